"""Calls that lay out areas of their own in the scratch, in scratch of exactly
the size their _scratch function promises: a guard behind it stays as it
was, and the results are those of a call with plenty.  Sizes at the ends of
each rule (one tile, counted or aggregated tiles, look-back; direct, claimed
and scanned permutes; small, grouped and scanned ranks; descriptors of one
workgroup, a few tiles, and so many that their sums are scanned)."""
import numpy as np
import pytest

from gpu_util import Guarded

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


def values(cv, n, ty, seed=1):
    import torch
    g = torch.Generator(device=cv.device)
    g.manual_seed(seed * 1000 + n)
    if ty == "d":
        return torch.randint(-999, 1000, (n,), generator=g, device=cv.device, dtype=torch.int32).to(torch.float64)
    return torch.randint(-2 ** 31, 2 ** 31, (n,), generator=g, device=cv.device, dtype=torch.int32)


def check(cv, name, units, call, outs):
    """call(scratch, out) twice; outs: how to make an output (or none)."""
    import torch
    a, b = outs(), outs()
    scr = Guarded(cv, units)
    ra = call(scr, a)
    scr.check(name)
    rb = call(cv.scratch(units), b)
    assert ra == rb, name
    if a is not None:
        assert torch.equal(a, b), name


SCANS = [1, 1024, 4097, 49_152, 49_153, 100_003, 1 << 23, (1 << 23) + 1, 20 << 20, (20 << 20) + 1]
PACKS = [1, 65_536, 65_537, 300_001, 1 << 24, (1 << 24) + 1]
PERMUTES = [1, 8192, 8193, 1 << 18, (1 << 21) - 1, 1 << 21, (1 << 21) + 1, 1 << 24, (1 << 24) + 1, (1 << 25) + 1]
RANKS = [1, 8193, 16_385, 1 << 19, (1 << 19) + 1, 1 << 21, (1 << 22) + 1, 1 << 23, (1 << 23) + 1]


@pytest.mark.parametrize("ty", ["z", "d"])
@pytest.mark.parametrize("n", SCANS)
def test_scans_and_reductions(cv, n, ty):
    import torch
    L, s = cv.lib, values(cv, n, ty)
    print("guarded scan", n, ty, flush=True)
    new = lambda: torch.full_like(s, 5)
    for op in ("add", "max"):
        f, r = getattr(L, f"{op}_su{ty}"), getattr(L, f"{op}_ru{ty}")
        check(cv, f"{op}_su{ty} {n}", getattr(L, f"{op}_su{ty}_scratch")(n), lambda scr, d: f(d, s, n, scr), new)
        check(cv, f"{op}_ru{ty} {n}", getattr(L, f"{op}_ru{ty}_scratch")(n), lambda scr, d: r(s, n, scr), lambda: None)
    assert L.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("ty", ["z", "d"])
@pytest.mark.parametrize("n", PACKS)
def test_packs(cv, n, ty):
    import torch
    L, s = cv.lib, values(cv, n, ty)
    f = (values(cv, n, "z", 2) & 1).contiguous()
    k = int(f.sum())
    print("guarded pack", n, ty, flush=True)
    check(cv, f"pk1 {n}", L.pk1_luv_scratch(n), lambda scr, d: L.pk1_luv(f, n, scr), lambda: None)
    p = getattr(L, f"pk2_lu{ty}")
    check(cv, f"pk2 {n}", getattr(L, f"pk2_lu{ty}_scratch")(n), lambda scr, d: p(d, s, f, n, k, scr),
          lambda: torch.full((k,), 5, dtype=s.dtype, device=cv.device))
    assert L.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("ty", ["z", "d"])
@pytest.mark.parametrize("n", PERMUTES)
def test_permutes(cv, n, ty):
    import torch
    L, s = cv.lib, values(cv, n, ty)
    g = torch.Generator(device=cv.device)
    g.manual_seed(n)
    p = torch.randperm(n, generator=g, device=cv.device).to(torch.int32)
    print("guarded permute", n, ty, flush=True)
    new = lambda: torch.full_like(s, 5)
    f, e = getattr(L, f"smp_pu{ty}"), getattr(L, f"dpe_pu{ty}")
    check(cv, f"smp {n}", getattr(L, f"smp_pu{ty}_scratch")(n), lambda scr, d: f(d, s, p, n, scr), new)
    k = max(1, n // 3)
    check(cv, f"dpe {n}", getattr(L, f"dpe_pu{ty}_scratch")(k, n), lambda scr, d: e(d, s, p, s, k, n, scr), new)
    assert L.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("ty", ["z", "d"])
@pytest.mark.parametrize("n", RANKS)
def test_ranks(cv, n, ty):
    import torch
    L, s = cv.lib, values(cv, n, ty)
    rng = np.random.default_rng(n)
    new = lambda: torch.full((n,), 5, dtype=torch.int32, device=cv.device)
    print("guarded rank", n, ty, flush=True)
    f, e = getattr(L, f"rku_lu{ty}"), getattr(L, f"rkd_le{ty}")
    check(cv, f"rku_lu{ty} {n}", getattr(L, f"rku_lu{ty}_scratch")(n), lambda scr, d: f(d, s, n, scr), new)
    for m in (2, 70_000):
        lens = np.bincount(rng.integers(0, m, n), minlength=m).astype(np.int32)
        sd = cv.segd(lens)
        check(cv, f"rkd_le{ty} {n} {m}", getattr(L, f"rkd_le{ty}_scratch")(n, m), lambda scr, d: e(d, s, sd, n, m, scr), new)
    assert L.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("n,m", [(5, 2), (3000, 4096), (3000, 4097), (200_000, 3), (1 << 20, 20_000), (300_000, 250_000),
                                 (1 << 22, (1 << 22) + 2049), (1 << 26, 7)])
def test_descriptors_and_segmented_calls(cv, n, m):
    import torch
    L = cv.lib
    rng = np.random.default_rng(n + m)
    lens = torch.from_numpy(np.bincount(rng.integers(0, m, n), minlength=m).astype(np.int32)).to(cv.device)
    words = L.siz_fos(n, m) * 2
    print("guarded descriptor", n, m, flush=True)
    check(cv, f"mke_fov {n} {m}", L.mke_fov_scratch(n, m), lambda scr, d: L.mke_fov(d, lens, n, m, scr),
          lambda: torch.zeros(words + 64, dtype=torch.int32, device=cv.device))
    sd = cv.segd(lens)
    for ty in "zd":
        s = values(cv, n, ty)
        f, r = getattr(L, f"add_se{ty}"), getattr(L, f"max_re{ty}")
        check(cv, f"add_se{ty} {n} {m}", getattr(L, f"add_se{ty}_scratch")(n, m),
              lambda scr, d: f(d, s, sd, n, m, scr), lambda: torch.full_like(s, 5))
        check(cv, f"max_re{ty} {n} {m}", getattr(L, f"max_re{ty}_scratch")(n, m),
              lambda scr, d: r(d, s, sd, n, m, scr), lambda: torch.full((m,), 5, dtype=s.dtype, device=cv.device))
    assert L.cvlhip_check_device_errors() == 0
