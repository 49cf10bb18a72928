"""Permutes with collisions and defaults (dpe, dfp, fpm) against numpy's
assignment in element order (the last writer wins): the ends of the place
kernel's lanes and workgroups (1024 destinations), both sides of the rule for
few sources (below n_d / 32 of at least 2^21 destinations), repeated indices,
flags, results over their default vector and off 16-byte alignment, and
indices out of range."""
import numpy as np
import pytest

from gpu_util import eq, host

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (5, 3), (1000, 1023), (3000, 1024), (1000, 1025), (40_000, 30_000), (1 << 17, 1 << 22),
          ((1 << 17) - 1, 1 << 22), (1, 1 << 22), (900_000, (1 << 20) + 3), (30_000, (1 << 22) - 1), (0, 2000),
          (1 << 16, 1 << 21), ((1 << 16) - 1, 1 << 21), (1000, (1 << 21) - 1)]


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


@pytest.mark.parametrize("n,n_d", SHAPES)
@pytest.mark.parametrize("ty", ["z", "d"])
def test_default_permutes(cv, ty, n, n_d):
    import torch
    L = cv.lib
    rng = np.random.default_rng(n * 7 + n_d)
    dt = np.float64 if ty == "d" else np.int32
    s, v = np.arange(1, n + 1).astype(dt), -np.arange(1, n_d + 1).astype(dt)
    idx = rng.integers(0, n_d, n).astype(np.int32)             # with repeats
    f = rng.integers(0, 2, n).astype(np.int32)
    dev = lambda a: torch.from_numpy(a).to(cv.device)
    ds, di, df = dev(s), dev(idx), dev(f)
    print("default permute", ty, n, n_d, flush=True)
    for kind in ("dpe", "dfp", "fpm"):
        live = np.ones(n, bool) if kind == "dpe" else f != 0
        want = v.copy()
        want[idx[live]] = s[live]                                # numpy assigns in order: the last one stays
        scr = cv.scratch(getattr(L, f"{kind}_pu{ty}_scratch")(n, n_d))
        for shift in (0, 1):
            buf = torch.full((n_d + 2 + shift,), 99, dtype=ds.dtype, device=cv.device)
            d = buf[shift:shift + n_d]
            for over in (False, True):
                dv = d if over else dev(v)
                if over or kind == "fpm":
                    d.copy_(dev(v))                              # fpm keeps what nobody aims at
                fn = getattr(L, f"{kind}_pu{ty}")
                if kind == "dpe":
                    fn(d, ds, di, dv, n, n_d, scr)
                elif kind == "dfp":
                    fn(d, ds, di, df, dv, n, n_d, scr)
                else:
                    fn(d, ds, di, df, n, n_d, scr)
                eq(host(d), want, f"{kind} {shift} {over}")
                assert torch.all(buf[shift + n_d:] == 99)
    assert L.cvlhip_check_device_errors() == 0
    if n:
        bad = idx.copy()
        bad[0] = n_d
        want = v.copy()
        want[bad[1:]] = s[1:]
        d = torch.empty(n_d, dtype=ds.dtype, device=cv.device)
        getattr(L, f"dpe_pu{ty}")(d, ds, dev(bad), dev(v), n, n_d, scr)
        eq(host(d), want, "out of range")
        assert L.cvlhip_check_device_errors() != 0
