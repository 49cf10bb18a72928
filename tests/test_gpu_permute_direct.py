"""Permutes that are scattered directly: the ends of each workgroup shape
(2^18, 2^19, 2^23 elements) and of the rule itself (2^21 ints, 2^24
doubles), aligned or not, and the errors that the partition reports too:
indices out of range, and indices that are no permutation (a destination
block of 8192 elements that more than 8192 indices aim at)."""
import numpy as np
import pytest

from gpu_util import eq, host

pytestmark = pytest.mark.gpu

EDGES = {"z": [8193, (1 << 18) - 1, 1 << 18, (1 << 18) + 1, (1 << 19) + 1, 1 << 21, (1 << 21) + 1],
         "d": [8193, (1 << 18) + 1, 1 << 19, (1 << 19) + 3, 1 << 23, (1 << 23) + 1, 1 << 24, (1 << 24) + 1]}


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


def call(cv, ty, d, s, p, n):
    getattr(cv.lib, f"smp_pu{ty}")(d, s, p, n, cv.scratch(getattr(cv.lib, f"smp_pu{ty}_scratch")(n)))


@pytest.mark.parametrize("ty,n", [(ty, n) for ty in "zd" for n in EDGES[ty]])
def test_direct_permute_edges(cv, ty, n):
    import torch
    dt = torch.float64 if ty == "d" else torch.int32
    g = torch.Generator(device=cv.device)
    g.manual_seed(n)
    print("direct permute", ty, n, flush=True)
    for shift in (0, 1):
        p = torch.empty(n + shift, dtype=torch.int32, device=cv.device)[shift:]
        s = torch.empty(n + shift, dtype=dt, device=cv.device)[shift:]
        p.copy_(torch.randperm(n, generator=g, device=cv.device))
        s.copy_(torch.arange(n, device=cv.device) * 3 - n)
        d = torch.zeros(n + 1, dtype=dt, device=cv.device)
        call(cv, ty, d, s, p, n)
        want = torch.empty(n, dtype=dt, device=cv.device)
        want[p.long()] = s
        assert torch.equal(d[:n], want), (ty, n, shift)
        assert float(d[n]) == 0.0
    assert cv.lib.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("ty", ["z", "d"])
@pytest.mark.parametrize("n", [9000, 300_000, 1_000_003])
def test_direct_permute_errors(cv, ty, n):
    """One duplicate into a full block raises the error word, as does an
    index out of range; the other values land and nothing outside is
    written."""
    import torch
    dt = torch.float64 if ty == "d" else torch.int32
    rng = np.random.default_rng(n)
    for kind in ("duplicate", "range"):
        p = rng.permutation(n).astype(np.int32)
        if kind == "duplicate":
            k = int(np.nonzero(p == n - 1)[0][0])
            p[k] = 3                                     # block 0 gets one index too many
        else:
            p[5], p[7] = n + 1000, -3
        s = torch.arange(n, device=cv.device).to(dt)
        buf = torch.full((n + 4096,), -7, dtype=dt, device=cv.device)
        print("direct permute error", ty, n, kind, flush=True)
        call(cv, ty, buf[:n], s, torch.from_numpy(p).to(cv.device), n)
        assert cv.lib.cvlhip_check_device_errors() != 0, kind
        assert torch.all(buf[n:] == -7)
        got, ok = host(buf[:n]), (p >= 0) & (p < n)
        if kind == "duplicate":
            ok[p == 3] = False
        eq(got[p[ok]].astype(np.int64), np.arange(n)[ok], kind)
