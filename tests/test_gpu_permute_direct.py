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


CLAIM = {"z": [3_000_001, 1 << 25, (1 << 25) + 1], "d": [(1 << 24) + 5, 3 << 23, (3 << 23) + 1]}


@pytest.mark.parametrize("ty,n", [(ty, n) for ty in "zd" for n in CLAIM[ty]])
@pytest.mark.parametrize("order", ["random", "rotate", "reverse"])
def test_partition_first_pass(cv, ty, n, order):
    """The partition's first pass claims its slots up to 2^25 ints or 3 2^23
    doubles and takes them from histograms above; rotations and reversals
    send whole waves to one bucket."""
    import torch
    dt = torch.float64 if ty == "d" else torch.int32
    i = torch.arange(n, device=cv.device)
    g = torch.Generator(device=cv.device)
    g.manual_seed(n)
    p = {"random": lambda: torch.randperm(n, generator=g, device=cv.device), "rotate": lambda: (i + n // 3) % n,
         "reverse": lambda: n - 1 - i}[order]().int()
    s = (i * 7 - n).to(dt)
    d = torch.zeros(n + 1, dtype=dt, device=cv.device)
    print("partition first pass", ty, n, order, flush=True)
    call(cv, ty, d, s, p, n)
    want = torch.empty(n, dtype=dt, device=cv.device)
    want[p.long()] = s
    assert torch.equal(d[:n], want) and float(d[n]) == 0.0
    assert cv.lib.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("ty,n", [("z", 5000), ("z", 3_000_001), ("z", (1 << 25) + 9), ("d", (1 << 24) + 5)])
def test_partition_errors(cv, ty, n):
    """A duplicate and an index out of range where the permute partitions (or
    scatters one block in LDS, which sees the range only)."""
    import torch
    dt = torch.float64 if ty == "d" else torch.int32
    p = torch.randperm(n, device=cv.device).int()
    s = torch.arange(n, device=cv.device).to(dt)
    buf = torch.full((n + 4096,), -7, dtype=dt, device=cv.device)
    for kind in ("duplicate", "range"):
        q = p.clone()
        if kind == "duplicate":
            if n <= 8192:
                continue
            q[(p == n - 1).nonzero()[0, 0]] = 3
        else:
            q[5], q[7] = n + 1000, -3
        print("partition error", ty, n, kind, flush=True)
        call(cv, ty, buf[:n], s, q, n)
        assert cv.lib.cvlhip_check_device_errors() != 0, kind
        assert torch.all(buf[n:] == -7)


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
