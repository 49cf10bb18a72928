"""Unsegmented scans in one small tile (4096 and 16384 ints, 2048 and 8192
doubles) and over tile aggregates (tiles of 8192 ints or 4096 doubles, up to
2^23 ints or 20 2^20 doubles): the ends of each rule and of the tiles, results
over their inputs, unaligned vectors, and the order-sensitive double maximum
(which of two equal zeros comes last)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

INTS = [1, 4095, 4096, 4097, 16384, 16385, 49152, 49153, 7 * 8192, 7 * 8192 + 1, 1_000_003, 1 << 23, (1 << 23) + 1]
DOUBLES = [1, 2048, 2049, 8192, 8193, 16384, 16385, 9 * 4096, 9 * 4096 + 1, 1_000_003, 20 << 20, (20 << 20) + 1]


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


def vec(x, shift):
    import torch
    t = torch.empty(x.numel() + shift + 1, dtype=x.dtype, device=x.device)[shift:]
    t[:-1] = x
    t[-1] = 99
    return t


@pytest.mark.parametrize("n", INTS)
def test_int_scans(cv, n):
    import torch
    L = cv.lib
    g = torch.Generator(device=cv.device)
    g.manual_seed(n)
    x = torch.randint(-2 ** 31, 2 ** 31, (n,), generator=g, device=cv.device, dtype=torch.int32)
    want = {"add": torch.cumsum(x, 0, dtype=torch.int64) - x, "max": torch.full((n,), -2 ** 31, device=cv.device)}
    want["add"] = ((want["add"] + 2 ** 31) & 0xFFFFFFFF) - 2 ** 31
    want["max"][1:] = torch.cummax(x, 0).values[:-1]
    print("int scans", n, flush=True)
    for op in ("add", "max"):
        scr = cv.scratch(getattr(L, f"{op}_suz_scratch")(n))
        for shift in (0, 1):
            s, d = vec(x, shift), vec(torch.zeros_like(x), shift)
            getattr(L, f"{op}_suz")(d, s, n, scr)
            assert torch.equal(d[:n].long(), want[op]) and int(d[n]) == 99, (op, shift)
            getattr(L, f"{op}_suz")(s, s, n, scr)
            assert torch.equal(s[:n].long(), want[op]) and int(s[n]) == 99, (op, shift, "in place")
    assert L.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("n", DOUBLES)
def test_double_scans(cv, n):
    import torch
    L = cv.lib
    g = torch.Generator(device=cv.device)
    g.manual_seed(n)
    x = torch.rand(n, generator=g, device=cv.device, dtype=torch.float64) * 2 - 1
    hi = torch.round(x * 2.0 ** 30)                          # sums of the leading bits are exact in integers
    h, lo = hi.long(), x - hi * 2.0 ** -30
    exact = (torch.cumsum(h, 0) - h).double() * 2.0 ** -30 + (torch.cumsum(lo, 0) - lo)
    bound = 2 * (np.ceil(np.log2(max(n, 2))) + 2) * 2.0 ** -53 * torch.cumsum(x.abs(), 0)
    top = torch.full_like(x, float(np.float32(-1.0e36)))
    top[1:] = torch.cummax(x, 0).values[:-1]
    print("double scans", n, flush=True)
    first = None
    for shift in (0, 1):
        scr = cv.scratch(L.add_sud_scratch(n))
        s, d = vec(x, shift), vec(torch.zeros_like(x), shift)
        L.add_sud(d, s, n, scr)
        assert bool(((d[:n] - exact).abs() <= bound).all()) and float(d[n]) == 99, shift
        first = d[:n].clone() if first is None else first
        assert torch.equal(d[:n], first), "a scan's bits differ between calls"
        L.max_sud(d, s, n, scr)
        assert torch.equal(d[:n], top) and float(d[n]) == 99, shift
        L.add_sud(s, s, n, scr)
        assert torch.equal(s[:n], first), "in place"
    assert L.cvlhip_check_device_errors() == 0


def test_zero_signs(cv):
    """Zeros of both signs in a descending tail: the running maximum keeps the
    last of equal values, across tiles."""
    import torch
    n = 100_000
    x = np.full(n, -1.0)
    x[10_000], x[50_000], x[70_000] = 0.0, -0.0, 0.0
    d = torch.empty(n, dtype=torch.float64, device=cv.device)
    cv.lib.max_sud(d, torch.from_numpy(x).to(cv.device), n, cv.scratch(cv.lib.max_sud_scratch(n)))
    got = np.signbit(d.cpu().numpy())
    assert not got[10_001:50_001].any() and got[50_001:70_001].all() and not got[70_001:].any()
