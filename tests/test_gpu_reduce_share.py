"""Host-returning reductions whose blocks combine in the last one to finish:
one block, the edges of the counter groups (31, 32 and 33 blocks of 1024
ints or 512 doubles) and the most blocks, calls of different operators, types
and sizes following each other over the same words, and the ordered double
maximum (the last of equal values, so the sign of a zero), against exact
results."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

INTS = [1, 1024, 1025, 31 * 1024, 31 * 1024 + 1, 32 * 1024, 33 * 1024, 64 * 1024 + 7, 2048 * 1024, 2048 * 1024 + 1, 5_000_003]


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


@pytest.mark.parametrize("n", INTS)
def test_reductions_follow_each_other(cv, n):
    import torch
    L = cv.lib
    rng = np.random.default_rng(n)
    z = rng.integers(-2 ** 31, 2 ** 31, n).astype(np.int32)
    d = rng.uniform(-1, 1, (n + 1) // 2)
    dz, dd = torch.from_numpy(z).to(cv.device), torch.from_numpy(d).to(cv.device)
    scr = cv.scratch(L.add_rud_scratch(n))
    total = int(np.sum(z, dtype=np.int64)) & 0xFFFFFFFF
    want = {"add_ruz": total - (1 << 32) if total >> 31 else total, "max_ruz": int(z.max()), "min_ruz": int(z.min()),
            "xor_ruz": int(np.bitwise_xor.reduce(z)), "pk1_luv": int(np.count_nonzero(z))}
    exact = float(np.sum(d.astype(np.longdouble)))
    tol = 2 * (np.ceil(np.log2(max(d.size, 2))) + 2) * 2.0 ** -53 * float(np.abs(d).sum())
    print("reductions", n, flush=True)
    first = None
    for _ in range(3):
        for name, w in want.items():
            assert getattr(L, name)(dz, n, scr) == w, name
            assert L.max_rud(dd, d.size, scr) == d.max()
            assert L.min_rud(dd, d.size, scr) == d.min()
        s = L.add_rud(dd, d.size, scr)
        assert abs(s - exact) <= tol
        first = s if first is None else first
        assert s == first, "a sum's bits differ between calls"
        assert L.add_ruz(dz, min(n, 1500), scr) == int(np.sum(z[:1500], dtype=np.int64).astype(np.int32))
    assert L.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("n", [512, 40_000, 3_000_000])
def test_ordered_maximum(cv, n):
    """Zeros of both signs under an all-negative rest: the serial fold keeps
    the last of equal values."""
    import torch
    L = cv.lib
    x = np.full(n, -1.0)
    for a, b in ((n // 3, 2 * n // 3), (2 * n // 3, n // 3)):
        y = x.copy()
        y[a], y[b] = 0.0, -0.0
        r = L.max_rud(torch.from_numpy(y).to(cv.device), n, cv.scratch(L.max_rud_scratch(n)))
        assert r == 0.0 and np.signbit(r) == np.signbit(y[max(a, b)]), n
