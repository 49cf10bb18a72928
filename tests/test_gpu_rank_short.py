"""Ranks of vectors that one workgroup holds (at most 16384 ints or 8192
doubles): every count of keys per lane, one key less and more than it takes,
the last length of that path and the first after it, against the C oracle.
Keys: random, all equal, few values, one varying digit, signed zeros,
infinities and NaN among doubles; ranks up and down, aligned or not."""
import numpy as np
import pytest

from gpu_util import eq, host
from oracle import oracle as O

pytestmark = pytest.mark.gpu

INTS = [1, 2, 63, 64, 65, 1000, 1023, 1024, 1025, 2048, 2049, 3073, 4097, 6145, 8193, 12289, 16383, 16384, 16385]
DOUBLES = [1, 64, 1023, 1025, 2049, 3072, 4097, 6145, 8191, 8192, 8193]


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


def check(cv, x, ty, what):
    import torch
    n = x.size
    for shift in (0, 1):
        t = torch.empty(n + shift, dtype=torch.float64 if ty == "d" else torch.int32, device=cv.device)
        s = t[shift:]
        s.copy_(torch.from_numpy(x))
        d = torch.full((n + 1,), -7, dtype=torch.int32, device=cv.device)
        for ud, up in (("u", True), ("d", False)):
            L = cv.lib
            getattr(L, f"rk{ud}_lu{ty}")(d, s, n, cv.scratch(getattr(L, f"rk{ud}_lu{ty}_scratch")(n)))
            eq(host(d[:n]), O.rank(x, up), f"{what} {ud} shift {shift}")
            assert int(d[n]) == -7, what
    assert cv.lib.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("n", INTS)
def test_short_int_ranks(cv, n):
    rng = np.random.default_rng(n)
    print("short int rank", n, flush=True)
    check(cv, rng.integers(-2 ** 31, 2 ** 31, n).astype(np.int32), "z", f"random {n}")
    check(cv, np.full(n, -5, np.int32), "z", f"equal {n}")
    check(cv, rng.integers(0, 3, n).astype(np.int32), "z", f"few {n}")
    check(cv, (rng.integers(0, 256, n) << 16).astype(np.int32), "z", f"digit 2 {n}")


@pytest.mark.parametrize("n", DOUBLES)
def test_short_double_ranks(cv, n):
    rng = np.random.default_rng(n)
    print("short double rank", n, flush=True)
    check(cv, rng.uniform(-1, 1, n), "d", f"random {n}")
    check(cv, rng.integers(-2, 3, n).astype(np.float64), "d", f"few {n}")
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, -np.nan, 5e-324, 1.7e308])
    check(cv, special[rng.integers(0, special.size, n)], "d", f"special {n}")
