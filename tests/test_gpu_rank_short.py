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


# The ends of each rule above one workgroup: small tiles (to 2^19 keys),
# grouped tile counts and direct ranks (to 2^23), then the column scans and
# the inverse's first pass inside the last one.
LONG = [16385, 32769, (1 << 19) - 1, 1 << 19, (1 << 19) + 1, (1 << 21) + 1, 1 << 23, (1 << 23) + 1]


@pytest.mark.parametrize("n", LONG)
def test_rank_rules(cv, n):
    import torch
    rng = np.random.default_rng(n)
    print("rank rules", n, flush=True)
    for ty, x in (("z", rng.integers(-2 ** 31, 2 ** 31, n).astype(np.int32)), ("d", rng.uniform(-1, 1, n))):
        s = torch.from_numpy(x).to(cv.device)
        d = torch.empty(n, dtype=torch.int32, device=cv.device)
        order = np.argsort(x, kind="stable")
        want = np.empty(n, np.int32)
        want[order] = np.arange(n, dtype=np.int32)
        L = cv.lib
        getattr(L, f"rku_lu{ty}")(d, s, n, cv.scratch(getattr(L, f"rku_lu{ty}_scratch")(n)))
        eq(host(d), want, f"rank {ty} {n}")
    assert cv.lib.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("n", [20_001, (1 << 19) + 3, (1 << 21) + 5])
def test_segmented_rank_rules(cv, n):
    """Segment passes after the key passes, empty segments among them, and
    keys all equal (only segment passes reorder anything, then nothing)."""
    import torch
    rng = np.random.default_rng(n)
    lens = rng.geometric(1 / 40, size=n).astype(np.int64)
    lens = lens[np.cumsum(lens) <= n]
    lens = np.append(lens, n - lens.sum())
    lens = np.insert(lens, [0, 5, lens.size // 2], 0).astype(np.int32)
    sd = cv.segd(lens)
    for kind in ("random", "equal", "low"):
        x = {"random": rng.integers(-2 ** 31, 2 ** 31, n), "equal": np.full(n, 3), "low": rng.integers(0, 200, n)}[kind]
        x = x.astype(np.int32)
        s = torch.from_numpy(x).to(cv.device)
        d = torch.empty(n, dtype=torch.int32, device=cv.device)
        print("segmented rank", n, kind, flush=True)
        cv.lib.rku_lez(d, s, sd, n, lens.size, cv.scratch(cv.lib.rku_lez_scratch(n, lens.size)))
        eq(host(d), O.rank(x, True, lens), f"segmented rank {kind} {n}")
    assert cv.lib.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("n", [16_385, 40_003, (1 << 19) + 3, (1 << 21) + 5])
def test_ranks_whose_lowest_digit_is_constant(cv, n):
    """Pass 0 is launched before the host knows that it has nothing to do:
    ints that vary in higher digits only or not at all, doubles of whole
    numbers, plain and segmented, up and down, aligned or not."""
    import torch
    rng = np.random.default_rng(n)
    lens = np.bincount(rng.integers(0, 700, n), minlength=700).astype(np.int32)
    sd, L = cv.segd(lens), cv.lib
    keys = {"equal": np.full(n, -9, np.int32), "digit 1": (rng.integers(0, 256, n) << 8).astype(np.int32),
            "digit 3": (rng.integers(-128, 128, n) << 24).astype(np.int32),
            "digits 1 to 3": (rng.integers(-2 ** 23, 2 ** 23, n) << 8).astype(np.int32),
            "whole": rng.integers(-500, 500, n).astype(np.float64), "equal d": np.full(n, 0.1)}
    for kind, x in keys.items():
        ty = "d" if x.dtype == np.float64 else "z"
        print("constant low digit", n, kind, flush=True)
        for shift in (0, 1):
            s = torch.empty(n + shift, dtype=torch.float64 if ty == "d" else torch.int32, device=cv.device)[shift:]
            s.copy_(torch.from_numpy(x))
            d = torch.empty(n, dtype=torch.int32, device=cv.device)
            for ud in "ud":
                getattr(L, f"rk{ud}_lu{ty}")(d, s, n, cv.scratch(getattr(L, f"rk{ud}_lu{ty}_scratch")(n)))
                eq(host(d), O.rank(x, ud == "u"), f"{kind} {n} {ud}")
        getattr(L, f"rku_le{ty}")(d, s, sd, n, lens.size, cv.scratch(getattr(L, f"rku_le{ty}_scratch")(n, lens.size)))
        eq(host(d), O.rank(x, True, lens), f"segmented {kind} {n}")
    assert L.cvlhip_check_device_errors() == 0
