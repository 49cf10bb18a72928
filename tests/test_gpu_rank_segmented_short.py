"""Segmented ranks of short vectors, against the C oracle, in scratch of
exactly the promised size with a guard behind it: lengths at the edges of the
small tiles, few segments and more than elements (three digits of segment
numbers), empty ones among them; ints and doubles, up and down."""
import numpy as np
import pytest

from gpu_util import Guarded, eq, host
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 129, 192, 193, 1000, 1024, 1025, 4097])
def test_short_segmented_ranks(cv, n):
    import torch
    L = cv.lib
    rng = np.random.default_rng(n)
    for m in (2, 3, 300, 70_000):
        lens = np.bincount(rng.integers(0, m, n), minlength=m).astype(np.int32)
        sd = cv.segd(lens)
        for ty, x in (("z", rng.integers(-50, 50, n).astype(np.int32)), ("z", np.full(n, 7, np.int32)),
                      ("d", rng.uniform(-1, 1, n)), ("d", rng.integers(-2, 3, n).astype(np.float64))):
            s = torch.from_numpy(x).to(cv.device)
            for ud in "ud":
                print("short segmented rank", n, m, ty, ud, flush=True)
                f = getattr(L, f"rk{ud}_le{ty}")
                scr = Guarded(cv, getattr(L, f"rk{ud}_le{ty}_scratch")(n, m))
                d = torch.full((n + 1,), -7, dtype=torch.int32, device=cv.device)
                f(d, s, sd, n, m, scr)
                eq(host(d[:n]), O.rank(x, ud == "u", lens), f"rk{ud}_le{ty} n={n} m={m}")
                assert int(d[n]) == -7
                scr.check(f"rk{ud}_le{ty} n={n} m={m}")
    assert L.cvlhip_check_device_errors() == 0
