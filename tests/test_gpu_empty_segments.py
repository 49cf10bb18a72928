"""Identities of empty segments, written by the reduction's own launch (no
more segments than elements, at most 2^20) or by one before it: both sides of
both bounds, short and long vectors, leading, trailing and adjacent empty
segments, for the serial identities of + and max."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def shapes():
    rng = np.random.default_rng(9)

    def some(n, m):                      # n elements thrown into m segments
        return np.bincount(rng.integers(0, m, n), minlength=m).astype(np.int32)
    return [("short", some(500, 400)), ("more_segments", some(500, 501)), ("equal", some(3000, 3000)),
            ("mid", np.insert(some(100_000, 60_000), [0, 0, 60_000], 0)), ("mid_more", some(40_000, 200_000)),
            ("last_folded", some(1 << 20, 1 << 20)), ("first_not", some((1 << 20) + 1, (1 << 20) + 1)),
            ("mostly_empty", np.concatenate([np.zeros(5000, np.int32), [70_000], np.zeros(60_000, np.int32)]))]


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


@pytest.mark.parametrize("name,lens", shapes(), ids=[s[0] for s in shapes()])
def test_empty_segment_identities(cv, name, lens):
    import torch
    lens = np.asarray(lens, np.int32)
    n, m = int(lens.sum()), lens.size
    rng = np.random.default_rng(n)
    z, x = rng.integers(-1000, 1000, n).astype(np.int32), rng.uniform(-1, 1, n)
    at = np.concatenate([[0], np.cumsum(lens)[:-1]])[lens > 0]
    want = {"add_rez": np.zeros(m, np.int32), "max_rez": np.full(m, -2 ** 31, np.int32),
            "max_red": np.full(m, np.float64(np.float32(-1.0e36)))}
    want["add_rez"][lens > 0] = np.add.reduceat(z, at)
    want["max_rez"][lens > 0] = np.maximum.reduceat(z, at)
    want["max_red"][lens > 0] = np.maximum.reduceat(x, at)
    sd = cv.segd(lens)
    print("empty segments", name, n, m, flush=True)
    for fn, w in want.items():
        src = torch.from_numpy(x if fn.endswith("d") else z).to(cv.device)
        d = torch.full((m + 1,), 5, dtype=src.dtype, device=cv.device)
        getattr(cv.lib, fn)(d, src, sd, n, m, cv.scratch(getattr(cv.lib, fn + "_scratch")(n, m)))
        assert np.array_equal(d[:m].cpu().numpy(), w), fn
        assert float(d[m]) == 5
    assert cv.lib.cvlhip_check_device_errors() == 0
