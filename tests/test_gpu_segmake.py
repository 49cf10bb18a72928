"""Segmented distribute and index: runs of four ints or two doubles, at the
ends of tiles (1024 elements; 2048 from 2^21 elements on), segments shorter
and longer than a run, empty ones first, last and in a row, on aligned and
unaligned results."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


def lengths(kind, n, rng):
    if kind == "ones":
        return np.ones(n, np.int32)
    mean = {"short": 3, "mid": 30, "long": 5000}[kind]
    z = rng.geometric(1 / mean, size=n // mean + 16).astype(np.int64)
    z = z[np.cumsum(z) <= n]
    z = np.append(z, n - z.sum())
    if kind != "long":
        z = np.insert(z, [0, 0, z.size // 2, z.size // 2, z.size], 0)
    return z.astype(np.int32)


@pytest.mark.parametrize("n", [1, 3, 1023, 1024, 1025, 40_001, (1 << 21) - 1, 1 << 21, (1 << 21) + 2049])
@pytest.mark.parametrize("kind", ["ones", "short", "mid", "long"])
def test_segmented_distribute_and_index(cv, n, kind):
    import torch
    L, dev = cv.lib, cv.device
    rng = np.random.default_rng(n)
    lens = lengths(kind, n, rng)
    m = lens.size
    sd = cv.segd(lens)
    l = torch.from_numpy(lens.astype(np.int64)).to(dev)
    own = torch.repeat_interleave(torch.arange(m, device=dev), l)
    at = torch.arange(n, device=dev) - (torch.cumsum(l, 0) - l)[own]
    init = torch.from_numpy(rng.integers(-2 ** 31, 2 ** 31, m).astype(np.int32)).to(dev)
    step = torch.from_numpy(rng.integers(-5, 6, m).astype(np.int32)).to(dev)
    val = torch.rand(m, device=dev, dtype=torch.float64)
    want = (init.long()[own] + step.long()[own] * at).to(torch.int32)
    print("segmented make", kind, n, m, flush=True)
    for shift in (0, 1):
        d = torch.full((n + 1 + shift,), -7, device=dev, dtype=torch.int32)[shift:]
        e = torch.full((n + 1 + shift,), -7, device=dev, dtype=torch.float64)[shift:]
        L.ind_lez(d, init, step, sd, n, m, None)
        assert torch.equal(d[:n], want) and int(d[n]) == -7, shift
        L.dis_vez(d, init, sd, n, m, None)
        assert torch.equal(d[:n], init[own]) and int(d[n]) == -7, shift
        L.dis_ved(e, val, sd, n, m, None)
        assert torch.equal(e[:n], val[own]) and float(e[n]) == -7.0, shift
    assert L.cvlhip_check_device_errors() == 0
