"""Shared helpers for the GPU parity tests: device tensors in, numpy out,
every call through the C-ABI of libcvl_hip.so."""
import math

import numpy as np


def dtype_of(ty):
    import torch
    return torch.float64 if ty == "d" else torch.int32


def np_dtype(ty):
    return np.float64 if ty == "d" else np.int32


def host(t):
    return t.detach().cpu().numpy()


def eq(a, b, what=""):
    a = np.asarray(a)
    b = np.asarray(b)
    assert a.shape == b.shape, (what, a.shape, b.shape)
    if a.dtype == np.float64:
        ok = np.array_equal(a.view(np.int64), b.view(np.int64))
    else:
        ok = np.array_equal(a, b)
    if not ok:
        bad = np.nonzero(a != b)[0] if a.dtype != np.float64 else np.nonzero(a.view(np.int64) != b.view(np.int64))[0]
        raise AssertionError(f"{what}: {bad.size} mismatches, first at {bad[:5]}: got {a[bad[:5]]} want {b[bad[:5]]}")


def fp_add_tol(absprefix, seglen):
    """Tolerance for a float +-scan element: 2(ceil(log2 L)+2) 2^-53 sum|x|."""
    L = max(int(seglen), 2)
    return 2.0 * (math.ceil(math.log2(L)) + 2) * 2.0 ** -53 * absprefix


def fp_add_tol_vec(absprefix, seglen):
    """Vector form of fp_add_tol."""
    L = np.maximum(np.asarray(seglen, np.int64), 2)
    return 2.0 * (np.ceil(np.log2(L)) + 2) * 2.0 ** -53 * np.asarray(absprefix)


def seg_lengths_per_element(lens):
    lens = np.asarray(lens, np.int64)
    return np.repeat(lens, lens)


class Guarded:
    """Scratch of exactly the promised units, followed by a guard that no
    kernel may write: use it as the call's scratch, then call check()."""
    GUARD = 32 << 10

    def __init__(self, cv, units):
        import torch
        self.nbytes = 8 * int(units)
        self.buf = torch.full((self.nbytes + self.GUARD,), 0xA5, dtype=torch.uint8, device=cv.device)

    def data_ptr(self):
        return self.buf.data_ptr()

    def check(self, what=""):
        bad = (self.buf[self.nbytes:] != 0xA5).nonzero()
        assert bad.numel() == 0, f"{what}: {bad.numel()} bytes written past the scratch, first at +{int(bad[0])}"
