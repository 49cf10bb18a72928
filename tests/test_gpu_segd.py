"""Segment descriptors (mke_fov) read back section by section and compared
with their definition, for both construction paths: one workgroup for small
descriptors (m and the bitmap's word count at most 4096), three kernels
otherwise (tile sums, offsets, bitmap words).

Layout (byte offsets, each section 256-byte aligned): header (n, m as
int64) at 0; lens[m] at 256; offs[m+1] (exclusive sums, offs[m] = n); nz
(ids of the non-empty segments, in order); wcnt[W+1] (segment heads in the
32-element words before each word); heads[W+8] (bit k of word k/32 set when
a non-empty segment starts at element k).  W = ceil(n / 32).  The lengths
are the serial CVL's whole descriptor (nesl/cvl/serial/facilt.c:118-144)."""
import numpy as np
import pytest

from gpu_util import host

pytestmark = pytest.mark.gpu


def up256(b):
    return (b + 255) & ~255


def layout(n, m):
    words = (n + 31) // 32
    lens = 256
    offs = up256(lens + 4 * m)
    nz = up256(offs + 4 * (m + 1))
    wcnt = up256(nz + 4 * m)
    heads = up256(wcnt + 4 * (words + 1))
    return words, lens, offs, nz, wcnt, heads


def want(lens):
    lens = np.asarray(lens, np.int64)
    n, m = int(lens.sum()), lens.size
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    nz = np.nonzero(lens > 0)[0]
    words = (n + 31) // 32
    heads = np.zeros(words + 8, np.uint32)
    starts = offs[:-1][lens > 0]
    np.bitwise_or.at(heads, starts // 32, (np.uint32(1) << (starts % 32).astype(np.uint32)))
    pc = np.array([bin(int(h)).count("1") for h in heads[:words]], np.int64)
    wcnt = np.concatenate([[0], np.cumsum(pc)])
    return n, m, offs, nz, words, heads, wcnt


def shapes():
    rng = np.random.default_rng(21)

    def split(n, m, empty=0.0):
        cuts = np.sort(rng.integers(0, n + 1, m - 1))
        lens = np.diff(np.concatenate([[0], cuts, [n]]))
        if empty:
            lens[rng.random(m) < empty] = 0
        return lens.astype(np.int32)
    return [
        ("small", split(5000, 100, 0.1)),
        ("small_edge", split(4096 * 32, 4096, 0.1)),     # the largest one-workgroup descriptor
        ("few_long", split(500_000, 3000, 0.05)),        # one tile of lengths, bitmap above 4096 words
        ("mid_tiles", split(700_000, 20_000, 0.2)),      # several tiles of lengths and of words, empties
        ("mid_edge", split(1 << 20, 1 << 15, 0.1)),      # 8 tiles of each, exactly
        ("many_short", split(120_000, 50_000, 0.2)),     # more than 4096 lengths
        ("large_long", split(1 << 21, 70_000)),
        ("large_many", split(300_000, 200_000, 0.3)),
        ("all_empty", np.zeros(5000, np.int32)),
        ("singletons", np.ones(100_003, np.int32)),     # every bit of every bitmap word set
        ("pairs_empty", np.tile(np.array([1, 0, 2], np.int32), 40_000)),
        ("empty_ends", np.concatenate([[0, 0], split(200_000, 9000), [0]]).astype(np.int32)),
    ]


@pytest.mark.parametrize("name,lens", shapes(), ids=[s[0] for s in shapes()])
def test_descriptor_sections(cv, name, lens):
    n, m, offs, nz, words, heads, wcnt = want(lens)
    print("segd", name, n, m, flush=True)
    sd = cv.segd(lens)
    raw = host(sd.buf).view(np.uint8)
    W, o_lens, o_offs, o_nz, o_wcnt, o_heads = layout(n, m)
    assert W == words
    hdr = raw[:16].view(np.int64)
    assert hdr[0] == n and hdr[1] == m
    i32 = lambda off, k: raw[off:off + 4 * k].view(np.int32)
    assert np.array_equal(i32(o_lens, m), lens)
    assert np.array_equal(i32(o_offs, m + 1), offs)
    assert np.array_equal(i32(o_nz, nz.size), nz)
    assert np.array_equal(i32(o_wcnt, words + 1), wcnt)
    assert np.array_equal(raw[o_heads:o_heads + 4 * (words + 8)].view(np.uint32), heads)
    assert cv.lib.cvlhip_check_device_errors() == 0


@pytest.fixture(scope="module")
def cv():
    from neslgpu_amd.cvl import Cvl
    return Cvl()


# The three-kernel build at the edges of its tiles (2048 lengths) and chunks
# (256 bitmap words, 8192 elements), with segments that span many chunks (a
# wave writes their head counts together), and enough tiles that their sums
# are scanned by a kernel of their own (above 2048 tiles).
def edge_shapes():
    rng = np.random.default_rng(5)
    long = np.array([0, 40_000, 1, 0, 8192, 8191, 1, 300_000, 0, 2_000_000, 3, 0], np.int32)
    return [("one_tile", np.full(2048, 100, np.int32)), ("tile_and_one", np.full(2049, 100, np.int32)),
            ("long", long), ("one_long", np.array([0, 9_000_000, 0], np.int32)),
            ("chunk_heads", np.full(300, 8192, np.int32)), ("chunk_ragged", np.full(301, 8191, np.int32)),
            ("long_many", np.concatenate([np.ones(5000, np.int32), long, np.ones(5000, np.int32)])),
            ("many_tiles", rng.integers(0, 3, 2048 * 2048 + 17).astype(np.int32))]


@pytest.mark.parametrize("name,lens", edge_shapes(), ids=[s[0] for s in edge_shapes()])
def test_descriptor_edges(cv, name, lens):
    print("segd edge", name, lens.size, flush=True)
    lens64 = lens.astype(np.int64)
    n, m = int(lens64.sum()), lens.size
    offs = np.concatenate([[0], np.cumsum(lens64)])
    nz = np.nonzero(lens > 0)[0]
    W, o_lens, o_offs, o_nz, o_wcnt, o_heads = layout(n, m)
    bits = np.zeros((W + 8) * 32, np.uint8)
    bits[offs[:-1][lens > 0]] = 1
    heads = np.packbits(bits, bitorder="little").view(np.uint32)
    wcnt = np.concatenate([[0], np.cumsum(bits[:W * 32].reshape(W, 32).sum(1, dtype=np.int64))])
    raw = host(cv.segd(lens).buf).view(np.uint8)
    i32 = lambda off, k: raw[off:off + 4 * k].view(np.int32)
    assert list(raw[:16].view(np.int64)) == [n, m]
    assert np.array_equal(i32(o_lens, m), lens)
    assert np.array_equal(i32(o_offs, m + 1), offs)
    assert np.array_equal(i32(o_nz, nz.size), nz)
    assert np.array_equal(i32(o_wcnt, W + 1), wcnt)
    assert np.array_equal(raw[o_heads:o_heads + 4 * (W + 8)].view(np.uint32), heads)
    # the length-class histogram (elements, then segments, of class 2^c..2^(c+1))
    cls = np.minimum(np.log2(lens64[nz]).astype(int), 20)
    hist = raw[24:24 + 4 * 42].view(np.uint32)
    assert np.array_equal(hist[:21], np.bincount(cls, lens64[nz], 21)[:21])
    assert np.array_equal(hist[21:], np.bincount(cls, minlength=21))
    assert cv.lib.cvlhip_check_device_errors() == 0


@pytest.mark.parametrize("n", [(1 << 25) - 1024, 1 << 25, (1 << 25) + 1024, 1 << 28])
def test_long_vectors_keep_the_widest_tiles(cv, n):
    """Scans from 2^25 elements on, and reductions above, have the 8-row
    schedule, whatever a network prefers; below, the network's choice."""
    import torch
    from neslgpu_amd import dispatch as D
    from test_gpu_dispatch import forcing_params
    L, m = cv.lib, n // 256
    lens = np.full(m, 256, np.int32)
    lens[-1] += n - m * 256
    saved = torch.empty(D.mlp_dims(L)[3], dtype=torch.float32, device=cv.device)
    L.cvlhip_sched_get_params(saved)
    had = L.cvlhip_sched_has_model()
    try:
        for arm in (1, 2, 4):
            L.cvlhip_sched_set_params(torch.from_numpy(forcing_params(D.mlp_dims(L), arm)).to(cv.device))
            sd = cv.segd(lens)
            picks = [L.cvlhip_segd_pick(sd, red, size) for red in (0, 1) for size in (4, 8)]
            print("picks", n, arm, picks, flush=True)
            scan, red = arm if n < 1 << 25 else 0, arm if n <= 1 << 25 else 0
            assert picks == [scan, scan, red, red]
            for (k, op, ty), pick in zip(D.KINDS, picks):
                assert D.admitted(D.features(cv, sd, k, ty))[0, arm] == (pick == arm)
    finally:
        L.cvlhip_sched_set_params(saved if had else None)


# Lengths that do not sum to n: the bitmap holds the heads below n, and every
# head count is defined (the memory holds garbage before), in both builds.
def off_sums():
    rng = np.random.default_rng(17)
    few = np.array([0, 60, 0, 40], np.int32)
    many = rng.integers(0, 40, 9000).astype(np.int32)
    return [("small_short", few, 100_000), ("small_long", many[:4000], 30_000), ("few_short", few, 500_000),
            ("none", np.zeros(3, np.int32), 400_000), ("many_short", many, 1_000_003), ("chunks_short", many, 1 << 20),
            ("many_long", many, 100_000), ("chunks_long", many, 1 << 17), ("one_past", few, 8192 * 40 + 1)]


@pytest.mark.parametrize("name,lens,n", off_sums(), ids=[s[0] for s in off_sums()])
def test_lengths_that_do_not_sum_to_n(cv, name, lens, n):
    import torch
    print("segd off sum", name, lens.size, n, int(lens.sum()), flush=True)
    L, m = cv.lib, lens.size
    buf = torch.full((L.siz_fos(n, m) * 2 + 64,), 0x7F7F7F7F, dtype=torch.int32, device=cv.device)
    L.mke_fov(buf, torch.from_numpy(lens).to(cv.device), n, m, cv.scratch(L.mke_fov_scratch(n, m)))
    offs = np.concatenate([[0], np.cumsum(lens.astype(np.int64))])
    at = offs[:-1][lens > 0]
    W, o_lens, o_offs, o_nz, o_wcnt, o_heads = layout(n, m)
    bits = np.zeros((W + 8) * 32, np.uint8)
    bits[at[at < n]] = 1
    raw = host(buf).view(np.uint8)
    i32 = lambda off, k: raw[off:off + 4 * k].view(np.int32)
    assert list(raw[:16].view(np.int64)) == [n, m]
    assert np.array_equal(i32(o_offs, m + 1), offs)
    assert np.array_equal(i32(o_nz, at.size), np.nonzero(lens > 0)[0])
    assert np.array_equal(raw[o_heads:o_heads + 4 * (W + 8)].view(np.uint32),
                          np.packbits(bits, bitorder="little").view(np.uint32))
    assert np.array_equal(i32(o_wcnt, W + 1), np.concatenate([[0], np.cumsum(bits[:W * 32].reshape(W, 32).sum(1, dtype=np.int64))]))
