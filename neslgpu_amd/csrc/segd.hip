// segd.hip -- segment descriptor construction: mke_fov, len_fos, siz_fos,
// cpy_wus (ref nesl/cvl/serial/facilt.c:106-144, elwise.c:291-298).
//
// mke_fov turns the m lengths into the descriptor laid out in segd.hpp:
// offsets (a scan of the lengths), the list of non-empty segments, the head
// bitmap and the per-word head counts.  It runs once per descriptor; every
// segmented kernel then finds boundaries from the bitmap.  Small
// descriptors are built by one workgroup, larger ones by three kernels (sums
// of the lengths per tile; offsets; bitmap and head counts), none of which
// waits for another workgroup.
#include "cvl_hip.hpp"
#include "segd.hpp"
#include "scan.hpp"
#include "mlp.hpp"
#include "../../include/cvl.h"
#include "../../include/cvl_hip_ext.h"

#include <stddef.h>
#include <stdlib.h>

// The trained dispatcher network, generated at build time from
// neslgpu_amd/dispatch_model.npz (sched_model.inc in the build directory).
#if __has_include("sched_model.inc")
#include "sched_model.inc"
#endif

namespace cvlhip {

// ---- the dispatcher's pick
// Parameters of the network that picks a schedule for every descriptor of
// at least kSchedMinN elements (mlp.hpp for the layout).
#ifdef CVLHIP_SCHED_MODEL_PARAMS
__device__ float g_sched_params[kParams] = {CVLHIP_SCHED_MODEL_PARAMS};
static int g_sched_model = 1;
#else
__device__ float g_sched_params[kParams];
static int g_sched_model = 0;
#endif
// CVLHIP_SCHED=0 in the environment starts the library with the
// dispatcher off (every segmented op then runs the flat 8-row schedule).
static int sched_enabled_at_load() {
    const char *e = getenv("CVLHIP_SCHED");
    return !(e && e[0] == '0' && e[1] == 0);
}
static int g_sched_enabled = sched_enabled_at_load();

constexpr int kHist = 2 * kLenClasses;

// A workgroup's histogram is kept in kHistCopies copies, one for every
// kHistCopies-th lane, since the lanes of a wave mostly add to the same few
// classes and LDS atomics on one word take turns (k_segd_offsets 5.1 -> 4.5 us
// at 16384 lengths).
constexpr int kHistCopies = 8;
__device__ __forceinline__ void hist_add(unsigned *h, unsigned len) {
    if (len == 0) return;
    int c = 31 - __clz(len);
    if (c >= kLenClasses) c = kLenClasses - 1;
    const int copy = threadIdx.x % kHistCopies;
    atomicAdd(h + c * kHistCopies + copy, len);
    atomicAdd(h + (kLenClasses + c) * kHistCopies + copy, 1u);
}
__device__ __forceinline__ unsigned hist_get(const unsigned *h, int i) {
    unsigned s = 0;
#pragma unroll
    for (int k = 0; k < kHistCopies; k++) s += h[i * kHistCopies + k];
    return s;
}

// Waves 0..3 of a workgroup of THREADS (at least 256) each pick the schedule
// of one kind of operation (sched_slot order) from the histogram `hist`;
// thread 0 stores the picks in the header.  Every thread of the workgroup
// must call it.
template <int THREADS>
__device__ void sched_pick_block(SegdHeader *hdr, int64_t n, int64_t m, const unsigned *hist, unsigned *s_pick) {
    // The network's parameters and the histogram are staged in LDS with
    // one coalesced pass first, so the forward passes wait for memory once
    // instead of once per layer.
    __shared__ float s_P[kLdsParams];
    __shared__ unsigned s_h[kHist];
    stage_params<THREADS>(g_sched_params, s_P);
    if (threadIdx.x < kHist) s_h[threadIdx.x] = hist[threadIdx.x];
    __syncthreads();
    const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (w < 4) {
        const bool red = (w >> 1) != 0, dbl = (w & 1) != 0;
        const float f = sched_feature(lane < kF ? lane : 0, n, m, s_h, s_h + kLenClasses, dbl, red);
        const int a = mlp_pick_wave(s_P, f, sched_admitted(max_len_class(s_h + kLenClasses), n, m, red));
        if (lane == 0) s_pick[w] = (unsigned)a;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned p = 0;
        for (int k = 0; k < 4; k++) p |= (s_pick[k] & 15u) << (4 * k);
        hdr->sched = (kSchedMagic << 16) | p;
    }
}

// ---- small descriptors: the whole construction in one workgroup
// (m and the bitmap's word count at most kSmallSegd), instead of a dozen
// launches; descriptors of short vectors are built very often by
// interpreted programs.
constexpr int kSmallThreads = 1024;
constexpr int kSmallPer = 4;
constexpr int kSmallSegd = kSmallThreads * kSmallPer;

// Exclusive scan over the workgroup of one value per thread (wrapping
// unsigned +); every thread must call it.  *total receives the sum.
__device__ unsigned block_exclusive_scan(unsigned x, unsigned *s_wave, unsigned *total) {
    const int tid = threadIdx.x, lane = tid % kWave, w = tid / kWave;
    constexpr int W = kSmallThreads / kWave;
    const unsigned inc = wave_inclusive_scan(x, AddU());
    __syncthreads();                                    // s_wave may still be read from a previous call
    if (lane == kWave - 1) s_wave[w] = inc;
    __syncthreads();
    if (tid < kWave) {
        const unsigned t = tid < W ? s_wave[tid] : 0u;
        const unsigned ti = wave_inclusive_scan(t, AddU());
        if (tid < W) s_wave[tid] = ti - t;
        if (tid == W - 1) *total = ti;
    }
    __syncthreads();
    return s_wave[w] + inc - x;
}

__global__ __launch_bounds__(kSmallThreads) void k_segd_small(const int *__restrict__ lens_in, SegdHeader *hdr,
                                                               int *lens, int *offs, int *nz, int *wcnt,
                                                               uint32_t *heads, int64_t n, int64_t m, int64_t words,
                                                               int pick) {
    __shared__ unsigned s_wave[kSmallThreads / kWave];
    __shared__ unsigned s_total;
    __shared__ uint32_t s_heads[kSmallSegd + 8];
    __shared__ unsigned s_hc[kHist * kHistCopies];
    __shared__ unsigned s_hist[kHist];
    __shared__ unsigned s_pick[4];
    const int tid = threadIdx.x;
    if (tid < kHist * kHistCopies) s_hc[tid] = 0u;     // ordered by the barriers of the scans below
    unsigned len[kSmallPer], off[kSmallPer], pos[kSmallPer];
    unsigned lsum = 0, psum = 0;
#pragma unroll
    for (int k = 0; k < kSmallPer; k++) {
        const int64_t g = (int64_t)tid * kSmallPer + k;
        len[k] = g < m ? (unsigned)lens_in[g] : 0u;
        off[k] = lsum;
        pos[k] = psum;
        lsum += len[k];
        psum += (g < m && (int)len[k] > 0) ? 1u : 0u;
    }
    const unsigned lbase = block_exclusive_scan(lsum, s_wave, &s_total);
    const unsigned ltot = s_total;
    const unsigned pbase = block_exclusive_scan(psum, s_wave, &s_total);
    for (int64_t i = tid; i < words + 8; i += kSmallThreads) s_heads[i] = 0u;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSmallPer; k++) {
        const int64_t g = (int64_t)tid * kSmallPer + k;
        if (g < m) {
            const int o = (int)(lbase + off[k]);
            if (lens != lens_in) lens[g] = (int)len[k];
            offs[g] = o;
            if ((int)len[k] > 0) {
                nz[pbase + pos[k]] = (int)g;
                if (o >= 0 && (int64_t)o < n) atomicOr(&s_heads[o >> 5], 1u << (o & 31));
                hist_add(s_hc, len[k]);
            }
        }
    }
    if (tid == 0) {
        offs[m] = (int)ltot;
        hdr->n = n;
        hdr->m = m;
        hdr->stats = kStatsMagic;
    }
    __syncthreads();
    if (tid < kHist) hdr->hist[tid] = s_hist[tid] = hist_get(s_hc, tid);
    __syncthreads();
    if (pick) sched_pick_block<kSmallThreads>(hdr, n, m, s_hist, s_pick);
    else if (tid == 0) hdr->sched = 0u;
    unsigned hc[kSmallPer], csum = 0;
#pragma unroll
    for (int k = 0; k < kSmallPer; k++) {
        const int64_t wd = (int64_t)tid * kSmallPer + k;
        const uint32_t h = wd < words ? s_heads[wd] : 0u;
        hc[k] = csum;
        csum += (unsigned)__popc(h);
        if (wd < words) heads[wd] = h;
    }
    if (tid < 8) heads[words + tid] = 0u;
    const unsigned cbase = block_exclusive_scan(csum, s_wave, &s_total);
#pragma unroll
    for (int k = 0; k < kSmallPer; k++) {
        const int64_t wd = (int64_t)tid * kSmallPer + k;
        if (wd < words) wcnt[wd] = (int)(cbase + hc[k]);
    }
    if (tid == 0) wcnt[words] = (int)s_total;
}

// ---- larger descriptors
// k_segd_sums adds up each tile of kTile lengths; k_segd_offsets, whose tiles
// add up the sums before them, writes offs, the lengths copy, nz, the
// histogram and the first head count (wcnt) of each chunk of kChunk elements;
// k_segd_words builds each chunk's bitmap words in LDS from the starts of
// its segments and writes them with the other head counts.  No workgroup
// waits for another, nothing is cleared first but the histogram, and the
// bitmap is written once, without atomics.  Two look-back kernels behind a
// clear, which waited across the chip and set the bits with atomics in
// memory, took 21.1 us for 300007 lengths of 5 10^6 elements and 19.2 for
// 16384 of about 500000, these three 13.8 and 12.6, most of it latency of
// dependent loads.
constexpr int kTileThreads = 512;
constexpr int kTile = kTileThreads * 4;         // lengths per tile
// Threads of k_segd_words: with 256, chunks of many short segments wait for
// twice as many rounds of loads (16384 one-element segments: 7.3 against
// 5.6 us).
constexpr int kChunkThreads = 512;
constexpr int kChunkWords = 256;                // bitmap words per workgroup of k_segd_words
constexpr int kChunk = kChunkWords * 32;        // elements per chunk
// Above this many tiles the sums are scanned by a kernel of their own
// instead of being added up by every tile.
constexpr int64_t kDirectTiles = 4 * kTileThreads;
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

struct SegPair {                    // (sum of lengths mod 2^32) | (count of non-empty) << 32
    using T = uint64_t;
    __host__ __device__ static T neutral() { return 0; }
    __device__ T operator()(T a, T b) const {
        return (uint64_t)(uint32_t)((uint32_t)a + (uint32_t)b) | (((a >> 32) + (b >> 32)) << 32);
    }
    __device__ static T of(unsigned len) { return (uint64_t)len | ((uint64_t)((int)len > 0) << 32); }
};

// Sum over a workgroup of W waves, in every thread.
template <int W>
__device__ __forceinline__ uint64_t block_sum(uint64_t x, uint64_t *s_wave) {
    const SegPair op;
    const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const uint64_t r = wave_reduce(x, op);
    __syncthreads();                         // s_wave may still be read from a previous use
    if (lane == 0) s_wave[w] = r;
    __syncthreads();
    uint64_t tot = 0;
#pragma unroll
    for (int i = 0; i < W; i++) tot = op(tot, s_wave[i]);
    return tot;
}

// Four lengths of a tile from segment g0 on (0 past the last).
__device__ __forceinline__ void load_lengths(const int *__restrict__ lens, int64_t g0, int64_t m, unsigned (&len)[4]) {
    if (((uintptr_t)lens & 15) == 0 && g0 + 4 <= m) {
        const i32x4 v = *(const i32x4 *)(lens + g0);
        len[0] = (unsigned)v.x;
        len[1] = (unsigned)v.y;
        len[2] = (unsigned)v.z;
        len[3] = (unsigned)v.w;
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) len[k] = g0 + k < m ? (unsigned)lens[g0 + k] : 0u;
    }
}

// parts[t]: the SegPair sum of tile t.  Workgroup 0 also clears the header
// from its schedule word to the end of the histogram.
__global__ __launch_bounds__(kTileThreads) void k_segd_sums(const int *__restrict__ lens, int64_t m,
                                                             uint64_t *__restrict__ parts, SegdHeader *hdr) {
    __shared__ uint64_t s_wave[kTileThreads / kWave];
    const int tid = threadIdx.x;
    if (blockIdx.x == 0) {
        if (tid < kHist) hdr->hist[tid] = 0u;
        if (tid == 0) hdr->sched = hdr->stats = 0u;
    }
    unsigned len[4];
    load_lengths(lens, (int64_t)blockIdx.x * kTile + tid * 4, m, len);
    const SegPair op;
    uint64_t sum = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) sum = op(sum, SegPair::of(len[k]));
    const uint64_t tot = block_sum<kTileThreads / kWave>(sum, s_wave);
    if (tid == 0) parts[blockIdx.x] = tot;
}

// Exclusive scan of the tile sums in place, one workgroup.
__global__ __launch_bounds__(kSmallThreads) void k_segd_scan_sums(uint64_t *parts, int64_t tiles) {
    constexpr int W = kSmallThreads / kWave;
    __shared__ uint64_t s_wave[W];
    const SegPair op;
    const int tid = threadIdx.x, w = tid / kWave, lane = tid % kWave;
    uint64_t carry = 0;
    for (int64_t base = 0; base < tiles; base += kSmallThreads) {
        const uint64_t x = base + tid < tiles ? parts[base + tid] : 0;
        const uint64_t inc = wave_inclusive_scan(x, op);
        __syncthreads();
        if (lane == kWave - 1) s_wave[w] = inc;
        __syncthreads();
        uint64_t before = carry;
#pragma unroll
        for (int i = 0; i < W; i++) {
            if (i < w) before = op(before, s_wave[i]);
            carry = op(carry, s_wave[i]);
        }
        uint64_t ex = shfl_up1(inc);
        if (lane == 0) ex = 0;
        if (base + tid < tiles) parts[base + tid] = op(before, ex);
    }
}

// `scanned`: parts holds exclusive sums, else the tiles' own.  Of wcnt it
// writes the first word of each chunk; *count: the number of non-empty
// segments.
__global__ __launch_bounds__(kTileThreads) void k_segd_offsets(const int *__restrict__ lens_in, SegdHeader *hdr,
                                                                int *lens, int *offs, int *nz,
                                                                int *__restrict__ wcnt,
                                                                const uint64_t *__restrict__ parts, int scanned,
                                                                int *__restrict__ count, int64_t n, int64_t m) {
    constexpr int W = kTileThreads / kWave;
    __shared__ uint64_t s_wave[W];
    __shared__ unsigned s_hist[kHist * kHistCopies];
    const SegPair op;
    const int tid = threadIdx.x, w = tid / kWave, lane = tid % kWave;
    const int64_t tile = blockIdx.x;
    const int64_t g0 = tile * kTile + tid * 4;
    if (tid < kHist * kHistCopies) s_hist[tid] = 0u;   // ordered by the barriers below
    unsigned len[4];
    load_lengths(lens_in, g0, m, len);
    // the tiles before this one
    uint64_t P = 0;
    if (scanned) {
        P = parts[tile];
    } else if (tile > 0) {
        uint64_t s = 0;
        for (int64_t i = tid; i < tile; i += kTileThreads) s = op(s, parts[i]);
        P = block_sum<W>(s, s_wave);
    }
    uint64_t loc[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        loc[k] = sum;
        sum = op(sum, SegPair::of(len[k]));
    }
    const uint64_t inc = wave_inclusive_scan(sum, op);
    __syncthreads();
    if (lane == kWave - 1) s_wave[w] = inc;
    __syncthreads();
    uint64_t through = P;                       // this tile and those before it
#pragma unroll
    for (int i = 0; i < W; i++) {
        through = op(through, s_wave[i]);
        if (i < w) P = op(P, s_wave[i]);
    }
    uint64_t ex = shfl_up1(inc);
    if (lane == 0) ex = 0;
    P = op(P, ex);
    int o4[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint64_t q = op(P, loc[k]);
        o4[k] = (int)(uint32_t)q;
        const bool live = g0 + k < m && (int)len[k] > 0;
        if (live) {
            nz[q >> 32] = (int)(g0 + k);
            hist_add(s_hist, len[k]);
        }
        // the chunks that start after this segment's head and no later than
        // its end: a lane's own few, or, for a long segment, its wave's work
        int j = 0, j1 = 0;
        if (live && o4[k] >= 0) {
            const int64_t end = (int64_t)o4[k] + len[k];
            j = o4[k] / kChunk + 1;
            j1 = (int)((end < n - 1 ? end : n - 1) / kChunk) + 1;
        }
        const int rank = (int)(q >> 32) + 1;
        const bool wide = j1 - j > 4;
        if (!wide)
            for (; j < j1; j++) wcnt[(int64_t)j * kChunkWords] = rank;
        for (uint64_t rest = ballot(wide); rest; rest &= rest - 1) {
            const int l = __builtin_ctzll(rest);
            const int from = shfl(j, l), to = shfl(j1, l), r = shfl(rank, l);
            for (int i = from + lane; i < to; i += kWave) wcnt[(int64_t)i * kChunkWords] = r;
        }
    }
    // (a descriptor in a CVL arena starts on an 8-byte unit: check)
    const bool a16 = (((uintptr_t)offs | (uintptr_t)lens) & 15) == 0;
    if (a16 && g0 + 4 <= m) {    // g0 is a multiple of 4
        *(i32x4 *)(offs + g0) = i32x4{o4[0], o4[1], o4[2], o4[3]};
        if (lens != lens_in) *(i32x4 *)(lens + g0) = i32x4{(int)len[0], (int)len[1], (int)len[2], (int)len[3]};
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (g0 + k < m) {
                offs[g0 + k] = o4[k];
                if (lens != lens_in) lens[g0 + k] = (int)len[k];
            }
        }
    }
    __syncthreads();
    const bool only = gridDim.x == 1;             // one tile: k_segd_sums did not run
    if (tid < kHist) {
        const unsigned h = hist_get(s_hist, tid);
        if (only) hdr->hist[tid] = h;
        else if (h) atomicAdd(&hdr->hist[tid], h);
    }
    if (tile == (int64_t)gridDim.x - 1) {
        // chunks that start past the last segment's end (lengths that sum to
        // less than n): all heads are before them
        const int end = (int)(uint32_t)through;
        if (end >= 0)
            for (int64_t j = end / kChunk + 1 + tid; j * kChunk < n; j += kTileThreads)
                wcnt[j * kChunkWords] = (int)(through >> 32);
        if (tid == 0) {
            offs[m] = end;
            *count = (int)(through >> 32);
            hdr->n = n;
            hdr->m = m;
            hdr->stats = kStatsMagic;
            if (only) hdr->sched = 0u;
        }
    }
    if (tile == 0 && tid == 0 && n > 0) wcnt[0] = 0;
}

// The bitmap words and head counts of one chunk.  Each head of the chunk
// marks a byte of LDS (distinct bytes: no atomics however short the
// segments), which the threads then pack into a word each.  With `pick`, the
// launch has one workgroup more than chunks, and that last workgroup picks
// the schedules from the histogram k_segd_offsets completed.
__global__ __launch_bounds__(kChunkThreads) void k_segd_words(const int *__restrict__ offs, const int *__restrict__ nz,
                                                             const int *__restrict__ count, int *wcnt, uint32_t *heads,
                                                             int64_t words, int64_t chunks, SegdHeader *hdr, int64_t n,
                                                             int64_t m, int pick) {
    constexpr int W = kChunkWords / kWave;
    __shared__ __attribute__((aligned(16))) unsigned char s_mark[kChunk];
    __shared__ unsigned s_wave[W];
    __shared__ unsigned s_pick[4];
    const int tid = threadIdx.x, w = tid / kWave, lane = tid % kWave;
    const int64_t c = blockIdx.x;
    if (c == chunks) {
        sched_pick_block<kChunkThreads>(hdr, n, m, hdr->hist, s_pick);
        return;
    }
    const int64_t w0 = c * kChunkWords, next = w0 + kChunkWords;
    const int all = *count;
    int r0 = n > 0 ? wcnt[w0] : 0, r1 = next < words ? wcnt[next] : all;
    // (negative lengths, or sums that wrap, leave some of these unwritten: clamp)
    r0 = r0 < 0 ? 0 : (r0 > all ? all : r0);
    r1 = r1 > all ? all : r1;
    for (int i = tid; i < kChunk / 16; i += kChunkThreads) ((u32x4 *)s_mark)[i] = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();
    const int64_t lo = c * kChunk;
    const bool ident = all == m;                  // no empty segment: nz is the identity
#pragma unroll 8
    for (int r = r0 + tid; r < r1; r += kChunkThreads) {
        const int64_t o = offs[ident ? r : nz[r]];
        if (o >= lo && o < lo + kChunk && o < n) s_mark[o - lo] = 1;
    }
    __syncthreads();
    uint32_t h = 0;
    if (tid < kChunkWords)
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const u32x4 v = ((const u32x4 *)s_mark)[tid * 2 + q];
        // four 0/1 bytes to four bits: the top nibble of a product that
        // adds each byte once, shifted to its bit
        h |= (((v.x * 0x10204080u) >> 28) | ((v.y * 0x10204080u) >> 28 << 4) | ((v.z * 0x10204080u) >> 28 << 8) |
              ((v.w * 0x10204080u) >> 28 << 12)) << (16 * q);
    }
    const unsigned cnt = (unsigned)__popc(h);
    const unsigned inc = wave_inclusive_scan(cnt, AddU());
    if (w < W && lane == kWave - 1) s_wave[w] = inc;
    __syncthreads();
    if (tid >= kChunkWords) return;
    unsigned base = (unsigned)r0 + inc - cnt;
#pragma unroll
    for (int i = 0; i < W; i++)
        if (i < w) base += s_wave[i];
    if (w0 + tid < words) {
        heads[w0 + tid] = h;
        wcnt[w0 + tid] = (int)base;          // the first word's: the clamped count
    }
    if (c == chunks - 1) {
        if (tid < 8) heads[words + tid] = 0u;
        if (tid == kChunkWords - 1) wcnt[words] = (int)(base + cnt);     // all heads
    }
}

// The count of non-empty segments, then, from byte 256, the tile sums in 16
// bytes per kSmallSegd lengths.
int64_t segd_build_scratch_bytes(int64_t n, int64_t m) {
    SegdLayout L(n, m);
    const int64_t ta = (m + kSmallSegd - 1) / kSmallSegd, tb = (L.words + kSmallSegd - 1) / kSmallSegd;
    static_assert(2 * kTile >= kSmallSegd, "the sums fit");
    return 256 + 16 * (ta + 1) + 16 * (tb + 1) + 256;
}

void segd_build(void *sd, const void *lens_in, int64_t n, int64_t m, void *scratch) {
    SegdLayout L(n, m);
    char *b = (char *)sd;
    SegdHeader *hdr = (SegdHeader *)(b + L.hdr);
    const int pick = g_sched_enabled && g_sched_model && n >= kSchedMinN;
    int *lens = (int *)(b + L.lens);
    int *offs = (int *)(b + L.offs);
    int *nz = (int *)(b + L.nz);
    int *wcnt = (int *)(b + L.wcnt);
    uint32_t *heads = (uint32_t *)(b + L.heads);
    if (!scratch) usage_error("mke_fov called without scratch");

    if (m <= kSmallSegd && L.words <= kSmallSegd) {
        k_segd_small<<<1, kSmallThreads, 0, g_stream>>>((const int *)lens_in, hdr, lens, offs, nz, wcnt, heads, n,
                                                        m, L.words, pick);
        LAUNCHCHECK();
        return;
    }
    const int64_t tiles = (m + kTile - 1) / kTile;
    const int64_t chunks = L.words > 0 ? (L.words + kChunkWords - 1) / kChunkWords : 1;
    int *count = (int *)scratch;
    uint64_t *parts = (uint64_t *)((char *)scratch + 256);
    if (tiles > 1) {
        k_segd_sums<<<(unsigned)tiles, kTileThreads, 0, g_stream>>>((const int *)lens_in, m, parts, hdr);
        LAUNCHCHECK();
    }
    const int scanned = tiles > kDirectTiles;
    if (scanned) {
        k_segd_scan_sums<<<1, kSmallThreads, 0, g_stream>>>(parts, tiles);
        LAUNCHCHECK();
    }
    // (at least one tile, so that the header of a descriptor without segments is written)
    k_segd_offsets<<<(unsigned)(tiles > 0 ? tiles : 1), kTileThreads, 0, g_stream>>>(
        (const int *)lens_in, hdr, lens, offs, nz, wcnt, parts, scanned, count, n, m);
    LAUNCHCHECK();
    k_segd_words<<<(unsigned)(chunks + (pick ? 1 : 0)), kChunkThreads, 0, g_stream>>>(offs, nz, count, wcnt, heads, L.words,
                                                                                  chunks, hdr, n, m, pick);
    LAUNCHCHECK();
}

}  // namespace cvlhip

using namespace cvlhip;

extern "C" {

// ---- the dispatcher's network in the descriptor build
void cvlhip_sched_set_params(const float *params) {
    if (!params) {                    // back to no network: descriptors get no pick
        g_sched_model = 0;
        return;
    }
    HIPCHECK(hipMemcpyToSymbolAsync(HIP_SYMBOL(g_sched_params), params, sizeof(float) * kParams, 0,
                                    hipMemcpyDeviceToDevice, g_stream));
    g_sched_model = 1;
}
void cvlhip_sched_get_params(float *params) {
    HIPCHECK(hipMemcpyFromSymbolAsync(params, HIP_SYMBOL(g_sched_params), sizeof(float) * kParams, 0,
                                      hipMemcpyDeviceToDevice, g_stream));
}
int cvlhip_sched_has_model(void) { return g_sched_model; }
void cvlhip_sched_enable(int on) { g_sched_enabled = on != 0; }
int cvlhip_sched_min_n(void) { return (int)kSchedMinN; }

int siz_fos(int n, int m) { return units_for_bytes(SegdLayout(n, m).bytes); }

// Byte offset of the m segment lengths inside a descriptor, so a host may
// read them in place instead of copying them out with len_fos.
int cvlhip_segd_lengths_offset(void) { return (int)SegdLayout(0, 0).lens; }

void mke_fov(vec_p sd, vec_p l, int n, int m, vec_p scratch) { segd_build(sd, l, n, m, scratch); }
int mke_fov_scratch(int n, int m) { return units_for_bytes(segd_build_scratch_bytes(n, m)); }
// The descriptor is larger than the lengths vector, so it cannot be built
// over it.
unsigned int mke_fov_inplace(void) { return INPLACE_NONE; }

void len_fos(vec_p l, vec_p sd, int n, int m, vec_p scratch) {
    (void)scratch;
    if (m > 0)
        HIPCHECK(hipMemcpyAsync(l, (const char *)sd + SegdLayout(n, m).lens, 4 * (size_t)m, hipMemcpyDeviceToDevice,
                                g_stream));
}
int len_fos_scratch(int n, int m) { (void)n; (void)m; return 0; }
// The lengths sit after the descriptor's header, so writing them over the
// descriptor would overlap the source.
unsigned int len_fos_inplace(void) { return INPLACE_NONE; }

// Copy of a whole descriptor (ref elwise.c:291-298 copies the m lengths,
// which is the whole serial descriptor).
void cpy_wus(vec_p d, vec_p s, int n, int m, vec_p scratch) {
    (void)scratch;
    if (d != s) HIPCHECK(hipMemcpyAsync(d, s, (size_t)SegdLayout(n, m).bytes, hipMemcpyDeviceToDevice, g_stream));
}
int cpy_wus_scratch(int n, int m) { (void)n; (void)m; return 0; }
unsigned int cpy_wus_inplace(void) { return INPLACE_1; }

}  // extern "C"
