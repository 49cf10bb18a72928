// pack.hip -- pack: stable compaction of the elements whose flag is true
// (ref nesl/cvl/serial/library.c:51-164; the VCODE PACK driver is
// nesl/vcode/main.c:577-642).
//
// pk2: each tile loads its flags and values, ranks the true flags with a
// wave-wide scan of per-lane counts, gets the number of true flags before the
// tile -- from a look-back in the same kernel, or, for mid-size vectors, from
// a count of every tile before it -- and writes the kept values to their final
// positions.  The segmented pack keeps the flat order
// (library.c:139-164), so it is the same kernel; pk1_lev, the per-segment
// counts, is a segmented reduction.
#include "cvl_hip.hpp"
#include "lookback.hpp"
#include "scan.hpp"
#include "../../include/cvl.h"

namespace cvlhip {

template <class T> struct VecN;
template <> struct VecN<int> {
    static constexpr int V = 4;
    typedef int vt __attribute__((ext_vector_type(4)));
    typedef int ft __attribute__((ext_vector_type(4)));
};
template <> struct VecN<double> {
    static constexpr int V = 2;
    typedef double vt __attribute__((ext_vector_type(2)));
    typedef int ft __attribute__((ext_vector_type(2)));
};

#ifndef CVLHIP_PACK_ROWS
#define CVLHIP_PACK_ROWS 8
#endif
constexpr int kPackRows = CVLHIP_PACK_ROWS;

template <class T, int R, int B = kBlock>
struct PackShape {
    static constexpr int V = VecN<T>::V;
    static constexpr int ROW = kWave * V;
    static constexpr int WAVES = B / kWave;
    static constexpr int WAVE_ELEMS = R * ROW;
    static constexpr int TILE = WAVES * WAVE_ELEMS;
};

// Flags set per tile of k_pack<T, R, B> (COUNTED), whose workgroups then add
// up the tiles before theirs instead of looking back.
template <class T, int R, int B>
__global__ __launch_bounds__(B) void k_pack_count(const int *__restrict__ f, int64_t n, int *__restrict__ counts,
                                                  int aligned) {
    using S = PackShape<T, R, B>;
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    constexpr int PER = S::TILE / B;
    static_assert(PER % 4 == 0, "runs of four flags per lane");
    __shared__ int s_w[S::WAVES];
    const int64_t t0 = (int64_t)blockIdx.x * S::TILE;
    int c = 0;
    if (aligned && t0 + S::TILE <= n) {
#pragma unroll
        for (int g = 0; g < PER / 4; g++) {
            const i32x4 v = *(const i32x4 *)(f + t0 + ((int64_t)g * B + threadIdx.x) * 4);
            c += (v.x != 0) + (v.y != 0) + (v.z != 0) + (v.w != 0);
        }
    } else {
        for (int64_t k = t0 + threadIdx.x; k < n && k < t0 + S::TILE; k += B) c += f[k] != 0;
    }
    c = wave_reduce(c, AddZ());
    if (threadIdx.x % kWave == 0) s_w[threadIdx.x / kWave] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int i = 0; i < S::WAVES; i++) tot += s_w[i];
        counts[blockIdx.x] = tot;
    }
}

// COUNTED: `status` holds the tiles' counts of k_pack_count (and there is no
// counter), else look-back status words.
template <class T, int R, int B, bool COUNTED>
__global__ __launch_bounds__(B) void k_pack(const T *__restrict__ s, const int *__restrict__ f,
                                                 T *__restrict__ d, int64_t n, int64_t dlim,
                                                 uint64_t *__restrict__ status, unsigned *__restrict__ counter,
                                                 int aligned_i, unsigned *__restrict__ err) {
    using S = PackShape<T, R, B>;
    constexpr int V = S::V;
    const AddZ add;
    const bool aligned = aligned_i != 0;
    __shared__ unsigned s_tile;
    __shared__ int s_wcnt[S::WAVES];
    __shared__ int s_wbase[S::WAVES];
    __shared__ T s_run[S::WAVES][S::ROW];   // one row's kept values, compacted

    if constexpr (!COUNTED) {
        if (threadIdx.x == 0) s_tile = counter ? atomicAdd(counter, 1u) : blockIdx.x;   // no counter: one tile
        __syncthreads();
    }
    const int64_t tile = COUNTED ? (int64_t)blockIdx.x : (int64_t)s_tile;
    const int w = threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    const int64_t wbase = tile * S::TILE + (int64_t)w * S::WAVE_ELEMS + (int64_t)lane * V;

    __shared__ int s_before[S::WAVES];
    if constexpr (COUNTED) {
        int before = 0;
        for (int64_t i = threadIdx.x; i < tile; i += B) before += ((const int *)status)[i];
        before = wave_reduce(before, add);
        if (lane == 0) s_before[w] = before;      // read after the barrier below
    }
    T x[R][V];
    uint32_t fb[R];
    int pos[R];          // rank of the lane's first kept element within the wave
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int64_t base = wbase + (int64_t)r * S::ROW;
        fb[r] = 0;
        if (aligned && base + V <= n) {
            typename VecN<T>::vt v = *(const typename VecN<T>::vt *)(s + base);
            typename VecN<T>::ft g = *(const typename VecN<T>::ft *)(f + base);
#pragma unroll
            for (int k = 0; k < V; k++) { x[r][k] = v[k]; fb[r] |= (g[k] != 0) << k; }
        } else {
#pragma unroll
            for (int k = 0; k < V; k++) {
                bool in = base + k < n;
                x[r][k] = in ? s[base + k] : T(0);
                fb[r] |= (in && f[base + k] != 0) << k;
            }
        }
    }
    int carry = 0;
    int rtot[R];         // kept values per row of the wave
#pragma unroll
    for (int r = 0; r < R; r++) {
        int c = __popc(fb[r]);
        int inc = wave_inclusive_scan(c, add);
        pos[r] = carry + inc - c;
        rtot[r] = bcast_last(inc);
        carry += rtot[r];
    }
    if (lane == 0) s_wcnt[w] = carry;
    __syncthreads();
    if (w == 0) {
        int tot = 0, wb[S::WAVES];
#pragma unroll
        for (int i = 0; i < S::WAVES; i++) { wb[i] = tot; tot += s_wcnt[i]; }
        int P = 0;
        if constexpr (COUNTED) {
#pragma unroll
            for (int i = 0; i < S::WAVES; i++) P += s_before[i];
        } else if (tile == 0) {
            if (lane == 0) TileStatus<int>::publish(status, 0, kPrefix, tot);
        } else {
            if (lane == 0) TileStatus<int>::publish(status, tile, kAggregate, tot);
            P = lookback(status, tile, add, err);
            if (lane == 0) TileStatus<int>::publish(status, tile, kPrefix, P + tot);
        }
        if (lane == 0) {
#pragma unroll
            for (int i = 0; i < S::WAVES; i++) s_wbase[i] = P + wb[i];
        }
    }
    __syncthreads();
    // Row by row, the wave compacts its kept values in LDS and writes them
    // as one contiguous run: every store instruction covers 64 consecutive
    // output elements.
    const int64_t ob = s_wbase[w];
    T *run = s_run[w];
    int rbase = 0;            // kept values of earlier rows of this wave
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int rcount = rtot[r];
        int o = pos[r] - rbase;
#pragma unroll
        for (int k = 0; k < V; k++) {
            if ((fb[r] >> k) & 1u) run[o++] = x[r][k];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (int i = lane; i < rcount; i += kWave) {
            const int64_t at = ob + rbase + i;
            if (at < dlim) d[at] = run[i];
            else *err = 1u;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        rbase += rcount;
    }
}

// Vectors of several look-back tiles and at most this length count their
// flags per tile first and pack in tiles an eighth as large: the flags are
// read twice, from the caches, but no tile waits for another, nothing is
// cleared and mid-size vectors reach every CU.  us per PACK (count to the
// host, then this) against the look-back: ints 40000 20 -> 19, 10^6 23 -> 20, 4
// 10^6 29 -> 24, 16 10^6 62 -> 56; doubles 10^6 22 -> 20, 8 10^6 50 -> 43, 16
// 10^6 80 -> 73.  Above, the second reading leaves the caches, and the last
// tiles add up more than 4096 counts of ints, 8192 of doubles.
constexpr int64_t kPackCountedMax = (int64_t)1 << 24;
constexpr int kPackCountedRows = 4;

constexpr int64_t kPackHeader = 256;

// The look-back tiles' status words, or the counted tiles' counts.
template <class T>
int64_t pack_scratch_bytes(int64_t n) {
    using S = PackShape<T, kPackRows>;
    using C = PackShape<T, kPackCountedRows>;
    const int64_t counted = n < kPackCountedMax ? n : kPackCountedMax;
    const int64_t status = 8 * ((n + S::TILE - 1) / S::TILE), counts = 4 * ((counted + C::TILE - 1) / C::TILE);
    return kPackHeader + (counts > status ? counts : status) + 256;
}

// Threads per pack workgroup (one tile, one look-back).  Measured on MI355X
// with 8-row tiles and 256 / 512 / 1024 threads: 2^28 int 0.735 / 0.599 /
// 0.558 ms, 2^27 double 0.462 / 0.458 / 0.459 (16-row tiles of 256
// threads: 0.694 and 0.578).  Scratch sizes assume 256 threads, the most
// tiles.
template <class T>
constexpr int pack_block() { return 1024; }

// Packs the n elements of s whose flag is set into d, which holds dlim.
template <class T>
void pack(void *d, const void *s, const void *f, int64_t n, int64_t dlim, void *scratch) {
    constexpr int B = pack_block<T>();
    static_assert(B >= kBlock, "scratch sizes count tiles of kBlock threads");
    using S = PackShape<T, kPackRows, B>;
    if (n <= 0) return;
    if (!scratch) usage_error("pack called without scratch");
    int64_t tiles = (n + S::TILE - 1) / S::TILE;
    if (tiles > 1 && n <= kPackCountedMax) {
        constexpr int R = kPackCountedRows;
        using C = PackShape<T, R, kBlock>;
        const unsigned g = (unsigned)((n + C::TILE - 1) / C::TILE);
        int *counts = (int *)((char *)scratch + kPackHeader);
        k_pack_count<T, R, kBlock><<<g, kBlock, 0, g_stream>>>((const int *)f, n, counts, ((uintptr_t)f & 15) == 0);
        LAUNCHCHECK();
        k_pack<T, R, kBlock, true><<<g, kBlock, 0, g_stream>>>(
            (const T *)s, (const int *)f, (T *)d, n, dlim, (uint64_t *)counts, nullptr,
            (((uintptr_t)s | (uintptr_t)f) & 15) == 0, device_error_word());
        LAUNCHCHECK();
        return;
    }
    if (tiles > 1) fill_u32(scratch, 0, (kPackHeader + 8 * tiles) / 4);
    int aligned = (((uintptr_t)s | (uintptr_t)f) & 15) == 0;
    k_pack<T, kPackRows, B, false><<<(unsigned)tiles, B, 0, g_stream>>>(
        (const T *)s, (const int *)f, (T *)d, n, dlim, (uint64_t *)((char *)scratch + kPackHeader),
        tiles > 1 ? (unsigned *)scratch : nullptr, aligned, device_error_word());
    LAUNCHCHECK();
}

}  // namespace cvlhip

using namespace cvlhip;

extern "C" {

int pk1_luv(vec_p f, int len, vec_p scratch) { return reduce_unseg<CountB>(f, len, scratch); }
int pk1_luv_scratch(int len) { return units_for_bytes(kReduceScratchBytes); (void)len; }
unsigned int pk1_luv_inplace(void) { return INPLACE_NONE; }

void pk1_lev(vec_p ds, vec_p f, vec_p sd, int n, int m, vec_p scratch) {
    reduce_seg<CountB>(ds, f, sd, n, m, scratch);
}
int pk1_lev_scratch(int n, int m) {
    (void)m;
    int64_t a = scan_scratch_bytes<AddZ>(n), b = kReduceScratchBytes;
    const int64_t c = seg_reduce_scratch_bytes(n, 4);       // pk1_lev: the segmented count
    if (c > a) a = c;
    return units_for_bytes(a > b ? a : b);
}
unsigned int pk1_lev_inplace(void) { return INPLACE_NONE; }

#define PK2U(NAME, T)                                                                  \
    void NAME(vec_p d, vec_p s, vec_p f, int src_len, int dest_len, vec_p scratch) {   \
        pack<T>(d, s, f, src_len, dest_len, scratch);                                  \
    }                                                                                  \
    int NAME##_scratch(int len) { return units_for_bytes(pack_scratch_bytes<T>(len)); } \
    unsigned int NAME##_inplace(void) { return INPLACE_NONE; }
PK2U(pk2_luz, int)
PK2U(pk2_lub, int)
PK2U(pk2_lud, double)

#define PK2E(NAME, T)                                                                  \
    void NAME(vec_p d, vec_p s, vec_p f, vec_p sd_s, int n_s, int m_s, vec_p sd_d, int n_d, int m_d, \
              vec_p scratch) {                                                         \
        (void)sd_s; (void)m_s; (void)sd_d; (void)m_d;                                  \
        pack<T>(d, s, f, n_s, n_d, scratch);                                           \
    }                                                                                  \
    int NAME##_scratch(int s_vec_len, int s_seg_len, int d_vec_len, int d_seg_len) {   \
        (void)s_seg_len; (void)d_vec_len; (void)d_seg_len;                             \
        return units_for_bytes(pack_scratch_bytes<T>(s_vec_len));                      \
    }                                                                                  \
    unsigned int NAME##_inplace(void) { return INPLACE_NONE; }
PK2E(pk2_lez, int)
PK2E(pk2_leb, int)
PK2E(pk2_led, double)

}  // extern "C"
