// permute.hip -- permute, back-permute and their flagged / default variants
// (ref nesl/cvl/serial/vprims.c:347-467, vecops.c:11-286).
//
//   smp  d[i[k]] = s[k]                       (a permutation)
//   bck  d[k]    = s[i[k]]                    (gather)
//   fpm  d[i[k]] = s[k] where f[k]
//   bfp  d[k]    = f[k] ? s[i[k]] : 0
//   dpe  d = v, then d[i[k]] = s[k]
//   dfp  d = v, then d[i[k]] = s[k] where f[k]
// Segmented forms offset each index by the start of its segment (the source
// segment for scatters, the destination segment for gathers), found in O(1)
// from the descriptor's head bitmap.
//
// Indices are checked against the destination (scatter) or source (gather)
// length: an out-of-range index skips the access and raises the device
// error word instead of faulting.  Scatters whose indices may repeat (fpm,
// dpe, dfp) resolve collisions as the serial loop does: the last writer in
// element order wins.  They first record, per destination, the largest
// source position aimed at it (atomicMax), then each destination takes the
// value of that position or its default.
#include "cvl_hip.hpp"
#include "segd.hpp"
#include "partition.hpp"
#include "../../include/cvl.h"

namespace cvlhip {

static int pgrid(int64_t n) {
    int g = grid_for(n, kBlock * 4);
    return g > 16384 ? 16384 : g;
}

#define GRID_STRIDE(i, n)                                                        \
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (n); \
         i += (int64_t)gridDim.x * blockDim.x)

// Segment base of element k for a scatter / gather; sv.m <= 1 means none.
struct SegBase {
    SegdView key;          // descriptor that owns element k (selects g)
    const int *base_offs;  // offsets of the other side (null: same as key)
    bool seg;
    __device__ __forceinline__ int64_t base(int64_t k) const {
        if (!seg) return 0;
        int g = key.seg_of(k);
        return base_offs ? base_offs[g] : key.offs[g];
    }
};

template <class T>
__global__ void k_gather(T *__restrict__ d, const T *__restrict__ s, const int *__restrict__ idx,
                         const int *__restrict__ f, int64_t n_d, int64_t n_s, SegBase sb, unsigned *err) {
    GRID_STRIDE(k, n_d) {
        if (f && !f[k]) { d[k] = T(0); continue; }
        int64_t p = sb.base(k) + idx[k];
        if (p >= 0 && p < n_s) d[k] = s[p];
        else { d[k] = T(0); *err = 1u; }
    }
}

// The plain gather, d[k] = s[i[k]] for every k: four elements per lane, their
// loads of s in flight together.  Bound by the random loads of s, about 60 G/s
// once s exceeds an XCD's L2.  STREAM (long vectors): the indices and the
// result pass by the caches, which are left to s.  An SpMV product of 2^26
// nonzeros whose x holds 2^22 / 2^20 doubles: 1614 / 1158 us with one element
// per lane, 1609 / 1139 with four, 1600 / 1097 streamed (of 3 10^6 nonzeros
// all the same; non-temporal loads of x: 1931 / 1603).
constexpr int kGatherTile = kBlock * 4;
constexpr int64_t kGatherStreamMin = 1 << 22;
template <class T, bool STREAM>
__global__ __launch_bounds__(kBlock) void k_gather_flat(T *d, const T *__restrict__ s, const int *idx, int64_t n_d,
                                                        int64_t n_s, int aligned, unsigned *err) {
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    constexpr int E = 16 / (int)sizeof(T);
    typedef T vt __attribute__((ext_vector_type(E)));
    const int64_t t0 = (int64_t)blockIdx.x * kGatherTile;
    if (aligned && t0 + kGatherTile <= n_d) {
        const i32x4 *const p = (const i32x4 *)(idx + t0) + threadIdx.x;
        const i32x4 q = STREAM ? __builtin_nontemporal_load(p) : *p;
        T v[4];
        bool bad = false;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = q[k];
            const bool in = i >= 0 && i < n_s;
            bad |= !in;
            const T x = s[in ? i : 0];
            v[k] = in ? x : T(0);
        }
        vt *const o = (vt *)(d + t0) + threadIdx.x * (4 / E);
#pragma unroll
        for (int h = 0; h < 4 / E; h++) {
            vt w;
#pragma unroll
            for (int k = 0; k < E; k++) w[k] = v[h * E + k];
            if (STREAM) __builtin_nontemporal_store(w, o + h);
            else o[h] = w;
        }
        if (bad) *err = 1u;
        return;
    }
    for (int64_t k = t0 + threadIdx.x; k < n_d && k < t0 + kGatherTile; k += kBlock) {
        const int64_t i = idx[k];
        if (i >= 0 && i < n_s) d[k] = s[i];
        else { d[k] = T(0); *err = 1u; }
    }
}

// Last-writer-wins scatter, pass 1: win[p] = max source position aimed at p.
__global__ void k_claim(int *__restrict__ win, const int *__restrict__ idx, const int *__restrict__ f, int64_t n,
                        int64_t n_d, SegBase sb, unsigned *err) {
    GRID_STRIDE(k, n) {
        if (f && !f[k]) continue;
        int64_t p = sb.base(k) + idx[k];
        if (p >= 0 && p < n_d) atomicMax(win + p, (int)k);
        else *err = 1u;
    }
}

// Few sources: only the words of win they aim at are cleared, and pass 2 goes
// by source.
__global__ void k_unclaim(int *__restrict__ win, const int *__restrict__ idx, const int *__restrict__ f, int64_t n,
                          int64_t n_d, SegBase sb) {
    GRID_STRIDE(k, n) {
        if (f && !f[k]) continue;
        const int64_t p = sb.base(k) + idx[k];
        if (p >= 0 && p < n_d) win[p] = -1;
    }
}
template <class T>
__global__ void k_scatter_won(T *__restrict__ d, const T *__restrict__ s, const int *__restrict__ idx,
                              const int *__restrict__ f, const int *__restrict__ win, int64_t n, int64_t n_d,
                              SegBase sb) {
    GRID_STRIDE(k, n) {
        if (f && !f[k]) continue;
        const int64_t p = sb.base(k) + idx[k];
        if (p >= 0 && p < n_d && win[p] == (int)k) d[p] = s[k];
    }
}

// Pass 2, by destination: d[p] = s[win[p]] where some source position won,
// the default v[p] (or d's own value, without v) elsewhere.  Coalesced in win,
// v and d; the random access is a read of s, where writing from the source
// side took a random read of win and a random write of d, after a copy of v.
// Four elements per lane.  us per call, source side -> this: a random order
// with a default, 10^6 ints 70 -> 50, 2^26 5596 -> 4061; half of 2^26 doubles
// in order, in place, 572 -> 521.
template <class T>
__global__ __launch_bounds__(kBlock) void k_place_won(T *d, const T *__restrict__ s, const T *v,
                                                      const int *__restrict__ win, int64_t n_d, int aligned) {
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    const int64_t e = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * 4;
    if (e >= n_d) return;
    int w[4];
    if (aligned && e + 4 <= n_d) {
        const i32x4 q = *(const i32x4 *)(win + e);
        w[0] = q.x; w[1] = q.y; w[2] = q.z; w[3] = q.w;
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) w[k] = e + k < n_d ? win[e + k] : -1;
    }
    T x[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        x[k] = T(0);
        if (w[k] >= 0) x[k] = s[w[k]];
        else if (v && e + k < n_d) x[k] = v[e + k];
    }
#pragma unroll
    for (int k = 0; k < 4; k++)
        if (e + k < n_d && (w[k] >= 0 || v)) d[e + k] = x[k];
}

static SegBase no_seg() {
    SegBase b{SegdView(nullptr, 0, 0), nullptr, false};
    return b;
}

template <class T>
void gather(void *d, const void *s, const void *idx, const void *f, int64_t n_d, int64_t n_s, SegBase sb) {
    if (n_d <= 0) return;
    if (!f && !sb.seg && n_s > 0) {        // (with nothing to gather from, every index is out of range)
        const int aligned = (((uintptr_t)d | (uintptr_t)idx) & 15) == 0;
        const unsigned g = (unsigned)grid_for(n_d, kGatherTile);
        if (n_d >= kGatherStreamMin)
            k_gather_flat<T, true><<<g, kBlock, 0, g_stream>>>((T *)d, (const T *)s, (const int *)idx, n_d, n_s, aligned,
                                                              device_error_word());
        else
            k_gather_flat<T, false><<<g, kBlock, 0, g_stream>>>((T *)d, (const T *)s, (const int *)idx, n_d, n_s, aligned,
                                                               device_error_word());
        LAUNCHCHECK();
        return;
    }
    k_gather<T><<<pgrid(n_d), kBlock, 0, g_stream>>>((T *)d, (const T *)s, (const int *)idx, (const int *)f, n_d,
                                                     n_s, sb, device_error_word());
    LAUNCHCHECK();
}

// Scatter in which several k may aim at one destination; `win` is n_d ints
// of scratch.  v: the default of destinations nobody aims at (null: they
// keep their contents).
// Few sources (below n_d / 32 of 2^21 or more) go by source: 16 10^6 ints
// in place, 0.1% of them aimed at, 14 us against 34 by destination, 6% 56
// against 64, 11% 73 against 75; in random order, with a default to copy, 31
// against 54, 103 against 96, 172 against 138.  Short destinations always go
// by destination, which is a launch less: 1% aimed at in random order with a
// default, 10^6 ints 15.5 by source and 12.8 by destination, 2 10^6 16.1 and
// 17.3, 3 10^6 17.3 and 22.0 (doubles 15.8 and 14.2, 18.2 and 19.7, 21.8 and
// 26.2).
template <class T>
void scatter_lww(void *d, const void *s, const void *idx, const void *f, const void *v, int64_t n, int64_t n_d,
                 SegBase sb, void *win) {
    if (v == d) v = nullptr;
    if (n_d <= 0) return;
    if (n <= 0) {
        if (v) HIPCHECK(hipMemcpyAsync(d, v, (size_t)n_d * sizeof(T), hipMemcpyDeviceToDevice, g_stream));
        return;
    }
    if (!win) { usage_error("permute with collisions needs scratch"); return; }
    const bool few = n_d >= (1 << 21) && n < n_d / 32;
    if (few) {
        if (v) HIPCHECK(hipMemcpyAsync(d, v, (size_t)n_d * sizeof(T), hipMemcpyDeviceToDevice, g_stream));
        k_unclaim<<<pgrid(n), kBlock, 0, g_stream>>>((int *)win, (const int *)idx, (const int *)f, n, n_d, sb);
        LAUNCHCHECK();
    } else {
        fill_u32(win, 0xffffffffu, n_d);
    }
    k_claim<<<pgrid(n), kBlock, 0, g_stream>>>((int *)win, (const int *)idx, (const int *)f, n, n_d, sb,
                                              device_error_word());
    LAUNCHCHECK();
    if (few) {
        k_scatter_won<T><<<pgrid(n), kBlock, 0, g_stream>>>((T *)d, (const T *)s, (const int *)idx, (const int *)f,
                                                            (const int *)win, n, n_d, sb);
        LAUNCHCHECK();
        return;
    }
    k_place_won<T><<<grid_for(n_d, kBlock * 4), kBlock, 0, g_stream>>>((T *)d, (const T *)s, (const T *)v,
                                                                      (const int *)win, n_d, ((uintptr_t)win & 15) == 0);
    LAUNCHCHECK();
}

}  // namespace cvlhip

using namespace cvlhip;

static int lww_units(int n_d) { return units_for_bytes(4 * (int64_t)(n_d > 0 ? n_d : 0) + 256); }

#define SEGB(sd, n, m, other) SegBase{SegdView(sd, n, m), other, (m) > 1}

#define PERMS(TY, T, W)                                                                                   \
    void smp_pu##TY(vec_p d, vec_p s, vec_p i, int len, vec_p scratch) {                                   \
        partition_permute<T>(d, s, (const int *)i, nullptr, len, 0, scratch);                             \
    }                                                                                                     \
    int smp_pu##TY##_scratch(int len) { return units_for_bytes(partition_permute_scratch_bytes(len, W)); } \
    unsigned int smp_pu##TY##_inplace(void) { return INPLACE_NONE; }                                      \
    void smp_pe##TY(vec_p d, vec_p s, vec_p i, vec_p sd, int n, int m, vec_p scratch) {                    \
        partition_permute<T>(d, s, (const int *)i, sd, n, m, scratch);                                    \
    }                                                                                                     \
    int smp_pe##TY##_scratch(int n, int m) { (void)m; return units_for_bytes(partition_permute_scratch_bytes(n, W)); } \
    unsigned int smp_pe##TY##_inplace(void) { return INPLACE_NONE; }                                      \
    void bck_pu##TY(vec_p d, vec_p s, vec_p i, int s_len, int d_len, vec_p scratch) {                     \
        (void)scratch;                                                                                    \
        gather<T>(d, s, i, nullptr, d_len, s_len, no_seg());                                              \
    }                                                                                                     \
    int bck_pu##TY##_scratch(int s_len, int d_len) { (void)s_len; (void)d_len; return 0; }                \
    unsigned int bck_pu##TY##_inplace(void) { return INPLACE_2; }                                         \
    void bck_pe##TY(vec_p d, vec_p s, vec_p i, vec_p sd_s, int n_s, int m_s, vec_p sd_d, int n_d, int m_d,  \
                    vec_p scratch) {                                                                      \
        (void)scratch;                                                                                    \
        if (m_s <= 1) { gather<T>(d, s, i, nullptr, n_d, n_s, no_seg()); return; }                         \
        SegdView src(sd_s, n_s, m_s);                                                                     \
        gather<T>(d, s, i, nullptr, n_d, n_s, SegBase{SegdView(sd_d, n_d, m_d), src.offs, true});         \
    }                                                                                                     \
    int bck_pe##TY##_scratch(int a, int b, int c, int e) { (void)a; (void)b; (void)c; (void)e; return 0; } \
    unsigned int bck_pe##TY##_inplace(void) { return INPLACE_2; }                                         \
    void fpm_pu##TY(vec_p d, vec_p s, vec_p i, vec_p f, int len_src, int len_dest, vec_p scratch) {        \
        scatter_lww<T>(d, s, i, f, nullptr, len_src, len_dest, no_seg(), scratch);                        \
    }                                                                                                     \
    int fpm_pu##TY##_scratch(int s_len, int d_len) { (void)s_len; return lww_units(d_len); }             \
    unsigned int fpm_pu##TY##_inplace(void) { return INPLACE_NONE; }                                      \
    void fpm_pe##TY(vec_p d, vec_p s, vec_p i, vec_p f, vec_p sd_s, int n_s, int m_s, vec_p sd_d, int n_d,  \
                    int m_d, vec_p scratch) {                                                             \
        if (m_s <= 1) { scatter_lww<T>(d, s, i, f, nullptr, n_s, n_d, no_seg(), scratch); return; }                 \
        SegdView dst(sd_d, n_d, m_d);                                                                     \
        scatter_lww<T>(d, s, i, f, nullptr, n_s, n_d, SegBase{SegdView(sd_s, n_s, m_s), dst.offs, true}, scratch);  \
    }                                                                                                     \
    int fpm_pe##TY##_scratch(int a, int b, int c, int e) { (void)a; (void)b; (void)e; return lww_units(c); } \
    unsigned int fpm_pe##TY##_inplace(void) { return INPLACE_NONE; }                                      \
    void bfp_pu##TY(vec_p d, vec_p s, vec_p i, vec_p f, int len_src, int len_dest, vec_p scratch) {        \
        (void)scratch;                                                                                    \
        gather<T>(d, s, i, f, len_dest, len_src, no_seg());                                               \
    }                                                                                                     \
    int bfp_pu##TY##_scratch(int s_len, int d_len) { (void)s_len; (void)d_len; return 0; }                \
    unsigned int bfp_pu##TY##_inplace(void) { return INPLACE_NONE; }                                      \
    void bfp_pe##TY(vec_p d, vec_p s, vec_p i, vec_p f, vec_p sd_s, int n_s, int m_s, vec_p sd_d, int n_d,  \
                    int m_d, vec_p scratch) {                                                             \
        (void)scratch;                                                                                    \
        if (m_s <= 1) { gather<T>(d, s, i, f, n_d, n_s, no_seg()); return; }                               \
        SegdView src(sd_s, n_s, m_s);                                                                     \
        gather<T>(d, s, i, f, n_d, n_s, SegBase{SegdView(sd_d, n_d, m_d), src.offs, true});               \
    }                                                                                                     \
    int bfp_pe##TY##_scratch(int a, int b, int c, int e) { (void)a; (void)b; (void)c; (void)e; return 0; } \
    unsigned int bfp_pe##TY##_inplace(void) { return INPLACE_NONE; }                                      \
    void dpe_pu##TY(vec_p d, vec_p s, vec_p i, vec_p v, int len_src, int len_dest, vec_p scratch) {        \
        scatter_lww<T>(d, s, i, nullptr, v, len_src, len_dest, no_seg(), scratch);                           \
    }                                                                                                     \
    int dpe_pu##TY##_scratch(int s_len, int d_len) { (void)s_len; return lww_units(d_len); }             \
    unsigned int dpe_pu##TY##_inplace(void) { return INPLACE_3; }                                         \
    void dpe_pe##TY(vec_p d, vec_p s, vec_p i, vec_p v, vec_p sd_s, int n_s, int m_s, vec_p sd_d, int n_d,  \
                    int m_d, vec_p scratch) {                                                             \
        if (m_s <= 1) { scatter_lww<T>(d, s, i, nullptr, v, n_s, n_d, no_seg(), scratch); return; }           \
        SegdView dst(sd_d, n_d, m_d);                                                                     \
        scatter_lww<T>(d, s, i, nullptr, v, n_s, n_d, SegBase{SegdView(sd_s, n_s, m_s), dst.offs, true}, scratch); \
    }                                                                                                     \
    int dpe_pe##TY##_scratch(int a, int b, int c, int e) { (void)a; (void)b; (void)e; return lww_units(c); } \
    unsigned int dpe_pe##TY##_inplace(void) { return INPLACE_3; }                                         \
    void dfp_pu##TY(vec_p d, vec_p s, vec_p i, vec_p f, vec_p v, int len_src, int len_dest, vec_p scratch) { \
        scatter_lww<T>(d, s, i, f, v, len_src, len_dest, no_seg(), scratch);                                 \
    }                                                                                                     \
    int dfp_pu##TY##_scratch(int s_len, int d_len) { (void)s_len; return lww_units(d_len); }             \
    unsigned int dfp_pu##TY##_inplace(void) { return INPLACE_4; }                                         \
    void dfp_pe##TY(vec_p d, vec_p s, vec_p i, vec_p f, vec_p v, vec_p sd_s, int n_s, int m_s, vec_p sd_d,  \
                    int n_d, int m_d, vec_p scratch) {                                                    \
        if (m_s <= 1) { scatter_lww<T>(d, s, i, f, v, n_s, n_d, no_seg(), scratch); return; }                 \
        SegdView dst(sd_d, n_d, m_d);                                                                     \
        scatter_lww<T>(d, s, i, f, v, n_s, n_d, SegBase{SegdView(sd_s, n_s, m_s), dst.offs, true}, scratch);  \
    }                                                                                                     \
    int dfp_pe##TY##_scratch(int a, int b, int c, int e) { (void)a; (void)b; (void)e; return lww_units(c); } \
    unsigned int dfp_pe##TY##_inplace(void) { return INPLACE_4; }

extern "C" {
PERMS(z, int, 4)
PERMS(b, int, 4)
PERMS(d, double, 8)
}
