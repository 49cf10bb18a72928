// elwise.hip -- elementwise operations, distribute, index, extract,
// replace, copies and RAND (ref nesl/cvl/serial/elwise.c:128-298,
// vprims.c:203-344, library.c:9-49, facilt.c:292-312).
//
// An elementwise workgroup owns a tile and each lane U vectors of it (16 bytes
// of the widest operand), all loaded before the first is used; one read of
// each input and one write of the output.  Arithmetic follows C on the
// host: int overflow wraps, int / and % truncate, floating point is compiled
// without contraction (-ffp-contract=off) so + - * / and sqrt round exactly
// as the serial CVL; libm transcendentals may differ in the last ulp.
#include "cvl_hip.hpp"
#include "elwise_ops.hpp"
#include "segd.hpp"
#include "../../include/cvl.h"
#include "../../include/cvl_hip_ext.h"

#include <math.h>

namespace cvlhip {


static int ew_grid(int64_t n) {
    int g = grid_for(n, kBlock * 4);
    return g > 16384 ? 16384 : g;
}

// ------------------------------------------------------------------ kernels
// V consecutive elements of one operand, as one load or store.
template <class T, int V> struct EwVec { typedef T type __attribute__((ext_vector_type(V))); };

// Elements per lane and vector: 16 bytes of the widest operand.
template <class... T>
constexpr int ew_lane() {
    size_t w = 4;
    ((w = sizeof(T) > w ? sizeof(T) : w), ...);
    return (int)(16 / w);
}

// Vectors per lane of a long vector; vectors so short that larger tiles would
// leave CUs without a workgroup take one.  Bound by memory.  Nine calls of
// quickhull's test (three of four 24 B/element) of 2^26 doubles, and five of
// 16-byte-per-element int work: 2708 and 866 us with grid-stride loops of one
// element per lane, 2335 and 751 with two vectors per lane (5.6 and 5.7
// TB/s), 2322 and 758 with four, 2418 and 770 with eight; of 4 10^6 elements,
// which the caches hold, 139 and 43, then 126 and 39, 129 and 48, 137 and 44.
constexpr int kEwLong = 2;
constexpr int64_t kEwLongMin = 1 << 21;

// A workgroup's tile is kBlock * U * V elements, V = ew_lane; the last one,
// and vectors that do not start on 16 bytes, go element by element.  d may be
// one of the inputs (all of a lane's loads precede its stores).
template <class F, int U>
__global__ __launch_bounds__(kBlock) void k_ew2(typename F::Out *d, const typename F::In *a, const typename F::In *b,
                                                int64_t n, int aligned) {
    using In = typename F::In;
    using Out = typename F::Out;
    constexpr int V = ew_lane<In, Out>();
    using VI = typename EwVec<In, V>::type;
    using VO = typename EwVec<Out, V>::type;
    const F f;
    const int64_t t0 = (int64_t)blockIdx.x * (kBlock * U * V);
    if (aligned && t0 + kBlock * U * V <= n) {
        VI x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t e = t0 + (u * kBlock + (int)threadIdx.x) * V;
            x[u] = *(const VI *)(a + e);
            y[u] = *(const VI *)(b + e);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            VO o;
#pragma unroll
            for (int k = 0; k < V; k++) o[k] = f(x[u][k], y[u][k]);
            *(VO *)(d + t0 + (u * kBlock + (int)threadIdx.x) * V) = o;
        }
        return;
    }
    for (int64_t i = t0 + threadIdx.x; i < n && i < t0 + kBlock * U * V; i += kBlock) d[i] = f(a[i], b[i]);
}

template <class F, int U>
__global__ __launch_bounds__(kBlock) void k_ew1(typename F::Out *d, const typename F::In *a, int64_t n, int aligned) {
    using In = typename F::In;
    using Out = typename F::Out;
    constexpr int V = ew_lane<In, Out>();
    using VI = typename EwVec<In, V>::type;
    using VO = typename EwVec<Out, V>::type;
    const F f;
    const int64_t t0 = (int64_t)blockIdx.x * (kBlock * U * V);
    if (aligned && t0 + kBlock * U * V <= n) {
        VI x[U];
#pragma unroll
        for (int u = 0; u < U; u++) x[u] = *(const VI *)(a + t0 + (u * kBlock + (int)threadIdx.x) * V);
#pragma unroll
        for (int u = 0; u < U; u++) {
            VO o;
#pragma unroll
            for (int k = 0; k < V; k++) o[k] = f(x[u][k]);
            *(VO *)(d + t0 + (u * kBlock + (int)threadIdx.x) * V) = o;
        }
        return;
    }
    for (int64_t i = t0 + threadIdx.x; i < n && i < t0 + kBlock * U * V; i += kBlock) d[i] = f(a[i]);
}

template <class T, int U>
__global__ __launch_bounds__(kBlock) void k_sel(T *d, const int *f, const T *a, const T *b, int64_t n, int aligned) {
    constexpr int V = ew_lane<T>();
    using VF = typename EwVec<int, V>::type;
    using VT = typename EwVec<T, V>::type;
    const int64_t t0 = (int64_t)blockIdx.x * (kBlock * U * V);
    if (aligned && t0 + kBlock * U * V <= n) {
        VF g[U];
        VT x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t e = t0 + (u * kBlock + (int)threadIdx.x) * V;
            g[u] = *(const VF *)(f + e);
            x[u] = *(const VT *)(a + e);
            y[u] = *(const VT *)(b + e);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            VT o;
#pragma unroll
            for (int k = 0; k < V; k++) o[k] = g[u][k] ? x[u][k] : y[u][k];
            *(VT *)(d + t0 + (u * kBlock + (int)threadIdx.x) * V) = o;
        }
        return;
    }
    for (int64_t i = t0 + threadIdx.x; i < n && i < t0 + kBlock * U * V; i += kBlock) d[i] = f[i] ? a[i] : b[i];
}

// The value at(k) in every element k of d.
template <class T, class F, int U>
__global__ __launch_bounds__(kBlock) void k_make(T *d, F at, int64_t n, int aligned) {
    constexpr int V = ew_lane<T>();
    using VT = typename EwVec<T, V>::type;
    const int64_t t0 = (int64_t)blockIdx.x * (kBlock * U * V);
    if (aligned && t0 + kBlock * U * V <= n) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t e = t0 + (u * kBlock + (int)threadIdx.x) * V;
            VT o;
#pragma unroll
            for (int k = 0; k < V; k++) o[k] = at(e + k);
            *(VT *)(d + e) = o;
        }
        return;
    }
    for (int64_t i = t0 + threadIdx.x; i < n && i < t0 + kBlock * U * V; i += kBlock) d[i] = at(i);
}
template <class T>
struct ConstAt {
    T v;
    __device__ T operator()(int64_t) const { return v; }
};
struct StepAt {
    int init, step;
    __device__ int operator()(int64_t i) const { return (int)((unsigned)init + (unsigned)step * (unsigned)i); }
};

// Are all operands 16-byte aligned?
template <class... P>
static int ew_aligned(P... p) {
    return (((uintptr_t)p | ...) & 15) == 0;
}

template <class F>
static void launch_ew2(void *d, const void *a, const void *b, int64_t n) {
    using In = typename F::In;
    using Out = typename F::Out;
    constexpr int T1 = kBlock * ew_lane<In, Out>();
    const int al = ew_aligned(d, a, b);
    if (n < kEwLongMin)
        k_ew2<F, 1><<<grid_for(n, T1), kBlock, 0, g_stream>>>((Out *)d, (const In *)a, (const In *)b, n, al);
    else
        k_ew2<F, kEwLong><<<grid_for(n, T1 * kEwLong), kBlock, 0, g_stream>>>((Out *)d, (const In *)a, (const In *)b, n, al);
    LAUNCHCHECK();
}
// U: vectors per lane of a long vector; 1 for functions long enough to hide
// the loads.
template <class F, int U>
static void launch_ew1(void *d, const void *a, int64_t n) {
    using In = typename F::In;
    using Out = typename F::Out;
    constexpr int T1 = kBlock * ew_lane<In, Out>();
    const int al = ew_aligned(d, a);
    if (U == 1 || n < kEwLongMin)
        k_ew1<F, 1><<<grid_for(n, T1), kBlock, 0, g_stream>>>((Out *)d, (const In *)a, n, al);
    else
        k_ew1<F, U><<<grid_for(n, T1 * U), kBlock, 0, g_stream>>>((Out *)d, (const In *)a, n, al);
    LAUNCHCHECK();
}
template <class T>
static void launch_sel(void *d, const void *f, const void *a, const void *b, int64_t n) {
    constexpr int T1 = kBlock * ew_lane<T>();
    const int al = ew_aligned(d, f, a, b);
    if (n < kEwLongMin)
        k_sel<T, 1><<<grid_for(n, T1), kBlock, 0, g_stream>>>((T *)d, (const int *)f, (const T *)a, (const T *)b, n, al);
    else
        k_sel<T, kEwLong><<<grid_for(n, T1 * kEwLong), kBlock, 0, g_stream>>>((T *)d, (const int *)f, (const T *)a,
                                                                              (const T *)b, n, al);
    LAUNCHCHECK();
}
template <class T, class F>
static void launch_make(void *d, F at, int64_t n) {
    constexpr int T1 = kBlock * ew_lane<T>();
    if (n < kEwLongMin) k_make<T, F, 1><<<grid_for(n, T1), kBlock, 0, g_stream>>>((T *)d, at, n, ew_aligned(d));
    else k_make<T, F, kEwLong><<<grid_for(n, T1 * kEwLong), kBlock, 0, g_stream>>>((T *)d, at, n, ew_aligned(d));
    LAUNCHCHECK();
}

// one element written by one lane (scalar replace without a host wait)
template <class T>
__global__ void k_put1(T *p, T v) {
    if (threadIdx.x == 0) *p = v;
}

// One element to the host mailbox (ext_vu*).
template <class T>
__global__ void k_ext_post(const T *p, Mailbox *mb, unsigned long long seq) {
    if (threadIdx.x == 0) mailbox_post(mb, seq, scalar_bits(*p));
}

// Segmented distribute and index: a lane makes runs of 16 bytes, four ints or
// two doubles, which share one bitmap word.  Its head count gives the segment
// of the first element, the head bits after it those of the others; rows of a
// wave without a head inside any run look one segment up per run.  Bound by
// the chain of two or three dependent loads, so a lane of a long vector has
// the lookups of eight elements in flight, else of four, and there are no
// branches per element (with them the double distribute below took 16.6 us).
// MAKE_SEGDES, DIST and INDEX of ints, one element per lane and lookup -> this:
// 16 10^6 elements in 100 / 10^6 / 4 10^6 segments 85 -> 55, 106 -> 73, 161 ->
// 123 us; 5 10^6 elements in 300007: the index kernel 13.9 -> 9.5.  One run of
// ints per lane is as fast to 2^20 elements and 5% slower at 16 10^6, four up
// to 3 us slower.  Doubles, one element per lane and lookup / runs of four, whose
// two stores each leave half of a line / this: 5 10^6 in 300007 segments 13.1 /
// 11.6 / 11.0 us, 2^25 in 20000 55.5 / 60.6 / 53.7, 2^26 in 2^22 221 / 172 / 156.
template <int R>
struct SegRun {
    int seg[R];            // (a valid segment past the last element, too)
    unsigned turn;         // bit k > 0: a segment starts at element k
    bool split;            // some run of the wave holds more than one segment
};
template <int R, int U>
__device__ __forceinline__ void seg_runs(const SegdView &sv, int64_t t0, bool ne, SegRun<R> (&r)[U]) {
    static_assert(32 % R == 0, "a run lies in one bitmap word");
    uint32_t h[U];
    int c[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int64_t e = t0 + ((int64_t)u * kBlock + threadIdx.x) * R;
        const int64_t w = (e < sv.n ? e : sv.n - 1) >> 5;
        h[u] = sv.heads[w];
        c[u] = sv.wcnt[w];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int64_t e = t0 + ((int64_t)u * kBlock + threadIdx.x) * R;
        const int64_t f = e < sv.n ? e : sv.n - 1;                 // no bit is set past the last element
        const int sh = (int)(f & 31);
        r[u].turn = e < sv.n ? (h[u] >> sh) & ((1u << R) - 2u) : 0u;
        r[u].split = ballot(r[u].turn != 0u) != 0;
        int g = c[u] + __popc(h[u] & ((2u << sh) - 1u)) - 1;       // among the non-empty segments
#pragma unroll
        for (int k = 0; k < R; k++) {
            g += (r[u].turn >> k) & 1u;
            r[u].seg[k] = g;
        }
    }
    if (ne) return;
#pragma unroll
    for (int u = 0; u < U; u++) {
        if (r[u].split) {
#pragma unroll
            for (int k = 0; k < R; k++) r[u].seg[k] = sv.nz[r[u].seg[k]];
        } else {
            r[u].seg[0] = sv.nz[r[u].seg[0]];
        }
    }
}
// A run is one 16-byte store, wherever d starts: global memory takes those at
// any multiple of 4 bytes.  (One store per element where d is off 16 bytes:
// 2^26 ints in 10^6 segments 106 us instead of 80, 3 10^6 7.3 instead of 4.7.)
template <class T, int R>
__device__ __forceinline__ void store_run(T *d, int64_t e, int64_t n, const T (&x)[R]) {
    static_assert(R == ew_lane<T>(), "16 bytes");
    typedef typename EwVec<T, R>::type VT __attribute__((aligned(sizeof(T))));
    if (e + R <= n) {
        VT o;
#pragma unroll
        for (int k = 0; k < R; k++) o[k] = x[k];
        *(VT *)(d + e) = o;
    } else {
#pragma unroll
        for (int k = 0; k < R; k++)
            if (e + k < n) d[e + k] = x[k];
    }
}

template <class T, int U>
__global__ __launch_bounds__(kBlock) void k_dist_seg(T *__restrict__ d, const T *__restrict__ v, SegdView sv) {
    constexpr int R = ew_lane<T>();
    const int64_t t0 = (int64_t)blockIdx.x * (kBlock * R * U);
    SegRun<R> r[U];
    seg_runs(sv, t0, sv.all_nonempty(), r);
    T x[U][R];
#pragma unroll
    for (int u = 0; u < U; u++) {
        if (r[u].split) {
#pragma unroll
            for (int k = 0; k < R; k++) x[u][k] = v[r[u].seg[k]];
        } else {
            const T one = v[r[u].seg[0]];
#pragma unroll
            for (int k = 0; k < R; k++) x[u][k] = one;
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++) store_run(d, t0 + ((int64_t)u * kBlock + threadIdx.x) * R, sv.n, x[u]);
}

template <int U>
__global__ __launch_bounds__(kBlock) void k_index_seg(int *__restrict__ d, const int *__restrict__ init,
                                                      const int *__restrict__ st, SegdView sv) {
    const int64_t t0 = (int64_t)blockIdx.x * (kBlock * 4 * U);
    SegRun<4> r[U];
    seg_runs(sv, t0, sv.all_nonempty(), r);
    int x[U][4];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int64_t e = t0 + ((int64_t)u * kBlock + threadIdx.x) * 4;
        unsigned at[4], step[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int g = r[u].seg[r[u].split ? k : 0];
            at[k] = step[k] = 0;
            if (k == 0 || r[u].split) {
                at[k] = (unsigned)init[g];
                step[k] = (unsigned)st[g];
            }
        }
        // an element is its segment's first value, or a step past the last one
        x[u][0] = (int)(at[0] + step[0] * (unsigned)(e - sv.offs[r[u].seg[0]]));
#pragma unroll
        for (int k = 1; k < 4; k++) {
            const bool turn = (r[u].turn >> k) & 1u;
            x[u][k] = (int)(turn ? at[k] : (unsigned)x[u][k - 1] + step[r[u].split ? k : 0]);
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++) store_run(d, t0 + ((int64_t)u * kBlock + threadIdx.x) * 4, sv.n, x[u]);
}

template <class T>
static void launch_dist_seg(void *d, const void *v, SegdView sv) {
    constexpr int R = ew_lane<T>(), T1 = kBlock * R;
    if (sv.n < kEwLongMin)
        k_dist_seg<T, 4 / R><<<grid_for(sv.n, T1 * (4 / R)), kBlock, 0, g_stream>>>((T *)d, (const T *)v, sv);
    else
        k_dist_seg<T, 8 / R><<<grid_for(sv.n, T1 * (8 / R)), kBlock, 0, g_stream>>>((T *)d, (const T *)v, sv);
    LAUNCHCHECK();
}

template <class T>
__global__ void k_ext_seg(T *__restrict__ d, const T *__restrict__ s, const int *__restrict__ idx, SegdView sv,
                          unsigned *err) {
    int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; g < sv.m; g += (int64_t)gridDim.x * blockDim.x) {
        int64_t p = (int64_t)sv.offs[g] + idx[g];
        if (p >= 0 && p < sv.n) d[g] = s[p];
        else *err = 1u;
    }
}

template <class T>
__global__ void k_rep_seg(T *__restrict__ d, const int *__restrict__ idx, const T *__restrict__ v, SegdView sv,
                          unsigned *err) {
    int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; g < sv.m; g += (int64_t)gridDim.x * blockDim.x) {
        int64_t p = (int64_t)sv.offs[g] + idx[g];
        if (p >= 0 && p < sv.n) d[p] = v[g];
        else *err = 1u;
    }
}

// ------------------------------------------------------------------ RAND
// lrand48: X' = (a X + c) mod 2^48, value = X' >> 17 (POSIX).  Element k of
// a call uses the (k+1)-th state after the call's starting state; each
// thread jumps to its first state with the affine map raised to its offset.
static uint64_t g_rand_state = 0;   // glibc's unseeded lrand48 starts at 0
constexpr uint64_t kLcgA = 0x5DEECE66DULL, kLcgC = 0xBULL, kMask48 = (1ULL << 48) - 1;

struct Affine { uint64_t a, c; };   // x -> a x + c (mod 2^48)

__host__ __device__ inline Affine compose(Affine f, Affine g) {   // g after f
    return Affine{(g.a * f.a) & kMask48, (g.a * f.c + g.c) & kMask48};
}
__host__ __device__ inline Affine lcg_pow(uint64_t k) {
    Affine r{1, 0}, b{kLcgA, kLcgC};
    while (k) {
        if (k & 1) r = compose(r, b);
        b = compose(b, b);
        k >>= 1;
    }
    return r;
}

constexpr int kRandPer = 16;

__global__ void k_rand(int *__restrict__ d, const int *__restrict__ s, int64_t n, uint64_t x0) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t k0 = t * kRandPer;
    if (k0 >= n) return;
    Affine j = lcg_pow((uint64_t)k0);
    uint64_t x = (j.a * x0 + j.c) & kMask48;
    for (int u = 0; u < kRandPer && k0 + u < n; u++) {
        x = (kLcgA * x + kLcgC) & kMask48;
        int r = (int)(x >> 17);
        int m = s[k0 + u];
        d[k0 + u] = m != 0 ? r % m : 0;
    }
}

// ------------------------------------------------------------------ splitmix
__device__ __forceinline__ uint64_t sm64(uint64_t seed, uint64_t k) {
    uint64_t z = seed + (k + 1) * 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

__global__ void k_splitmix_u32(uint32_t *d, int64_t n, uint64_t seed) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (int64_t)gridDim.x * blockDim.x) d[i] = (uint32_t)(sm64(seed, (uint64_t)i) >> 32);
}

__global__ void k_splitmix_f64(double *d, int64_t n, uint64_t seed, double lo, double hi) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        double u = (double)(sm64(seed, (uint64_t)i) >> 11) * 0x1.0p-53;
        d[i] = lo + (hi - lo) * u;
    }
}

}  // namespace cvlhip

using namespace cvlhip;

// ------------------------------------------------------------------ CVL entry points
#define NOSCR(NAME, FLAG)                                     \
    int NAME##_scratch(int len) { (void)len; return 0; }      \
    unsigned int NAME##_inplace(void) { return FLAG; }

#define EW2(NAME, F, FLAG)                                                                    \
    void NAME(vec_p d, vec_p s1, vec_p s2, int len, vec_p scratch) {                          \
        (void)scratch;                                                                        \
        if (len <= 0) return;                                                                 \
        launch_ew2<F>(d, s1, s2, len);                                                        \
    }                                                                                         \
    NOSCR(NAME, FLAG)

#define EW1(NAME, F, FLAG) EW1U(NAME, F, FLAG, kEwLong)
#define EW1U(NAME, F, FLAG, U)                                                                 \
    void NAME(vec_p d, vec_p s, int len, vec_p scratch) {                                     \
        (void)scratch;                                                                        \
        if (len <= 0) return;                                                                 \
        launch_ew1<F, U>(d, s, len);                                                          \
    }                                                                                         \
    NOSCR(NAME, FLAG)

// In-place flags as in the serial CVL (elwise.c:128-177): an output may
// overwrite any input of the same width.
#define IP12 (INPLACE_1 | INPLACE_2)

extern "C" {

EW2(max_wuz, MaxZf, IP12) EW2(max_wud, MaxDf, IP12)
EW2(min_wuz, MinZf, IP12) EW2(min_wud, MinDf, IP12)
EW2(add_wuz, AddZf, IP12) EW2(add_wud, AddDf, IP12)
EW2(sub_wuz, SubZf, IP12) EW2(sub_wud, SubDf, IP12)
EW2(mul_wuz, MulZf, IP12) EW2(mul_wud, MulDf, IP12)
EW2(div_wuz, DivZf, IP12) EW2(div_wud, DivDf, IP12)
EW2(grt_wuz, GrtZf, IP12) EW2(grt_wud, GrtDf, INPLACE_NONE)
EW2(les_wuz, LesZf, IP12) EW2(les_wud, LesDf, INPLACE_NONE)
EW2(geq_wuz, GeqZf, IP12) EW2(geq_wud, GeqDf, INPLACE_NONE)
EW2(leq_wuz, LeqZf, IP12) EW2(leq_wud, LeqDf, INPLACE_NONE)
EW2(lsh_wuz, LshZf, IP12)
EW2(rsh_wuz, RshZf, IP12)
EW2(mod_wuz, ModZf, IP12)
EW2(eql_wub, EqlBf, IP12) EW2(eql_wuz, EqlZf, IP12) EW2(eql_wud, EqlDf, INPLACE_NONE)
EW2(neq_wub, NeqBf, IP12) EW2(neq_wuz, NeqZf, IP12) EW2(neq_wud, NeqDf, INPLACE_NONE)
EW2(xor_wub, XorBf, IP12)
EW2(ior_wub, IorBf, IP12)
EW2(and_wub, AndBf, IP12)
EW2(ior_wuz, IorZf, IP12)
EW2(and_wuz, AndZf, IP12)
EW2(xor_wuz, XorZf, IP12)

EW1(not_wub, NotBf, INPLACE_1)
EW1(not_wuz, NotZf, INPLACE_1)
EW1(int_wud, IntDf, INPLACE_NONE)
EW1(int_wub, IntBf, INPLACE_1)
EW1(dbl_wuz, DblZf, INPLACE_NONE)
EW1(boo_wuz, BooZf, INPLACE_1)
EW1(flr_wud, FlrDf, INPLACE_NONE)
EW1(cei_wud, CeiDf, INPLACE_NONE)
EW1(trn_wud, TrnDf, INPLACE_NONE)
EW1(rou_wud, RouDf, INPLACE_NONE)
EW1U(exp_wud, ExpDf, INPLACE_1, 1)
EW1U(log_wud, LogDf, INPLACE_1, 1)
EW1(sqt_wud, SqtDf, INPLACE_1)
EW1U(sin_wud, SinDf, INPLACE_1, 1)
EW1U(cos_wud, CosDf, INPLACE_1, 1)
EW1U(tan_wud, TanDf, INPLACE_1, 1)
EW1U(asn_wud, AsnDf, INPLACE_1, 1)
EW1U(acs_wud, AcsDf, INPLACE_1, 1)
EW1U(atn_wud, AtnDf, INPLACE_1, 1)
EW1U(snh_wud, SnhDf, INPLACE_1, 1)
EW1U(csh_wud, CshDf, INPLACE_1, 1)
EW1U(tnh_wud, TnhDf, INPLACE_1, 1)

#define CPY(NAME, W)                                                                           \
    void NAME(vec_p d, vec_p s, int len, vec_p scratch) {                                      \
        (void)scratch;                                                                         \
        if (len <= 0 || d == s) return;                                                        \
        HIPCHECK(hipMemcpyAsync(d, s, (size_t)len * W, hipMemcpyDeviceToDevice, g_stream));    \
    }                                                                                          \
    NOSCR(NAME, INPLACE_1)
CPY(cpy_wuz, 4)
CPY(cpy_wub, 4)
CPY(cpy_wud, 8)

#define SEL(NAME, T)                                                                           \
    void NAME(vec_p d, vec_p s1, vec_p s2, vec_p s3, int len, vec_p scratch) {                 \
        (void)scratch;                                                                         \
        if (len <= 0) return;                                                                  \
        launch_sel<T>(d, s1, s2, s3, len);                                                     \
    }                                                                                          \
    NOSCR(NAME, INPLACE_1 | INPLACE_2 | INPLACE_3)
SEL(sel_wuz, int)
SEL(sel_wub, int)
SEL(sel_wud, double)

// ---- RAND
void rnd_wuz(vec_p d, vec_p s, int len, vec_p scratch) {
    (void)scratch;
    if (len <= 0) return;
    int64_t threads = ((int64_t)len + kRandPer - 1) / kRandPer;
    k_rand<<<grid_for(threads, kBlock), kBlock, 0, g_stream>>>((int *)d, (const int *)s, len, g_rand_state);
    LAUNCHCHECK();
    Affine j = lcg_pow((uint64_t)len);
    g_rand_state = (j.a * g_rand_state + j.c) & kMask48;
}
NOSCR(rnd_wuz, INPLACE_1)

// rnd_foz: the serial CVL on Linux calls srandom(seed) (facilt.c:292-312),
// which does not reseed lrand48; RAND's stream is therefore unaffected.
void rnd_foz(int seed) { (void)seed; }

void cvlhip_rand_set_state(unsigned long long s) { g_rand_state = s & kMask48; }
unsigned long long cvlhip_rand_get_state(void) { return g_rand_state; }

// ---- distribute / index
#define DIS(NAME, T)                                                                           \
    void NAME(vec_p d, T v, int len, vec_p scratch) {                                          \
        (void)scratch;                                                                         \
        if (len <= 0) return;                                                                  \
        launch_make<T>(d, ConstAt<T>{v}, len);                                                 \
    }                                                                                          \
    NOSCR(NAME, INPLACE_NONE)
DIS(dis_vuz, int)
DIS(dis_vud, double)
void dis_vub(vec_p d, cvl_bool v, int len, vec_p scratch) {
    (void)scratch;
    if (len <= 0) return;
    launch_make<int>(d, ConstAt<int>{v}, len);
}
NOSCR(dis_vub, INPLACE_NONE)

#define DISSEG(NAME, T, UNSEG)                                                                 \
    void NAME(vec_p d, vec_p v, vec_p sd, int n, int m, vec_p scratch) {                       \
        (void)scratch;                                                                         \
        if (n <= 0) return;                                                                    \
        SegdView sv(sd, n, m);                                                                 \
        launch_dist_seg<T>(d, v, sv);                                                          \
    }                                                                                          \
    int NAME##_scratch(int n, int m) { (void)n; (void)m; return 0; }                           \
    unsigned int NAME##_inplace(void) { return INPLACE_NONE; }
DISSEG(dis_vez, int, dis_vuz)
DISSEG(dis_veb, int, dis_vub)
DISSEG(dis_ved, double, dis_vud)

void ind_luz(vec_p d, int init, int stride, int count, vec_p scratch) {
    (void)scratch;
    if (count <= 0) return;
    launch_make<int>(d, StepAt{init, stride}, count);
}
NOSCR(ind_luz, INPLACE_NONE)

void ind_lez(vec_p d, vec_p init, vec_p stride, vec_p dest_segd, int vec_len, int seg_count, vec_p scratch) {
    (void)scratch;
    if (vec_len <= 0) return;
    SegdView sv(dest_segd, vec_len, seg_count);
    constexpr int T1 = kBlock * 4;
    if (vec_len < kEwLongMin)
        k_index_seg<1><<<grid_for(vec_len, T1), kBlock, 0, g_stream>>>((int *)d, (const int *)init, (const int *)stride, sv);
    else
        k_index_seg<2><<<grid_for(vec_len, T1 * 2), kBlock, 0, g_stream>>>((int *)d, (const int *)init, (const int *)stride,
                                                                          sv);
    LAUNCHCHECK();
}
int ind_lez_scratch(int n, int m) { (void)n; (void)m; return 0; }
unsigned int ind_lez_inplace(void) { return INPLACE_NONE; }

// ---- extract / replace of one element
// EXT has a one-lane kernel post the element to the host mailbox and waits
// for it (the caller needs the value); REP writes it with a one-lane kernel
// that takes the value as an argument, so it queues behind earlier work
// without a host wait.
#define EXT(NAME, T)                                                                           \
    T NAME(vec_p V, int i, int len, vec_p scratch) {                                           \
        (void)scratch;                                                                         \
        if (i < 0 || i >= len) { usage_error(#NAME ": index %d outside [0,%d)", i, len); return (T)0; } \
        Mailbox *mb = mailbox_device();                                                        \
        const unsigned long long seq = mailbox_next();                                         \
        k_ext_post<T><<<1, 64, 0, g_stream>>>((const T *)V + i, mb, seq);                      \
        LAUNCHCHECK();                                                                         \
        return scalar_from_bits<T>(mailbox_wait(seq));                                         \
    }                                                                                          \
    NOSCR(NAME, INPLACE_NONE)
EXT(ext_vuz, int)
EXT(ext_vub, cvl_bool)
EXT(ext_vud, double)

#define REP(NAME, T, NORM)                                                                     \
    void NAME(vec_p V, int i, T val, int len, vec_p scratch) {                                 \
        (void)scratch;                                                                         \
        if (i < 0 || i >= len) { usage_error(#NAME ": index %d outside [0,%d)", i, len); return; } \
        k_put1<T><<<1, 64, 0, g_stream>>>((T *)V + i, (T)NORM(val));                          \
        LAUNCHCHECK();                                                                         \
    }                                                                                          \
    NOSCR(NAME, INPLACE_NONE)
#define IDENT(x) (x)
#define NOTNOT(x) ((x) != 0)
REP(rep_vuz, int, IDENT)
REP(rep_vub, cvl_bool, NOTNOT)
REP(rep_vud, double, IDENT)

#define EXTSEG(NAME, T)                                                                        \
    void NAME(vec_p d, vec_p s, vec_p i, vec_p sd, int n, int m, vec_p scratch) {              \
        (void)scratch;                                                                         \
        if (m <= 0) return;                                                                    \
        SegdView sv(sd, n, m);                                                                 \
        k_ext_seg<T><<<grid_for(m, kBlock), kBlock, 0, g_stream>>>((T *)d, (const T *)s, (const int *)i, sv, \
                                                                   device_error_word());       \
        LAUNCHCHECK();                                                                         \
    }                                                                                          \
    int NAME##_scratch(int n, int m) { (void)n; (void)m; return 0; }                           \
    unsigned int NAME##_inplace(void) { return INPLACE_2; }
EXTSEG(ext_vez, int)
EXTSEG(ext_veb, int)
EXTSEG(ext_ved, double)

#define REPSEG(NAME, T)                                                                        \
    void NAME(vec_p d, vec_p s, vec_p v, vec_p sd, int n, int m, vec_p scratch) {              \
        (void)scratch;                                                                         \
        if (m <= 0) return;                                                                    \
        SegdView sv(sd, n, m);                                                                 \
        k_rep_seg<T><<<grid_for(m, kBlock), kBlock, 0, g_stream>>>((T *)d, (const int *)s, (const T *)v, sv, \
                                                                   device_error_word());       \
        LAUNCHCHECK();                                                                         \
    }                                                                                          \
    int NAME##_scratch(int n, int m) { (void)n; (void)m; return 0; }                           \
    unsigned int NAME##_inplace(void) { return INPLACE_NONE; }
REPSEG(rep_vez, int)
REPSEG(rep_veb, int)
REPSEG(rep_ved, double)

// ---- synthetic inputs
void cvlhip_fill_splitmix_u32(vec_p d, long long n, unsigned long long seed) {
    if (n <= 0) return;
    k_splitmix_u32<<<ew_grid(n), kBlock, 0, g_stream>>>((uint32_t *)d, n, seed);
    LAUNCHCHECK();
}
void cvlhip_fill_splitmix_f64(vec_p d, long long n, unsigned long long seed, double lo, double hi) {
    if (n <= 0) return;
    k_splitmix_f64<<<ew_grid(n), kBlock, 0, g_stream>>>((double *)d, n, seed, lo, hi);
    LAUNCHCHECK();
}

}  // extern "C"
