// rank.hip -- stable radix rank: rank[i] = position of s[i] in the stable
// sort of s (ref nesl/cvl/serial/rank.c:40-362).
//
// Same digit sequence as the reference: 8-bit digits, least significant
// first, over the transformed 32-bit key (int: key ^ 0x80000000 up,
// key ^ 0x7fffffff down) or the two transformed 32-bit fields of a double
// (low word first), then, for segmented ranks, over the segment number; the
// rank is the final position minus the segment's offset.  A stable LSD sort
// is unique, so any pass that sees a single digit value can be skipped
// without changing the result: one histogram pass reads all keys first and
// the host launches only the passes that reorder something.
//
// Each reordering pass is a histogram kernel (per-tile digit counts), a
// column scan of those counts (each tile's offset in each digit's bucket)
// and a scatter kernel -- or, with CVLHIP_RANK_CHAIN, the scatter kernel
// alone, its tiles chaining the digit offsets with a look-back (tiles
// claimed in order, one chained word per tile and digit): a tile of 4096
// elements ranks its digits stably with a wave-level multisplit (8 ballots
// give each lane the lanes holding the same digit), stages the tile in LDS in
// digit order and writes each digit's run contiguously (keys, then
// indices).  The last pass leaves the sorted order of indices; the rank is
// its inverse, rank[order[p]] = p (minus the segment offset), computed by
// the coalesced permutation engine of partition.hip.
//
// A vector of at most kBlockRankMax4 ints or kBlockRankMax8 doubles is ranked
// by one workgroup in one launch (k_rank_block).  Up to kRankDirectMax keys
// the passes run without the column scan (grouped tile counts) and the last
// one stores the ranks itself (kDirect).
#include "cvl_hip.hpp"
#include "segd.hpp"
#include "lookback.hpp"
#include "partition.hpp"
#include "colscan.hpp"
#include "../../include/cvl.h"

namespace cvlhip {

constexpr int kRadix = 256;
static_assert(kRadix == kTileScanCols, "per-tile digit counts are scanned 256 wide");
#ifndef CVLHIP_RANK_THREADS
#define CVLHIP_RANK_THREADS 512     // 4096-key tiles: 2.03 -> 1.97 ms at 2^26 against 8192
#endif
#ifndef CVLHIP_RANK_ITEMS
#define CVLHIP_RANK_ITEMS 8
#endif
// 1: each pass chains its tiles' digit offsets with a look-back inside the
// scatter kernel (tiles claimed in order) instead of a per-tile histogram
// kernel and a column scan before it.
#ifndef CVLHIP_RANK_CHAIN
#define CVLHIP_RANK_CHAIN 0
#endif
constexpr bool kRankChain = CVLHIP_RANK_CHAIN != 0;
constexpr int kRankThreads = CVLHIP_RANK_THREADS;        // waves of 64
static_assert(kRankThreads >= 256, "one thread per digit");
constexpr int kRankItems = CVLHIP_RANK_ITEMS;            // per lane
constexpr int kRankTile = kRankThreads * kRankItems;     // keys per tile

// Tiles of vectors short enough that 4096-key tiles would leave most CUs
// without one.
constexpr int kRankSmallThreads = 256, kRankSmallItems = 4;

// ---------------------------------------------------------------- key transforms
// KeyT: uint32_t (int ranks) or uint64_t (double ranks, low field in the low
// 32 bits).
__device__ __forceinline__ uint32_t int_key(int s, bool up) {
    return (uint32_t)s ^ (up ? 0x80000000u : 0x7fffffffu);
}
__device__ __forceinline__ uint64_t dbl_key(double s, bool up) {
    uint64_t b = __builtin_bit_cast(uint64_t, s);
    uint32_t lo = (uint32_t)b, hi = (uint32_t)(b >> 32);
    bool neg = (b >> 63) != 0;
    uint32_t flo = neg ? ~lo : lo;
    uint32_t fhi = neg ? ~hi : (hi ^ 0x80000000u);
    if (!up) { flo = ~flo; fhi = ~fhi; }
    return ((uint64_t)fhi << 32) | flo;
}

// ---------------------------------------------------------------- histogram
// hist[p][d]: number of elements whose digit in pass p is d, for the key
// passes (from the keys) -- segment passes are counted by k_seg_hist.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Keys are read 16 bytes per lane when the input is 16-byte aligned
// (`aligned`); the counts do not depend on which lane sees which key.
template <bool DBL>
__global__ __launch_bounds__(kBlock) void k_key_hist(const void *__restrict__ s, int64_t n, bool up, bool aligned,
                                                     unsigned *__restrict__ hist) {
    constexpr int P = DBL ? 8 : 4;
    constexpr int V = DBL ? 2 : 4;               // keys per 16 bytes
    __shared__ unsigned sh[P][kRadix];
    for (int i = threadIdx.x; i < P * kRadix; i += kBlock) (&sh[0][0])[i] = 0;
    __syncthreads();
    auto count = [&](uint64_t key) {
#pragma unroll
        for (int p = 0; p < P; p++) atomicAdd(&sh[p][(key >> (8 * p)) & 255], 1u);
    };
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    const int64_t nv = aligned ? n / V : 0;
    for (int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x; k < nv; k += stride) {
        const u32x4 w = ((const u32x4 *)s)[k];
        if constexpr (DBL) {
            count(dbl_key(__builtin_bit_cast(double, ((uint64_t)w.y << 32) | w.x), up));
            count(dbl_key(__builtin_bit_cast(double, ((uint64_t)w.w << 32) | w.z), up));
        } else {
            count(int_key((int)w.x, up));
            count(int_key((int)w.y, up));
            count(int_key((int)w.z, up));
            count(int_key((int)w.w, up));
        }
    }
    for (int64_t k = nv * V + (int64_t)blockIdx.x * kBlock + threadIdx.x; k < n; k += stride)
        count(DBL ? dbl_key(((const double *)s)[k], up) : int_key(((const int *)s)[k], up));
    __syncthreads();
    for (int i = threadIdx.x; i < P * kRadix; i += kBlock)
        if ((&sh[0][0])[i]) atomicAdd(hist + i, (&sh[0][0])[i]);
}

// Which passes run.  A pass whose digit takes one value over all keys keeps
// the order and is skipped; the digit takes one value iff none of its bits
// is 1 in one key and 0 in another, i.e. shares no bit with (OR of the keys)
// AND (OR of the complemented keys).  The keys' OR words come from the
// first pass's histogram kernel; those of the segment numbers (segmented
// ranks: the numbers of the non-empty segments) from k_seg_or, as `words`
// [0] (OR of the numbers) and [1] (OR of their complements), one per
// 256-byte line, in kOrCopies copies (workgroup b adds to copy
// b % kOrCopies, so fewer atomics queue on each word).
constexpr int kOrStride = 64;
constexpr int kOrWords = 2;
constexpr int kOrCopies = 8;
struct OrU {
    using T = uint32_t;
    __host__ __device__ static constexpr uint32_t neutral() { return 0u; }
    __device__ __forceinline__ uint32_t operator()(uint32_t a, uint32_t b) const { return a | b; }
};

// The workgroup's OR of v[0..NW) into words[first..first+NW): one atomic
// per word and workgroup.
template <int NW>
__device__ __forceinline__ void or_publish(const uint32_t (&v)[NW], unsigned *__restrict__ words, int first) {
    __shared__ uint32_t s_or[kBlock / kWave][NW];
    const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
#pragma unroll
    for (int k = 0; k < NW; k++) {
        const uint32_t r = wave_reduce(v[k], OrU());
        if (lane == 0) s_or[w][k] = r;
    }
    __syncthreads();
    if (threadIdx.x < NW) {
        uint32_t r = 0;
#pragma unroll
        for (int i = 0; i < kBlock / kWave; i++) r |= s_or[i][threadIdx.x];
        if (r) atomicOr(words + ((blockIdx.x % kOrCopies) * kOrWords + first + threadIdx.x) * kOrStride, r);
    }
}

// The runs: the per-tile words of the first pass's keys (k_rank_hist with
// ORW: bits that differ from key 0, two words per tile) folded with the
// segment words of k_seg_or (when segmented); bit p of the posted mask is
// set when pass p reorders something (key passes first, then segment
// passes).  One workgroup.  It also leaves the mask in *word, for the pass
// behind it.
constexpr int kOrPostThreads = 1024;
__global__ __launch_bounds__(kOrPostThreads) void k_or_post(const uint32_t *__restrict__ parts, int64_t nparts,
                                                           const uint32_t *__restrict__ seg_words, int key_passes,
                                                           int seg_passes, Mailbox *mb, unsigned long long seq,
                                                           unsigned *__restrict__ word) {
    __shared__ uint32_t s_or[kOrPostThreads / kWave][2];
    const int tid = threadIdx.x, w = tid / kWave, lane = tid % kWave;
    uint32_t v[2] = {0, 0};
    for (int64_t t = tid; t < nparts; t += kOrPostThreads) {
        const uint2 q = *(const uint2 *)(parts + 2 * t);
        v[0] |= q.x;
        v[1] |= q.y;
    }
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const uint32_t r = wave_reduce(v[k], OrU());
        if (lane == 0) s_or[w][k] = r;
    }
    __syncthreads();
    if (tid == 0) {
        uint32_t o[2] = {0, 0};
        for (int i = 0; i < kOrPostThreads / kWave; i++)
            for (int k = 0; k < 2; k++) o[k] |= s_or[i][k];
        const uint64_t kdiff = ((uint64_t)o[1] << 32) | o[0];
        uint32_t so = 0, sc = 0;
        if (seg_words)
            for (int c = 0; c < kOrCopies; c++) {
                so |= seg_words[(c * kOrWords + 0) * kOrStride];
                sc |= seg_words[(c * kOrWords + 1) * kOrStride];
            }
        const uint32_t sdiff = so & sc;
        unsigned long long mask = 0;
        for (int p = 0; p < key_passes; p++)
            if ((kdiff >> (8 * p)) & 255u) mask |= 1ull << p;
        for (int q = 0; q < seg_passes; q++)
            if ((sdiff >> (8 * q)) & 255u) mask |= 1ull << (key_passes + q);
        *word = (unsigned)mask;
        mailbox_post(mb, seq, mask);
    }
}

__global__ __launch_bounds__(kBlock) void k_seg_or(const int *__restrict__ lens, int64_t m,
                                                   unsigned *__restrict__ words) {
    uint32_t o = 0, c = 0;
    for (int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x; g < m; g += (int64_t)gridDim.x * kBlock)
        if (lens[g] != 0) {
            o |= (uint32_t)g;
            c |= ~(uint32_t)g;
        }
    const uint32_t v[2] = {o, c};
    or_publish<2>(v, words, 0);
}

// Segment-number digits: segment g contributes lens[g] elements.
__global__ void k_seg_hist(const int *__restrict__ lens, int64_t m, int npass, unsigned *__restrict__ hist) {
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < m; g += (int64_t)gridDim.x * blockDim.x) {
        unsigned L = (unsigned)lens[g];
        if (!L) continue;
        for (int p = 0; p < npass; p++) atomicAdd(hist + p * kRadix + ((g >> (8 * p)) & 255), L);
    }
}

// Exclusive scan of each pass's 256 counts (one block per pass).
__global__ void k_hist_scan(unsigned *hist, unsigned *starts) {
    __shared__ unsigned sh[kRadix];
    const int p = blockIdx.x, d = threadIdx.x;
    unsigned v = hist[p * kRadix + d];
    sh[d] = v;
    __syncthreads();
    for (int o = 1; o < kRadix; o <<= 1) {
        unsigned t = d >= o ? sh[d - o] : 0;
        __syncthreads();
        sh[d] += t;
        __syncthreads();
    }
    starts[p * kRadix + d] = sh[d] - v;
}

// ---------------------------------------------------------------- multisplit
// A wave ranks its ITEMS x 64 keys by one 8-bit digit, stably: item j of a
// lane is element j * 64 + lane of the wave's span, of which `count` exist.
// dig: each item's digit; loc: its place among the wave's items of that
// digit; cnt (256 counters of this wave, zero on entry): items per digit.
// FULL: every element of the span exists (all but the last wave of a
// vector), so no lane is masked out.
template <bool FULL, int ITEMS, class KeyT>
__device__ __forceinline__ void multisplit(const KeyT (&key)[ITEMS], int shift, int lane, int64_t count, unsigned *cnt,
                                           unsigned (&dig)[ITEMS], unsigned (&loc)[ITEMS]) {
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        const bool in = FULL || (int64_t)j * kWave + lane < count;
        const KeyT k = key[j];
        const unsigned d = in ? (unsigned)((k >> shift) & 255) : 0u;
        dig[j] = d;
        // lanes of this round holding the same digit: those that agree
        // with this lane in every bit of the digit, the AND over the
        // bits of (lanes with the bit set) XNOR (all lanes if this lane
        // has it set, none if not).  Per bit four instructions: the
        // sign-extended bit, its lane mask (a compare of that value,
        // which the compiler would otherwise rebuild from a shift of the
        // digit), and one 3-input bit operation (v_bitop3, gfx950) per
        // half of the mask: acc & ~(spread ^ mask), truth table 0x84
        // over (spread, acc, mask).
        uint32_t plo = ~0u, phi = ~0u;
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const uint32_t spread = (uint32_t)__builtin_amdgcn_sbfe((int)d, b, 1);   // 0 or ~0: bit b
            const uint64_t bb = __builtin_amdgcn_uicmp(spread, 0u, 33);            // lanes with bit b (ICMP_NE)
            plo = __builtin_amdgcn_bitop3_b32(spread, plo, (uint32_t)bb, 0x84);
            phi = __builtin_amdgcn_bitop3_b32(spread, phi, (uint32_t)(bb >> 32), 0x84);
        }
        if constexpr (!FULL) {             // lanes past the end are no one's peers
            const uint64_t act = ballot(in);
            plo &= (uint32_t)act;
            phi &= (uint32_t)(act >> 32);
        }
        // peers in lanes below this one (v_mbcnt: the set bits of a
        // 64-lane mask below the current lane)
        const unsigned before = __builtin_amdgcn_mbcnt_hi(phi, __builtin_amdgcn_mbcnt_lo(plo, 0u));
        const uint64_t peers = ((uint64_t)phi << 32) | plo;
        const unsigned old = cnt[d];
        loc[j] = old + before;
        // the highest lane of each digit group advances the counter
        const bool leader = in && (peers >> lane) == 1ull;
        if (leader) cnt[d] = old + before + 1;
    }
}

// ---------------------------------------------------------------- short vectors
// The rank of a vector that one workgroup holds: keys and original indices
// (16 bits) stay in registers and LDS through all digit passes, so the call
// is one launch with no host wait instead of 14 launches and one wait.  The
// passes are bound by the multisplit's instructions on one CU (about 45 per
// 64 keys and pass), the rest by barriers and LDS latency.  Against the
// passes below, us per call: 1000 ints 67 -> 7.4, 5000 74 -> 16, 16000 99 ->
// 37; 1000 doubles 126 -> 14, 8192 146 -> 43.
// ITEMS: keys per lane, the fewest that hold the vector (idle lanes still
// take their share of every round).
constexpr int kBlockRankThreads = 1024;

template <class KeyT, int ITEMS>
__global__ __launch_bounds__(kBlockRankThreads) void k_rank_block(const void *__restrict__ s, int n, int up,
                                                                  int *__restrict__ rank) {
    constexpr int W = kBlockRankThreads / kWave, TILE = kBlockRankThreads * ITEMS, SPAN = kWave * ITEMS;
    constexpr int NW = sizeof(KeyT) / 4, P = sizeof(KeyT);
    static_assert(TILE <= 65536, "16-bit indices");
    __shared__ __attribute__((aligned(16))) unsigned s_cnt[W][kRadix];
    __shared__ KeyT s_key[TILE];
    __shared__ unsigned short s_idx[TILE];
    __shared__ uint32_t s_or[NW][W];
    const int tid = threadIdx.x, w = tid / kWave, lane = tid % kWave;
    const int wb = w * SPAN;
    auto key_at = [&](int e) -> KeyT {
        if constexpr (NW == 2) return dbl_key(((const double *)s)[e], up);
        else return int_key(((const int *)s)[e], up);
    };
    auto clear = [&] {
        const u32x4 z = {0u, 0u, 0u, 0u};
        for (int i = tid; i < W * kRadix / 4; i += kBlockRankThreads) ((u32x4 *)&s_cnt[0][0])[i] = z;
    };
    KeyT key[ITEMS];
    unsigned idx[ITEMS];
    const KeyT k0 = key_at(0);
    KeyT x = 0;
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        const int e = wb + j * kWave + lane;
        idx[j] = (unsigned)e;
        key[j] = e < n ? key_at(e) : k0;
    }
    clear();
#pragma unroll
    for (int j = 0; j < ITEMS; j++) x |= key[j] ^ k0;
#pragma unroll
    for (int k = 0; k < NW; k++) {
        const uint32_t r = wave_reduce((uint32_t)((uint64_t)x >> (32 * k)), OrU());
        if (lane == 0) s_or[k][w] = r;
    }
    __syncthreads();
    // the bits in which some key differs from key 0: a pass none of whose
    // bits is among them keeps the order and is skipped
    uint64_t diff = 0;
#pragma unroll
    for (int k = 0; k < NW; k++) {
        uint32_t r = 0;
#pragma unroll
        for (int i = 0; i < W; i++) r |= s_or[k][i];
        diff |= (uint64_t)r << (32 * k);
    }
    if (diff == 0) {                       // all keys equal
        for (int i = tid; i < n; i += kBlockRankThreads) rank[i] = i;
        return;
    }
    for (int p = 0; p < P; p++) {
        const uint64_t rest = diff >> (8 * p);
        if (rest == 0) break;
        if ((rest & 255) == 0) continue;
        const bool last = (rest >> 8) == 0;
        unsigned dig[ITEMS], loc[ITEMS];
        if (wb + SPAN <= n) multisplit<true>(key, 8 * p, lane, SPAN, s_cnt[w], dig, loc);
        else if (wb < n) multisplit<false>(key, 8 * p, lane, n - wb, s_cnt[w], dig, loc);
        __syncthreads();
        if (w == 0) {
            // where each wave's items of each digit start: lane l takes the
            // digits 4l .. 4l+3
            u32x4 t = {0u, 0u, 0u, 0u};
#pragma unroll 4
            for (int i = 0; i < W; i++) t += *(const u32x4 *)&s_cnt[i][4 * lane];
            const unsigned all = t.x + t.y + t.z + t.w;
            const unsigned at = wave_inclusive_scan(all, AddU()) - all;
            u32x4 run = {at, at + t.x, at + t.x + t.y, at + t.x + t.y + t.z};
#pragma unroll 4
            for (int i = 0; i < W; i++) {
                const u32x4 c = *(const u32x4 *)&s_cnt[i][4 * lane];
                *(u32x4 *)&s_cnt[i][4 * lane] = run;
                run += c;
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            if (wb + j * kWave + lane >= n) continue;
            const unsigned at = s_cnt[w][(key[j] >> (8 * p)) & 255] + loc[j];
            if (last) {
                s_idx[idx[j]] = (unsigned short)at;      // the rank, by original index
            } else {
                s_key[at] = key[j];
                s_idx[at] = (unsigned short)idx[j];
            }
        }
        __syncthreads();
        if (last) break;
        clear();
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const int e = wb + j * kWave + lane;
            if (e < n) {
                key[j] = s_key[e];
                idx[j] = s_idx[e];
            }
        }
        __syncthreads();
    }
    for (int i = tid; i < n; i += kBlockRankThreads) rank[i] = (int)s_idx[i];
}

// The longest vector it takes: 112 KiB of the 160 KiB LDS for ints, 96 KiB
// for doubles.  There it still takes less than half the time of the passes
// (figures above); twice as many keys do not fit.
constexpr int kBlockRankMax4 = 16 * kBlockRankThreads, kBlockRankMax8 = 8 * kBlockRankThreads;

template <class KeyT, int ITEMS>
static void launch_rank_block(const void *s, int n, bool up, int *rank) {
    if constexpr (ITEMS > 1)
        if (n <= (ITEMS > 8 ? ITEMS - 4 : ITEMS > 4 ? ITEMS - 2 : ITEMS - 1) * kBlockRankThreads) {
            launch_rank_block<KeyT, (ITEMS > 8 ? ITEMS - 4 : ITEMS > 4 ? ITEMS - 2 : ITEMS - 1)>(s, n, up, rank);
            return;
        }
    k_rank_block<KeyT, ITEMS><<<1, kBlockRankThreads, 0, g_stream>>>(s, n, up, rank);
    LAUNCHCHECK();
}

// ---------------------------------------------------------------- one pass
struct PassArgs {
    const void *src;         // first pass: the original values; else keys_in
    bool vec4;               // keys of 4 bytes or less (source 0, 2, 5, 6), read four at a time
    const int *idx_in;       // null on the first pass (index = position)
    void *keys_out;          // null when the next passes need no keys
    int kout;                // bytes per key in keys_out (8, 4, 2 or 1)
    int oshift;              // keys_out holds key >> oshift
    int *idx_out;            // the element order after this pass
    const unsigned *starts;  // 256 bucket starts of this pass
    const unsigned *tile_ofs;  // tiles x 256: elements of each digit in earlier tiles
    uint32_t *chain;           // or null: tiles x 256 chain words (chain_exclusive)
    unsigned *ticket;          // the chain's tile counter
    int parity;                // the chain's state set
    int64_t n;
    int shift;               // digit = (field >> shift) & 255
    // 0: int values, 1: double values, 2: keys32, 3: keys64, 4: segment
    // number, 5: keys16, 6: keys8.  Stored keys keep only the bits the
    // remaining passes read, shifted down: after the second of four 8-bit
    // passes a 32-bit key needs 16 bits, after the third 8.
    int source;
    int up;
    SegdView seg;                  // segment of an element (segmented ranks)
    unsigned *err;                 // device error word
    // The last pass of an unsegmented rank, fused with the first partition
    // pass of the inverse (partition_invert_begin): instead of the order it
    // writes the pairs (index, position) into child index >> clog of
    // `pairs`, at the tile's slot from tile_ofs2 (tiles x 256, the column
    // scan of the per-tile child counts that k_rank_hist wrote to hist2).
    uint2 *pairs;
    const unsigned *tile_ofs2;
    int clog;
    // Grouped tiles: tile_ofs holds the tiles' own counts, groups the
    // counts of each kRankGroup tiles together (ngroups x 256), and the pass
    // adds up what lies before its tile itself; starts is not read.
    unsigned *groups;
    int64_t ngroups;
    const unsigned *runs;    // pass 0, launched before the host knows: does nothing unless bit 0 is set here
    // The last pass with a direct inverse: rank[index] = position, minus the
    // start of the index's segment when rel is set.
    int *rank;
    int rel;
};

constexpr int kRankGroup = 32;            // tiles per group
constexpr int kRankGroups = 64;           // most groups that a pass adds up

// Which order a pass leaves: kOrder writes the element order (and the keys
// the next passes need), kFuse the inverse's first partition pass, kDirect
// the ranks themselves.
enum RankOut { kOrder, kFuse, kDirect };

// Key of element e for this pass (ix = its original index).
template <class KeyT>
__device__ __forceinline__ KeyT pass_key(const PassArgs &a, int64_t e, int ix) {
    if (a.source == 0) return (KeyT)int_key(((const int *)a.src)[e], a.up);
    if (a.source == 1) return (KeyT)dbl_key(((const double *)a.src)[e], a.up);
    if (a.source == 2) return (KeyT)((const uint32_t *)a.src)[e];
    if (a.source == 3) return (KeyT)((const uint64_t *)a.src)[e];
    if (a.source == 5) return (KeyT)((const uint16_t *)a.src)[e];
    if (a.source == 6) return (KeyT)((const uint8_t *)a.src)[e];
    return (KeyT)(uint32_t)a.seg.seg_of(ix);
}

// Four consecutive stored fields from e (a multiple of 4; the arrays are
// 256-byte aligned, the original values 16-byte aligned when vec4 is set),
// widened to 32 bits: the raw int for source 0, else the stored key.
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef unsigned char u8x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 load_fields4(const PassArgs &a, int64_t e) {
    if (a.source == 5) {
        const u16x4 h = *(const u16x4 *)((const uint16_t *)a.src + e);
        return u32x4{h.x, h.y, h.z, h.w};
    }
    if (a.source == 6) {
        const u8x4 c = *(const u8x4 *)((const uint8_t *)a.src + e);
        return u32x4{c.x, c.y, c.z, c.w};
    }
    return *(const u32x4 *)((const uint32_t *)a.src + e);
}

// keys_out[pos] = key >> oshift, in KOUT bytes.
template <class KeyT, int KOUT>
__device__ __forceinline__ void store_key(const PassArgs &a, int64_t pos, KeyT k) {
    const KeyT v = k >> a.oshift;
    if constexpr (KOUT == 1) ((uint8_t *)a.keys_out)[pos] = (uint8_t)v;
    else if constexpr (KOUT == 2) ((uint16_t *)a.keys_out)[pos] = (uint16_t)v;
    else ((KeyT *)a.keys_out)[pos] = v;
}

// Per-tile digit counts of one pass, as a tiles x 256 matrix (tile t =
// elements [t*kRankTile, (t+1)*kRankTile) of the current order).
// With B2 (the fused last pass) it also counts each tile's elements per
// child of the inverse's first partition pass (index >> a.clog) into hist2.
// With ORW (the first pass, launched before the host knows which passes
// run) it also writes the bits in which the tile's keys differ from key 0
// to or_parts[2 tile], [2 tile + 1] (low, high 32 bits) for k_or_post.
template <class KeyT, bool B2, bool ORW = false, int TH = kRankThreads, int IT = kRankItems>
__global__ __launch_bounds__(TH) void k_rank_hist(PassArgs a, unsigned *__restrict__ hist,
                                                            unsigned *__restrict__ hist2,
                                                            uint32_t *__restrict__ or_parts = nullptr) {
    __shared__ unsigned s_hist[kRadix];
    __shared__ unsigned s_hist2[B2 ? kRadix : 1];
    const int tid = threadIdx.x;
    // ORW: key 0 of the vector, the reference every tile compares with
    // (read first, so that its latency hides behind the tile's loads)
    KeyT k0 = 0;
    if constexpr (ORW) k0 = pass_key<KeyT>(a, 0, 0);
    for (int i = tid; i < kRadix; i += TH) {
        s_hist[i] = 0;
        if constexpr (B2) s_hist2[i] = 0;
    }
    __syncthreads();
    const int64_t tile = blockIdx.x;      // rows are whole 1 KiB stores: launch order
    const int64_t t0 = tile * (TH * IT);
    // Item j is element t0 + ((j / 4) * TH + tid) * 4 + j % 4: runs
    // of four per lane, one 16-byte load each for 4-byte keys.
    static_assert(IT % 4 == 0, "runs of four keys per lane");
    KeyT kv[IT];
    bool in[IT];
#pragma unroll
    for (int g = 0; g < IT / 4; g++) {
        const int64_t e0 = t0 + ((int64_t)g * TH + tid) * 4;
        if (a.vec4 && e0 + 4 <= a.n) {
            const u32x4 w = load_fields4(a, e0);
            const uint32_t x[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                kv[g * 4 + c] = (KeyT)(a.source == 0 ? int_key((int)x[c], a.up) : x[c]);
                in[g * 4 + c] = true;
            }
        } else {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int64_t e = e0 + c;
                const int j = g * 4 + c;
                in[j] = e < a.n;
                kv[j] = 0;
                if (in[j]) kv[j] = pass_key<KeyT>(a, e, a.source == 4 ? (a.idx_in ? a.idx_in[e] : (int)e) : 0);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < IT; j++)
        if (in[j]) atomicAdd(&s_hist[(kv[j] >> a.shift) & 255], 1u);
    if constexpr (ORW) {
        // the bits in which some key of the tile differs from key 0 of the
        // vector (the same reference in every tile): a digit takes one value
        // over all keys iff none of its bits differs anywhere
        constexpr int NW = sizeof(KeyT) / 4;
        __shared__ uint32_t s_or[TH / kWave][NW];
        KeyT x = 0;
#pragma unroll
        for (int j = 0; j < IT; j++)
            if (in[j]) x |= kv[j] ^ k0;
        const int w = tid / kWave, lane = tid % kWave;
#pragma unroll
        for (int k = 0; k < NW; k++) {
            const uint32_t r = wave_reduce((uint32_t)((uint64_t)x >> (32 * k)), OrU());
            if (lane == 0) s_or[w][k] = r;
        }
        __syncthreads();
        if (tid < 2) {
            uint32_t r = 0;
            if (tid < NW)
#pragma unroll
                for (int i = 0; i < TH / kWave; i++) r |= s_or[i][tid];
            or_parts[2 * tile + tid] = r;
        }
    }
    if constexpr (B2) {
        // the elements' original indices: children of the inverse
#pragma unroll
        for (int g = 0; g < IT / 4; g++) {
            const int64_t e0 = t0 + ((int64_t)g * TH + tid) * 4;
            int ix[4];
            if (a.idx_in && e0 + 4 <= a.n) {
                const u32x4 w = *(const u32x4 *)((const uint32_t *)a.idx_in + e0);
                ix[0] = (int)w.x; ix[1] = (int)w.y; ix[2] = (int)w.z; ix[3] = (int)w.w;
            } else {
#pragma unroll
                for (int c = 0; c < 4; c++) ix[c] = e0 + c < a.n ? (a.idx_in ? a.idx_in[e0 + c] : (int)(e0 + c)) : -1;
            }
#pragma unroll
            for (int c = 0; c < 4; c++)
                if (e0 + c < a.n && (unsigned)ix[c] < (unsigned)a.n) atomicAdd(&s_hist2[(unsigned)ix[c] >> a.clog], 1u);
        }
    }
    __syncthreads();
    for (int d = tid; d < kRadix; d += TH) {
        const unsigned c = s_hist[d];
        hist[tile * kRadix + d] = c;
        if (a.groups && c) atomicAdd(a.groups + (tile / kRankGroup) * kRadix + d, c);
        if constexpr (B2) hist2[tile * kRadix + d] = s_hist2[d];
    }
}

// KOUT: bytes per key written to keys_out (a.kout), 0 when no keys are.
// OUT: what it leaves (RankOut); GRP: grouped tile counts; TH x IT: the tile.
template <class KeyT, int KOUT, RankOut OUT, bool GRP, int TH = kRankThreads, int IT = kRankItems>
__global__ __launch_bounds__(TH) void k_rank_pass(PassArgs a) {
    static_assert(OUT == kOrder || KOUT == 0, "the last pass writes no keys");
    static_assert(TH >= kRadix, "one thread per digit");
    constexpr bool FUSE = OUT == kFuse;
    constexpr int W = TH / kWave;
    constexpr int kWaveSpan = kWave * IT;     // consecutive keys per wave
    // s_cnt: per-wave digit counts, then per-wave starts within a digit;
    // s_stage: keys, then (reinterpreted) indices, in digit order.  FUSE:
    // the 8-byte pairs in child order, staged once every position is known,
    // over both (then dead): 32 KiB instead of 8 + 32, so three workgroups
    // of LDS become four.
    constexpr int kCntBytes = W * kRadix * 4;
    constexpr int kStageBytes = (TH * IT) * (int)sizeof(KeyT);
    constexpr int kPairBytes = (TH * IT) * 8;
    constexpr int kRaw = (FUSE && kPairBytes > kCntBytes + kStageBytes) ? kPairBytes : kCntBytes + kStageBytes;
    __shared__ __attribute__((aligned(16))) unsigned char s_raw[kRaw];
    unsigned(*const s_cnt)[kRadix] = (unsigned(*)[kRadix])s_raw;
    KeyT *const s_stage = (KeyT *)(s_raw + kCntBytes);
    __shared__ unsigned s_tot[kRadix];
    __shared__ unsigned s_lstart[kRadix];     // tile-local start of each digit's run
    __shared__ unsigned s_gbase[kRadix];      // global position of the run
    __shared__ unsigned char s_dig[FUSE ? 1 : (TH * IT)];
    __shared__ unsigned s_c2[FUSE ? kRadix : 1];   // FUSE: per-child counts, then starts, of the tile
    __shared__ unsigned s_g2[FUSE ? kRadix : 1];   // FUSE: the tile's slot in each child
    __shared__ unsigned s_all[GRP ? kRadix : 1];   // GRP: each digit's count in the whole vector
    __shared__ unsigned s_placed;                  // FUSE: pairs staged
    __shared__ unsigned s_tile;

    unsigned go = 1u;
    if constexpr (GRP)
        if (a.runs) go = *a.runs;
    const int tid = threadIdx.x;
    const int w = tid / kWave, lane = tid % kWave;
    for (int i = tid; i < W * kRadix; i += TH) (&s_cnt[0][0])[i] = 0;
    if constexpr (FUSE)
        for (int i = tid; i < kRadix; i += TH) s_c2[i] = 0;
    // a chained pass numbers its tiles in the order they start; the
    // order of the tiles' runs within a digit is then their data order
    if (kRankChain && a.chain && tid == 0) s_tile = atomicAdd(a.ticket, 1u);
    __syncthreads();
    const int64_t tile = (kRankChain && a.chain) ? (int64_t)s_tile : xcd_tile(blockIdx.x, gridDim.x);
    const int64_t t0 = tile * (TH * IT);
    const int64_t count = a.n - t0 < (TH * IT) ? a.n - t0 : (TH * IT);
    const int64_t wb = t0 + (int64_t)w * kWaveSpan;

    if constexpr (GRP) {
        // Elements of each digit in the earlier tiles of this tile's group
        // and in the earlier groups, and in all groups: at most kRankGroup +
        // kRankGroups loads per thread, ahead of the tile's own loads.
        const int64_t g = tile / kRankGroup;
        for (int q = tid; q < 2 * kRadix; q += TH) {
            const int d = q % kRadix;
            unsigned before = 0, all = 0;
            if (q < kRadix) {
#pragma unroll 8
                for (int64_t r = g * kRankGroup; r < tile; r++) before += a.tile_ofs[r * kRadix + d];
                s_gbase[d] = before;
            } else {
#pragma unroll 8
                for (int64_t r = 0; r < a.ngroups; r++) {
                    const unsigned c = a.groups[r * kRadix + d];
                    all += c;
                    before += r < g ? c : 0u;
                }
                s_lstart[d] = before;
                s_all[d] = all;
            }
        }
    }

    KeyT key[IT];
    int idx[IT];
    unsigned dig[IT];
    unsigned loc[IT];

    // Item j of a lane is element wb + j*64 + lane: each round of the
    // multisplit below holds 64 consecutive elements, which keeps it stable.
    // A whole span of 4-byte keys is read with 16-byte loads (lane l gets
    // elements 4l..4l+3 of each 256) and put in that order through the
    // wave's own part of s_stage, which is free until the staging phase.
    if constexpr (sizeof(KeyT) == 4) {
        if (a.vec4 && wb + kWaveSpan <= a.n) {
            static_assert(IT % 4 == 0, "runs of four keys per lane");
            uint32_t *sw = (uint32_t *)s_stage + (int64_t)w * kWaveSpan;
            auto transpose = [&](auto load4, uint32_t (&out)[IT]) {
#pragma unroll
                for (int g = 0; g < IT / 4; g++) {
                    const u32x4 v = load4(wb + g * 4 * kWave + 4 * lane);
                    *(u32x4 *)(sw + g * 4 * kWave + 4 * lane) = v;
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                for (int j = 0; j < IT; j++) out[j] = sw[j * kWave + lane];
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            };
            uint32_t raw[IT];
            transpose([&](int64_t e) { return load_fields4(a, e); }, raw);
#pragma unroll
            for (int j = 0; j < IT; j++) key[j] = (KeyT)(a.source == 0 ? int_key((int)raw[j], a.up) : raw[j]);
            if (a.idx_in) {
                transpose([&](int64_t e) { return *(const u32x4 *)((const uint32_t *)a.idx_in + e); }, raw);
#pragma unroll
                for (int j = 0; j < IT; j++) idx[j] = (int)raw[j];
            } else {
#pragma unroll
                for (int j = 0; j < IT; j++) idx[j] = (int)(wb + (int64_t)j * kWave + lane);
            }
            goto loaded;
        }
    }
#pragma unroll
    for (int j = 0; j < IT; j++) {
        const int64_t e = wb + (int64_t)j * kWave + lane;
        KeyT k = 0;
        int ix = 0;
        if (e < a.n) {
            ix = a.idx_in ? a.idx_in[e] : (int)e;
            k = pass_key<KeyT>(a, e, ix);
        }
        key[j] = k;
        idx[j] = ix;
    }
loaded:
    if constexpr (GRP)
        if (!(go & 1u)) return;          // (asked behind the loads: 1 us a call less than in front of them)
    if (wb + kWaveSpan <= a.n) multisplit<true>(key, a.shift, lane, kWaveSpan, s_cnt[w], dig, loc);
    else multisplit<false>(key, a.shift, lane, a.n - wb, s_cnt[w], dig, loc);
    __syncthreads();

    // Per digit: wave starts within the digit, the tile count, and the
    // global start of the tile's run (bucket start + earlier tiles).
    if (tid < kRadix) {
        const int d = tid;
        unsigned run = 0;
#pragma unroll
        for (int i = 0; i < W; i++) {
            const unsigned c = s_cnt[i][d];
            s_cnt[i][d] = run;
            run += c;
        }
        s_tot[d] = run;
        if constexpr (GRP) {
            s_gbase[d] += s_lstart[d];
        } else {
            const unsigned prefix = (kRankChain && a.chain)
                                        ? chain_exclusive(a.chain, tile, kRadix, d, run, a.parity, a.err)
                                        : a.tile_ofs[tile * kRadix + d];
            s_gbase[d] = a.starts[d] + prefix;
        }
    }
    __syncthreads();
    // tile-local digit starts: exclusive scan of the 256 totals (one wave)
    if (tid < kWave) {
        unsigned c[kRadix / kWave], t = 0;
#pragma unroll
        for (int i = 0; i < kRadix / kWave; i++) { c[i] = s_tot[tid * (kRadix / kWave) + i]; t += c[i]; }
        unsigned run = wave_inclusive_scan(t, AddU()) - t;
        unsigned gc[kRadix / kWave] = {}, grun = 0;     // grouped: the digits' starts in the whole vector
        if constexpr (GRP) {
            unsigned gt = 0;
#pragma unroll
            for (int i = 0; i < kRadix / kWave; i++) { gc[i] = s_all[tid * (kRadix / kWave) + i]; gt += gc[i]; }
            grun = wave_inclusive_scan(gt, AddU()) - gt;
        }
#pragma unroll
        for (int i = 0; i < kRadix / kWave; i++) {
            const int d = tid * (kRadix / kWave) + i;
            s_lstart[d] = run;
            s_gbase[d] += grun - run;       // now: global position of local slot 0 of digit d's run
            run += c[i];
            grun += gc[i];
        }
    }
    __syncthreads();

    if constexpr (OUT == kDirect) {
        // Every element's sorted position is its rank: store it where the
        // element came from.
#pragma unroll
        for (int j = 0; j < IT; j++) {
            const int64_t e = wb + (int64_t)j * kWave + lane;
            if (e >= a.n) continue;
            const unsigned d = dig[j];
            const unsigned pos = s_gbase[d] + s_lstart[d] + s_cnt[w][d] + loc[j];
            if ((unsigned)idx[j] < (unsigned)a.n)
                a.rank[idx[j]] = (int)pos - (a.rel ? a.seg.offs[a.seg.seg_of(idx[j])] : 0);
            else
                atomicOr(a.err, 1u);
        }
        return;
    }

    if constexpr (FUSE) {
        // Every element's sorted position is known here: place the pair
        // (index, position) in child index >> clog of the inverse's first
        // partition pass, staged in child order, each child's run written
        // contiguously at the tile's slot in that child.
        uint2 *const s_pair = (uint2 *)s_raw;   // written only after the barrier below: s_cnt is read here
        unsigned ch[IT], rk[IT], pos[IT];
#pragma unroll
        for (int j = 0; j < IT; j++) {
            const int64_t e = wb + (int64_t)j * kWave + lane;
            ch[j] = 0xFFFFFFFFu;
            if (e < a.n) {
                const unsigned d = dig[j];
                pos[j] = s_gbase[d] + s_lstart[d] + s_cnt[w][d] + loc[j];
                if ((unsigned)idx[j] < (unsigned)a.n) {
                    ch[j] = (unsigned)idx[j] >> a.clog;
                    rk[j] = atomicAdd(&s_c2[ch[j]], 1u);
                } else {
                    atomicOr(a.err, 1u);
                }
            }
        }
        __syncthreads();
        if (tid < kWave) {          // child starts within the tile (one wave)
            unsigned c[kRadix / kWave], t = 0;
#pragma unroll
            for (int i = 0; i < kRadix / kWave; i++) { c[i] = s_c2[tid * (kRadix / kWave) + i]; t += c[i]; }
            unsigned run = wave_inclusive_scan(t, AddU()) - t;
#pragma unroll
            for (int i = 0; i < kRadix / kWave; i++) {
                s_c2[tid * (kRadix / kWave) + i] = run;
                run += c[i];
            }
            if (tid == kWave - 1) s_placed = run;
        }
        for (int i = tid; i < kRadix; i += TH) s_g2[i] = a.tile_ofs2[tile * kRadix + i];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IT; j++)
            if (ch[j] != 0xFFFFFFFFu) s_pair[s_c2[ch[j]] + rk[j]] = make_uint2((unsigned)idx[j], pos[j]);
        __syncthreads();
        // s_pair[0 .. placed): the tile's elements with a valid index, by
        // child (index < n < 2^(clog + 8), so every child is below 256)
        const int placed = (int)s_placed;
        const int64_t csize = (int64_t)1 << a.clog;
        for (int i = tid; i < placed; i += TH) {
            const uint2 pr = s_pair[i];
            const unsigned c = pr.x >> a.clog;
            const int64_t at = (int64_t)c * csize + s_g2[c] + (i - s_c2[c]);
            const int64_t cend = ((int64_t)c + 1) * csize < a.n ? ((int64_t)c + 1) * csize : a.n;
            if (at < cend) a.pairs[at] = pr;
            else atomicOr(a.err, 1u);
        }
        return;
    }

    // Stage in digit order, then write each digit's run contiguously:
    // first the keys (when a later pass needs them), then the indices.
    unsigned slot[IT];
#pragma unroll
    for (int j = 0; j < IT; j++) {
        const int64_t e = wb + (int64_t)j * kWave + lane;
        slot[j] = 0;
        if (e < a.n) {
            slot[j] = s_lstart[dig[j]] + s_cnt[w][dig[j]] + loc[j];
            s_dig[slot[j]] = (unsigned char)dig[j];
            if constexpr (KOUT > 0) s_stage[slot[j]] = key[j];
        }
    }
    __syncthreads();
    // Staged element i = tid + k * TH goes to s_gbase[its digit]
    // + i, for the keys and then for the indices.  (s_gbase[d] >= 0: the
    // tile's elements below digit d are among all elements below it.)
    unsigned spos[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const int i = tid + k * TH;
        spos[k] = i < count ? s_gbase[s_dig[i]] + (unsigned)i : 0xFFFFFFFFu;
    }
    if constexpr (KOUT > 0) {
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const int i = tid + k * TH;
            if (i < count) {
                if (spos[k] < a.n) store_key<KeyT, KOUT>(a, spos[k], s_stage[i]);
                else atomicOr(a.err, 1u);
            }
        }
        __syncthreads();
    }
    int *s_idx = (int *)s_stage;
#pragma unroll
    for (int j = 0; j < IT; j++) {
        const int64_t e = wb + (int64_t)j * kWave + lane;
        if (e < a.n) s_idx[slot[j]] = idx[j];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const int i = tid + k * TH;
        if (i < count) {
            if (spos[k] < a.n) a.idx_out[spos[k]] = s_idx[i];
            else atomicOr(a.err, 1u);
        }
    }
}

// rank[k] = k - (segment offset): the result when no pass reorders anything.
__global__ void k_rank_identity(int *rank, int64_t n, SegdView seg, int segmented) {
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
        rank[k] = (int)(segmented ? k - seg.offs[seg.seg_of(k)] : k);
}

// ---------------------------------------------------------------- host driver
// Up to this many keys the tiles' counts are grouped (no column scans), pass
// 0 runs without waiting for the host, and the last pass stores the ranks
// directly: one scattered 4-byte store per key, which stays in the caches
// while the result is small, in place of the inverse's four or five launches.
// us per call against the column scans and the partitioned inverse: 17000
// ints 96 -> 44, 250000 101 -> 51, 10^6 116 -> 72, 3 10^6 152 -> 114, 5 10^6
// 191 -> 171, 8 10^6 246 -> 236; 250000 doubles 182 -> 105, 3 10^6 303 -> 247,
// 8 10^6 620 -> 592.  Above, a pass would add up more than kRankGroups
// groups per tile, and the scattered stores miss the caches.
constexpr int64_t kRankDirectMax = (int64_t)kRankGroups * kRankGroup * kRankTile;
// Up to this many keys tiles are small: 250000 ints 51 against 57 us, 500000
// 57 against 62, but 10^6 75 against 72.
constexpr int64_t kRankSmallMax = (int64_t)1 << 19;
constexpr int kRankSmallTile = kRankSmallThreads * kRankSmallItems;
static_assert(kRankSmallMax <= (int64_t)kRankGroups * kRankGroup * kRankSmallTile, "small tiles are grouped");
constexpr int kRankPasses = 12;           // most passes: 8 of a double, 4 of a segment number

// Byte offsets of the areas in a rank's scratch.  Every area's whole size is
// counted, rows of 256 words per tile, group and pass rounded up as the
// kernels write them; areas that share their bytes are never in use together.
struct RankScratch {
    int64_t keysA, keysB, idxA, idxB, hist, starts, counters, status, scan_status, status2, orparts, invert, bytes;
    int64_t groups;                                    // grouped tiles of kRankTile: the group counts of each pass
    int64_t small_counts, small_groups, small_orparts;   // small tiles: tile counts, group counts, OR words
    RankScratch(int64_t n, bool dbl) {
        auto up = [](int64_t b) { return (b + 255) & ~(int64_t)255; };
        auto most = [](int64_t a, int64_t b) { return a > b ? a : b; };
        auto parts = [](int64_t k, int64_t size) { return (k + size - 1) / size; };
        constexpr int64_t row = 4 * kRadix;
        const int64_t kw = dbl ? 8 : 4;
        const int64_t tiles = most(parts(n, kRankTile), 1);
        keysA = 0;
        keysB = up(keysA + kw * n);
        idxA = up(keysB + kw * n);
        idxB = up(idxA + 4 * n);
        hist = up(idxB + 4 * n);
        starts = up(hist + kRankPasses * row);
        counters = up(starts + kRankPasses * row);
        status = up(counters + 4 * 16);
        // one column-scan status region per pass, one for the fused last
        // pass's child counts and one for the speculative first pass, cleared
        // together; grouped tiles have no column scan and keep their group
        // counts there
        groups = scan_status = up(status + row * tiles);
        const int64_t ngroups = tiles < kRankGroups * kRankGroup ? parts(tiles, kRankGroup) : kRankGroups;
        const int64_t scan_bytes = most((kRankPasses + 2) * 8 * tile_scan_status_words(tiles), kRankPasses * row * ngroups);
        // the fused last pass's per-tile child counts; the first pass's
        // per-tile OR words
        status2 = up(scan_status + scan_bytes);
        orparts = up(status2 + row * tiles);
        // the inverse's scratch.  Small tiles' counts lie in it: their passes
        // are done before an inverse (or none) runs.
        invert = up(orparts + 8 * tiles);
        bytes = up(invert + partition_permute_scratch_bytes(n, 4));
        const int64_t small_tiles = most(parts(n, kRankSmallTile), 1);
        small_counts = invert;
        small_groups = small_counts + row * small_tiles;
        small_orparts = small_groups + kRankPasses * row * parts(small_tiles, kRankGroup);
        if (n <= kRankSmallMax) bytes = most(bytes, up(small_orparts + 8 * small_tiles));
    }
};

static unsigned *g_hist_host = nullptr;

template <int TH, int IT, bool B2, bool ORW>
static void launch_hist(const PassArgs &a, int64_t tiles, bool dbl, unsigned *hist, unsigned *hist2, uint32_t *or_parts) {
    if (dbl) k_rank_hist<uint64_t, B2, ORW, TH, IT><<<(unsigned)tiles, TH, 0, g_stream>>>(a, hist, hist2, or_parts);
    else k_rank_hist<uint32_t, B2, ORW, TH, IT><<<(unsigned)tiles, TH, 0, g_stream>>>(a, hist, hist2, or_parts);
    LAUNCHCHECK();
}

// An order-writing pass: the kernel of the key width it writes.
template <bool GRP, int TH, int IT>
static void launch_order(const PassArgs &a, dim3 grid, bool dbl) {
    if (dbl) {
        if (a.keys_out) k_rank_pass<uint64_t, 8, kOrder, GRP, TH, IT><<<grid, TH, 0, g_stream>>>(a);
        else k_rank_pass<uint64_t, 0, kOrder, GRP, TH, IT><<<grid, TH, 0, g_stream>>>(a);
    } else if (!a.keys_out) {
        k_rank_pass<uint32_t, 0, kOrder, GRP, TH, IT><<<grid, TH, 0, g_stream>>>(a);
    } else if (a.kout == 1) {
        k_rank_pass<uint32_t, 1, kOrder, GRP, TH, IT><<<grid, TH, 0, g_stream>>>(a);
    } else if (a.kout == 2) {
        k_rank_pass<uint32_t, 2, kOrder, GRP, TH, IT><<<grid, TH, 0, g_stream>>>(a);
    } else {
        k_rank_pass<uint32_t, 4, kOrder, GRP, TH, IT><<<grid, TH, 0, g_stream>>>(a);
    }
    LAUNCHCHECK();
}

// One grouped pass.
template <int TH, int IT>
static void launch_grouped(const PassArgs &a, int64_t tiles, bool dbl, bool last) {
    const dim3 grid((unsigned)tiles);
    if (!last) return launch_order<true, TH, IT>(a, grid, dbl);
    if (dbl) k_rank_pass<uint64_t, 0, kDirect, true, TH, IT><<<grid, TH, 0, g_stream>>>(a);
    else k_rank_pass<uint32_t, 0, kDirect, true, TH, IT><<<grid, TH, 0, g_stream>>>(a);
    LAUNCHCHECK();
}

void rank_run(int *rank, const void *s, int64_t n, bool dbl, bool up, const void *sd, int64_t m, void *scratch) {
    if (n <= 0) return;
    if (!scratch) usage_error("rank called without scratch");
    if (n > 0x7fffffffLL) usage_error("rank: too many keys");
    RankScratch L(n, dbl);
    char *b = (char *)scratch;
    unsigned *hist = (unsigned *)(b + L.hist);
    unsigned *starts = (unsigned *)(b + L.starts);
    const bool segmented = sd != nullptr && m > 1;
    if (!segmented && n <= (dbl ? kBlockRankMax8 : kBlockRankMax4)) {
        if (dbl) launch_rank_block<uint64_t, kBlockRankMax8 / kBlockRankThreads>(s, (int)n, up, rank);
        else launch_rank_block<uint32_t, kBlockRankMax4 / kBlockRankThreads>(s, (int)n, up, rank);
        return;
    }
    SegdView seg(sd, n, segmented ? m : 0);
    const int key_passes = dbl ? 8 : 4;
    int seg_passes = 0;
    if (segmented) {
        int64_t mm = m - 1;
        while (mm > 0) { seg_passes++; mm >>= 8; }
    }
    const int total = key_passes + seg_passes;

    const bool chain = kRankChain && n < (int64_t)kChainMask;
    const bool aligned = ((uintptr_t)s & 15) == 0;
    const bool grouped = !chain && n <= kRankDirectMax;
    const bool small = grouped && n <= kRankSmallMax;
    const int tile = small ? kRankSmallTile : kRankTile;
    const int64_t tiles = (n + tile - 1) / tile;
    const int64_t ngroups = (tiles + kRankGroup - 1) / kRankGroup;
    const int64_t sw = tile_scan_status_words((n + kRankTile - 1) / kRankTile);
    unsigned *tile_ofs = (unsigned *)(b + (small ? L.small_counts : L.status));
    uint64_t *scan_status = (uint64_t *)(b + L.scan_status);
    uint32_t *or_parts = (uint32_t *)(b + (small ? L.small_orparts : L.orparts));
    unsigned *groups = (unsigned *)(b + (small ? L.small_groups : L.groups));      // ngroups x 256 per pass
    int gs = grid_for(m, kBlock);
    if (gs > 4096) gs = 4096;
    bool runs[12] = {};
    unsigned *tile_ofs2 = (unsigned *)(b + L.status2);
    InvertFirstPass inv{};
    void *keys[2] = {b + L.keysA, b + L.keysB};
    int *idxs[2] = {(int *)(b + L.idxA), (int *)(b + L.idxB)};
    int cur = -1;   // buffer holding the current (keys, idx); -1 = original input
    int kshift = 0;  // the stored keys are the transformed keys >> kshift
    int kbytes = dbl ? 8 : 4;

    PassArgs a0{};
    a0.n = n;
    a0.up = up;
    a0.seg = seg;
    a0.source = dbl ? 1 : 0;
    a0.src = s;
    a0.vec4 = !dbl && aligned;
    a0.err = device_error_word();
    a0.tile_ofs = tile_ofs;
    a0.groups = grouped ? groups : nullptr;
    a0.ngroups = ngroups;
    bool first_counted = false;             // pass 0's tile counts are taken and scanned
    if (chain) {
        if (!g_hist_host) HIPCHECK(hipHostMalloc(&g_hist_host, 4 * 12 * kRadix, hipHostMallocDefault));
        int g = grid_for(n, kBlock * 16);
        if (g > 2048) g = 2048;
        // chained passes need every digit's start up front: full histograms
        fill_u32(hist, 0, 12 * kRadix);
        if (dbl) k_key_hist<true><<<g, kBlock, 0, g_stream>>>(s, n, up, aligned, hist);
        else k_key_hist<false><<<g, kBlock, 0, g_stream>>>(s, n, up, aligned, hist);
        LAUNCHCHECK();
        if (seg_passes) {
            k_seg_hist<<<gs, kBlock, 0, g_stream>>>(seg.lens, m, seg_passes, hist + key_passes * kRadix);
            LAUNCHCHECK();
        }
        k_hist_scan<<<total, kRadix, 0, g_stream>>>(hist, starts);
        LAUNCHCHECK();
        HIPCHECK(hipMemcpyAsync(g_hist_host, hist, 4 * (size_t)total * kRadix, hipMemcpyDeviceToHost, g_stream));
        HIPCHECK(hipStreamSynchronize(g_stream));
        for (int p = 0; p < total; p++) {
            int nonzero = 0;
            for (int d = 0; d < kRadix; d++) nonzero += g_hist_host[p * kRadix + d] != 0;
            runs[p] = nonzero > 1;
        }
    } else {
        // Pass 0's tile counts, which nearly always serve, also give the
        // keys' OR words; k_or_post posts which passes run to the host.
        // Behind it the device clears the scan status regions and the
        // inverse's counters and column-scans pass 0's counts (or, with
        // grouped tiles, runs pass 0), covering the host's wait and its next
        // launches.
        unsigned *words = hist, *mask_word = (unsigned *)(b + L.counters);
        static_assert(kOrCopies * kOrWords * kOrStride <= 12 * kRadix, "the OR words fit the histogram space");
        if (seg_passes) {
            fill_u32(words, 0, kOrCopies * kOrWords * kOrStride);
            k_seg_or<<<gs, kBlock, 0, g_stream>>>(seg.lens, m, words);
            LAUNCHCHECK();
        }
        // the group counts of every pass
        if (grouped) fill_u32(groups, 0, (int64_t)total * kRadix * ngroups);
        if (small) launch_hist<kRankSmallThreads, kRankSmallItems, false, true>(a0, tiles, dbl, tile_ofs, nullptr, or_parts);
        else launch_hist<kRankThreads, kRankItems, false, true>(a0, tiles, dbl, tile_ofs, nullptr, or_parts);
        const unsigned long long seq = mailbox_next();
        k_or_post<<<1, kOrPostThreads, 0, g_stream>>>(or_parts, tiles, seg_passes ? words : nullptr, key_passes,
                                                      seg_passes, mailbox_device(), seq, mask_word);
        LAUNCHCHECK();
        // An unsegmented rank whose inverse takes two or more partition
        // passes runs the first of them inside its last pass (kFuse): the
        // pass knows every element's sorted position as it places it, so the
        // order is never written and read back.
        if (!segmented && !grouped) inv = partition_invert_begin(n, b + L.invert);
        if (grouped) {
            // Pass 0 is launched whether or not its digit varies, so that
            // the device works through the host's wait, and reads the mask
            // itself (8 10^6 equal ints: 73 us when it runs all the same, 58
            // so, 56 with the host asked first).
            PassArgs a = a0;
            a.keys_out = keys[0];
            a.oshift = dbl ? 0 : 8;
            a.idx_out = idxs[0];
            a.kout = kbytes;
            a.runs = mask_word;
            if (small) launch_grouped<kRankSmallThreads, kRankSmallItems>(a, tiles, dbl, false);
            else launch_grouped<kRankThreads, kRankItems>(a, tiles, dbl, false);
        } else {
            fill_u32(scan_status, 0, 2 * sw * 14);   // status regions: 12 passes, the inverse's counts, pass 0's
            tile_scan(tile_ofs, tiles, nullptr, scan_status + 13 * sw, true, starts);
            first_counted = true;
        }
        const unsigned long long mask = mailbox_wait(seq);
        for (int p = 0; p < total; p++) runs[p] = (mask >> p) & 1u;
        if (grouped && runs[0]) {
            cur = 0;
            kshift = dbl ? 0 : 8;
        }
    }
    int run[12], nrun = 0;
    bool any = false;
    for (int p = 0; p < total; p++) {
        any = any || runs[p];
        if (runs[p] && !(grouped && p == 0)) run[nrun++] = p;
    }
    if (!any) {
        k_rank_identity<<<grid_for(n, kBlock * 4), kBlock, 0, g_stream>>>(rank, n, seg, segmented);
        LAUNCHCHECK();
        return;
    }
    // The last key pass that runs decides whether keys must still travel.
    int last_key_run = -1;
    for (int i = 0; i < nrun; i++) if (run[i] < key_passes) last_key_run = i;
    // pass 0's speculative counts serve when pass 0 runs, unless it is also
    // the fused last pass, which counts the inverse's children as well
    first_counted = first_counted && run[0] == 0 && !(inv.pairs && nrun == 1);

    // Chained passes: per-digit counts below 2^30 (n < 2^30); one set of
    // words for all passes (alternating state sets) and a tile counter per
    // pass, contiguous and cleared together.
    unsigned *tickets = (unsigned *)(b + L.counters);
    if (chain) fill_u32(tickets, 0, (L.status - L.counters) / 4 + kRadix * tiles);
    bool done = false;
    for (int i = 0; i < nrun; i++) {
        const int p = run[i];
        const int out = cur == 0 ? 1 : 0;
        PassArgs a = a0;
        a.starts = starts + p * kRadix;
        a.chain = chain ? (uint32_t *)tile_ofs : nullptr;
        a.ticket = tickets + i;
        a.parity = i & 1;
        a.idx_in = cur < 0 ? nullptr : idxs[cur];
        if (p < key_passes) {
            a.source = cur < 0 ? (dbl ? 1 : 0) : (dbl ? 3 : (kbytes == 4 ? 2 : (kbytes == 2 ? 5 : 6)));
            a.src = cur < 0 ? s : keys[cur];
            a.shift = 8 * p - kshift;
        } else {
            a.source = 4;
            a.src = nullptr;
            a.shift = 8 * (p - key_passes);
        }
        a.vec4 = a.source == 5 || a.source == 6 || ((a.source == 0 || a.source == 2) && ((uintptr_t)a.src & 15) == 0);
        a.keys_out = i < last_key_run ? keys[out] : nullptr;
        a.kout = kbytes;
        if (a.keys_out && !dbl) {
            // the next pass that reads keys is run[i + 1] (key passes come first)
            const int nshift = 8 * run[i + 1];
            const int width = 32 - nshift;
            a.kout = width > 16 ? 4 : (width > 8 ? 2 : 1);
            a.oshift = nshift - kshift;
        }
        a.idx_out = idxs[out];
        if (grouped) a.groups = groups + (int64_t)p * kRadix * ngroups;
        const bool last = i + 1 == nrun;
        const bool fuse = inv.pairs && last;
        a.pairs = fuse ? inv.pairs : nullptr;
        a.tile_ofs2 = tile_ofs2;
        a.clog = inv.clog;
        a.rank = rank;
        a.rel = segmented;
        if (!chain && !(i == 0 && first_counted)) {
            if (fuse) launch_hist<kRankThreads, kRankItems, true, false>(a, tiles, dbl, tile_ofs, tile_ofs2, nullptr);
            else if (small) launch_hist<kRankSmallThreads, kRankSmallItems, false, false>(a, tiles, dbl, tile_ofs, nullptr, nullptr);
            else launch_hist<kRankThreads, kRankItems, false, false>(a, tiles, dbl, tile_ofs, nullptr, nullptr);
            // the column scan also leaves the digits' starts (the scan of its totals)
            if (!grouped) tile_scan(tile_ofs, tiles, nullptr, scan_status + i * sw, true, starts + p * kRadix);
            // the children's totals go to the inverse's counters
            if (fuse) tile_scan(tile_ofs2, tiles, inv.cnt, scan_status + 12 * sw, true);
        }
        if (small) {
            launch_grouped<kRankSmallThreads, kRankSmallItems>(a, tiles, dbl, last);
        } else if (grouped) {
            launch_grouped<kRankThreads, kRankItems>(a, tiles, dbl, last);
        } else if (fuse) {
            if (dbl) k_rank_pass<uint64_t, 0, kFuse, false><<<(unsigned)tiles, kRankThreads, 0, g_stream>>>(a);
            else k_rank_pass<uint32_t, 0, kFuse, false><<<(unsigned)tiles, kRankThreads, 0, g_stream>>>(a);
            LAUNCHCHECK();
        } else {
            launch_order<false, kRankThreads, kRankItems>(a, dim3((unsigned)tiles), dbl);
        }
        if (a.keys_out) {
            kshift += a.oshift;
            kbytes = a.kout;
        }
        cur = out;
        done = grouped && last;
    }
    // rank = inverse of the final order
    if (done) return;
    if (inv.pairs) partition_invert_finish(rank, n, b + L.invert);
    else partition_invert(rank, idxs[cur], n, segmented ? sd : nullptr, m, b + L.invert);
}

int64_t rank_scratch_bytes(int64_t n, bool dbl) { return RankScratch(n, dbl).bytes; }

}  // namespace cvlhip

using namespace cvlhip;

#define RANKS(UD, UPV, TY, DBL)                                                                  \
    void rk##UD##_lu##TY(vec_p d, vec_p s, int len, vec_p scratch) {                             \
        rank_run((int *)d, s, len, DBL, UPV, nullptr, 0, scratch);                               \
    }                                                                                            \
    int rk##UD##_lu##TY##_scratch(int len) { return units_for_bytes(rank_scratch_bytes(len, DBL)); } \
    unsigned int rk##UD##_lu##TY##_inplace(void) { return INPLACE_NONE; }                        \
    void rk##UD##_le##TY(vec_p d, vec_p s, vec_p segd, int vec_len, int seg_count, vec_p scratch) { \
        rank_run((int *)d, s, vec_len, DBL, UPV, segd, seg_count, scratch);                      \
    }                                                                                            \
    int rk##UD##_le##TY##_scratch(int vec_len, int seg_count) {                                  \
        (void)seg_count;                                                                         \
        return units_for_bytes(rank_scratch_bytes(vec_len, DBL));                                \
    }                                                                                            \
    unsigned int rk##UD##_le##TY##_inplace(void) { return INPLACE_NONE; }

extern "C" {
RANKS(u, true, z, false)
RANKS(d, false, z, false)
RANKS(u, true, d, true)
RANKS(d, false, d, true)
}
