// mlp.hpp -- shape of the learned dispatcher's network and its one-wave
// forward pass used when a segment descriptor is built.  No counterpart in
// the reference.
//
// Network: x (kF features) -> ReLU(W1 x + b1) (kH) -> ReLU(W2 h1 + b2) (kH)
//          -> W3 h2 + b3 (kA outputs, one predicted log-time per schedule).
// Parameters live in one flat array in the order W1 b1 W2 b2 W3 b3
// (row-major W[out][in]).
#pragma once

#include "cvl_hip.hpp"
#include "segd.hpp"

namespace cvlhip {

constexpr int kF = 3 + 2 * kLenClasses + 2, kH = 32, kA = 6;
constexpr int kW1 = 0, kB1 = kW1 + kH * kF, kW2 = kB1 + kH, kB2 = kW2 + kH * kH, kW3 = kB2 + kH,
              kB3 = kW3 + kA * kH, kParams = kB3 + kA;
static_assert(kH <= kWave && kA <= kWave && kF <= kWave, "one wave holds a layer");

// Feature i of a descriptor of n elements in m segments whose length-class
// histogram is elems[]/segs[]:
//   [0] log2(n)/32   [1] log2(m)/32   [2] log2(max(n/m, 1))/20
//   [3 + c]      fraction of the elements in segments of class c
//   [3 + 21 + c] fraction of the segments in class c
//   [45] 1 for 8-byte values   [46] 1 for a reduction
__device__ __forceinline__ float sched_feature(int i, int64_t n, int64_t m, const uint32_t *elems,
                                               const uint32_t *segs, bool dbl, bool red) {
    const float nn = n > 0 ? (float)n : 1.f, mm = m > 0 ? (float)m : 1.f;
    if (i == 0) return log2f(nn) / 32.f;
    if (i == 1) return log2f(mm) / 32.f;
    if (i == 2) return log2f(nn / mm > 1.f ? nn / mm : 1.f) / 20.f;
    if (i < 3 + kLenClasses) return (float)elems[i - 3] / nn;
    if (i < 3 + 2 * kLenClasses) return (float)segs[i - 3 - kLenClasses] / mm;
    if (i == 3 + 2 * kLenClasses) return dbl ? 1.f : 0.f;
    if (i == 4 + 2 * kLenClasses) return red ? 1.f : 0.f;
    return 0.f;
}

// Schedules a descriptor admits whatever the network predicts.  The flat
// 8-row schedule (0) takes any descriptor.  The others are admitted for
// reductions up to 2^kOthersMaxLogN elements, the largest length the network
// was trained on, and for scans below it.  All arms of eleven kinds of lengths
// (Zipf, geometric, equal, uniform), total ms of 8 rows / the network's pick /
// the fastest arm: scans of 2^25 0.83 / 0.85 / 0.83 (doubles 1.60 / 1.76 /
// 1.60), 8 rows the fastest of every kind there and beyond; reductions of 2^25
// 0.95 / 0.61 / 0.61 (1.11 / 1.00 / 1.00), short segments gaining from 2 rows;
// but of 2^27 the pick was a wave per segment at twice the time of 8 rows for
// geometric(256) lengths.  The per-segment ones (3 thread, 4
// wave, 5 workgroup) give a segment one lane, wave or workgroup: one long
// segment serialises them and a few segments leave the chip idle, so each
// is admitted only when the longest segment is below 2^(kArmMaxClass + 1)
// and there are at least 2^kArmMinLogM segments.  (A workgroup takes 50 us for
// 2^16 elements: with that limit the network's pick for 700000 ints in 3500
// segments, one of them of 60000, took 52 us against 15 in flat tiles; of 209
// training workloads none is faster for segments above 2^14.)  cmax: the
// highest length class holding a segment (-1: none).  Bit a set: schedule a
// admitted.
constexpr int kArmMaxClass[3] = {5, 12, 13};
constexpr int kArmMinLogM[3] = {14, 11, 9};
constexpr int kOthersMaxLogN = 25;
__host__ __device__ inline unsigned sched_admitted(int cmax, int64_t n, int64_t m, bool reduce) {
    const int64_t most = (int64_t)1 << kOthersMaxLogN;
    if (reduce ? n > most : n >= most) return 1u;
    unsigned a = 7u;
    for (int k = 0; k < 3; k++)
        if (cmax <= kArmMaxClass[k] && m >= ((int64_t)1 << kArmMinLogM[k])) a |= 1u << (3 + k);
    return a;
}
__host__ __device__ inline int max_len_class(const uint32_t *segs) {
    int c = kLenClasses - 1;
    while (c >= 0 && segs[c] == 0) c--;
    return c;
}

// Parameters staged in LDS for mlp_pick_wave: rows of W2 and W3 one word
// longer than in the array, so that the lanes of a step (one row each) read
// different banks; W1's rows are of odd length already.
constexpr int kPitch = kH + 1;
constexpr int kLB2 = kW2 + kH * kPitch, kLW3 = kLB2 + kH, kLB3 = kLW3 + kA * kPitch, kLdsParams = kLB3 + kA;
__device__ __forceinline__ int lds_param(int i) {
    if (i < kW2) return i;
    if (i < kB2) return i + (i - kW2) / kH;
    if (i < kW3) return i - kB2 + kLB2;
    if (i < kB3) return i - kW3 + kLW3 + (i - kW3) / kH;
    return i - kB3 + kLB3;
}
// Stage the parameters (THREADS threads, which then need a barrier), all
// loads in flight together.
template <int THREADS>
__device__ __forceinline__ void stage_params(const float *__restrict__ params, float *s_P) {
    constexpr int PER = (kParams + THREADS - 1) / THREADS;
    float v[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const int i = k * THREADS + (int)threadIdx.x;
        v[k] = i < kParams ? params[i] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const int i = k * THREADS + (int)threadIdx.x;
        if (i < kParams) s_P[lds_param(i)] = v[k];
    }
}

// The value x has in lane i (the same i in every lane).
__device__ __forceinline__ float lane_value(float x, int i) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), i));
}

// Forward pass of one feature vector by one whole wave (lane i holds
// feature i); every lane returns the index of the smallest prediction among
// the admitted schedules (the first one on ties).  P: the staged parameters.
// Sums run in index order, so the same parameters and features always give
// the same pick.  Bound by latency: the steps are unrolled, so that their
// LDS reads are in flight together, and take the other lanes' values from
// registers (v_readlane) instead of LDS shuffles (with the launch that waits
// for the pick: 9.3 -> 4.6 us).
__device__ __forceinline__ int mlp_pick_wave(const float *__restrict__ P, float feature_of_lane, unsigned admitted) {
    const int lane = lane_id();
    const int j1 = lane < kH ? lane : kH - 1;       // lanes past a layer's width compute a copy
    float a = P[kB1 + j1];
#pragma unroll
    for (int i = 0; i < kF; i++) a += P[kW1 + j1 * kF + i] * lane_value(feature_of_lane, i);
    const float h1 = a > 0.f ? a : 0.f;
    a = P[kLB2 + j1];
#pragma unroll
    for (int i = 0; i < kH; i++) a += P[kW2 + j1 * kPitch + i] * lane_value(h1, i);
    const float h2 = a > 0.f ? a : 0.f;
    const int j3 = lane < kA ? lane : kA - 1;
    a = P[kLB3 + j3];
#pragma unroll
    for (int i = 0; i < kH; i++) a += P[kLW3 + j3 * kPitch + i] * lane_value(h2, i);
    int best = 0;                                   // flat8 is always admitted
    float by = lane_value(a, 0);
#pragma unroll
    for (int k = 1; k < kA; k++) {
        const float v = lane_value(a, k);
        if (((admitted >> k) & 1u) && v < by) { by = v; best = k; }
    }
    return best;
}

}  // namespace cvlhip
