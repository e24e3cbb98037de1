// Row staging shared by the f32-MFMA SSD forward and backward (ssd_f32.hip,
// ssd_f32_bwd.hip): chunks of 64 fused (step, rank) rows of strided [b, l, m,
// (h|g), W] tensors into LDS, and the per-row decay tables.
#pragma once

#include "bwd_core.h"
#include "common.h"

namespace mamba {

constexpr int kFR = 64;  // fused rows per chunk
constexpr double kFLog2e = 1.4426950408889634;

// The decays of a chunk's rows (lane = row) in log2 units, summed in 64 bits: the
// decay between two rows is a difference of sums that may be far larger than
// itself, and with sums in f32 it is off by their rounding (under strong decays
// that left dv and dB up to 1.8 times as far from 64 bits as sums taken row by row
// over 32).  cs + lo is the sum up to the row; the difference of two rows is
// (cs_i - cs_j) + (lo_i - lo_j), and f_exp of it costs less than an __expf.
struct FDecay {
    float cs, lo;
    float a, b;  // decay factors from the row to the chunk's end, and up to the row
    float end;   // the whole chunk's, in log2 units
};
__device__ __forceinline__ float f_exp(float x) { return __builtin_amdgcn_exp2f(x); }
// x: the row's log-decay.  At the least -2^14, whose exp is 0 as that of all below: a
// mask's lowest value or -inf, kept, would make the sums infinite in log2 units and
// every difference after it NaN (a NaN stays one).
__device__ __forceinline__ FDecay f_decay(double x) {
    x = x < -16384. ? -16384. : x;
    const double cs = wave_incl_scan64(x * kFLog2e), end = wave_lane64(cs, 63);
    FDecay d;
    d.cs = (float)cs;
    d.lo = fabsf(d.cs) < INFINITY ? (float)(cs - (double)d.cs) : 0.f;
    d.a = f_exp((float)(end - cs));
    d.b = f_exp(d.cs);
    d.end = (float)end;
    return d;
}

// four values of a row, as f32
template <typename T>
struct FRaw;
template <>
struct FRaw<float> {
    float4 v;
    __device__ __forceinline__ float4 get() const { return v; }
};
template <>
struct FRaw<bf16_t> {
    uint2 v;
    __device__ __forceinline__ float4 get() const {
        return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                           __uint_as_float(v.y & 0xffff0000u));
    }
};

// The rows of chunk c that thread tid stages: W values per row, NT threads.
// Rows past the sequence end read as zero.
template <typename T, int W, int NT>
__device__ __forceinline__ void f_fetch(FRaw<T> (&raw)[kFR * W / 4 / NT], const T* base, int64_t sl, int64_t sm, int L,
                                        int mshift, int c, int tid) {
    constexpr int RW = W / 4;
#pragma unroll
    for (int q = 0; q < kFR * W / 4 / NT; ++q) {
        const int e = tid + NT * q, row = e / RW, col = (e % RW) * 4;
        const int t = c * (kFR >> mshift) + (row >> mshift);
        const int64_t at = (int64_t)min(t, L - 1) * sl + (int64_t)(row & ((1 << mshift) - 1)) * sm + col;
        raw[q].v = *reinterpret_cast<const decltype(raw[q].v)*>(base + at);
    }
}
// flip: 0, or kFR - 1 for the rows in reverse
template <typename T, int W, int NT, int PITCH>
__device__ __forceinline__ void f_commit(const FRaw<T> (&raw)[kFR * W / 4 / NT], float* dst, int L, int mshift, int c,
                                         int tid, int flip = 0) {
    constexpr int RW = W / 4;
#pragma unroll
    for (int q = 0; q < kFR * W / 4 / NT; ++q) {
        const int e = tid + NT * q, row = e / RW, col = (e % RW) * 4;
        const int t = c * (kFR >> mshift) + (row >> mshift);
        const float4 z = {0.f, 0.f, 0.f, 0.f};
        *reinterpret_cast<float4*>(dst + (row ^ flip) * PITCH + col) = t < L ? raw[q].get() : z;
    }
}

// One wave's state tiles h[n][p] (rows n, columns p): tile t = slot + 4 q at
// rows 32 (t / (PB / 32)), columns 32 (t % (PB / 32)); QT tiles per wave, all
// present where the slot has any.
//   h <- dec h + sum_j B[j][n] (w_j v[j][p])
template <int PB, int N, int QT, int VP>
__device__ __forceinline__ void f_update(bwd_f32x16 (&acc)[QT], const float* sB, const float* sV, const float* w64, float dec,
                                         int slot, int i32, int hf) {
    constexpr int PT = PB / 32, TILES = PT * (N / 32), BP = N + 4;
    if (slot >= TILES) return;
#pragma unroll
    for (int q = 0; q < QT; ++q)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[q][r] *= dec;
    // a wave's tiles share their columns (4 is a multiple of PT)
    const float* Ap = sB + 4 * hf * BP + 32 * (slot / PT) + i32;
    const float* Bp = sV + 4 * hf * VP + 32 * (slot % PT) + i32;
#pragma unroll
    for (int s = 0; s < kFR / 8; ++s) {
        const float4 w = *reinterpret_cast<const float4*>(&w64[8 * s + 4 * hf]);
        const float wj[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float v = wj[k] * Bp[(8 * s + k) * VP];
#pragma unroll
            for (int q = 0; q < QT; ++q) acc[q] = bwd_mfma(Ap[(8 * s + k) * BP + 128 / PT * q], v, acc[q]);
        }
        if (s & 1) __builtin_amdgcn_sched_barrier(0);  // bounds the loads moved ahead (registers)
    }
}

}  // namespace mamba
