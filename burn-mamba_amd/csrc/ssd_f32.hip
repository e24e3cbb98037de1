// SSD forward with every product on f32 MFMA, split over sequence segments:
// f32 I/O (the reference's default float), and bf16 I/O of the shapes that the
// bf16 kernels do not take.  Headdim a multiple of 32, dstate 32, 64 or 128.
//
// The Mamba-2 SSD (src/mamba2/ssd/serial.rs:34-506) and the Mamba-3 single- and
// double-SSD (src/mamba3/single_ssd/ssd/serial_recalculated/serial_recalculated.rs:86-291,
// src/mamba3/double_ssd/ssd/serial.rs:118-409) are one recurrence on fused rows
// j = (step, rank); with cs the cumulative log-decay of a row's step,
//   y_i   = exp(cs_i) C_i . h + sum_j W_ij (C_i . B_j) v_j  (+ D v_i)
//   W_ij  = exp(cs_i - cs_j) sc_j (earlier step), gm_i (own step), 0 (later)
//   h'    = exp(cs_end) h + sum_j exp(cs_end - cs_j) sc_j v_j (x) B_j
// and Mamba-2 is one rank with sc = gm = dt.  Chunks are 64 fused rows whatever
// chunk_len says: the chunked form is exact for any length, so only rounding
// differs.
//
// Two launches (one when a (batch, head) is not split):
//   1. ssd_f32_state: one 4-wave workgroup per (batch, head, 64 columns of
//      headdim, segment but the last) forms the segment's state, the first from
//      the initial state, the others from zero.
//   2. ssd_f32_scan: one 8-wave workgroup per (.., segment) sums the earlier
//      segments' states into its entry state and walks the segment's chunks.
//      Segment 0 finds the initial state in the last segment's place in the
//      workspace, which has no state of its own there: only the first launch
//      reads it from its memory, which the scan may write (final_state may be
//      the same memory).
//      Waves 0-3 each form a 32 x 32 tile of y; waves 4-7 form C.B^T, then
//      update the state, which stays in their accumulators, so that on every
//      SIMD one wave's y tile runs beside another's update.
// What bounds it: the f32 MFMA rate (157 TFLOP/s) in the large, and one chunk's
// chain of three barriers in the small; the segments exist so that a launch
// covers the chip when (batch, head) alone does not.  Segments, and not a
// workgroup per chunk with every chunk's state in memory, because the states
// (32 KB at 64 x 128) would be most of the traffic.  Measured against the SIMT
// kernels (three launches), f32: 2 x 512 tokens, 8 heads 64 x 64, 62 -> 21 us;
// the block forward at 2 x 256, d_model 256, 64 x 64, rank 4, 357 -> 150 us; a
// training step at 2 x 4096, 32 heads 64 x 128, rank 4, 19.3 -> 6.5 ms (its
// forward 13.6 -> 0.9 ms).
//
// f32 MFMA 32x32x2 (see bwd_core.h): A[m][k] and B[k][n] are one value per lane
// (m or n = lane % 32, k = lane / 32).  The four products of a 16-byte LDS read
// take k = 8 s + 4 (lane / 32) + 0..3 on both sides.
#include <algorithm>

#include "ssd_f32.h"
#include "ssd_f32_rows.h"

namespace mamba {

// log-decay and weights of one fused row (lane) of a chunk, in flight
struct FTabRaw {
    float da, gm, sc;
};

struct FTables {
    float cs[kFR], lo[kFR], gm[kFR], sc[kFR];  // cs, lo: FDecay
    float w[kFR];  // sc exp(cs_end - cs): the weights of the state update
    float dec, end;
};

// What one workgroup works on.
struct FJob {
    int b, h, g, p0, s, c0, c1;
    int64_t hp;  // (batch, head, block of headdim)
};

__device__ __forceinline__ FJob f_job(const SsdF32Params& p, int nseg, int PB) {
    FJob j;
    const int npb = p.P / PB;
    const int u = blockIdx.x / nseg;
    j.s = blockIdx.x % nseg;
    j.hp = u;
    j.p0 = (u % npb) * PB;
    j.h = (u / npb) % p.H;
    j.b = u / npb / p.H;
    j.g = j.h / (p.H / p.G);
    j.c0 = j.s * p.cps;
    j.c1 = min(p.nch, j.c0 + p.cps);
    return j;
}

// one wave: lane = fused row
__device__ __forceinline__ FTabRaw f_tab_fetch(const SsdF32Params& p, const FJob& j, int c, int lane) {
    const int t = min(c * (kFR >> p.mshift) + (lane >> p.mshift), p.L - 1);
    FTabRaw r;
    r.da = p.da[(int64_t)j.b * p.da_sb + (int64_t)t * p.da_sl + (int64_t)j.h * p.da_sh];
    r.gm = p.gm ? p.gm[(int64_t)j.b * p.gm_sb + (int64_t)t * p.gm_sl + (int64_t)j.h * p.gm_sh] : 1.f;
    r.sc = p.sc ? p.sc[(int64_t)j.b * p.sc_sb + (int64_t)t * p.sc_sl + (int64_t)j.h * p.sc_sh] : 1.f;
    return r;
}
__device__ __forceinline__ FDecay f_tab_decay(const SsdF32Params& p, const FTabRaw& r, float A, int c, int lane) {
    const bool ok = c * (kFR >> p.mshift) + (lane >> p.mshift) < p.L;
    // a step's decay counts once, at its first rank
    return f_decay(ok && (lane & (p.M - 1)) == 0 ? (double)r.da * A : 0.);
}
__device__ __forceinline__ void f_tab_commit(const SsdF32Params& p, const FTabRaw& r, const FDecay& d, FTables& T, int c,
                                             int lane) {
    const bool ok = c * (kFR >> p.mshift) + (lane >> p.mshift) < p.L;
    const float sc = ok ? r.sc : 0.f;
    T.cs[lane] = d.cs;
    T.lo[lane] = d.lo;
    T.gm[lane] = ok ? r.gm : 0.f;
    T.sc[lane] = sc;
    T.w[lane] = d.a * sc;
    if (lane == 63) {
        T.dec = d.b;
        T.end = d.end;
    }
}

// The initial state's tile t (rows n 32 (t / (PB / 32)), columns p 32 (t % (PB / 32))).
template <int PB, int N>
__device__ __forceinline__ void f_h0(const SsdF32Params& p, const FJob& j, int t, int i32, int hf, bwd_f32x16& a) {
    constexpr int PT = PB / 32;
    const int64_t at = (int64_t)(j.p0 + 32 * (t % PT) + i32) * N + 32 * (t / PT) + 4 * hf;
    const int64_t bh = (int64_t)j.b * p.H + j.h, pn = (int64_t)p.P * N;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float4 x = {0.f, 0.f, 0.f, 0.f};
        if (p.h0) x = *reinterpret_cast<const float4*>(p.h0 + bh * pn + at + 8 * k);
        if (p.init_hpr) {
            const float4 i = *reinterpret_cast<const float4*>(p.init_hpr + j.h * pn + at + 8 * k);
            x.x += i.x; x.y += i.y; x.z += i.z; x.w += i.w;
        }
        a[4 * k] = x.x; a[4 * k + 1] = x.y; a[4 * k + 2] = x.z; a[4 * k + 3] = x.w;
    }
}

template <int PB, int N>
struct FStateLds {
    float B[kFR * (N + 4)];
    float V[kFR * (PB + 8)];
    float w[kFR];  // as FTables
    float dec, end;
};

template <typename T, int PB, int N>
__global__ __launch_bounds__(256, 3) void ssd_f32_state(SsdF32Params p) {
    extern __shared__ __align__(16) char f_smem[];
    FStateLds<PB, N>& S = *reinterpret_cast<FStateLds<PB, N>*>(f_smem);
    constexpr int PT = PB / 32, TILES = PT * (N / 32), QT = (TILES + 3) / 4, NT = 256;
    const int tid = threadIdx.x, wv = wave_id(), lane = tid & 63, i32 = lane & 31, hf = lane >> 5;
    const FJob j = f_job(p, p.S - 1, PB);
    const T* vb = static_cast<const T*>(p.v) + (int64_t)j.b * p.v_sb + (int64_t)j.h * p.v_sh + j.p0;
    const T* Bb = static_cast<const T*>(p.Bm) + (int64_t)j.b * p.B_sb + (int64_t)j.g * p.B_sg;
    const float A = p.A ? p.A[j.h] : 1.f;
    FRaw<T> rb[kFR * N / 4 / NT], rv[kFR * PB / 4 / NT];
    FTabRaw rt = {0.f, 0.f, 0.f};
    bwd_f32x16 acc[QT];
    float* const seg = p.seg + j.hp * p.S * (int64_t)(N * PB) + lane;
#pragma unroll
    for (int q = 0; q < QT; ++q) {
        const int t = wv + 4 * q;
        if (t >= TILES) break;
        if (j.s == 0 && (p.h0 || p.init_hpr)) {
            f_h0<PB, N>(p, j, t, i32, hf, acc[q]);
            float* out = seg + (p.S - 1) * (int64_t)(N * PB) + t * 1024;
#pragma unroll
            for (int r = 0; r < 16; ++r) out[r * 64] = acc[q][r];
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[q][r] = 0.f;
        }
    }
    auto fetch = [&](int c) {
        f_fetch<T, N, NT>(rb, Bb, p.B_sl, p.B_sm, p.L, p.mshift, c, tid);
        f_fetch<T, PB, NT>(rv, vb, p.v_sl, p.v_sm, p.L, p.mshift, c, tid);
        if (wv == 0) rt = f_tab_fetch(p, j, c, lane);
    };
    auto commit = [&](int c) {
        f_commit<T, N, NT, N + 4>(rb, S.B, p.L, p.mshift, c, tid);
        f_commit<T, PB, NT, PB + 8>(rv, S.V, p.L, p.mshift, c, tid);
        if (wv == 0) {
            const FDecay d = f_tab_decay(p, rt, A, c, lane);
            S.w[lane] = c * (kFR >> p.mshift) + (lane >> p.mshift) < p.L ? d.a * rt.sc : 0.f;
            if (lane == 63) {
                S.dec = d.b;
                S.end = d.end;
            }
        }
    };
    fetch(j.c0);
    commit(j.c0);
    __syncthreads();
    float total = 0.f;
    for (int c = j.c0; c < j.c1; ++c) {
        if (c + 1 < j.c1) fetch(c + 1);
        total += S.end;
        f_update<PB, N, QT, PB + 8>(acc, S.B, S.V, S.w, S.dec, wv, i32, hf);
        __syncthreads();
        if (c + 1 < j.c1) commit(c + 1);
        __syncthreads();
    }
    float* out = seg + j.s * (int64_t)(N * PB);
#pragma unroll
    for (int q = 0; q < QT; ++q) {
        const int t = wv + 4 * q;
        if (t >= TILES) break;
#pragma unroll
        for (int r = 0; r < 16; ++r) out[t * 1024 + r * 64] = acc[q][r];
    }
    if (tid == 0) p.segd[j.hp * p.S + j.s] = total;
}

template <int PB, int N>
struct FScanLds {
    float B[kFR * (N + 4)];
    float C[kFR * (N + 4)];
    float V[kFR * (PB + 8)];
    float h[N * (PB + 8)];    // the state entering the chunk, [n][p]
    float W[kFR * (kFR + 8)];  // W_ij (C_i . B_j), [j][i]
    FTables T;
    float zero[32];  // read for v where there is no D: 0 v of an infinite v would be NaN
};

template <typename T, int PB, int N>
__global__ __launch_bounds__(512) void ssd_f32_scan(SsdF32Params p) {
    extern __shared__ __align__(16) char f_smem[];
    FScanLds<PB, N>& S = *reinterpret_cast<FScanLds<PB, N>*>(f_smem);
    constexpr int PT = PB / 32, TILES = PT * (N / 32), QT = (TILES + 3) / 4, NT = 512;
    constexpr int NP = N + 4, VP = PB + 8, WP = kFR + 8;
    const int tid = threadIdx.x, wv = wave_id(), lane = tid & 63, i32 = lane & 31, hf = lane >> 5;
    const FJob j = f_job(p, p.S, PB);
    const T* vb = static_cast<const T*>(p.v) + (int64_t)j.b * p.v_sb + (int64_t)j.h * p.v_sh + j.p0;
    const T* Bb = static_cast<const T*>(p.Bm) + (int64_t)j.b * p.B_sb + (int64_t)j.g * p.B_sg;
    const T* Cb = static_cast<const T*>(p.Cm) + (int64_t)j.b * p.C_sb + (int64_t)j.g * p.C_sg;
    T* yb = static_cast<T*>(p.y) + (int64_t)j.b * p.y_sb + (int64_t)j.h * p.y_sh + j.p0;
    const float A = p.A ? p.A[j.h] : 1.f;
    const float D = p.D ? p.D[j.h] : 0.f;
    const int steps = kFR >> p.mshift;
    FRaw<T> rb[kFR * N / 4 / NT], rc[kFR * N / 4 / NT], rv[kFR * PB / 4 / NT];
    FTabRaw rt = {0.f, 0.f, 0.f};
    FDecay rd = {0.f, 0.f, 0.f, 0.f, 0.f};
    auto fetch = [&](int c) {
        f_fetch<T, N, NT>(rb, Bb, p.B_sl, p.B_sm, p.L, p.mshift, c, tid);
        f_fetch<T, N, NT>(rc, Cb, p.C_sl, p.C_sm, p.L, p.mshift, c, tid);
        f_fetch<T, PB, NT>(rv, vb, p.v_sl, p.v_sm, p.L, p.mshift, c, tid);
        if (wv == 7) rt = f_tab_fetch(p, j, c, lane);
    };
    auto commit = [&](int c) {
        f_commit<T, N, NT, NP>(rb, S.B, p.L, p.mshift, c, tid);
        f_commit<T, N, NT, NP>(rc, S.C, p.L, p.mshift, c, tid);
        f_commit<T, PB, NT, VP>(rv, S.V, p.L, p.mshift, c, tid);
        if (wv == 7) f_tab_commit(p, rt, rd, S.T, c, lane);
    };
    const bool st = wv >= 4;  // wave-uniform
    const int w4 = wv & 3;
    bwd_f32x16 acc[QT];       // state waves: h[n][p]
    auto publish = [&]() {
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            const int t = w4 + 4 * q;
            if (t >= TILES) break;
            float* hp = S.h + 32 * (t / PT) * VP + 32 * (t % PT) + i32;
#pragma unroll
            for (int r = 0; r < 16; ++r) hp[bwd_row(r, hf) * VP] = acc[q][r];
        }
    };
    fetch(j.c0);
    if (st) {
        // the entering state: segment 0's end through the later ones, oldest first
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            const int t = w4 + 4 * q;
            if (t >= TILES) break;
            const float* sp = p.seg + j.hp * p.S * (int64_t)(N * PB) + t * 1024 + lane;
            if (p.S == 1) {
                f_h0<PB, N>(p, j, t, i32, hf, acc[q]);
                continue;
            }
            const bool zero = j.s == 0 && !p.h0 && !p.init_hpr;
            const int64_t first = j.s == 0 ? p.S - 1 : 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[q][r] = zero ? 0.f : sp[first * (N * PB) + r * 64];
#pragma unroll 4
            for (int u = 1; u < j.s; ++u) {
                const float dec = f_exp(p.segd[j.hp * p.S + u]);
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[q][r] = __builtin_fmaf(acc[q][r], dec, sp[(int64_t)u * (N * PB) + r * 64]);
            }
        }
        publish();
    }
    if (wv == 7) rd = f_tab_decay(p, rt, A, j.c0, lane);
    if (tid < 32) S.zero[tid] = 0.f;
    commit(j.c0);
    __syncthreads();
    // y waves: rows 32 it, columns 32 pt
    const int it = PT == 2 ? w4 >> 1 : w4 & 1, pt = PT == 2 ? w4 & 1 : 0;
    const bool yw = !st && (PT == 2 || w4 < 2);
    for (int c = j.c0; c < j.c1; ++c) {
        if (c + 1 < j.c1) fetch(c + 1);
        bwd_f32x16 ya;
        if (yw) {
            // y^T[p][i] = exp(cs_i) sum_n h[n][p] C[i][n]
#pragma unroll
            for (int r = 0; r < 16; ++r) ya[r] = 0.f;
            const float* Ap = S.h + 4 * hf * VP + 32 * pt + i32;
            const float* Bp = S.C + (32 * it + i32) * NP + 4 * hf;
#pragma unroll
            for (int s = 0; s < N / 8; ++s) {
                const float4 cv = *reinterpret_cast<const float4*>(Bp + 8 * s);
                const float cj[4] = {cv.x, cv.y, cv.z, cv.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) ya = bwd_mfma(Ap[(8 * s + k) * VP], cj[k], ya);
            }
            const float e = f_exp(S.T.cs[32 * it + i32]);
#pragma unroll
            for (int r = 0; r < 16; ++r) ya[r] *= e;
        }
        if (st && w4 < 3) {
            // tile (jt, wi) of C.B^T as [j][i]: (0, 0), (0, 1), (1, 1)
            const int jt = w4 >> 1, wi = (w4 + 1) >> 1;
            bwd_f32x16 a;
#pragma unroll
            for (int r = 0; r < 16; ++r) a[r] = 0.f;
            const float* Ap = S.B + (32 * jt + i32) * NP + 4 * hf;
            const float* Bp = S.C + (32 * wi + i32) * NP + 4 * hf;
#pragma unroll
            for (int s = 0; s < N / 8; ++s) {
                const float4 bv = *reinterpret_cast<const float4*>(Ap + 8 * s);
                const float4 cv = *reinterpret_cast<const float4*>(Bp + 8 * s);
                a = bwd_mfma(bv.x, cv.x, a);
                a = bwd_mfma(bv.y, cv.y, a);
                a = bwd_mfma(bv.z, cv.z, a);
                a = bwd_mfma(bv.w, cv.w, a);
            }
            const int i = 32 * wi + i32, si = i >> p.mshift;
            const float csi = S.T.cs[i], loi = S.T.lo[i], gmi = S.T.gm[i];
            float* Wp = S.W + 32 * jt * WP + i;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int jr = bwd_row(r, hf), jj = 32 * jt + jr, sj = jj >> p.mshift;
                const float k = sj < si ? f_exp((csi - S.T.cs[jj]) + (loi - S.T.lo[jj])) * S.T.sc[jj] : gmi;
                Wp[jr * WP] = sj <= si ? a[r] * k : 0.f;
            }
        }
        // wave 7 has no tile of C.B^T: the next chunk's decays
        if (wv == 7 && c + 1 < j.c1) rd = f_tab_decay(p, rt, A, c + 1, lane);
        __syncthreads();
        if (yw) {
            // += sum_j v[j][p] W[j][i]
            const float* Ap = S.V + 4 * hf * VP + 32 * pt + i32;
            const float* Bp = S.W + 4 * hf * WP + 32 * it + i32;
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int k = 0; k < 4; ++k) ya = bwd_mfma(Ap[(8 * s + k) * VP], Bp[(8 * s + k) * WP], ya);
            if (it)
#pragma unroll
                for (int s = 4; s < 8; ++s)
#pragma unroll
                    for (int k = 0; k < 4; ++k) ya = bwd_mfma(Ap[(8 * s + k) * VP], Bp[(8 * s + k) * WP], ya);
            // lane = row i, four consecutive columns per register quad
            const int i = 32 * it + i32, t = c * steps + (i >> p.mshift);
            if (t < p.L) {
                T* yr = yb + (int64_t)t * p.y_sl + (int64_t)(i & (p.M - 1)) * p.y_sm + 32 * pt + 4 * hf;
                const float* vr = p.D ? S.V + i * VP + 32 * pt + 4 * hf : S.zero + 4 * hf;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float4 x = *reinterpret_cast<const float4*>(vr + 8 * k);
                    const float o0 = __builtin_fmaf(D, x.x, ya[4 * k]), o1 = __builtin_fmaf(D, x.y, ya[4 * k + 1]);
                    const float o2 = __builtin_fmaf(D, x.z, ya[4 * k + 2]), o3 = __builtin_fmaf(D, x.w, ya[4 * k + 3]);
                    if constexpr (sizeof(T) == 4)
                        *reinterpret_cast<float4*>(yr + 8 * k) = make_float4(o0, o1, o2, o3);
                    else
                        *reinterpret_cast<uint2*>(yr + 8 * k) = make_uint2(pack_bf16x2(o0, o1), pack_bf16x2(o2, o3));
                }
            }
        }
        if (st) f_update<PB, N, QT, PB + 8>(acc, S.B, S.V, S.T.w, S.T.dec, w4, i32, hf);
        __syncthreads();
        if (c + 1 < j.c1) {
            commit(c + 1);
            if (st) publish();
            __syncthreads();
        }
    }
    if (st && j.s == p.S - 1) {
        const int64_t bh = (int64_t)j.b * p.H + j.h;
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            const int t = w4 + 4 * q;
            if (t >= TILES) break;
            float* out = p.hT + (bh * p.P + j.p0 + 32 * (t % PT) + i32) * N + 32 * (t / PT) + 4 * hf;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                *reinterpret_cast<float4*>(out + 8 * k) =
                    make_float4(acc[q][4 * k], acc[q][4 * k + 1], acc[q][4 * k + 2], acc[q][4 * k + 3]);
        }
    }
}

// ------------------------------------------------------------ host side --
static int f_pblock(const SsdF32Params& p) { return p.P % 64 == 0 ? 64 : 32; }

bool ssd_f32_plan(SsdF32Params* q) {
    SsdF32Params& p = *q;
    if (p.P % 32 != 0 || p.P > 256 || (p.N != 32 && p.N != 64 && p.N != 128)) return false;
    // a step's ranks lie in one 32-row tile: its own-step block is on the diagonal
    if (p.M < 1 || p.M > 32 || (p.M & (p.M - 1)) != 0) return false;
    // rows move as four values: 16 bytes of f32, 8 of bf16
    const uintptr_t al = p.io_dtype == MAMBA_BF16 ? 7u : 15u;
    for (const void* ptr : {p.v, p.Bm, p.Cm, (const void*)p.y})
        if (((uintptr_t)ptr & al) != 0) return false;
    for (const void* ptr : {(const void*)p.h0, (const void*)p.init_hpr, (const void*)p.hT})
        if (((uintptr_t)ptr & 15u) != 0) return false;
    for (int64_t s : {p.v_sb, p.v_sl, p.v_sm, p.v_sh, p.B_sb, p.B_sl, p.B_sm, p.B_sg, p.C_sb, p.C_sl, p.C_sm, p.C_sg,
                      p.y_sb, p.y_sl, p.y_sm, p.y_sh})
        if (s % 4 != 0) return false;
    p.mshift = __builtin_ctz(p.M);
    const int64_t steps = kFR >> p.mshift;
    p.nch = (int)((p.L + steps - 1) / steps);
    // Segments per (batch, head, block): the scan takes rounds of 256 workgroups
    // (one per CU at dstate 64 and 128, by 75 to 143 KB of LDS and up to 240
    // registers; at dstate 32, 53 to 66 KB, two fit, which is not counted), each as
    // long as a segment's chunks plus the entry state; the state pass half a chunk's
    // time per chunk at two workgroups per CU and another launch (about half a
    // chunk's time).
    const int64_t units = (int64_t)p.nb * p.H * (p.P / f_pblock(p));
    double best = 0.;
    for (int n = 1; n <= std::min(p.nch, 64); ++n) {
        const int cps = (p.nch + n - 1) / n, S = (p.nch + cps - 1) / cps;
        const int64_t rounds = (units * S + 255) / 256, pass = (units * (S - 1) + 511) / 512;
        const double cost = (double)rounds * (cps + 1. + 0.1 * S) + (S > 1 ? (double)pass * (0.5 * cps + 0.5) + 0.5 : 0.);
        if (best == 0. || cost < best) {
            best = cost;
            p.S = S;
            p.cps = cps;
        }
    }
    return units * p.S < (1ll << 31);
}

size_t ssd_f32_workspace(const SsdF32Params& p) {
    if (p.S == 1) return 0;
    const size_t units = (size_t)p.nb * p.H * p.S;
    return align_up(units * p.P * p.N * sizeof(float), 256) +
           align_up(units * (p.P / f_pblock(p)) * sizeof(float), 256);
}

template <typename T, int PB, int N>
static int f_run(SsdF32Params p, void* ws, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
    const int units = p.nb * p.H * (p.P / PB);
    p.seg = static_cast<float*>(ws);
    p.segd = p.seg + (p.S == 1 ? 0 : align_up((size_t)p.nb * p.H * p.S * p.P * p.N * sizeof(float), 256) / sizeof(float));
    // dynamic LDS above the 64 KB default (up to the CU's 160 KB)
    constexpr size_t lds_scan = sizeof(FScanLds<PB, N>), lds_state = sizeof(FStateLds<PB, N>);
    static_assert(lds_scan <= 160 * 1024, "LDS of a CU");
    MAMBA_CHECK_HIP(hipFuncSetAttribute((const void*)ssd_f32_scan<T, PB, N>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)lds_scan));
    if (p.S > 1) {
        hipLaunchKernelGGL((ssd_f32_state<T, PB, N>), dim3(units * (p.S - 1)), dim3(256), lds_state, stream, p);
        MAMBA_CHECK_LAUNCH();
    }
    if (ev0) MAMBA_CHECK_HIP(hipEventRecord(ev0, stream));
    hipLaunchKernelGGL((ssd_f32_scan<T, PB, N>), dim3(units * p.S), dim3(512), lds_scan, stream, p);
    MAMBA_CHECK_LAUNCH();
    if (ev1) MAMBA_CHECK_HIP(hipEventRecord(ev1, stream));
    return MAMBA_OK;
}

template <typename T, int PB>
static int f_run_n(const SsdF32Params& p, void* ws, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
    return p.N == 128  ? f_run<T, PB, 128>(p, ws, stream, ev0, ev1)
           : p.N == 64 ? f_run<T, PB, 64>(p, ws, stream, ev0, ev1)
                       : f_run<T, PB, 32>(p, ws, stream, ev0, ev1);
}

int ssd_f32_launch(const SsdF32Params& p, void* ws, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
    const bool wide = f_pblock(p) == 64;
    if (p.io_dtype == MAMBA_BF16)
        return wide ? f_run_n<bf16_t, 64>(p, ws, stream, ev0, ev1) : f_run_n<bf16_t, 32>(p, ws, stream, ev0, ev1);
    return wide ? f_run_n<float, 64>(p, ws, stream, ev0, ev1) : f_run_n<float, 32>(p, ws, stream, ev0, ev1);
}

}  // namespace mamba
