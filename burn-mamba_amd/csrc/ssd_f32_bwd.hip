// SSD backward with every product on f32 MFMA, split over sequence segments:
// headdim 64, dstate 64 or 128, f32 arithmetic, f32 or bf16 inputs.
//
// Reference: the Autodiff arms of Mamba2BackendExt::ssd_serial_recalculated
// (src/mamba2/ssd/serial_recalculated/backward.rs:29-321, gradient math
// combined_backward.rs:126-593), of Mamba3SingleSsdBackendExt::single_ssd_serial_
// recalculated (src/mamba3/single_ssd/ssd/serial_recalculated/backward.rs:27-299)
// and of the double-SSD one (double_ssd/ssd/serial_recalculated/backward.rs:27-275).
// All are the backward of ssd_f32.hip's recurrence on fused (step, rank) rows:
// with cs the cumulative log-decay in the chunk, a_j = exp(cs_end - cs_j),
// b_i = exp(cs_i), w_j = sc_j a_j, h the state entering the chunk, g the
// gradient of the state leaving it and
//   W_ij = e_ij sc_j, e_ij = exp(cs_i - cs_j)  (earlier step), gm_i (own step), 0 (later),
//   CB_ij = C_i . B_j,   DV_ij = dy_i . v_j,   T_ij = W_ij CB_ij DV_ij over earlier steps,
//   xu_j = v_j . g B_j,  uh_i = C_i . h^T dy_i
// the gradients are
//   dv_j = w_j g B_j + sum_i (W CB)_ij dy_i  (+ D dy_j)
//   dB_j = w_j g^T v_j + sum_i (W DV)_ij C_i,  dC_i = b_i h^T dy_i + sum_j (W DV)_ij B_j
//   dsc_t = sum over the step's rows j of  sum_i e_ij CB_ij DV_ij + a_j xu_j
//   dgm_t = sum over the step's own pairs of CB_ij DV_ij
//   dda_t = exp(cs_end) <g, h> + sum_{j before t} w_j xu_j + sum_{i from t on} b_i uh_i
//         + sum_{j before t} sum_i T_ij - sum_{i before t} sum_j T_ij
//   g <- exp(cs_end) g + sum_i b_i C_i (x) dy_i.
// Mamba-2: ddt = A dda + dsc + dgm, dA = sum dt dda, dD = sum DV_jj.
//
// Three launches (two when a (batch, head) is not split, one for 32 rows or fewer):
//   1. ssd_f32_bwd_seg: the states of all segments but the last from zero, and
//      the state gradients of all but the first.
//   2. ssd_f32_bwd_states (more than 32 rows): from its entry state, each segment's chunk-entry
//      states, written for the next launch.
//   3. ssd_f32_bwd_chunks: each segment's chunks in reverse, 8 waves with fixed
//      roles; g stays in registers in both layouts that the products take it in
//      ([n][p] on waves 0, 1, 6, 7, [p][n] on waves 2-5), so that each enters its MFMA
//      straight from the accumulators and LDS holds only the chunk's rows:
//        phase A  w0, 1, 6, 7: g B and xu (32 columns of p, half of n; the
//                 halves meet in LDS), and a 32 x 32 tile of CB and DV with W
//                 and T's row and column sums on w0, 6, 7;
//                 w2-5: g^T v, h^T dy, uh and <g, h> (32 columns of n each; at
//                 dstate 64 two waves share them, a row tile each)
//        phase B  w0, 1, 6, 7: dv, g; w2-5: dB, dC, g; w7: the per-step
//                 gradients.
// What bounds it: the f32 MFMA rate (157 TFLOP/s) and, close behind, HBM (inputs
// read three times, the entry states written and read, dB / dC per head).
// 64-row chunks halve the entry states and the barriers against 32-row ones.
// Sums over rows whose weights fall with the row (g, dv, dB) run from the last
// row: a term rounds at the size of the sum it meets, so the small ones go first.
// Measured: the backward at 2 x 4096 steps, 32 heads 64 x 128, rank 4, 5.6 ms ->
// 2.3 ms (reverse loop 4.53 -> 1.62 ms)
// against one workgroup per (batch, head, half of dstate) on
// 32-row chunks, which it replaces; at 2 x 2048, 80 heads, rank 1, 0.98 -> 0.82
// ms; and at dstate 64 (1 x 1024, 24 heads), where the SIMT kernels ran, 7.6 ms
// -> 0.08 ms.
// T: bf16 rows are widened on their way into LDS (the same values as an f32 copy,
// half the bytes of three passes, and no spills in the reverse loop): a bf16
// forward and backward at 2 x 2048, 80 heads, rank 1 943 -> 880 us with the four
// conversion launches gone.
#include <algorithm>
#include <type_traits>

#include "ssd_f32_bwd.h"
#include "ssd_f32_rows.h"

namespace mamba {

constexpr int kBP = 64;          // headdim
constexpr int kBVP = kBP + 4;    // pitch of v and dy rows and of the pair matrices

// acc += A B over 8 values of k: A is four accumulator registers (an operand
// that a product left in MFMA layout), B four consecutive values of a row
__device__ __forceinline__ bwd_f32x16 fb_acc4(const bwd_f32x16& g, int r0, float4 x, bwd_f32x16 acc) {
    acc = bwd_mfma(g[r0], x.x, acc);
    acc = bwd_mfma(g[r0 + 1], x.y, acc);
    acc = bwd_mfma(g[r0 + 2], x.z, acc);
    return bwd_mfma(g[r0 + 3], x.w, acc);
}
__device__ __forceinline__ bwd_f32x16 fb_row4(float4 a, float4 x, bwd_f32x16 acc) {
    acc = bwd_mfma(a.x, x.x, acc);
    acc = bwd_mfma(a.y, x.y, acc);
    acc = bwd_mfma(a.z, x.z, acc);
    return bwd_mfma(a.w, x.w, acc);
}
__device__ __forceinline__ float4 fb_ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
// one tile's column to a row of an output: four consecutive values per register
// quad, rows 8 apart; vec: the outputs are 16-byte aligned
__device__ __forceinline__ void fb_put(float* o, bool vec, const bwd_f32x16& a) {
    if (vec) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(o + 8 * q) = make_float4(a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]);
    } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) o[8 * (r >> 2) + (r & 3)] = a[r];
    }
}
__device__ __forceinline__ bwd_f32x16 fb_zero() {
    bwd_f32x16 z;
#pragma unroll
    for (int r = 0; r < 16; ++r) z[r] = 0.f;
    return z;
}

// bounds how far operand loads are moved ahead of their MFMAs (registers)
__device__ __forceinline__ void fb_fence() { __builtin_amdgcn_sched_barrier(0); }

struct FBJob {
    int b, h, grp, s, c0, c1;
    int64_t bh;
};
__device__ __forceinline__ FBJob fb_job(const SsdF32BwdParams& p, int u, int s) {
    FBJob j;
    j.s = s;
    j.bh = u;
    j.h = u % p.H;
    j.b = u / p.H;
    j.grp = j.h / (p.H / p.G);
    j.c0 = s * p.cps;
    j.c1 = min(p.nch, j.c0 + p.cps);
    return j;
}

// log-decay and weights of one fused row (lane) of chunk c; zero past the end
struct FBTab {
    float da, gm, sc;
};
__device__ __forceinline__ FBTab fb_tab(const SsdF32BwdParams& p, const FBJob& j, int c, int lane) {
    const int t0 = c * (kFR >> p.mshift) + (lane >> p.mshift), t = min(t0, p.L - 1);
    FBTab r;
    r.da = p.da[(int64_t)j.b * p.da_sb + (int64_t)t * p.da_sl + (int64_t)j.h * p.da_sh];
    r.gm = p.gm ? p.gm[(int64_t)j.b * p.gm_sb + (int64_t)t * p.gm_sl + (int64_t)j.h * p.gm_sh] : 1.f;
    r.sc = p.sc ? p.sc[(int64_t)j.b * p.sc_sb + (int64_t)t * p.sc_sl + (int64_t)j.h * p.sc_sh] : 1.f;
    if (t0 >= p.L) r.da = r.gm = r.sc = 0.f;
    return r;
}
// a step's decay counts once, at its first rank
__device__ __forceinline__ FDecay fb_decay(const SsdF32BwdParams& p, const FBTab& r, float A, int lane) {
    return f_decay((lane & (p.M - 1)) == 0 ? (double)r.da * A : 0.);
}

// The state entering segment s as [n][p] tiles (columns p on lanes), or as
// [p][n] tiles (columns n): four consecutive values of the row axis per load.
// Horner over the earlier segments (h), or over the later ones (g).  Of several
// segments the first launch alone reads d(final state), and copies it into the
// place of segment 0, which has no gradient of its own there: d(initial state),
// written by the last launch, may be the same memory.
template <int N, bool PN>
__device__ __forceinline__ void fb_entry(const SsdF32BwdParams& p, const FBJob& j, bool grad, int pt, int nt, int i32,
                                         int hf, bwd_f32x16& a) {
    const float* h0 = grad ? p.dfin : p.h0;
    const float* seg = grad ? p.gs : p.fs;
    const float* dec = grad ? p.gd : p.fd;
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = 0.f;
    // h0 and dfin are [p][n]; segments [n][p]
    const int lp = 32 * pt + (PN ? 4 * hf : i32), ln = 32 * nt + (PN ? i32 : 4 * hf);
    if (h0) {
        const float* q = (grad && p.S > 1 ? p.gs + j.bh * p.S * (kBP * N) : h0 + j.bh * (kBP * N)) + lp * N + ln;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int k = 8 * (r >> 2) + (r & 3);
            a[r] = q[PN ? k * N : k];
        }
    }
    const int n = grad ? p.S - 1 - j.s : j.s;
    for (int k = 0; k < n; ++k) {
        const int u = grad ? p.S - 1 - k : k;
        const float d = f_exp(dec[j.bh * p.S + u]);
        const float* q = seg + (j.bh * p.S + u) * (kBP * N) + ln * kBP + lp;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int e = 8 * (r >> 2) + (r & 3);
            a[r] = __builtin_fmaf(a[r], d, q[PN ? e : e * kBP]);
        }
    }
}

template <int N>
struct FBSegLds {
    float R[kFR * (N + 4)];   // B or C rows
    float X[kFR * kBVP];      // v or dy rows
    float w[kFR];
    float dec, end;
};

// One workgroup per (batch, head, segment, direction): blocks of direction 0
// form the state of segments 0 .. S - 2 from zero, those of direction 1 the
// state gradient that segments 1 .. S - 1 hand to the left, from zero.
template <int N, typename T>
__global__ __launch_bounds__(256, 3) void ssd_f32_bwd_seg(SsdF32BwdParams p) {
    __shared__ __align__(16) FBSegLds<N> S;
    constexpr int TILES = 2 * (N / 32), QT = TILES / 4, NT = 256;
    const int tid = threadIdx.x, wv = wave_id(), lane = tid & 63, i32 = lane & 31, hf = lane >> 5;
    const bool rev = blockIdx.x & 1;
    const int flip = rev ? kFR - 1 : 0;
    const int idx = blockIdx.x >> 1, u = idx / (p.S - 1), s0 = idx % (p.S - 1);
    const FBJob j = fb_job(p, u, rev ? s0 + 1 : s0);
    const T* xb = static_cast<const T*>(rev ? p.dy : p.v) +
                  (rev ? (int64_t)j.b * p.dy_sb + (int64_t)j.h * p.dy_sh : (int64_t)j.b * p.v_sb + (int64_t)j.h * p.v_sh);
    const T* rb = static_cast<const T*>(rev ? p.C : p.B) +
                  (rev ? (int64_t)j.b * p.C_sb + (int64_t)j.grp * p.C_sg : (int64_t)j.b * p.B_sb + (int64_t)j.grp * p.B_sg);
    const int64_t xsl = rev ? p.dy_sl : p.v_sl, xsm = rev ? p.dy_sm : p.v_sm;
    const int64_t rsl = rev ? p.C_sl : p.B_sl, rsm = rev ? p.C_sm : p.B_sm;
    const float A = p.A ? p.A[j.h] : 1.f;
    FRaw<T> rr[kFR * N / 4 / NT], rx[kFR * kBP / 4 / NT];
    FBTab rt = {0.f, 0.f, 0.f};
    bwd_f32x16 acc[QT];
#pragma unroll
    for (int q = 0; q < QT; ++q) acc[q] = fb_zero();
    auto fetch = [&](int c) {
        f_fetch<T, N, NT>(rr, rb, rsl, rsm, p.L, p.mshift, c, tid);
        f_fetch<T, kBP, NT>(rx, xb, xsl, xsm, p.L, p.mshift, c, tid);
        if (wv == 0) rt = fb_tab(p, j, c, lane);
    };
    auto commit = [&](int c) {
        f_commit<T, N, NT, N + 4>(rr, S.R, p.L, p.mshift, c, tid, flip);
        f_commit<T, kBP, NT, kBVP>(rx, S.X, p.L, p.mshift, c, tid, flip);
        if (wv == 0) {
            const FDecay d = fb_decay(p, rt, A, lane);
            S.w[lane ^ flip] = rev ? d.b : d.a * rt.sc;
            if (lane == 63) {
                S.dec = d.b;
                S.end = d.end;
            }
        }
    };
    const int nc = j.c1 - j.c0;
    auto at = [&](int k) { return rev ? j.c1 - 1 - k : j.c0 + k; };
    fetch(at(0));
    if (rev && j.s == p.S - 1 && p.dfin) {
        const float* in = p.dfin + j.bh * (kBP * N) + tid;
        float* to = p.gs + j.bh * p.S * (kBP * N) + tid;
        float v[kBP * N / NT];
#pragma unroll
        for (int e = 0; e < kBP * N / NT; ++e) v[e] = in[e * NT];
        commit(at(0));
#pragma unroll
        for (int e = 0; e < kBP * N / NT; ++e) to[e * NT] = v[e];
    } else {
        commit(at(0));
    }
    __syncthreads();
    float total = 0.f;
    for (int k = 0; k < nc; ++k) {
        if (k + 1 < nc) fetch(at(k + 1));
        total += S.end;
        f_update<kBP, N, QT, kBVP>(acc, S.R, S.X, S.w, S.dec, wv, i32, hf);
        __syncthreads();
        if (k + 1 < nc) commit(at(k + 1));
        __syncthreads();
    }
    float* out = (rev ? p.gs : p.fs) + (j.bh * p.S + j.s) * (kBP * N);
#pragma unroll
    for (int q = 0; q < QT; ++q) {
        const int t = wv + 4 * q;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            out[(32 * (t >> 1) + bwd_row(r, hf)) * kBP + 32 * (t & 1) + i32] = acc[q][r];
    }
    if (tid == 0) (rev ? p.gd : p.fd)[j.bh * p.S + j.s] = total;
}

// The chunk-entry states of one segment, as [p][n] tiles (pt + 2 nt) in
// accumulator order: hs[(b h, chunk)][tile][r][lane].
template <int N, typename T>
__global__ __launch_bounds__(256, 3) void ssd_f32_bwd_states(SsdF32BwdParams p) {
    __shared__ __align__(16) FBSegLds<N> S;
    constexpr int TILES = 2 * (N / 32), QT = TILES / 4, NT = 256, NP = N + 4;
    const int tid = threadIdx.x, wv = wave_id(), lane = tid & 63, i32 = lane & 31, hf = lane >> 5;
    const FBJob j = fb_job(p, blockIdx.x / p.S, blockIdx.x % p.S);
    const T* vb = static_cast<const T*>(p.v) + (int64_t)j.b * p.v_sb + (int64_t)j.h * p.v_sh;
    const T* Bb = static_cast<const T*>(p.B) + (int64_t)j.b * p.B_sb + (int64_t)j.grp * p.B_sg;
    const float A = p.A ? p.A[j.h] : 1.f;
    FRaw<T> rr[kFR * N / 4 / NT], rx[kFR * kBP / 4 / NT];
    FBTab rt = {0.f, 0.f, 0.f};
    bwd_f32x16 acc[QT];
    auto fetch = [&](int c) {
        f_fetch<T, N, NT>(rr, Bb, p.B_sl, p.B_sm, p.L, p.mshift, c, tid);
        f_fetch<T, kBP, NT>(rx, vb, p.v_sl, p.v_sm, p.L, p.mshift, c, tid);
        if (wv == 0) rt = fb_tab(p, j, c, lane);
    };
    auto commit = [&](int c) {
        f_commit<T, N, NT, NP>(rr, S.R, p.L, p.mshift, c, tid);
        f_commit<T, kBP, NT, kBVP>(rx, S.X, p.L, p.mshift, c, tid);
        if (wv == 0) {
            const FDecay d = fb_decay(p, rt, A, lane);
            S.w[lane] = d.a * rt.sc;
            if (lane == 63) S.dec = d.b;
        }
    };
    fetch(j.c0);
#pragma unroll
    for (int q = 0; q < QT; ++q) fb_entry<N, true>(p, j, false, wv & 1, (wv >> 1) + 2 * q, i32, hf, acc[q]);
    commit(j.c0);
    __syncthreads();
    for (int c = j.c0; c < j.c1; ++c) {
        if (c + 1 < j.c1) fetch(c + 1);
        float* dst = p.hs + ((j.bh * p.nch + c) * TILES + wv) * 1024 + lane;
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int r = 0; r < 16; ++r) dst[q * 4096 + r * 64] = acc[q][r];
        if (c + 1 < j.c1) {
            const float dec = S.dec;
#pragma unroll
            for (int q = 0; q < QT; ++q)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[q][r] *= dec;
            // h[p][n] += sum_j (w_j v[j][p]) B[j][n]
            const float* Ap = S.X + 4 * hf * kBVP + 32 * (wv & 1) + i32;
            const float* Bp = S.R + 4 * hf * NP + 32 * (wv >> 1) + i32;
#pragma unroll
            for (int s = 0; s < kFR / 8; ++s) {
                const float4 w = fb_ld4(&S.w[8 * s + 4 * hf]);
                const float wj[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float a = wj[k] * Ap[(8 * s + k) * kBVP];
#pragma unroll
                    for (int q = 0; q < QT; ++q) acc[q] = bwd_mfma(a, Bp[(8 * s + k) * NP + 64 * q], acc[q]);
                }
                if (s & 1) fb_fence();
            }
            __syncthreads();
            commit(c + 1);
            __syncthreads();
        }
    }
}

template <int N>
struct FBLds {
    float B[kFR * (N + 4)];
    float C[kFR * (N + 4)];
    float V[kFR * kBVP];
    float Y[kFR * kBVP];      // dy
    float E1[kFR * kBVP];     // [i][j] W CB
    float E2[kFR * kBVP];     // [i][j] W DV
    float cs[kFR], lo[kFR], gm[kFR], sc[kFR], av[kFR], bv[kFR], w[kFR];
    float zero[32];           // read for dy where there is no D: 0 dy of an infinite dy would be NaN
    float P[4][16 * 64];      // [pt, nh] its share of g B for the other row tile, accumulator order
    float xu[4][kFR];         // v_j . g B_j over 32 columns of p and half of n
    float uh[4][kFR];         // C_i . h^T dy_i over 32 columns of n
    float xg[2][kFR];         // [row tile][j] sum over its rows i of e_ij CB_ij DV_ij
    float rowm[2][kFR];       // [column tile][i] sum over its columns j of T_ij
    float dg[kFR];            // sum over the own step's j of CB_ij DV_ij
    float dxd[kFR];           // DV_jj
    float ghc[4];             // <g, h> over 32 columns of n
    float dec;
};

// What the last chunk's rows are.  A second row tile of zeros is left out (the sums
// are the same): in kernels of their own, as the loop is 1 to 3 % slower with it.
//   FB_FULL  anything
//   FB_ONE   a sequence of one chunk of at most 32 rows: no other, and its entry state
//            is the initial one, no states launch
//   FB_TAIL  two to four chunks in one segment, the last of at most 32 rows
// us against 32-row chunks and FB_FULL, dstate 128, f32: 12 heads, 16 positions 25.1 /
// 34.7 / 22.8; 256 (batch, head), 16 positions 39.3 / 47.0 / 33.5, 90 66.1 / 77.3 / 72.5, 140
// 93.0 / 105.9 / 101.  In several segments the last one's end is no earlier for it.
enum FBRows { FB_FULL, FB_ONE, FB_TAIL };
template <int N, typename T, FBRows R>
__global__ __launch_bounds__(512, 2) void ssd_f32_bwd_chunks(SsdF32BwdParams p) {
    extern __shared__ __align__(16) char fb_smem[];
    FBLds<N>& S = *reinterpret_cast<FBLds<N>*>(fb_smem);
    constexpr int NTN = N / 32, TILES = 2 * NTN, NT = 512, NP = N + 4;
    constexpr bool ONE = R == FB_ONE;
    constexpr int XT = N == 128 && !ONE ? 2 : 1;      // row tiles of dB and dC per wave
    const int tid = threadIdx.x, wv = wave_id(), lane = tid & 63, i32 = lane & 31, hf = lane >> 5;
    const FBJob j = fb_job(p, blockIdx.x / p.S, blockIdx.x % p.S);
    const T* vb = static_cast<const T*>(p.v) + (int64_t)j.b * p.v_sb + (int64_t)j.h * p.v_sh;
    const T* yb = static_cast<const T*>(p.dy) + (int64_t)j.b * p.dy_sb + (int64_t)j.h * p.dy_sh;
    const T* Bb = static_cast<const T*>(p.B) + (int64_t)j.b * p.B_sb + (int64_t)j.grp * p.B_sg;
    const T* Cb = static_cast<const T*>(p.C) + (int64_t)j.b * p.C_sb + (int64_t)j.grp * p.C_sg;
    const float A = p.A ? p.A[j.h] : 1.f;
    const float D = p.D ? p.D[j.h] : 0.f;
    const int ms = p.mshift, steps = kFR >> ms;
    const int pt = wv & 1;                                  // waves 0, 1, 6, 7
    const int nt = N == 128 ? wv - 2 : (wv - 2) & 1;        // waves 2-5
    const int own = N == 128 ? 0 : (wv - 2) >> 1;
    FRaw<T> rB[kFR * N / 4 / NT], rC[kFR * N / 4 / NT], rv[kFR * kBP / 4 / NT], ry[kFR * kBP / 4 / NT];
    FBTab rt = {0.f, 0.f, 0.f};
    FDecay rd = {0.f, 0.f, 0.f, 0.f, 0.f};
    auto fetch = [&](int c, int tid) {
        f_fetch<T, N, NT>(rB, Bb, p.B_sl, p.B_sm, p.L, ms, c, tid);
        f_fetch<T, N, NT>(rC, Cb, p.C_sl, p.C_sm, p.L, ms, c, tid);
        f_fetch<T, kBP, NT>(rv, vb, p.v_sl, p.v_sm, p.L, ms, c, tid);
        f_fetch<T, kBP, NT>(ry, yb, p.dy_sl, p.dy_sm, p.L, ms, c, tid);
        if (wv == 1) rt = fb_tab(p, j, c, tid & 63);
    };
    auto commit = [&](int c, int tid) {
        const int lane = tid & 63;
        f_commit<T, N, NT, NP>(rB, S.B, p.L, ms, c, tid);
        f_commit<T, N, NT, NP>(rC, S.C, p.L, ms, c, tid);
        f_commit<T, kBP, NT, kBVP>(rv, S.V, p.L, ms, c, tid);
        f_commit<T, kBP, NT, kBVP>(ry, S.Y, p.L, ms, c, tid);
        if (wv == 1) {
            S.cs[lane] = rd.cs;
            S.lo[lane] = rd.lo;
            S.gm[lane] = rt.gm;
            S.sc[lane] = rt.sc;
            S.av[lane] = rd.a;
            S.bv[lane] = rd.b;
            S.w[lane] = rd.a * rt.sc;
            if (lane == 63) S.dec = rd.b;
        }
    };
    // Each role runs its own loop over the chunks, with the same barriers (A |
    // B | commit |), so that no wave holds another role's accumulators.
    fetch(j.c1 - 1, tid);
    if (wv == 1) rd = fb_decay(p, rt, A, lane);
    if (tid < 32) S.zero[tid] = 0.f;
    if (wv < 2 || wv >= 6) {
        // 32 columns of p (pt) and half of n (nh): its share of g B for both row
        // tiles, a pair tile, then dv of row tile nh
        constexpr int GT = NTN / 2;
        const int nh = wv >= 6;
        bwd_f32x16 G[GT], acc[2];  // g[n][p] tiles (GT nh + k, pt); w g B as [p][j]
        float accA = 0.f, accD = 0.f;
#pragma unroll
        for (int k = 0; k < GT; ++k) fb_entry<N, false>(p, j, true, pt, GT * nh + k, i32, hf, G[k]);
        commit(j.c1 - 1, tid);
        __syncthreads();
        for (int c = j.c1 - 1; c >= j.c0; --c) {
            const int t0 = c * steps;
            const int RT = ONE || (R == FB_TAIL && c == p.nch - 1) ? 1 : 2, KS = 4 * RT;  // row tiles, groups of eight rows
            int tid = threadIdx.x;  // opaque per chunk: addresses and lane masks are formed in the loop
            asm volatile("" : "+v"(tid));
            const int lane = tid & 63, i32 = lane & 31, hf = lane >> 5;
            if (c > j.c0) fetch(c - 1, tid);
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                if (x >= RT) break;
                const int row = 32 * x + i32;
                const float* Bp = S.B + row * NP + 32 * GT * nh + 4 * hf;
                bwd_f32x16 a = fb_zero();
#pragma unroll
                for (int k = 0; k < GT; ++k) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) a = fb_acc4(G[k], 4 * q, fb_ld4(Bp + 32 * k + 8 * q), a);
                    fb_fence();
                }
                const float* vr = S.V + row * kBVP + 32 * pt + 4 * hf;
                float s = 0.f;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 v = fb_ld4(vr + 8 * q);
                    s += a[4 * q] * v.x + a[4 * q + 1] * v.y + a[4 * q + 2] * v.z + a[4 * q + 3] * v.w;
                }
                s += __shfl_xor(s, 32, 64);
                if (hf == 0) S.xu[2 * pt + nh][row] = s;
                const float w = S.w[row];
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[x][r] = a[r] * w;
            }
            if (RT == 2 || nh) {
                // the other row tile's share goes to its wave
                float* out = S.P[2 * pt + nh] + lane;
#pragma unroll
                for (int r = 0; r < 16; ++r) out[64 * r] = nh ? acc[0][r] : acc[1][r];
            }
            // pair tile (it, jt): CB and DV as [i][j] (columns j on lanes), weighted
            auto tile = [&](auto diag, int it, int jt) {
                constexpr bool DIAG = decltype(diag)::value;
                const float* Ac = S.C + (32 * it + i32) * NP + 4 * hf;
                const float* Bc = S.B + (32 * jt + i32) * NP + 4 * hf;
                const float* Ay = S.Y + (32 * it + i32) * kBVP + 4 * hf;
                const float* Bv = S.V + (32 * jt + i32) * kBVP + 4 * hf;
                const int jj = 32 * jt + i32, sj = jj >> ms, row0 = 32 * it + 4 * hf;
                float* e1 = S.E1 + row0 * kBVP + jj;
                float* e2 = S.E2 + row0 * kBVP + jj;
                bwd_f32x16 cb = fb_zero(), dx = fb_zero();
#pragma unroll
                for (int s = 0; s < N / 8; ++s) {
                    cb = fb_row4(fb_ld4(Ac + 8 * s), fb_ld4(Bc + 8 * s), cb);
                    if ((s & 3) == 3) fb_fence();
                    if (s == 7 && N == 128) {
                        // two sums of 64 products instead of one of 128; the first
                        // waits where the lane's W CB will go
#pragma unroll
                        for (int r = 0; r < 16; ++r) e1[(8 * (r >> 2) + (r & 3)) * kBVP] = cb[r];
                        cb = fb_zero();
                    }
                }
#pragma unroll
                for (int s = 0; s < kBP / 8; ++s) {
                    dx = fb_row4(fb_ld4(Ay + 8 * s), fb_ld4(Bv + 8 * s), dx);
                    if ((s & 3) == 3) fb_fence();
                }
                const float csj = S.cs[jj], loj = S.lo[jj], scj = S.sc[jj];
                float rl[16], rs[16], xg = 0.f, dd = 0.f;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 c4 = fb_ld4(&S.cs[row0 + 8 * q]), l4 = fb_ld4(&S.lo[row0 + 8 * q]);
                    const float4 g4 = fb_ld4(&S.gm[row0 + 8 * q]);
                    const float d[4] = {(c4.x - csj) + (l4.x - loj), (c4.y - csj) + (l4.y - loj),
                                        (c4.z - csj) + (l4.z - loj), (c4.w - csj) + (l4.w - loj)};
                    const float gi[4] = {g4.x, g4.y, g4.z, g4.w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int r = 4 * q + k;
                        if constexpr (N == 128) cb[r] += e1[(8 * q + k) * kBVP];
                        const float t = cb[r] * dx[r];
                        float e, W;
                        if constexpr (DIAG) {
                            // i's step against j's: later, own, earlier (selects: a
                            // dropped pair's values never enter a sum)
                            const int si = (row0 + 8 * q + k) >> ms;
                            const bool lower = si > sj, same = si == sj;
                            e = f_exp(lower ? d[k] : 0.f);
                            W = lower ? e * scj : gi[k];
                            rl[r] = lower ? W * t : 0.f;
                            rs[r] = same ? t : 0.f;
                            xg += lower ? e * t : 0.f;
                            dd = 4 * hf + 8 * q + k == i32 ? dx[r] : dd;
                            e1[(8 * q + k) * kBVP] = lower || same ? W * cb[r] : 0.f;
                            e2[(8 * q + k) * kBVP] = lower || same ? W * dx[r] : 0.f;
                        } else {
                            e = f_exp(d[k]);
                            W = e * scj;
                            rl[r] = W * t;
                            xg = __builtin_fmaf(e, t, xg);
                            e1[(8 * q + k) * kBVP] = W * cb[r];
                            e2[(8 * q + k) * kBVP] = W * dx[r];
                        }
                    }
                    fb_fence();
                }
                xg += __shfl_xor(xg, 32, 64);
                if (hf == 0) S.xg[it][jj] = xg;
                const int ri = 32 * it + bwd_row(i32 >> 1, hf);
                const float rsum = bwd_half_sum16(rl, i32);
                if ((i32 & 1) == 0) S.rowm[jt][ri] = rsum;
                if constexpr (DIAG) {
                    const float ssum = bwd_half_sum16(rs, i32);
                    if ((i32 & 1) == 0) S.dg[ri] = ssum;
                    if (((i32 >> 2) & 1) == hf) S.dxd[jj] = dd;
                }
            };
            if (wv == 0)
                tile(std::true_type{}, 0, 0);
            else if (RT == 2 && wv == 6)
                tile(std::false_type{}, 1, 0);
            else if (RT == 2 && wv == 7)
                tile(std::true_type{}, 1, 1);
            else if ((RT == 2 || wv == 1) && c > j.c0)  // wave 1 has no pair tile: the next chunk's decays
                rd = fb_decay(p, rt, A, lane);
            __syncthreads();
            if (RT == 2 || !nh) {
                const float* in = S.P[2 * pt + 1 - nh] + lane;
                bwd_f32x16 a;
#pragma unroll
                for (int r = 0; r < 16; ++r) a[r] = (nh ? acc[1][r] : acc[0][r]) + in[64 * r];
                const float* Ap = S.Y + 4 * hf * kBVP + 32 * pt + i32;
                const float* Bp = S.E1 + 4 * hf * kBVP + 32 * nh + i32;
#pragma unroll
                for (int s = 7; s >= 0; --s)
                    if (s < KS && s >= 4 * nh) {
#pragma unroll
                        for (int k = 3; k >= 0; --k) a = bwd_mfma(Ap[(8 * s + k) * kBVP], Bp[(8 * s + k) * kBVP], a);
                        if ((s & 1) == 0) fb_fence();
                    }
                const int row = 32 * nh + i32, t = t0 + (row >> ms);
                if (t < p.L) {
                    float* out = p.dv + ((((int64_t)j.b * p.L + t) * p.M + (row & (p.M - 1))) * p.H + j.h) * kBP +
                                 32 * pt + 4 * hf;
                    const float* yr = p.D ? S.Y + row * kBVP + 32 * pt + 4 * hf : S.zero + 4 * hf;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float4 y = fb_ld4(yr + 8 * q);
                        a[4 * q] = __builtin_fmaf(D, y.x, a[4 * q]);
                        a[4 * q + 1] = __builtin_fmaf(D, y.y, a[4 * q + 1]);
                        a[4 * q + 2] = __builtin_fmaf(D, y.z, a[4 * q + 2]);
                        a[4 * q + 3] = __builtin_fmaf(D, y.w, a[4 * q + 3]);
                    }
                    fb_put(out, p.vec, a);
                }
            }
            if (c > j.c0 || j.s == 0) {  // past the first chunk it is the gradient of h0
                const float dec = S.dec;
#pragma unroll
                for (int k = 0; k < GT; ++k)
#pragma unroll
                    for (int r = 0; r < 16; ++r) G[k][r] *= dec;
                const float* Cp = S.C + 4 * hf * NP + 32 * GT * nh + i32;
                const float* Yp = S.Y + 4 * hf * kBVP + 32 * pt + i32;
#pragma unroll
                for (int s = 7; s >= 0; --s) {
                    if (s >= KS) continue;
                    const float4 b4 = fb_ld4(&S.bv[8 * s + 4 * hf]);
                    const float bi[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
                    for (int e = 3; e >= 0; --e) {
                        const float y = bi[e] * Yp[(8 * s + e) * kBVP];
#pragma unroll
                        for (int k = 0; k < GT; ++k) G[k] = bwd_mfma(Cp[(8 * s + e) * NP + 32 * k], y, G[k]);
                    }
                    if ((s & 1) == 0) fb_fence();
                }
            }
            if (wv == 7) {
            // lane = fused row; a step's results on its first rank's lane
            float xu = (S.xu[0][lane] + S.xu[1][lane]) + (S.xu[2][lane] + S.xu[3][lane]);
            float uh = 0.f, gh = 0.f;
#pragma unroll
            for (int k = 0; k < NTN; ++k) {
                uh += S.uh[k][lane];
                gh += S.ghc[k];
            }
            float xg = lane < 32 && RT == 2 ? S.xg[0][lane] + S.xg[1][lane] : S.xg[RT - 1][lane];
            if (RT == 1 && lane >= 32) xu = uh = xg = 0.f;  // never formed
            const float sc = S.sc[lane];
            const float z = S.w[lane] * xu, pz = wave_incl_scan(z) - z;
            // T's pairs j before t <= i: those of t's own 32-row tile as column
            // less row sums before t (a pair wholly before t cancels); those of
            // the tile below the diagonal one-sided, with nothing to cancel, as
            // columns before t or rows from t on.  One scan of 64 rows instead
            // left dA 1.4 times as far from 64 bits.
            const float d = RT == 2 ? sc * S.xg[lane >> 5][lane] - S.rowm[lane >> 5][lane]
                            : lane < 32 ? sc * xg - S.rowm[0][lane] : 0.f;
            const float pd = half_incl_scan(d) - d;
            const int rl = lane < 32 ? lane : 95 - lane;  // rows 32 .. 63 from the last
            float px = 0.f;
            if (RT == 2) {
                const float x = lane < 32 ? sc * S.xg[1][lane] : S.rowm[0][rl], sx = __shfl(half_incl_scan(x), rl, 64);
                px = lane < 32 ? sx - x : sx;
            }
            // suffix sums of b_i uh_i: the scan runs from the last lane
            const float su = __shfl(wave_incl_scan(__shfl(S.bv[lane] * uh, 63 - lane, 64)), 63 - lane, 64);
            const float dda = S.dec * gh + pz + su + (px + pd);
            float ds = xg + S.av[lane] * xu, dg = RT == 2 || lane < 32 ? S.dg[lane] : 0.f;
            for (int o = 1; o < p.M; o <<= 1) {
                ds += __shfl_xor(ds, o, 64);
                dg += __shfl_xor(dg, o, 64);
            }
            const int t = t0 + (lane >> ms);
            if (t < p.L && (lane & (p.M - 1)) == 0) {
                const int64_t o = ((int64_t)j.b * p.L + t) * p.H + j.h;
                p.dda[o] = p.A ? __builtin_fmaf(A, dda, ds + dg) : dda;
                if (p.dsc) p.dsc[o] = ds;
                if (p.dgm) p.dgm[o] = dg;
                accA += sc * dda;
                accD += S.dxd[lane];
            }
            }
            __syncthreads();
            if (c > j.c0) {
                commit(c - 1, tid);
                __syncthreads();
            }
        }
        // the first segment's g, past its first chunk, is the gradient of h0
        if (j.s == 0) {
#pragma unroll
            for (int k = 0; k < GT; ++k) {
                float* out = p.dh0 + j.bh * (kBP * N) + (32 * pt + i32) * N + 32 * (GT * nh + k) + 4 * hf;
                fb_put(out, p.vec, G[k]);
            }
        }
        if (p.pA && wv == 7) {
            const float sA = wave_sum(accA), sD = wave_sum(accD);
            if (lane == 0) {
                p.pA[j.bh * p.S + j.s] = sA;
                p.pD[j.bh * p.S + j.s] = sD;
            }
        }
    } else {
        bwd_f32x16 G[4], acc[4];  // g[p][n] tiles (0..1, nt), the entry state's; dB^T, dC^T (2 + x)
        auto fetch_h = [&](int c, int lane) {
            const float* src = p.hs + ((j.bh * p.nch + c) * TILES + 2 * nt) * 1024 + lane;
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int r = 0; r < 16; ++r) G[2 + k][r] = src[k * 1024 + r * 64];
        };
        if (!ONE)
            fetch_h(j.c1 - 1, lane);
        else  // one chunk: its entry state is the initial one
#pragma unroll
            for (int k = 0; k < 2; ++k) fb_entry<N, true>(p, j, false, k, nt, i32, hf, G[2 + k]);
#pragma unroll
        for (int k = 0; k < 2; ++k) fb_entry<N, true>(p, j, true, k, nt, i32, hf, G[k]);
        commit(j.c1 - 1, tid);
        __syncthreads();
        for (int c = j.c1 - 1; c >= j.c0; --c) {
            const int t0 = c * steps;
            const int RT = ONE || (R == FB_TAIL && c == p.nch - 1) ? 1 : 2, KS = 4 * RT;  // row tiles, groups of eight rows
            int tid = threadIdx.x;  // opaque per chunk: addresses and lane masks are formed in the loop
            asm volatile("" : "+v"(tid));
            const int lane = tid & 63, i32 = lane & 31, hf = lane >> 5;
#pragma unroll
            for (int x = 0; x < XT; ++x) {
                if (RT == 1 && (XT == 2 ? x : own)) break;
                const int row = 32 * (XT == 2 ? x : own) + i32;
                const float* Vp = S.V + row * kBVP + 4 * hf;
                const float* Yp = S.Y + row * kBVP + 4 * hf;
                acc[x] = fb_zero();
                acc[2 + x] = fb_zero();
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        acc[x] = fb_acc4(G[k], 4 * q, fb_ld4(Vp + 32 * k + 8 * q), acc[x]);
                        acc[2 + x] = fb_acc4(G[2 + k], 4 * q, fb_ld4(Yp + 32 * k + 8 * q), acc[2 + x]);
                        if (q & 1) fb_fence();
                    }
                fb_fence();
                const float* cr = S.C + row * NP + 32 * nt + 4 * hf;
                float s = 0.f;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 v = fb_ld4(cr + 8 * q);
                    s += acc[2 + x][4 * q] * v.x + acc[2 + x][4 * q + 1] * v.y + acc[2 + x][4 * q + 2] * v.z +
                         acc[2 + x][4 * q + 3] * v.w;
                }
                s += __shfl_xor(s, 32, 64);
                if (hf == 0) S.uh[nt][row] = s;
                fb_fence();
                const float w = S.w[row], bi = S.bv[row];
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[x][r] *= w;
                    acc[2 + x][r] *= bi;
                }
            }
            fb_fence();
            float gh = 0.f;
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int r = 0; r < 16; ++r) gh = __builtin_fmaf(G[k][r], G[2 + k][r], gh);
            gh = wave_sum_dpp(gh);
            if (lane == 0 && own == 0) S.ghc[nt] = gh;
            if (c > j.c0) fetch_h(c - 1, lane);
            __syncthreads();
#pragma unroll
            for (int x = 0; x < XT; ++x) {
                if (RT == 1 && (XT == 2 ? x : own)) break;
                const int xt = XT == 2 ? x : own, row = 32 * xt + i32;
                const float* Cp = S.C + 4 * hf * NP + 32 * nt + i32;
                const float* Ep = S.E2 + 4 * hf * kBVP + 32 * xt + i32;
#pragma unroll
                for (int s = 7; s >= 0; --s)
                    if (s < KS && s >= 4 * xt) {
#pragma unroll
                        for (int k = 3; k >= 0; --k)
                            acc[x] = bwd_mfma(Cp[(8 * s + k) * NP], Ep[(8 * s + k) * kBVP], acc[x]);
                        if ((s & 1) == 0) fb_fence();
                    }
                const float* Bp = S.B + 4 * hf * NP + 32 * nt + i32;
                const float* Er = S.E2 + row * kBVP + 4 * hf;
#pragma unroll
                for (int s = 0; s < 8; ++s)
                    if (s < 4 * xt + 4) {
                        const float4 e = fb_ld4(Er + 8 * s);
                        acc[2 + x] = bwd_mfma(Bp[(8 * s) * NP], e.x, acc[2 + x]);
                        acc[2 + x] = bwd_mfma(Bp[(8 * s + 1) * NP], e.y, acc[2 + x]);
                        acc[2 + x] = bwd_mfma(Bp[(8 * s + 2) * NP], e.z, acc[2 + x]);
                        acc[2 + x] = bwd_mfma(Bp[(8 * s + 3) * NP], e.w, acc[2 + x]);
                        if (s & 1) fb_fence();
                    }
                fb_fence();
                const int t = t0 + (row >> ms);
                if (t < p.L) {
                    const int64_t o = ((((int64_t)j.b * p.L + t) * p.M + (row & (p.M - 1))) * p.H + j.h) * N + 32 * nt +
                                      4 * hf;
                    fb_put(p.dBh + o, p.vec, acc[x]);
                    fb_put(p.dCh + o, p.vec, acc[2 + x]);
                }
            }
            fb_fence();
            if (c > j.c0) {
                fetch(c - 1, tid);  // only now: dB's and dC's registers are free
                fb_fence();
                const float dec = S.dec;
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int r = 0; r < 16; ++r) G[k][r] *= dec;
                const float* Cp = S.C + 4 * hf * NP + 32 * nt + i32;
                const float* Yp = S.Y + 4 * hf * kBVP + i32;
#pragma unroll
                for (int s = 7; s >= 0; --s) {
                    if (s >= KS) continue;
                    const float4 b4 = fb_ld4(&S.bv[8 * s + 4 * hf]);
                    const float bi[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
                    for (int e = 3; e >= 0; --e) {
                        const float cv = bi[e] * Cp[(8 * s + e) * NP];
#pragma unroll
                        for (int k = 0; k < 2; ++k) G[k] = bwd_mfma(Yp[(8 * s + e) * kBVP + 32 * k], cv, G[k]);
                    }
                    if ((s & 1) == 0) fb_fence();
                }
            }
            __syncthreads();
            if (c > j.c0) {
                commit(c - 1, tid);
                __syncthreads();
            }
        }
    }
}

// ------------------------------------------------------------ host side --
size_t ssd_f32_bwd_workspace(const SsdF32BwdParams& p) {
    const size_t units = (size_t)p.nb * p.H, state = (size_t)kBP * p.N * sizeof(float);
    size_t n = align_up(units * p.nch * state, 256);
    if (p.G != p.H) n += 2 * align_up((size_t)p.nb * p.L * p.M * p.H * p.N * sizeof(float), 256);
    if (p.S > 1) n += 2 * align_up(units * p.S * state, 256) + 2 * align_up(units * p.S * sizeof(float), 256);
    if (p.A) n += 2 * align_up(units * p.S * sizeof(float), 256);
    return n;
}

bool ssd_f32_bwd_plan(SsdF32BwdParams* q, size_t limit) {
    SsdF32BwdParams& p = *q;
    if (p.P != kBP || (p.N != 64 && p.N != 128)) return false;
    // a step's ranks lie in one 32-row tile: its own-step block is on the diagonal
    if (p.M < 1 || p.M > 32 || (p.M & (p.M - 1)) != 0) return false;
    for (const void* ptr : {p.v, p.B, p.C, p.dy})  // four values per load
        if (((uintptr_t)ptr & (p.bf16 ? 7u : 15u)) != 0) return false;
    p.vec = true;
    for (const float* ptr : {p.dv, p.dBh, p.dCh, p.dh0})
        if (((uintptr_t)ptr & 15u) != 0) p.vec = false;
    for (int64_t s : {p.v_sb, p.v_sl, p.v_sm, p.v_sh, p.B_sb, p.B_sl, p.B_sm, p.B_sg, p.C_sb, p.C_sl, p.C_sm, p.C_sg,
                      p.dy_sb, p.dy_sl, p.dy_sm, p.dy_sh})
        if (s % 4 != 0) return false;
    p.mshift = __builtin_ctz(p.M);
    const int64_t steps = kFR >> p.mshift;
    p.nch = (int)((p.L + steps - 1) / steps);
    // In units of a chunk of the reverse loop (one workgroup per CU, rounds of
    // 256): a segment's chunks and its entry gradient; the state kernels about
    // a third of a chunk each at three workgroups per CU, and a launch.
    const int64_t units = (int64_t)p.nb * p.H;
    double best = 0.;
    for (int n = 1; n <= std::min(p.nch, 64); ++n) {
        SsdF32BwdParams t = p;
        t.cps = (p.nch + n - 1) / n;
        t.S = (p.nch + t.cps - 1) / t.cps;
        if (ssd_f32_bwd_workspace(t) > limit) continue;
        const int64_t r3 = (units * t.S + 255) / 256, r2 = (units * t.S + 767) / 768,
                      r1 = (2 * units * (t.S - 1) + 767) / 768;
        const double cost = (double)r3 * (t.cps + 0.5 + 0.05 * t.S) + (double)r2 * (0.35 * t.cps + 0.3) +
                            (t.S > 1 ? (double)r1 * 0.35 * t.cps + 0.4 : 0.);
        if (best == 0. || cost < best) {
            best = cost;
            p.S = t.S;
            p.cps = t.cps;
        }
    }
    return best > 0. && units * p.S * 2 < (1ll << 31);
}

static FBRows fb_rows(const SsdF32BwdParams& p) {
    const int64_t last = ((int64_t)p.L << p.mshift) - (int64_t)(p.nch - 1) * kFR;  // rows of the last chunk
    return p.S > 1 || p.nch > 4 || last > kFR / 2 ? FB_FULL : p.nch == 1 ? FB_ONE : FB_TAIL;
}

template <int N, typename T, FBRows R>
static int fb_run_as(const SsdF32BwdParams& p, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
    const int units = p.nb * p.H;
    // dynamic LDS above the 64 KB default (up to the CU's 160 KB)
    constexpr size_t lds = sizeof(FBLds<N>);
    static_assert(lds <= 160 * 1024, "LDS of a CU");
    MAMBA_CHECK_HIP(hipFuncSetAttribute((const void*)ssd_f32_bwd_chunks<N, T, R>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)lds));
    if (p.S > 1) {
        hipLaunchKernelGGL((ssd_f32_bwd_seg<N, T>), dim3(units * (p.S - 1) * 2), dim3(256), 0, stream, p);
        MAMBA_CHECK_LAUNCH();
    }
    if (R != FB_ONE) {
        hipLaunchKernelGGL((ssd_f32_bwd_states<N, T>), dim3(units * p.S), dim3(256), 0, stream, p);
        MAMBA_CHECK_LAUNCH();
    }
    if (ev0) MAMBA_CHECK_HIP(hipEventRecord(ev0, stream));
    hipLaunchKernelGGL((ssd_f32_bwd_chunks<N, T, R>), dim3(units * p.S), dim3(512), lds, stream, p);
    MAMBA_CHECK_LAUNCH();
    if (ev1) MAMBA_CHECK_HIP(hipEventRecord(ev1, stream));
    return MAMBA_OK;
}

template <int N, typename T>
static int fb_run(const SsdF32BwdParams& p, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
    switch (fb_rows(p)) {
        case FB_ONE: return fb_run_as<N, T, FB_ONE>(p, stream, ev0, ev1);
        case FB_TAIL: return fb_run_as<N, T, FB_TAIL>(p, stream, ev0, ev1);
        default: return fb_run_as<N, T, FB_FULL>(p, stream, ev0, ev1);
    }
}

int ssd_f32_bwd_launch(SsdF32BwdParams& p, void* ws, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
    const size_t units = (size_t)p.nb * p.H, state = (size_t)kBP * p.N * sizeof(float);
    char* at = static_cast<char*>(ws);
    auto take = [&](size_t bytes) {
        float* r = reinterpret_cast<float*>(at);
        at += align_up(bytes, 256);
        return r;
    };
    p.hs = take(units * p.nch * state);
    if (p.G != p.H) {
        const size_t plane = (size_t)p.nb * p.L * p.M * p.H * p.N * sizeof(float);
        p.dBh = take(plane);
        p.dCh = take(plane);
    }
    if (p.S > 1) {
        p.fs = take(units * p.S * state);
        p.gs = take(units * p.S * state);
        p.fd = take(units * p.S * sizeof(float));
        p.gd = take(units * p.S * sizeof(float));
    }
    if (p.A) {
        p.pA = take(units * p.S * sizeof(float));
        p.pD = take(units * p.S * sizeof(float));
    }
    if (p.bf16)
        return p.N == 128 ? fb_run<128, bf16_t>(p, stream, ev0, ev1) : fb_run<64, bf16_t>(p, stream, ev0, ev1);
    return p.N == 128 ? fb_run<128, float>(p, stream, ev0, ev1) : fb_run<64, float>(p, stream, ev0, ev1);
}

}  // namespace mamba
