// Batched f32 products for blocks of a few hundred tokens, on f32 MFMA:
//   C[z][m][n] = sum_k A[z][m][k] B[z][k][n], any layout with one unit stride
// per operand, so that a block reads its weights and activations where they are
// (transposed or not) instead of copying them into a library's preferred form.
//
// Why not the library alone: at 2 x 256 tokens, 512 channels it takes 256 x 256
// tiles for the transposed products, two workgroups on 256 CUs: out_proj 118 us
// and x_proj 25 us for 0.13 and 0.025 GFLOP, here 7.9 and 7.5 us.  Larger
// products stay with the library, which reaches 154 TFLOP/s.
//
// Tilings: 64 x 64 (a 32 x 32 tile per wave of four, 32 of K per step), and, where
// those would give fewer workgroups than CUs, 32 x 32 with 4, 8 or 16 waves sharing
// K (128, 256 or 512 per step), their tiles summed through LDS at the end in a fixed
// order.  Bound by launch and one load latency per step in the small; a lone
// tile's MFMAs take 1.7 us per 512 of K.
#include "bwd_core.h"
#include "common.h"

namespace mamba {

struct MmParams {
    int Z, M, N, K;
    const float* a; int64_t a_sz, a_sm, a_sk;
    const float* b; int64_t b_sz, b_sk, b_sn;
    float* c; int64_t c_sz, c_sm;  // unit stride along n
    bool a_vec, b_vec;             // 16-byte loads along the unit stride
    int tiles_m, tiles_n;
};

// An operand's W x KB block (W rows of M or columns of N, KB of K) in registers,
// then in LDS.  KC: K is the unit stride, LDS [w][KB + 4], operands read as 16
// bytes (4 of K); else LDS [k][W + 8], operands read a word at a time.
template <int W, int KB, bool KC, int NT>
struct MmBlock {
    static constexpr int NV = W * KB / 4 / NT;            // float4 per thread
    static constexpr int P = KC ? KB + 4 : W + 8;         // pitch
    static constexpr int WORDS = (KC ? W : KB) * P;
    float4 v[NV];

    __device__ __forceinline__ void load(const float* p, int64_t sw, int64_t sk, int w0, int k0, int nw, int nk,
                                         bool vec, int tid) {
        constexpr int RV = (KC ? KB : W) / 4;              // float4 per LDS row
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const int e = tid + NT * q, r = e / RV, c = (e % RV) * 4;
            const int w = w0 + (KC ? r : c), k = k0 + (KC ? c : r);
            float4 x = {0.f, 0.f, 0.f, 0.f};
            if (KC ? w < nw : k < nk) {
                const float* at = p + (int64_t)w * sw + (int64_t)k * sk;
                const int left = KC ? nk - k : nw - w;     // values along the unit stride
                if (vec && left >= 4) {
                    x = *reinterpret_cast<const float4*>(at);
                } else {
                    if (left > 0) x.x = at[0];
                    if (left > 1) x.y = at[1];
                    if (left > 2) x.z = at[2];
                    if (left > 3) x.w = at[3];
                }
            }
            v[q] = x;
        }
    }
    __device__ __forceinline__ void store(float* s, int tid) const {
        constexpr int RV = (KC ? KB : W) / 4;
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const int e = tid + NT * q;
            *reinterpret_cast<float4*>(s + (e / RV) * P + (e % RV) * 4) = v[q];
        }
    }
    // the operand values of w = w0 + lane % 32 at k = k0 + 4 (lane / 32) + 0..3
    static __device__ __forceinline__ float4 get(const float* s, int w, int k) {
        if constexpr (KC) {
            return *reinterpret_cast<const float4*>(s + w * P + k);
        } else {
            const float* at = s + k * P + w;
            return make_float4(at[0], at[P], at[2 * P], at[3 * P]);
        }
    }
};

// NS waves share K on a 32 x 32 tile; NS = 1: 64 x 64, a quarter per wave of 4
template <bool AK, bool BK, int NS>
__global__ __launch_bounds__(NS == 1 ? 256 : 64 * NS) void mm_f32_kernel(MmParams p) {
    constexpr bool SPLIT = NS > 1;
    constexpr int W = SPLIT ? 32 : 64, KB = 32 * NS, NT = SPLIT ? 64 * NS : 256;
    using MA = MmBlock<W, KB, AK, NT>;
    using MB = MmBlock<W, KB, BK, NT>;
    extern __shared__ __align__(16) float mm_smem[];
    float* sA = mm_smem;
    float* sB = mm_smem + MA::WORDS;
    const int tid = threadIdx.x, wv = wave_id(), lane = tid & 63, i32 = lane & 31, hf = lane >> 5;
    int t = blockIdx.x;
    const int tn = t % p.tiles_n;
    t /= p.tiles_n;
    const int tm = t % p.tiles_m, z = t / p.tiles_m;
    const float* a = p.a + (int64_t)z * p.a_sz;
    const float* b = p.b + (int64_t)z * p.b_sz;
    const int m0 = tm * W, n0 = tn * W;
    MA ra;
    MB rb;
    bwd_f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    const int wm = SPLIT ? 0 : 32 * (wv >> 1), wn = SPLIT ? 0 : 32 * (wv & 1), wk = SPLIT ? 32 * wv : 0;
    ra.load(a, p.a_sm, p.a_sk, m0, 0, p.M, p.K, p.a_vec, tid);
    rb.load(b, p.b_sn, p.b_sk, n0, 0, p.N, p.K, p.b_vec, tid);
    for (int k0 = 0; k0 < p.K; k0 += KB) {
        ra.store(sA, tid);
        rb.store(sB, tid);
        __syncthreads();
        if (k0 + KB < p.K) {
            ra.load(a, p.a_sm, p.a_sk, m0, k0 + KB, p.M, p.K, p.a_vec, tid);
            rb.load(b, p.b_sn, p.b_sk, n0, k0 + KB, p.N, p.K, p.b_vec, tid);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float4 x = MA::get(sA, wm + i32, wk + 8 * s + 4 * hf);
            const float4 y = MB::get(sB, wn + i32, wk + 8 * s + 4 * hf);
            acc = bwd_mfma(x.x, y.x, acc);
            acc = bwd_mfma(x.y, y.y, acc);
            acc = bwd_mfma(x.z, y.z, acc);
            acc = bwd_mfma(x.w, y.w, acc);
        }
        __syncthreads();
    }
    float* c = p.c + (int64_t)z * p.c_sz;
    const int n = n0 + wn + i32;
    if constexpr (SPLIT) {
        // the waves' tiles through LDS, added in wave order: every wave its
        // share of the rows
        static_assert(MA::WORDS + MB::WORDS >= NS * 1024, "room for the waves' tiles");
        constexpr int RW = 16 / NS;
#pragma unroll
        for (int r = 0; r < 16; ++r) mm_smem[wv * 1024 + r * 64 + lane] = acc[r];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < RW; ++q) {
            const int r = wv * RW + q;
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < NS; ++w) v += mm_smem[w * 1024 + r * 64 + lane];
            const int m = m0 + bwd_row(r, hf);
            if (m < p.M && n < p.N) c[(int64_t)m * p.c_sm + n] = v;
        }
        return;
    }
    if (n < p.N)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = m0 + wm + bwd_row(r, hf);
            if (m < p.M) c[(int64_t)m * p.c_sm + n] = acc[r];
        }
}

static int mm_params(const mamba_mm_f32_args* a, MmParams* out) {
    MAMBA_CHECK_ARG(a != nullptr, "args is NULL");
    MAMBA_CHECK_ARG(a->batch > 0 && a->m > 0 && a->n > 0 && a->k > 0, "sizes must be >= 1");
    MAMBA_CHECK_ARG(a->a && a->b && a->c, "a, b and c are required");
    MAMBA_CHECK_ARG((a->a_sm == 1 || a->a_sk == 1) && (a->b_sk == 1 || a->b_sn == 1),
                    "a and b need a unit stride in one of their last two axes");
    MmParams p;
    p.Z = a->batch; p.M = a->m; p.N = a->n; p.K = a->k;
    p.a = a->a; p.a_sz = a->a_sb; p.a_sm = a->a_sm; p.a_sk = a->a_sk;
    p.b = a->b; p.b_sz = a->b_sb; p.b_sk = a->b_sk; p.b_sn = a->b_sn;
    p.c = a->c; p.c_sz = a->c_sb; p.c_sm = a->c_sm;
    auto al = [](const void* q, int64_t s0, int64_t s1) { return ((uintptr_t)q & 15u) == 0 && s0 % 4 == 0 && s1 % 4 == 0; };
    p.a_vec = al(p.a, p.a_sz, p.a_sk == 1 ? p.a_sm : p.a_sk);
    p.b_vec = al(p.b, p.b_sz, p.b_sk == 1 ? p.b_sn : p.b_sk);
    *out = p;
    return MAMBA_OK;
}

template <bool AK, bool BK, int NS>
static int mm_run(MmParams p, hipStream_t s) {
    constexpr int W = NS > 1 ? 32 : 64, KB = 32 * NS, NT = NS > 1 ? 64 * NS : 256;
    constexpr int lds = (MmBlock<W, KB, AK, NT>::WORDS + MmBlock<W, KB, BK, NT>::WORDS) * 4;
    static_assert(lds <= 160 * 1024, "LDS of a CU");
    p.tiles_m = (p.M + W - 1) / W;
    p.tiles_n = (p.N + W - 1) / W;
    if (lds > 64 * 1024)
        MAMBA_CHECK_HIP(hipFuncSetAttribute((const void*)mm_f32_kernel<AK, BK, NS>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    hipLaunchKernelGGL((mm_f32_kernel<AK, BK, NS>), dim3((unsigned)((int64_t)p.Z * p.tiles_m * p.tiles_n)), dim3(NT), lds,
                       s, p);
    MAMBA_CHECK_LAUNCH();
    return MAMBA_OK;
}

// 64 x 64 tiles where they give every CU a workgroup; else 32 x 32 with K over 4
// waves, or over 8 or 16 where K is long and the tiles are still few (a step's load
// latency, about 2 us, is paid K / 256 or K / 512 times instead of K / 128; 512 x
// 512 of K = 256: 7.1 us with 16 waves, half of them idle, 5.3 with 8).
template <bool AK, bool BK>
static int mm_launch(const MmParams& p, hipStream_t s) {
    auto tiles = [&](int w) { return (int64_t)p.Z * ((p.M + w - 1) / w) * ((p.N + w - 1) / w); };
    if (tiles(64) >= 256) return mm_run<AK, BK, 1>(p, s);
    if (p.K <= 128 || tiles(32) > 512) return mm_run<AK, BK, 4>(p, s);
    return p.K <= 256 ? mm_run<AK, BK, 8>(p, s) : mm_run<AK, BK, 16>(p, s);
}

}  // namespace mamba

using namespace mamba;

extern "C" int mamba_mm_f32(const mamba_mm_f32_args* a, mamba_stream_t stream) {
    MmParams p;
    const int st = mm_params(a, &p);
    if (st != MAMBA_OK) return st;
    MAMBA_CHECK_ARG((int64_t)p.Z * ((p.M + 31) / 32) * ((p.N + 31) / 32) < (1ll << 31), "too many tiles");
    const hipStream_t s = (hipStream_t)stream;
    // a K of 1 has both strides free: any form reads it
    const bool ak = p.a_sk == 1, bk = p.b_sk == 1;
    if (ak) return bk ? mm_launch<true, true>(p, s) : mm_launch<true, false>(p, s);
    return bk ? mm_launch<false, true>(p, s) : mm_launch<false, false>(p, s);
}
