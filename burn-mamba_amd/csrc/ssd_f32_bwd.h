// The segment-parallel SSD backward on f32 MFMA (ssd_f32_bwd.hip), shared by
// the Mamba-2 and the Mamba-3 seams.
#pragma once

#include "common.h"

namespace mamba {

struct SsdF32BwdParams {
    int nb, L, M, mshift, H, P, G, N;  // L counts steps; M = 1 << mshift ranks per step
    int nch, S, cps;                   // chunks of 64 fused rows, segments, chunks per segment
    bool bf16;                         // v, B, C and dy are bf16 (f32 otherwise)
    const void* v; int64_t v_sb, v_sl, v_sm, v_sh;
    // log-decay per step: da (A == NULL), or dt with A[h] (Mamba-2)
    const float* da; int64_t da_sb, da_sl, da_sh;
    const float* A;
    // source weights of earlier steps (sc) and of the row's own step (gm); NULL: 1
    const float* gm; int64_t gm_sb, gm_sl, gm_sh;
    const float* sc; int64_t sc_sb, sc_sl, sc_sh;
    const void* B; int64_t B_sb, B_sl, B_sm, B_sg;
    const void* C; int64_t C_sb, C_sl, C_sm, C_sg;
    const float* D;        // dv += D[h] dy (Mamba-2), or NULL
    const float* h0;       // [b, h, p, n] or NULL
    const void* dy; int64_t dy_sb, dy_sl, dy_sm, dy_sh;
    const float* dfin;     // [b, h, p, n] or NULL
    float* dv;             // [b, l, m, h, p]
    float* dda;            // [b, l, h]: d(da), or with A the whole d(dt)
    float* dsc; float* dgm;  // [b, l, h] or NULL
    float* dBh; float* dCh;  // [b, l, m, h, n]
    float* dh0;            // [b, h, p, n]
    bool vec;              // every output is 16-byte aligned
    // workspace
    float* hs;             // [b h][chunk][tile][16][64] states entering the chunks
    float* fs; float* gs;  // [b h][S][n][p] segments' states and state gradients (0: dfin)
    float* fd; float* gd;  // [b h][S] segment log2-decays
    float* pA; float* pD;  // [b h][S] partial dA, dD (Mamba-2)
};

// Whether the kernels cover these shapes and layouts; fills nch, and S and cps
// for the fewest estimated rounds whose workspace is within `limit` bytes.
bool ssd_f32_bwd_plan(SsdF32BwdParams* p, size_t limit);
size_t ssd_f32_bwd_workspace(const SsdF32BwdParams& p);
// Places the workspace's parts (with ngroups < nheads dBh and dCh: the caller
// sums them over each group's heads; with A the pA and pD partials: over batch
// and segments) and launches.  ev0 / ev1 (nullable) are recorded around the
// reverse chunk loop.
int ssd_f32_bwd_launch(SsdF32BwdParams& p, void* ws, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1);

}  // namespace mamba
