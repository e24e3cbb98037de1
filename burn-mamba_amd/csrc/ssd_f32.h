// The segment-parallel f32 SSD forward on f32 MFMA (ssd_f32.hip), shared by
// the Mamba-2 and the Mamba-3 seams: both are the same recurrence on fused
// (step, rank) rows.
#pragma once

#include "common.h"

namespace mamba {

struct SsdF32Params {
    int nb, L, M, mshift, H, P, G, N;  // L counts steps; M = 1 << mshift ranks per step
    int nch, S, cps;                   // chunks of 64 fused rows, segments, chunks per segment
    int io_dtype;
    const void* v; int64_t v_sb, v_sl, v_sm, v_sh;
    // log-decay per step: da (A == NULL), or dt with A[h] (Mamba-2)
    const float* da; int64_t da_sb, da_sl, da_sh;
    const float* A;
    // source weights of earlier steps (sc) and of the row's own step (gm); NULL: 1
    const float* gm; int64_t gm_sb, gm_sl, gm_sh;
    const float* sc; int64_t sc_sb, sc_sl, sc_sh;
    const void* Bm; int64_t B_sb, B_sl, B_sm, B_sg;
    const void* Cm; int64_t C_sb, C_sl, C_sm, C_sg;
    const float* D;         // y += D[h] v (Mamba-2), or NULL
    const float* h0;        // [b, h, p, n] or NULL
    const float* init_hpr;  // [h, p, n] or NULL
    void* y; int64_t y_sb, y_sl, y_sm, y_sh;
    float* hT;
    float* seg;             // [b h pblock][S][N * PB] segments' end states (0: from the initial state, which S - 1 holds)
    float* segd;            // [b h pblock][S] segment log2-decays
};

// Whether the kernels cover these shapes and layouts; fills nch, S and cps.
bool ssd_f32_plan(SsdF32Params* p);
size_t ssd_f32_workspace(const SsdF32Params& p);
// ev0 / ev1 (nullable) are recorded around the scan kernel.
int ssd_f32_launch(const SsdF32Params& p, void* ws, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1);

}  // namespace mamba
