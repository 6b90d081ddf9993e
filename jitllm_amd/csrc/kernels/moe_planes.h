// A handful of routed pairs over packed planes (Q4_K), without grouping or combine, as moe.h has it over GGUF rows: the packed
// matvec on a pair's sheet, and for the down projections its chunk loop over the chunks of all of a row's pairs, a chunk's
// planes those of the pair it belongs to.
#pragma once
#include "matvec.h"
#include "mxfp4.h"
#include "packed.h"

#pragma clang fp contract(off)

template <int RW, int XPRE>
__device__ __forceinline__ void moe_planes_gather_body(const MoePlanesGatherArgs& m, uint8_t* smem) {
    const u32 c = blockIdx.y;
    const int y = blockIdx.z;
    PackedMatVecArgs p;
    p.out = m.out[y]; p.qs = m.qs[y]; p.d = m.d[y]; p.sc = m.sc[y]; p.x = m.x; p.nrows = m.nrows; p.k = m.k; p.stride = m.stride;
    p.per = m.per; p.nwaves = m.nwaves; p.ngroups = m.ngroups;
    p.q = nullptr; p.as = nullptr; p.s16 = nullptr; p.x2 = nullptr; p.resid = nullptr; p.alpha = 0.f; p.norm_out = nullptr;
    p.norm_eps = 0.f; p.inv_k = 0.0;
    const u32* sel = m.sel;
    size_t words = m.sheet_words;
    int row_step = m.row_step, ku = m.k_used, sel_stride = m.sel_stride, n_expert = m.n_expert;
    JL_NOW(p.out, p.qs, p.d, p.sc, p.x, p.nrows, p.k, p.stride, p.per, p.nwaves, p.ngroups, sel, words, row_step, ku, sel_stride, n_expert);
    const u32 row = sel ? c / (u32)ku : c;
    // (no selection: one matrix; an id no expert has: the last sheet, for a pair that adds nothing, see below)
    const u32 e = !sel ? 0u : min((u32)__builtin_amdgcn_readfirstlane((i32)as_global(sel)[row * (u32)sel_stride + (c - row * (u32)ku)]), (u32)n_expert - 1u);
    p.out = as_global(p.out) + (size_t)c * p.nrows;
    p.qs = as_global(p.qs) + (size_t)e * words; p.d = as_global(p.d) + (size_t)e * words; p.sc = as_global(p.sc) + (size_t)e * words;
    p.row0 = (int)e * row_step;
    p.x = as_global(p.x) + (size_t)row * p.k;
    packed_matvec_body<JL_Q4_KF, RW, XPRE, true>(p, smem);
}
template <int RW, int XPRE>
__device__ __forceinline__ void moe_planes_down_body(const MoePlanesDownArgs& args, uint8_t* smem) {
    constexpr int KP = 64 / RW, NB = 8 / KP;
    MoePlanesDownArgs m = args;
    JL_NOW(m.resid, m.qs, m.d, m.sc, m.g, m.u, m.sel, m.wt, m.sheet_words, m.nrows, m.k, m.row_step, m.stride, m.per, m.nwaves, m.ngroups,
           m.n_expert, m.sel_stride, m.k_used);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwaves = m.nwaves;
    const size_t tok = blockIdx.y;
    const u32* sel = m.sel ? as_global(m.sel) + tok * m.sel_stride : nullptr;   // (null: expert 0)
    const float* wt = m.wt ? as_global(m.wt) + tok * m.k_used : nullptr;        // (null: 1)
    float* resid = as_global(m.resid) + tok * m.nrows;
    int g = blockIdx.x;
    if ((m.ngroups & 7) == 0) g = (g & 7) * (m.ngroups >> 3) + (g >> 3);   // (neighbouring row runs to one XCD, as above)
    const int rl = lane % RW, b0 = lane / RW * NB, rr = min(g * RW + rl, m.nrows - 1);
    // lane i holds pair i's id and weight (an id no expert has: the last sheet is read for it and nothing added)
    const u32 last = (u32)m.n_expert - 1u, ids = sel ? sel[min(lane, m.k_used - 1)] : 0u;
    const float wts = wt ? wt[min(lane, m.k_used - 1)] : 1.f;

    const int row_chunks = m.k / 256, nchunks = row_chunks * m.k_used;
    PackedMatVecArgs p;   // the activation: the row's gated columns one behind the other
    p.k = m.k * m.k_used; p.x = as_global(m.g) + tok * p.k; p.x2 = as_global(m.u) + tok * p.k; p.per = m.per; p.stride = m.stride;
    p.norm_out = nullptr; p.q = nullptr; p.as = nullptr; p.s16 = nullptr;
    const u32 *qs = as_global(m.qs), *d = as_global(m.d), *sc = as_global(m.sc);
    uint8_t* my = smem + wave * JL_PK_WAVE_LDS;
    PkAct A;
    A.a = (const u32x4*)my; A.da = (const float*)(my + 256); A.ss = (const float*)(my + 288);
    PkX<true> X[XPRE];
#pragma unroll
    for (int i = 0; i < XPRE; i++) pk_load_x<true, true>(p, wave + i * nwaves, lane, X[i]);
    __builtin_amdgcn_s_barrier();
    float acc = 0.f;
    auto chunk = [&](int c, const PkX<true>& Xc) __attribute__((always_inline)) {
        const int pair = c / row_chunks, cc = c - pair * row_chunks;   // (uniform)
        const u32 id = (u32)__builtin_amdgcn_readlane((i32)ids, pair);
        const size_t e = min(id, last);
        p.qs = qs + e * m.sheet_words; p.d = d + e * m.sheet_words; p.sc = sc + e * m.sheet_words;
        const int row = (int)e * m.row_step + rr;
        PkWQ4KF<NB> w;
        pk_load<NB>(p, cc, b0, row, w);
        pk_stage_x<true, true>(p, c, lane, Xc, my);
        const float more = fmaf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(i32, wts), pair)), pk_dot<NB>(p, w, cc, b0, row, A), acc);
        acc = id <= last ? more : acc;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
#pragma unroll
    for (int i = 0; i < XPRE; i++) {
        const int c = wave + i * nwaves;
        if (c < nchunks) chunk(c, X[i]);
    }
    for (int c = wave + XPRE * nwaves; c < nchunks; c += nwaves) {
        PkX<true> Xc;
        pk_load_x<true, true>(p, c, lane, Xc);
        chunk(c, Xc);
    }
    float* red = (float*)(smem + nwaves * JL_PK_WAVE_LDS);
    red[wave * JL_PK_RED_STRIDE + lane] = acc;
    const int j = threadIdx.x & 15;
    const float base = resid[min(g * RW + (int)(threadIdx.x >> 4), m.nrows - 1)];
    lds_barrier();
    for (int r = threadIdx.x >> 4; r < RW; r += nwaves * 4) {
        float t = 0.f;
        if (j < nwaves) {
#pragma unroll
            for (int q = 0; q < KP; q++) t += red[j * JL_PK_RED_STRIDE + q * RW + r];
        }
        t += dpp_f32<JL_DPP_QUAD_XOR1, 0xf>(t);
        t += dpp_f32<JL_DPP_QUAD_XOR2, 0xf>(t);
        t += dpp_f32<JL_DPP_ROW_HALF_MIRROR, 0xf>(t);
        t += dpp_f32<JL_DPP_ROW_MIRROR, 0xf>(t);
        if (j == 0 && g * RW + r < m.nrows) resid[g * RW + r] = (r < nwaves * 4 ? base : resid[g * RW + r]) + t;
    }
}
