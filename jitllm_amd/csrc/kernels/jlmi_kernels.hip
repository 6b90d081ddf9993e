// The gfx950 code object: every kernel entry point the C ABI launches through
// hipModuleLaunchKernel.  Built with
//   hipcc --genco --offload-arch=gfx950 -O3 -ffp-contract=off ...
// Entry points are extern "C" so the host can look them up by name.
#include "common.h"
#include "dequant.h"
#include "few_i8.h"
#include "gemm_i8.h"
#include "gemm_q4k.h"
#include "gemm_q4k_k2.h"
#include "gemm_q4k_fold.h"
#include "matvec.h"
#include "moe.h"
#include "moe_cols.h"
#include "moe_planes.h"
#include "mxfp4.h"
#include "packed.h"
#include "quantize.h"

extern __shared__ __attribute__((aligned(16))) uint8_t jl_smem[];

// ------------------------------------------------------------- quantizer
// x [ntok][k] f32 -> q [ntok][k] int8, as [ntok][k/32], sum16 [ntok][k/16].
// grid = (ceil(k/4/256), ntok), block = 256: one thread per four elements.
// x2 (may be null): the activation is silu(x) * x2, the gated feed-forward block's, formed
// with the arithmetic of the fused matvec's own quantizer.
extern "C" __global__ __launch_bounds__(256) void jl_quantize_act(
    const float* __restrict__ x, int8_t* __restrict__ q, float* __restrict__ as,
    float* __restrict__ sum16, int k, int per, const float* __restrict__ x2) {
    const size_t tok = blockIdx.y;
    const int g4 = blockIdx.x * 256 + threadIdx.x;
    const bool live = g4 < k / 4;
    f32x4 v = live ? ((const f32x4*)(x + tok * (size_t)k))[g4] : f32x4{0.f, 0.f, 0.f, 0.f};
    if (x2) {
        const f32x4 u = live ? ((const f32x4*)(x2 + tok * (size_t)k))[g4] : f32x4{0.f, 0.f, 0.f, 0.f};
        v = f32x4{silu_f32(v.x) * u.x, silu_f32(v.y) * u.y, silu_f32(v.z) * u.z, silu_f32(v.w) * u.w};
    }
    u32 m = max(max(abs_bits(v.x), abs_bits(v.y)), max(abs_bits(v.z), abs_bits(v.w)));
    u32 amax = window_amax(live ? m : 0u, per);
    float d;
    i32 sum;
    u32 qq = quantize4(v, amax, d, sum);
    if (live) {
        ((u32*)(q + tok * (size_t)k))[g4] = qq;
        if ((g4 & 3) == 0) sum16[tok * (size_t)(k / 16) + (g4 >> 2)] = (float)sum;
        if ((g4 & 7) == 0) as[tok * (size_t)(k / 32) + (g4 >> 3)] = d;
    }
}

// --------------------------------------------------------------- dequant
extern "C" __global__ __launch_bounds__(256) void jl_dequant(
    const uint8_t* __restrict__ src, float* __restrict__ dst, size_t n, int type) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = dequant_elem(type, src, i);
}

// ---------------------------------------------------------------- matvec
// jl_matvec_<type>_r<rows per wavefront>; the workgroup is 64..1024 threads.
// MAXT is the largest workgroup the variant's register use allows.
// _x2, _x4: the same for an activation of two, of more float4 groups a thread, whose first two (four)
// groups a thread loads together ahead of its weights.
#define JL_MATVEC_KERNEL(T, TYPE, RPW, MAXT)                                                 \
    extern "C" __global__ __launch_bounds__(MAXT) void jl_matvec_##T##_r##RPW(MatVecArgs p) { \
        matvec_body<TYPE, RPW, 1>(p, jl_smem);                                               \
    }                                                                                        \
    extern "C" __global__ __launch_bounds__(MAXT) void jl_matvec_##T##_r##RPW##_x2(MatVecArgs p) { \
        matvec_body<TYPE, RPW, 2>(p, jl_smem);                                               \
    }                                                                                        \
    extern "C" __global__ __launch_bounds__(MAXT) void jl_matvec_##T##_r##RPW##_x4(MatVecArgs p) { \
        matvec_body<TYPE, RPW, 4>(p, jl_smem);                                               \
    }
// _res: one row a wavefront with resid[r] += weight * out[r] riding on the store (MatVecArgs.resid set);
// _pq: one row a wavefront over an activation that comes quantized (MatVecArgs.q / as / s16, x null)
#define JL_MATVEC_RES_KERNEL(T, TYPE)                                                               \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_##T##_r1_res(MatVecArgs p) {       \
        matvec_body<TYPE, 1, 1, true>(p, jl_smem);                                                  \
    }                                                                                               \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_##T##_r1_x2_res(MatVecArgs p) {    \
        matvec_body<TYPE, 1, 2, true>(p, jl_smem);                                                  \
    }                                                                                               \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_##T##_r1_x4_res(MatVecArgs p) {    \
        matvec_body<TYPE, 1, 4, true>(p, jl_smem);                                                  \
    }                                                                                               \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_##T##_r1_pq(MatVecArgs p) {        \
        matvec_body<TYPE, 1, 1, false, true>(p, jl_smem);                                           \
    }                                                                                               \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_##T##_r1_pq_res(MatVecArgs p) {    \
        matvec_body<TYPE, 1, 1, true, true>(p, jl_smem);                                            \
    }
JL_MATVEC_RES_KERNEL(q4k, JL_Q4_K) JL_MATVEC_RES_KERNEL(q8_0, JL_Q8_0) JL_MATVEC_RES_KERNEL(q6k, JL_Q6_KS)
JL_MATVEC_RES_KERNEL(q8_0p, JL_Q8_0P)
JL_MATVEC_KERNEL(q4k, JL_Q4_K, 1, 1024) JL_MATVEC_KERNEL(q4k, JL_Q4_K, 2, 1024) JL_MATVEC_KERNEL(q4k, JL_Q4_K, 4, 512)
JL_MATVEC_KERNEL(q8_0, JL_Q8_0, 1, 1024) JL_MATVEC_KERNEL(q8_0, JL_Q8_0, 2, 1024) JL_MATVEC_KERNEL(q8_0, JL_Q8_0, 4, 1024)
// (Q6_K over the staging layout made for it: JL_STAGE_Q6K in kernels/matvec.h)
JL_MATVEC_KERNEL(q6k, JL_Q6_KS, 1, 1024) JL_MATVEC_KERNEL(q6k, JL_Q6_KS, 2, 512) JL_MATVEC_KERNEL(q6k, JL_Q6_KS, 4, 512)
// Q8_0 with two blocks a lane-slot, every load 4-byte aligned (rows 4-byte aligned, k % 64 == 0);
// dynamic LDS = JL_ACT_LDS_BYTES_SHIFTED(k)
JL_MATVEC_KERNEL(q8_0p, JL_Q8_0P, 1, 1024) JL_MATVEC_KERNEL(q8_0p, JL_Q8_0P, 2, 1024) JL_MATVEC_KERNEL(q8_0p, JL_Q8_0P, 4, 512)

// grid = (row groups, matrices), block = 64..1024.  _n: an RMSNorm in front of the quantizer, _a: a gated
// activation, _na: both; _res: MatVecMultiArgs.resid set
#define JL_MATVEC_MULTI_PRE(T, TYPE, P, PRE, SUF, RES)                                                             \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_multi_##T##P##SUF(MatVecMultiArgs p) {            \
        matvec_multi_body<TYPE, 1, RES, PRE>(p, jl_smem);                                             \
    }                                                                                                              \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_multi_##T##P##_x2##SUF(MatVecMultiArgs p) {       \
        matvec_multi_body<TYPE, 2, RES, PRE>(p, jl_smem);                                                          \
    }                                                                                                              \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_multi_##T##P##_x4##SUF(MatVecMultiArgs p) {       \
        matvec_multi_body<TYPE, 4, RES, PRE>(p, jl_smem);                                             \
    }
#define JL_MATVEC_MULTI_FORMS(T, TYPE, SUF, RES)                                                                   \
    JL_MATVEC_MULTI_PRE(T, TYPE, , 0, SUF, RES) JL_MATVEC_MULTI_PRE(T, TYPE, _n, JL_PRE_NORM, SUF, RES)            \
    JL_MATVEC_MULTI_PRE(T, TYPE, _a, JL_PRE_ACT, SUF, RES) JL_MATVEC_MULTI_PRE(T, TYPE, _na, JL_PRE_NORM | JL_PRE_ACT, SUF, RES) \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_multi_##T##_q##SUF(MatVecMultiArgs p) {           \
        matvec_multi_body<TYPE, 0, RES>(p, jl_smem);                                                  \
    }
#define JL_MATVEC_MULTI_KERNEL(T, TYPE) JL_MATVEC_MULTI_FORMS(T, TYPE, , false) JL_MATVEC_MULTI_FORMS(T, TYPE, _res, true)
JL_MATVEC_MULTI_KERNEL(q4k, JL_Q4_K) JL_MATVEC_MULTI_KERNEL(q8_0, JL_Q8_0) JL_MATVEC_MULTI_KERNEL(q6k, JL_Q6_KS)
JL_MATVEC_MULTI_KERNEL(q8_0p, JL_Q8_0P)
// One matrix for several tokens
JL_MATVEC_MULTI_PRE(q4kf, JL_Q4_KF, , 0, , false) JL_MATVEC_MULTI_PRE(q6kw, JL_Q6_KW, , 0, , false)
// The same grid over matrices of different types (the reference's MatVecSegments,
// jit/gpu/kernels/matvec.go:1411-1431: a block's q, k and v in one launch whatever their
// formats).
#define JL_MATVEC_SEGMENTS(P, PRE, SUF, RES)                                                                       \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_segments##P##SUF(MatVecMultiArgs p) {             \
        matvec_segments_body<RES, PRE>(p, jl_smem);                                                                 \
    }
JL_MATVEC_SEGMENTS(, 0, , false) JL_MATVEC_SEGMENTS(_n, JL_PRE_NORM, , false) JL_MATVEC_SEGMENTS(_a, JL_PRE_ACT, , false)
JL_MATVEC_SEGMENTS(_na, JL_PRE_NORM | JL_PRE_ACT, , false) JL_MATVEC_SEGMENTS(, 0, _res, true) JL_MATVEC_SEGMENTS(_n, JL_PRE_NORM, _res, true)
JL_MATVEC_SEGMENTS(_a, JL_PRE_ACT, _res, true) JL_MATVEC_SEGMENTS(_na, JL_PRE_NORM | JL_PRE_ACT, _res, true)

// The same with 32 or 16 lanes a row, for rows of at most that many slots
#define JL_MATVEC_LANES(T, TYPE, L)                                                                                \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_##T##_r1_l##L(MatVecArgs p) {                     \
        matvec_body<TYPE, 1, 1, false, false, L>(p, jl_smem);                                                      \
    }                                                                                                              \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_multi_##T##_l##L(MatVecMultiArgs p) {             \
        matvec_multi_body<TYPE, 1, false, 0, L>(p, jl_smem);                                                       \
    }                                                                                                              \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_multi_##T##_n_l##L(MatVecMultiArgs p) {           \
        matvec_multi_body<TYPE, 1, false, JL_PRE_NORM, L>(p, jl_smem);                                             \
    }
#define JL_MATVEC_LANES_TYPES(L)                                                                                   \
    JL_MATVEC_LANES(q4k, JL_Q4_K, L) JL_MATVEC_LANES(q8_0, JL_Q8_0, L) JL_MATVEC_LANES(q6k, JL_Q6_KS, L)           \
    JL_MATVEC_LANES(q8_0p, JL_Q8_0P, L)                                                                            \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_segments_l##L(MatVecMultiArgs p) {                \
        matvec_segments_body<false, 0, L>(p, jl_smem);                                                             \
    }                                                                                                              \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_segments_n_l##L(MatVecMultiArgs p) {              \
        matvec_segments_body<false, JL_PRE_NORM, L>(p, jl_smem);                                                   \
    }
JL_MATVEC_LANES_TYPES(32) JL_MATVEC_LANES_TYPES(16)
#define JL_MATVEC_TOKENS_LANES(T, TYPE, L)                                                                         \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_multi_##T##_l##L(MatVecMultiArgs p) {             \
        matvec_multi_body<TYPE, 1, false, 0, L>(p, jl_smem);                                                       \
    }
JL_MATVEC_TOKENS_LANES(q4kf, JL_Q4_KF, 32) JL_MATVEC_TOKENS_LANES(q4kf, JL_Q4_KF, 16)
JL_MATVEC_TOKENS_LANES(q6kw, JL_Q6_KW, 32) JL_MATVEC_TOKENS_LANES(q6kw, JL_Q6_KW, 16)

// -------------------------------------------------- few tokens, int8 matrix cores
extern "C" __global__ __launch_bounds__(256) void jl_few_prep(FewI8PrepArgs p) { few_i8_prep_body(p); }
// jl_few_<type>_<rows | planes>_t<token tiles>r<row tiles>: grid = (row tiles, experts, matrices)
#define JL_FEW_KERNEL(T, TYPE, P, PL, NT, RT, W256)                                                             \
    extern "C" __global__ __launch_bounds__(512, TYPE == JL_Q6_K && !W256 && PL && NT == 4 && RT == 2 ? 3 : 2)  \
    void jl_few_##T##_##P##_t##NT##r##RT(FewI8Args p) {                                                         \
        few_i8_body<TYPE, PL, NT, RT, W256>(p, jl_smem);                                                        \
    }
#define JL_FEW_SIZES(T, TYPE, P, PL, W256)                                                                      \
    JL_FEW_KERNEL(T, TYPE, P, PL, 1, 1, W256) JL_FEW_KERNEL(T, TYPE, P, PL, 1, 2, W256)                         \
    JL_FEW_KERNEL(T, TYPE, P, PL, 2, 1, W256) JL_FEW_KERNEL(T, TYPE, P, PL, 3, 1, W256)                         \
    JL_FEW_KERNEL(T, TYPE, P, PL, 3, 2, W256) JL_FEW_KERNEL(T, TYPE, P, PL, 4, 1, W256)                         \
    JL_FEW_KERNEL(T, TYPE, P, PL, 4, 2, W256)
#define JL_FEW_WIDE(T, TYPE, W256)                                                                              \
    JL_FEW_KERNEL(T, TYPE, planes, true, 1, 4, W256) JL_FEW_KERNEL(T, TYPE, planes, true, 2, 2, W256)           \
    JL_FEW_KERNEL(T, TYPE, planes, true, 2, 4, W256)
#define JL_FEW_FORMS(T, TYPE, W256)                                                                             \
    JL_FEW_SIZES(T, TYPE, rows, false, W256) JL_FEW_SIZES(T, TYPE, planes, true, W256) JL_FEW_WIDE(T, TYPE, W256)
JL_FEW_FORMS(q8_0, JL_Q8_0, false) JL_FEW_FORMS(q4k, JL_Q4_K, false) JL_FEW_FORMS(q6k, JL_Q6_K, false)
JL_FEW_FORMS(q4kw, JL_Q4_K, true) JL_FEW_FORMS(q6kw, JL_Q6_K, true)   // (the k-quant window)

// ---------------------------------------------------------- packed planes
// grid = (ceil(nrows/256), k/256 or k/32 for Q8_0), block = 256
extern "C" __global__ __launch_bounds__(256) void jl_pack_weights(PackArgs p) { pack_weights_body(p); }
// grid = (ceil(nrows/64), ceil(k/256)), block = 256
#define JL_UNPACK_KERNEL(T, TYPE)                                                              \
    extern "C" __global__ __launch_bounds__(256) void jl_unpack_##T(UnpackArgs p) {            \
        __shared__ __attribute__((aligned(16))) uint8_t lds[JL_UNPACK_LDS];                    \
        unpack_body<TYPE>(p, lds);                                                             \
    }
JL_UNPACK_KERNEL(q4k, JL_Q4_K) JL_UNPACK_KERNEL(q6k, JL_Q6_K) JL_UNPACK_KERNEL(q8_0, JL_Q8_0) JL_UNPACK_KERNEL(mxfp4, JL_MXFP4)
// jl_matvec_packed_<type>_w<rows per wavefront>: grid = ceil(nrows/RW), block = 64..1024
// XPRE = chunks whose activation loads go out ahead of the weights (register budget).
// jl_matvec_packed_<type>_w<RW> quantizes f32 x itself; jl_matvec_packed_q8_<type>_w<RW>
// takes activations already quantized.
#define JL_PACKED_KERNEL(T, TYPE, RW, XPRE)                                                                  \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_packed_##T##_w##RW(PackedMatVecArgs p) {    \
        packed_matvec_body<TYPE, RW, XPRE, true>(p, jl_smem);                                                \
    }                                                                                                        \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_packed_q8_##T##_w##RW(PackedMatVecArgs p) { \
        packed_matvec_body<TYPE, RW, XPRE, false>(p, jl_smem);                                               \
    }
JL_PACKED_KERNEL(q4k, JL_Q4_K, 64, 4) JL_PACKED_KERNEL(q4k, JL_Q4_K, 32, 4) JL_PACKED_KERNEL(q4k, JL_Q4_K, 16, 4)
JL_PACKED_KERNEL(q8_0, JL_Q8_0, 64, 2) JL_PACKED_KERNEL(q8_0, JL_Q8_0, 32, 4) JL_PACKED_KERNEL(q8_0, JL_Q8_0, 16, 4)
JL_PACKED_KERNEL(q6k, JL_Q6_K, 64, 4) JL_PACKED_KERNEL(q6k, JL_Q6_K, 32, 4) JL_PACKED_KERNEL(q6k, JL_Q6_K, 16, 4)
// jl_matvec_packed_multi[_act|_norm]_<type>_w<RW>: grid = (ceil(nrows/RW), matrices)
#define JL_PACKED_MULTI_KERNEL(T, TYPE, RW, XPRE)                                                               \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_packed_multi_##T##_w##RW(PackedMultiArgs p) {  \
        packed_matvec_multi_body<TYPE, RW, XPRE, false>(p, jl_smem);                                            \
    }                                                                                                           \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_packed_multi_act_##T##_w##RW(PackedMultiArgs p) { \
        packed_matvec_multi_body<TYPE, RW, 2, true>(p, jl_smem);                                                \
    }                                                                                                           \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_packed_multi_norm_##T##_w##RW(PackedMultiArgs p) { \
        packed_matvec_multi_body<TYPE, RW, 2, true, true>(p, jl_smem);                                          \
    }
JL_PACKED_MULTI_KERNEL(q4k, JL_Q4_K, 64, 4) JL_PACKED_MULTI_KERNEL(q4k, JL_Q4_K, 32, 4) JL_PACKED_MULTI_KERNEL(q4k, JL_Q4_K, 16, 4)
JL_PACKED_MULTI_KERNEL(q8_0, JL_Q8_0, 64, 2) JL_PACKED_MULTI_KERNEL(q8_0, JL_Q8_0, 32, 4) JL_PACKED_MULTI_KERNEL(q8_0, JL_Q8_0, 16, 4)
JL_PACKED_MULTI_KERNEL(q6k, JL_Q6_K, 64, 4) JL_PACKED_MULTI_KERNEL(q6k, JL_Q6_K, 32, 4) JL_PACKED_MULTI_KERNEL(q6k, JL_Q6_K, 16, 4)
#define JL_PACKED_TOKENS_KERNEL(RW)                                                                             \
    extern "C" __global__ __launch_bounds__(1024) void jl_matvec_packed_multi_q4kf_w##RW(PackedMultiArgs p) {   \
        packed_matvec_multi_body<JL_Q4_KF, RW, 4, false>(p, jl_smem);                                           \
    }
JL_PACKED_TOKENS_KERNEL(64) JL_PACKED_TOKENS_KERNEL(32) JL_PACKED_TOKENS_KERNEL(16)   // (one matrix for several tokens)

// ------------------------------------------------------------ prefill GEMM
// grid = (k/256, tok_pad/4), block = 256: one wavefront per (token, super-block)
// some more tokens: grid = (ceil(nrows / 32), ceil(ntok / 64)), block = 512
extern "C" __global__ __launch_bounds__(512) void jl_gemm_q4k_few32(GemmArgs p) {
    __shared__ __attribute__((aligned(16))) float part[8 * 2 * 1024];
    gemm_q4k_few32_body<2>(p, part);
}
extern "C" __global__ __launch_bounds__(256) void jl_gemm_prep_q4k(GemmPrepArgs p) {
    __shared__ u32 lds[JL_GEMM_PREP_LDS_WORDS];
    gemm_prep_q4k_body<4>(p, lds);
}
// the same with sixteen wavefronts a workgroup (few tokens): block = 1024
extern "C" __global__ __launch_bounds__(1024) void jl_gemm_prep_q4k_w16(GemmPrepArgs p) {
    __shared__ u32 lds[JL_GEMM_PREP_LDS_WORDS];
    gemm_prep_q4k_body<16>(p, lds);
}
// grid = (tok_pad/128, ceil(nrows/64)), block = 256, two workgroups per CU; and the
// 128-row form on 512 threads
extern "C" __global__ __launch_bounds__(256, 2) void jl_gemm_q4k_r64(GemmArgs p) {
    gemm_split_slice(p);
    gemm_q4k_body<1>(p, jl_smem, blockIdx.x * JL_GEMM_TILE, blockIdx.y * 64);
}
// The int8 form (kernels/gemm_i8.h): prep grid = (ceil(k/256), tok_pad/32), block = 1024; matrix kernel
// jl_gemm_i8_<type>_<shape>: grid = (token tiles, row tiles, K splits), block = 256, dynamic LDS = JL_GEMM_I8_LDS_BYTES;
// shape r4t4: 128 tokens x 128 rows (Q8_0: the others have no registers for it), r2t4: 128 x 64.  jl_moe_gemm_i8_...:
// the same tile per expert, and r2t2, Q6_K with the window of 32: 64 columns x 128 rows.
extern "C" __global__ __launch_bounds__(1024) void jl_gemm_i8_prep(GemmPrepArgs p) {
    __shared__ u32 lds[JL_GEMM_I8_PREP_WORDS];
    gemm_i8_prep_body(p, lds);
}
extern "C" __global__ __launch_bounds__(1024) void jl_moe_gemm_i8_prep(MoeGemmPrepArgs p) {
    __shared__ u32 lds[JL_GEMM_I8_PREP_WORDS];
    moe_gemm_i8_prep_body(p, lds);
}
template <int TYPE, bool W256, int RT, int TW>
__device__ __forceinline__ void moe_gemm_i8_tiles(const MoeGemmArgs& p) {
    constexpr u32 ROWS = 32 * RT * (4 / TW);
    const u32 rtiles = ((u32)p.nrows + ROWS - 1) / ROWS;
    const u32 ntiles = p.wl[0];
    const u32 per_mat = ntiles * rtiles, total = per_mat * (u32)p.nmat;
    for (u32 idx = blockIdx.x; idx < total; idx += gridDim.x) {   // uniform across the workgroup
        const u32 mat = idx / per_mat, rem = idx - mat * per_mat;
        const u32 t = rem / rtiles, rt = rem - t * rtiles;
        const u32 ent = p.wl[4 + p.nslots + t];
        const int e = (int)(ent & 0xFFFFu), ctile = (int)(ent >> 16);
        const u32 c_lo = p.start[e], c_hi = p.start[e + 1];
        const int slot0 = (int)(c_lo >> 5) + e;
        GemmArgs g;
        g.w = p.bank[mat] + (size_t)e * p.sheet_bytes;
        g.bq = p.bq; g.da = p.da; g.dsum = p.dsum;
        g.nrows = p.nrows; g.k = p.k; g.row_bytes = p.row_bytes;
        g.tok_pad = 32 * p.nslots;
        g.ntok = 32 * slot0 + (int)(c_hi - c_lo);    // tokens are positions in the workspace
        g.out_stride = p.nrows; g.sb_per = 0;
        g.out = p.out[mat] + ((ptrdiff_t)c_lo - (ptrdiff_t)32 * slot0) * p.nrows;   // workspace position -> column
        gemm_i8_body<TYPE, W256, RT, TW>(g, jl_smem, 32 * slot0 + 32 * TW * ctile, (int)(rt * ROWS));
        __syncthreads();   // the tile's LDS is free for the next one
    }
}
#define JL_GEMM_I8_DENSE(T, TYPE, W256, RT, TW, OCC)                                                               \
    extern "C" __global__ __launch_bounds__(256, OCC) void jl_gemm_i8_##T##_r##RT##t##TW(GemmArgs p) {             \
        gemm_i8_split_slice<TYPE, W256>(p);                                                                        \
        gemm_i8_body<TYPE, W256, RT, TW>(p, jl_smem, blockIdx.x * 32 * TW, blockIdx.y * 32 * RT * (4 / TW));       \
    }
#define JL_GEMM_I8_MOE(T, TYPE, W256, RT, TW, OCC)                                                                 \
    extern "C" __global__ __launch_bounds__(256, OCC) void jl_moe_gemm_i8_##T##_r##RT##t##TW(MoeGemmArgs p) {      \
        moe_gemm_i8_tiles<TYPE, W256, RT, TW>(p);                                                                  \
    }
#define JL_GEMM_I8_SHAPES(T, TYPE, W256, OCC)                                                                      \
    JL_GEMM_I8_DENSE(T, TYPE, W256, 2, 4, OCC) JL_GEMM_I8_MOE(T, TYPE, W256, 2, 4, OCC)
JL_GEMM_I8_SHAPES(q8_0, JL_Q8_0, false, 3) JL_GEMM_I8_SHAPES(q4k, JL_Q4_K, false, 2) JL_GEMM_I8_SHAPES(q6k, JL_Q6_K, false, 2)
JL_GEMM_I8_SHAPES(q6kw, JL_Q6_K, true, 2)
JL_GEMM_I8_MOE(q6k, JL_Q6_K, false, 2, 2, 2)
extern "C" __global__ __launch_bounds__(512) void jl_gemm_i8_q8_0_r4t8(GemmArgs p) {
    gemm_i8_split_slice<JL_Q8_0, false>(p);
    const int y = blockIdx.y;
    if (y < p.tall) gemm_i8_body<JL_Q8_0, false, 4, 8>(p, jl_smem, blockIdx.x * 256, y * 128);
    else gemm_i8_body<JL_Q8_0, false, 2, 8>(p, jl_smem, blockIdx.x * 256, 64 * (y + p.tall));   // (128 tall + 64 (y - tall))
}
JL_GEMM_I8_DENSE(q8_0, JL_Q8_0, false, 4, 4, 2) JL_GEMM_I8_MOE(q8_0, JL_Q8_0, false, 4, 4, 2)
extern "C" __global__ __launch_bounds__(512) void jl_gemm_q4k_r128(GemmArgs p) {
    gemm_q4k_body<2>(p, jl_smem, blockIdx.x * JL_GEMM_TILE, blockIdx.y * 128);
}
// the folded-scale form (kernels/gemm_q4k_fold.h): its prep, block = 1024, and its wide tile,
// grid = (tok_pad/256, ceil(nrows/128)), block = 512, dynamic LDS = JL_GEMM_FOLD_LDS_BYTES
extern "C" __global__ __launch_bounds__(1024) void jl_gemm_prep_q4k_fold(GemmPrepArgs p) {
    __shared__ u32 lds[JL_GEMM_PREP_LDS_WORDS + 32];
    gemm_prep_q4k_body<16, false, true>(p, lds);
}
extern "C" __global__ __launch_bounds__(512) void jl_gemm_q4k_fold_wide(GemmArgs p) { gemm_q4k_fold_wide_body<false>(p, jl_smem); }
// the same tile on four wavefronts of 64 tokens: block = 256, two workgroups a CU
extern "C" __global__ __launch_bounds__(256, 2) void jl_gemm_q4k_fold_wide4(GemmArgs p) { gemm_q4k_fold_wide4_body(p, jl_smem); }
extern "C" __global__ __launch_bounds__(512) void jl_gemm_q4k_wide(GemmArgs p) {
    gemm_split_slice(p);
    gemm_q4k_wide_body<false>(p, jl_smem);
}
// 128 tokens x 64 rows over the whole of K, the K halves on two groups of four wavefronts:
// grid = (tok_pad/128, ceil(nrows/64)), block = 512, dynamic LDS = JL_GEMM_K2_LDS_BYTES
extern "C" __global__ __launch_bounds__(512) void jl_gemm_q4k_k2(GemmArgs p) { gemm_q4k_k2_body<false>(p, jl_smem); }
extern "C" __global__ __launch_bounds__(512) void jl_gemm_q4k_k2_planes(GemmArgs p) { gemm_q4k_k2_body<true>(p, jl_smem); }
// The same two tiles reading the weights from packed planes (GemmArgs.pqs / pd / psc), after the
// prep in the planes' K order: no rows are restored first.
extern "C" __global__ __launch_bounds__(1024) void jl_gemm_prep_q4k_planes(GemmPrepArgs p) {
    __shared__ u32 lds[JL_GEMM_PREP_LDS_WORDS];
    gemm_prep_q4k_body<16, true>(p, lds);
}
extern "C" __global__ __launch_bounds__(256, 2) void jl_gemm_q4k_r64_planes(GemmArgs p) {
    gemm_split_slice(p);
    gemm_q4k_body<1, false, true>(p, jl_smem, blockIdx.x * JL_GEMM_TILE, blockIdx.y * 64);
}
extern "C" __global__ __launch_bounds__(512) void jl_gemm_q4k_wide_planes(GemmArgs p) {
    gemm_split_slice(p);
    gemm_q4k_wide_body<true>(p, jl_smem);
}
extern "C" __global__ __launch_bounds__(256) void jl_gemm_w16_prep_q4k(GemmW16PrepArgs p) {
    __shared__ u32 raw[32 * 37];
    gemm_w16_prep_q4k_body(p, raw);
}
extern "C" __global__ __launch_bounds__(256, 2) void jl_gemm_q4k_w16(GemmW16Args p) { gemm_q4k_w16_body(p, jl_smem); }

// ------------------------------------------------------- mixture of experts
// grid = rows, block = 64
extern "C" __global__ __launch_bounds__(64) void jl_moe_route(MoeRouteArgs p) { moe_route_body<16>(p); }
extern "C" __global__ __launch_bounds__(64) void jl_moe_route_g2(MoeRouteArgs p) { moe_route_body<2>(p); }
extern "C" __global__ __launch_bounds__(64) void jl_moe_route_g4(MoeRouteArgs p) { moe_route_body<4>(p); }
// grid = (token groups, 8 at most, experts, ceil(token groups / 8)), by_expert: (experts, token groups); block = 128; a group is
// JL_LOGITS_TOK tokens
extern "C" __global__ __launch_bounds__(128) void jl_moe_logits(MoeLogitsArgs p) {
    __shared__ float part[JL_LOGITS_TOK * 128];
    moe_logits_body<1>(p, part);
}
// more tokens: grid = (..., ceil(experts / EB), ...)
#define JL_MOE_LOGITS(NAME, EB, F16)                                                        \
    extern "C" __global__ __launch_bounds__(128, 4) void jl_moe_logits_##NAME(MoeLogitsArgs p) {  \
        __shared__ float part[2 * JL_LOGITS_TOK * 128];                                     \
        moe_logits_body<EB, F16>(p, part);                                                  \
    }
JL_MOE_LOGITS(e2, 2, false) JL_MOE_LOGITS(e2_f16, 2, true) JL_MOE_LOGITS(e4, 4, false) JL_MOE_LOGITS(e4_f16, 4, true)
JL_MOE_LOGITS(e8, 8, false) JL_MOE_LOGITS(e8_f16, 8, true)
// one workgroup of 1024 threads (n_expert <= 1024)
extern "C" __global__ __launch_bounds__(1024) void jl_moe_group(MoeGroupArgs p) {
    __shared__ u32 scount[2048];
    __shared__ __attribute__((aligned(16))) uint16_t skeys[JL_MOE_GROUP_KEYS];
    moe_group_body(p, scount, skeys);
}
// the linear-time form: a workgroup of 1024 threads for 1024 pairs, dynamic LDS = JL_MOE_GROUP2_LDS(experts)
extern "C" __global__ __launch_bounds__(1024) void jl_moe_group2(MoeGroupArgs p) { moe_group2_body(p, jl_smem); }
// grid = (ceil(k/4/256), ncols), block = 256
extern "C" __global__ __launch_bounds__(256) void jl_moe_quant(MoeQuantArgs p) { moe_quant_body(p); }
// grid = (row shares, n_expert, matrices), block = 512, dynamic LDS = 8 staged columns
#define JL_MOE_KERNEL(T, TYPE, LPR)                                                               \
    extern "C" __global__ __launch_bounds__(512) void jl_moe_matvec_##T##_l##LPR(MoeMatVecArgs p) { \
        moe_matvec_body<TYPE, LPR>(p, jl_smem);                                                   \
    }
JL_MOE_KERNEL(q4k, JL_Q4_K, 4) JL_MOE_KERNEL(q4k, JL_Q4_K, 8)
JL_MOE_KERNEL(q4k, JL_Q4_K, 16) JL_MOE_KERNEL(q4k, JL_Q4_K, 32) JL_MOE_KERNEL(q4k, JL_Q4_K, 64)
JL_MOE_KERNEL(q8_0, JL_Q8_0, 4) JL_MOE_KERNEL(q8_0, JL_Q8_0, 8)
JL_MOE_KERNEL(q8_0, JL_Q8_0, 16) JL_MOE_KERNEL(q8_0, JL_Q8_0, 32) JL_MOE_KERNEL(q8_0, JL_Q8_0, 64)
JL_MOE_KERNEL(q6k, JL_Q6_K, 4) JL_MOE_KERNEL(q6k, JL_Q6_K, 8)
JL_MOE_KERNEL(q6k, JL_Q6_K, 16) JL_MOE_KERNEL(q6k, JL_Q6_K, 32) JL_MOE_KERNEL(q6k, JL_Q6_K, 64)
// banks of packed planes: grid = (ceil(nrows/64), n_expert, matrices), block = 64 * wavefronts (<= 8),
// dynamic LDS = wavefronts * JL_MOEP_TB * 256
extern "C" __global__ __launch_bounds__(512) void jl_moe_matvec_planes_q4k(MoePlanesArgs p) {
    moe_matvec_planes_body(p, jl_smem);
}
// a matvec a routed column: grid = (row groups, columns, matrices), block = 1024, dynamic LDS as jl_matvec_multi_*; the down
// projections of a row's pairs: grid = (row groups, rows), block <= 1024, 128 bytes of LDS behind the staging area
#define JL_MOE_GATHER_L(T, TYPE, L)                                                                                                            \
    extern "C" __global__ __launch_bounds__(1024) void jl_moe_gather_##T##_l##L(MoeGatherArgs p) { moe_gather_body<TYPE, 0, L>(p, jl_smem); }         \
    extern "C" __global__ __launch_bounds__(1024) void jl_moe_gather_##T##_a_l##L(MoeGatherArgs p) { moe_gather_body<TYPE, JL_PRE_ACT, L>(p, jl_smem); } \
    extern "C" __global__ __launch_bounds__(1024) void jl_moe_gather_##T##_down_l##L(MoeGatherDownArgs p) { moe_gather_down_body<TYPE, L>(p, jl_smem); }
#define JL_MOE_GATHER(T, TYPE) JL_MOE_GATHER_L(T, TYPE, 8) JL_MOE_GATHER_L(T, TYPE, 16) JL_MOE_GATHER_L(T, TYPE, 32) JL_MOE_GATHER_L(T, TYPE, 64)
JL_MOE_GATHER(q4k, JL_Q4_KF) JL_MOE_GATHER(q8_0, JL_Q8_0) JL_MOE_GATHER(q8_0p, JL_Q8_0P) JL_MOE_GATHER(q6k, JL_Q6_KS) JL_MOE_GATHER(q6kw, JL_Q6_KW)
// over planes: grid = (ceil(nrows/RW), pairs, 2) and (ceil(nrows/RW), rows), block <= 1024, dynamic LDS = JL_PK_LDS_BYTES
#define JL_MOE_PLANES_GATHER(RW)                                                                                          \
    extern "C" __global__ __launch_bounds__(1024) void jl_moe_planes_gather_w##RW(MoePlanesGatherArgs p) {                \
        moe_planes_gather_body<RW, 1>(p, jl_smem);                                                                        \
    }                                                                                                                     \
    extern "C" __global__ __launch_bounds__(1024) void jl_moe_planes_down_w##RW(MoePlanesDownArgs p) {                    \
        moe_planes_down_body<RW, 2>(p, jl_smem);                                                                          \
    }
JL_MOE_PLANES_GATHER(16) JL_MOE_PLANES_GATHER(32) JL_MOE_PLANES_GATHER(64)
// experts of some tens of columns (kernels/moe_cols.h): prep grid = ceil(records * k/256 / 16); matrices: dynamic LDS = JL_MC_LDS_BYTES
#define JL_MOE_COLS(T, KO)                                                                                                         \
    extern "C" __global__ __launch_bounds__(256) void jl_moe_cols_prep_##T(MoeColsPrepArgs p) { moe_cols_prep_body<KO>(p); }      \
    extern "C" __global__ __launch_bounds__(256, 2) void jl_moe_cols_##T(MoeColsArgs p) { moe_cols_body<KO>(p, jl_smem); }
JL_MOE_COLS(q4k, 0) JL_MOE_COLS(q4k_planes, 1) JL_MOE_COLS(q6k, 2)
// grid = (ceil(n_embd/4/256), rows), block = 256
extern "C" __global__ __launch_bounds__(256) void jl_moe_combine(MoeCombineArgs p) { moe_combine_body(p); }

// ------------------------------------------------------------------- MXFP4
// grid = (ceil(ntok/128), ceil(nrows/128), K splits), block = 256, dynamic LDS = 4 stages of 128 x 272 B
extern "C" __global__ __launch_bounds__(256) void jl_mxfp4_prep(MxPrepArgs p) {
    __shared__ u32x4 lds[32 * 33];
    mx_prep_body(p, lds);
}
extern "C" __global__ __launch_bounds__(256) void jl_moe_gemm_prep(MoeGemmPrepArgs p) {
    __shared__ u32 lds[JL_GEMM_PREP_LDS_WORDS];
    moe_gemm_prep_body<false>(p, lds);
}
extern "C" __global__ __launch_bounds__(256) void jl_moe_gemm_prep_planes(MoeGemmPrepArgs p) {
    __shared__ u32 lds[JL_GEMM_PREP_LDS_WORDS];
    moe_gemm_prep_body<true>(p, lds);
}
extern "C" __global__ __launch_bounds__(256, 2) void jl_moe_gemm_q4k(MoeGemmArgs p) { moe_gemm_q4k_body(p, jl_smem); }
// Sixteen columns a group, weights from HBM straight into matrix operands.
// prep: grid = ceil(ncols/4), block = 256; main (CH super-blocks a step): grid = 8 * ceil(n_expert/8) * row blocks * matrices,
// block = 64 * nwaves (<= 512), dynamic LDS = (k/256) * JL_MOE_G16_SB_WORDS * 4
extern "C" __global__ __launch_bounds__(256) void jl_moe_g16_prep(MoeG16PrepArgs p) {
    __shared__ u32 lds[4 * 72];
    moe_g16_prep_body<0>(p, lds);
}
extern "C" __global__ __launch_bounds__(256) void jl_moe_g16_prep_planes(MoeG16PrepArgs p) {
    __shared__ u32 lds[4 * 72];
    moe_g16_prep_body<1>(p, lds);
}
// _c: fragments from the prep kernel's workspace; _f / _g: the columns (plain / silu(x) * x2) quantized by
// the kernel itself; _d: groups of 32 columns (two token tiles); g16p: the sheets are packed planes
#define JL_MOE_G16_FORMS(NAME, KO, CH)                                                                                          \
    extern "C" __global__ __launch_bounds__(512) void jl_moe_##NAME##_c##CH(MoeG16Args p) { moe_g16_body<CH, 0, KO>(p, jl_smem); } \
    extern "C" __global__ __launch_bounds__(512) void jl_moe_##NAME##_f##CH(MoeG16Args p) { moe_g16_body<CH, 1, KO>(p, jl_smem); } \
    extern "C" __global__ __launch_bounds__(512) void jl_moe_##NAME##_g##CH(MoeG16Args p) { moe_g16_body<CH, 2, KO>(p, jl_smem); } \
    extern "C" __global__ __launch_bounds__(512) void jl_moe_##NAME##_d##CH(MoeG16Args p) { moe_g16_body<CH, 0, KO, 2>(p, jl_smem); }
#define JL_MOE_G16_KERNEL(CH) JL_MOE_G16_FORMS(g16, 0, CH) JL_MOE_G16_FORMS(g16p, 1, CH)
JL_MOE_G16_KERNEL(1) JL_MOE_G16_KERNEL(2) JL_MOE_G16_KERNEL(3)
// Experts with many columns: the prefill GEMM's 128-token x 64-row tile placed per expert.  An
// expert's column groups are consecutive slots of the prepared workspace, so to the tile they
// are a token range; columns past the expert's last are computed and not stored.  The
// workgroups stride over (row tile, column tile of the work list, matrix), so none is empty.
// grid = up to two workgroups a CU, block = 256, dynamic LDS as jl_gemm_q4k_r64.
// PL (Q4_K): the banks are packed planes, an expert's sheet a plane set of its own or a row range
// of the bank's (MoeGemmArgs.pqs ...); the tile is the plane form of the prefill GEMM's.
template <bool PL>
__device__ __forceinline__ void moe_gemm_tiles(const MoeGemmArgs& p) {
    const u32 rtiles = (u32)(p.nrows + 63) / 64;
    const u32 ntiles = p.wl[0];
    const u32 per_mat = ntiles * rtiles, total = per_mat * (u32)p.nmat;
    for (u32 idx = blockIdx.x; idx < total; idx += gridDim.x) {   // uniform across the workgroup
        const u32 mat = idx / per_mat, rem = idx - mat * per_mat;
        const u32 t = rem / rtiles, rt = rem - t * rtiles;
        const u32 ent = p.wl[4 + p.nslots + t];
        const int e = (int)(ent & 0xFFFFu), ctile = (int)(ent >> 16);
        const u32 c_lo = p.start[e], c_hi = p.start[e + 1];
        const int ncol = (int)(c_hi - c_lo);
        const int slot0 = (int)(c_lo >> 5) + e;
        GemmArgs g;
        if (PL) {
            const size_t ew = (size_t)e * p.sheet_words;
            g.pqs = p.pqs[mat] + ew; g.pd = p.pd[mat] + ew; g.psc = p.psc[mat] + ew;
            g.prow0 = e * p.row_step; g.pstride = p.pstride; g.psb0 = 0;
            g.w = nullptr;
        } else {
            g.w = p.bank[mat] + (size_t)e * p.sheet_bytes;
        }
        g.bq = p.bq; g.da = p.da;
        g.nrows = p.nrows; g.k = p.k; g.row_bytes = p.row_bytes;
        g.tok_pad = 32 * p.nslots;
        g.ntok = 32 * slot0 + ncol;                  // tokens are positions in the workspace
        g.out_stride = p.nrows; g.sb_per = 0;
        g.out = p.out[mat] + ((ptrdiff_t)c_lo - (ptrdiff_t)32 * slot0) * p.nrows;   // workspace position -> column
        gemm_q4k_body<1, true, PL>(g, jl_smem, 32 * slot0 + 128 * ctile, (int)rt * 64);
        __syncthreads();   // the tile's LDS is free for the next one
    }
}
extern "C" __global__ __launch_bounds__(256, 2) void jl_moe_gemm_r64(MoeGemmArgs p) { moe_gemm_tiles<false>(p); }
extern "C" __global__ __launch_bounds__(256, 2) void jl_moe_gemm_r64_planes(MoeGemmArgs p) { moe_gemm_tiles<true>(p); }
// grid = 1, block = 1024
extern "C" __global__ __launch_bounds__(1024) void jl_moe_worklist(MoeWorklistArgs p) {
    __shared__ u32 tot[16];
    moe_worklist_body(p, tot);
}
extern "C" __global__ __launch_bounds__(512) void jl_mxfp4_gemm(MxGemmArgs p) { mx_gemm_body<4>(p, jl_smem); }
extern "C" __global__ __launch_bounds__(512) void jl_mxfp4_gemm_r96(MxGemmArgs p) { mx_gemm_body<3>(p, jl_smem); }
extern "C" __global__ __launch_bounds__(256) void jl_sum_parts(SumPartsArgs p) { sum_parts_body(p); }
// grid = ceil(nrows/4), block = 256: one wavefront per row, ntok <= 8
extern "C" __global__ __launch_bounds__(256) void jl_mxfp4_matvec(MxGemmArgs p) { mx_matvec_body(p); }
// one token, _b<blocks a lane holds>: grid = ceil(nrows / (4 wavefronts * 4 rows)), block = 256
extern "C" __global__ __launch_bounds__(256) void jl_mxfp4_matvec1_b1(MxGemmArgs p) { mx_matvec1_body<1>(p); }
extern "C" __global__ __launch_bounds__(256) void jl_mxfp4_matvec1_b2(MxGemmArgs p) { mx_matvec1_body<2>(p); }
extern "C" __global__ __launch_bounds__(256) void jl_mxfp4_matvec1_b3(MxGemmArgs p) { mx_matvec1_body<3>(p); }
// ntok <= 8 over packed planes, _r<rows a workgroup>: grid = ceil(nrows/R), block = 64 * nwaves,
// LDS = nwaves * 8 * 64 floats
extern "C" __global__ __launch_bounds__(1024) void jl_mxfp4_matvec_planes_r64(MxPlanesArgs p) {
    mx_planes_matvec_body<64, 6>(p, (float*)jl_smem);
}
extern "C" __global__ __launch_bounds__(1024) void jl_mxfp4_matvec_planes_r32(MxPlanesArgs p) {
    mx_planes_matvec_body<32, 3>(p, (float*)jl_smem);
}
extern "C" __global__ __launch_bounds__(1024) void jl_mxfp4_matvec_planes_r16(MxPlanesArgs p) {
    mx_planes_matvec_body<16, 2>(p, (float*)jl_smem);
}
// MXFP4 planes x bf16 beyond a handful of tokens: prep grid = (ceil(ceil(k/64) / 4), tok_pad/32),
// block = 256; GEMM grid = 8 * ceil(tiles of 64 x 64 / 8), block = 256, dynamic LDS = 64 KiB
extern "C" __global__ __launch_bounds__(256) void jl_mxfp4_planes_prep(MxPlanesPrepArgs p) { mx_planes_prep_body(p); }
extern "C" __global__ __launch_bounds__(256, 2) void jl_mxfp4_planes_gemm(MxPlanesGemmArgs p) {
    mx_planes_gemm_body<2>(p, (float*)jl_smem);
}
extern "C" __global__ __launch_bounds__(256, 2) void jl_mxfp4_planes_gemm_r96(MxPlanesGemmArgs p) {
    mx_planes_gemm_body<3>(p, (float*)jl_smem);
}
// the opt-in block-scaled form over packed planes: prep grid = (ceil(ceil(k/64) / 4), tok_pad/32),
// block = 256; GEMM grid = 8 * ceil(tiles of 64 x 64 / 8), block = 256, dynamic LDS = 64 KiB
extern "C" __global__ __launch_bounds__(256) void jl_mxfp4_scaled_prep(MxScaledPrepArgs p) { mx_scaled_prep_body(p); }
extern "C" __global__ __launch_bounds__(256, 2) void jl_mxfp4_scaled_gemm(MxScaledGemmArgs p) {
    mx_scaled_gemm_body(p, (float*)jl_smem);
}
// A few tokens: prep grid = (ceil(k/128), tiles of 16 tokens), block = 256; kernel grid = (ceil(nrows/16), chunks),
// block = 512; _t<NT>: up to 16 NT tokens, _c<NT>: chunks of 16 NT of more
extern "C" __global__ __launch_bounds__(256) void jl_mxfp4_prep_few(MxPrepArgs p) { mx_prep_few_body(p); }
#define JL_MX_FEW_KERNEL(NAME, NT, PL, CHUNKS)                                                 \
    extern "C" __global__ __launch_bounds__(512) void jl_mxfp4_few_##NAME(MxGemmArgs p) {      \
        __shared__ __attribute__((aligned(16))) float part[8 * NT * 256];                      \
        mx_few_body<NT, PL, CHUNKS>(p, part);                                                  \
    }
JL_MX_FEW_KERNEL(t1, 1, false, false) JL_MX_FEW_KERNEL(t2, 2, false, false)
JL_MX_FEW_KERNEL(t3, 3, false, false) JL_MX_FEW_KERNEL(t4, 4, false, false)
JL_MX_FEW_KERNEL(c3, 3, false, true) JL_MX_FEW_KERNEL(c4, 4, false, true)
JL_MX_FEW_KERNEL(planes_t1, 1, true, false) JL_MX_FEW_KERNEL(planes_t2, 2, true, false)
JL_MX_FEW_KERNEL(planes_t3, 3, true, false) JL_MX_FEW_KERNEL(planes_t4, 4, true, false)
JL_MX_FEW_KERNEL(planes_c3, 3, true, true) JL_MX_FEW_KERNEL(planes_c4, 4, true, true)
// the same in one launch: kernel grid = (ceil(nrows / (16 RT)), chunks of 16 NT tokens), block = 512, dynamic LDS = JL_MX_ONE_LDS(k, NT)
#define JL_MX_ONE_KERNEL(NT, RT)                                                                                                                       \
    extern "C" __global__ __launch_bounds__(512) void jl_mxfp4_one_t##NT##r##RT(MxGemmArgs p) { mx_one_body<NT, RT, false>(p, jl_smem); }               \
    extern "C" __global__ __launch_bounds__(512) void jl_mxfp4_one_planes_t##NT##r##RT(MxGemmArgs p) { mx_one_body<NT, RT, true>(p, jl_smem); }
JL_MX_ONE_KERNEL(1, 1) JL_MX_ONE_KERNEL(2, 1) JL_MX_ONE_KERNEL(3, 1) JL_MX_ONE_KERNEL(4, 1)
JL_MX_ONE_KERNEL(1, 2) JL_MX_ONE_KERNEL(2, 2) JL_MX_ONE_KERNEL(3, 2) JL_MX_ONE_KERNEL(4, 2)

// A Q4_K weight is d * sc * q - dmin * m with sc, m <= 63 and q <= 15: a super-block whose
// |d| * 945 + |dmin| * 63 passes the largest f16 cannot be folded (a NaN or infinite scale
// fails the comparison and is flagged too).  grid = ceil(nblocks/256), block = 256.
extern "C" __global__ __launch_bounds__(256) void jl_q4k_fold_range(FoldRangeArgs a) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.nblocks) return;
    const u32 h = *(const u32*)(a.w + i * 144);
    const float d = fabsf(half_bits_to_f32((uint16_t)(h & 0xFFFF))), dmin = fabsf(half_bits_to_f32((uint16_t)(h >> 16)));
    if (!(d * 945.f + dmin * 63.f <= 65504.f)) atomicOr(a.flag, 1u);
}

// A dense feed-forward block's pieces between its prefill GEMMs: g = silu(g) * u, n a multiple of four;
// resid[r] += wt[r] * y[r] (wt null: 1), grid = (ceil(n_embd / 4 / 256), rows).
extern "C" __global__ __launch_bounds__(256) void jl_silu_mul(float* __restrict__ g, const float* __restrict__ u, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i * 4 >= n) return;
    const f32x4 a = ((const f32x4*)g)[i], b = ((const f32x4*)u)[i];
    ((f32x4*)g)[i] = f32x4{silu_f32(a.x) * b.x, silu_f32(a.y) * b.y, silu_f32(a.z) * b.z, silu_f32(a.w) * b.w};
}
extern "C" __global__ __launch_bounds__(256) void jl_add_rows(float* __restrict__ resid, const float* __restrict__ y,
                                                              const float* __restrict__ wt, int n_embd) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i * 4 >= n_embd) return;
    const size_t o = (size_t)blockIdx.y * n_embd / 4 + i;
    const float w = wt ? wt[blockIdx.y] : 1.0f;
    const f32x4 v = ((const f32x4*)y)[o];
    f32x4 r = ((f32x4*)resid)[o];
    r.x += w * v.x; r.y += w * v.y; r.z += w * v.z; r.w += w * v.w;
    ((f32x4*)resid)[o] = r;
}

// ------------------------------------------------- host-pointer calls: operands and results
// A host-pointer call's activations and results are tens of kilobytes: what a copy through the runtime costs
// (two pageable copies and a stream wait: 31 us round a 5 us matvec) is latency, not bytes.  jl_host_in copies
// the operands from pinned host memory, 16 bytes a lane, in stream order with the matrix work; results are
// stored to pinned host memory by the kernels that make them, and jl_host_done behind them raises the call's
// number there, which the calling thread watches.  (A kernel that copied the results out and raised the number
// itself took 4.7 us for 16 KB; this one takes an empty launch.)
extern "C" __global__ __launch_bounds__(256) void jl_host_in(const u32x4* __restrict__ src, u32x4* __restrict__ dst, u32 n) {
    for (u32 i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) dst[i] = src[i];
}
extern "C" __global__ __launch_bounds__(64) void jl_host_done(u32* flag, u32 number) {
    if (threadIdx.x == 0) __hip_atomic_store(flag, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ------------------------------------------------------------------ probes
// What one launch costs on this machine before any arithmetic: jl_probe_read streams nvec
// 16-byte vectors with every thread keeping eight loads in flight and folds them into a word
// that is stored only if it matches a value random data never gives; jl_probe_empty returns
// at once.  Timed by the benchmark beside the kernels they bound.  grid and block are free.
extern "C" __global__ __launch_bounds__(1024) void jl_probe_read(const u32x4* __restrict__ src, size_t nvec,
                                                                  u32* __restrict__ sink) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    u32x4 acc = u32x4{0u, 0u, 0u, 0u};
    for (; i + 7 * stride < nvec; i += 8 * stride) {
        u32x4 v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = __builtin_nontemporal_load(src + i + j * stride);
#pragma unroll
        for (int j = 0; j < 8; j++) acc ^= v[j];
    }
    for (; i < nvec; i += stride) acc ^= __builtin_nontemporal_load(src + i);
    if ((acc.x ^ acc.y ^ acc.z ^ acc.w) == 0x9e3779b9u && sink) sink[0] = acc.x;
}
// What the matrix cores deliver with nothing to wait for: every wavefront issues `iters` rounds
// of four independent 32x32x16 f16 matrix instructions on registers (jl_probe_mfma), and the
// same with five f32 multiply-adds issued after each of them (jl_probe_mfma_v5, the vector load
// of the prefill GEMM's loop).  2 * 32 * 32 * 16 flops an instruction.
template <int V>
__device__ __forceinline__ void probe_mfma_body(size_t iters, u32* sink) {
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    typedef float f16v __attribute__((ext_vector_type(16)));
    h8 a, b;
#pragma unroll
    for (int i = 0; i < 8; i++) { a[i] = (_Float16)(int)(threadIdx.x & 3); b[i] = (_Float16)(int)(threadIdx.x & 1); }
    f16v acc[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[j][e] = 0.f;
    float v[5];
#pragma unroll
    for (int i = 0; i < 5; i++) v[i] = (float)threadIdx.x + (float)i;
    const float c = __uint_as_float(0x3f7ff000u + (threadIdx.x & 1)), d = 0.5f;
    for (size_t it = 0; it < iters; it++) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc[j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < V; i++) v[i] = fmaf(v[i], c, d);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (V > 0) __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
        }
    }
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) s += acc[j][e];
#pragma unroll
    for (int i = 0; i < 5; i++) s += v[i];
    if (sink && __float_as_uint(s) == 0x9e3779b9u) sink[0] = 1;
}
extern "C" __global__ __launch_bounds__(1024) void jl_probe_mfma(const u32x4* __restrict__, size_t iters, u32* __restrict__ sink) {
    probe_mfma_body<0>(iters, sink);
}
extern "C" __global__ __launch_bounds__(1024) void jl_probe_mfma_v5(const u32x4* __restrict__, size_t iters, u32* __restrict__ sink) {
    probe_mfma_body<5>(iters, sink);
}
extern "C" __global__ __launch_bounds__(1024) void jl_probe_empty(const u32x4* __restrict__, size_t, u32* __restrict__) {}
// Holds the stream for `ticks` ticks of the 100 MHz constant clock and touches no memory: what a
// benchmark enqueues in front of a timed window so that the window's launches are all queued
// before the first one starts.  One wavefront; the wait is bounded by the clock, so it always ends.
extern "C" __global__ __launch_bounds__(64) void jl_probe_wait(const u32x4* __restrict__, size_t ticks, u32* __restrict__) {
    const uint64_t t0 = wall_clock64();
    while (wall_clock64() - t0 < ticks) __builtin_amdgcn_s_sleep(8);
}
