// Few tokens (or few columns an expert) on the int8 matrix cores: Q8_0, Q6_K and Q4_K, GGUF rows or
// packed planes, any activation window.
//
// The weights are read once, at whatever pace memory gives, and everything else has to fit under
// that.  v_mfma_i32_16x16x32_i8 takes a quantized weight as it is -- no conversion to f16, no scale
// multiplied in -- so what is left for the vector unit is the unpacking of nibbles (none for Q8_0)
// and, for every 16 rows x 16 tokens x 32 of K, the conversion of four int32 sums and their two
// scales: 18 to 23 vector instructions a matrix instruction.  A 128-token tile (gemm_i8.h) spends
// the same on 12 tokens as on 128 and adds K slices in a second launch.  Counters at 16 tokens (14336 x 4096,
// Q6_K 4096 x 14336 at 12; kernel alone, traced): Q4_K rows 12.8 us and planes 11.6, Q6_K rows 15.6, Q8_0
// rows 14.9; the vector unit issues 21 to 33 % of the time, the matrix cores 4 to 7 %, wavefronts wait for
// data 38 to 49 %, L1 answers 8.6 to 14.8 of 42 to 51 thousand cycles.  What is left is the serial chain of a
// wavefront's few steps (a super-block's weights, through LDS, matrix instruction, scales) behind the prep's launch.
//
//   * A workgroup owns 16 RT rows and up to 16 NT columns; its wavefronts split K (wavefront w takes
//     super-blocks w, w + nwaves, ...: a row's bytes are asked for side by side) and their partial tiles
//     are added through LDS in wavefront order: one launch after the prep.
//   * More tokens than a workgroup's columns: groups of tgroup token tiles on grid y, each of which reads the weights
//     again (from L2 while the groups of a row tile run together).  64 tokens in smaller groups where more workgroups are
//     worth it (1.025 over 17 to 64 tokens), and beyond 64 where the estimates put it before the tiles: 208 drawn
//     matmuls of 60 to 780 tokens 1.175 times as fast as without.
//   * L1 would be the next bound after memory: a vector load costs it one access for every 64-byte line that a
//     quad of ADJACENT lanes touches, so the matrix operand's own lane order (lane % 16 = row) would cost 64
//     accesses a 1 KiB load where 16 do.  GGUF rows are therefore loaded along the row, 16 bytes a lane, and
//     change lanes through the wavefront's own corner of LDS; over planes a lane loads one word of RT
//     consecutive rows (so row tile j of a workgroup is rows RT r + j), and the four header words of a Q4_K
//     super-block are one load by the four lane groups.
//   * Lane (r = lane % 16, g = lane / 16) holds, for a block of 32, eight values of row r, in an order of
//     the weights' own (jl_few_order), and the prep lays the int8 activations out to match: four blocks'
//     values in two 16-byte loads, their scales in one.
//   * D has rows on registers and tokens on lanes, so a token's scale is one value a lane, and the
//     rows' scales, which every lane of the row's column needs, take a turn through the wavefront's
//     own corner of LDS (one 16-byte read a block for all NT token tiles).
//   * Q6_K: a block of 32 has two sub-scales; the matrix instruction runs twice with the other
//     half's lanes zeroed, and both sums meet their integer scales in v_mad_i32_i24.  The weight is
//     4 (q - 32) as an int8 (six bits at the top of the byte, sign bit flipped), the 1/4 goes into d.
//   * Q4_K: the minimums meet d_a * (sum of the block's a).
//   * With the k-quant window (W256) one d_a covers a super-block: Q6_K and Q4_K sum integers (sc * dot,
//     m * sum of a) in v_mad_i32_i24 over the super-block and turn to f32 once.
//
// start / slots: column group g of expert e is slot start[e]/16 + e + g, as in the mixture's other
// kernels; a plain matrix is one expert whose columns are the tokens (start null).
#pragma once
#include "args.h"
#include "common.h"
#include "quantize.h"

#pragma clang fp contract(off)

// Word `w` (elements 4w.. of a block of 32) of a token's int8 block goes to lane group g, half h.
// order 0: GGUF rows, Q8_0 planes (lane group g holds elements 8g..8g+7); order 1: Q4_K planes (4g.. and
// 16 + 4g..); order 2: Q6_K planes (run of 16 g/2: 4(g%2).. and 8 + 4(g%2)..)
__device__ __forceinline__ void jl_few_order(int order, int w, int& g, int& h) {
    if (order == 0) { g = w >> 1; h = w & 1; }
    else if (order == 1) { g = w & 3; h = w >> 2; }
    else { g = (w >> 2) * 2 + (w & 1); h = (w >> 1) & 1; }
}

// One wavefront per (column, 256 elements): quantize, lay out.  K past the end is zero (values and
// scales) up to a multiple of 128; columns that fill no group's last slot keep what was there (their
// results are not stored).  grid = (ceil(k / 256), ceil(ncols / 4)), block = 256.
__device__ __forceinline__ void few_i8_prep_body(const FewI8PrepArgs& args) {
    FewI8PrepArgs p = args;
    JL_NOW(p.x, p.x2, p.src, p.start, p.bq, p.da, p.ds, p.k, p.per, p.ncols, p.n_expert, p.nslots, p.nch, p.order, p.isum);
    p.x = as_global(p.x); p.x2 = as_global(p.x2); p.src = as_global(p.src); p.start = as_global(p.start);
    p.bq = as_global(p.bq); p.da = as_global(p.da); p.ds = as_global(p.ds);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const u32 c = blockIdx.y * 4 + wave;
    if (c >= (u32)p.ncols) return;   // whole wavefronts, no barrier below
    const int ch = blockIdx.x, g4 = ch * 64 + lane;
    // (a column of no expert -- the grouping leaves ids that no expert has out -- has no source row either)
    const u32 ncols = p.start ? p.start[p.n_expert] : (u32)p.ncols;
    u32 row = p.src ? p.src[c] : c;
    if (c >= ncols) row = 0;
    const bool live = g4 < p.k / 4;
    const int gc = live ? g4 : p.k / 4 - 1;
    f32x4 v = ((const f32x4*)(p.x + row * (size_t)p.k))[gc];
    f32x4 u = {0.f, 0.f, 0.f, 0.f};
    if (p.x2) u = ((const f32x4*)(p.x2 + row * (size_t)p.k))[gc];
    if (c >= ncols) return;   // the whole wavefront
    u32 slot = c >> 4, i = c & 15;
    if (p.start) {
        // the column's expert: the last whose first column is not past it
        u32 cnt = 0, lo = 0;
        for (int base = 0; base <= p.n_expert; base += 64) {
            const int idx = base + lane;
            const u32 s = idx <= p.n_expert ? p.start[idx] : 0xFFFFFFFFu;
            const bool le = s <= c;
            cnt += (u32)__builtin_popcountll(__ballot(le));
            lo = max(lo, le ? s : 0u);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) lo = max(lo, (u32)__shfl_xor((int)lo, off, 64));
        slot = (lo >> 4) + (cnt - 1) + ((c - lo) >> 4);
        i = (c - lo) & 15;
    }
    if (p.x2) v = f32x4{silu_f32(v.x) * u.x, silu_f32(v.y) * u.y, silu_f32(v.z) * u.z, silu_f32(v.w) * u.w};
    if (!live) v = f32x4{0.f, 0.f, 0.f, 0.f};
    const u32 m = max(max(abs_bits(v.x), abs_bits(v.y)), max(abs_bits(v.z), abs_bits(v.w)));
    const u32 amax = p.per == 8 ? wave_amax_256(m) : window_amax(m, p.per);
    float d;
    i32 s16;
    const u32 q = quantize4(v, amax, d, s16);
    const i32 s32 = s16 + dpp_i32<JL_DPP_ROW_HALF_MIRROR, 0xf>(0, s16);
    const int ks = (lane >> 3) & 3, c128 = ch * 2 + (lane >> 5);
    if (c128 >= p.nch) return;
    int g, h;
    jl_few_order(p.order, lane & 7, g, h);
    const size_t at = (size_t)c128 * p.nslots + slot;
    p.bq[((at * 2 + (ks >> 1)) * 64 + 16 * g + i) * 4 + (ks & 1) * 2 + h] = q;
    if ((lane & 7) == 0) {
        if (!live) d = 0.f;
        p.da[(at * 16 + i) * 4 + ks] = d;
        if (p.ds) p.ds[(at * 16 + i) * 4 + ks] = p.isum ? __uint_as_float((u32)s32) : d * (float)s32;
    }
}

// Uniform base + a lane's 32-bit byte offset, the addressing form that costs no vector instruction.
// (few_pin keeps the compiler from folding the offset into 64-bit lane addresses outside the loop.)
template <class T> __device__ __forceinline__ T few_ld(const void* base, u32 off) { return *(const T*)((const uint8_t*)base + off); }
__device__ __forceinline__ void few_pin(u32& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void few_lds_fence() {   // a wavefront's own LDS operations complete in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// X's odd sixteens of lanes <-> Y's even ones.
__device__ __forceinline__ void swap16(u32& x, u32& y) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    x = r[0]; y = r[1];
}

// One word of RT consecutive rows of a plane (4-byte aligned).
struct __attribute__((packed, aligned(4))) u32x2_a4 { u32x2 v; };
template <int RT> __device__ __forceinline__ void few_words(const void* base, u32 off, u32* o) {
    if constexpr (RT == 4) {
        const u32x4 v = few_ld<u32x4_a4>(base, off).v;
        o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    } else if constexpr (RT == 2) {
        const u32x2 v = few_ld<u32x2_a4>(base, off).v;
        o[0] = v.x; o[1] = v.y;
    } else {
        o[0] = few_ld<u32>(base, off);
    }
}

struct FewMat { const uint8_t* w; const u32 *qs, *dp, *sp; };   // the expert's sheet

// ---------------------------------------------------------------- what a lane computes with
// A row tile's eight-value groups of a half super-block (four blocks of 32), before the cheap decode of one
// block: Q8_0 the values, Q4_K and Q6_K the nibble words (rows: pairs of blocks share them) and bit pairs.
template <int TYPE, bool PL> struct FewR;
template <bool PL> struct FewR<JL_Q8_0, PL> { u32 v[4][2]; };
template <> struct FewR<JL_Q4_K, false> { u32 v[2][2]; };
template <> struct FewR<JL_Q4_K, true> { u32 v[4]; };
template <> struct FewR<JL_Q6_K, false> { u32 v[2][2], h[2]; };
template <> struct FewR<JL_Q6_K, true> { u32 v[4], h[4]; };

// The lane's eight int8 weights of block s (0..3).
template <int TYPE, bool PL>
__device__ __forceinline__ u32x2 few_decode(const FewR<TYPE, PL>& R, int s, int g) {
    if constexpr (TYPE == JL_Q8_0) {
        return u32x2{R.v[s][0], R.v[s][1]};
    } else if constexpr (TYPE == JL_Q4_K) {
        const u32 M = 0x0F0F0F0Fu;
        if constexpr (PL) return u32x2{R.v[s] & M, (R.v[s] >> 4) & M};
        else {
            const u32 x = R.v[s >> 1][0], y = R.v[s >> 1][1];
            return (s & 1) ? u32x2{(x >> 4) & M, (y >> 4) & M} : u32x2{x & M, y & M};
        }
    } else {
        const u32 L = 0x3C3C3C3Cu, T = 0xC0C0C0C0u, S = 0x80808080u;
        if constexpr (PL) {
            const u32 w = R.v[s], h = R.h[s];
            const int sh = 2 * (g & 1);
            return u32x2{(((w << 2) & L) | ((h << (6 - sh)) & T)) ^ S, (((w >> 2) & L) | ((h << (2 - sh)) & T)) ^ S};
        } else {
            const u32 x = R.v[s & 1][0], y = R.v[s & 1][1];
            const int sh = 6 - 2 * s;
            return u32x2{(((s >= 2 ? x >> 2 : x << 2) & L) | ((R.h[0] << sh) & T)) ^ S,
                         (((s >= 2 ? y >> 2 : y << 2) & L) | ((R.h[1] << sh) & T)) ^ S};
        }
    }
}

// The scales of a lane's row for lane group g's block (runs 2g, 2g + 1), into the tile's scale area:
// Q8_0: [4 blocks][16] d;  Q4_K: [4][16] d*sc, [4][16] dmin*m, or with W256 the integers sc and m, [16] d, [16] dmin;
// Q6_K: [8 runs][16] int32 sc, [16] d/4.
__device__ __forceinline__ void few_put_q8(u32 d, int g, int r, float* lds) { lds[g * 16 + r] = half_bits_to_f32((uint16_t)d); }
template <bool W256>
__device__ __forceinline__ void few_put_q4k(u32 dd, u32 sc, u32 m, int g, int r, float* lds) {
    const float d = half_bits_to_f32((uint16_t)(dd & 0xFFFF)), dmin = half_bits_to_f32((uint16_t)(dd >> 16));
    if constexpr (W256) {
        lds[g * 16 + r] = __uint_as_float(sc);
        lds[64 + g * 16 + r] = __uint_as_float(m);
        lds[128 + r] = d;
        lds[144 + r] = dmin;
    } else {
        lds[g * 16 + r] = d * (float)sc;
        lds[64 + g * 16 + r] = dmin * (float)m;
    }
}
__device__ __forceinline__ void few_put_q6k(u32 d, i32 s0, i32 s1, int g, int r, float* lds) {
    i32* is = (i32*)lds;
    is[(2 * g) * 16 + r] = s0;
    is[(2 * g + 1) * 16 + r] = s1;
    lds[128 + r] = half_bits_to_f32((uint16_t)(d & 0xFFFF)) * 0.25f;
}

__device__ __forceinline__ i32x4 mfma_i8(u32x2 a, u32x2 b, i32x4 c) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, a), __builtin_bit_cast(long, b), c, 0, 0, 0);
}

// One slot's activations of four blocks: int8, scales, and (Q4_K) scale * sum or the sum itself (W256).
template <int TYPE, bool W256> struct FewA {
    u32x4 a[2];
    f32x4 da, ds;
    float d1;
    __device__ __forceinline__ void load(const FewI8Args& p, int c128, u32 slot, u32 va, u32 vd) {
        const size_t at = (size_t)(u32)(c128 * p.nslots) + slot;
        a[0] = few_ld<u32x4>(p.bq + at * 512, va);
        a[1] = few_ld<u32x4>(p.bq + at * 512 + 256, va);
        if constexpr (W256) d1 = few_ld<float>(p.da + at * 64, vd);
        else da = few_ld<f32x4>(p.da + at * 64, vd);
        if constexpr (TYPE == JL_Q4_K) ds = few_ld<f32x4>(p.ds + at * 64, vd);
    }
    __device__ __forceinline__ u32x2 block(int s) const {
        const u32x4 q = a[s >> 1];
        return (s & 1) ? u32x2{q.z, q.w} : u32x2{q.x, q.y};
    }
};

// Four blocks of RT row tiles against NT slots: half H of a super-block.  m0: all ones in the lane groups of a block's first
// run (Q6_K).  P, M (W256): the super-block's integer sums, scaled once, behind its second half, the larger product d P unrounded.
// (Scaled after each half, d P rounded first, and the wavefronts' sums added one after the other: NMSE against 64 bits at K = 4096
// 8.8e-15 for Q4_K, so 6.5e-15, the tiles 7.5e-15; Q6_K 5.3e-15, so 3.9e-15, the tiles 4.8e-15.  And half as many scalings: Q4_K
// 14336 x 4096, 48 tokens 24.4 -> 21.5 us, Q6_K 4096 x 4096, 96 tokens 17.6 -> 16.4.)
// Q6_K, window 32: the half's four blocks are summed with the tokens' scales alone, and the sum meets the row's scale once: four
// vector instructions a result and block where each product met both in five.  44 shapes of 2 to 400 tokens 0.967 times as long
// (5649 x 13824 planes, 35 tokens 49.1 -> 45.2 us, 4663 x 3840 rows, 42 tokens 19.2 -> 18.6), NMSE against 64 bits 4.4e-15 -> 4.1e-15
// at K = 1024, 6.2e-15 -> 5.2e-15 at 2560.  (Summed over the super-block: 4.9e-15 and 5.9e-15.)
template <int TYPE, bool PL, int NT, int RT, bool W256, int H>
__device__ __forceinline__ void few_blocks(const FewR<TYPE, PL>* R, const float* sc, const FewA<TYPE, W256>* X, u32 m0, int g,
                                           i32x4 (*P)[NT], i32x4 (*M)[NT], f32x4 (*acc)[NT]) {
    const i32x4 zero = {0, 0, 0, 0};
    constexpr bool SUMS = TYPE == JL_Q6_K && !W256;
    f32x4 sum[RT][NT];
    if constexpr (SUMS)
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int t = 0; t < NT; t++) sum[rt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (W256 && H == 0)
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int t = 0; t < NT; t++) { P[rt][t] = zero; M[rt][t] = zero; }
    // (planes, four token tiles: a row tile's four blocks one after the other, so that one tile's sums are held, 168 registers for 175
    // and three wavefronts a SIMD for two)
    constexpr int OUTER = SUMS && PL && NT == 4 ? RT : 1, INNER = RT / OUTER;
#pragma unroll
    for (int u = 0; u < 4 * OUTER; u++) {
        const int s = u & 3;
        // (block by block: the compiler would gather the scale reads and decodes of all four, and sink
        // the sums' arithmetic behind the loop: registers)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int rt = (u >> 2) * INNER; rt < ((u >> 2) + 1) * INNER; rt++) {
            const u32x2 b = few_decode<TYPE, PL>(R[rt], s, g);
            const float* scr = sc + rt * (JL_FEW_SC_BYTES / 4);
            if constexpr (TYPE == JL_Q6_K) {
                const u32x2 b0 = u32x2{b.x & m0, b.y & m0}, b1 = u32x2{b.x & ~m0, b.y & ~m0};
                const i32x4 s0 = ((const i32x4*)scr)[(2 * s) * 4 + g], s1 = ((const i32x4*)scr)[(2 * s + 1) * 4 + g];
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const u32x2 a = X[t].block(s);
                    const i32x4 y0 = mfma_i8(b0, a, zero), y1 = mfma_i8(b1, a, zero);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const i32 v = __mul24(y0[i], s0[i]) + __mul24(y1[i], s1[i]);
                        if constexpr (W256) P[rt][t][i] += v;
                        else sum[rt][t][i] = fmaf((float)v, X[t].da[s], sum[rt][t][i]);
                    }
                    // (the products of four tiles in flight made 129 registers, and 128 are two workgroups of eight wavefronts a CU: planes
                    // 2401 x 1280, 151 tokens 14.6 us, so 12.1)
                    if constexpr (SUMS && PL && NT == 4 && RT == 1)
                        if (t == 1) __builtin_amdgcn_sched_barrier(0);
                }
            } else if constexpr (TYPE == JL_Q4_K && W256) {
                const i32x4 s4 = ((const i32x4*)scr)[s * 4 + g], m4 = ((const i32x4*)(scr + 64))[s * 4 + g];
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const i32x4 y = mfma_i8(b, X[t].block(s), zero);
                    const i32 A = (i32)__float_as_uint(X[t].ds[s]);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        P[rt][t][i] += __mul24(y[i], s4[i]);
                        M[rt][t][i] += __mul24(A, m4[i]);
                    }
                }
            } else {
                const f32x4 s4 = ((const f32x4*)scr)[s * 4 + g];
                f32x4 m4 = {0.f, 0.f, 0.f, 0.f};
                if constexpr (TYPE == JL_Q4_K) m4 = ((const f32x4*)(scr + 64))[s * 4 + g];
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const i32x4 y = mfma_i8(b, X[t].block(s), zero);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        acc[rt][t][i] = fmaf((float)y[i], s4[i] * X[t].da[s], acc[rt][t][i]);
                        if constexpr (TYPE == JL_Q4_K) acc[rt][t][i] = fmaf(-m4[i], X[t].ds[s], acc[rt][t][i]);
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if constexpr (W256) asm volatile("" : "+v"(P[rt][t]));
                else if constexpr (SUMS) asm volatile("" : "+v"(sum[rt][t]));
                else asm volatile("" : "+v"(acc[rt][t]));
                if constexpr (W256 && TYPE == JL_Q4_K) asm volatile("" : "+v"(M[rt][t]));
            }
        }
        if constexpr (OUTER > 1)
            if (s == 3) {
                const int rt = u >> 2;
                __builtin_amdgcn_sched_barrier(0);
                const f32x4 d4 = ((const f32x4*)(sc + rt * (JL_FEW_SC_BYTES / 4) + 128))[g];
#pragma unroll
                for (int t = 0; t < NT; t++) {
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[rt][t][i] = fmaf(sum[rt][t][i], d4[i], acc[rt][t][i]);
                    asm volatile("" : "+v"(acc[rt][t]));
                }
            }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (SUMS && OUTER == 1)
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            const f32x4 d4 = ((const f32x4*)(sc + rt * (JL_FEW_SC_BYTES / 4) + 128))[g];
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[rt][t][i] = fmaf(sum[rt][t][i], d4[i], acc[rt][t][i]);
        }
    if constexpr (W256 && H == 1)
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            const float* scr = sc + rt * (JL_FEW_SC_BYTES / 4);
            const f32x4 d4 = ((const f32x4*)(scr + 128))[g];
            f32x4 n4 = {0.f, 0.f, 0.f, 0.f};
            if constexpr (TYPE == JL_Q4_K) n4 = ((const f32x4*)(scr + 144))[g];
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float v;
                    if constexpr (TYPE == JL_Q4_K) v = fmaf(d4[i], (float)P[rt][t][i], -(n4[i] * (float)M[rt][t][i]));
                    else v = d4[i] * (float)P[rt][t][i];
                    acc[rt][t][i] = fmaf(v, X[t].d1, acc[rt][t][i]);
                }
        }
}

// ---------------------------------------------------------------- GGUF rows, a super-block (256 of K) at a time
// A row tile's 16 x 256 weights are 16 PC pieces of 16 bytes, loaded along the rows (a wavefront's lanes take
// consecutive pieces) and kept in LDS rows of STRIDE bytes.  Q8_0 (rows of whole 64s, 4-byte aligned: the host
// checks): 272 bytes, every piece 4-byte aligned.  Q4_K: 144 bytes.  Q6_K: 210 bytes that begin 0 or 2 bytes
// past a 4-byte boundary: 13 pieces from that boundary on, then the last two pairs of bytes by 2-byte loads.
template <int TYPE> struct FewRows;
template <> struct FewRows<JL_Q8_0> { static constexpr int PC = 17, NI = 5, STRIDE = 272, SB = 272; };
template <> struct FewRows<JL_Q4_K> { static constexpr int PC = 9, NI = 3, STRIDE = 144, SB = 144; };
template <> struct FewRows<JL_Q6_K> { static constexpr int PC = 13, NI = 4, STRIDE = 224, SB = 210; };
template <int TYPE> struct FewRowW { u32x4 v[FewRows<TYPE>::NI]; u32 tail; };
template <int TYPE, int RT> struct FewRowAddr { u32 row[RT][FewRows<TYPE>::NI], piece[FewRows<TYPE>::NI], lds[FewRows<TYPE>::NI], tail[RT], mine[RT]; };

template <int TYPE, int RT>
__device__ __forceinline__ void few_rows_load(const FewI8Args& p, const uint8_t* w, int sb, const FewRowAddr<TYPE, RT>& ad, FewRowW<TYPE>* W) {
    typedef FewRows<TYPE> F;
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
#pragma unroll
        for (int i = 0; i < F::NI; i++) {
            if constexpr (TYPE == JL_Q4_K) W[rt].v[i] = few_ld<u32x4>(w + (size_t)sb * 144, ad.row[rt][i]);
            else if constexpr (TYPE == JL_Q8_0) {
                // K may end inside the last unit: a piece that passes the row's end is its last 16 bytes
                const u32 o = min((u32)sb * 272u + ad.piece[i], (u32)p.row_bytes - 16u);
                W[rt].v[i] = few_ld<u32x4_a4>(w, ad.row[rt][i] + o).v;
            } else W[rt].v[i] = few_ld<u32x4_a4>(w, ((ad.row[rt][i] + (u32)sb * 210u) & ~3u) + ad.piece[i]).v;
        }
        if constexpr (TYPE == JL_Q6_K) W[rt].tail = few_ld<uint16_t>(w + (size_t)sb * 210, ad.tail[rt]);
    }
}

template <int TYPE, int RT>
__device__ __forceinline__ void few_rows_stage(const FewI8Args& p, int sb, const FewRowAddr<TYPE, RT>& ad, const FewRowW<TYPE>* W,
                                               uint8_t* st, int lane) {
    typedef FewRows<TYPE> F;
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        uint8_t* s = st + rt * 16 * F::STRIDE;
#pragma unroll
        for (int i = 0; i < F::NI; i++) {
            if constexpr (TYPE == JL_Q8_0) {
                const u32 o = (u32)sb * 272u + ad.piece[i], past = o - min(o, (u32)p.row_bytes - 16u);
                ((u32x4_a4*)(s + ad.lds[i] - past))->v = W[rt].v[i];
            } else *(u32x4*)(s + ad.lds[i]) = W[rt].v[i];
        }
        if constexpr (TYPE == JL_Q6_K) {
            const u32 a0 = (ad.tail[rt] + (u32)sb * 210u) & 2u;   // (field offsets of the tail are even multiples of... 208, 206)
            const int l = lane < 32 ? lane : 0, f = l < 16 ? 208 : 206;
            *(uint16_t*)(s + (l & 15) * F::STRIDE + ((a0 ^ (f & 2)) + f)) = (uint16_t)W[rt].tail;
        }
    }
}

// Half h (128 of K) of the staged super-block: the row's scales to the scale area, the lane's words to R.
template <int TYPE, int RT, bool W256>
__device__ __forceinline__ void few_rows_half(const FewI8Args& p, int sb, int h, const FewRowAddr<TYPE, RT>& ad, const uint8_t* st, float* sc,
                                              int g, int r, FewR<TYPE, false>* R) {
    typedef FewRows<TYPE> F;
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        const uint8_t* s = st + rt * 16 * F::STRIDE + r * F::STRIDE;
        float* scr = sc + rt * (JL_FEW_SC_BYTES / 4);
        if constexpr (TYPE == JL_Q8_0) {
            const u32 d = *(const uint16_t*)(s + (4 * h + g) * 34);
            few_put_q8(sb * 8 + 4 * h + g < p.k / 32 ? d : 0u, g, r, scr);   // (past K: whatever LDS held)
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const u32* q = (const u32*)(s + (4 * h + b) * 34 + (b & 1 ? 2 : 0) + 8 * g);   // 4-byte aligned
                if (b & 1) { R[rt].v[b][0] = q[0]; R[rt].v[b][1] = q[1]; }
                else {
                    const u32 x = q[0], y = q[1], z = q[2];
                    R[rt].v[b][0] = __builtin_amdgcn_alignbyte(y, x, 2);
                    R[rt].v[b][1] = __builtin_amdgcn_alignbyte(z, y, 2);
                }
            }
        } else if constexpr (TYPE == JL_Q4_K) {
            const u32x4 hd = *(const u32x4*)s;
            // bytes of the scale fields of sub-block g or 4 + g (format/quant/dequant.go:360-365)
            const u32 b0 = hd.y >> (8 * g), b1 = hd.z >> (8 * g), b2 = hd.w >> (8 * g);
            const u32 k = h ? (b2 & 0xF) | (((b0 >> 6) & 3) << 4) : b0 & 63;
            const u32 m = h ? ((b2 >> 4) & 0xF) | (((b1 >> 6) & 3) << 4) : b1 & 63;
            few_put_q4k<W256>(hd.x, k, m, g, r, scr);
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const u32x2 q = *(const u32x2*)(s + 16 + h * 64 + b * 32 + 8 * g);
                R[rt].v[b][0] = q.x; R[rt].v[b][1] = q.y;
            }
        } else {
            const u32 a0 = (ad.mine[rt] + (u32)sb * 210u) & 2u;
            const u32 two = *(const uint16_t*)(s + a0 + 192 + 8 * h + 2 * g);
            few_put_q6k(*(const uint16_t*)(s + a0 + 208), (i32)(int8_t)(two & 0xFF), (i32)(int8_t)(two >> 8), g, r, scr);
            auto eight = [&](int f, u32& x, u32& y) {
                const u32* q = (const u32*)(s + f + 8 * g);
                const u32 u = q[0], v = q[1], z = q[2];
                x = __builtin_amdgcn_alignbyte(v, u, a0);
                y = __builtin_amdgcn_alignbyte(z, v, a0);
            };
            eight(64 * h, R[rt].v[0][0], R[rt].v[0][1]);
            eight(64 * h + 32, R[rt].v[1][0], R[rt].v[1][1]);
            eight(128 + 32 * h, R[rt].h[0], R[rt].h[1]);
        }
    }
}

// ---------------------------------------------------------------- planes, half a super-block (128 of K) at a time
template <int TYPE> struct FewPlaneW;
template <> struct FewPlaneW<JL_Q8_0> { u32 q[4][2], d; };
template <> struct FewPlaneW<JL_Q4_K> { u32 q[4], h; };
template <> struct FewPlaneW<JL_Q6_K> { u32 q[4], h[2], sc, d; };
// vr: byte offset of the lane's first row's word; vg, vh the lane group's shares; hp, hstep its header plane (Q4_K)
struct FewPlaneAddr { u32 vr, vg, vh, hstep; const uint8_t* hp; };

template <int TYPE, int RT>
__device__ __forceinline__ void few_planes_load(const FewI8Args& p, const FewMat& m, int c, const FewPlaneAddr& ad, int g, FewPlaneW<TYPE>* W) {
    const size_t st = (size_t)p.pstride;
    u32 t[RT];
    if constexpr (TYPE == JL_Q8_0) {
        const int nb = p.k / 32;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const u32* b = m.qs + (size_t)min(c * 4 + s, nb - 1) * 8 * st;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                few_words<RT>(b + h * st, ad.vr + ad.vg, t);
#pragma unroll
                for (int j = 0; j < RT; j++) W[j].q[s][h] = t[j];
            }
        }
        // two rows a word of the D plane: RT rows from an even or an odd one on
        const u32 o = (u32)min(c * 4 + g, nb - 1) * (((u32)p.pstride + 1) / 2) * 4u + ((ad.vr >> 3) << 2);
        const u32 odd = (ad.vr >> 2) & 1;
        if constexpr (RT == 1) {
            W[0].d = few_ld<u32>(m.dp, o) >> (16 * odd);
        } else {
            const u32 last = few_ld<u32>(m.dp, o + (RT / 2 - 1 + odd) * 4u);
            u32 d[RT / 2];
            few_words<RT / 2>(m.dp, o, d);
#pragma unroll
            for (int j = 0; j < RT / 2; j++) {
                const u32 nx = j + 1 < RT / 2 ? d[j + 1] : last;
                const u32 both = odd ? (d[j] >> 16) | (nx << 16) : d[j];
                W[2 * j].d = both;
                W[2 * j + 1].d = both >> 16;
            }
        }
    } else if constexpr (TYPE == JL_Q4_K) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            few_words<RT>(m.qs + (size_t)(c * 4 + s) * 4 * st, ad.vr + ad.vg, t);
#pragma unroll
            for (int j = 0; j < RT; j++) W[j].q[s] = t[j];
        }
        few_words<RT>(ad.hp + (size_t)(u32)(c >> 1) * ad.hstep, 0, t);   // lane group 0: d, 1..3: the scale words
#pragma unroll
        for (int j = 0; j < RT; j++) W[j].h = t[j];
    } else {
        // lane group g: run g / 2 of the block, primary word g % 2; the run's third word for two blocks at
        // once (even lane groups the first's, odd the second's)
#pragma unroll
        for (int s = 0; s < 4; s++) {
            few_words<RT>(m.qs + (size_t)(c * 8 + 2 * s) * 3 * st, ad.vr + ad.vg, t);
#pragma unroll
            for (int j = 0; j < RT; j++) W[j].q[s] = t[j];
        }
#pragma unroll
        for (int s = 0; s < 2; s++) {
            few_words<RT>(m.qs + (size_t)(c * 8 + 4 * s) * 3 * st, ad.vr + ad.vh, t);
#pragma unroll
            for (int j = 0; j < RT; j++) W[j].h[s] = t[j];
        }
        few_words<RT>(m.sp + (size_t)c * 2 * st, ad.vr + ((g >> 1) ? (u32)p.pstride * 4u : 0u), t);
#pragma unroll
        for (int j = 0; j < RT; j++) W[j].sc = t[j];
        few_words<RT>(m.dp + (size_t)(c >> 1) * st, ad.vr, t);
#pragma unroll
        for (int j = 0; j < RT; j++) W[j].d = t[j];
    }
}

template <int TYPE, int RT, bool W256>
__device__ __forceinline__ void few_planes_half(int c, const FewPlaneW<TYPE>* W, float* sc, int g, int r, FewR<TYPE, true>* R) {
    if constexpr (TYPE == JL_Q4_K) {
        // the header words go round: each lane of a row gets all four
#pragma unroll
        for (int j = 0; j < RT; j++) ((u32*)(sc + j * (JL_FEW_SC_BYTES / 4) + 160))[r * 4 + g] = W[j].h;
        few_lds_fence();
    }
#pragma unroll
    for (int j = 0; j < RT; j++) {
        float* scr = sc + j * (JL_FEW_SC_BYTES / 4);
        if constexpr (TYPE == JL_Q8_0) {
            few_put_q8(W[j].d, g, r, scr);
#pragma unroll
            for (int s = 0; s < 4; s++) { R[j].v[s][0] = W[j].q[s][0]; R[j].v[s][1] = W[j].q[s][1]; }
        } else if constexpr (TYPE == JL_Q4_K) {
            const u32x4 h = ((const u32x4*)(scr + 160))[r];
            // bits 12 s .. 12 s + 11 of the 96-bit stream; s = g (bits 0, 12, 24, 36) or 4 + g (48, 60, 72, 84)
            const u32 a = (c & 1) ? (g < 2 ? h.z : h.w) : (g < 3 ? h.y : h.z);
            const u32 b = (c & 1) ? h.w : h.z;
            const u32 f = (u32)((((uint64_t)b << 32) | a) >> ((12 * ((c & 1) * 4 + g)) & 31));
            few_put_q4k<W256>(h.x, f & 63, (f >> 6) & 63, g, r, scr);
#pragma unroll
            for (int s = 0; s < 4; s++) R[j].v[s] = W[j].q[s];
        } else {
            const u32 two = W[j].sc >> (16 * (g & 1));
            few_put_q6k(W[j].d, (i32)(two & 0xFF) - 128, (i32)((two >> 8) & 0xFF) - 128, g, r, scr);
#pragma unroll
            for (int s = 0; s < 4; s++) R[j].v[s] = W[j].q[s];
#pragma unroll
            for (int s = 0; s < 2; s++) {
                u32 a = W[j].h[s], b = W[j].h[s];
                swap16(a, b);
                R[j].h[2 * s] = a; R[j].h[2 * s + 1] = b;
            }
        }
    }
}

// Q6_K, window 32: result (row r, token tok of a slot) block by block.  A row's scale that is infinite meets the sum of four blocks
// above; the decode matvec's infinities and NaN are those of its products with the blocks one by one.
template <bool PL>
__device__ __forceinline__ float few_q6_one(const FewI8Args& p, const FewMat& m, int e, int r, u32 slot, int tok) {
    const uint8_t* row = PL ? nullptr : m.w + (size_t)r * p.row_bytes;
    const size_t n = (size_t)p.pstride, at = (size_t)(p.prow0 + e * p.row_step + r);
    float o = 0.f;
#pragma unroll 1
    for (int b = 0; b < p.k / 32; b++) {
        const int sb = b >> 3, half = (b >> 2) & 1, s = b & 3;
        const size_t x = (size_t)(b >> 2) * p.nslots + slot;
        const u32* a = (const u32*)p.bq + x * 512 + (s >> 1) * 256 + tok * 4 + 2 * (s & 1);
        const uint8_t* blk = PL ? nullptr : row + (size_t)sb * 210;
        i32 P = 0;
#pragma unroll
        for (int run = 0; run < 2; run++) {
            u32x4 lo, hi = {0u, 0u, 0u, 0u};   // the run's words
            u32 hw = 0;
            i32 sc, v = 0;
            if constexpr (PL) {
                const u32* w = m.qs + ((size_t)(sb * 16 + half * 8 + 2 * s + run) * 3) * n + at;
                lo = u32x4{w[0], w[n], w[0] >> 4, w[n] >> 4};
                hw = w[2 * n];
                sc = (i32)((m.sp[((size_t)sb * 4 + 2 * half + (s >> 1)) * n + at] >> (16 * (s & 1) + 8 * run)) & 255) - 128;
            } else {
                lo = ld16_a2(blk + 64 * half + 32 * (s & 1) + 16 * run);
                hi = ld16_a2(blk + 128 + 32 * half + 16 * run);
                sc = (int8_t)blk[192 + 8 * half + 2 * s + run];
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const u32 h2 = PL ? hw >> (2 * i) : hi[i] >> (2 * s), q = ((PL ? lo[i] : lo[i] >> (4 * (s >> 1))) & 0x0F0F0F0Fu) | ((h2 & 0x03030303u) << 4);
                int g, h;
                jl_few_order(PL ? 2 : 0, 4 * run + i, g, h);
                v = dot4(0xE0E0E0E0u, a[g * 64 + h], dot4(q, a[g * 64 + h], v));   // q - 32
            }
            P += sc * v;
        }
        const u32 d = PL ? m.dp[(size_t)sb * n + at] : (u32)ld2(blk + 208);
        o = fmaf((float)P, half_bits_to_f32((uint16_t)d) * p.da[x * 64 + 4 * tok + s], o);
    }
    return o;
}

// grid = (ceil(nrows / (16 RT)), experts or token groups, matrices), block = 64 * p.nwaves, dynamic LDS: JL_FEW_LDS_BYTES.
template <int TYPE, bool PL, int NT, int RT, bool W256>
__device__ __forceinline__ void few_i8_body(const FewI8Args& args, uint8_t* smem) {
    FewI8Args p;   // the matrix's arguments, asked for at once
    {
        const int mat = blockIdx.z;
        p.out[0] = args.out[mat];
        p.w[0] = PL ? nullptr : args.w[mat];
        p.pqs[0] = PL ? args.pqs[mat] : nullptr; p.pd[0] = PL ? args.pd[mat] : nullptr; p.psc[0] = PL && TYPE != JL_Q8_0 ? args.psc[mat] : nullptr;
        p.resid = args.resid; p.bq = args.bq; p.da = args.da; p.ds = TYPE == JL_Q4_K ? args.ds : nullptr; p.start = args.start;
        p.sheet_bytes = PL ? 0 : args.sheet_bytes; p.sheet_words = PL ? args.sheet_words : 0;
        p.row_step = PL ? args.row_step : 0; p.prow0 = PL ? args.prow0 : 0; p.pstride = PL ? args.pstride : 0;
        p.nrows = args.nrows; p.k = args.k; p.row_bytes = PL ? 0 : args.row_bytes; p.ncols = args.ncols; p.nslots = args.nslots;
        p.nch = args.nch; p.nwaves = args.nwaves; p.tgroup = args.tgroup;
        if constexpr (PL) {
            JL_NOW(p.out[0], p.pqs[0], p.pd[0], p.psc[0], p.resid, p.bq, p.da, p.ds, p.start, p.sheet_words, p.row_step, p.prow0, p.pstride,
                   p.nrows, p.k, p.ncols, p.nslots, p.nch, p.nwaves, p.tgroup);
            p.pqs[0] = as_global(p.pqs[0]); p.pd[0] = as_global(p.pd[0]); p.psc[0] = as_global(p.psc[0]);
        } else {
            JL_NOW(p.out[0], p.w[0], p.resid, p.bq, p.da, p.ds, p.start, p.sheet_bytes, p.nrows, p.k, p.row_bytes, p.ncols, p.nslots, p.nch,
                   p.nwaves, p.tgroup);
            p.w[0] = as_global(p.w[0]);
        }
        p.out[0] = as_global(p.out[0]); p.resid = as_global(p.resid); p.bq = as_global(p.bq); p.da = as_global(p.da); p.ds = as_global(p.ds);
        p.start = as_global(p.start);
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), nw = p.nwaves;
    const int r16 = lane & 15, g = lane >> 4;
    const int e = p.start ? blockIdx.y : 0;
    u32 col0 = 0, ncol = (u32)p.ncols;
    if (p.start) {
        col0 = (u32)__builtin_amdgcn_readfirstlane((i32)p.start[e]);
        ncol = (u32)__builtin_amdgcn_readfirstlane((i32)p.start[e + 1]) - col0;
        if (ncol == 0) return;
    }
    const int r0 = blockIdx.x * 16 * RT;
    FewMat m;
    m.w = PL ? nullptr : p.w[0] + (size_t)e * p.sheet_bytes;
    m.qs = PL ? p.pqs[0] + (size_t)e * p.sheet_words : nullptr;
    m.dp = PL ? p.pd[0] + (size_t)e * p.sheet_words : nullptr;
    m.sp = PL && TYPE != JL_Q8_0 ? p.psc[0] + (size_t)e * p.sheet_words : nullptr;
    u32 va = 16u * lane, vd = 16u * r16;
    float* sc = (float*)(smem + wave * JL_FEW_WAVE_BYTES(TYPE, PL, RT));
    uint8_t* st = (uint8_t*)sc + JL_FEW_SC_BYTES * RT;   // GGUF rows: the staged super-block
    // Q6_K: the lane groups that hold a block's first run of sixteen
    const u32 m0 = g < 2 ? 0xFFFFFFFFu : 0u;
    const u32 t_lo = p.start ? 0u : blockIdx.y * (u32)p.tgroup;
    const u32 ntile = p.start ? (ncol + 15) >> 4 : min((ncol + 15) >> 4, t_lo + (u32)p.tgroup);
    ncol = min(ncol, 16u * ntile);   // (a last tile of NT past the group's: not this workgroup's to store)
    const u32 slot0 = (col0 >> 4) + (u32)e;

    FewPlaneAddr pa;
    FewRowAddr<TYPE, RT> ra;
    if constexpr (PL) {
        // row tile j: rows RT r + j, the last rows' lanes moved back so that no load passes the row range
        const u32 w4 = (u32)p.pstride * 4u;
        pa.vr = (u32)(p.prow0 + e * p.row_step + min(r0 + RT * r16, p.nrows - RT)) * 4u;
        pa.vg = 0; pa.vh = 0; pa.hstep = 0; pa.hp = nullptr;
        if constexpr (TYPE == JL_Q8_0) pa.vg = 2u * g * w4;
        else if constexpr (TYPE == JL_Q4_K) {
            pa.vg = (u32)g * w4;
            pa.hp = (const uint8_t*)(g ? m.sp + (size_t)(g - 1) * p.pstride : m.dp) + pa.vr;
            pa.hstep = g ? 3u * w4 : w4;
        } else {
            pa.vg = (u32)((g >> 1) * 3 + (g & 1)) * w4;
            pa.vh = (u32)((g >> 1) * 3 + 2 + (g & 1) * 6) * w4;
        }
    } else {
        typedef FewRows<TYPE> F;
#pragma unroll
        for (int i = 0; i < F::NI; i++) {
            const int idx = min(i * 64 + lane, 16 * F::PC - 1), rr = idx / F::PC, pc = idx % F::PC;
            ra.piece[i] = 16u * pc;
            ra.lds[i] = (u32)(rr * F::STRIDE + 16 * pc);
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
                ra.row[rt][i] = (u32)min(r0 + rt * 16 + rr, p.nrows - 1) * (u32)p.row_bytes + (TYPE == JL_Q4_K ? ra.piece[i] : 0u);
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            ra.mine[rt] = (u32)min(r0 + rt * 16 + r16, p.nrows - 1) * (u32)p.row_bytes;
            const int l = lane < 32 ? lane : 0;
            ra.tail[rt] = (u32)min(r0 + rt * 16 + (l & 15), p.nrows - 1) * (u32)p.row_bytes + (l < 16 ? 208u : 206u);
        }
    }

    for (u32 t0 = t_lo; t0 < ntile; t0 += NT) {
        f32x4 acc[RT][NT];
        i32x4 P[RT][NT], M[RT][NT];
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int t = 0; t < NT; t++) acc[rt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        u32 slot[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) slot[t] = slot0 + min(t0 + t, ntile - 1);   // (past the last: its results are not stored)
        auto load_a = [&](int c128, FewA<TYPE, W256>* X) {
#pragma unroll
            for (int t = 0; t < NT; t++) X[t].load(p, c128, slot[t], va, vd);
        };

        // The next unit is on its way while one is worked on, in two register sets that take turns (a copy
        // from one to the other would wait for the data, and a request behind a branch would make every
        // wait before it count for nothing: the last unit is peeled).  Activations go out ahead of the
        // weights: a wavefront's loads return in order, and they come from L2.
        if constexpr (PL) {
            // (with four token tiles the activations are asked for when their chunk begins: registers)
            constexpr bool AHEAD = NT <= 2;
            FewPlaneW<TYPE> W0[RT], W1[RT];
            FewA<TYPE, W256> X0[NT], X1[NT];
            auto pin = [&]() { few_pin(va); few_pin(vd); few_pin(pa.vg); few_pin(pa.vh); few_pin(pa.vr); };
            auto load_w = [&](int c, FewPlaneW<TYPE>* W) { few_planes_load<TYPE, RT>(p, m, c, pa, g, W); };
            auto compute = [&](auto H, int sb, const FewPlaneW<TYPE>* W, const FewA<TYPE, W256>* X) {
                constexpr int h = decltype(H)::value;
                FewR<TYPE, true> R[RT];
                few_planes_half<TYPE, RT, W256>(2 * sb + h, W, sc, g, r16, R);
                few_lds_fence();
                few_blocks<TYPE, true, NT, RT, W256, h>(R, sc, X, m0, g, P, M, acc);
                few_lds_fence();
            };
            // (super-blocks w, w + nwaves, ... of wavefront w, the halves in turn: the order of the rows' form,
            // whose bits these are)
            const int nsb = p.nch / 2;
            int sb = wave;
            if (sb < nsb) {
                if (AHEAD) load_a(2 * sb, X0);
                load_w(2 * sb, W0);
                for (; sb + nw < nsb; sb += nw) {
                    pin();
                    if (AHEAD) load_a(2 * sb + 1, X1); else load_a(2 * sb, X0);
                    load_w(2 * sb + 1, W1);
                    compute(GemmIntC<0>{}, sb, W0, X0);
                    pin();
                    if (AHEAD) load_a(2 * (sb + nw), X0); else load_a(2 * sb + 1, X0);
                    load_w(2 * (sb + nw), W0);
                    compute(GemmIntC<1>{}, sb, W1, AHEAD ? X1 : X0);
                }
                pin();
                if (AHEAD) load_a(2 * sb + 1, X1); else load_a(2 * sb, X0);
                load_w(2 * sb + 1, W1);
                compute(GemmIntC<0>{}, sb, W0, X0);
                if (!AHEAD) load_a(2 * sb + 1, X0);
                compute(GemmIntC<1>{}, sb, W1, AHEAD ? X1 : X0);
            }
        } else {
            // A super-block's registers are free once it is staged, so one set is enough: stage, ask for the
            // halves' activations, then for the next super-block, then work.  (NT > 1: the second half's
            // activations, and the next super-block behind them, between the halves.)
            FewRowW<TYPE> W[RT];
            FewA<TYPE, W256> X0[NT], X1[NT];
            auto pin = [&]() {
                few_pin(va); few_pin(vd);
#pragma unroll
                for (int i = 0; i < FewRows<TYPE>::NI; i++) {
                    few_pin(ra.piece[i]);
#pragma unroll
                    for (int rt = 0; rt < RT; rt++) few_pin(ra.row[rt][i]);
                }
#pragma unroll
                for (int rt = 0; rt < RT; rt++) { few_pin(ra.tail[rt]); few_pin(ra.mine[rt]); }
            };
            auto half = [&](int sb, auto H, const FewA<TYPE, W256>* X) {
                constexpr int h = decltype(H)::value;
                FewR<TYPE, false> R[RT];
                few_rows_half<TYPE, RT, W256>(p, sb, h, ra, st, sc, g, r16, R);
                few_lds_fence();
                few_blocks<TYPE, false, NT, RT, W256, h>(R, sc, X, m0, g, P, M, acc);
                few_lds_fence();
            };
            auto unit = [&](int sb, int next) {   // next < 0: the last
                few_rows_stage<TYPE, RT>(p, sb, ra, W, st, lane);
                few_lds_fence();
                pin();
                load_a(2 * sb, X0);
                if constexpr (NT == 1) {
                    load_a(2 * sb + 1, X1);
                    if (next >= 0) few_rows_load<TYPE, RT>(p, m.w, next, ra, W);
                    half(sb, GemmIntC<0>{}, X0);
                    half(sb, GemmIntC<1>{}, X1);
                } else {
                    half(sb, GemmIntC<0>{}, X0);
                    load_a(2 * sb + 1, X0);
                    if (next >= 0) few_rows_load<TYPE, RT>(p, m.w, next, ra, W);
                    half(sb, GemmIntC<1>{}, X0);
                }
            };
            const int nsb = p.nch / 2;
            int sb = wave;
            if (sb < nsb) {
                pin();
                few_rows_load<TYPE, RT>(p, m.w, sb, ra, W);
                for (; sb + nw < nsb; sb += nw) unit(sb, sb + nw);
                unit(sb, -1);
            }
        }

        // the wavefronts' partial tiles, [wavefront][token][16 RT rows + 4]
        constexpr int RS = 16 * RT + 4;
        float* red = (float*)smem;
        __syncthreads();
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int t = 0; t < NT; t++) {
                float* o = red + ((size_t)wave * 16 * NT + t * 16 + r16) * RS;
                if constexpr (!PL || RT == 1) {
                    *(f32x4*)(o + rt * 16 + 4 * g) = acc[rt][t];
                } else {
                    // (lanes that were moved back repeat rows that others hold too: the same values)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int at = min(r0 + RT * (4 * g + i), p.nrows - RT) + rt - r0;
                        if (at >= 0) o[at] = acc[rt][t][i];
                    }
                }
            }
        __syncthreads();
        const u32 left = ncol - t0 * 16;
        for (int i = threadIdx.x; i < 16 * NT * 16 * RT; i += nw * 64) {
            const int tok = i / (16 * RT), rr = i % (16 * RT);
            // (by pairs: one after the other the eight additions round four and a half times a result's size, so three)
            const float* at = red + tok * RS + rr;
            constexpr int W = 16 * NT * RS;
            float v = 0.f;
            int q = 0;
            for (; q + 4 <= nw; q += 4, at += 4 * W) v += (at[0] + at[W]) + (at[2 * W] + at[3 * W]);
            for (; q < nw; q++, at += W) v += at[0];
            if constexpr (TYPE == JL_Q6_K && !W256) {
                // Again where a row's scale is infinite or four blocks' sum passes the largest f32, but not where the token has a scale that
                // is no number: its blocks' integers are zero, its sums NaN in every row and form.  (4096 x 4096, 12 tokens, one of them with
                // an infinite activation: 485 us without that second look, 22 as a call without.)  Sixteen lanes in a row hold one token.
                const bool mine = (u32)tok < left && r0 + rr < p.nrows && !__builtin_isfinite(v);
                if (__ballot(mine)) {
                    u32 l = threadIdx.x & 63;
                    few_pin(l);   // (nothing of this ahead of the wavefront's super-blocks, in registers of theirs)
                    bool bad = false;
                    if ((u32)tok < left)
                        for (int x = l & 15; x < p.k / 128; x += 16) {
                            const f32x4 d = *(const f32x4*)(p.da + ((size_t)x * p.nslots + slot0 + t0 + (tok >> 4)) * 64 + 4 * (tok & 15));
#pragma unroll
                            for (int b = 0; b < 4; b++) bad |= !__builtin_isfinite(d[b]);
                        }
                    const bool token = ((u32)(__ballot(bad) >> (l & 48)) & 0xFFFFu) == 0;
                    if (mine && token) v = few_q6_one<PL>(p, m, e, r0 + rr, slot0 + t0 + (tok >> 4), tok & 15);
                }
            }
            if ((u32)tok < left && r0 + rr < p.nrows) {
                const size_t o = (size_t)(col0 + t0 * 16 + tok) * p.nrows + r0 + rr;
                if (p.out[0]) p.out[0][o] = v;
                if (p.resid) p.resid[o] += v;
            }
        }
        if (t0 + NT < ntile) __syncthreads();
    }
}
