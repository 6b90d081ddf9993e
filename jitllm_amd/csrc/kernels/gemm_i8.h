// Prefill GEMM, and the mixture's tile per expert, on the int8 matrix cores: Q8_0, Q4_K and Q6_K with the activation
// window of 32 (the window of a model that holds a type with 32-element blocks, jit/cpu/matvec.go:46-62), Q6_K
// with the k-quant window of 256.  Per (token, row) it is the decode matvec's value (format/quant/dequant.go:
// 148-157, :360-397 and :443-470 for the weights, jit/cpu/packedgemm.go:54-58 for the identity with the matvec):
//
//   window 32    out[t][r] = sum_b d_a[t,b] * d[r,b] * P[t,r,b],  P = sum_{l<32} q[r,b,l] * a[t,b,l]
//                (Q4_K: d = d * sc of the sub-block, minus (dmin * m) * (d_a * sum of the block's a))
//   window 256   out[t][r] = sum_sb d_a[t,sb] * d[r,sb] * P[t,r,sb]
//
// v_mfma_i32_32x32x32_i8 takes a block of 32 a time, exactly.  Q6_K's weight is sc * (q - 32), thirteen bits: it goes in
// as two int8 operands, 128 * hi + lo, whose sums are put together as integers.
//
// What bounds it.  Window 32: both scales change every 32 of K, so an output element costs vector instructions a block.  Q8_0 and
// Q4_K: two, since the sums leave the matrix core as floats (below); with a conversion, a product and a multiply-add it was
// three, 53 vector instructions a matrix instruction with everything else, now 37.  Q8_0, 2048 tokens x 4096 -> 14336, tiles of
// 256 tokens x 128 rows: the vector unit issues 76 % of the time and the matrix instructions take most of the rest, the two do
// not overlap on a SIMD; L1 0.35 of 0.69 million cycles (0.70 of 0.67 under tiles of 128 tokens, whose weights' narrow loads bound
// it then): 320 us, 363 before, 460 as f16 operands.  Q6_K, two operands and two matrix instructions a block: four
// vector instructions an output element and block, now three and an eighth (a super-block's sum meets the row's scale once): 14336 x 4096,
// 2048 tokens 621 -> 568 us, 12957 x 1536, 1138 147 -> 136, NMSE against 64 bits 1.4e-14 -> 4.8e-15 (13183 x 1280, 102 tokens).
// Window 256 (551 us as f16 operands, 14336 -> 4096, now 400): 12 vector instructions a matrix instruction, most of
// them the making of Q6_K's two operands, which every workgroup of 128 tokens does anew; vector unit 43 %, matrix cores 27 %, L1
// 0.66 of 0.85 million cycles.
//
// A workgroup of four wavefronts (TW = 8: eight) owns 32 TW tokens x 32 RT (4 / TW) rows, a wavefront 32 tokens x 32 RT rows.  A
// stage is 128 of K: the threads turn the rows' bytes into operands in LDS (thread = row, block of 32), one stage ahead of
// the matrix work and dealt over it, two buffers and one barrier a stage.  A tile's scaling runs under the next
// tile's matrix instruction.  Rows sit on lanes (stores are contiguous), tokens on registers; activation fragments
// come from L2 into a register ring a stage ahead.
//
// Prep (gemm_i8_prep_group): x f32 -> bq [k/128 stages][groups of 32 tokens][4 blocks][64 lanes][16] int8, lane (t = lane %
// 32, kg = lane / 32) holding elements 16 kg .. of the block; da [k/32][tok_pad] (window 256: [k/256][tok_pad]) and, for
// Q4_K, dsum likewise.
#pragma once
#include "gemm_q4k.h"

#pragma clang fp contract(off)

// A buffer: operand planes, rows of 128 bytes whose sixteen-byte pieces are permuted by the row (piece c of row r lies at
// c ^ r % 8: a wavefront's reads, one piece of 32 rows, spread over all banks without padding); window 32: the rows'
// scales [rows][4 blocks] and the tokens' [4 blocks][32 tw], Q4_K: twice.
#define JL_GEMM_I8_BUF_BYTES(planes, rows, tw, w32, mins) \
    ((planes) * (rows) * 128 + ((w32) ? ((mins) + 1) * ((rows) * 16 + 4 * 32 * (tw) * 4) : 0))
#define JL_GEMM_I8_LDS_BYTES(planes, rows, tw, w32, mins) (2 * JL_GEMM_I8_BUF_BYTES(planes, rows, tw, w32, mins))
#define JL_GEMM_I8_PREP_WORDS (32 * 65)

typedef i32 i32x16 __attribute__((ext_vector_type(16)));
typedef short i16x2 __attribute__((ext_vector_type(2)));

// One chunk of 256 elements of a group of 32 tokens: quantize, lay out.  load(t): this lane's four elements of
// token t (zero past the end).  block = 1024: sixteen wavefronts, two tokens each (the chain of tokens a wavefront
// quantizes is the kernel's length).
template <class Load>
__device__ __forceinline__ void gemm_i8_prep_group(u32* sq, int ch, int grp, int ngrp, int k, int per, u32* bq, float* da, float* dsum, Load load) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tok_pad = 32 * ngrp;
    const bool in = ch * 256 + 4 * lane < k;
    f32x4 v[2];
#pragma unroll
    for (int i = 0; i < 2; i++) v[i] = load(wave * 2 + i, in);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int t = wave * 2 + i;
        const u32 m = max(max(abs_bits(v[i].x), abs_bits(v[i].y)), max(abs_bits(v[i].z), abs_bits(v[i].w)));
        const u32 amax = per == 8 ? wave_amax_256(m) : window_amax(m, per);
        float d;
        i32 s16;
        sq[t * 65 + lane] = quantize4(v[i], amax, d, s16);
        const i32 s32 = s16 + dpp_i32<JL_DPP_ROW_HALF_MIRROR, 0xf>(0, s16);
        if (per == 8) {
            if (lane == 0) da[(size_t)ch * tok_pad + grp * 32 + t] = d;
        } else if ((lane & 7) == 0 && in) {
            const size_t at = (size_t)(ch * 8 + (lane >> 3)) * tok_pad + grp * 32 + t;
            da[at] = d;
            if (dsum) dsum[at] = d * (float)s32;
        }
    }
    __syncthreads();
    const int f = threadIdx.x >> 6, t = lane & 31, kg = lane >> 5;   // fragment f: stage half f / 4, block f % 4
    const int stage = 2 * ch + (f >> 2);
    if (f < 8 && stage < k / 128) {
        const u32* s = sq + t * 65 + 8 * f + 4 * kg;
        ((u32x4*)bq)[(((size_t)stage * ngrp + grp) * 4 + (f & 3)) * 64 + lane] = u32x4{s[0], s[1], s[2], s[3]};
    }
}
// grid = (ceil(k/256), tok_pad/32), block = 1024
__device__ __forceinline__ void gemm_i8_prep_body(const GemmPrepArgs& args, u32* sq) {
    GemmPrepArgs p = args;
    JL_NOW(p.x, p.bq, p.da, p.dsum, p.ntok, p.tok_pad, p.k, p.per);
    const float* x = as_global(p.x);
    const int ch = blockIdx.x, grp = blockIdx.y, lane = threadIdx.x & 63;
    gemm_i8_prep_group(sq, ch, grp, p.tok_pad >> 5, p.k, p.per, (u32*)as_global(p.bq), as_global(p.da), as_global(p.dsum), [&](int t, bool in) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (grp * 32 + t < p.ntok && in) v = *(const f32x4*)(x + (size_t)(grp * 32 + t) * p.k + ch * 256 + 4 * lane);
        return v;
    });
}

// K split: sb_per stages to a workgroup (k-quants: an even number), partial sums to slab z
template <int TYPE, bool W256> __device__ __forceinline__ void gemm_i8_split_slice(GemmArgs& p) {
    if (p.sb_per == 0) return;
    const int s0 = blockIdx.z * p.sb_per;
    const int n = min(p.sb_per, p.k / 128 - s0);
    p.w += TYPE == JL_Q8_0 ? (size_t)s0 * 4 * 34 : (size_t)(s0 / 2) * (TYPE == JL_Q6_K ? 210 : 144);
    if (TYPE == JL_Q4_K) p.dsum += (size_t)s0 * 4 * p.tok_pad;
    p.bq += (size_t)s0 * (p.tok_pad >> 5) * (4096 / 2);
    p.da += W256 ? (size_t)(s0 / 2) * p.tok_pad : (size_t)s0 * 4 * p.tok_pad;
    p.k = 128 * n;
    p.out += (size_t)blockIdx.z * p.ntok * p.out_stride;
}

// A thread's bytes of a weight stage: one block (run) of 32.
template <int TYPE> struct GemmI8Raw;
template <> struct GemmI8Raw<JL_Q8_0> { u32x4 q[2]; u32 d; };
template <> struct GemmI8Raw<JL_Q4_K> { u32x4 q[2], h; };
template <> struct GemmI8Raw<JL_Q6_K> { u32x4 q[2], h[2]; u32 d; };   // d: the super-block's | the run's two scales << 16

// One sum out[t][r] of a window-32 tile, block by block as integers turned to f32, row: the weight row's first block.
template <int TYPE>
__device__ __forceinline__ float gemm_i8_one(const GemmArgs& p, const uint8_t* row, int t) {
    const u32x4* a = (const u32x4*)p.bq + ((size_t)(t >> 5) * 4) * 64 + (t & 31);
    float o = 0.f;
#pragma unroll 1
    for (int b = 0; b < p.k / 32; b++) {
        const u32x4* f = a + ((size_t)(b >> 2) * (p.tok_pad >> 5) * 4 + (b & 3)) * 64;
        if constexpr (TYPE == JL_Q6_K) {
            const uint8_t* blk = row + (size_t)(b >> 3) * 210;
            const int n = (b >> 2) & 1, g = b & 3;
            i32 P = 0;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const u32x4 lo = ld16_a2(blk + 64 * n + 32 * (g & 1) + 16 * h), hi = ld16_a2(blk + 128 + 32 * n + 16 * h), v = f[32 * h];
                i32 s = 0;
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const u32 q = ((lo[c] >> (4 * (g >> 1))) & 0x0F0F0F0Fu) | (((hi[c] >> (2 * g)) & 0x03030303u) << 4);
                    s = dot4(0xE0E0E0E0u, v[c], dot4(q, v[c], s));   // q - 32
                }
                P += (int8_t)blk[192 + 8 * n + 2 * g + h] * s;
            }
            // (both scales first: a token's may be large enough for its product with P to pass the largest f32 alone)
            o = fmaf((float)P, p.da[(size_t)b * p.tok_pad + t] * half_bits_to_f32(ld2(blk + 208)), o);
            continue;
        }
        const uint8_t* blk = TYPE == JL_Q4_K ? row + (size_t)(b >> 3) * 144 : row + (size_t)b * 34;
        const uint8_t* q = TYPE == JL_Q4_K ? blk + 16 + 32 * ((b & 7) >> 1) : blk + 2;
        i32 P = 0;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const u32x4 w = ld16_a2(q + 16 * h), v = f[32 * h];
#pragma unroll
            for (int c = 0; c < 4; c++) P = dot4(TYPE == JL_Q4_K ? (w[c] >> (4 * (b & 1))) & 0x0F0F0F0Fu : w[c], v[c], P);
        }
        const size_t at = (size_t)b * p.tok_pad + t;
        if constexpr (TYPE == JL_Q4_K) {
            const u32x4 h = ld16_a2(blk);
            u32 sc, mn;
            scale_min_k4(b & 7, h.y, h.z, h.w, sc, mn);
            o = fmaf((float)P * p.da[at], half_bits_to_f32((uint16_t)(h.x & 0xFFFF)) * (float)sc, o);
            o = fmaf(p.dsum[at], -(half_bits_to_f32((uint16_t)(h.x >> 16)) * (float)mn), o);
        } else {
            o = fmaf((float)P * p.da[at], half_bits_to_f32(ld2(blk)), o);
        }
    }
    return o;
}

// t0, r0: the tile's first token and row.
template <int TYPE, bool W256, int RT, int TW>
__device__ __forceinline__ void gemm_i8_body(const GemmArgs& p, uint8_t* smem, int t0, int r0) {
    constexpr bool Q6 = TYPE == JL_Q6_K, Q4 = TYPE == JL_Q4_K;
    constexpr int NPL = Q6 ? 2 : 1, NW = TW > 4 ? TW : 4, ROWS = 32 * RT * (NW / TW);
    constexpr bool HALVES = ROWS < 16 * NW;   // fewer blocks than threads: two threads a block of 32, sixteen bytes each
    constexpr int NB = HALVES ? 1 : ROWS / (16 * NW);
    static_assert(!HALVES || TYPE == JL_Q8_0, "two threads a block: Q8_0");
    constexpr int BUF = JL_GEMM_I8_BUF_BYTES(NPL, ROWS, TW, !W256, Q4), O_D = NPL * ROWS * 128, O_DA = O_D + ROWS * 16,
                  O_M = O_DA + 4 * 32 * TW * 4, O_DS = O_M + ROWS * 16;
    // One operand, window 32: the sums start at the bits of M = 1.5 * 2^23, so that what comes out of the matrix core IS the float
    // M + P (|P| <= 32 * 127 * 128 < 2^22), and P * d = fma(M + P, d, -M d) with -M d exact (d has 17 bits at most): no
    // conversion.  (A row with a scale that is infinite comes out as NaN so: it is summed again where it is stored.)
    constexpr bool MAGIC = !W256 && NPL == 1;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), tg = TW < 4 ? wave % TW : wave;
    const bool live = t0 + 32 * tg < p.ntok;                   // else no token of its 32 exists
    const int arow = lane & 31, kg = lane >> 5;
    const int nsteps = p.k / 128;
    // this thread's share of a weight stage: block (run) qb of rows tid / 4 + 64 i
    const int qb = HALVES ? (tid >> 1) & 3 : tid & 3, myrow = HALVES ? tid >> 3 : tid >> 2;
    const uint8_t* wrow[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) wrow[i] = p.w + (size_t)min(r0 + myrow + 16 * NW * i, p.nrows - 1) * p.row_bytes;
    GemmI8Raw<TYPE> raw[NB];
    float rda[2] = {0.f, 0.f}, rds[2] = {0.f, 0.f};
    auto load_w = [&](int step, int i) __attribute__((always_inline)) {
        step = min(step, nsteps - 1);
        GemmI8Raw<TYPE>& r = raw[i];
        if constexpr (Q6) {
            const uint8_t* blk = wrow[i] + (size_t)(step >> 1) * 210;
            const int n = step & 1;
            r.q[0] = ld16_a2(blk + 64 * n + 32 * (qb & 1));
            r.q[1] = ld16_a2(blk + 64 * n + 32 * (qb & 1) + 16);
            r.h[0] = ld16_a2(blk + 128 + 32 * n);
            r.h[1] = ld16_a2(blk + 128 + 32 * n + 16);
            r.d = ((u32)ld2(blk + 192 + 8 * n + 2 * qb) << 16) | (W256 ? 0u : (u32)ld2(blk + 208));
        } else if constexpr (Q4) {
            // sub-block 4 * n + qb: nibble qb % 2 of the 32 bytes of group 2 * n + qb / 2
            const uint8_t* blk = wrow[i] + (size_t)(step >> 1) * 144;
            const int g = 2 * (step & 1) + (qb >> 1);
            r.h = ld16_a2(blk);
            r.q[0] = ld16_a2(blk + 16 + 32 * g);
            r.q[1] = ld16_a2(blk + 32 + 32 * g);
        } else {
            const uint8_t* blk = wrow[i] + (size_t)(4 * step + qb) * 34;
            r.d = ld2(blk);
            r.q[0] = ld16_a2(blk + 2 + (HALVES ? 16 * (tid & 1) : 0));
            if constexpr (!HALVES) r.q[1] = ld16_a2(blk + 18);
        }
    };
    // window 32: the stage's token scales, 4 blocks x 32 TW tokens
    auto load_scales = [&](int step) __attribute__((always_inline)) {
        step = min(step, nsteps - 1);
#pragma unroll
        for (int u = 0; u < 2 * TW / NW; u++) {
            const int idx = tid + 64 * NW * u, b = idx / (32 * TW), t = min(t0 + idx % (32 * TW), p.tok_pad - 1);
            rda[u] = p.da[(size_t)(4 * step + b) * p.tok_pad + t];
            if constexpr (Q4) rds[u] = p.dsum[(size_t)(4 * step + b) * p.tok_pad + t];
        }
    };
    // Half h of the thread's block of row set i of stage `step`, as operand bytes in `buf`; with h = 0 its scales.
    auto slice = [&](uint8_t* buf, int step, int i, int h) __attribute__((always_inline)) {
        const GemmI8Raw<TYPE>& r = raw[i];
        const int row = myrow + 16 * NW * i;
        uint8_t* dst = buf + row * 128 + 16 * ((2 * qb + (HALVES ? tid & 1 : h)) ^ (row & 7));
        float *sD = (float*)(buf + O_D) + row * 4 + qb, *sM = (float*)(buf + O_M) + row * 4 + qb;
        if constexpr (Q6) {
            const int nsh = 4 * (qb >> 1), hsh = (2 * qb - 4) & 31;
            const short sc = (short)(int8_t)(r.d >> (16 + 8 * h));
            const i16x2 S = {sc, sc}, B = {(short)(-32 * sc), (short)(-32 * sc)};
            u32x4 hi, lo;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                // (a rotation puts the two high bits at bits 4-5 of their byte)
                const u32 q = ((r.q[h][c] >> nsh) & 0x0F0F0F0Fu) | (__builtin_amdgcn_alignbit(r.h[h][c], r.h[h][c], hsh) & 0x30303030u);
                const u32 e = __builtin_amdgcn_perm(0, q, 0x0C020C00u), o = __builtin_amdgcn_perm(0, q, 0x0C030C01u);
                // sc * (q - 32) of bytes 0, 2 and 1, 3: 128 * hi + lo, 0 <= lo < 128
                const i16x2 ve = __builtin_bit_cast(i16x2, e) * S + B, vo = __builtin_bit_cast(i16x2, o) * S + B;
                const i16x2 sh7 = {7, 7};
                hi[c] = __builtin_amdgcn_perm(__builtin_bit_cast(u32, vo >> sh7), __builtin_bit_cast(u32, ve >> sh7), 0x06020400u);
                lo[c] = __builtin_amdgcn_perm(__builtin_bit_cast(u32, vo), __builtin_bit_cast(u32, ve), 0x06020400u) & 0x7F7F7F7Fu;
            }
            *(u32x4*)dst = hi;
            *(u32x4*)(dst + ROWS * 128) = lo;
            if (!W256 && h == 0) *sD = half_bits_to_f32((uint16_t)(r.d & 0xFFFF));
        } else if constexpr (Q4) {
            const int nsh = 4 * (qb & 1);
            u32x4 v;
#pragma unroll
            for (int c = 0; c < 4; c++) v[c] = (r.q[h][c] >> nsh) & 0x0F0F0F0Fu;
            *(u32x4*)dst = v;
            if (h == 0) {
                u32 sc, mn;
                scale_min_k4(4 * (step & 1) + qb, r.h.y, r.h.z, r.h.w, sc, mn);
                *sD = half_bits_to_f32((uint16_t)(r.h.x & 0xFFFF)) * (float)sc;
                *sM = -(half_bits_to_f32((uint16_t)(r.h.x >> 16)) * (float)mn);
            }
        } else {
            *(u32x4*)dst = r.q[h];
            if (h == 0) *sD = half_bits_to_f32((uint16_t)r.d);
        }
    };
    auto put_scales = [&](uint8_t* buf) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2 * TW / NW; u++) {
            ((float*)(buf + O_DA))[tid + 64 * NW * u] = rda[u];
            if constexpr (Q4) ((float*)(buf + O_DS))[tid + 64 * NW * u] = rds[u];
        }
    };
    // Part b (0..3) of the work that readies stage `step` in `buf`, and its places refilled with the stage behind it.
    auto part = [&](uint8_t* buf, int step, int b) __attribute__((always_inline)) {
        if constexpr (NB == 2) {
            slice(buf, step, b >> 1, b & 1);
            if (b & 1) load_w(step + 1, b >> 1);
        } else if constexpr (HALVES) {
            if (b == 0) slice(buf, step, 0, 0);   // (both of a block's threads store its scale)
            if (b == 0) load_w(step + 1, 0);
        } else {
            if (b < 2) slice(buf, step, 0, b);
            if (b == 1) load_w(step + 1, 0);
        }
        if (!W256 && b == 2) {
            put_scales(buf);
            load_scales(step + 1);
        }
    };
#pragma unroll
    for (int i = 0; i < NB; i++) load_w(0, i);
    if (!W256) load_scales(0);
#pragma unroll
    for (int b = 0; b < 4; b++) part(smem, 0, b);
    if (!live) {   // (uniform: this wavefront only readies weights)
        lds_barrier();
        for (int step = 0; step < nsteps; step++) {
#pragma unroll
            for (int b = 0; b < 4; b++) part(smem + ((step + 1) & 1) * BUF, step + 1, b);
            lds_barrier();
        }
        return;
    }

    // fragment (step, block) of this wavefront's 32 tokens
    const size_t ngrp = (size_t)(p.tok_pad >> 5), mygrp = (size_t)(t0 >> 5) + tg;
    auto a_frag = [&](int step, int b) {
        return ((const i32x4*)p.bq)[(((size_t)step * ngrp + mygrp) * 4 + b) * 64 + lane];
    };
    f32x16 out[RT];
#pragma unroll
    for (int j = 0; j < RT; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) out[j][e] = 0.f;
    i32x4 ring[4];
#pragma unroll
    for (int b = 0; b < 4; b++) ring[b] = a_frag(0, b);
    const int row0 = TW < 4 ? 32 * RT * (wave / TW) : 0;   // the wavefront's first row of the tile
    const i32x16 zero = {0};
    int piece[4];   // where the lane's piece of a block lies in its row
#pragma unroll
    for (int b = 0; b < 4; b++) piece[b] = 16 * ((2 * b + kg) ^ (arow & 7));
    lds_barrier();

    if constexpr (W256) {
        i32x16 ah[RT], al[RT];
        const uint8_t* drow[RT];
#pragma unroll
        for (int j = 0; j < RT; j++) drow[j] = p.w + (size_t)min(r0 + row0 + 32 * j + arow, p.nrows - 1) * p.row_bytes + 208;
        const float* dap = p.da + t0 + 32 * tg + 4 * kg;
        // (the half of the super-block is a compile-time constant: nothing in the loop is behind a branch)
        auto stage = [&](auto HALF, int step) __attribute__((always_inline)) {
            constexpr int half = decltype(HALF)::value;
            uint8_t *cur = smem + half * BUF, *nxt = smem + (half ^ 1) * BUF;
            const uint8_t* w0 = cur + (row0 + arow) * 128;
            const int nstep = min(step + 1, nsteps - 1);
            f32x4 dav[4];
            uint16_t db[RT];
            if (half) {
#pragma unroll
                for (int i = 0; i < 4; i++) dav[i] = *(const f32x4*)(dap + (size_t)(step >> 1) * p.tok_pad + 8 * i);
#pragma unroll
                for (int j = 0; j < RT; j++) db[j] = ld2(drow[j] + (size_t)(step >> 1) * 210);
            }
            i32x4 wf[2][2];
            auto read_w = [&](int n) __attribute__((always_inline)) {   // tile n = RT * block + row group
#pragma unroll
                for (int pl = 0; pl < 2; pl++)
                    wf[n & 1][pl] = *(const i32x4*)(w0 + (pl * ROWS + 32 * (n % RT)) * 128 + piece[n / RT]);
            };
            read_w(0);
#pragma unroll
            for (int n = 0; n < 4 * RT; n++) {
                const int b = n / RT, j = n % RT;
                const bool first = half == 0 && b == 0;
                if (n + 1 < 4 * RT) read_w(n + 1);
                ah[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ring[b], wf[n & 1][0], first ? zero : ah[j], 0, 0, 0);
                al[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ring[b], wf[n & 1][1], first ? zero : al[j], 0, 0, 0);
                if (j == RT - 1) {
                    ring[b] = a_frag(nstep, b);
                    part(nxt, step + 1, b);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (half) {
#pragma unroll
                for (int j = 0; j < RT; j++) {
                    const float dd = half_bits_to_f32(db[j]);
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        out[j][e] = fmaf(dav[e >> 2][e & 3], dd * (float)((ah[j][e] << 7) + al[j][e]), out[j][e]);
                }
            }
            lds_barrier();
        };
        for (int step = 0; step < nsteps; step += 2) {
            stage(GemmIntC<0>{}, step);
            stage(GemmIntC<1>{}, step + 1);
        }
    } else if constexpr (Q6) {
        // The row's scale holds for a super-block, the token's for a block: the blocks are summed with the token's scale alone, and
        // the super-block's sum meets the row's once, three vector instructions an element and block (shift and add, conversion,
        // multiply-add) where a product and a multiply-add with both scales made it four.  (A row with a scale that is infinite
        // is summed again where it is stored, block by block.)  The tile of 128 rows has no registers for the second set of sums.
        constexpr bool SUMS = TW >= 4;
        i32x16 acc[2][2];
        f32x16 sum[SUMS ? RT : 1];
        f32x4 dav[4];
        float d[RT];   // the row scales of the super-block that is summed
#pragma unroll
        for (int pl = 0; pl < 2; pl++) acc[1][pl] = zero;
#pragma unroll
        for (int j = 0; j < RT; j++) {
            d[j] = 0.f;
#pragma unroll
            for (int e = 0; e < 16; e++) sum[SUMS ? j : 0][e] = 0.f;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) dav[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        // s, row tile j's sums = (begin: nothing) + y, scaled; move: the block ends, and the token scales of the next take each quarter's place
        auto scale = [&](bool begin, bool move, const i32x16 (&y)[2], int j, const float* next) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
#pragma unroll
                for (int e = 4 * i; e < 4 * i + 4; e++) {
                    const float v = (float)((y[0][e] << 7) + y[1][e]);
                    if constexpr (SUMS) sum[j][e] = begin ? v * dav[i][e & 3] : fmaf(v, dav[i][e & 3], sum[j][e]);
                    else out[j][e] = fmaf(v * dav[i][e & 3], d[j], out[j][e]);
                }
                if (move) dav[i] = *(const f32x4*)(next + 8 * i);
            }
        };
        auto fold = [&]() __attribute__((always_inline)) {
            if constexpr (!SUMS) return;
#pragma unroll
            for (int j = 0; j < RT; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) out[j][e] = fmaf(sum[SUMS ? j : 0][e], d[j], out[j][e]);
        };
        auto stage = [&](auto HALF, int step) __attribute__((always_inline)) {
            constexpr int half = decltype(HALF)::value;
            uint8_t *cur = smem + half * BUF, *nxt = smem + (half ^ 1) * BUF;
            const uint8_t* w0 = cur + (row0 + arow) * 128;
            const int nstep = min(step + 1, nsteps - 1);
            i32x4 wf[2][2];
            auto read_w = [&](int n) __attribute__((always_inline)) {   // tile n = RT * block + row group
#pragma unroll
                for (int pl = 0; pl < 2; pl++)
                    wf[n & 1][pl] = *(const i32x4*)(w0 + (pl * ROWS + 32 * (n % RT)) * 128 + piece[n / RT]);
            };
            const float* sDa = (const float*)(cur + O_DA) + 32 * tg + 4 * kg;
            read_w(0);
#pragma unroll
            for (int n = 0; n < 4 * RT; n++) {
                const int b = n / RT, j = n % RT;
                if (n + 1 < 4 * RT) read_w(n + 1);
#pragma unroll
                for (int pl = 0; pl < 2; pl++)
                    acc[n & 1][pl] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ring[b], wf[n & 1][pl], zero, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                // the tile before
                if (j == 0) scale(half == 0 && b == 1, true, acc[1], RT - 1, sDa + b * 32 * TW);
                else scale(half == 0 && b == 0, false, acc[(n + 1) & 1], j - 1, nullptr);
                if (half == 0 && n == 0) {   // the super-block before is whole
                    fold();
#pragma unroll
                    for (int i = 0; i < RT; i++) d[i] = ((const float*)(cur + O_D))[(row0 + 32 * i + arow) * 4];
                }
                if (j == RT - 1) {
                    ring[b] = a_frag(nstep, b);
                    part(nxt, step + 1, b);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            lds_barrier();
        };
        for (int step = 0; step < nsteps; step += 2) {
            stage(GemmIntC<0>{}, step);
            stage(GemmIntC<1>{}, step + 1);
        }
        scale(false, false, acc[1], RT - 1, nullptr);
        fold();
    } else {
        i32x16 first = {0};
        if constexpr (MAGIC) {
#pragma unroll
            for (int e = 0; e < 16; e++) first[e] = 0x4B400000;
            asm volatile("" : "+v"(first));   // (held in registers: as a constant it is moved in anew for every instruction)
        }
        // Three wavefronts a SIMD (Q8_0, two row tiles): a tile's scaling right behind its own matrix instruction, whose latency the
        // other wavefronts fill; a second accumulator would be spilled.
        constexpr bool ONE = MAGIC && !Q4 && RT == 2 && TW == 4;
        i32x16 acc[ONE ? 1 : 2];
        f32x4 dav[4], dsv[4];
        float pd = 0.f, pm = 0.f, pc = 0.f;   // the row scales of the tile whose sums wait in the other accumulator; -M * pd
        acc[ONE ? 0 : 1] = zero;
#pragma unroll
        for (int i = 0; i < 4; i++) { dav[i] = f32x4{0.f, 0.f, 0.f, 0.f}; dsv[i] = f32x4{0.f, 0.f, 0.f, 0.f}; }
        // o += the sums y, scaled; next: where the token scales of the block behind lie, which take each quarter's
        // place when it has been used (MOVE: the block ends)
        auto scale = [&](auto MOVE, const i32x16& y, f32x16& o, const float* next, const float* next_s) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
#pragma unroll
                for (int e = 4 * i; e < 4 * i + 4; e++) {
                    if constexpr (MAGIC) {
                        const i32 v = y[e];   // (a copy: bit_cast of a vector's element takes another element's bits)
                        o[e] = fmaf(fmaf(__builtin_bit_cast(float, v), pd, pc), dav[i][e & 3], o[e]);
                    } else {
                        o[e] = fmaf((float)y[e] * dav[i][e & 3], pd, o[e]);
                    }
                    if constexpr (Q4) o[e] = fmaf(dsv[i][e & 3], pm, o[e]);
                }
                if constexpr (decltype(MOVE)::value) {
                    dav[i] = *(const f32x4*)(next + 8 * i);
                    if constexpr (Q4) dsv[i] = *(const f32x4*)(next_s + 8 * i);
                }
            }
        };
        for (int step = 0; step < nsteps; step++) {
            uint8_t *cur = smem + (step & 1) * BUF, *nxt = smem + ((step + 1) & 1) * BUF;
            const uint8_t* w0 = cur + (row0 + arow) * 128;
            const int nstep = min(step + 1, nsteps - 1);
            i32x4 wf[2];
            auto read_w = [&](int n) __attribute__((always_inline)) {   // tile n = RT * block + row group
                wf[n & 1] = *(const i32x4*)(w0 + 32 * (n % RT) * 128 + piece[n / RT]);
            };
            const float *sDa = (const float*)(cur + O_DA) + 32 * tg + 4 * kg, *sDs = (const float*)(cur + O_DS) + 32 * tg + 4 * kg;
            read_w(0);
            f32x4 dd[RT], dm[RT];
#pragma unroll
            for (int j = 0; j < RT; j++) {
                dd[j] = *(const f32x4*)((const float*)(cur + O_D) + (row0 + 32 * j + arow) * 4);
                if constexpr (Q4) dm[j] = *(const f32x4*)((const float*)(cur + O_M) + (row0 + 32 * j + arow) * 4);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < 4 * RT; n++) {
                const int b = n / RT, j = n % RT;
                if (n + 1 < 4 * RT) read_w(n + 1);
                if constexpr (ONE) {
                    if (j == 0) {
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            dav[i] = *(const f32x4*)(sDa + b * 32 * TW + 8 * i);
                            if constexpr (Q4) dsv[i] = *(const f32x4*)(sDs + b * 32 * TW + 8 * i);
                        }
                    }
                    acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ring[b], wf[n & 1], first, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    pd = dd[j][b];
                    pc = -12582912.f * pd;
                    if constexpr (Q4) pm = dm[j][b];
                    if (j == RT - 1) {
                        ring[b] = a_frag(nstep, b);
                        part(nxt, step + 1, b);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    scale(GemmIntC<0>{}, acc[0], out[j], nullptr, nullptr);
                    __builtin_amdgcn_sched_barrier(0);
                    continue;
                }
                acc[n & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ring[b], wf[n & 1], MAGIC ? first : zero, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                // the tile before
                if (j == 0) scale(GemmIntC<1>{}, acc[1], out[RT - 1], sDa + b * 32 * TW, sDs + b * 32 * TW);
                else scale(GemmIntC<0>{}, acc[(n + 1) & 1], out[j - 1], nullptr, nullptr);
                pd = dd[j][b];
                if constexpr (MAGIC) pc = -12582912.f * pd;
                if constexpr (Q4) pm = dm[j][b];
                if (j == RT - 1) {
                    ring[b] = a_frag(nstep, b);
                    part(nxt, step + 1, b);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            lds_barrier();
        }
        if constexpr (!ONE) scale(GemmIntC<0>{}, acc[1], out[RT - 1], nullptr, nullptr);
    }
    // store: lane = row (contiguous in memory), register = token
#pragma unroll
    for (int j = 0; j < RT; j++) {
        const int r = r0 + row0 + 32 * j + arow;
        if (r >= p.nrows) continue;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int t = t0 + 32 * tg + 8 * (e >> 2) + 4 * kg + (e & 3);
            if (t < p.ntok) p.out[(size_t)t * p.out_stride + r] = out[j][e];
        }
    }
    // An infinite scale makes a row's every sum NaN (Q6_K: NaN or infinite), whatever the token.  The decode matvec and the few-token
    // kernel give the product's infinities there, and NaN where it has none.  Not so where the token has a scale that is no number: its
    // blocks' integers are zero, its sums NaN in every row and form.  (Without that second look one infinite activation had every row
    // of sixteen tokens summed again, one by one: Q6_K 14336 x 4096, 2048 tokens 93.8 ms for 0.68, Q8_0 9.8 for 0.37.)
    if constexpr (MAGIC || (Q6 && !W256)) {
        u32 l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(l));   // (nothing of this ahead of the stages, in registers of theirs)
        const int lrow = l & 31, lkg = l >> 5;
        float sum = 0.f;   // (a product of zero with what is no number is NaN, and so is a sum with it)
#pragma unroll
        for (int j = 0; j < RT; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) sum = fmaf(out[j][e], 0.f, sum);
        const int elems = __ballot(__builtin_isnan(sum)) ? 16 : 0;   // uniform
#pragma unroll 1
        for (int e = 0; e < elems; e++) {
            const int t = t0 + 32 * tg + 8 * (e >> 2) + 4 * lkg + (e & 3);
            bool odd = false, bad = false;
#pragma unroll 1
            for (int j = 0; j < RT; j++) {
                const int r = r0 + row0 + 32 * j + lrow;
                if (t < p.ntok && r < p.nrows) odd |= !__builtin_isfinite(p.out[(size_t)t * p.out_stride + r]);   // (as stored above)
            }
            if (__ballot(odd) == 0) continue;   // uniform
            if (t < p.ntok)   // the lanes of a token look its scales through
                for (int b = lrow; b < p.k / 32; b += 32) bad |= !__builtin_isfinite(p.da[(size_t)b * p.tok_pad + t]);
            if ((u32)(__ballot(bad) >> (32 * lkg)) == 0) {
#pragma unroll 1
                for (int j = 0; j < RT; j++) {
                    const int r = r0 + row0 + 32 * j + lrow;
                    if (t >= p.ntok || r >= p.nrows) continue;
                    float* o = p.out + (size_t)t * p.out_stride + r;
                    if (!__builtin_isfinite(*o)) *o = gemm_i8_one<TYPE>(p, p.w + (size_t)r * p.row_bytes, t);
                }
            }
        }
    }
}
