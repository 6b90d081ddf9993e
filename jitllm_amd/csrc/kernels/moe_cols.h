// Grouped expert matmul for experts of some tens of columns (a prompt through a mixture block): Q4_K sheets, GGUF rows or
// packed planes, and Q6_K rows, the k-quant activation window of 256.  Per (column, row) it is the decode matvec's value.
//
// A wavefront owns 32 rows and up to 64 columns, and turns its rows' bytes into the matrix operand in registers, once for
// all of the columns (groups of 32 columns decoded a sheet twice at 48 columns an expert, tiles of 128 x 64 staged the decoded
// operand in LDS); no weight is written back to LDS.  Four such wavefronts a workgroup share the columns, which come to LDS
// half a super-block (Q6_K: a whole one) at a time by loads that write LDS directly, as do Q4_K's rows.  Source rows are
// quantized once each (the prep), not once a column: a column's record is found through the routing's own list.
//
// 128 experts, 48 columns each, us (prep included): Q4_K, two banks of 768 x 2048 177 -> 98; 2048 x 768 98 -> 67; Q6_K
// 2048 x 768 115 -> 87.  The block of 777 rows, top 8 (Q4_K, Q6_K down): 339 -> 234, 216 with all that came behind (router, lists, the first
// rows asked for ahead of the columns).
//
// What bounds it (two banks of 768 x 2048, timestamps in the kernel): a super-block takes 1.0 us of work -- vector
// instructions, eight a matrix instruction (decoding 4.5 at 64 columns, the epilogue 3), which a SIMD issues one after the
// other with its matrix instructions -- and 1.0 us of waiting for the rows, of which one super-block is on the way at a
// time (two workgroups of 72 KB of LDS fill a CU; one workgroup of eight wavefronts with two or three on the way gained
// nothing, its wavefronts wait for each other).  Rows straight into registers, a lane a row: 97 us against 86 (sixteen
// bytes of 64 lines an instruction keep L1 busy all of the time, Q6_K 79 against 71).
#pragma once
#include "gemm_i8.h"

#pragma clang fp contract(off)

// KO: 0 Q4_K GGUF rows, 1 Q4_K planes, 2 Q6_K rows.  A wavefront takes four (record, super-block) tasks.
template <int KO>
__device__ __forceinline__ void moe_cols_prep_body(const MoeColsPrepArgs& args) {
    MoeColsPrepArgs p = args;
    JL_NOW(p.x, p.x2, p.src, p.rec, p.aug, p.da, p.k, p.nrec);
    constexpr int TB = 4;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const float *x = as_global(p.x), *x2 = as_global(p.x2);
    const u32* src = as_global(p.src);
    const u32 nsb = (u32)p.k / 256, ntask = (u32)p.nrec * nsb, t0 = (blockIdx.x * 4 + wave) * TB;
    if (t0 >= ntask) return;
    f32x4 v[TB], u[TB];
#pragma unroll
    for (int b = 0; b < TB; b++) {
        const u32 t = min(t0 + b, ntask - 1), r = t / nsb, sb = t - r * nsb;
        const size_t at = (size_t)(src ? (u32)__builtin_amdgcn_readfirstlane((i32)src[r]) : r) * p.k + sb * 256 + 4 * lane;
        v[b] = *(const f32x4*)(x + at);
        u[b] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (x2) u[b] = *(const f32x4*)(x2 + at);
    }
#pragma unroll
    for (int b = 0; b < TB; b++) {
        const u32 t = t0 + b;
        if (t >= ntask) break;   // uniform
        f32x4 w = v[b];
        if (x2) w = f32x4{silu_f32(w.x) * u[b].x, silu_f32(w.y) * u[b].y, silu_f32(w.z) * u[b].z, silu_f32(w.w) * u[b].w};
        const u32 m = max(max(abs_bits(w.x), abs_bits(w.y)), max(abs_bits(w.z), abs_bits(w.w)));
        float d;
        i32 sum16;
        const u32 q = quantize4(w, wave_amax_256(m), d, sum16);
        if (lane == 0) as_global(p.da)[t] = d;
        u32* rec = as_global(p.rec) + (size_t)t * (JL_MC_REC(KO == 2) / 4);
        if constexpr (KO == 2) {
            rec[lane] = q;
        } else {
            const i32 a32 = sum16 + dpp_i32<JL_DPP_ROW_HALF_MIRROR, 0xf>(0, sum16);
            const int sub = lane >> 3;
            if ((lane & 7) == 0) {
                _Float16* aug = (_Float16*)as_global(p.aug) + (size_t)t * 16;
                aug[sub] = (_Float16)(float)(a32 & 31);
                aug[8 + sub] = (_Float16)(float)(a32 >> 5);
            }
            auto f = [](u32 x, int b2) { return (_Float16)(float)(int8_t)(x >> (8 * b2)); };
            const f16x2 p02 = {f(q, 0), f(q, 2)}, p13 = {f(q, 1), f(q, 3)};
            // the word's high nibbles' partner is eight lanes on (rows: the next sub-block) or four (planes: elements + 16)
            constexpr int SHL = KO == 1 ? 0x104 : 0x108;
            const u32 a = __builtin_bit_cast(u32, p02), c = __builtin_bit_cast(u32, p13);
            const u32 a2 = (u32)dpp_i32<SHL, 0xf>(0, (i32)a), c2 = (u32)dpp_i32<SHL, 0xf>(0, (i32)c);
            const int ks = KO == 1 ? 4 * (sub & 3) + (lane & 3) : 8 * ((sub >> 1) & 1) + (lane & 7);
            if ((lane & (KO == 1 ? 4 : 8)) == 0) ((u32x4*)rec)[2 * ks + (sub >> 2)] = u32x4{a, a2, c, c2};
        }
    }
}

// Bytes b0 and b1 of w, integers up to 63, as a pair of f16: (1024 + n) by its bits, then m * n + a in one exact step.
__device__ __forceinline__ f16x2 mc_pair(u32 w, int b0, int b1, f16x2 m, f16x2 a) {
    const u32 v = __builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | (u32)b0 | ((u32)b1 << 16));
    return __builtin_elementwise_fma(__builtin_bit_cast(f16x2, v), m, a);
}
// The multipliers and addends of moe_g16_word for the sub-block pair in bytes 2 hh and 2 hh + 1 of w (scales of six bits).
__device__ __forceinline__ void mc_scales(u32 w, int hh, GemmWideScale& k) {
    const f16x2 one = {(_Float16)1.0f, (_Float16)1.0f}, m1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
    const f16x2 m64 = {(_Float16)-64.0f, (_Float16)-64.0f}, r16 = {(_Float16)0.0625f, (_Float16)0.0625f};
    k.mlo = mc_pair(w, 2 * hh, 2 * hh, one, m1024);
    k.alo = k.mlo * m1024;
    const f16x2 hi = mc_pair(w, 2 * hh + 1, 2 * hh + 1, one, m1024);
    k.mhi = hi * r16;
    k.ahi = hi * m64;
}
// The minimums of a Q4_K super-block as a matrix operand: times 1 for the low bits of the columns' sums (kg = 0), 32 for the rest.
__device__ __forceinline__ f16x8 mc_mins(u32 lo, u32 hi, int kg) {
    const _Float16 mul = kg ? (_Float16)32.0f : (_Float16)1.0f, add = kg ? (_Float16)-32768.0f : (_Float16)-1024.0f;
    const f16x2 m = {mul, mul}, a = {add, add};
    const u32x4 o = {__builtin_bit_cast(u32, mc_pair(lo, 0, 1, m, a)), __builtin_bit_cast(u32, mc_pair(lo, 2, 3, m, a)),
                     __builtin_bit_cast(u32, mc_pair(hi, 0, 1, m, a)), __builtin_bit_cast(u32, mc_pair(hi, 2, 3, m, a))};
    return __builtin_bit_cast(f16x8, o);
}

// lane = row (contiguous in memory), register = column
template <int G>
__device__ __forceinline__ void mc_store(const MoeColsArgs& p, const f32x16 (&out)[G], int mat, int r, int kg, u32 c0, int n) {
    float* o = p.out[mat];
    asm volatile("" : "+v"(r));   // (the addresses are formed here, not kept in registers over the loop)
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = 32 * g + 8 * (i >> 2) + 4 * kg + (i & 3);
            if (r < p.nrows && t < n) o[(size_t)(c0 + t) * p.nrows + r] = out[g][i];
        }
}

// A lane's places among a Q4_K tile's rows: 18 instructions of 64 pieces, nine pieces a row; four a wavefront, the last two the first two
// wavefronts'.
struct MoeColsQ4Rows { u32 woff[4], xoff; };
__device__ __forceinline__ void moe_cols_q4_places(const MoeColsArgs& p, int last, MoeColsQ4Rows& w) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    auto piece_at = [&](int i) {
        const int idx = 64 * i + lane, row = idx / 9;
        return (u32)min(row, last) * (u32)p.row_bytes + 16 * (u32)(idx - 9 * row);
    };
#pragma unroll
    for (int i = 0; i < 4; i++) w.woff[i] = piece_at(4 * wave + i);
    w.xoff = piece_at(16 + (wave & 1));
}
// Asks for the first super-block's rows.
__device__ __forceinline__ void moe_cols_q4_rows(uint8_t* smem, const uint8_t* sheet, const MoeColsQ4Rows& w) {
    constexpr int O_W = 2 * JL_MC_A;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const u32 lds0 = lds_address(smem);
#pragma unroll
    for (int i = 0; i < 4; i++) load_lds16(sheet, w.woff[i], __builtin_amdgcn_readfirstlane(lds0 + O_W + 4096 * wave + 1024 * i));
    if (wave < 2) load_lds16(sheet, w.xoff, __builtin_amdgcn_readfirstlane(lds0 + O_W + 1024 * (16 + wave)));
}
// Q4_K rows.  G: groups of 32 columns (n columns exist).  The rows' bytes come to LDS as they lie, 144 contiguous bytes a
// row (straight into registers, a lane a row, is sixteen bytes of 64 lines an instruction), and each wavefront reads its own.
// asked: the first super-block's rows are already on their way.
template <int G>
__device__ __forceinline__ void moe_cols_q4_tile(const MoeColsArgs& p, uint8_t* smem, const uint8_t* sheet, const MoeColsQ4Rows& w, bool asked, int mat, int r0, u32 c0, int n) {
    constexpr int O_W = 2 * JL_MC_A, O_AUG = O_W + 2 * JL_MC_W, O_DA = O_AUG + 2 * 64 * 32;
    constexpr int NA = 2 * G;   // a wavefront's instructions for half a super-block of columns; NS: for its weights, sums, scales
    constexpr int NS = 5;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, kg = lane >> 5, nsb = p.k / 256;
    const u32 lds0 = lds_address(smem);
    const u32 crec = p.map ? p.map[c0 + min(lane, n - 1)] : c0 + min(lane, n - 1);
    u32 woff[4], xoff = w.xoff;
#pragma unroll
    for (int i = 0; i < 4; i++) woff[i] = w.woff[i];
    // the fifth: weights, or 32 columns' sums (wavefronts 2, 3); and wavefront 0 brings the scales
    const uint8_t* xbase = wave < 2 ? sheet : p.aug;
    const u32 xstep = wave < 2 ? 144 : 32, xto = wave < 2 ? O_W + 1024 * (16 + wave) : O_AUG + 1024 * (wave & 1), xpar = wave < 2 ? JL_MC_W : 64 * 32;
    const u32 srec = (u32)__shfl((int)crec, 32 * (wave & 1) + (lane >> 1), 64);
    if (wave >= 2) xoff = srec * (u32)(nsb * 32) + 16 * (lane & 1);
    // columns: four an instruction, sixteen pieces each; piece P of column c lies at place P ^ c % 16, so that a fragment's
    // reads spread over the banks
    u32 aoff[NA];
#pragma unroll
    for (int i = 0; i < NA; i++) {
        const int col = 4 * NA * wave + 4 * i + (lane >> 4);
        aoff[i] = (u32)__shfl((int)crec, col, 64) * (u32)(nsb * 512) + 16 * ((lane & 15) ^ (col & 15));
    }
    const u32 doff = crec * (u32)(nsb * 4);
    auto load_a = [&](int h) __attribute__((always_inline)) {
        const uint8_t* base = p.rec + (size_t)h * 256;
        const u32 to = lds0 + (h & 1) * JL_MC_A + 1024 * NA * wave;
#pragma unroll
        for (int i = 0; i < NA; i++) load_lds16(base, aoff[i], __builtin_amdgcn_readfirstlane(to + 1024 * i));
    };
    auto load_w = [&](int sb, auto ROWS) __attribute__((always_inline)) {
        const uint8_t* base = sheet + (size_t)sb * 144;
        const u32 to = lds0 + O_W + (sb & 1) * JL_MC_W + 4096 * wave;
        if constexpr (decltype(ROWS)::value != 0)
#pragma unroll
            for (int i = 0; i < 4; i++) load_lds16(base, woff[i], __builtin_amdgcn_readfirstlane(to + 1024 * i));
        if (decltype(ROWS)::value != 0 || wave >= 2) load_lds16(xbase + (size_t)sb * xstep, xoff, __builtin_amdgcn_readfirstlane(lds0 + xto + (sb & 1) * xpar));
        if (wave == 0) load_lds4((const uint8_t*)p.da + (size_t)sb * 4, doff, __builtin_amdgcn_readfirstlane(lds0 + O_DA + (sb & 1) * 256));
    };
    load_a(0);
    if (!asked) moe_cols_q4_rows(smem, sheet, w);   // uniform
    load_w(0, GemmIntC<0>{});
    f32x16 out[G], acc[G];
    const f32x16 zero = {0.f};
#pragma unroll
    for (int g = 0; g < G; g++) out[g] = zero;
    u32 mask_lo = 0x000F000Fu, mask_hi = 0x00F000F0u, magic = 0x64006400u;
    asm volatile("" : "+v"(mask_lo), "+v"(mask_hi), "+v"(magic));
    u32 place[8];
#pragma unroll
    for (int i = 0; i < 8; i++) place[i] = l32 * 256 + 16 * ((2 * i + kg) ^ (l32 & 15));
    const uint8_t* wlane = smem + O_W + (32 * wave + l32) * 144;

    auto stage = [&](auto PAR, int sb) __attribute__((always_inline)) {
        constexpr int cur = decltype(PAR)::value;
        const uint8_t* W = wlane + cur * JL_MC_W;
        const bool more = sb + 1 < nsb;   // uniform
        u32x4 hd, q[4];
        GemmScaleBytes six;   // this lane's six-bit scales of half kg are sc, the minimums all eight
        u32 sc6 = 0;
#pragma unroll
        for (int hf = 0; hf < 2; hf++) {
            // This half's columns, and with the first half the super-block's weights, have arrived everywhere; the place of
            // the half before is free.  (The requests behind them that may be out: the next super-block's weights.)
            if (hf == 0 || !more) wait_loads<0>();
            else if (wave == 0) wait_loads<NS + 1>();
            else wait_loads<NS>();
            lds_barrier();
            if (hf == 0 || more) load_a(2 * sb + hf + 1);
            if (hf == 0 && more) load_w(sb + 1, GemmIntC<1>{});
            const uint8_t* A = smem + hf * JL_MC_A;
            if (hf == 0) {
                hd = *(const u32x4*)W;
                q[0] = *(const u32x4*)(W + 16 + 64 * kg);
                q[1] = *(const u32x4*)(W + 32 + 64 * kg);
            }
            f16x8 af[3][G];
            u32x4 bw[2];
            GemmWideScale sc;
            auto read_a = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
                for (int g = 0; g < G; g++) af[ks % 3][g] = *(const f16x8*)(A + g * 8192 + place[ks]);
            };
            // half x of K-step ks's word: four weights
            auto decode = [&](int ks, int x) __attribute__((always_inline)) {
                const u32 w0 = q[2 * hf + (ks >> 2)][ks & 3], w = x ? w0 >> 8 : w0;
                auto nib = [&](u32 v, u32 mask) { return __builtin_bit_cast(f16x2, (v & mask) | magic); };
                bw[ks & 1][2 * x] = __builtin_bit_cast(u32, __builtin_elementwise_fma(nib(w, mask_lo), sc.mlo, sc.alo));
                bw[ks & 1][2 * x + 1] = __builtin_bit_cast(u32, __builtin_elementwise_fma(nib(w, mask_hi), sc.mhi, sc.ahi));
            };
            read_a(0);
            read_a(1);
            if (hf == 0) {
                six = gemm_scale_bytes(hd.y, hd.z, hd.w);
                u32 lo6 = hd.y & 0x3F3F3F3Fu, hi6 = (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u);
                asm volatile("" : "+v"(lo6), "+v"(hi6));   // (a select, not a branch)
                sc6 = kg ? hi6 : lo6;
            }
            mc_scales(sc6, hf, sc);
            decode(0, 0);
            decode(0, 1);
#pragma unroll
            for (int ks = 0; ks < 8; ks++) {
                if (ks + 2 < 8) read_a(ks + 2);
                if (hf == 0 && (ks == 4 || ks == 5)) q[ks - 2] = *(const u32x4*)(W + 16 * (ks - 1) + 64 * kg);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int g = 0; g < G; g++) {
                    acc[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[ks % 3][g], __builtin_bit_cast(f16x8, bw[ks & 1]),
                                                                    hf == 0 && ks == 0 ? zero : acc[g], 0, 0, 0);
                    if (ks + 1 < 8) {
                        if (g == 0) decode(ks + 1, 0);
                        if (g == G - 1) decode(ks + 1, 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        // out += d_a * (d * P - dmin * M)
        const f16x8 mm = mc_mins(six.mn_lo, six.mn_hi, kg);
        const float dd = half_bits_to_f32((uint16_t)(hd.x & 0xFFFF)), dmin = half_bits_to_f32((uint16_t)(hd.x >> 16));
        const float* sda = (const float*)(smem + O_DA + cur * 256) + 4 * kg;
#pragma unroll
        for (int g = 0; g < G; g++) {
            const f16x8 aug = *(const f16x8*)(smem + O_AUG + cur * 2048 + (32 * g + l32) * 32 + 16 * kg);
            const f32x16 accM = __builtin_amdgcn_mfma_f32_32x32x16_f16(aug, mm, zero, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const f32x4 dav = *(const f32x4*)(sda + 32 * g + 8 * i);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float uu = fmaf(dd, acc[g][4 * i + j], -(dmin * accM[4 * i + j]));
                    out[g][4 * i + j] = fmaf(dav[j], uu, out[g][4 * i + j]);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int sb = 0; sb < nsb; sb += 2) {
        stage(GemmIntC<0>{}, sb);
        if (sb + 1 < nsb) stage(GemmIntC<1>{}, sb + 1);
    }
    mc_store<G>(p, out, mat, r0 + 32 * wave + l32, kg, c0, n);
    lds_barrier();   // LDS is free for the next columns
}

// Q6_K rows: 210-byte blocks lie on two-byte boundaries, so the rows' bytes come through registers (sixteen bytes a lane along
// the row), a super-block ahead, and are laid down in LDS when the one before has been used.
template <int G>
__device__ __forceinline__ void moe_cols_q6_tile(const MoeColsArgs& p, uint8_t* smem, int e, int mat, int r0, u32 c0, int n) {
    constexpr int A_SB = 64 * 256, O_W = 2 * A_SB, O_D = O_W + JL_MC_Q6_W + 128 * 16, O_DA = O_D + 128 * 2;
    constexpr int NA = 2 * G, AR = 3;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, kg = lane >> 5, nsb = p.k / 256;
    const u32 lds0 = lds_address(smem);
    const u32 crec = p.map ? p.map[c0 + min(lane, n - 1)] : c0 + min(lane, n - 1);
    const uint8_t* sheet = p.bank[mat] + (size_t)e * p.sheet_bytes + (size_t)r0 * p.row_bytes;
    const int last = p.nrows - 1 - r0;
    // thirteen pieces a row, and the two bytes behind them; the last round is half empty (it repeats the last piece, which
    // goes to a place of no use)
    u32 woff[7], wto[7];
#pragma unroll
    for (int i = 0; i < 7; i++) {
        const int idx = min(tid + 256 * i, 128 * 13 - 1), row = idx / 13, pc = idx - 13 * row;
        woff[i] = (u32)min(row, last) * (u32)p.row_bytes + 16 * (u32)pc;
        wto[i] = O_W + (tid + 256 * i < 128 * 13 ? row * 208 + 16 * pc : JL_MC_Q6_W + 16 * (tid - 128));
    }
    const u32 doff = (u32)min(tid & 127, last) * (u32)p.row_bytes + 208;
    u32x4 raw[7];
    u32 rd = 0;
    float rda = 0.f;
    auto load_w = [&](int sb) __attribute__((always_inline)) {
        const uint8_t* base = sheet + (size_t)sb * 210;
#pragma unroll
        for (int i = 0; i < 7; i++) raw[i] = ld16_a2(base + woff[i]);
        rd = ld2(base + doff);
        rda = p.da[(size_t)crec * nsb + sb];
    };
    auto put_w = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 7; i++) *(u32x4*)(smem + wto[i]) = raw[i];
        *(uint16_t*)(smem + O_D + 2 * (tid & 127)) = (uint16_t)rd;
        *(float*)(smem + O_DA + 4 * lane) = rda;   // (every wavefront the same values)
    };
    u32 aoff[NA];   // columns, as in the Q4_K tile
#pragma unroll
    for (int i = 0; i < NA; i++) {
        const int col = 4 * NA * wave + 4 * i + (lane >> 4);
        aoff[i] = (u32)__shfl((int)crec, col, 64) * (u32)(nsb * 256) + 16 * ((lane & 15) ^ (col & 15));
    }
    auto load_a = [&](int sb) __attribute__((always_inline)) {
        const uint8_t* base = p.rec + (size_t)sb * 256;
        const u32 to = lds0 + (sb & 1) * A_SB + 1024 * NA * wave;
#pragma unroll
        for (int i = 0; i < NA; i++) load_lds16(base, aoff[i], __builtin_amdgcn_readfirstlane(to + 1024 * i));
    };
    load_a(0);
    load_w(0);
    f32x16 out[G];
    const f32x16 fzero = {0.f};
#pragma unroll
    for (int g = 0; g < G; g++) out[g] = fzero;
    const uint8_t* W = smem + O_W + (32 * wave + l32) * 208;
    const u32 place = (u32)l32 * 256 + 16 * ((8 * kg) ^ (l32 & 15));
    const i32x16 zero = {0};
    for (int sb = 0; sb < nsb; sb++) {
        wait_loads<0>();    // this super-block's columns (in LDS) and weights (in registers) are here
        lds_barrier();   // ... everywhere, and the one before has been used
        put_w();
        if (sb + 1 < nsb) load_a(sb + 1);
        load_w(min(sb + 1, nsb - 1));
        lds_barrier();
        const uint8_t* A = smem + (sb & 1) * A_SB;
        u32x4 q[4], h[2];
#pragma unroll
        for (int v = 0; v < 2; v++) h[v] = *(const u32x4*)(W + 128 + 32 * kg + 16 * v);
        const u32x2 sc8 = *(const u32x2*)(W + 192 + 8 * kg);
#pragma unroll
        for (int v = 0; v < 4; v++) q[v] = *(const u32x4*)(W + 64 * kg + 16 * v);
        i32x16 ah[G], al[G];
        i32x4 af[AR][G], hi[2], lo[2];
        auto read_a = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < G; g++) af[ks % AR][g] = *(const i32x4*)(A + g * 8192 + (place ^ (16 * ks)));
        };
        // word c of K-step ks: four weights sc * (q - 32) = 128 * hi + lo, 0 <= lo < 128
        auto decode = [&](int ks, int c) __attribute__((always_inline)) {
            const int nsh = 4 * (ks >> 2), hsh = (4 * (ks >> 2) + 2 * ((ks >> 1) & 1) - 4) & 31;
            const short sc = (short)(int8_t)(sc8[ks >> 2] >> (8 * (ks & 3)));
            const i16x2 S = {sc, sc}, B = {(short)(-32 * sc), (short)(-32 * sc)}, sh7 = {7, 7};
            // (a rotation puts the two high bits at bits 4-5 of their byte)
            const u32 v = ((q[ks & 3][c] >> nsh) & 0x0F0F0F0Fu) | (__builtin_amdgcn_alignbit(h[ks & 1][c], h[ks & 1][c], hsh) & 0x30303030u);
            const u32 ev = __builtin_amdgcn_perm(0, v, 0x0C020C00u), od = __builtin_amdgcn_perm(0, v, 0x0C030C01u);
            const i16x2 ve = __builtin_bit_cast(i16x2, ev) * S + B, vo = __builtin_bit_cast(i16x2, od) * S + B;
            hi[ks & 1][c] = (i32)__builtin_amdgcn_perm(__builtin_bit_cast(u32, vo >> sh7), __builtin_bit_cast(u32, ve >> sh7), 0x06020400u);
            lo[ks & 1][c] = (i32)(__builtin_amdgcn_perm(__builtin_bit_cast(u32, vo), __builtin_bit_cast(u32, ve), 0x06020400u) & 0x7F7F7F7Fu);
        };
#pragma unroll
        for (int ks = 0; ks < AR - 1; ks++) read_a(ks);
#pragma unroll
        for (int c = 0; c < 4; c++) decode(0, c);
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            if (ks + AR - 1 < 8) read_a(ks + AR - 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < G; g++) {
                // (the next K-step's four words are decoded under the matrix instructions of this one)
                ah[g] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[ks % AR][g], hi[ks & 1], ks == 0 ? zero : ah[g], 0, 0, 0);
                if (ks + 1 < 8) {
                    decode(ks + 1, 4 / G * g);
                    if (G == 1) decode(ks + 1, 1);
                }
                __builtin_amdgcn_sched_barrier(0);
                al[g] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[ks % AR][g], lo[ks & 1], ks == 0 ? zero : al[g], 0, 0, 0);
                if (ks + 1 < 8) {
                    decode(ks + 1, G == 1 ? 2 : 2 * g + 1);
                    if (G == 1) decode(ks + 1, 3);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        const float dd = half_bits_to_f32(*(const uint16_t*)(smem + O_D + 2 * (32 * wave + l32)));
        const float* sda = (const float*)(smem + O_DA) + 4 * kg;
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const f32x4 dav = *(const f32x4*)(sda + 32 * g + 8 * i);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    out[g][4 * i + j] = fmaf(dav[j], dd * (float)((ah[g][4 * i + j] << 7) + al[g][4 * i + j]), out[g][4 * i + j]);
            }
        __builtin_amdgcn_sched_barrier(0);
    }
    mc_store<G>(p, out, mat, r0 + 32 * wave + l32, kg, c0, n);
    wait_loads<0>();
    lds_barrier();   // LDS is free for the next columns
}

// Q4_K planes: a lane's words of its row straight into registers, a super-block ahead (every request is 32 rows' words of a plane).
struct MoeColsPlaneWords { u32x4 h, q[4]; };   // (d, dmin) and the words of six-bit fields; words of K-steps 4 v ..
template <int G>
__device__ __forceinline__ void moe_cols_planes_tile(const MoeColsArgs& p, uint8_t* smem, int e, int mat, int r0, u32 c0, int n) {
    constexpr int REC = 512, BUF = 64 * REC, O_AUG = 2 * BUF, AUG = 64 * 32, O_DA = O_AUG + 2 * AUG, NW = 20,
                  AR = 3;   // fragments of the columns in flight: K-step ks + 2's are asked for with ks's matrix work
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, kg = lane >> 5, nsb = p.k / 256;
    const int row = min(r0 + 32 * wave + l32, p.nrows - 1);

    // ---- weights: a uniform base and a 32-bit lane offset
    const size_t pst = (size_t)p.pstride, at = (size_t)e * p.sheet_words + (size_t)e * p.row_step;
    const char *pq = (const char*)(p.pqs[mat] + at), *pd = (const char*)(p.pd[mat] + at), *ps = (const char*)(p.psc[mat] + at);
    const u32 rowo = 4 * (u32)row, qo = 4 * ((u32)kg * 16 * (u32)p.pstride + (u32)row);
    MoeColsPlaneWords raw[2];
    auto load_w = [&](int sb, MoeColsPlaneWords& r) __attribute__((always_inline)) {
        auto at32 = [&](const char* base, size_t plane, u32 off) { return *(const u32*)(base + 4 * plane * pst + off); };
        r.h = u32x4{at32(pd, sb, rowo), at32(ps, 3 * sb, rowo), at32(ps, 3 * sb + 1, rowo), at32(ps, 3 * sb + 2, rowo)};
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
            for (int c = 0; c < 4; c++) r.q[v][c] = at32(pq, (size_t)sb * 32 + 4 * v + c, qo);
    };
    auto arrived = [&](MoeColsPlaneWords& r) __attribute__((always_inline)) {
        asm volatile("" : "+v"(r.h), "+v"(r.q[0]), "+v"(r.q[1]), "+v"(r.q[2]), "+v"(r.q[3]));
    };

    // ---- columns: a wavefront brings the records of 8 G of them into LDS, two an instruction; piece P of column c lies
    // at place P ^ c of its record, so that a fragment's 32 reads spread over the banks
    const u32 crec = p.map ? p.map[c0 + min(lane, n - 1)] : c0 + min(lane, n - 1);
    constexpr int PP = REC / 16;                     // pieces a record
    constexpr int CI = 64 / PP, NI = 8 * G / CI;     // columns an instruction, instructions
    u32 voff[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int col = 8 * G * wave + CI * i + lane / PP;
        voff[i] = (u32)__shfl((int)crec, col, 64) * (u32)(nsb * REC) + 16 * ((lane % PP) ^ (col % PP));
    }
    const u32 lds0 = lds_address(smem);
    auto dma = [&](int sb) __attribute__((always_inline)) {
        const uint8_t* base = p.rec + (size_t)sb * REC;
        const u32 to = lds0 + (sb & 1) * BUF + 8 * G * REC * wave;
#pragma unroll
        for (int i = 0; i < NI; i++) load_lds16(base, voff[i], __builtin_amdgcn_readfirstlane(to + 1024 * i));
    };
    // block sums (thread = column tid / 4, eight bytes) and scales (thread = column), through registers
    const u32 arec = (u32)__shfl((int)crec, 16 * wave + (lane >> 2), 64);
    u32x2 raug = {0u, 0u};
    float rda = 0.f;
    auto load_s = [&](int sb) __attribute__((always_inline)) {
        raug = *(const u32x2*)(p.aug + ((size_t)arec * nsb + sb) * 32 + 8 * (tid & 3));
        rda = p.da[(size_t)crec * nsb + sb];
    };
    auto put_s = [&](int sb) __attribute__((always_inline)) {
        *(u32x2*)(smem + O_AUG + (sb & 1) * AUG + 8 * tid) = raug;
        *(float*)(smem + O_DA + (sb & 1) * 256 + 4 * lane) = rda;   // (every wavefront the same values)
    };

    dma(0);
    load_s(0);
    load_w(0, raw[0]);
    f32x16 out[G];
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
        for (int i = 0; i < 16; i++) out[g][i] = 0.f;
    put_s(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NW) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");

    u32 mask_lo = 0x000F000Fu, mask_hi = 0x00F000F0u, magic = 0x64006400u;
    asm volatile("" : "+v"(mask_lo), "+v"(mask_hi), "+v"(magic));
    const u32 abase = (u32)l32 * REC + 16 * (kg ^ l32);

    auto stage = [&](auto PAR, int sb) __attribute__((always_inline)) {
        constexpr int cur = decltype(PAR)::value;
        const bool more = sb + 1 < nsb;   // uniform
        // The weights have to be here before the next requests go out: the compiler does not count the loads into LDS, so a
        // wait for the weights put behind them would be one for them as well.
        arrived(raw[cur]);
        if (more) dma(sb + 1);
        load_s(min(sb + 1, nsb - 1));
        load_w(min(sb + 1, nsb - 1), raw[cur ^ 1]);
        __builtin_amdgcn_sched_barrier(0);
        const uint8_t* A = smem + cur * BUF;
        const MoeColsPlaneWords& r = raw[cur];
        const float* sda = (const float*)(smem + O_DA + cur * 256) + 4 * kg;
        f32x16 acc[G];
        const f32x16 zero = {0.f};
        f16x8 af[AR][G];
        u32x4 bw[2];
        auto read_a = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < G; g++) af[ks % AR][g] = *(const f16x8*)(A + g * 32 * REC + (abase ^ (32 * ks)));
        };
        // K-step ks's word: the lane's scales of it, then its eight weights in two halves
        GemmWideScale sc;
        auto scales = [&](int ks) __attribute__((always_inline)) {
            if ((ks & 3) == 0) gemm_wide_scale_planes(r.h, 4 * kg + (ks >> 2), sc);
        };
        auto decode = [&](int ks, int h) __attribute__((always_inline)) {
            const u32 w = h ? r.q[ks >> 2][ks & 3] >> 8 : r.q[ks >> 2][ks & 3];
            auto nib = [&](u32 v, u32 mask) { return __builtin_bit_cast(f16x2, (v & mask) | magic); };
            bw[ks & 1][2 * h] = __builtin_bit_cast(u32, __builtin_elementwise_fma(nib(w, mask_lo), sc.mlo, sc.alo));
            bw[ks & 1][2 * h + 1] = __builtin_bit_cast(u32, __builtin_elementwise_fma(nib(w, mask_hi), sc.mhi, sc.ahi));
        };
#pragma unroll
        for (int ks = 0; ks < AR - 1; ks++) read_a(ks);
        scales(0);
        decode(0, 0);
        decode(0, 1);
#pragma unroll
        for (int ks = 0; ks < 16; ks++) {
            if (ks + AR - 1 < 16) read_a(ks + AR - 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < G; g++) {
                acc[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[ks % AR][g], __builtin_bit_cast(f16x8, bw[ks & 1]), ks == 0 ? zero : acc[g], 0, 0, 0);
                if (ks + 1 < 16) {
                    if (g == 0) {
                        scales(ks + 1);
                        decode(ks + 1, 0);
                    }
                    if (g == G - 1) decode(ks + 1, 1);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        const float mul = kg == 0 ? 1.0f : 32.0f;
        f16x8 mm;
#pragma unroll
        for (int b = 0; b < 8; b++) mm[b] = (_Float16)((float)gemm_stream_field(r.h, 2 * b + 1) * mul);
        const float dd = half_bits_to_f32((uint16_t)(r.h.x & 0xFFFF)), dmin = half_bits_to_f32((uint16_t)(r.h.x >> 16));
#pragma unroll
        for (int g = 0; g < G; g++) {
            const f16x8 aug = *(const f16x8*)(smem + O_AUG + cur * AUG + (32 * g + l32) * 32 + 16 * kg);
            const f32x16 accM = __builtin_amdgcn_mfma_f32_32x32x16_f16(aug, mm, zero, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const f32x4 dav = *(const f32x4*)(sda + 32 * g + 8 * i);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float uu = fmaf(dd, acc[g][4 * i + j], -(dmin * accM[4 * i + j]));
                    out[g][4 * i + j] = fmaf(dav[j], uu, out[g][4 * i + j]);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) put_s(sb + 1);
        // the next super-block's records have arrived (its weights may still be on the way)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NW) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    for (int sb = 0; sb < nsb; sb += 2) {
        stage(GemmIntC<0>{}, sb);
        if (sb + 1 < nsb) stage(GemmIntC<1>{}, sb + 1);
    }
    mc_store<G>(p, out, mat, r0 + 32 * wave + l32, kg, c0, n);
    lds_barrier();   // LDS is free for the next columns
}

// grid = 8 * ceil(items / 8), block = 256; item = ((expert, matrix), block of 128 rows, share of the columns), the XCD that
// the workgroup's number names taking a run of them, so that an expert's columns are fetched into one L2.
template <int KO>
__device__ __forceinline__ void moe_cols_body(const MoeColsArgs& p, uint8_t* smem) {
    const u32 per_xcd = gridDim.x >> 3, item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (item >= (u32)p.items) return;
    const u32 z = item % (u32)p.shares, i1 = item / (u32)p.shares, rb = i1 % (u32)p.rblocks, i2 = i1 / (u32)p.rblocks;
    const int mat = __builtin_amdgcn_readfirstlane((int)(i2 % (u32)p.nmat)), e = __builtin_amdgcn_readfirstlane((int)(i2 / (u32)p.nmat));
    const int r0 = __builtin_amdgcn_readfirstlane((int)rb * 128);
    const uint8_t* sheet = p.bank[mat] + (size_t)e * p.sheet_bytes + (size_t)r0 * p.row_bytes;
    MoeColsQ4Rows w4;
    if constexpr (KO == 0) moe_cols_q4_places(p, p.nrows - 1 - r0, w4);
    const u32 c_hi = p.start[e + 1], c_lo = p.start[e] + 64 * z;
    for (u32 c0 = c_lo; c0 < c_hi; c0 += 64 * (u32)p.shares) {   // uniform
        const int n = (int)min(64u, c_hi - c0);
        // The rows' bytes, from memory the first time, are asked for ahead of the columns, which wait for the records' numbers.  Ahead of start as
        // well they save even routing nothing (1.00, 55 banks and column counts), and a workgroup without columns, which brings 18 KB for
        // nothing, costs uneven routing: 128 experts of 2048 x 768, eight of them with columns, 32 an expert on average 84 us, so 64; half of the
        // experts 53 and 48.
        if (KO == 0 && c0 == c_lo) moe_cols_q4_rows(smem, sheet, w4);
        auto tile = [&](auto G) __attribute__((always_inline)) {
            constexpr int g = decltype(G)::value;
            if constexpr (KO == 0) moe_cols_q4_tile<g>(p, smem, sheet, w4, c0 == c_lo, mat, r0, c0, n);
            else if constexpr (KO == 1) moe_cols_planes_tile<g>(p, smem, e, mat, r0, c0, n);
            else moe_cols_q6_tile<g>(p, smem, e, mat, r0, c0, n);
        };
        if (n > 32) tile(GemmIntC<2>{});
        else tile(GemmIntC<1>{});
    }
}
