// Kernel argument blocks, shared by the device code and the host launcher.
// Plain C layouts: the host passes each struct by value as the kernel's single
// parameter.
#pragma once
#include <stdint.h>

// ---- dynamic LDS of the decode matvecs, as the kernels divide it and the host asks for it
// Bytes of LDS the staging area needs for a k-element activation.
#define JL_ACT_LDS_BYTES(k) ((k) + ((k) / 32) * 4 + ((k) / 16) * 4)
// the grouped kernels' RMSNorm: up to sixteen partial sums and the scale, behind the staging area
#define JL_NORM_LDS_BYTES 160
// ... and with the second copy of the int8 values that the Q8_0 pair form reads (k % 64 == 0)
#define JL_ACT_LDS_BYTES_SHIFTED(k) (JL_ACT_LDS_BYTES(k) + (k) + 16)
// A wavefront's private LDS: 256 int8 activations, 8 scales, 16 half-block sums.
#define JL_PK_WAVE_LDS 384
// Dynamic LDS of a workgroup of `nw` wavefronts: the private areas, then the
// partial sums [nw][64], rows one word apart in banks.
#define JL_PK_RED_STRIDE 65
#define JL_PK_LDS_BYTES(nw) ((nw) * (JL_PK_WAVE_LDS + JL_PK_RED_STRIDE * 4))

struct MatVecArgs {
    float* out;          // [nrows]
    const uint8_t* w;    // GGUF row-major blocks
    const float* x;      // f32 activations (fused quantize) or null
    const int8_t* q;     // pre-quantized activations (split form) or null
    const float* as;     // [k/32] activation scales
    const float* s16;    // [k/16] activation sums
    int nrows, k;
    int row_bytes;
    int per;             // activation window / 32 (fused form)
    int nwaves;          // wavefronts per workgroup (the launch's block / 64)
    int ngroups;         // workgroups (the launch's grid)
    float* resid;        // optional: resid[r] += alpha * out[r] (times sigmoid(*resid_gate) when resid_gate is set)
    const float* resid_gate;
    float alpha;
};

// Several decode matvecs of one type in one launch (grid y = matrix): matrix i computes
// out[i][0:nrows[i]] = w[i] . act(i), act(i) = x + i*xstride (xstride 0: one shared
// activation), optionally silu(x) * (x2 + i*xstride); matrix 0 may also add
// alpha * out[0] into resid.
#define JL_MAX_MULTI 16
struct MatVecMultiArgs {
    float* out[JL_MAX_MULTI];
    const uint8_t* w[JL_MAX_MULTI];
    int nrows[JL_MAX_MULTI];
    const float* x;
    const float* x2;     // null: plain activation
    float* resid;        // null: none
    float alpha;
    const float* resid_gate;   // null, or one logit: the residual weight is alpha * sigmoid(*resid_gate)
    size_t xstride;      // elements
    int k, row_bytes, per, nwaves, ngroups;
    // the mixed-type kernel only: each matrix's type (JL_TYPE_*) and bytes per row
    int type[JL_MAX_MULTI];
    int row_bytes_of[JL_MAX_MULTI];
    // the _q entry points: one activation for every matrix, quantized beforehand (x unused)
    const int8_t* q;
    const float* as;
    const float* s16;
    const float* norm_w; // null: none; else the activation is RMSNorm(x) * norm_w first
    float* norm_out;     // optional: the normed activation, written once
    float norm_eps;
    double inv_k;        // 1 / k
};

// Activation preparation for the Q4_K prefill GEMM: quantize x and lay it out
// in matrix-fragment order, bq [k/128 stages][tok_pad/32][9][64][8] f16, da [k/256][tok_pad].
struct GemmPrepArgs {
    const float* x;      // [ntok][k]
    uint16_t* bq;        // f16 bits
    float* da;
    int ntok, tok_pad, k;
    float* dsum = nullptr;   // window 32, optional: d_a * (sum of the block's int8) [k/32][tok_pad]
    int per = 0;             // the int8 prep: activation window / 32
};

struct GemmArgs {
    float* out;          // [ntok][out_stride]; a launch may cover a slice of the rows
    const uint8_t* w;    // GGUF row-major Q4_K (of the slice)
    const uint16_t* bq;
    const float* da;
    int nrows, k, ntok, tok_pad;   // nrows of the slice
    int row_bytes;
    int out_stride;      // floats between tokens in out
    int sb_per;          // K split: super-blocks per blockIdx.z (0 = whole K), out = slab z of [gridDim.z][ntok][out_stride]
    const float* dsum = nullptr;   // window 32, Q4_K: the prep's d_a * block sums
    int tall = 1 << 24;   // Q8_0, 256 tokens x 128 rows: row tiles of 128, those behind them are of 64
    // the weights as packed planes (the kernels' plane forms; w is unused then): QS, D and SC
    // planes of a buffer of pstride rows, this launch's first row at prow0 (nrows counted from
    // it), its first super-block psb0 (a K split moves it)
    const uint32_t* pqs = nullptr;
    const uint32_t* pd = nullptr;
    const uint32_t* psc = nullptr;
    int prow0 = 0, pstride = 0, psb0 = 0;
};

// Few tokens on the int8 matrix cores (kernels/few_i8.h).  The prep's layout, by chunk (128 of K) and slot
// (16 columns): bq [chunk][slot][2 pairs of blocks][64 lanes][4 words] int8, da and ds [chunk][slot][16
// columns][4 blocks] (the columns' scales, and scale * sum of the block's values; ds only where the
// weights have minimums).
struct FewI8PrepArgs {
    const float* x;
    const float* x2;        // null: plain activation, else silu(x) * x2
    const uint32_t* src;    // null: column c reads row c
    const uint32_t* start;  // null: one group, column c in slot c / 16
    uint32_t* bq;
    float* da;
    float* ds;              // may be null
    int k, per, ncols, n_expert, nslots, nch, order;
    int isum;               // ds: the block sums themselves, as integers
};
#define JL_FEW_SC_BYTES 896   // a row tile's scales, and the header words on their way to them
// a wavefront's LDS: scales, and over GGUF rows a staged super-block (ggml types 8, 12, 14)
#define JL_FEW_WAVE_BYTES(type, planes, rt) \
    ((rt) * (JL_FEW_SC_BYTES + ((planes) ? 0 : 16 * ((type) == 8 ? 272 : (type) == 12 ? 144 : 224))))
#define JL_FEW_RED_BYTES(nw, nt, rt) ((nw) * 16 * (nt) * (16 * (rt) + 4) * 4)
struct FewI8Args {
    float* out[2];          // [column][nrows]; may be null when resid is set
    const uint8_t* w[2];    // GGUF: sheets of sheet_bytes
    const uint32_t* pqs[2];
    const uint32_t* pd[2];
    const uint32_t* psc[2];
    float* resid;           // null, or resid[column][nrows] += the result
    const uint32_t* bq;
    const float* da;
    const float* ds;
    const uint32_t* start;  // null: one expert of ncols columns
    size_t sheet_bytes, sheet_words;
    int nrows, k, row_bytes, ncols, nslots, nch, nwaves;
    int prow0, row_step, pstride;
    int tgroup;             // start null: token tiles a workgroup, grid y = the groups of them
};

// Mixture block on the matrix cores (Q4_K, activation window 256).  An expert's columns are
// cut into groups of 32; group g of expert e has the workspace slot start[e]/32 + e + g
// (distinct for distinct groups, below ncols/32 + n_expert + 1 = nslots).  The prep kernel
// gathers, quantizes and lays out the groups' activations as the prefill GEMM's fragments,
// bq [k/128 stages][nslots][9][64 lanes][8] f16 and da [k/256][32*nslots]; the matrix kernel
// meets them with the expert's sheet, out[mat][column][nrows].
//
// Most (expert, group) pairs of a grid sized for the fullest expert are empty, and an empty
// workgroup still costs its dispatch, so the kernels walk a work list instead, written by
// jl_moe_worklist from start[]: wl[0] = number of 128-column tiles, wl[4 + s] = expert of
// slot s (all ones: unused), wl[4 + nslots + t] = tile t as expert | (tile of the expert << 16).
struct MoeWorklistArgs {
    const uint32_t* start;
    uint32_t* wl;
    int n_expert, nslots;
    int tile_log2 = 7;    // columns a tile
};

struct MoeGemmPrepArgs {
    const float* x;       // [.][k]
    const float* x2;      // optional: activation is silu(x) * x2
    const uint32_t* src;  // optional: column -> row of x (identity when null)
    const uint32_t* start;
    const uint32_t* wl;
    uint16_t* bq;
    float* da;
    int k, nslots;
    int per = 0;          // the int8 prep: activation window / 32
    float* dsum = nullptr;
};

struct MoeGemmArgs {
    float* out[2];
    const uint8_t* bank[2];
    const uint16_t* bq;
    const float* da;
    const uint32_t* start;
    const uint32_t* wl;
    size_t sheet_bytes;
    int nrows, k, row_bytes, nslots, nmat;
    // the banks as packed planes (plane form of the tile kernel; bank[] unused): expert e's planes
    // are pqs / pd / psc [mat] + e * sheet_words (u32 words; 0 when the bank is ONE plane set), its
    // first row e * row_step inside them (0 when every expert has its own sheet), pstride rows a
    // plane set
    const uint32_t* pqs[2] = {nullptr, nullptr};
    const uint32_t* pd[2] = {nullptr, nullptr};
    const uint32_t* psc[2] = {nullptr, nullptr};
    size_t sheet_words = 0;
    int row_step = 0, pstride = 0;
    const float* dsum = nullptr;   // the int8 form, Q4_K: d_a * block sums
};

// A decode matvec a routed column (moe_gather_body): grid y = column, z = matrix.
struct MoeGatherArgs {
    float* out[2];          // [column][nrows]
    const uint8_t* bank[2];
    const float* x;
    const float* x2;        // null: plain activation, else silu(x) * x2
    const uint32_t* src;    // null: column c reads row c
    const uint32_t* start;  // null: column c is pair c of sel, which reads row c / k_used
    const uint32_t* sel;    // [row][sel_stride]; null as well: one expert, column c reads row c
    size_t sheet_bytes;
    int nrows, k, row_bytes, per, nwaves, ngroups, n_expert, sel_stride, k_used;
};

// resid[row] += sum over the row's pairs of wt * (down sheet of the pair's expert . silu(g) u)  (moe_gather_down_body):
// grid y = row.
struct MoeGatherDownArgs {
    float* resid;           // [row][nrows]
    const uint8_t* bank;
    const float *g, *u;     // [pair][k]
    const uint32_t* sel;    // [row][sel_stride]; null: expert 0 (k_used 1)
    const float* wt;        // [row][k_used]; null: 1
    size_t sheet_bytes;
    uint32_t slots_inv;     // 2^32 / (slots of a sheet's row), rounded up
    int nrows, k, row_bytes, per, nwaves, ngroups, n_expert, sel_stride, k_used;
};

// The same two steps over packed planes: column = pair of sel (null: column c reads row c, expert 0); sheet_words, row_step: from an expert's planes, rows to the next's.
struct MoePlanesGatherArgs {
    float* out[2];          // [pair][nrows]
    const uint32_t *qs[2], *d[2], *sc[2];
    const float* x;         // [row][k]
    const uint32_t* sel;
    size_t sheet_words;
    int nrows, k, row_step, stride, per, nwaves, ngroups, n_expert, sel_stride, k_used;
};
struct MoePlanesDownArgs {
    float* resid;           // [row][nrows]
    const uint32_t *qs, *d, *sc;
    const float *g, *u;     // [pair][k]
    const uint32_t* sel;
    const float* wt;        // [row][k_used]
    size_t sheet_words;
    int nrows, k, row_step, stride, per, nwaves, ngroups, n_expert, sel_stride, k_used;
};

// Grouped expert matmul for experts of some tens of columns (kernels/moe_cols.h): rec [record][k/256][512 or 256 bytes],
// aug [record][k/256][32 bytes], da [record][k/256].
// A column's record of one super-block: the operand pieces of sixteen bytes in the order the weights decode to
// (Q4_K: f16, piece 2 ks + kg of K-step ks = 0..15; Q6_K: int8, piece 8 kg + ks, ks = 0..7).
#define JL_MC_REC(q6) ((q6) ? 256 : 512)
// its dynamic LDS: Q4_K rows (columns by halves of a super-block, rows as they lie), Q6_K rows, Q4_K planes
#define JL_MC_A (64 * 256)      // half a super-block of 64 columns
#define JL_MC_W (128 * 144)
#define JL_MC_Q4_LDS (2 * JL_MC_A + 2 * JL_MC_W + 2 * (64 * 32 + 64 * 4))
#define JL_MC_Q6_W (128 * 208)
#define JL_MC_Q6_LDS (2 * 64 * 256 + JL_MC_Q6_W + 128 * 16 + 128 * 2 + 64 * 4)
#define JL_MC_PLANES_LDS (2 * (64 * 512 + 64 * 32 + 64 * 4))
struct MoeColsPrepArgs {
    const float* x;
    const float* x2;        // null: plain activation, else silu(x) * x2
    const uint32_t* src;    // null: record r is row r of x
    uint32_t* rec;
    uint32_t* aug;
    float* da;
    int k, nrec;
};
struct MoeColsArgs {
    float* out[2];
    const uint8_t* bank[2];
    const uint32_t* pqs[2] = {nullptr, nullptr};   // packed planes, as in MoeG16Args
    const uint32_t* pd[2] = {nullptr, nullptr};
    const uint32_t* psc[2] = {nullptr, nullptr};
    const uint8_t* rec;
    const uint8_t* aug;
    const float* da;
    const uint32_t* map;    // column -> record (null: its own)
    const uint32_t* start;
    size_t sheet_bytes, sheet_words = 0;
    int nrows, k, row_bytes, nmat, rblocks, shares, items, row_step = 0, pstride = 0;
};

// Grouped expert matmul, sixteen columns a group (moe_g16_body).  Column group g of expert e is
// slot (start[e] >> 4) + e + g of the prepared workspace; a slot holds, for every super-block,
// JL_MOE_G16_SB_WORDS words: eight matrix fragments of 64 lanes x 16 bytes (half, K-step), the
// sub-block sums' fragment (32 lanes x 16 bytes) and the sixteen columns' scales.
#define JL_MX1_RPW 2   // rows a wavefront of the one-token MXFP4 matvec walks (2880 x 2880: 1 / 2 / 3 / 4 rows 4.46 / 4.18 / 4.22 / 4.30 us)
#define JL_MOE_G16_SB_WORDS 2192
#define JL_MOE_G16_LDS_WORDS 2224   // the same in LDS, the fragments 65 vectors apart
struct MoeG16PrepArgs {
    const float* x;
    const float* x2;        // null: plain activation
    const uint32_t* src;    // null: column c reads row c
    const uint32_t* start;  // [n_expert + 1]
    uint32_t* ws;
    int k, n_expert, ncols;
};
struct MoeG16Args {
    float* out[2];
    const uint8_t* bank[2];
    const uint32_t* ws;
    const uint32_t* start;
    size_t sheet_bytes;
    int nrows, k, row_bytes;
    int tiles_wg;           // tiles of sixteen rows a workgroup owns
    int blocks, nmat, n_expert, nwaves;   // row blocks an (expert, matrix); wavefronts a workgroup
    // the banks as packed planes (plane form; bank[] and sheet_bytes unused): expert e's planes are
    // pqs / pd / psc [mat] + e * sheet_words (u32 words; 0 when the bank is ONE plane set), its first
    // row e * row_step inside them (0 when every expert has its own sheet), pstride rows a plane set
    const uint32_t* pqs[2] = {nullptr, nullptr};
    const uint32_t* pd[2] = {nullptr, nullptr};
    const uint32_t* psc[2] = {nullptr, nullptr};
    size_t sheet_words = 0;
    int row_step = 0, pstride = 0;
    // fused form: the columns are quantized by the matrix kernel itself (ws unused)
    const float* x = nullptr;
    const float* x2 = nullptr;
    const uint32_t* src = nullptr;
};

// Two-pass form of the Q4_K prefill GEMM.  Pass one expands the weights once per call into
// f16 matrix fragments, w16 [ceil(nrows/64)][k/128 stages][18 fragments][64 lanes] 16-byte
// vectors (fragment 2*ks+g: K-step ks of the tile's row group g; 16+g: the minimum columns,
// meaningful in second halves) and wsc [k/256][nrows_pad] (d, dmin); pass two is the matrix
// kernel with nothing left to dequantize.
struct GemmW16PrepArgs {
    const uint8_t* w;    // GGUF row-major Q4_K
    void* w16;           // 16-byte vectors
    float* wsc;          // pairs (d, dmin)
    int nrows, nrows_pad, k, row_bytes;
};

struct GemmW16Args {
    float* out;          // [ntok][nrows]
    const void* w16;
    const float* wsc;
    const uint16_t* bq;
    const float* da;
    int nrows, nrows_pad, k, ntok, tok_pad;
    int ntt, nrt;        // token tiles (128) and row tiles (64)
};

// Mixture-of-experts grouping: sel [rows][sel_stride] expert ids (the first k_used of
// each row are the selection) -> start [n_expert+1], perm [rows*k_used] (column ->
// row), pos [rows*k_used] (pair -> column).
// Dynamic LDS of the linear-time form (moe_group2_body).
#define JL_MOE_GROUP2_LDS(nexp) (16 * (nexp) * 2 + (2 * (nexp) + 16) * 4)
struct MoeGroupArgs {
    const uint32_t* sel;
    uint32_t* start;
    uint32_t* perm;
    uint32_t* pos;
    int sel_stride, rows, k_used, n_expert;
    int chunks = 1;         // 1024s of pairs a workgroup (moe_group2_body)
    uint32_t* wl[2] = {};   // null, or the work lists (MoeWorklistArgs) of tiles of 64 and of 128 columns
    int nslots = 0;
};

// Router: softmax over all experts, the k largest by (score descending, index ascending),
// weights = selected scores over their sum.  sel [rows][sel_stride] (first k_used filled),
// wt [rows][k_used].
struct MoeRouteArgs {
    const float* logits;    // [rows][n_expert]
    uint32_t* sel;
    float* wt;
    int n_expert, k_used, sel_stride;
};

// Router logits: logits[t][r] = sum_i W[r][i] * x[t][i], W f32 or f16 (the one matrix of a
// mixture block that is not quantized).
struct MoeLogitsArgs {
    const void* w;          // [n_expert][k], f32 or f16
    const float* x;         // [ntok][k]
    float* logits;          // [ntok][n_expert]
    int n_expert, k, ntok, f16;
    int by_expert;          // the grid's order: 0 token groups side by side, 1 expert rows (moe_logits_body)
};

// Column activations of a mixture pass: column c reads x[src(c)] (or silu(x[src(c)]) *
// x2[src(c)]) and is quantized like any activation vector: q [ncols][k] int8,
// as [ncols][k/32], s16 [ncols][k/16].
struct MoeQuantArgs {
    const float* x;
    const float* x2;        // null: plain activation
    const uint32_t* src;    // null: column c reads row c
    int8_t* q;
    float* as;
    float* s16;
    int k, per;
    const uint32_t* start;  // [n_expert + 1]: columns from start[n_expert] on belong to no expert and are left alone
    int n_expert;
    // chunked form (q, as, s16 unused): column c's 256-element chunk i as 88 consecutive words at
    // chunked + (c * k/256 + i) * 88 -- 64 of int8 values, 8 scales, 16 half-block sums -- so a
    // reader addresses everything it needs of a (column, chunk) from one base
    uint32_t* chunked = nullptr;
};

// Grouped expert matvec over columns sorted by expert: out[m][c][0:nrows] =
// bank[m] sheet(expert of c) . column c, columns already quantized (MoeQuantArgs).
struct MoeMatVecArgs {
    float* out[2];
    const uint8_t* bank[2];
    const int8_t* q;
    const float* as;
    const float* s16;
    const uint32_t* start;  // [n_expert + 1]
    size_t sheet_bytes;
    int nrows, k, row_bytes;
    int nwaves;             // wavefronts per workgroup
    int shares;             // workgroups one (expert, matrix) is split into, by rows
};

// The same over banks of packed planes (moe_matvec_planes_body): expert e's planes are
// pqs / pd / psc [m] + e * sheet_words (u32 words; 0 when a bank is ONE plane set), its first
// row e * row_step inside them (0 when every expert has a sheet of its own), pstride rows a
// plane set.
struct MoePlanesArgs {
    float* out[2];
    const uint32_t* pqs[2];
    const uint32_t* pd[2];
    const uint32_t* psc[2];
    const uint32_t* chunked;   // the columns, quantized in the chunked form (MoeQuantArgs.chunked)
    const uint32_t* start;  // [n_expert + 1]
    size_t sheet_words;
    int row_step, pstride;
    int nrows, k;
    int nwaves;             // wavefronts per workgroup: they split the 256-element chunks of K
};

struct MoeCombineArgs {
    float* resid;           // [rows][n_embd], accumulated into
    const float* y;         // [ncols][n_embd]
    const float* wt;        // [rows][k_used]
    const uint32_t* sel;    // [rows][sel_stride]
    const uint32_t* pos;    // [rows*k_used]; not read for an id that no expert has
    int sel_stride, k_used, n_embd;
    uint32_t last_id;       // ids past this one are no expert's and add nothing
};

// MXFP4 weights x bf16 activations: out [ntok][nrows] f32.
// bf16 activations x [ntok][k] -> matrix fragments xf [ceil(k/256) stages][tok_pad/32][16]
// [64 lanes][8 bf16]: fragment ks of a stage holds, for lane 32*kg + t%32, the eight values
// x[t][256*stage + 16*ks + 8*kg ..]; tokens past ntok and K past k are zero.
struct MxPrepArgs {
    const uint16_t* x;
    uint16_t* xf;
    int ntok, tok_pad, k;
};

// The one-launch few-token kernel (mx_one_body): token tiles of a group of activations (4 KB) a wavefront has room for, as many as
// it works on at most (two row tiles' sums have to fit); dynamic LDS of its eight wavefronts.
#define JL_MX_ONE_SLOTS(k, nt) (((k) + 1023) / 1024 * (nt) < 4 ? ((k) + 1023) / 1024 * (nt) : 4)
#define JL_MX_ONE_LDS(k, nt) (8 * 4096 * JL_MX_ONE_SLOTS(k, nt))
struct MxGemmArgs {
    float* out;
    const uint8_t* w;     // GGUF row-major MXFP4 blocks (17 bytes per 32)
    const uint16_t* x;    // bf16 bits: [ntok][k] for the matvec, fragment order (MxPrepArgs) for the GEMM
    int tok_pad;          // GEMM: tokens padded to whole tiles of 128
    int nrows, k, ntok;
    int row_bytes;
    int nsplit;           // workgroups along K (grid z); > 1: partial sums go to part
    float* part;          // [nsplit][ntok][nrows], summed by jl_sum_parts
    // the few-token kernel over packed planes (w unused): rows row0 .. of planes of `stride` rows
    const uint32_t* qs = nullptr;
    const uint32_t* d = nullptr;
    int row0 = 0, stride = 0;
};

// MXFP4 planes x a handful of bf16 tokens: rows row0 .. row0+nrows of planes of `stride` rows.
struct MxPlanesArgs {
    float* out;           // [ntok][nrows]
    const uint32_t* qs;   // [k/32][4][stride]: a block's 16 code bytes, four words
    const uint32_t* d;    // [k/32][ceil(stride/4)]: E8M0 exponent minus one, four rows a word
    const uint32_t* x;    // [ntok][k] bf16 bits, read two a word
    int nrows, k, ntok, row0, stride;
    int nwaves;           // wavefronts of a workgroup; they split the blocks of K
};

// MXFP4 planes x bf16, more than a handful of tokens, the planes read where they lie:
// activation fragments in the planes' K order.
struct MxPlanesPrepArgs {
    const uint16_t* x;    // [ntok][k] bf16 bits
    uint32_t* xa;         // [K-step of 64][token tile of 32][4 matrix K-steps][64 lanes][4 words]
    int ntok, tok_pad, k;
    // GGUF rows to turn into planes on the way (null: the weights are planes already)
    const uint8_t* w = nullptr;
    uint32_t* qs = nullptr;
    uint32_t* d = nullptr;
    int nrows = 0, stride = 0;   // stride a multiple of 64
};

struct MxPlanesGemmArgs {
    float* out;           // [ntok][nrows]
    const uint32_t* qs;   // rows row0 .. row0+nrows of planes of `stride` rows
    const uint32_t* d;
    const uint32_t* xa;
    int nrows, k, ntok, tok_pad, row0, stride;
};

// The opt-in block-scaled form: activations as MX fp8 (e4m3 codes, one E8M0 scale a token and
// block of 32) in the operand order of the 32x32x64 scaled matrix instruction.
struct MxScaledPrepArgs {
    const uint16_t* x;    // [ntok][k] bf16 bits
    uint32_t* xa;         // [K-step][token tile][64 lanes][8 words]
    uint8_t* xs;          // [K-step][token tile][64 lanes]
    int ntok, tok_pad, k;
};

struct MxScaledGemmArgs {
    float* out;           // [ntok][nrows]
    const uint32_t* qs;   // MXFP4 planes, rows row0 .. row0+nrows of `stride`
    const uint32_t* d;
    const uint32_t* xa;
    const uint8_t* xs;
    int nrows, k, ntok, tok_pad, row0, stride;
};

// out[i] = part[0][i] + part[1][i] + ... in that order.
struct SumPartsArgs {
    float* out;
    const float* part;
    size_t n;
    int nsplit;
};

// GGUF row-major blocks -> the reference's device planes (and back, for Q4_K).
struct PackArgs {
    const uint8_t* src;   // [nrows][k / block] GGUF blocks
    uint32_t* qs;
    uint32_t* d;
    uint32_t* sc;         // null for formats without a scale plane
    int nrows, k, type;
    uint32_t* flag;       // MXFP4: set to 1 when a block's exponent cannot be stored (else untouched)
};

// Scale range of a Q4_K matrix for the folded-scale GEMM (kernels/gemm_q4k_fold.h).
struct FoldRangeArgs {
    const uint8_t* w;     // GGUF super-blocks, 144 bytes each
    size_t nblocks;
    uint32_t* flag;       // set to 1 when a super-block's weights can pass the f16 range (else untouched)
};

struct UnpackArgs {
    uint8_t* dst;         // [nrows][k/256] Q4_K super-blocks
    const uint32_t* qs;
    const uint32_t* d;
    const uint32_t* sc;
    int nrows, k, row0, stride;
};

// Decode matvec over the planes: rows row0 .. row0+nrows of a buffer of `stride` rows.
struct PackedMatVecArgs {
    float* out;           // [nrows]
    const uint32_t* qs;
    const uint32_t* d;
    const uint32_t* sc;
    const float* x;       // f32 activations (fused quantize) or null
    const int8_t* q;      // pre-quantized activations or null
    const float* as;
    const float* s16;
    int nrows, k, row0, stride;
    int per;              // activation window / 32
    int nwaves;           // wavefronts per workgroup (the launch's block / 64)
    int ngroups;          // workgroups (the launch's grid.x)
    const float* x2;      // gated kernels only: the activation is silu(x) * x2
    float* resid;         // null: none; else resid[r] += alpha * out[r]
    float alpha;
    float* norm_out;      // norm kernels only: null, or where the normed activation goes
    float norm_eps;
    double inv_k;        // 1 / k
};

// Several packed matvecs of one type and shape in one launch, grid = (row groups,
// matrices): matrix y has its own planes and first row (an expert's sheet inside its bank's
// planes: the same plane pointers, row0 = expert * rows) and reads x + y * xstride.
struct PackedMultiArgs {
    float* out[JL_MAX_MULTI];
    const uint32_t* qs[JL_MAX_MULTI];
    const uint32_t* d[JL_MAX_MULTI];
    const uint32_t* sc[JL_MAX_MULTI];
    int row0[JL_MAX_MULTI];
    const float* x;
    const float* x2;      // null: plain activation
    size_t xstride;       // elements
    int nrows, k, stride, per, nwaves, ngroups;
    float* resid;         // null: none; else resid[r] += alpha * out[0][r] (matrix 0 only)
    float alpha;
    const float* resid_gate;    // null, or one logit: the residual weight is alpha * sigmoid(*resid_gate)
    const float* norm_w;  // norm kernels only: RMSNorm weights [k]; every x_j is normed ahead of its quantizer
    float* norm_out;      // null, or where matrix 0's normed activation goes
    float norm_eps;
    double inv_k;        // 1 / k
};
