// Host side of the C ABI declared in include/jlmi.h.
//
// One context = one device, one stream, one gfx950 code object loaded with
// hipModuleLoad and its kernels resolved by name.  Entry points validate
// shapes on the host before any launch (a kernel is never started on operands
// it does not fit), translate the reference's operator contracts into kernel
// launches, and report served / declined / error.  There is no CPU compute path
// here: when the code object or the device is missing, creation fails.
#include "../../include/jlmi.h"

#include <dlfcn.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <atomic>
#include <mutex>
#include <thread>
#include <string>
#include <vector>

#include "hip_api.h"
#include "kernels/args.h"
#include "scratch.h"

namespace {

thread_local std::string g_create_error;
const HipApi* H = nullptr;  // the process-wide HIP runtime, resolved by the first jl_ctx_create

struct Tuning {
    int rpw = 0, block = 0, grid = 0;
    int act_split = 0;          // grouped matvec with a gated activation: 1 always quantize it in its own launch, 2 never
    int xpre = 0;               // decode matvec: 1 / 2 / 4 float4 groups of x a thread loads ahead of its weights
    int q8pair = 0;             // Q8_0 rows: 2 keeps one block a lane-slot (2-byte-aligned loads)
    int packed_rw = 0, packed_block = 0, moe_group = 0, moe_logits = 0;
    int moe_shares = 0;
    int gemm_rows = 0;
    int gemm_form = 0;
    int gemm_split = 0;
    int gemm_prep = 0;
    int gemm_planes = 0;
    int gemm_few = 0;           // the int8 few-token form: 1 wherever it fits, 2 never; 3: decode matvecs in one launch
    int few_nt = 0, few_rt = 0, few_waves = 0;
    int gemm_i8 = 0;            // the int8 tile forms, Q8_0: 1 / 2 / 3 ask for 128 x 128 / 128 x 64 / 256 x 128 tiles
    int moe_form = 0;
    int moe_g16 = 0;
    int gemm_fold = 0, gemm_fold_waves = 0;
    int moe_chunk = 0;
    int moe_waves = 0;
    int moe_lpr = 0;
    int matvec_lanes = 0;
    int mx_rows = 0;
    int mx_scaled = 0;          // 1: packed MXFP4 matmul on the block-scaled fp8 x fp4 matrix instruction (lossy)
    int mx_planes = 0;          // packed MXFP4: 2 restores rows first; 64 / 32 / 16 rows a workgroup of the plane
                                // matvec; rows and planes: 3 / 4 the tiles of 64 / 96 rows
    int mx_split = 0;
    int gemm_tall = 0;   // Q8_0, 256 tokens x 128 rows: 1 no tiles of 64 rows, 2 + n those behind n of 128
    int mx_few = 0, mx_few_min = 0;   // MXFP4: the few-token form up to / from this many tokens
    int mx_one = 0;                   // ... in one launch: 1 never, 11 / 12 wherever it can be, that many row tiles a workgroup
};

// The code object's kernels by name.  Looked up on every launch, so without a string to allocate or a tree to
// walk: open addressing over the names' hashes.
struct KernelTable {
    struct Slot { uint64_t hash = 0; std::string name; hipFunction_t fn = nullptr; };
    std::vector<Slot> slots;
    size_t used = 0;
    static uint64_t hash_of(const char* s) {
        uint64_t h = 1469598103934665603ull;   // FNV-1a
        for (; *s; s++) h = (h ^ (uint8_t)*s) * 1099511628211ull;
        return h ? h : 1;
    }
    hipFunction_t find(const char* name) const {
        if (slots.empty()) return nullptr;
        const uint64_t h = hash_of(name);
        for (size_t i = h & (slots.size() - 1); slots[i].hash; i = (i + 1) & (slots.size() - 1))
            if (slots[i].hash == h && slots[i].name == name) return slots[i].fn;
        return nullptr;
    }
    void add(const std::string& name, hipFunction_t fn) {
        if (2 * (used + 1) > slots.size()) {
            std::vector<Slot> old(slots.empty() ? 64 : 2 * slots.size());
            old.swap(slots);
            used = 0;
            for (const Slot& o : old)
                if (o.hash) add(o.name, o.fn);
        }
        const uint64_t h = hash_of(name.c_str());
        size_t i = h & (slots.size() - 1);
        while (slots[i].hash && slots[i].name != name) i = (i + 1) & (slots.size() - 1);
        if (!slots[i].hash) used++;
        slots[i] = Slot{h, name, fn};
    }
};

// A kernel's name put together from its parts.
struct Name {
    char s[64];
    unsigned n = 0;
    Name() { s[0] = 0; }
    Name& operator<<(const char* p) {
        while (*p && n < sizeof s - 1) s[n++] = *p++;
        s[n] = 0;
        return *this;
    }
    Name& operator<<(char ch) {
        const char t[2] = {ch, 0};
        return *this << t;
    }
    Name& operator<<(int v) {
        char t[12];
        int i = 11;
        t[i] = 0;
        do t[--i] = (char)('0' + v % 10);
        while ((v /= 10) && i > 0);
        return *this << (t + i);
    }
    operator const char*() const { return s; }
};

struct Resident {
    void* dev = nullptr;
    size_t bytes = 0;
};

// A block whose feed-forward weights jl_prep_layer made resident: one device allocation, the
// pieces' addresses in it.
struct Layer {
    jl_layer_plan plan;          // host pointers cleared
    void* mem = nullptr;         // the allocation
    // packed = 0: the matrices' (banks') bytes; packed = 1: plane sets
    const void *gate = nullptr, *up = nullptr, *down = nullptr;
    const uint32_t *gp[3] = {nullptr, nullptr, nullptr}, *upl[3] = {nullptr, nullptr, nullptr},
                   *dp[3] = {nullptr, nullptr, nullptr};
    const float* norm_w = nullptr;
    const float* router = nullptr;
};

}  // namespace

struct jl_ctx {
    int device = 0;
    int act_window = 32;
    hipStream_t stream = nullptr;
    hipModule_t module = nullptr;
    KernelTable fn;
    std::string err;
    std::mutex mu;  // serialises the host-pointer seam (one staging area per context)
    std::atomic<std::thread::id> mu_owner{};   // the thread inside mu (jl_forget must not try it again)
    // jl_forget only queues its range here, under a lock no launch or upload path holds; the
    // host-pointer calls apply the queue (unlink + hipFree) before their residency lookup
    std::mutex forget_mu;
    std::vector<std::pair<uintptr_t, uintptr_t>> pending_forget;
    // Q4_K matrices (device address -> rows, k) whose scales jl_fold_admit_dev found inside the
    // f16 range: the only ones the folded-scale GEMM form is used for (under forget_mu)
    std::map<uintptr_t, std::pair<int, int>> fold_ok;
    bool no_device = false;   // created with device < 0: host-side bookkeeping only
    // the static device array of scratch.hip on this context's device (null: the lookup
    // failed and static_err says why), and the state of a call that lives on it
    void* static_scratch = nullptr;
    size_t static_scratch_bytes = 0;
    std::string static_err;
    Tuning tune;
    int gemm_min_tok = 3;  // below this a per-token matvec loop is as fast (3.8 us a token against 8.9 us for up to 16)
    int num_cu = 0;
    size_t lds_limit = 0;
    uint8_t few_simd[5][2][4][3] = {};   // wavefronts a SIMD holds of jl_few_*: form, planes, token tiles - 1, row tiles / 2 (0: not built)
    std::atomic<unsigned long long> launches{0};   // kernels launched so far (jl_launch_count)

    // prefill GEMM workspace (quantized activations in stage layout), grown on demand
    void* gemm_ws = nullptr;
    size_t gemm_ws_bytes = 0;
    std::vector<std::pair<int, int>> reserved;   // (tokens, features) jl_reserve has sized the workspaces for

    void* w16_ws = nullptr;   // expanded weights of the two-pass GEMM
    size_t w16_ws_bytes = 0;

    void* mx_ws = nullptr;      // partial sums of a K-split matmul (MXFP4, Q4_K)
    size_t mx_ws_bytes = 0;
    uint32_t* one_group = nullptr;   // (0, n) for n = 0..16: column ranges of a single group of n columns
    void* moe_q_ws = nullptr;   // quantized column activations of a mixture pass
    size_t moe_q_ws_bytes = 0;
    void* act_ws = nullptr;     // a long gated activation, quantized once for a grouped matvec
    size_t act_ws_bytes = 0;

    // rows restored to GGUF order for the GEMM over packed planes
    void* unpack_ws = nullptr;
    size_t unpack_ws_bytes = 0;
    void* flag_ws = nullptr;    // one word the MXFP4 packer raises when it must refuse
    size_t flag_ws_bytes = 0;

    // mixture-of-experts workspace (grouping tables and intermediate columns)
    void* moe_ws = nullptr;
    size_t moe_ws_bytes = 0;

    // blocks prepared by jl_prep_layer, and the workspace their runs share (router logits,
    // selection and weights of a mixture; gate and up of a dense block at one row)
    std::map<int, Layer> layers;
    void* layer_ws = nullptr;
    size_t layer_ws_bytes = 0;
    // a block's router logits and, when it is not handed a place for them, selection and weights
    void* moe_route_ws = nullptr;
    size_t moe_route_ws_bytes = 0;

    // host-pointer seam state
    std::map<const void*, Resident> resident;
    void* stage_x = nullptr;    // device
    void* stage_out = nullptr;  // device
    size_t stage_x_bytes = 0, stage_out_bytes = 0;
    // pinned host memory the small operands and results of a host-pointer call go through, and the word
    // that is raised to the call's number when its results are in
    void* pin = nullptr;
    size_t pin_bytes = 0;
    volatile uint32_t* pin_flag = nullptr;
    uint32_t pin_number = 0;
};

namespace {

// What a call in progress on THIS thread has switched on for its context: jl_reserve_shape
// walks a launch path with launching off (dry_run), jl_matmul_static_dev carves workspaces
// from the static array instead of the heap (no_alloc).  Kept per thread and tagged with the
// context, so a launch that another thread makes on the same context meanwhile is a launch.
struct CallState {
    const jl_ctx* ctx = nullptr;
    bool dry_run = false;
    bool no_alloc = false;
    size_t static_used = 0;
};
thread_local CallState g_call;
bool call_dry_run(const jl_ctx* c) { return g_call.ctx == c && g_call.dry_run; }
bool call_no_alloc(const jl_ctx* c) { return g_call.ctx == c && g_call.no_alloc; }
// Switches the state on for a scope; nests (a dry run inside a no-alloc call).
struct CallScope {
    CallState saved;
    CallScope(const jl_ctx* c, bool dry_run, bool no_alloc) : saved(g_call) {
        if (g_call.ctx != c) g_call = CallState{};
        g_call.ctx = c;
        g_call.dry_run = g_call.dry_run || dry_run;
        g_call.no_alloc = g_call.no_alloc || no_alloc;
    }
    ~CallScope() { g_call = saved; }
};

// c->mu with its owner recorded.
struct CtxLock {
    jl_ctx* c;
    explicit CtxLock(jl_ctx* ctx) : c(ctx) {
        c->mu.lock();
        c->mu_owner.store(std::this_thread::get_id());
    }
    ~CtxLock() {
        c->mu_owner.store(std::thread::id());
        c->mu.unlock();
    }
};

int fail(jl_ctx* c, int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (c) c->err = buf;
    else g_create_error = buf;
    return code;
}

#define HIP_TRY(c, call)                                                              \
    do {                                                                              \
        hipError_t e_ = (call);                                                       \
        if (e_ != hipSuccess)                                                         \
            return fail((c), JL_ERR_HIP, "%s: %s", #call, H->GetErrorString(e_));     \
    } while (0)

std::string default_code_object() {
    Dl_info info;
    if (dladdr((void*)&jl_ctx_create, &info) && info.dli_fname) {
        std::string p = info.dli_fname;
        size_t s = p.rfind('/');
        return (s == std::string::npos ? std::string(".") : p.substr(0, s)) + "/jlmi_gfx950.hsaco";
    }
    return "jlmi_gfx950.hsaco";
}

struct TypeInfo {
    const char* tag;   // kernel-name fragment
    int block_elems, block_bytes;
    int slot_elems;    // elements one lane-slot of the matvec kernel covers
};

const TypeInfo* type_info(int type) {
    static const TypeInfo q8 = {"q8_0", 32, 34, 32};
    static const TypeInfo q4k = {"q4k", 256, 144, 64};
    static const TypeInfo q6k = {"q6k", 256, 210, 64};
    switch (type) {
    case JL_TYPE_Q8_0: return &q8;
    case JL_TYPE_Q4_K: return &q4k;
    case JL_TYPE_Q6_K: return &q6k;
    }
    return nullptr;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Largest workgroup of the matvec variant with `rpw` rows per wavefront, 0 when the
// code object has no such variant (kernels/jlmi_kernels.hip).
int matvec_max_block(int type, int rpw, bool q8_pair = false) {
    if (rpw == 1) return 1024;
    if (rpw == 2) return type == JL_TYPE_Q6_K ? 512 : 1024;
    if (rpw == 4) return type == JL_TYPE_Q8_0 && !q8_pair ? 1024 : 512;
    return 0;
}

// Float4 groups of the activation that a thread of a matvec loads ahead of its weights: all of them up to two,
// else four ("matvec.xpre" = 1, 2 or 4 asks for one).  A group that is loaded when its turn comes waits out a
// trip to memory behind the weights (Q4_K 4096 x 8192 6.0 us with one ahead, 5.5 with all).
int x_groups(const jl_ctx* c, int k, int threads) {
    if (c->tune.xpre == 1 || c->tune.xpre == 2 || c->tune.xpre == 4) return c->tune.xpre;
    return k / 4 > 2 * threads ? 4 : k / 4 > threads ? 2 : 1;
}

hipStream_t pick_stream(jl_ctx* c, void* s) { return s ? (hipStream_t)s : c->stream; }

// LDS of the decode matvec: int8 activations, a scale per 32, a sum per 16
size_t act_lds_bytes(int k) { return JL_ACT_LDS_BYTES((size_t)k); }

// Q8_0 rows in the form that takes two blocks a lane-slot with every load 4-byte aligned
// (kernels/matvec.h): rows on 4-byte boundaries, an even number of blocks a row, room in
// LDS for the second copy of the activations.
bool q8_pair_form(const jl_ctx* c, int type, const void* w, int k) {
    return type == JL_TYPE_Q8_0 && c->tune.q8pair != 2 && k % 64 == 0 && ((uintptr_t)w & 3) == 0 &&
           act_lds_bytes(k) + (size_t)k + 16 <= c->lds_limit;
}

// counted: whether jl_launch_count counts it (a host-pointer call's copies are not).
int launch(jl_ctx* c, const char* name, unsigned gx, unsigned gy, unsigned block, unsigned lds,
           hipStream_t st, void** params, unsigned gz = 1, bool counted = true) {
    const hipFunction_t f = c->fn.find(name);
    if (!f) return fail(c, JL_ERR_ARG, "kernel %s is not in the code object", name);
    if (call_dry_run(c)) return JL_OK;
    HIP_TRY(c, H->ModuleLaunchKernel(f, gx, gy, gz, block, 1, 1, lds, st, params, nullptr));
    if (counted) c->launches++;
    return JL_OK;
}

// Grows a context-owned device buffer.  Growing frees the old one, which kernels enqueued by
// earlier calls -- on the context's stream or on any stream a caller passed -- may still
// read, so the whole device is waited for first.  Never reached once the buffer is large
// enough (jl_reserve, jl_reserve_shape).
int grow(jl_ctx* c, void** buf, size_t* have, size_t need) {
    if (*have >= need) return JL_OK;
    if (call_no_alloc(c)) {
        // a call that must not allocate: the next piece of the static array, or an error.  (A
        // workspace asked for a second time with a larger size gets a new, larger piece: the
        // one it had stays taken until the call ends.)
        const size_t off = (g_call.static_used + 255) & ~(size_t)255;
        if (off + need > c->static_scratch_bytes)
            return fail(c, JL_ERR_NOMEM, "this shape needs %zu bytes of workspace on top of %zu already carved; the static "
                        "scratch holds %zu", need, off, c->static_scratch_bytes);
        *buf = (char*)c->static_scratch + off;
        *have = need;
        g_call.static_used = off + need;
        return JL_OK;
    }
    if (*buf) {
        HIP_TRY(c, H->DeviceSynchronize());
        HIP_TRY(c, H->Free(*buf));
    }
    *buf = nullptr;
    *have = 0;
    HIP_TRY(c, H->Malloc(buf, need));
    *have = need;
    return JL_OK;
}

// Shape checks shared by every matvec entry point.  Returns JL_OK, JL_DECLINED or an error.
int matvec_check(jl_ctx* c, int type, int nrows, int k, const TypeInfo** ti_out) {
    const TypeInfo* ti = type_info(type);
    if (!ti) return JL_DECLINED;
    if (nrows <= 0 || k <= 0) return fail(c, JL_ERR_ARG, "matvec: nrows=%d k=%d", nrows, k);
    if (k % ti->block_elems != 0) return JL_DECLINED;
    size_t lds = (size_t)k + (size_t)(k / 32) * 4 + (size_t)(k / 16) * 4;
    if (lds > c->lds_limit) return JL_DECLINED;  // activation does not fit LDS
    if ((size_t)(k / ti->block_elems) * ti->block_bytes > 0x7fffffffu) return JL_DECLINED;
    *ti_out = ti;
    return JL_OK;
}

// Lanes a row for the decode matvecs: a row of at most 32 (16) slots takes 32 (16) lanes of a wavefront, which then has two (four)
// rows a step; the same sums in the same order (the lanes left out added zeros).  From eight rows a CU; below, the launch is
// its ramp.  us, 64 lanes -> 32 -> 16, weights in turn: Q4_K 8192 x 1024 4.8 -> 3.4 -> 3.1 (the host's launch), 32768 x 1024 11.5 ->
// 7.4 -> 5.5, 8192 x 2048 5.0 -> 4.2, 16384 x 2048 7.9 -> 5.9, 65536 x 2048 22.6 -> 15.5; Q6_K 8192 x 1024 5.8 -> 4.2 -> 3.5, 16384 x 2048
// 10.2 -> 8.2; Q8_0 16384 x 1024 6.9 -> 5.3 -> 5.8, 65536 x 1024 20.9 -> 15.3 -> 14.4, 16384 x 2048 9.0 -> 8.6.
int matvec_lanes(const jl_ctx* c, int slots, long rows) {
    const int lanes = c->tune.matvec_lanes ? c->tune.matvec_lanes : rows <= 8L * c->num_cu ? 64 : slots <= 16 ? 16 : 32;
    return slots <= lanes ? lanes : 64;
}

int matvec_launch(jl_ctx* c, float* out, int type, const void* w, const float* x, const int8_t* q,
                  const float* as, const float* s16, int nrows, int k, hipStream_t st, float* resid = nullptr,
                  float alpha = 0.f, const float* resid_gate = nullptr) {
    const TypeInfo* ti = nullptr;
    int rc = matvec_check(c, type, nrows, k, &ti);
    if (rc != JL_OK) return rc;
    if (!out || !w) return fail(c, JL_ERR_ARG, "matvec: null operand");
    if (x && !aligned16(x)) return JL_DECLINED;
    if (!x && (!q || !as || !s16)) return fail(c, JL_ERR_ARG, "matvec: no activation");
    if (q && !aligned16(q)) return JL_DECLINED;
    if (type == JL_TYPE_Q4_K && !aligned16(w)) return JL_DECLINED;
    if (((uintptr_t)w & 1) != 0) return JL_DECLINED;

    // Shape choice, from sweeps on MI355X: one row (or step of rows) per wavefront.  At most sixteen a CU: one workgroup a CU of as
    // many wavefronts as it has rows, eight at least (the workgroup quantizes x; Q4_K 1500 x 13312 on eight 6.9 us, on
    // sixteen 7.8; 3000 x 11008 on twelve 6.2 and 6.6; 6144 x 2048 two rows a step, 4.1 as two workgroups a CU, so 3.3).  Taller ones: a persistent grid over the row groups with
    // sixteen wavefronts a CU for the k-quants, whose registers leave room for no more (a second round of workgroups
    // quantizes x again: Q6_K 10822 x 768 7.0 us -> 5.6, 14336 x 4096 10.2 -> 8.6), as two workgroups of eight, which
    // cover each other's barriers (9988 x 5120 Q6_K 9.4 against 10.3 as one; 6000 x 4096 Q4_K 4.5 and 4.5);
    // Q8_0: two workgroups of twelve, or, up to two rounds of them, one of sixteen wavefronts (8192 x 4096 7.3 against
    // 6.8); from forty rows a CU with the two-block form, K = 3584 to 5120, two of eight (weights from memory, eight
    // against twelve: 14336 x 4096 11.8 and 12.4, 12800 x 5120 14.7 and 15.7, 10240 x 3584 8.0 and 9.3; from cache the
    // same, 10.3 and 10.5, 12.1 and 12.5, 6.6 and 7.2; outside that range the ones gain what the others lose: 14336 x 2560
    // 8.1 and 8.4, from cache 6.8 and 6.3, 14336 x 14336 41.6 and 39.4).
    int rpw = c->tune.rpw, block = c->tune.block;
    if (rpw <= 0 || resid || !x) rpw = 1;   // (the kernels with the residual add or a quantized activation: one row a wavefront)
    if (rpw != 1 && rpw != 2 && rpw != 4) return fail(c, JL_ERR_ARG, "matvec: rpw=%d", rpw);
    const bool pair = q8_pair_form(c, type, w, k);
    const int slots = k / (type == JL_TYPE_Q8_0 && !pair ? 32 : 64);
    int lanes = rpw == 1 && x && !resid ? matvec_lanes(c, slots, nrows) : 64;
    const int steps = (nrows + 64 / lanes - 1) / (64 / lanes);   // of a wavefront, all rows
    const bool small = steps <= 16 * c->num_cu;
    const bool one_per_cu = small || (type == JL_TYPE_Q8_0 && pair && nrows <= 32 * c->num_cu && k >= 4096);
    if (block <= 0)
        block = small ? 64 * std::max(8, (steps + c->num_cu - 1) / c->num_cu) : one_per_cu ? 1024 :
                type == JL_TYPE_Q8_0 && !(pair && nrows >= 40 * c->num_cu && k >= 3584 && k <= 5120) ? 768 : 512;
    if (block % 64 != 0 || block > 1024) return fail(c, JL_ERR_ARG, "matvec: block=%d", block);
    if (block > matvec_max_block(type, rpw, pair)) block = matvec_max_block(type, rpw, pair);
    const int xpre = x_groups(c, k, block);
    if (xpre != 1) lanes = 64;   // (a tuned workgroup: rows that short are one group a thread otherwise)
    const int rows_per_block = (block / 64) * rpw * (64 / lanes);
    long groups = ((long)nrows + rows_per_block - 1) / rows_per_block;
    long grid = c->tune.grid > 0 ? c->tune.grid : (long)c->num_cu * (one_per_cu && rpw == 1 ? 1 : 2);
    if (grid > groups) grid = groups;
    if (grid < 1) grid = 1;

    MatVecArgs a;
    a.out = out;
    a.w = (const uint8_t*)w;
    a.x = x;
    a.q = q;
    a.as = as;
    a.s16 = s16;
    a.nrows = nrows;
    a.k = k;
    a.row_bytes = (k / ti->block_elems) * ti->block_bytes;
    a.per = c->act_window / 32;
    a.nwaves = block / 64;
    a.ngroups = (int)grid;
    a.resid = resid; a.alpha = alpha; a.resid_gate = resid ? resid_gate : nullptr;
    Name name;
    name << "jl_matvec_" << (pair ? "q8_0p" : ti->tag) << "_r" << rpw << (!x ? "_pq" : xpre == 4 ? "_x4" : xpre == 2 ? "_x2" : "") << (resid ? "_res" : "");
    if (lanes != 64) name << "_l" << lanes;
    void* params[] = {&a};
    unsigned lds = (unsigned)(act_lds_bytes(k) + (pair ? (size_t)k + 16 : 0));
    return launch(c, name, (unsigned)grid, 1, (unsigned)block, lds, st, params);
}

// The forms for several tokens or routed pairs: Q6_K has one for the k-quant window.
const char* q6_tag(const jl_ctx* c, int type) { return type == JL_TYPE_Q6_K && c->act_window == 256 ? "q6kw" : type_info(type)->tag; }

// m matrices of one type in one launch (kernels/matvec.h, matvec_multi_body).
// tokens: one plain matrix for m activations (tokens_matvec_launch).
// types: null when every matrix is of `type`; else the type of each (the mixed-type kernel).
int matvec_multi_launch(jl_ctx* c, int type, int m, float* const* outs, const void* const* ws, const int* rows,
                        const float* x, size_t xstride, const float* x2, float* resid, float alpha, int k,
                        hipStream_t st, const float* norm_w = nullptr, float norm_eps = 0.f,
                        float* norm_out = nullptr, const int* types = nullptr, const float* resid_gate = nullptr,
                        bool tokens = false) {
    if (m < 1 || m > JL_MAX_MULTI) return fail(c, JL_ERR_ARG, "matvec multi: %d matrices", m);
    const TypeInfo* ti = nullptr;
    const TypeInfo* tis[JL_MAX_MULTI];
    int max_rows = 0;
    for (int i = 0; i < m; i++) {
        const int t = types ? types[i] : type;
        int rc = matvec_check(c, t, rows[i], k, &ti);
        if (rc != JL_OK) return rc;
        tis[i] = ti;
        if (!outs[i] || !ws[i]) return fail(c, JL_ERR_ARG, "matvec multi: null operand");
        if (t == JL_TYPE_Q4_K && !aligned16(ws[i])) return JL_DECLINED;
        if (((uintptr_t)ws[i] & 1) != 0) return JL_DECLINED;
        if (rows[i] > max_rows) max_rows = rows[i];
    }
    if (!x || !aligned16(x) || (x2 && !aligned16(x2)) || (xstride % 4) != 0) return JL_DECLINED;
    if ((norm_w && !aligned16(norm_w)) || (norm_out && !aligned16(norm_out))) return JL_DECLINED;
    MatVecMultiArgs a;
    memset(&a, 0, sizeof a);
    for (int i = 0; i < m; i++) {
        a.out[i] = outs[i];
        a.w[i] = (const uint8_t*)ws[i];
        a.nrows[i] = rows[i];
        a.type[i] = types ? types[i] : type;
        a.row_bytes_of[i] = (k / tis[i]->block_elems) * tis[i]->block_bytes;
    }
    a.x = x; a.x2 = x2; a.resid = resid; a.alpha = alpha; a.resid_gate = resid ? resid_gate : nullptr;
    a.xstride = xstride;
    a.norm_w = norm_w; a.norm_eps = norm_eps; a.norm_out = norm_out; a.inv_k = 1.0 / k;
    a.k = k; a.row_bytes = (k / ti->block_elems) * ti->block_bytes; a.per = c->act_window / 32;
    bool pair = !types;
    for (int i = 0; i < m && pair; i++) pair = q8_pair_form(c, type, ws[i], k);
    // Sixteen wavefronts a workgroup, one row each.  As many workgroups as are resident at once over all the
    // matrices -- one a CU, two for the paired Q8_0 form, whose registers allow them -- because one more round of
    // workgroups stages (norms, gates) the activation once more (us, with 512 workgroups for every type -> now:
    // gate + up with a norm in front Q4_K 2048 / 7168 7.9 -> 6.7, 4096 / 14336 13.0 -> 12.3, Q6_K 1536 / 4608 9.6 -> 7.1;
    // q + k + v of a 4096 k-quant block 8.2 -> 6.1); never more row groups than a matrix has.
    const int nwaves = 16, xpre = x_groups(c, k, nwaves * 64);
    int lanes = 64;
    if (!x2 && !resid && (types || xpre == 1) && (m > 1 || types || norm_w)) {
        long total = 0;
        bool plain8 = false;   // (the mixed-type kernel reads Q8_0 rows a block a slot)
        for (int i = 0; i < m; i++) {
            total += rows[i];
            plain8 |= (types ? types[i] : type) == JL_TYPE_Q8_0 && !pair;
        }
        lanes = matvec_lanes(c, k / (plain8 ? 32 : 64), total);
    }
    const int step = nwaves * (64 / lanes);
    const long slots = c->tune.grid > 0 ? c->tune.grid : (pair ? 2L : 1L) * c->num_cu;
    long lo = 1, gx = ((long)max_rows + step - 1) / step;
    while (lo < gx) {   // the largest gx whose workgroups with work are at most `slots`
        const long mid = (lo + gx + 1) / 2;
        long n = 0;
        for (int i = 0; i < m; i++) n += std::min(mid, ((long)rows[i] + step - 1) / step);
        if (n <= slots) lo = mid; else gx = mid - 1;
    }
    // (one matrix for several activations, a token each: a row group's workgroups on one XCD, whose L2 then holds its rows)
    bool same = m > 1 && gx > 8;
    for (int i = 1; i < m && same; i++) same = ws[i] == ws[0];
    if (same) gx &= ~7L;
    a.nwaves = nwaves; a.ngroups = (int)gx;
    Name name;
    // "matvec.act_split" = 1: a gated activation shared by the group's matrices is formed and
    // quantized once, by the quantizer kernel, and the matvec stages the int8 copy (the same
    // values, bit for bit).  Not the default: the extra launch costs what it saves (Q6_K
    // 4096 x 14336 over silu(gate) * up: 15.2 us against 14.4 with every workgroup forming it).
    const bool split_act = x2 && !types && !norm_w && xstride == 0 && c->tune.act_split == 1;
    // A single matrix with nothing in front of its quantizer but (perhaps) that activation is the
    // plain decode matvec with the residual add riding on it: its kernel carries no norm or gate
    // code and keeps every row loop in registers (Q6_K 4096 x 14336: 10.8 against 12.2 us).
    if (m == 1 && !types && !norm_w && (!x2 || split_act) && c->tune.act_split != 3) {
        const int8_t* q = nullptr;
        const float *as = nullptr, *s16 = nullptr;
        if (x2) {
            const size_t o_as = ((size_t)k + 255) & ~(size_t)255, o_s16 = o_as + (((size_t)(k / 32) * 4 + 255) & ~(size_t)255);
            int rc = grow(c, &c->act_ws, &c->act_ws_bytes, o_s16 + (size_t)(k / 16) * 4);
            if (rc != JL_OK) return rc;
            int8_t* qq = (int8_t*)c->act_ws;
            float* asw = (float*)((char*)c->act_ws + o_as);
            float* s16w = (float*)((char*)c->act_ws + o_s16);
            int per = c->act_window / 32;
            void* qp[] = {(void*)&x, (void*)&qq, (void*)&asw, (void*)&s16w, (void*)&k, (void*)&per, (void*)&x2};
            rc = launch(c, "jl_quantize_act", (unsigned)((k / 4 + 255) / 256), 1, 256, 0, st, qp);
            if (rc != JL_OK) return rc;
            q = qq; as = asw; s16 = s16w;
        }
        return matvec_launch(c, outs[0], type, ws[0], x2 ? nullptr : x, q, as, s16, rows[0], k, st, resid, alpha,
                             resid_gate);
    }
    if (split_act) {
        const size_t o_as = ((size_t)k + 255) & ~(size_t)255, o_s16 = o_as + (((size_t)(k / 32) * 4 + 255) & ~(size_t)255);
        int rc = grow(c, &c->act_ws, &c->act_ws_bytes, o_s16 + (size_t)(k / 16) * 4);
        if (rc != JL_OK) return rc;
        int8_t* q = (int8_t*)c->act_ws;
        float* as = (float*)((char*)c->act_ws + o_as);
        float* s16 = (float*)((char*)c->act_ws + o_s16);
        int per = c->act_window / 32;
        void* qp[] = {(void*)&x, (void*)&q, (void*)&as, (void*)&s16, (void*)&k, (void*)&per, (void*)&x2};
        rc = launch(c, "jl_quantize_act", (unsigned)((k / 4 + 255) / 256), 1, 256, 0, st, qp);
        if (rc != JL_OK) return rc;
        a.x = nullptr; a.x2 = nullptr; a.q = q; a.as = as; a.s16 = s16;
        name << "jl_matvec_multi_" << (pair ? "q8_0p" : ti->tag) << "_q" << (resid ? "_res" : "");
        void* params[] = {&a};
        unsigned lds = (unsigned)(act_lds_bytes(k) + (pair ? (size_t)k + 16 : 0));
        return launch(c, name, (unsigned)gx, (unsigned)m, nwaves * 64, lds, st, params);
    }
    if (types) name << "jl_matvec_segments";
    else name << "jl_matvec_multi_" << (pair ? "q8_0p" : tokens && type == JL_TYPE_Q4_K ? "q4kf" : tokens ? q6_tag(c, type) : ti->tag);
    name << (norm_w ? x2 ? "_na" : "_n" : x2 ? "_a" : "") << (types || xpre == 1 ? "" : xpre == 4 ? "_x4" : "_x2") << (resid ? "_res" : "");
    if (lanes != 64) name << "_l" << lanes;
    void* params[] = {&a};
    // (+ 16 to round the staging area up)
    unsigned lds = (unsigned)(act_lds_bytes(k) + (pair ? (size_t)k + 16 : 0) + 16 + JL_NORM_LDS_BYTES);
    return launch(c, name, (unsigned)gx, (unsigned)m, nwaves * 64, lds, st, params);
}

int ensure_stage(jl_ctx* c, void** buf, size_t* have, size_t need) { return grow(c, buf, have, need); }

// Applies the ranges jl_forget queued: every device copy keyed inside one of them is
// unlinked and freed.  Called with c->mu held, before a residency lookup.
void drain_forget(jl_ctx* c) {
    std::vector<std::pair<uintptr_t, uintptr_t>> todo;
    {
        std::lock_guard<std::mutex> g(c->forget_mu);
        todo.swap(c->pending_forget);
    }
    for (const auto& r : todo)
        for (auto it = c->resident.begin(); it != c->resident.end();) {
            const uintptr_t k0 = (uintptr_t)it->first;
            if (k0 >= r.first && k0 < r.second) {
                if (!c->no_device) (void)H->Free(it->second.dev);
                it = c->resident.erase(it);
            } else {
                ++it;
            }
        }
}

// Device copy of host weight bytes, keyed on the host pointer.
int resident_weight(jl_ctx* c, const void* w, size_t bytes, void** dev) {
    auto it = c->resident.find(w);
    if (it != c->resident.end() && it->second.bytes == bytes) {
        *dev = it->second.dev;
        return JL_OK;
    }
    if (it != c->resident.end()) {
        HIP_TRY(c, H->Free(it->second.dev));
        c->resident.erase(it);
    }
    void* d = nullptr;
    HIP_TRY(c, H->Malloc(&d, bytes));
    hipError_t e = H->Memcpy(d, w, bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)H->Free(d);
        return fail(c, JL_ERR_HIP, "weight upload: %s", H->GetErrorString(e));
    }
    c->resident[w] = Resident{d, bytes};
    *dev = d;
    return JL_OK;
}

int ws_ensure(jl_ctx* c, void** buf, size_t* have, size_t need);
// The work lists a block's grouping made for tiles of 64 and of 128 columns.
struct MoeLists { uint32_t* wl[2]; int nslots; };
int moe_matvec_launch(jl_ctx* c, float* out0, float* out1, int type, const void* bank0, const void* bank1,
                      const float* x, const float* x2, const uint32_t* src, const uint32_t* start,
                      int n_expert, int ncols, int nrows, int k, hipStream_t st,
                      const jl_packed_bank* pb0 = nullptr, const jl_packed_bank* pb1 = nullptr, int nsrc = 0, const MoeLists* lists = nullptr);

// plane banks of a mixture: from this many columns an expert (on average) the matrix-core tile
// per expert takes over from the dot-product form ("moe.form" = 1 / 4 forces one)
constexpr long kMoePlaneTileCols = 14;
constexpr int kGemmTile = 128;         // tokens and rows per workgroup (kernels/gemm_q4k.h)
constexpr int kGemmStride = 152;       // f16 per stage row
constexpr unsigned gemm_lds_bytes(int rows) {   // two weight stages, row scales, token scales
    return 2u * rows * kGemmStride * 2u + 2u * 2u * rows * 4u + 2u * kGemmTile * 4u;
}
constexpr unsigned kGemmLdsBytes = gemm_lds_bytes(128);
constexpr size_t kGemmAStageBytes = 9 * 1024;  // per 32 tokens and stage: nine fragments of 64 lanes x 16 B

size_t gemm_ws_need(int ntok, int k) {
    size_t tok_pad = ((size_t)ntok + 255) / 256 * 256;   // the widest token tile of any form
    size_t nsb = (size_t)k / 256;
    return nsb * 2 * (tok_pad / 32) * kGemmAStageBytes + nsb * tok_pad * 4;
}

int gemm_ws_ensure(jl_ctx* c, size_t need) { return grow(c, &c->gemm_ws, &c->gemm_ws_bytes, need); }

// Calls jl_reserve covers allocate nothing, whatever their rows: a workspace that grows with the rows is then only
// used as far as it is there.  K slices: the Q4_K and MXFP4 forms cut a grid to at most two rounds of the CUs, whose
// tiles this many bytes hold; the int8 tiles, whose rule has no such bound, keep to it where it is all there is.
bool reserved_for(const jl_ctx* c, int ntok, int k) {
    for (const auto& r : c->reserved)
        if (ntok <= r.first && k <= r.second) return true;
    return false;
}
size_t slab_reserve(const jl_ctx* c) { return (size_t)c->num_cu * 256 * 128 * 4; }

constexpr size_t kGemmW16StageVecs = 1152;   // JL_GEMM_W16_STAGE_VECS
constexpr unsigned kGemmW16LdsBytes = 2u * 1152u * 16u + 2u * kGemmTile * 4u;

// Two-pass form: expand the weights into f16 fragments once, then the matrix kernel.
int gemm_q4k_w16_launch(jl_ctx* c, float* out, const void* w, const uint16_t* bq, const float* da, int nrows,
                        int k, int ntok, int tok_pad, hipStream_t st) {
    const int nsb = k / 256;
    const int nrt = (nrows + 63) / 64, nrows_pad = nrt * 64, ntt = tok_pad / kGemmTile;
    const size_t w16_bytes = (size_t)nrt * 2 * nsb * kGemmW16StageVecs * 16;
    const size_t need = w16_bytes + (size_t)nsb * nrows_pad * 8;
    int rcw = grow(c, &c->w16_ws, &c->w16_ws_bytes, need);
    if (rcw != JL_OK) return rcw;
    float* wsc = (float*)((char*)c->w16_ws + w16_bytes);
    GemmW16PrepArgs pa;
    pa.w = (const uint8_t*)w; pa.w16 = c->w16_ws; pa.wsc = wsc;
    pa.nrows = nrows; pa.nrows_pad = nrows_pad; pa.k = k; pa.row_bytes = nsb * 144;
    void* pp[] = {&pa};
    int rc = launch(c, "jl_gemm_w16_prep_q4k", (unsigned)nsb, (unsigned)(nrows_pad / 32), 256, 0, st, pp);
    if (rc != JL_OK) return rc;
    GemmW16Args ga;
    ga.out = out; ga.w16 = c->w16_ws; ga.wsc = wsc; ga.bq = bq; ga.da = da;
    ga.nrows = nrows; ga.nrows_pad = nrows_pad; ga.k = k; ga.ntok = ntok; ga.tok_pad = tok_pad;
    ga.ntt = ntt; ga.nrt = nrt;
    void* gp[] = {&ga};
    const unsigned groups = (unsigned)((nrt + 7) / 8 * 8) * (unsigned)ntt;
    return launch(c, "jl_gemm_q4k_w16", groups, 1, 256, kGemmW16LdsBytes, st, gp);
}

// Q4_K prefill GEMM on the f16 matrix cores; operands are device pointers.  Forms (tuning
// key "gemm.form", 0 = choose): 1 = 128-token x 64-row tiles, weights dequantized in the
// kernel; 2 = 256-token x 128-row tiles, a wavefront across all 128 rows (least L1 traffic
// per matrix instruction, for grids that still fill the chip); 3 = weights expanded once
// per call into f16 fragments, then 128 x 64 tiles; 6 = 128 x 64 tiles that walk the whole of K,
// its halves on two groups of four wavefronts (grids of half a round up to one round of the chip).
struct PlaneRef {
    const uint32_t *qs, *d, *sc;
    int row, stride;
};

constexpr int kGemmWideTok = 256;
// JL_GEMM_K2_LDS_BYTES: two groups of (two weight stages, minimum columns, row scales, token scales)
constexpr unsigned kGemmK2LdsBytes = 2u * (2u * 64u * 136u * 2u + 2u * 64u * 24u * 2u + 2u * 64u * 2u * 4u + 2u * 128u * 4u);
constexpr unsigned kGemmWideLdsBytes = 2u * 128u * 136u * 2u + 2u * 128u * 24u * 2u + 2u * 128u * 2u * 4u + 2u * kGemmWideTok * 4u;   // JL_GEMM_WIDE_LDS_BYTES

// A grid of at most a round and a half of 32-row workgroups: the form that takes a lane's operand
// words straight from GGUF rows (no plane form of it exists).
bool gemm_q4k_few_applies(const jl_ctx* c, int nrows, int k, int ntok) {
    const int form = c->tune.gemm_form;
    if ((size_t)nrows * (size_t)(k / 256) * 144 >= ((size_t)1 << 32)) return false;
    const long few32_groups = (long)((nrows + 31) / 32) * ((ntok + 63) / 64);
    return ((form == 0 && 2 * few32_groups <= 3L * c->num_cu) || (form == 5 && ntok <= 1024)) && ntok > 64;
}

// pl: the weights as packed planes (w unused): the tiled forms read them where they lie.  The
// caller has checked that gemm_q4k_few_applies() is false.
int gemm_q4k_launch(jl_ctx* c, float* out, const void* w, const float* x, int nrows, int k, int ntok,
                    hipStream_t st, const PlaneRef* pl = nullptr) {
    int form = c->tune.gemm_form;
    if (pl && form == 3) form = 0;
    if (!pl && gemm_q4k_few_applies(c, nrows, k, ntok)) {
        // some more than few tokens, few enough rows: 32-row x 64-token workgroups that split K,
        // one to a CU, while the grid is at most a round and a half (4096 rows: up to 192
        // tokens; measured against the tiled forms, 128 tokens x 4096 rows 24.6 -> 16.5 us;
        // at 14336 rows the tiled forms win)
        const int tok_pad = (ntok + 63) / 64 * 64, nsb = k / 256;
        int rc = gemm_ws_ensure(c, gemm_ws_need(tok_pad, k));
        if (rc != JL_OK) return rc;
        uint16_t* bq = (uint16_t*)c->gemm_ws;
        float* da = (float*)((char*)c->gemm_ws + (size_t)nsb * 2 * (tok_pad / 32) * kGemmAStageBytes);
        GemmPrepArgs pa;
        pa.x = x; pa.bq = bq; pa.da = da; pa.ntok = ntok; pa.tok_pad = tok_pad; pa.k = k;
        void* pp[] = {&pa};
        rc = launch(c, "jl_gemm_prep_q4k_w16", (unsigned)nsb, (unsigned)(tok_pad / 32), 1024, 0, st, pp);
        if (rc != JL_OK) return rc;
        GemmArgs ga;
        ga.out = out; ga.w = (const uint8_t*)w; ga.bq = bq; ga.da = da;
        ga.nrows = nrows; ga.k = k; ga.ntok = ntok; ga.tok_pad = tok_pad; ga.row_bytes = nsb * 144;
        ga.out_stride = nrows; ga.sb_per = 0;
        void* gp[] = {&ga};
        return launch(c, "jl_gemm_q4k_few32", (unsigned)((nrows + 31) / 32), (unsigned)(tok_pad / 64), 512, 0, st, gp);
    }
    if (form == 4 || form == 5) form = 0;   // outside the few-token forms' range
    const bool k2_fits = (k / 256) % 4 == 0 && kGemmK2LdsBytes <= c->lds_limit;
    if (form == 0 && k2_fits) {
        // 128 x 64 tiles over the whole of K: from half a round of the chip up to one round nothing
        // has to be cut along K and added afterwards (measured against the forms below, us:
        // 512 tokens x 4096 rows 32.0 against 37.9, 384 x 4096 29.4 against 35.9, 128 x 14336
        // 27.9 against 36.2, 256 x 4096 26.5 against 27.7; two rounds and more go to the wide tile)
        const long k2_groups = (long)((ntok + kGemmTile - 1) / kGemmTile) * ((nrows + 63) / 64);
        if (k2_groups <= c->num_cu && 2 * k2_groups >= c->num_cu) form = 6;
    }
    if (form == 0) {
        const long wide_groups = (long)((ntok + kGemmWideTok - 1) / kGemmWideTok) * ((nrows + 127) / 128);
        // from a quarter of the CUs on: a smaller grid is widened along K below (measured
        // against the 64-row tiles: 1024 tokens x 4096 rows 56 against 62 us, 512 x 4096 38 against 40)
        // (not for a last token tile that is mostly padding: 128 tokens x 14336 rows 40 against 45 us)
        const bool padded = (ntok % kGemmWideTok) != 0 && (ntok % kGemmWideTok) <= kGemmWideTok / 2 && ntok < 2 * kGemmWideTok;
        form = 4 * wide_groups >= 3 * (long)c->num_cu || (4 * wide_groups >= (long)c->num_cu && !padded) ? 2 : 1;
    }
    if (form == 2 && kGemmWideLdsBytes > c->lds_limit) form = 1;
    if (form == 6 && !k2_fits) form = 1;
    // the opt-in folded-scale form (kernels/gemm_q4k_fold.h): asked for with "gemm.fold" = 1,
    // and only for a matrix whose scales jl_fold_admit_dev has checked
    bool fold = false;
    if (c->tune.gemm_fold == 1 && form == 2 && !pl && 2u * 128u * 136u * 2u <= c->lds_limit) {
        std::lock_guard<std::mutex> g(c->forget_mu);
        auto it = c->fold_ok.find((uintptr_t)w);
        fold = it != c->fold_ok.end() && it->second.first == nrows && it->second.second == k;
    }
    const int tile = form == 2 ? kGemmWideTok : kGemmTile;
    const int tok_pad = (ntok + tile - 1) / tile * tile;
    const int nsb = k / 256;
    int rc = gemm_ws_ensure(c, gemm_ws_need(tok_pad, k));
    if (rc != JL_OK) return rc;
    uint16_t* bq = (uint16_t*)c->gemm_ws;
    float* da = (float*)((char*)c->gemm_ws + (size_t)nsb * 2 * (tok_pad / 32) * kGemmAStageBytes);
    GemmPrepArgs pa;
    pa.x = x; pa.bq = bq; pa.da = da; pa.ntok = ntok; pa.tok_pad = tok_pad; pa.k = k;
    void* pp[] = {&pa};
    // sixteen wavefronts a workgroup: the chain of tokens a wavefront quantizes one after the other
    // is the kernel's length (whole matmul, 512 tokens x 4096 rows: 41.0 -> 39.7 us; 2048 tokens:
    // 87.1 -> 83.4; "gemm.prep" = 4 asks for four wavefronts)
    const bool prep16 = c->tune.gemm_prep != 4;
    // (the plane kernels take the activations in the planes' K order: their own prep)
    rc = launch(c, fold ? "jl_gemm_prep_q4k_fold" : pl ? "jl_gemm_prep_q4k_planes" : prep16 ? "jl_gemm_prep_q4k_w16" : "jl_gemm_prep_q4k",
                (unsigned)nsb, (unsigned)(tok_pad / 32), fold || pl || prep16 ? 1024 : 256, 0, st, pp);
    if (rc != JL_OK) return rc;
    if (form == 3) return gemm_q4k_w16_launch(c, out, w, bq, da, nrows, k, ntok, tok_pad, st);
    GemmArgs ga;
    if (pl) { ga.pqs = pl->qs; ga.pd = pl->d; ga.psc = pl->sc; ga.prow0 = pl->row; ga.pstride = pl->stride; }
    ga.out = out; ga.w = (const uint8_t*)w; ga.bq = bq; ga.da = da;
    ga.nrows = nrows; ga.k = k; ga.ntok = ntok; ga.tok_pad = tok_pad; ga.row_bytes = nsb * 144;
    ga.out_stride = nrows; ga.sb_per = 0;
    void* gp[] = {&ga};
    if (fold) {
        // four wavefronts a workgroup, two workgroups a CU, from a full round of the chip on;
        // eight below (measured, us: 2048 tokens x 14336 rows 238 against 251; 1024 x 4096
        // 59.7 against 55.1; a round or so, 2048 x 4096 and 512 x 14336, the same)
        const long groups = (long)(tok_pad / kGemmWideTok) * ((nrows + 127) / 128);
        const bool w8 = c->tune.gemm_fold_waves == 8 || (c->tune.gemm_fold_waves != 4 && groups < (long)c->num_cu);
        return launch(c, w8 ? "jl_gemm_q4k_fold_wide" : "jl_gemm_q4k_fold_wide4", (unsigned)(tok_pad / kGemmWideTok),
                      (unsigned)((nrows + 127) / 128), w8 ? 512 : 256, 2u * 128u * 136u * 2u, st, gp);   // JL_GEMM_FOLD_LDS_BYTES
    }
    if (form == 6)   // 128 x 64 tiles over the whole of K, the K halves on two groups of wavefronts
        return launch(c, pl ? "jl_gemm_q4k_k2_planes" : "jl_gemm_q4k_k2", (unsigned)(tok_pad / kGemmTile), (unsigned)((nrows + 63) / 64), 512,
                      kGemmK2LdsBytes, st, gp);
    int rows_left = nrows;
    if (form == 2) {
        // One workgroup per CU: a grid of f full rounds and a last round at most half full
        // leaves half the chip idle for a whole round.  The rows of that last round go to the
        // 128 x 64 tiles instead (two workgroups per CU), which fill the chip once more.
        const long ntt = tok_pad / kGemmWideTok, nrt = (nrows + 127) / 128;
        const long full = ntt * nrt / c->num_cu, rem = ntt * nrt - full * c->num_cu;
        long nrt_wide = nrt;
        if (c->tune.gemm_form == 0 && full >= 1 && rem > 0 && 2 * rem <= c->num_cu) nrt_wide = full * c->num_cu / ntt;
        ga.nrows = nrt_wide == nrt ? nrows : (int)(nrt_wide * 128);
        // a grid of at most half the CUs is widened along K, partial slabs added in order
        int wsplit = c->tune.gemm_split > 0 ? c->tune.gemm_split : (c->tune.gemm_form == 0 ? (int)(c->num_cu / (ntt * nrt)) : 1);
        if (wsplit > 8) wsplit = 8;
        if (wsplit > nsb) wsplit = nsb;
        if (wsplit > 1) {
            const int per = (nsb + wsplit - 1) / wsplit;
            wsplit = (nsb + per - 1) / per;   // no empty split
        }
        if (wsplit > 1 && nrt_wide == nrt) {
            const size_t n = (size_t)ntok * nrows;
            rc = ws_ensure(c, &c->mx_ws, &c->mx_ws_bytes, n * wsplit * 4);
            if (rc != JL_OK) return rc;
            ga.out = (float*)c->mx_ws; ga.sb_per = (nsb + wsplit - 1) / wsplit;
            rc = launch(c, pl ? "jl_gemm_q4k_wide_planes" : "jl_gemm_q4k_wide", (unsigned)ntt, (unsigned)nrt, 512,
                        kGemmWideLdsBytes, st, gp, (unsigned)wsplit);
            if (rc != JL_OK) return rc;
            SumPartsArgs sa;
            sa.out = out; sa.part = (const float*)c->mx_ws; sa.n = n; sa.nsplit = wsplit;
            void* sp[] = {&sa};
            return launch(c, "jl_sum_parts", (unsigned)((n + 255) / 256), 1, 256, 0, st, sp);
        }
        rc = launch(c, pl ? "jl_gemm_q4k_wide_planes" : "jl_gemm_q4k_wide", (unsigned)ntt, (unsigned)nrt_wide, 512,
                    kGemmWideLdsBytes, st, gp);
        rows_left = nrows - ga.nrows;
        if (rc != JL_OK || rows_left == 0) return rc;
        if (pl) ga.prow0 += ga.nrows;
        else ga.w += (size_t)ga.nrows * ga.row_bytes;
        ga.out += ga.nrows;
        ga.nrows = rows_left;
    }
    // 64-row workgroups, two to a CU, unless asked for the 128-row form
    const int rows = c->tune.gemm_rows == 128 && !pl ? 128 : 64;
    const char* const r64 = pl ? "jl_gemm_q4k_r64_planes" : "jl_gemm_q4k_r64";
    if (rows == 64 && rows_left == nrows) {
        // a grid that leaves most of the chip idle (few tokens) is widened along K
        const long groups = (long)(tok_pad / kGemmTile) * ((nrows + 63) / 64);
        int nsplit = c->tune.gemm_split > 0 ? c->tune.gemm_split
                     : (c->tune.gemm_form == 0 && groups <= c->num_cu ? (int)(2 * c->num_cu / groups) : 1);
        if (nsplit > 8) nsplit = 8;
        if (nsplit > nsb) nsplit = nsb;
        if (nsplit > 1) {
            const int per = (nsb + nsplit - 1) / nsplit;
            nsplit = (nsb + per - 1) / per;   // no empty split
            const size_t n = (size_t)ntok * nrows;
            rc = ws_ensure(c, &c->mx_ws, &c->mx_ws_bytes, n * nsplit * 4);
            if (rc != JL_OK) return rc;
            ga.out = (float*)c->mx_ws; ga.sb_per = per;
            rc = launch(c, r64, (unsigned)(tok_pad / kGemmTile), (unsigned)((nrows + 63) / 64), 256,
                        gemm_lds_bytes(64), st, gp, (unsigned)nsplit);
            if (rc != JL_OK) return rc;
            SumPartsArgs sa;
            sa.out = out; sa.part = (const float*)c->mx_ws; sa.n = n; sa.nsplit = nsplit;
            void* sp[] = {&sa};
            return launch(c, "jl_sum_parts", (unsigned)((n + 255) / 256), 1, 256, 0, st, sp);
        }
    }
    return launch(c, rows == 128 ? "jl_gemm_q4k_r128" : r64, (unsigned)(tok_pad / kGemmTile),
                  (unsigned)((rows_left + rows - 1) / rows), rows == 128 ? 512 : 256, gemm_lds_bytes(rows), st, gp);
}

// The int8 tile forms (kernels/gemm_i8.h): Q8_0, Q4_K and Q6_K with window 32, Q6_K with the k-quant window.
struct I8Shape { int rt, tw; };
unsigned gemm_i8_lds(const jl_ctx* c, int type, I8Shape f) {   // JL_GEMM_I8_LDS_BYTES
    const unsigned planes = type == JL_TYPE_Q6_K ? 2 : 1, rows = 32u * f.rt * (f.tw < 4 ? 4 / f.tw : 1), mins = type == JL_TYPE_Q4_K;
    return 2u * (planes * rows * 128u + (c->act_window == 32 ? (mins + 1) * (rows * 16u + 4u * 32u * f.tw * 4u) : 0u));
}
bool gemm_i8_applies(const jl_ctx* c, int type, int nrows, int k, int ntok) {
    if (type != JL_TYPE_Q8_0 && type != JL_TYPE_Q4_K && type != JL_TYPE_Q6_K) return false;
    if (c->act_window != 32 && !(c->act_window == 256 && type == JL_TYPE_Q6_K)) return false;
    return k % 128 == 0 && ntok <= 65535 * 4 && (nrows + 63) / 64 <= 65535 && (k + 255) / 256 <= 65535;
}
Name gemm_i8_name(const char* pre, const jl_ctx* c, int type, I8Shape f) {
    Name n;
    n << pre << "_i8_" << type_info(type)->tag << (c->act_window == 256 ? "w_r" : "_r") << f.rt << "t" << f.tw;
    return n;
}

size_t gemm_i8_acts(int type, int ntok, int k) {   // bytes of the activations' fragments and scales
    const size_t tok_pad = ((size_t)ntok + 127) / 128 * 128;
    return (size_t)(k / 128) * (tok_pad / 32) * 4096 + (type == JL_TYPE_Q4_K ? 2 : 1) * (size_t)(k / 32) * tok_pad * 4;
}
// The tile and the slices of K of a launch, and what the tiles should take.
struct I8Plan { I8Shape f; int nsplit; double us; int tall; };
I8Plan gemm_i8_plan(const jl_ctx* c, int type, int nrows, int k, int ntok) {
    const bool q6 = type == JL_TYPE_Q6_K, q4 = type == JL_TYPE_Q4_K;
    const int nstage = k / 128;
    const int unit = q6 || q4 ? 2 : 1, nunit = nstage / unit;   // stages a split is made of
    // Shape and K split by what they should take.  A wavefront's 32 x 32 x 32 block costs its SIMD `many` us with two or
    // three wavefronts there and `alone` with one; workgroups are resident two (128 x 128: Q8_0 only, the others have no
    // registers for it) or three (128 x 64; two for the k-quants) a CU; the slabs of a split a launch (hidden under the
    // tail of the tiles) and a trip through memory.  Fitted to 19 shapes (1024 x 4096 to 14336 x 4096, 100 to 2048 tokens)
    // of every type at 1 to 8 splits, 6 % each; the pick is within 5 % of the best split at all but eight of the 76.  (One
    // pair of constants for every type left the k-quants uncut: window 32, 512 tokens of 4096 x 4096 Q4_K 62 against 52
    // in two, Q6_K 80 against 66, 900 tokens of 1700 x 8192 112 against 85 and 143 against 105.)
    // (Q8_0's and Q4_K's since their sums come as floats: 512 to 2048 tokens of five shapes.)  Q8_0, 256 tokens x 128 rows on eight
    // wavefronts, one workgroup a CU: a weight's narrow loads, which fill L1 under the 128-token tile (0.70 of 0.67 million cycles), serve
    // twice the tokens; 2048 tokens of 4096 x 14336 330 -> 303, 1024 of 14336 x 4096 177 -> 160, 512 93 -> 85, but 1500 of 8192 x 2048,
    // a round and a half, 84 (90 so).
    struct Shape { int rt, tw, cap; double many, alone; };
    static const Shape q8_shapes[] = {{4, 8, 1, 0.073, 0.146}, {4, 4, 2, 0.081, 0.115}, {2, 4, 3, 0.086, 0.122}};
    const Shape one = {2, 4, 2, q4 ? 0.106 : c->act_window == 32 ? 0.160 : 0.097, q4 ? 0.165 : c->act_window == 32 ? 0.241 : 0.131};
    const bool q8 = type == JL_TYPE_Q8_0;
    I8Shape f = {2, 4};
    int nsplit = 1, tall = 1 << 24;
    double best = 1e30;
    // Slabs as far as the static array has room for them behind the activations, in every call, so that a call that may
    // not allocate is served where one without slices fits, with the slices of the call that may (without that bound one
    // drawn shape in thirteen was refused for its slices; by the estimate it costs 0.3 % on average).
    const size_t n = (size_t)ntok * nrows, acts = (gemm_i8_acts(type, ntok, k) + 255) & ~(size_t)255;
    size_t most = acts < jl_static_scratch_bytes() ? jl_static_scratch_bytes() - acts : 0;
    if (reserved_for(c, ntok, k)) most = std::min(most, slab_reserve(c));
    for (int i = 0; i < (q8 ? 3 : 1); i++) {
        const Shape& h = q8 ? q8_shapes[i] : one;
        if (q8 && c->tune.gemm_i8 > 0 && i != c->tune.gemm_i8 % 3) continue;
        const int rt = h.rt, waves = h.tw / 4;   // (of a workgroup on a SIMD)
        const long cap = h.cap, groups = (long)((ntok + 32 * h.tw - 1) / (32 * h.tw)) * ((nrows + 32 * rt - 1) / (32 * rt));
        for (int s = 1; s <= 8 && s <= nunit; s++) {
            if (c->tune.gemm_split > 0 && s != std::min(std::min(c->tune.gemm_split, 8), nunit)) continue;
            const int per = (nunit + s - 1) / s;
            if ((nunit + per - 1) / per != s) continue;   // no empty split
            if (s > 1 && n * s * 4 > most) continue;
            const long wgs = groups * s, full = wgs / (cap * c->num_cu), left = wgs - full * cap * c->num_cu;
            const double block = 4 * rt * per * unit;     // of a wavefront
            double us = full * (0.15 + h.many * waves * cap * block);
            if (left) us += 0.15 + std::max(h.many * waves * ((left + c->num_cu - 1) / c->num_cu), h.alone) * block;
            if (s > 1) us += 0.25 + 1.16e-6 * (s + 1) * n;
            // 256 tokens x 128 rows: a last round of at most half of the CUs gives its rows to tiles of 64 instead, which take 0.59 of a
            // tile's time and fill it (17 shapes whose tiles are these anyway, K 256 to 2688: 0.94 of the time on average, none more than 0.97;
            // 2048 tokens of 14336 x 4096, 3.5 rounds, 334 -> 322).  With it these tiles take over from the others from K = 1536 on alone
            // (25 shapes 0.93, none slower; below, 18 shapes, 0.96 to 1.14: a short chain's start, which the estimate leaves out, is longer here).
            int high = 1 << 24;
            if (h.tw == 8 && s == 1 && full && left && c->tune.gemm_tall != 1) {
                const long ttiles = (ntok + 255) / 256, tall_n = full * c->num_cu / ttiles, low = ((nrows - 128 * tall_n + 63) / 64) * ttiles;
                const double mixed = full * (0.15 + h.many * waves * block) + 0.15 + 0.59 * h.many * waves * block;
                if (low <= c->num_cu && mixed < us) {
                    high = (int)tall_n;
                    if (k >= 1536) us = mixed;
                }
            }
            if (us < best) { best = us; f = {rt, h.tw}; nsplit = s; tall = high; }
        }
    }
    return {f, nsplit, best, c->tune.gemm_tall > 1 ? c->tune.gemm_tall - 2 : tall};
}

int gemm_i8_launch(jl_ctx* c, float* out, int type, const void* w, const float* x, int nrows, int k, int ntok, hipStream_t st) {
    const bool q6 = type == JL_TYPE_Q6_K, q4 = type == JL_TYPE_Q4_K;
    const int tok_pad = (ntok + 127) / 128 * 128, nstage = k / 128;
    const size_t bq_bytes = (size_t)nstage * (tok_pad / 32) * 4096, da_bytes = (size_t)(k / 32) * tok_pad * 4;
    int rc = gemm_ws_ensure(c, bq_bytes + (q4 ? 2 : 1) * da_bytes);
    if (rc != JL_OK) return rc;
    GemmPrepArgs pa;
    pa.x = x; pa.bq = (uint16_t*)c->gemm_ws; pa.da = (float*)((char*)c->gemm_ws + bq_bytes);
    pa.ntok = ntok; pa.tok_pad = tok_pad; pa.k = k; pa.per = c->act_window / 32;
    if (q4) pa.dsum = (float*)((char*)pa.da + da_bytes);   // the minimums meet d_a * block sums
    void* pp[] = {&pa};
    rc = launch(c, "jl_gemm_i8_prep", (unsigned)((k + 255) / 256), (unsigned)(tok_pad / 32), 1024, 0, st, pp);
    if (rc != JL_OK) return rc;
    GemmArgs ga;
    ga.out = out; ga.w = (const uint8_t*)w; ga.bq = pa.bq; ga.da = pa.da; ga.dsum = pa.dsum;
    ga.nrows = nrows; ga.k = k; ga.ntok = ntok; ga.tok_pad = tok_pad;
    ga.row_bytes = q6 ? (k / 256) * 210 : q4 ? (k / 256) * 144 : (k / 32) * 34;
    ga.out_stride = nrows; ga.sb_per = 0;
    void* gp[] = {&ga};
    const int unit = q6 || q4 ? 2 : 1, nunit = nstage / unit;   // stages a split is made of
    const I8Plan plan = gemm_i8_plan(c, type, nrows, k, ntok);
    const I8Shape f = plan.f;
    const int nsplit = plan.nsplit;
    const size_t n = (size_t)ntok * nrows;
    const int tt = 32 * f.tw, tr = 32 * f.rt, per = (nunit + nsplit - 1) / nsplit;
    if (nsplit > 1) {
        rc = ws_ensure(c, &c->mx_ws, &c->mx_ws_bytes, n * nsplit * 4);
        if (rc != JL_OK) return rc;
        ga.out = (float*)c->mx_ws; ga.sb_per = per * unit;
    }
    int rtiles = (nrows + tr - 1) / tr;
    if (f.tw == 8 && plan.tall < rtiles) {
        ga.tall = plan.tall;
        rtiles = plan.tall + (nrows - 128 * plan.tall + 63) / 64;
    }
    rc = launch(c, gemm_i8_name("jl_gemm", c, type, f), (unsigned)((ntok + tt - 1) / tt), (unsigned)rtiles, 64u * f.tw,
                gemm_i8_lds(c, type, f), st, gp, (unsigned)nsplit);
    if (rc != JL_OK || nsplit == 1) return rc;
    SumPartsArgs sa;
    sa.out = out; sa.part = (const float*)c->mx_ws; sa.n = n; sa.nsplit = nsplit;
    void* sp[] = {&sa};
    return launch(c, "jl_sum_parts", (unsigned)((n + 255) / 256), 1, 256, 0, st, sp);
}

// Few tokens, or few columns an expert, on the int8 matrix cores (kernels/few_i8.h): up to two
// matrices (banks) of one type and shape over the same columns.
struct FewCall {
    int type = 0, nrows = 0, k = 0, ncols = 0, nmat = 1, n_expert = 1;
    const void* w[2] = {nullptr, nullptr};        // GGUF rows
    const PlaneRef* pl[2] = {nullptr, nullptr};   // or planes
    size_t sheet_bytes = 0, sheet_words = 0;
    int row_step = 0;
    const float *x = nullptr, *x2 = nullptr;
    const uint32_t *src = nullptr, *start = nullptr;
    float *out[2] = {nullptr, nullptr}, *resid = nullptr;
};

// K in chunks of 128 (Q8_0 may end inside one); GGUF row offsets and plane words within 32 bits
bool few_fits(const jl_ctx* c, int type, bool planes, int nrows, int k, int ncols, int stride) {
    const TypeInfo* ti = type_info(type);
    if (!ti || c->tune.gemm_few == 2 || k % ti->block_elems || ncols > 65535 * 4 || (k + 255) / 256 > 65535) return false;
    if (planes)   // (a lane's offset: up to twelve planes of Q6_K's, the whole D plane of Q8_0's)
        return (size_t)stride * 4 * 12 < ((size_t)1 << 32) && (type != JL_TYPE_Q8_0 || (size_t)(k / 32) * (((size_t)stride + 1) / 2) * 4 < ((size_t)1 << 32));
    if (type == JL_TYPE_Q8_0 && k % 64) return false;   // (rows on 4-byte boundaries)
    return (size_t)nrows * (size_t)(k / ti->block_elems) * ti->block_bytes < ((size_t)1 << 32);
}

int few_form(int type, bool w256) { return type == JL_TYPE_Q8_0 ? 2 : type == JL_TYPE_Q4_K ? w256 : 3 + w256; }

// A workgroup's token tiles (of 16), row tiles (of 16) and wavefronts, over which K is dealt.
struct FewShape { int nt, rt, nw; double us = 0; };   // us: what launch and prep should take (one matrix)

// Token tiles: what the (average) group fills.  Two rules for the other two.
//
// One group: the least of an estimate, in units of a wavefront's step of 256 alone on its SIMD.  Workgroups of eight or
// four wavefronts run in rounds of `cap` a CU (registers of the fullest SIMD, and LDS), the last with what is left; a round takes `e` (its
// start, the reduction) and ceil(K / 256 / wavefronts) steps, a step a serial chain (longer with more row tiles) and a
// part of each wavefront the SIMD holds.  Fitted to 34 shapes (1024 x 1024 to 14336 x 4096) of every type, window and
// layout at 8, 24, 40 and 64 tokens over everything that is built: the pick is 1 to 3 % behind the best on average.
// Against always eight wavefronts, and row tiles where most CUs kept a workgroup, geometric means over them: 8 and 24
// tokens 2 to 4 % faster, 64 tokens 9 %, the worst loss 11 % and the largest gain 66 %: a workgroup over a round's end
// costs a whole round (rows of 9216 x 1280, window 32, 64 tokens: Q6_K 25.7 against 15.5).  (Three, five and six
// wavefronts are the best of some shapes and, estimated so, the worst of others: 5120 x 5120 Q6_K, 64 tokens, five 38.6,
// eight 25.7.)  Three token tiles: 33 to 48 tokens took four (40 tokens 24 % faster, never slower).
//
// Groups of a mixture (grid: rows, banks, experts; most groups part empty): row tiles as many as leave most CUs a
// workgroup, eight wavefronts.  More rows a workgroup share the activations' loads, and over planes widen the weights'
// (14336 x 4096 / 4096 x 4096, us, row tiles 1 / 2 / 4: Q8_0 planes 16 tokens 28.8 20.6 18.7 / 11.6 11.3 14.7; Q4_K
// planes 20.1 15.4 14.4 / 8.4 9.4 12.6; Q4_K rows 18.2 16.4 - / 8.5 10.2 -; Q8_0 rows 64 tokens 39.3 35.0 - /
// 13.5 18.0 -).
FewShape few_shape(const jl_ctx* c, int type, bool w256, bool planes, int nrows, int k, int ncols, bool groups, int n_expert, int nmat) {
    const int nsb = (k + 255) / 256, form = few_form(type, w256);
    const long avg = ((long)ncols + n_expert - 1) / n_expert, sheets = (long)n_expert * nmat, cus = c->num_cu;
    FewShape f = {1, 1, std::min(8, nsb)};
    if (groups) {
        f.nt = avg <= 16 ? 1 : avg <= 32 ? 2 : 4;
        // Rows, more than 32 columns.  Many workgroups: three token tiles where a CU holds three workgroups of them for four of two, else, k-quants,
        // two (four would take every group's activations and registers for columns that most experts do not have; Q8_0's are few enough, and from
        // K = 4096 on a second pass costs more).  us, two / three / four tiles, window 32, 36 columns: Q8_0 128 x 768 x 2048 twice 209 / 162 / 222,
        // 60 x 1280 x 2048 162 / 124 / 172, Q6_K 128 x 2048 x 768 123 / 115 / 156, 60 x 2048 x 1280 131 / 150 / 155, 100 x 512 x 1024 42 / 40 / 47;
        // 48 columns 238 / 221 / 230, 178 / 161 / 174, 139 / 147 / 161, 152 / 201 / 167, 47 / 52 / 49, 8 x 4096 x 4096 85 / 92 / 76.
        // Few workgroups, fewer than eight a CU of one row tile: they run at once, and the launch lasts as long as the passes of its fullest expert
        // (columns taken as dealt at random).  Three tiles where its columns should fit them: 36 columns, Q8_0 8 x 512 x 1024 9.5 / 7.9 / 8.5.  Else
        // four: 44 columns 9.7 / 10.7 / 8.7, Q6_K 2 x 1024 x 4096 twice 17 / 19 / 14, the same 8 with the k-quant window 10.2 / 11.1 / 8.9; two
        // where four would come with two row tiles, whose pass is twice as long, and K is short: Q8_0 8 x 512 x 512 twice 10.0 / 11.2 / 11.4.
        // 486 launches of 2 to 128 experts, 33 to 54 columns: 1.0 % behind the best of the three, always four 10 %.
        if (avg > 32 && !planes) {
            const int w = (f.nw + 3) / 4, two = c->few_simd[form][0][1][0] / w, three = c->few_simd[form][0][2][0] / w;
            const bool packs = 4 * three >= 3 * two, q8 = type == JL_TYPE_Q8_0;
            const long wgs = (nrows + 15) / 16 * sheets;
            const auto any_over = [&](int n) { return 1 - std::pow(1 - 0.5 * std::erfc((n + 0.5 - avg) / std::sqrt(2.0 * avg)), n_expert); };
            if (avg <= 34 && !packs && wgs > 2 * cus) f.nt = 2;   // (Q6_K 8 x 4096 x 4096, 33 columns 57 / 71 / 73)
            else if (wgs >= 8 * cus) {
                if (avg <= (q8 && nsb < 16 ? 48 : 44) && packs) f.nt = 3;
                else if (!q8 && nsb < 16) f.nt = 2;
            } else if (any_over(48) < 0.3 && (packs || wgs <= 2 * cus)) f.nt = 3;
            else if (nsb < 8 && (nrows + 31) / 32 * sheets >= cus) f.nt = 2;
            else if (any_over(64) >= 0.5) f.nt = packs ? 3 : 2;
        }
    }
    else f.nt = (int)std::min<long>((avg + 15) / 16, 4);
    if (c->tune.few_nt) f.nt = c->tune.few_nt;
    if (groups) {
        if (planes ? (nrows + 31) / 32 * sheets >= cus : (f.nt == 4 || (f.nt == 1 && type == JL_TYPE_Q4_K)) && (nrows + 31) / 32 * sheets >= cus)
            f.rt = 2;
        if (planes && f.nt <= 2 && (f.nt == 2 || type != JL_TYPE_Q6_K) && (nrows + 63) / 64 * sheets * 10 >= cus * 7) f.rt = 4;
    } else {
        // More than one token tile: the token tiles a workgroup takes by time, us: the prep, rounds of `start`, steps of a chain and of
        // the wavefronts the SIMD holds, both longer with every token tile.  Fitted to 12 shapes (1024 x 1024 to 14336 x 4096) at
        // 32 to 512 tokens with one to four token tiles 6 to 10 % each; the pick is 1.5
        // to 3 % behind the best.  Up to 64 tokens a split has to promise a seventh more, and Q8_0 planes, where the fit is worst, have
        // none (17 to 64 tokens, against all of them in one workgroup: Q4_K planes 1526 x 5120, 52 tokens 16.3 -> 12.5, Q6_K 1114 x
        // 10752, 57 tokens 29.6 -> 21.9; most shapes keep the one).
        static const struct { double start, chain0, chain1, part0, part1; } cost[5][2] = {   // [few_form()][planes]
            {{2.16, 0.53, 0.12, 0.00, 0.23}, {3.74, 0.82, 0.04, 0.00, 0.24}}, {{2.51, 0.36, 0.17, 0.06, 0.21}, {3.86, 0.37, 0.27, 0.23, 0.12}},
            {{1.88, 0.55, 0.19, 0.13, 0.16}, {3.90, 0.07, 0.17, 0.48, 0.16}}, {{1.92, 0.14, 0.52, 0.39, 0.14}, {3.41, 0.77, 0.36, 0.36, 0.18}},
            {{1.99, 0.12, 0.47, 0.36, 0.11}, {3.68, 0.66, 0.29, 0.37, 0.12}}};
        const auto& q = cost[form][planes];
        const int nt_lo = avg > (planes && type == JL_TYPE_Q8_0 ? 64 : 16) && !c->tune.few_nt ? 1 : f.nt, nt_hi = f.nt;
        double least = 1e30;
        f.us = 1e30;
        for (int nt = nt_lo; nt <= nt_hi; nt++) {
            const long tgroups = ((avg + 15) / 16 + nt - 1) / nt;
            // (over planes more row tiles get wider loads of the weights, which is most of a step with one token tile)
            const double e = planes && nt <= 2 ? 0.5 : 3, more = !planes ? 1.6 : nt == 1 ? 1.2 : 1.4;
            double best = 1e30, us = 0;
            FewShape g = {nt, 1, std::min(8, nsb)};
            for (int w : {8, 4}) {
                const int nw = std::min(w, nsb);
                double part = 0.25 * nw, chain = 1;
                for (int rt : {1, 2, 4}) {
                    const int simd = nt > 4 ? 0 : c->few_simd[form][planes][nt - 1][rt / 2];
                    if (!simd || nrows < rt) break;
                    const size_t lds = std::max(nw * JL_FEW_WAVE_BYTES(type, planes, rt), JL_FEW_RED_BYTES(nw, nt, rt));
                    if (lds > c->lds_limit) break;
                    const long cap = std::max<long>(1, std::min<long>(simd / ((nw + 3) / 4), (long)(c->lds_limit / lds)));
                    const long wgs = (nrows + 16 * rt - 1) / (16 * rt) * sheets * tgroups, full = wgs / (cap * cus), left = (wgs - full * cap * cus + cus - 1) / cus;
                    const int steps = (nsb + nw - 1) / nw;
                    double t = full * (e + steps * (chain + part * cap));
                    if (left) t += e + steps * (chain + part * left);
                    if (t < best) {
                        best = t; g.rt = rt; g.nw = nw;
                        const long rounds = full + (left > 0);
                        us = rounds * (q.start + steps * chain * (q.chain0 + q.chain1 * nt)) + steps * part * (full * cap + left) * (q.part0 + q.part1 * nt);
                    }
                    part *= more; chain *= 2;
                }
            }
            us += (planes ? 5.2 : 6.4) + (planes ? 1.9e-6 : 1.7e-6) * avg * k;
            const double weighed = avg <= 64 && nt < nt_hi ? 1.15 * us : us;
            if (best < 1e30 && weighed < least) { least = weighed; f = g; f.us = us; }
        }
        if (least == 1e30) f = {nt_hi, 1, std::min(8, nsb), 1e30};
    }
    if (c->tune.few_rt) f.rt = c->tune.few_rt;
    if (nrows < f.rt) f.rt = 1;
    if (c->tune.few_waves) f.nw = std::min(c->tune.few_waves, nsb);
    else if (c->tune.few_rt || groups) f.nw = std::min(8, nsb);
    while (f.nw > 1 && (size_t)f.nw * JL_FEW_WAVE_BYTES(type, planes, f.rt) > c->lds_limit) f.nw--;
    return f;
}

int few_launch(jl_ctx* c, const FewCall& f, hipStream_t st) {
    const bool planes = f.pl[0] != nullptr;
    const TypeInfo* ti = type_info(f.type);
    const int nch = (f.k + 255) / 256 * 2;
    const int nslots = f.start ? f.ncols / 16 + f.n_expert + 1 : (f.ncols + 15) / 16;
    const size_t q_bytes = (size_t)nch * nslots * 2048, s_bytes = (size_t)nch * nslots * 256;
    void** ws = f.start ? &c->moe_q_ws : &c->gemm_ws;
    int rc = grow(c, ws, f.start ? &c->moe_q_ws_bytes : &c->gemm_ws_bytes, q_bytes + 2 * s_bytes);
    if (rc != JL_OK) return rc;
    FewI8PrepArgs pa;
    pa.x = f.x; pa.x2 = f.x2; pa.src = f.src; pa.start = f.start;
    pa.bq = (uint32_t*)*ws; pa.da = (float*)((char*)*ws + q_bytes);
    pa.ds = f.type == JL_TYPE_Q4_K ? (float*)((char*)*ws + q_bytes + s_bytes) : nullptr;
    pa.k = f.k; pa.per = c->act_window / 32; pa.ncols = f.ncols; pa.n_expert = f.n_expert; pa.nslots = nslots;
    pa.nch = nch;
    pa.order = f.type == JL_TYPE_Q8_0 || !planes ? 0 : f.type == JL_TYPE_Q4_K ? 1 : 2;
    const bool w256 = f.type != JL_TYPE_Q8_0 && c->act_window == 256;
    pa.isum = w256;
    void* pp[] = {&pa};
    rc = launch(c, "jl_few_prep", (unsigned)((f.k + 255) / 256), (unsigned)((f.ncols + 3) / 4), 256, 0, st, pp);
    if (rc != JL_OK) return rc;
    FewI8Args a;
    memset(&a, 0, sizeof a);
    for (int m = 0; m < f.nmat; m++) {
        a.out[m] = f.out[m];
        a.w[m] = (const uint8_t*)f.w[m];
        if (planes) { a.pqs[m] = f.pl[m]->qs; a.pd[m] = f.pl[m]->d; a.psc[m] = f.pl[m]->sc; }
    }
    a.resid = f.resid; a.bq = pa.bq; a.da = pa.da; a.ds = pa.ds; a.start = f.start;
    a.sheet_bytes = f.sheet_bytes; a.sheet_words = f.sheet_words; a.row_step = f.row_step;
    if (planes) { a.prow0 = f.pl[0]->row; a.pstride = f.pl[0]->stride; }
    a.nrows = f.nrows; a.k = f.k; a.row_bytes = (f.k / ti->block_elems) * ti->block_bytes;
    a.ncols = f.ncols; a.nslots = nslots; a.nch = nch;
    const FewShape sh = few_shape(c, f.type, w256, planes, f.nrows, f.k, f.ncols, f.start != nullptr, f.n_expert, f.nmat);
    const int nt = sh.nt, rt = sh.rt, nw = sh.nw;
    a.nwaves = nw;
    const int ntile = (f.ncols + 15) / 16, tgroups = (ntile + nt - 1) / nt;
    a.tgroup = f.start ? 0 : (ntile + tgroups - 1) / tgroups;
    const unsigned lds = (unsigned)std::max(nw * JL_FEW_WAVE_BYTES(f.type, planes, rt), JL_FEW_RED_BYTES(nw, nt, rt));
    if (lds > c->lds_limit) return JL_DECLINED;
    Name name;
    name << "jl_few_" << ti->tag << (w256 ? "w_" : "_") << (planes ? "planes" : "rows") << "_t" << nt << "r" << rt;
    void* ap[] = {&a};
    return launch(c, name, (unsigned)((f.nrows + 16 * rt - 1) / (16 * rt)), (unsigned)(f.start ? f.n_expert : tgroups), (unsigned)(64 * nw), lds, st, ap,
                  (unsigned)f.nmat);
}

int packed_matvec_multi_launch(jl_ctx* c, int type, int m, float* const* outs, const PlaneRef* pls, const float* x, size_t xstride, const float* up,
                               float* resid, float alpha, const float* resid_gate, const float* norm_w, float norm_eps, float* norm_out, int nrows,
                               int k, hipStream_t st, bool tokens = false);
// A few tokens as that many decode matvecs in one launch (each reads the weights, the later ones from L2).
int tokens_matvec_launch(jl_ctx* c, float* out, int type, const void* w, const PlaneRef* pl, const float* x, int nrows, int k, int ntok, hipStream_t st) {
    float* outs[JL_MAX_MULTI];
    const void* ws[JL_MAX_MULTI];
    PlaneRef pls[JL_MAX_MULTI];
    int rows[JL_MAX_MULTI];
    for (int t = 0; t < ntok; t++) {
        outs[t] = out + (size_t)t * nrows; ws[t] = w; rows[t] = nrows;
        if (pl) pls[t] = *pl;
    }
    return pl ? packed_matvec_multi_launch(c, type, ntok, outs, pls, x, k, nullptr, nullptr, 0.f, nullptr, nullptr, 0.f, nullptr, nrows, k, st, true)
              : matvec_multi_launch(c, type, ntok, outs, ws, rows, x, k, nullptr, nullptr, 0.f, k, st, nullptr, 0.f, nullptr, nullptr, nullptr, true);
}
// Where: the few-token form is two launches, this is one.  Over rows a workgroup's sixteen wavefronts make `passes` steps of their
// lanes a row, each a chain of trips (Q8_0, two workgroups a CU: at least its bytes); over planes a wavefront goes through its share
// of K, longer with wider runs of rows, and longer where eight does not divide the runs (a run's workgroups then share no XCD).
// Two tokens of a k-quant always (they were two launches of the matvec), else up to eight where that is an eighth (planes: a fifth) below the
// few-token estimate.  us, before -> so: Q4_K 4096 x 4096 2 / 4 tokens 8.9 -> 6.3 / 9.2 -> 8.6, 2048 x 2048 8 tokens 8.9 -> 6.2, 14336 x
// 4096 2 tokens 16.3 -> 12.1, 4 tokens 16.5 (18.1 so); Q6_K 4096 x 14336 2 tokens 24.0 -> 16.1; Q8_0 planes 4096 x 4096 2 / 4 tokens
// 13.0 -> 8.0 / 12.9 (9.0 so).
bool tokens_matvec_wanted(const jl_ctx* c, int type, bool planes, int nrows, int k, int ntok, int stride) {
    if (ntok < 2 || ntok > JL_MAX_MULTI) return false;
    if (c->tune.gemm_few == 3) return true;
    if (ntok > 8 || c->tune.gemm_few || c->tune.gemm_form || c->gemm_min_tok != 3) return false;
    // (Short rows over planes, where one launch takes wider runs and a lane the more blocks of a row: NMSE against 64 bits at K =
    // 256 to 512, Q6_K two tokens 5.5e-15 and two launches 4.0e-15, Q8_0 three 5.2e-15 and the few-token kernel 4.3e-15.)
    if (planes && k < 1024 && type != JL_TYPE_Q4_K) return false;
    if (ntok == 2 && type != JL_TYPE_Q8_0) return true;
    // (Q6_K over planes, and short rows under a shorter window: the matvec's sums round more than the few-token kernel's, NMSE
    // against 64 bits 8.3e-15 and 4.8e-15 for eight tokens at K = 2048 over planes, 4.6e-15 and 4.3e-15 for three at K = 512)
    if (type == JL_TYPE_Q6_K && (planes || (c->act_window != 256 && k < 1024))) return false;
    if (!few_fits(c, type, planes, nrows, k, ntok, stride)) return false;
    const TypeInfo* ti = type_info(type);
    const bool q8 = type == JL_TYPE_Q8_0;
    const long cus = c->num_cu;
    const double mb = 1e-6 * nrows * ((double)k / ti->block_elems * ti->block_bytes);
    double us;
    if (!planes) {   // (matvec_multi_launch)
        const int slots = (k + 63) / 64, lanes = matvec_lanes(c, slots, (long)nrows * ntok), step = 16 * (64 / lanes);
        const long groups = (nrows + step - 1) / step;
        long gx = std::min(groups, std::max(1L, (q8 ? 2 : 1) * cus / ntok));
        if (gx > 8) gx &= ~7L;
        const double trips = (double)((groups + gx - 1) / gx) * ((slots + lanes - 1) / lanes);
        us = q8 ? std::max(4.3 + 0.125 * ntok * mb, 4.3 + (slots > 64 ? 2.2 : 1.5) * trips) : 4.3 + (type == JL_TYPE_Q4_K ? 1.0 : 1.28) * trips;
    } else {         // (packed_matvec_multi_launch)
        int rw = 64;
        while (rw > 16 && (long)ntok * ((nrows + rw - 1) / rw) < cus * 3 / 4) rw >>= 1;
        const long runs = (nrows + rw - 1) / rw, wgs = runs * ntok;
        const int nch = (k + 255) / 256, nw = std::min(nch, wgs <= cus ? 16 : 8);
        const double trips = (double)((wgs + (nw > 8 ? 1 : 3) * cus - 1) / ((nw > 8 ? 1 : 3) * cus)) * ((nch + nw - 1) / nw);
        const bool whole = runs % 8 == 0;
        us = std::max(4.3 + (whole ? 0.12 : 0.2) * ntok * mb, 4.5 + trips * (rw == 64 ? 3.1 : rw == 32 ? 2.2 : 1.8) * (whole ? 1 : 1.3));
    }
    return us < (planes ? 0.78 : 0.87) * few_shape(c, type, !q8 && c->act_window == 256, planes, nrows, k, ntok, false, 1, 1).us;
}

// Where the int8 few-token form serves a plain matmul.
bool few_applies(const jl_ctx* c, int type, bool planes, int nrows, int k, int ntok, int stride) {
    if (!few_fits(c, type, planes, nrows, k, ntok, stride)) return false;
    if (c->tune.gemm_few == 1 || (c->tune.gemm_form == 4 && ntok <= 64)) return true;
    if (c->tune.gemm_form != 0) return false;
    if (ntok > 64) {
        // Beyond one group of 64 the groups of tokens are workgroups of their own, and the weights' bytes come again from L2:
        // where the estimate is below a tiled GEMM's (which pays its slices of K, their sum and, over planes, the rows made anew).
        // Against those, us: Q8_0 2048 x 2048 96 tokens 18.2 -> 10.0, 4096 x 4096 256 planes 39.5 -> 29.2; Q4_K window 32 8192 x 2048
        // 128 29.4 -> 20.7, 1024 x 1024 512 22 -> 14; Q6_K 4096 x 4096 128 26.1 -> 23.8, window 32 32.2 -> 25.9; Q4_K 2048 x 8192 96
        // 27.4 -> 19.9, planes 34.4 -> 20.5.  The tiles stay, 14336 x 4096: Q8_0 rows 128 tokens 42.8 (51.9 so).
        // (A twelfth off the tiles' estimate for both errors.)
        if (ntok > 1024 || ntok < c->gemm_min_tok || c->tune.gemm_few || c->tune.gemm_split || c->tune.gemm_i8) return false;
        const size_t need = (size_t)((k + 255) / 256 * 2) * ((ntok + 15) / 16) * 2560;
        if (need > jl_static_scratch_bytes()) return false;
        const bool w256 = type == JL_TYPE_Q4_K && c->act_window == 256;
        double tiles = 1e30;
        if (w256 && gemm_q4k_few_applies(c, nrows, k, ntok)) {
            const long groups = (long)((nrows + 31) / 32) * ((ntok + 63) / 64), rounds = (groups + c->num_cu - 1) / c->num_cu;
            tiles = 8.9 + 3.2e-6 * ntok * k + 0.5 * rounds * (k / 256);   // (over planes 3 us and more above that: one choice for both layouts)
        } else if (!w256 && gemm_i8_applies(c, type, nrows, k, ntok)) {
            const I8Plan p = gemm_i8_plan(c, type, nrows, k, ntok);
            tiles = 11.7 + 1e-6 * ((ntok + 127) / 128 * 128) * k + 1.03 * p.us + (p.nsplit > 1 ? 1.8 : 0) + (planes ? 4.3 + 0.16e-6 * nrows * k : 0);
        }
        if (tiles == 1e30) return false;   // (nothing to be measured against: as before)
        return few_shape(c, type, type != JL_TYPE_Q8_0 && c->act_window == 256, planes && !w256, nrows, k, ntok, false, 1, 1).us < 0.92 * tiles;
    }
    // (two tokens: two matvecs are as fast for the k-quants, not for Q8_0: 21 against 22 us, 9.6 against 10.6)
    return ntok >= (type == JL_TYPE_Q8_0 ? 2 : c->gemm_min_tok);
}

// out [ntok][nrows] = x [ntok][k] W^T on device operands: the matrix-core GEMM where it
// applies, else one fused matvec launch per token (same values, token by token).
int matmul_launch(jl_ctx* c, float* out, int type, const void* w, const float* x, int nrows, int k,
                  int ntok, hipStream_t st) {
    const TypeInfo* ti = nullptr;
    int rc = matvec_check(c, type, nrows, k, &ti);
    if (rc != JL_OK) return rc;
    if (!out || !w || !x || ntok <= 0) return fail(c, JL_ERR_ARG, "matmul: bad operand");
    if (!aligned16(x) || (k % 4) != 0) return JL_DECLINED;
    if (tokens_matvec_wanted(c, type, false, nrows, k, ntok, 0)) {
        rc = tokens_matvec_launch(c, out, type, w, nullptr, x, nrows, k, ntok, st);
        if (rc != JL_DECLINED) return rc;
    }
    if (few_applies(c, type, false, nrows, k, ntok, 0) && ((uintptr_t)w & (type == JL_TYPE_Q4_K ? 15 : 3)) == 0) {
        FewCall f;
        f.type = type; f.nrows = nrows; f.k = k; f.ncols = ntok; f.w[0] = w; f.x = x; f.out[0] = out;
        rc = few_launch(c, f, st);
        if (rc != JL_DECLINED) return rc;
    }
    if (ntok >= c->gemm_min_tok && c->tune.gemm_form != 9 && ((uintptr_t)w & (type == JL_TYPE_Q4_K ? 15 : 1)) == 0 &&
        gemm_i8_applies(c, type, nrows, k, ntok))
        return gemm_i8_launch(c, out, type, w, x, nrows, k, ntok, st);
    const bool gemm = type == JL_TYPE_Q4_K && c->act_window == 256 && ntok >= c->gemm_min_tok &&
                      aligned16(w) && ntok <= 65535 * 4 && kGemmLdsBytes <= c->lds_limit;
    if (gemm) return gemm_q4k_launch(c, out, w, x, nrows, k, ntok, st);
    // Q8_0, a handful of tokens: the grouped dot-product kernel with the tokens as the columns
    // of a single group streams the rows once and beats the 128-token tile (14336 x 4096:
    // 2 tokens 17.4 against 21.7 us token by token, 3 tokens 18.6 against 35.2 for the tile, 8 tokens
    // 26.9 against 34.3, 12 tokens 41.8 against 34.5; Q6_K rows are too long for that kernel: 62 us at 3)
    if (type == JL_TYPE_Q8_0 && ntok >= 2 && ntok <= 8 && c->tune.gemm_form == 0 && aligned16(w) &&
        (size_t)nrows * ti->block_bytes * (k / ti->block_elems) % 2 == 0) {
        rc = moe_matvec_launch(c, out, nullptr, type, w, nullptr, x, nullptr, nullptr, c->one_group + 2 * ntok, 1, ntok,
                               nrows, k, st);
        if (rc != JL_DECLINED) return rc;
    }
    for (int t = 0; t < ntok; t++) {
        rc = matvec_launch(c, out + (size_t)t * nrows, type, w, x + (size_t)t * k, nullptr, nullptr,
                           nullptr, nrows, k, st);
        if (rc != JL_OK) return rc;
    }
    return JL_OK;
}

int ws_ensure(jl_ctx* c, void** buf, size_t* have, size_t need) { return grow(c, buf, have, need); }

// Words of the three planes of an nrows x k matrix (jit/gpu/kernels/pack.go:580-621).
bool packed_words(int type, size_t nrows, int k, size_t* nq, size_t* nd, size_t* nsc) {
    if (k <= 0 || nrows == 0) return false;
    switch (type) {
    case JL_TYPE_Q4_K:
        if (k % 256) return false;
        *nq = nrows * (size_t)(k / 32) * 4; *nd = nrows * (size_t)(k / 256); *nsc = *nd * 3;
        return true;
    case JL_TYPE_Q6_K:
        if (k % 256) return false;
        *nq = nrows * (size_t)(k / 16) * 3; *nd = nrows * (size_t)(k / 256); *nsc = nrows * (size_t)(k / 64);
        return true;
    case JL_TYPE_Q8_0:
        if (k % 32) return false;
        *nq = nrows * (size_t)(k / 32) * 8; *nd = (size_t)(k / 32) * ((nrows + 1) / 2); *nsc = 0;
        return true;
    case JL_TYPE_MXFP4:   // DSlots 4: an exponent byte a row, four rows a word (pack.go:543-575)
        if (k % 32) return false;
        *nq = nrows * (size_t)(k / 32) * 4; *nd = (size_t)(k / 32) * ((nrows + 3) / 4); *nsc = 0;
        return true;
    }
    return false;
}

int packed_check(jl_ctx* c, int type, const PlaneRef& pl, int nrows, int k, const TypeInfo** ti) {
    *ti = type_info(type);
    if (!*ti) return JL_DECLINED;
    if (nrows <= 0 || k <= 0 || pl.row < 0 || pl.stride <= 0)
        return fail(c, JL_ERR_ARG, "packed: nrows=%d k=%d row=%d stride=%d", nrows, k, pl.row, pl.stride);
    if ((long)pl.row + nrows > pl.stride)
        return fail(c, JL_ERR_ARG, "packed: rows %d..%d outside a buffer of %d rows", pl.row, pl.row + nrows, pl.stride);
    if (k % (*ti)->block_elems != 0) return JL_DECLINED;
    if (!pl.qs || !pl.d || (type != JL_TYPE_Q8_0 && !pl.sc)) return fail(c, JL_ERR_ARG, "packed: null plane");
    if (((uintptr_t)pl.qs | (uintptr_t)pl.d | (uintptr_t)pl.sc) & 3) return JL_DECLINED;
    return JL_OK;
}

int packed_matvec_launch(jl_ctx* c, float* out, int type, const PlaneRef& pl, const float* x,
                         const int8_t* q, const float* as, const float* s16, int nrows, int k,
                         hipStream_t st) {
    const TypeInfo* ti = nullptr;
    int rc = packed_check(c, type, pl, nrows, k, &ti);
    if (rc != JL_OK) return rc;
    if (!out) return fail(c, JL_ERR_ARG, "packed matvec: null out");
    if (x && !aligned16(x)) return JL_DECLINED;
    if (!x && (!q || !as || !s16)) return fail(c, JL_ERR_ARG, "packed matvec: no activation");
    if (q && ((uintptr_t)q & 3)) return JL_DECLINED;
    // Rows per wavefront: the widest run that still gives three CUs in four a
    // workgroup (from sweeps: 224 workgroups of 64-row runs beat 448 of 32-row runs).
    int rw = c->tune.packed_rw;
    if (rw <= 0) {
        rw = 64;
        while (rw > 16 && (nrows + rw - 1) / rw < c->num_cu * 3 / 4) rw >>= 1;
    }
    if (rw != 16 && rw != 32 && rw != 64) return fail(c, JL_ERR_ARG, "packed matvec: rw=%d", rw);
    const int nchunks = (k + 255) / 256;
    // sixteen-row runs: eight wavefronts a workgroup, two workgroups a CU (measured against sixteen,
    // us: Q4_K 4096 x 4096 4.87 against 5.06, Q6_K 4096 x 14336 14.46 against 14.69)
    int nw = c->tune.packed_block > 0 ? c->tune.packed_block / 64 : rw == 16 ? 8 : 16;
    if (nw > nchunks) nw = nchunks;
    if (nw < 1 || nw > 16) return fail(c, JL_ERR_ARG, "packed matvec: block=%d", nw * 64);
    PackedMatVecArgs a;
    a.out = out; a.qs = pl.qs; a.d = pl.d; a.sc = pl.sc;
    a.x = x; a.q = q; a.as = as; a.s16 = s16;
    a.nrows = nrows; a.k = k; a.row0 = pl.row; a.stride = pl.stride; a.per = c->act_window / 32;
    a.nwaves = nw; a.ngroups = (nrows + rw - 1) / rw;
    a.x2 = nullptr; a.resid = nullptr; a.alpha = 0.f; a.norm_out = nullptr; a.norm_eps = 0.f; a.inv_k = 0.0;
    Name name;
    name << "jl_matvec_packed_" << (x ? "" : "q8_") << ti->tag << "_w" << rw;
    void* params[] = {&a};
    return launch(c, name, (unsigned)((nrows + rw - 1) / rw), 1, (unsigned)(nw * 64),
                  (unsigned)JL_PK_LDS_BYTES(nw), st, params);
}

// m packed matvecs of one type and shape in one launch (grid.y = matrix): each with its
// own planes and first row, reading x + j * xstride; up gates the activation.
int packed_matvec_multi_launch(jl_ctx* c, int type, int m, float* const* outs, const PlaneRef* pls,
                               const float* x, size_t xstride, const float* up, float* resid, float alpha,
                               const float* resid_gate, const float* norm_w, float norm_eps, float* norm_out,
                               int nrows, int k, hipStream_t st, bool tokens) {
    if (m < 1 || m > JL_MAX_MULTI) return fail(c, JL_ERR_ARG, "packed multi: %d matrices", m);
    // the norm precedes gate and up, the gated activation precedes down: never both
    if (norm_w && (up || !aligned16(norm_w) || (norm_out && !aligned16(norm_out)))) return JL_DECLINED;
    const TypeInfo* ti = nullptr;
    for (int j = 0; j < m; j++) {
        int rc = packed_check(c, type, pls[j], nrows, k, &ti);
        if (rc != JL_OK) return rc;
        if (!outs[j]) return fail(c, JL_ERR_ARG, "packed multi: null out");
        if (pls[j].stride != pls[0].stride) return JL_DECLINED;
    }
    if (!x || !aligned16(x) || (up && !aligned16(up)) || (xstride % 4) != 0) return JL_DECLINED;
    // rows per wavefront: the widest run that still gives three CUs in four a workgroup,
    // counting every matrix's row groups
    int rw = c->tune.packed_rw;
    if (rw <= 0) {
        rw = 64;
        while (rw > 16 && (long)m * ((nrows + rw - 1) / rw) < c->num_cu * 3 / 4) rw >>= 1;
    }
    if (rw != 16 && rw != 32 && rw != 64) return fail(c, JL_ERR_ARG, "packed multi: rw=%d", rw);
    const int nchunks = (k + 255) / 256;
    // eight wavefronts a workgroup, two and more workgroups a CU, unless there is not one a CU to be had: sixteen then
    // (gated block of 4096 / 14336 over planes, us: gate + up on eight, down on sixteen 26.6 where sixteen and eight
    // took 29.1; 2816 / 7936 down on sixteen 14.2 against 14.9)
    int nw = c->tune.packed_block > 0 ? c->tune.packed_block / 64 : (long)m * ((nrows + rw - 1) / rw) <= c->num_cu ? 16 : 8;
    if (nw > nchunks) nw = nchunks;
    if (nw < 1 || nw > 16) return fail(c, JL_ERR_ARG, "packed multi: block=%d", nw * 64);
    PackedMultiArgs a;
    memset(&a, 0, sizeof a);
    for (int j = 0; j < m; j++) {
        a.out[j] = outs[j]; a.qs[j] = pls[j].qs; a.d[j] = pls[j].d; a.sc[j] = pls[j].sc; a.row0[j] = pls[j].row;
    }
    a.x = x; a.x2 = up; a.xstride = xstride; a.resid = resid; a.alpha = alpha;
    a.resid_gate = resid ? resid_gate : nullptr;
    a.norm_w = norm_w; a.norm_eps = norm_eps; a.norm_out = norm_w ? norm_out : nullptr; a.inv_k = 1.0 / k;
    a.nrows = nrows; a.k = k; a.stride = pls[0].stride; a.per = c->act_window / 32;
    a.nwaves = nw; a.ngroups = (nrows + rw - 1) / rw;
    Name name;
    name << "jl_matvec_packed_multi_" << (up ? "act_" : norm_w ? "norm_" : "") << (tokens && type == JL_TYPE_Q4_K ? "q4kf" : ti->tag) << "_w" << rw;
    void* params[] = {&a};
    return launch(c, name, (unsigned)a.ngroups, (unsigned)m, (unsigned)(nw * 64),
                  (unsigned)(JL_PK_LDS_BYTES(nw) + (norm_w ? 16 + JL_NORM_LDS_BYTES : 0)), st, params);
}

// MXFP4 planes (QS and D only): rows row .. row+nrows of a buffer of `stride` rows.
int mx_planes_check(jl_ctx* c, const PlaneRef& pl, int nrows, int k) {
    if (nrows <= 0 || k <= 0 || pl.row < 0 || pl.stride <= 0)
        return fail(c, JL_ERR_ARG, "mxfp4 planes: nrows=%d k=%d row=%d stride=%d", nrows, k, pl.row, pl.stride);
    if ((long)pl.row + nrows > pl.stride)
        return fail(c, JL_ERR_ARG, "mxfp4 planes: rows %d..%d outside a buffer of %d rows", pl.row, pl.row + nrows,
                    pl.stride);
    if (!pl.qs || !pl.d) return fail(c, JL_ERR_ARG, "mxfp4 planes: null plane");
    if (k % 32 != 0 || k / 32 > 65535 || (((uintptr_t)pl.qs | (uintptr_t)pl.d) & 3)) return JL_DECLINED;
    return JL_OK;
}

int unpack_launch(jl_ctx* c, int type, const PlaneRef& pl, int nrows, int k, void* dst, hipStream_t st) {
    UnpackArgs a;
    a.dst = (uint8_t*)dst; a.qs = pl.qs; a.d = pl.d; a.sc = pl.sc;
    a.nrows = nrows; a.k = k; a.row0 = pl.row; a.stride = pl.stride;
    void* params[] = {&a};
    const char* name = type == JL_TYPE_Q4_K ? "jl_unpack_q4k" : type == JL_TYPE_Q6_K ? "jl_unpack_q6k" : type == JL_TYPE_Q8_0 ? "jl_unpack_q8_0" : "jl_unpack_mxfp4";
    return launch(c, name, (unsigned)((nrows + 63) / 64), (unsigned)((k + 255) / 256), 256, 0, st, params);
}

int packed_matmul_launch(jl_ctx* c, float* out, int type, const PlaneRef& pl, const float* x, int nrows,
                         int k, int ntok, hipStream_t st) {
    const TypeInfo* ti = nullptr;
    int rc = packed_check(c, type, pl, nrows, k, &ti);
    if (rc != JL_OK) return rc;
    if (!out || !x || ntok <= 0) return fail(c, JL_ERR_ARG, "packed matmul: bad operand");
    if (!aligned16(x) || (k % 4) != 0) return JL_DECLINED;
    if (tokens_matvec_wanted(c, type, true, nrows, k, ntok, pl.stride)) {
        rc = tokens_matvec_launch(c, out, type, nullptr, &pl, x, nrows, k, ntok, st);
        if (rc != JL_DECLINED) return rc;
    }
    if (few_applies(c, type, true, nrows, k, ntok, pl.stride)) {
        FewCall f;
        f.type = type; f.nrows = nrows; f.k = k; f.ncols = ntok; f.pl[0] = &pl; f.x = x; f.out[0] = out;
        rc = few_launch(c, f, st);
        if (rc != JL_DECLINED) return rc;
    }
    // the matrix-core forms read GGUF rows: the planes are turned back into rows in a workspace
    const bool gemm = type == JL_TYPE_Q4_K && c->act_window == 256 && ntok >= c->gemm_min_tok &&
                      ntok <= 65535 * 4 && kGemmLdsBytes <= c->lds_limit && k / 256 <= 65535;
    const bool i8 = ntok >= c->gemm_min_tok && c->tune.gemm_form != 9 && gemm_i8_applies(c, type, nrows, k, ntok);
    // Q4_K with the k-quant window: the tiled forms read the planes where they lie; only the
    // few-token forms, which take a lane's operand words straight from GGUF rows, restore rows first
    if (gemm && c->tune.gemm_planes != 2 && !gemm_q4k_few_applies(c, nrows, k, ntok) && (size_t)pl.stride * 4 < ((size_t)1 << 31))
        return gemm_q4k_launch(c, out, nullptr, x, nrows, k, ntok, st, &pl);
    if (gemm || i8) {
        rc = ws_ensure(c, &c->unpack_ws, &c->unpack_ws_bytes, (size_t)nrows * (size_t)(k / ti->block_elems) * ti->block_bytes);
        if (rc != JL_OK) return rc;
        rc = unpack_launch(c, type, pl, nrows, k, c->unpack_ws, st);
        if (rc != JL_OK) return rc;
        return gemm ? gemm_q4k_launch(c, out, c->unpack_ws, x, nrows, k, ntok, st)
                    : gemm_i8_launch(c, out, type, c->unpack_ws, x, nrows, k, ntok, st);
    }
    for (int t = 0; t < ntok; t++) {
        rc = packed_matvec_launch(c, out + (size_t)t * nrows, type, pl, x + (size_t)t * k, nullptr, nullptr,
                                  nullptr, nrows, k, st);
        if (rc != JL_OK) return rc;
    }
    return JL_OK;
}

// The int8 tile placed per expert: work list, columns quantized and laid out group by group, tiles.
int moe_gemm_i8_launch(jl_ctx* c, float* out0, float* out1, int type, const void* bank0, const void* bank1, const float* x,
                       const float* x2, const uint32_t* src, const uint32_t* start, int n_expert, int ncols, int nrows, int k,
                       I8Shape f, hipStream_t st, const MoeLists* lists) {
    const TypeInfo* ti = type_info(type);
    const bool q4 = type == JL_TYPE_Q4_K;
    const int nslots = ncols / 32 + n_expert + 1, nstage = k / 128, tile = 32 * f.tw;
    const long tiles_max = ncols / tile + n_expert;
    if (nslots > 65535 || n_expert > 65535) return JL_DECLINED;
    const int row_bytes = (k / ti->block_elems) * ti->block_bytes, nmat = bank1 ? 2 : 1, tr = 32 * f.rt * (4 / f.tw);
    const long work = tiles_max * ((nrows + tr - 1) / tr) * nmat;
    if (work >= (1L << 31)) return JL_DECLINED;
    const size_t bq_bytes = (size_t)nstage * nslots * 4096, da_bytes = (size_t)(k / 32) * nslots * 128;
    const size_t o_wl = bq_bytes + (q4 ? 2 : 1) * da_bytes;
    int rc = ws_ensure(c, &c->moe_q_ws, &c->moe_q_ws_bytes, o_wl + (size_t)(4 + nslots + tiles_max) * 4);
    if (rc != JL_OK) return rc;
    char* ws = (char*)c->moe_q_ws;
    MoeWorklistArgs wa;
    wa.start = start; wa.wl = (uint32_t*)(ws + o_wl); wa.n_expert = n_expert; wa.nslots = nslots;
    wa.tile_log2 = f.tw == 4 ? 7 : 6;
    void* wp[] = {&wa};
    if (lists && lists->nslots == nslots) wa.wl = lists->wl[wa.tile_log2 - 6];   // (made by the grouping)
    else if ((rc = launch(c, "jl_moe_worklist", 1, 1, 1024, 0, st, wp)) != JL_OK) return rc;
    MoeGemmPrepArgs pa;
    pa.x = x; pa.x2 = x2; pa.src = src; pa.start = start; pa.wl = wa.wl;
    pa.bq = (uint16_t*)ws; pa.da = (float*)(ws + bq_bytes); pa.k = k; pa.nslots = nslots; pa.per = c->act_window / 32;
    if (q4) pa.dsum = (float*)(ws + bq_bytes + da_bytes);
    void* pp[] = {&pa};
    rc = launch(c, "jl_moe_gemm_i8_prep", (unsigned)((k + 255) / 256), (unsigned)nslots, 1024, 0, st, pp);
    if (rc != JL_OK) return rc;
    MoeGemmArgs ga;
    ga.out[0] = out0; ga.out[1] = out1;
    ga.bank[0] = (const uint8_t*)bank0; ga.bank[1] = (const uint8_t*)bank1;
    ga.bq = pa.bq; ga.da = pa.da; ga.dsum = pa.dsum; ga.start = start; ga.wl = wa.wl;
    ga.sheet_bytes = (size_t)nrows * row_bytes; ga.nrows = nrows; ga.k = k; ga.row_bytes = row_bytes;
    ga.nslots = nslots; ga.nmat = nmat;
    void* gp[] = {&ga};
    const long cap = f.rt == 4 || type != JL_TYPE_Q8_0 ? 2 : 3;
    return launch(c, gemm_i8_name("jl_moe_gemm", c, type, f), (unsigned)std::min(work, cap * c->num_cu), 1, 256, gemm_i8_lds(c, type, f), st, gp);
}

// Blocks of rows an expert's matrix is cut into by the groups-of-columns kernels ("moe.form" = 3): one workgroup of eight
// wavefronts a CU (the same age on every SIMD, tiles handed out as they get to them: two younger workgroups of four
// measured 4 % slower).  An expert is worked on by XCD e % 8 alone, so the grid runs in rounds of that XCD's CUs, a round
// taking its fill of LDS and the tiles a wavefront has: the split that is estimated least, the fewest blocks among equals.
// Fitted to 19 shapes (8 to 128 experts of 512 x 1024 to 2304 x 768) at 2, 4, 6 and 8 columns an expert and every number of
// blocks, 9 % each; the pick is 0.6 % behind the best on average, at most 19 (rounds of all CUs without the fill, the rule
// before: 5.7, at most 64: 46 x 1536 x 1024 twice, eight columns, twelve blocks 41 us, two 25.4).  "moe.waves" = 4: the
// two-workgroup form.
int moe_g16_blocks(const jl_ctx* c, int nrows, int k, int n_expert, int ncols, int nmat, int nwaves) {
    const int tiles = (nrows + 15) / 16, sets = (tiles + nwaves - 1) / nwaves;
    if (c->tune.moe_shares > 0) return std::min(c->tune.moe_shares, sets);
    // (experts that can have a column: at most one a column)
    const long slots = std::max(1, c->num_cu / 8) * (nwaves == 4 ? 2L : 1L), n_xcd = (std::min<long>(n_expert, ncols) + 7) / 8;
    const double nsb = k / 256, fill = 1.62 + (0.22 + 0.074 * std::min(16.0, (double)ncols / n_expert)) * nsb, tile = 0.19 + 0.6 * nsb;
    int best = 1;
    double best_cost = 1e30;
    for (int nb = 1; nb <= sets && nb <= 64; nb++) {
        const long tiles_wg = (tiles + nb - 1) / nb, blocks = (tiles + tiles_wg - 1) / tiles_wg;
        const long per_wave = (tiles_wg + nwaves - 1) / nwaves, rounds = (blocks * nmat * n_xcd + slots - 1) / slots;
        const double cost = rounds * (fill + per_wave * tile);
        if (cost < best_cost) { best_cost = cost; best = nb; }
    }
    return best;
}

// Banks with the k-quant window, more than eight columns an expert on average: whether the int8 few-token kernel takes less
// time than the columns against decoded rows (kernels/moe_cols.h), us by what each has to do (millions of the banks'
// elements, a pass of the columns a time; super-blocks of a row, the chain of a small grid), fitted to 38 (Q4_K) and 19
// (Q6_K) shapes, 8 to 128 experts of 512 x 1024 to 2816 x 1024 at 3 to 64 columns.  Chosen so, a launch takes 0.5 % (Q4_K)
// and 1.3 % (Q6_K) more than the best of every form on average from twelve columns on, at most 24 (8 x 512 x 1024, 32
// columns 13.3 us against 10.7) and 46 %; always the columns 1.9 %, always the few-token kernel 49, groups of 32 41 %.
bool moe_few_faster(int type, int n_expert, int ncols, int nmat, int nrows, int k) {
    const double avg = (double)ncols / n_expert, nsb = k / 256, melem = 1e-6 * n_expert * nmat * (double)nrows * k;
    const auto over = [&](int n) { return 0.5 * std::erfc((n + 0.5 - avg) / std::sqrt(2 * avg)); };   // an expert's columns pass n
    const int nt = avg <= 16 ? 1 : avg <= 32 ? 2 : 4;   // (few_shape takes fewer where those are faster than four)
    const double passes = melem * (1 + over(16 * nt));
    if (type == JL_TYPE_Q4_K) {
        if (avg >= 32) return false;
        const double few = 5.3 + 1.15 * (0.5 + 0.95e-6 * ncols * k + passes * (nt == 1 ? 0.157 : 0.241));
        return few < std::max(7 + 1.1 * nsb, 5.5 + 0.155 * melem) * (1 + 0.3 * over(32));
    }
    return 6.0 + passes * (nt == 1 ? 0.267 : nt == 2 ? 0.377 : 0.76) < 8.6 + 0.81 * nsb + melem * (0.247 + 0.113 * over(32) + 0.475 * over(64));
}

// What a grouped matmul asks of its one or two banks of n_expert sheets of nrows x k, whichever kernel serves them
// and whether or not anything is grouped: GGUF rows (bank0, bank1) or packed planes (pb0, pb1).  `two` says that the
// call has a second output.  Reads nothing of the device, so it can go in front of everything else.
int moe_banks_check(jl_ctx* c, int type, bool planes, const void* bank0, const void* bank1, const jl_packed_bank* pb0,
                    const jl_packed_bank* pb1, bool two, int n_expert, int nrows, int k) {
    const TypeInfo* ti = type_info(type);
    if (!ti) return JL_DECLINED;
    if (nrows <= 0 || k <= 0 || n_expert <= 0) return fail(c, JL_ERR_ARG, "moe matvec: %d experts of %d x %d", n_expert, nrows, k);
    if ((planes ? pb1 != nullptr : bank1 != nullptr) != two) return fail(c, JL_ERR_ARG, "moe matvec: second matrix needs both bank and out");
    if (planes) {
        if (!pb0) return fail(c, JL_ERR_ARG, "moe matvec: null bank");
        for (const jl_packed_bank* b : {pb0, pb1}) {
            if (!b) continue;
            if (!b->qs || !b->d || !b->sc || b->stride <= 0) return fail(c, JL_ERR_ARG, "moe matvec: null plane");
            if ((((uintptr_t)b->qs | (uintptr_t)b->d | (uintptr_t)b->sc) & 3) || (b->sheet_bytes & 3)) return JL_DECLINED;
            // an expert's rows must lie inside a plane set: its own sheet, or its range of the bank's
            if (b->sheet_bytes ? b->stride < nrows : (long)b->stride < (long)n_expert * nrows)
                return fail(c, JL_ERR_ARG, "moe matvec: plane sets of %d rows do not hold %d experts x %d rows", b->stride,
                            n_expert, nrows);
            if (b->sheet_bytes != pb0->sheet_bytes || b->stride != pb0->stride) return JL_DECLINED;   // one layout a launch
        }
        // plane sheets are served in Q4_K with the k-quant window
        if (type != JL_TYPE_Q4_K || c->act_window != 256) return JL_DECLINED;
        if ((size_t)pb0->stride * 4 >= ((size_t)1 << 31)) return JL_DECLINED;
    } else {
        if (!bank0) return fail(c, JL_ERR_ARG, "moe matvec: null bank");
        if (!aligned16(bank0) || (bank1 && !aligned16(bank1))) return JL_DECLINED;
    }
    if (k % 256 != 0 || n_expert > 65535) return JL_DECLINED;
    const size_t sheet = (size_t)nrows * (size_t)(k / ti->block_elems) * ti->block_bytes;
    return (type == JL_TYPE_Q4_K ? sheet % 16 : sheet % 2) != 0 ? JL_DECLINED : JL_OK;
}

// Lanes a row for the gather kernels: of 64, 32 and 16 (8: rows of eight slots at most) the width that leaves the fewest without a slot while every CU still gets
// a workgroup.
// Whole block, us, 64 -> 32 / 16 lanes for gate + up: Q4_K, 32 slots a row (K 2048), 8 / 32 / 96 pairs of 128 experts 22.6 -> 21.8 /
// 20.8, 36.6 -> 31.2 / 31.7, 95.7 -> 76.4 / 77.3; 44 slots (three of sixteen lanes), 16 / 60 pairs of 60 43.5 -> 42.6 / 40.1, 116 ->
// 114 / 103; too few workgroups, 2 pairs of 24 experts of 1280 rows, 40 slots, 18.2 -> 19.4 / 19.7.  Q8_0 gains only while a lane
// has one slot: 28 slots 70 -> 66 / 67, 44 slots 59.7 -> 63.4 / 63.6.
int gather_lanes(const jl_ctx* c, int type, int nslots, int nrows, long matvecs) {
    int best = 64;
    double most = nslots / (64.0 * ((nslots + 63) / 64));
    for (int lanes = 32; lanes >= (nslots <= 8 ? 8 : 16); lanes /= 2) {
        const double used = nslots / ((double)lanes * ((nslots + lanes - 1) / lanes));
        const int rows = 16 * (64 / lanes);
        if (used > most && (type != JL_TYPE_Q8_0 || nslots <= lanes) && (nrows + rows - 1) / rows * matvecs >= c->num_cu) best = lanes, most = used;
    }
    return best;
}

// A decode matvec a routed column (kernels/moe.h: moe_gather_body), GGUF banks.  start null: column c is pair c of sel.
int moe_gather_launch(jl_ctx* c, float* out0, float* out1, int type, const void* bank0, const void* bank1, const float* x, const float* x2,
                      const uint32_t* src, const uint32_t* start, const uint32_t* sel, int sel_stride, int k_used, int n_expert, int ncols,
                      int nrows, int k, hipStream_t st) {
    const TypeInfo* ti = type_info(type);
    MoeGatherArgs a;
    a.out[0] = out0; a.out[1] = out1; a.bank[0] = (const uint8_t*)bank0; a.bank[1] = (const uint8_t*)bank1;
    a.x = x; a.x2 = x2; a.src = src; a.start = start; a.sel = sel; a.sel_stride = sel_stride; a.k_used = k_used; a.n_expert = n_expert;
    a.nrows = nrows; a.k = k; a.row_bytes = (k / ti->block_elems) * ti->block_bytes; a.per = c->act_window / 32;
    a.sheet_bytes = (size_t)nrows * a.row_bytes;
    const int nmat = bank1 ? 2 : 1;
    const bool pair = q8_pair_form(c, type, bank0, k) && (!bank1 || q8_pair_form(c, type, bank1, k)) && a.sheet_bytes % 4 == 0;
    const size_t lds = act_lds_bytes(k) + (pair ? (size_t)k + 16 : 0) + 16;
    if (lds > c->lds_limit || ncols > 65535) return JL_DECLINED;
    // one round of workgroups, as the grouped matvecs (two a CU for the paired Q8_0 form)
    a.nwaves = 16;
    const int lpr = gather_lanes(c, type, k / (type == JL_TYPE_Q8_0 && !pair ? 32 : 64), nrows, (long)ncols * nmat), per_group = 16 * (64 / lpr);
    const long slots = (pair ? 2L : 1L) * c->num_cu, groups = (nrows + per_group - 1) / per_group;
    a.ngroups = (int)std::max(1L, std::min(groups, slots / ((long)ncols * nmat)));
    if (!start && !sel && a.ngroups > 8) a.ngroups &= ~7;   // (one matrix: a row group's workgroups on one XCD)
    Name name;
    name << "jl_moe_gather_" << (pair ? "q8_0p" : q6_tag(c, type)) << (x2 ? "_a" : "") << "_l" << lpr;
    void* params[] = {&a};
    return launch(c, name, (unsigned)a.ngroups, (unsigned)ncols, 1024, (unsigned)lds, st, params, (unsigned)nmat);
}

// Whether a block's pairs go without grouping (moe_gather_ffn).  That saves two launches and the grouped kernels' setup, and reads a
// sheet again for every pair that shares its expert with another, but faster (from L2 and the memory-side cache where it is read
// again) than the grouped kernels, which make 5 TB/s of a few columns a sheet, over planes 7 and a longer setup; the rows' choices
// are taken as evenly spread.  Fitted to 862 (Q4_K, k-quant window), 450 (planes) and 1724 (the others) blocks, 2 to 128 experts of
// 768 x 2048 to 14336 x 4096 at 1 to 32 rows: 0.7, 2.4 and 0.6 % behind the better of the two, at most 9, 4 and 11 % slower than
// grouped.  (One line for all, 6.5 and 3.65 TB/s and 13 us: 16 experts top-4 of 14336 x 4096, six rows 273 -> 349 us, planes of
// 4096 x 4096 221 -> 267 at 64 experts and sixteen.)  The whole block, grouped -> so, us, at pairs: Q4_K 128 experts top-8 of 768 x 2048 with Q6_K down 35 -> 22 (8), 56 -> 30
// (32), 97 -> 79 (96), 122 -> 118 (192), 134 -> 163 (320: grouped); 60 top-4 of 1792 x 2816 33 -> 25 (4), 127 -> 98 (60), 142 -> 146
// (92), 138 -> 162 (120: grouped); 8 top-2 of 2048 x 2816 28 -> 20 (2), 50 -> 36 (16), 49 -> 51 (24: grouped); 32 top-4 of 1024 x
// 2048 47 -> 31 (32), 49 -> 44 (64), 49 -> 58 (80: grouped).  Q8_0 60 top-4 of 1792 x 2816 36 -> 27 (4), 174 -> 159 (60), 221 -> 250 (92:
// grouped); 32 top-4 of 1024 x 2048, Q6_K down, 57 -> 41 (32), 80 -> 66 (64), 84 -> 99 (96: grouped).
// Over planes (Q4_K) 128 top-8 of 768 x 2048 36 -> 21 (8), 63 -> 44 (64), 83 -> 68 (128), 108 -> 108 (256: grouped); 60 top-4 of 1792 x
// 2816 39 -> 24 (4), 108 -> 100 (64), 143 -> 171 (128: grouped); 8 top-2 of 1024 x 1536 30 -> 16 (2), 42 -> 29 (32).
// Q4_K and Q6_K rows of sheets under 512 x 512 keep the grouped form, whose launches a caller can count on there
// (tests/test_gpu_moe.py), though they would gain as well.
bool moe_gather_ffn_wanted(const jl_ctx* c, int type, int down_type, bool planes, int rows, int k_used, int n_expert, int n_ffn, int n_embd) {
    const double pairs = (double)rows * k_used, sheet = (double)n_ffn * n_embd;
    if (pairs > 256 || (!planes && type != JL_TYPE_Q8_0 && sheet < 512.0 * 512.0)) return false;
    const TypeInfo *t = type_info(type), *d = type_info(down_type);
    const double mb = sheet * 1e-6 * (2.0 * t->block_bytes / t->block_elems + (double)d->block_bytes / d->block_elems);
    const double touched = n_expert * (1.0 - std::pow(1.0 - std::min(1.0, (double)k_used / n_expert), rows));
    struct { double again, grouped, setup; } q = {8, 5.6, 14};
    if (planes) q = {7.5, 7, 20};
    else if (type == JL_TYPE_Q4_K && c->act_window == 256) q = {6.5, 5, 18};
    return pairs * mb / q.again < q.setup + touched * mb / q.grouped;
}

// A routed block of a handful of pairs without its grouping and combine: the pairs themselves are the columns of gate + up,
// and the down projections of a row's pairs are one matvec that adds into the residual stream.  JL_DECLINED (nothing
// enqueued) where the activations of a row do not fit LDS.
int moe_gather_ffn(jl_ctx* c, float* resid, int type, int down_type, const void* gate, const void* up, const void* down, const float* x,
                   const uint32_t* sel, int sel_stride, const float* wt, int rows, int k_used, int n_expert, int n_ffn, int n_embd,
                   float* g, float* u, hipStream_t st) {
    const TypeInfo* ti = type_info(down_type);
    MoeGatherDownArgs a;
    a.resid = resid; a.bank = (const uint8_t*)down; a.g = g; a.u = u; a.sel = sel; a.wt = wt;
    a.nrows = n_embd; a.k = n_ffn; a.row_bytes = (n_ffn / ti->block_elems) * ti->block_bytes; a.per = c->act_window / 32;
    a.sheet_bytes = (size_t)n_embd * a.row_bytes;
    a.n_expert = n_expert; a.sel_stride = sel_stride; a.k_used = k_used;
    const long kk = (long)k_used * n_ffn;
    if (kk > 65536 || act_lds_bytes((int)kk) + 256 > c->lds_limit || act_lds_bytes(n_embd) + 256 > c->lds_limit) return JL_DECLINED;
    const bool pair = q8_pair_form(c, down_type, down, (int)kk) && n_ffn % 64 == 0 && a.row_bytes % 4 == 0 &&
                      act_lds_bytes((int)kk) + (size_t)kk + 256 <= c->lds_limit;
    const size_t lds = act_lds_bytes((int)kk) + (pair ? (size_t)kk + 16 : 0) + 16 + 128;
    const uint32_t row_slots = (uint32_t)(n_ffn / (down_type == JL_TYPE_Q8_0 && !pair ? 32 : 64));
    a.slots_inv = 0xFFFFFFFFu / row_slots + 1u;
    int rc = moe_gather_launch(c, g, u, type, gate, up, x, nullptr, nullptr, nullptr, sel, sel_stride, k_used, n_expert, rows * k_used,
                               n_ffn, n_embd, st);
    if (rc != JL_OK) return rc;
    // (eight and four wavefronts a workgroup: the same at one row, 2 and 9 us slower at 32 pairs)
    a.nwaves = 16;
    const int lpr = gather_lanes(c, down_type, (int)row_slots * k_used, n_embd, rows), per_group = 16 * (64 / lpr);
    const long slots = (pair ? 2L : 1L) * c->num_cu, groups = (n_embd + per_group - 1) / per_group;
    a.ngroups = (int)std::max(1L, std::min(groups, slots / rows));
    if (!sel && a.ngroups > 8) a.ngroups &= ~7;
    Name name;
    name << "jl_moe_gather_" << (pair ? "q8_0p" : q6_tag(c, down_type)) << "_down_l" << lpr;
    void* params[] = {&a};
    return launch(c, name, (unsigned)a.ngroups, (unsigned)rows, 1024, (unsigned)lds, st, params);
}

// The same over packed planes.  Rows a workgroup and its wavefronts as the packed matvecs have them (other widths and eight against
// sixteen wavefronts: within 4 % at 8 to 128 pairs, sixteen-row runs from 32 pairs up to 40 % slower).
int moe_planes_gather_ffn(jl_ctx* c, float* resid, const jl_packed_bank* pg, const jl_packed_bank* pu, const jl_packed_bank* pd, const float* x,
                          const uint32_t* sel, int sel_stride, const float* wt, int rows, int k_used, int n_expert, int n_ffn, int n_embd,
                          float* g, float* u, hipStream_t st) {
    if (k_used > 16 || (long)rows * k_used > 65535 || (long)k_used * n_ffn > (1L << 24)) return JL_DECLINED;
    auto width = [&](int nrows, long matvecs) {   // rows a workgroup: the widest run that still gives three CUs in four a workgroup
        int rw = c->tune.packed_rw;
        if (rw != 16 && rw != 32 && rw != 64)
            for (rw = 64; rw > 16 && matvecs * ((nrows + rw - 1) / rw) < c->num_cu * 3 / 4;) rw >>= 1;
        return rw;
    };
    auto waves = [&](long groups, int nchunks) { return std::min(nchunks, c->tune.packed_block > 0 ? c->tune.packed_block / 64 : groups <= c->num_cu ? 16 : 8); };
    MoePlanesGatherArgs a;
    a.out[0] = g; a.out[1] = u;
    a.qs[0] = pg->qs; a.d[0] = pg->d; a.sc[0] = pg->sc; a.qs[1] = pu->qs; a.d[1] = pu->d; a.sc[1] = pu->sc;
    a.x = x; a.sel = sel; a.sheet_words = pg->sheet_bytes / 4; a.row_step = pg->sheet_bytes ? 0 : n_ffn; a.stride = pg->stride;
    a.nrows = n_ffn; a.k = n_embd; a.per = c->act_window / 32; a.n_expert = n_expert; a.sel_stride = sel_stride; a.k_used = k_used;
    const int pairs = rows * k_used, rw = width(n_ffn, 2L * pairs);
    a.ngroups = (n_ffn + rw - 1) / rw;
    a.nwaves = waves(2L * pairs * a.ngroups, n_embd / 256);
    Name name;
    name << "jl_moe_planes_gather_w" << rw;
    void* params[] = {&a};
    int rc = launch(c, name, (unsigned)a.ngroups, (unsigned)pairs, 64u * a.nwaves, (unsigned)JL_PK_LDS_BYTES(a.nwaves), st, params, 2);
    if (rc != JL_OK) return rc;
    MoePlanesDownArgs b;
    b.resid = resid; b.qs = pd->qs; b.d = pd->d; b.sc = pd->sc; b.g = g; b.u = u; b.sel = sel; b.wt = wt;
    b.sheet_words = pd->sheet_bytes / 4; b.row_step = pd->sheet_bytes ? 0 : n_embd; b.stride = pd->stride;
    b.nrows = n_embd; b.k = n_ffn; b.per = c->act_window / 32; b.n_expert = n_expert; b.sel_stride = sel_stride; b.k_used = k_used;
    const int dw = width(n_embd, rows);
    b.ngroups = (n_embd + dw - 1) / dw;
    b.nwaves = waves((long)rows * b.ngroups, k_used * (n_ffn / 256));
    Name dname;
    dname << "jl_moe_planes_down_w" << dw;
    void* dparams[] = {&b};
    return launch(c, dname, (unsigned)b.ngroups, (unsigned)rows, 64u * b.nwaves, (unsigned)JL_PK_LDS_BYTES(b.nwaves), st, dparams);
}

// The columns of an expert against rows decoded in registers (kernels/moe_cols.h): the source rows quantized once each
// (nsrc of them, src naming each column's; nsrc = 0: not known, a record a column), then the matrices.
int moe_cols_launch(jl_ctx* c, float* out0, float* out1, int type, const void* bank0, const void* bank1, const jl_packed_bank* pb0,
                    const jl_packed_bank* pb1, const float* x, const float* x2, const uint32_t* src, const uint32_t* start, int n_expert,
                    int ncols, int nrows, int k, int nsrc, hipStream_t st) {
    const TypeInfo* ti = type_info(type);
    const bool q6 = type == JL_TYPE_Q6_K, planes = pb0 != nullptr, mapped = src && nsrc > 0 && nsrc <= ncols;
    const size_t nsb = (size_t)k / 256, nrec = mapped ? nsrc : ncols, rec = JL_MC_REC(q6);
    const int nmat = (planes ? pb1 != nullptr : bank1 != nullptr) ? 2 : 1;
    const unsigned lds = q6 ? JL_MC_Q6_LDS : planes ? JL_MC_PLANES_LDS : JL_MC_Q4_LDS;
    // (32-bit offsets in the kernels: records, and half a super-block's words of every row of the planes)
    if (nrec * nsb * rec >= ((size_t)1 << 32) || (planes && (size_t)pb0->stride >= ((size_t)1 << 25)) || lds > c->lds_limit) return JL_DECLINED;
    const double avg = (double)ncols / n_expert;
    const long rblocks = (nrows + 127) / 128, shares = avg <= 48 ? 1 : (long)(avg * 1.2 / 64) + 1, items = rblocks * shares * nmat * n_expert;
    if (items >= (1L << 30)) return JL_DECLINED;
    const size_t o_aug = nrec * nsb * rec, o_da = o_aug + (q6 ? 0 : nrec * nsb * 32);
    int rc = ws_ensure(c, &c->moe_q_ws, &c->moe_q_ws_bytes, o_da + nrec * nsb * 4);
    if (rc != JL_OK) return rc;
    char* ws = (char*)c->moe_q_ws;
    const char* tag = q6 ? "q6k" : planes ? "q4k_planes" : "q4k";
    MoeColsPrepArgs pa;
    pa.x = x; pa.x2 = x2; pa.src = mapped ? nullptr : src; pa.rec = (uint32_t*)ws; pa.aug = (uint32_t*)(ws + o_aug); pa.da = (float*)(ws + o_da);
    pa.k = k; pa.nrec = (int)nrec;
    void* pp[] = {&pa};
    Name name;
    name << "jl_moe_cols_prep_" << tag;
    rc = launch(c, name, (unsigned)((nrec * nsb + 15) / 16), 1, 256, 0, st, pp);
    if (rc != JL_OK) return rc;
    MoeColsArgs ga;
    ga.out[0] = out0; ga.out[1] = out1;
    ga.bank[0] = (const uint8_t*)bank0; ga.bank[1] = (const uint8_t*)bank1;
    if (planes) {
        const jl_packed_bank* pbs[2] = {pb0, pb1};
        for (int m = 0; m < nmat; m++) { ga.pqs[m] = pbs[m]->qs; ga.pd[m] = pbs[m]->d; ga.psc[m] = pbs[m]->sc; }
        ga.sheet_words = pb0->sheet_bytes / 4;
        ga.row_step = pb0->sheet_bytes ? 0 : nrows;
        ga.pstride = pb0->stride;
    }
    ga.rec = (const uint8_t*)ws; ga.aug = (const uint8_t*)ws + o_aug; ga.da = pa.da; ga.map = mapped ? src : nullptr; ga.start = start;
    ga.nrows = nrows; ga.k = k; ga.row_bytes = (k / ti->block_elems) * ti->block_bytes; ga.sheet_bytes = (size_t)nrows * ga.row_bytes;
    ga.nmat = nmat; ga.rblocks = (int)rblocks; ga.shares = (int)shares; ga.items = (int)items;
    void* gp[] = {&ga};
    Name gname;
    gname << "jl_moe_cols_" << tag;
    return launch(c, gname, (unsigned)((items + 7) / 8 * 8), 1, 256, lds, st, gp);
}

// pb0 / pb1: the banks as packed planes (bank0 / bank1 unused then): the per-expert kernels
// read an expert's sheet where it lies in the bank's pages.
int moe_matvec_launch(jl_ctx* c, float* out0, float* out1, int type, const void* bank0, const void* bank1,
                      const float* x, const float* x2, const uint32_t* src, const uint32_t* start,
                      int n_expert, int ncols, int nrows, int k, hipStream_t st, const jl_packed_bank* pb0,
                      const jl_packed_bank* pb1, int nsrc, const MoeLists* lists) {
    const TypeInfo* ti = nullptr;
    int rc = matvec_check(c, type, nrows, k, &ti);
    if (rc != JL_OK) return rc;
    const bool planes = pb0 != nullptr;
    if (!out0 || !x || !start || ncols <= 0) return fail(c, JL_ERR_ARG, "moe matvec: bad operand");
    rc = moe_banks_check(c, type, planes, bank0, bank1, pb0, pb1, out1 != nullptr, n_expert, nrows, k);
    if (rc != JL_OK) return rc;
    if (!aligned16(x) || (x2 && !aligned16(x2)) || ncols > 65535) return JL_DECLINED;
    const int row_bytes = (k / ti->block_elems) * ti->block_bytes;
    const size_t sheet = (size_t)nrows * row_bytes;
    // The int8 forms, by columns an expert on average (us of one matrix of 128 experts x 2048 x 768 / 32 x 2048 x 1024 /
    // 16 x 1024 x 2048, what they replace -> them; "moe.form" = 5 forces the few-token kernel, 6, 7, 8 the tiles of 128
    // columns x 64 rows, 64 x 128 (Q6_K, window 32: else as 6) and, Q8_0, 128 x 128):
    //   Q8_0 window 32    1: 39/16/13 -> 36/15/12   8: 90/29/25 -> 53/21/14   32: 235/71/69 -> 92/30/20   128: 853/238/236 -> 170/56/41
    //   Q6_K window 32    1: 32/16/15 -> 39/16/12   8: 98/40/31 -> 62/22/15   32: 308/110/89 -> 114/37/25   128: 1065/403/304 -> 254/86/60
    //   Q6_K window 256   2: 48/20/18 -> 47/19/14   8: 67/27/30 -> 59/21/15   48: 179/47/48 -> 111/38/28    128: 238/81/56 -> 183/61/43
    // The few-token kernel reads an expert's sheet once for 16 to 64 columns (few_shape) and the columns once for every row tile, so it
    // gives way to the tiles where the columns are the more; a tile of 64 columns needs two workgroups a CU.  From 40 columns on
    // (52 for Q6_K's rows of up to 1024), window 32, Q8_0 takes tiles of 128 columns, Q6_K of 64, Q4_K from 56 on 128.  us, few-token kernel /
    // tiles: Q8_0 60 x 1280 x 2048 twice, 40 columns 127 / 140, 46 156 / 141, 60 x 2048 x 1280, 42 columns 101 / 82; Q6_K 60 x 2048 x 1280, 46 columns
    // 150 / 102; K up to 1024, 48 / 53 columns: 128 x 2048 x 768 135 / 126, 140 / 133, 128 x 2880 x 768 193 / 182, 199 / 184, 60 x 1536 x 1024 twice
    // 127 / 122, 129 / 131, 128 x 1024 x 1024 94 / 90, 99 / 104, 32 x 2048 x 768 38 / 37, 40 / 49, 128 x 2048 x 512 95 / 100, 100 / 104, 60 x 2048 x 512 46 /
    // 50, 47 / 56.  Tiles of 64 columns were Q8_0's and Q4_K's too: blocks of 128 experts of 768 x 2048, 54 columns 348 (321 on 128) and, spilling,
    // 1912 (few-token kernel 410).  (The tiles would be faster earlier in places, for long rows and in the largest Q6_K banks; their one chain of
    // sums rounds more than the few-token kernel's.)  With a
    // column or two an expert Q6_K's dot-product kernel is as fast while rows are short.  Q4_K with the k-quant window
    // has the forms below, and the few-token kernel where moe_few_faster finds it faster.
    {
        const bool q4w = type == JL_TYPE_Q4_K && c->act_window == 256, q6 = type == JL_TYPE_Q6_K;
        const int nmat = (planes ? pb1 != nullptr : bank1 != nullptr) ? 2 : 1;
        const double avg = (double)ncols / n_expert;
        const long tiles64 = (long)n_expert * nmat * ((nrows + 127) / 128);   // workgroups of a tile of 64 columns an expert
        const bool align = sheet % (type == JL_TYPE_Q4_K ? 16 : 4) == 0;
        int form = c->tune.moe_form;
        if (q6 && !planes && c->act_window == 256 && (form == 3 || form == 4)) form += 2;   // (their Q6_K forms)
        // A handful of columns: a decode matvec each (the whole block's us with both of its matvecs, as it was -> so, at 64 lanes a row).  Q4_K, 128 experts of 768 x 2048,
        // 8 / 16 / 24 columns 42 -> 33 / 44 -> 40 / 46 -> 49, 60 of 1792 x 2816, 4 / 16 / 32 / 48 columns 53 -> 32 / 71 -> 52 /
        // 94 -> 86 / 114 -> 127, 8 of 1024 x 1536, 2 / 16 / 24 columns 31 -> 22 / 38 -> 38 / 39 -> 47; Q6_K down projections the
        // same; Q8_0, whose other form costs an expert more: the first 8 / 64 / 96 columns 52 -> 34 / 109 -> 96 / 128 -> 138,
        // the second 57 -> 34 at 4, 191 -> 177 at 64, 8 x 1024 x 1536 at 24 columns 41 -> 43.  Q4_K and Q6_K sheets under 512 x 512
        // keep the grouped form, whose launches a caller can count on there (tests/test_gpu_moe.py), though they would gain as
        // well: 8 experts of 256 x 512, 12 columns 28.7 against 21.9.
        // It reads a sheet again for every column that shares it, which shows where sheets are large: at 6 TB/s, against the
        // few-token kernel's 4 for the sheets that have a column (taken as evenly spread) and 5 us of prep.  us, that kernel / so:
        // Q6_K 4096 x 14336, 2 experts, 6 / 16 columns 32 / 58, 33 / 92, 4 experts 16 columns 56 / 103.  Q4_K with the k-quant window
        // has a slower one: 14336 x 4096 twice, 4 experts, 8 / 12 columns 92 / 70, 93 / 113; one matrix the same on average.  (512
        // and 256 launches, 2 to 16 experts of 1024 x 2048 to 14336 x 4096, 2 to 32 columns: 1.3 and 1.9 % behind the better of
        // the two; by the columns alone 7.5 and 2.4.)
        const double mb = 1e-6 * nmat * sheet, reads = mb * ncols;
        const bool shared = q4w ? ncols > 8 && nmat == 2 && reads >= 280
                                : reads / 6 >= 5 + mb / 4 * n_expert * (1 - std::pow(1 - 1.0 / n_expert, ncols));
        const bool gather = !shared && (type == JL_TYPE_Q8_0 ? ncols <= 16 || (ncols <= 64 && avg <= 1.1)
                                                 : (long)nrows * k >= 512L * 512 && ncols <= ((double)nrows * k >= 2.4e6 && avg <= 0.6 ? 32 : 16));
        if (form == 0 && !planes && (type == JL_TYPE_Q8_0 || type == JL_TYPE_Q4_K || q6) && gather) form = 10;
        if (form == 0 && (c->act_window == 32 || c->act_window == 256) && !planes) {
            if (q4w) form = ncols <= 8L * n_expert ? 0 : moe_few_faster(type, n_expert, ncols, nmat, nrows, k) ? 5 : 9;
            else if (q6 && c->act_window == 256 && avg > 8 && avg < 60) form = moe_few_faster(type, n_expert, ncols, nmat, nrows, k) ? 5 : 9;
            else if (q6 && avg < (c->act_window == 32 ? 3 : 2) && k < 2048) form = 0;
            else if (avg < (q6 ? c->act_window == 256 ? 28 : k <= 1024 ? 52 : 40 : 40)) form = 5;
            else if (avg < (q6 && c->act_window == 32 ? 64 : 56)) form = tiles64 < 2 * c->num_cu || type == JL_TYPE_Q4_K ? 5 : q6 && c->act_window == 32 ? 7 : 6;
            else form = type == JL_TYPE_Q8_0 && avg >= 64 && tiles64 >= 2 * c->num_cu ? 8 : 6;
        }
        // Planes (gate + up + down of 128 x 768 x 2048 and 32 x 1024 x 2048, the block's us, the forms below against columns):
        // 12 columns 149 / 74 against 159 / 70, 16 157 / 75 against 167 / 72, 25 248 / 92 against 194 / 80, 48 363 / 135
        // against 275 / 105, 64 384 / 151 against 380 / 138, 128 (the second) 219 against 208.
        if (form == 0 && q4w && planes && ncols >= 16L * n_expert) form = 9;
        if (form == 5 && !align && c->tune.moe_form == 0 && avg >= 6) form = 6;
        if (form == 10 && !planes) {
            rc = moe_gather_launch(c, out0, out1, type, bank0, bank1, x, x2, src, start, nullptr, 0, 1, n_expert, ncols, nrows, k, st);
            if (rc != JL_DECLINED) return rc;
        }
        if (form == 9 && c->act_window == 256 && (type == JL_TYPE_Q4_K || (q6 && !planes))) {
            rc = moe_cols_launch(c, out0, out1, type, bank0, bank1, pb0, pb1, x, x2, src, start, n_expert, ncols, nrows, k, nsrc, st);
            if (rc != JL_DECLINED) return rc;
        }
        if (form >= 6 && !planes && gemm_i8_applies(c, type, nrows, k, ncols)) {
            rc = moe_gemm_i8_launch(c, out0, out1, type, bank0, bank1, x, x2, src, start, n_expert, ncols, nrows, k,
                                    form == 7 && q6 && c->act_window == 32 ? I8Shape{2, 2} : form == 8 && type == JL_TYPE_Q8_0 ? I8Shape{4, 4} : I8Shape{2, 4}, st, lists);
            if (rc != JL_DECLINED) return rc;
        }
        if (form == 5 && align && few_fits(c, type, planes, nrows, k, ncols, planes ? pb0->stride : 0)) {
            FewCall f;
            f.type = type; f.nrows = nrows; f.k = k; f.ncols = ncols; f.nmat = nmat;
            f.n_expert = n_expert; f.x = x; f.x2 = x2; f.src = src; f.start = start; f.out[0] = out0; f.out[1] = out1;
            PlaneRef a{}, b{};
            if (planes) {
                a = PlaneRef{pb0->qs, pb0->d, pb0->sc, 0, pb0->stride};
                if (pb1) b = PlaneRef{pb1->qs, pb1->d, pb1->sc, 0, pb1->stride};
                f.pl[0] = &a; f.pl[1] = pb1 ? &b : nullptr;
                f.sheet_words = pb0->sheet_bytes / 4; f.row_step = pb0->sheet_bytes ? 0 : nrows;
            } else {
                f.w[0] = bank0; f.w[1] = bank1; f.sheet_bytes = sheet;
            }
            rc = few_launch(c, f, st);
            if (rc != JL_DECLINED) return rc;
        }
    }
    // Q4_K with the k-quant activation window can also run on the matrix cores (tuning
    // "moe.form" = 2: groups of 32 columns, a wavefront to itself; 3: groups of 16, the weights
    // decoded in registers, below; 4: the prefill GEMM's tile).  Their vector work does not grow
    // with the number of columns.  Measured at the 128-expert shape, top-8 (router + gate + up +
    // down + combine, whole block, us; forms 1 / 2 / 3 with groups of 16 / 3 with groups of 32 / 4):
    //   16 rows 73 / 155 / 85 / - / -       64 rows 133 / 210 / 110 / - / -     128 rows 191 / 223 / 130 / 137 / 302
    //   192 rows - / 232 / 171 / 147 / 309  256 rows 333 / 238 / 187 / 157 / 315  512 rows - / 301 / 281 / 243 / 352
    //   1024 rows - / 426 / 489 / 372 / 400 1280 rows - / 501 / 577 / 475 / 435   2048 rows - / 709 / 831 / 639 / 623
    // so form 3 takes over from two columns an expert on average.  Above eight the columns against decoded rows
    // ("moe.form" = 9, above) have replaced groups of 32 and form 4 over GGUF rows (777 rows: 339 -> 234 us), and over planes
    // from sixteen; form 4 is left to what they decline, form 2 to "moe.form" = 2.
    // Form 3: groups of sixteen columns on the 16 x 16 x 32 matrix instruction, the weights decoded
    // in registers straight into its operand (Q4_K GGUF sheets or packed planes, the k-quant window; the group's
    // fragments for the whole of K sit in LDS).  Its steady state runs at the rate of a plain read;
    // the library picks it from two (over planes three) columns an expert on average up to 72, wherever
    // the fragments fit in LDS (one workgroup a CU runs either way: 100 experts x 512 x 2560, six columns, 63 -> 35 us);
    // "moe.form" = 3 forces it.
    {
        const int nsb = k / 256;
        const size_t frag16 = (size_t)nsb * JL_MOE_G16_LDS_WORDS * 4;   // a token tile's fragments
        const size_t lds16 = frag16 + 16;                               // and the tile counter
        const size_t nslots16 = (size_t)ncols / 16 + (size_t)n_expert + 1;
        const bool can16 = type == JL_TYPE_Q4_K && c->act_window == 256 && lds16 <= c->lds_limit &&
                           (size_t)nrows * row_bytes < ((size_t)1 << 32);
        const bool pick16 = c->tune.moe_form == 0 &&
                            (long)ncols >= (planes ? 3L : 2L) * n_expert && (long)ncols < 72L * n_expert;
        if (can16 && (c->tune.moe_form == 3 || pick16)) {
            // up to eight columns an expert the matrix kernel quantizes them itself: no prep launch,
            // no workspace ("moe.group16" = 1 forces the prep kernel, 2 the fused form).  (An expert of more than
            // sixteen is read twice, and that workgroup can be the launch's length; how often one is depends on the
            // routing.  Gate + up / down of 768 x 2048, means of eight random routings, fused against groups of 32:
            // 8 columns, 64 experts 31.4 / 18.3 against 37.5 / 24.2, 96 72 / 32 against 75 / 40, 112 64 / 52 against
            // 64 / 63, 128 68 / 32 against 69 / 38; 9 columns, 64 34 / 20 against 38 / 24, 112 72 / 55 against 64 / 63,
            // 128 75 / 36 against 70 / 38.)
            const bool fused = c->tune.moe_g16 == 2 || (c->tune.moe_g16 == 0 && (long)ncols <= 8L * n_expert);
            // beyond groups of 32 (two token tiles, a decoded word meets both), so
            // that an expert of 17-32 columns reads its sheet once ("moe.group16" = 3 forces them)
            const bool two = !fused && 2 * frag16 + 16 <= c->lds_limit &&
                             (c->tune.moe_g16 == 3 || c->tune.moe_g16 == 0);
            MoeG16PrepArgs pa;
            pa.ws = nullptr;
            if (!fused) {
                rc = ws_ensure(c, &c->moe_q_ws, &c->moe_q_ws_bytes, nslots16 * nsb * JL_MOE_G16_SB_WORDS * 4);
                if (rc != JL_OK) return rc;
                pa.x = x; pa.x2 = x2; pa.src = src; pa.start = start; pa.ws = (uint32_t*)c->moe_q_ws;
                pa.k = k; pa.n_expert = n_expert; pa.ncols = ncols;
                void* pp[] = {&pa};
                rc = launch(c, planes ? "jl_moe_g16_prep_planes" : "jl_moe_g16_prep", (unsigned)((ncols + 3) / 4), 1,
                            256, 0, st, pp);
                if (rc != JL_OK) return rc;
            }
            MoeG16Args ga;
            ga.out[0] = out0; ga.out[1] = out1;
            ga.bank[0] = (const uint8_t*)bank0; ga.bank[1] = (const uint8_t*)bank1;
            ga.ws = pa.ws; ga.start = start;
            if (fused) { ga.x = x; ga.x2 = x2; ga.src = src; }
            ga.sheet_bytes = sheet; ga.nrows = nrows; ga.k = k; ga.row_bytes = row_bytes;
            if (planes) {
                const jl_packed_bank* pbs[2] = {pb0, pb1};
                for (int m = 0; m < (pb1 ? 2 : 1); m++) { ga.pqs[m] = pbs[m]->qs; ga.pd[m] = pbs[m]->d; ga.psc[m] = pbs[m]->sc; }
                ga.sheet_words = pb0->sheet_bytes / 4;
                ga.row_step = pb0->sheet_bytes ? 0 : nrows;
                ga.pstride = pb0->stride;
            }
            const int nmat = (planes ? pb1 != nullptr : bank1 != nullptr) ? 2 : 1, tiles = (nrows + 15) / 16;
            const int nwaves = !two && c->tune.moe_waves == 4 ? 4 : 8;
            const int best_blocks = moe_g16_blocks(c, nrows, k, n_expert, ncols, nmat, nwaves);
            ga.tiles_wg = (tiles + best_blocks - 1) / best_blocks;   // handed out inside the workgroup as its wavefronts get to them
            ga.blocks = (tiles + ga.tiles_wg - 1) / ga.tiles_wg;
            ga.nmat = nmat; ga.n_expert = n_expert; ga.nwaves = nwaves;
            const long grid = 8L * ((n_expert + 7) / 8) * ga.blocks * nmat;
            if (grid >= (1L << 31)) return JL_DECLINED;
            // super-blocks a step: all of a short row, else two (288 contiguous bytes a row; four
            // measured 10 % slower at K = 2048: twice the bytes in flight before the first step)
            // (over planes one: a lane's twelve loads of a super-block go to twelve planes, and more
            // of them in flight measured 5 % slower)
            int ch = planes ? 1 : (nsb <= 3 ? nsb : 2);
            if (c->tune.moe_chunk >= 1 && c->tune.moe_chunk <= 3) ch = std::min(c->tune.moe_chunk, nsb);
            Name name;
            name << "jl_moe_g16" << (planes ? "p_" : "_") << (fused ? (x2 ? 'g' : 'f') : two ? 'd' : 'c') << ch;
            void* gp[] = {&ga};
            return launch(c, name, (unsigned)grid, 1, (unsigned)(64 * nwaves), (unsigned)(two ? 2 * frag16 + 16 : lds16), st, gp);
        }
    }
    if (planes && c->tune.moe_form != 4 && (c->tune.moe_form == 1 || (long)ncols < kMoePlaneTileCols * n_expert)) {
        // few columns an expert: the dot-product form over planes (rows on lanes, a lane's share of a
        // chunk loaded once for all the expert's columns, the columns as scalar operands)
        if ((size_t)ncols * (k / 256) * 88 >= ((size_t)1 << 32)) return JL_DECLINED;   // 32-bit word offsets in the kernel
        // the columns quantized once, chunk by chunk: 88 words a (column, 256 elements)
        rc = ws_ensure(c, &c->moe_q_ws, &c->moe_q_ws_bytes, (size_t)ncols * (k / 256) * 88 * 4);
        if (rc != JL_OK) return rc;
        MoeQuantArgs qa;
        qa.x = x; qa.x2 = x2; qa.src = src;
        qa.q = nullptr; qa.as = nullptr; qa.s16 = nullptr; qa.chunked = (uint32_t*)c->moe_q_ws;
        qa.k = k; qa.per = c->act_window / 32; qa.start = start; qa.n_expert = n_expert;
        void* qparams[] = {&qa};
        rc = launch(c, "jl_moe_quant", (unsigned)((k / 4 + 255) / 256), (unsigned)ncols, 256, 0, st, qparams);
        if (rc != JL_OK) return rc;
        MoePlanesArgs a;
        const jl_packed_bank* pbs[2] = {pb0, pb1};
        const int nmat = pb1 ? 2 : 1;
        for (int m = 0; m < 2; m++) {
            a.out[m] = m == 0 ? out0 : out1;
            a.pqs[m] = m < nmat ? pbs[m]->qs : nullptr; a.pd[m] = m < nmat ? pbs[m]->d : nullptr;
            a.psc[m] = m < nmat ? pbs[m]->sc : nullptr;
        }
        a.chunked = qa.chunked; a.start = start;
        a.sheet_words = pb0->sheet_bytes / 4; a.row_step = pb0->sheet_bytes ? 0 : nrows; a.pstride = pb0->stride;
        a.nrows = nrows; a.k = k;
        a.nwaves = std::min(8, k / 256);
        void* params[] = {&a};
        return launch(c, "jl_moe_matvec_planes_q4k", (unsigned)((nrows + 63) / 64), (unsigned)n_expert, (unsigned)(a.nwaves * 64),
                      (unsigned)(a.nwaves * 8 * 256), st, params, (unsigned)nmat);   // JL_MOEP_TB columns a pass
    }
    const bool many_cols = c->tune.moe_form == 0 && (long)ncols >= 10L * n_expert;   // (72 and more get here)
    if (type == JL_TYPE_Q4_K && c->act_window == 256 && (planes || c->tune.moe_form == 4 || many_cols || c->tune.moe_form == 2) &&
        4u * 19968u <= c->lds_limit) {   // JL_MOEG_WAVE_LDS
        const int nslots = ncols / 32 + n_expert + 1, nsb = k / 256;
        const int tiles_max = ncols / 128 + n_expert;
        if (nslots > 65535) return JL_DECLINED;
        auto up256 = [](size_t v) { return (v + 255) & ~(size_t)255; };
        const size_t bq_bytes = (size_t)2 * nsb * nslots * kGemmAStageBytes;
        const size_t o_wl = bq_bytes + up256((size_t)nsb * nslots * 32 * 4);
        rc = ws_ensure(c, &c->moe_q_ws, &c->moe_q_ws_bytes, o_wl + (size_t)(4 + nslots + tiles_max) * 4);
        if (rc != JL_OK) return rc;
        // the work list of groups and tiles, from start[]
        MoeWorklistArgs wa;
        wa.start = start; wa.wl = (uint32_t*)((char*)c->moe_q_ws + o_wl);
        wa.n_expert = n_expert; wa.nslots = nslots;
        void* wp[] = {&wa};
        rc = launch(c, "jl_moe_worklist", 1, 1, 1024, 0, st, wp);
        if (rc != JL_OK) return rc;
        MoeGemmPrepArgs pa;
        pa.x = x; pa.x2 = x2; pa.src = src; pa.start = start; pa.wl = wa.wl;
        pa.bq = (uint16_t*)c->moe_q_ws; pa.da = (float*)((char*)c->moe_q_ws + bq_bytes);
        pa.k = k; pa.nslots = nslots;
        void* pp[] = {&pa};
        rc = launch(c, planes ? "jl_moe_gemm_prep_planes" : "jl_moe_gemm_prep", (unsigned)nsb, (unsigned)nslots, 256, 0, st, pp);
        if (rc != JL_OK) return rc;
        MoeGemmArgs ga;
        ga.out[0] = out0; ga.out[1] = out1;
        ga.bank[0] = (const uint8_t*)bank0; ga.bank[1] = (const uint8_t*)bank1;
        ga.bq = pa.bq; ga.da = pa.da; ga.start = start; ga.wl = wa.wl;
        ga.sheet_bytes = sheet; ga.nrows = nrows; ga.k = k; ga.row_bytes = row_bytes;
        ga.nslots = nslots; ga.nmat = (planes ? pb1 != nullptr : bank1 != nullptr) ? 2 : 1;
        if (planes) {
            const jl_packed_bank* pbs[2] = {pb0, pb1};
            for (int m = 0; m < ga.nmat; m++) { ga.pqs[m] = pbs[m]->qs; ga.pd[m] = pbs[m]->d; ga.psc[m] = pbs[m]->sc; }
            ga.sheet_words = pb0->sheet_bytes / 4;
            ga.row_step = pb0->sheet_bytes ? 0 : nrows;
            ga.pstride = pb0->stride;
        }
        void* gp[] = {&ga};
        const long rtiles = (nrows + 63) / 64;
        if (planes) {
            if (kGemmLdsBytes > c->lds_limit || (long)tiles_max * rtiles * ga.nmat >= (1L << 31)) return JL_DECLINED;
            const long work = (long)tiles_max * rtiles * ga.nmat;
            return launch(c, "jl_moe_gemm_r64_planes", (unsigned)std::min<long>(work, 2L * c->num_cu), 1, 256,
                          gemm_lds_bytes(64), st, gp);
        }
        if ((c->tune.moe_form == 4 || (c->tune.moe_form == 0 && (long)ncols >= 56L * n_expert)) &&
            kGemmLdsBytes <= c->lds_limit && n_expert <= 65535 && (long)tiles_max * rtiles * ga.nmat < (1L << 31)) {
            const long work = (long)tiles_max * rtiles * ga.nmat;
            return launch(c, "jl_moe_gemm_r64", (unsigned)std::min<long>(work, 2L * c->num_cu), 1, 256, gemm_lds_bytes(64), st, gp);
        }
        return launch(c, "jl_moe_gemm_q4k", (unsigned)((nrows + 255) / 256), (unsigned)nslots, 256, 4u * 19968u, st, gp,
                      (unsigned)ga.nmat);
    }
    if (planes) return JL_DECLINED;   // (no LDS for the tile form on this device)
    const int nslots = k / ti->slot_elems;
    // lanes per row: the width that leaves the fewest lanes without a slot (a row of 12 slots
    // on 16 lanes idles a quarter of them; on 4 lanes, three slots each, none); among equals
    // eight lanes, several slots a lane, measured best (sweeps at the 128-expert shape);
    // tuning "moe.lpr" overrides
    int lpr = 64, waste = 1 << 30;
    for (int cand : {8, 16, 4, 32, 64}) {
        const int w = (nslots + cand - 1) / cand * cand - nslots;
        if (w < waste) { waste = w; lpr = cand; }
    }
    {
        // (100 * a + b: a for rows of more than 16 slots, b for shorter ones)
        const int tl = c->tune.moe_lpr > 64 ? (nslots > 16 ? c->tune.moe_lpr / 100 : c->tune.moe_lpr % 100) : c->tune.moe_lpr;
        if (tl == 4 || tl == 8 || tl == 16 || tl == 32 || tl == 64) lpr = tl;
    }
    const size_t act = ((size_t)k + (size_t)(k / 32) * 4 + (size_t)(k / 16) * 4 + 15) & ~(size_t)15;
    const size_t lds = 8 * act;
    if (lds > c->lds_limit) return JL_DECLINED;

    // every column's activation, quantized once: q [ncols][k], as [ncols][k/32], s16 [ncols][k/16]
    auto up256 = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t o_as = up256((size_t)ncols * k), o_s16 = o_as + up256((size_t)ncols * (k / 32) * 4);
    rc = ws_ensure(c, &c->moe_q_ws, &c->moe_q_ws_bytes, o_s16 + up256((size_t)ncols * (k / 16) * 4));
    if (rc != JL_OK) return rc;
    char* qws = (char*)c->moe_q_ws;
    MoeQuantArgs qa;
    qa.x = x; qa.x2 = x2; qa.src = src;
    qa.q = (int8_t*)qws; qa.as = (float*)(qws + o_as); qa.s16 = (float*)(qws + o_s16);
    qa.k = k; qa.per = c->act_window / 32; qa.start = start; qa.n_expert = n_expert;
    void* qparams[] = {&qa};
    rc = launch(c, "jl_moe_quant", (unsigned)((k / 4 + 255) / 256), (unsigned)ncols, 256, 0, st, qparams);
    if (rc != JL_OK) return rc;

    MoeMatVecArgs a;
    a.out[0] = out0; a.out[1] = out1;
    a.bank[0] = (const uint8_t*)bank0; a.bank[1] = (const uint8_t*)bank1;
    a.q = qa.q; a.as = qa.as; a.s16 = qa.s16; a.start = start;
    a.sheet_bytes = sheet; a.nrows = nrows; a.k = k; a.row_bytes = row_bytes;
    // A workgroup of four wavefronts covers 4 * 2 * (64 / lpr) rows per step; at the kernel's
    // ~150 registers three such workgroups fill a CU's twelve wavefront slots, where one of
    // eight wavefronts leaves four empty (sweeps at the 128-expert, 64-row shape: 210 -> 150 us
    // for the block).  Row shares: about twelve workgroups per CU when every expert is in use,
    // each share at least one step.
    const int nmat = bank1 ? 2 : 1, nwaves = c->tune.moe_waves > 0 && c->tune.moe_waves <= 8 ? c->tune.moe_waves : 4;
    const int rows_per_step = nwaves * 2 * (64 / lpr);  // JL_MOE_U row groups per wavefront step
    int shares = c->tune.moe_shares;
    if (shares <= 0) {
        shares = (12 * c->num_cu + n_expert * nmat - 1) / (n_expert * nmat);
        const int most = (nrows + rows_per_step - 1) / rows_per_step;
        if (shares > most) shares = most;
    }
    if (shares < 1) shares = 1;
    if (shares > 65535) shares = 65535;
    a.nwaves = nwaves; a.shares = shares;
    Name name;
    name << "jl_moe_matvec_" << ti->tag << "_l" << lpr;
    void* params[] = {&a};
    return launch(c, name, (unsigned)shares, (unsigned)n_expert, nwaves * 64, (unsigned)lds, st, params, (unsigned)nmat);
}

}  // namespace

extern "C" {

int jl_ctx_create(jl_ctx** out, const jl_options* opts) {
    if (!out) return fail(nullptr, JL_ERR_ARG, "jl_ctx_create: null out");
    *out = nullptr;
    if (!H) {
        std::string why;
        H = hip_api(&why);
        if (!H) return fail(nullptr, JL_ERR_HIP, "%s", why.c_str());
    }
    jl_ctx* c = new (std::nothrow) jl_ctx;
    if (!c) return fail(nullptr, JL_ERR_NOMEM, "out of memory");
    c->device = opts ? opts->device : 0;
    c->act_window = (opts && opts->act_window) ? opts->act_window : 32;
    std::string path = (opts && opts->code_object) ? opts->code_object : default_code_object();

    auto bail = [&](int code, const std::string& msg) {
        g_create_error = msg;
        jl_ctx_destroy(c);
        return code;
    };
    if (c->act_window != 32 && c->act_window != 64 && c->act_window != 128 && c->act_window != 256)
        return bail(JL_ERR_ARG, "act_window must be 32, 64, 128 or 256");
    if (c->device < 0) {
        // no device: the host-side bookkeeping (residency keys, the forget queue, the lock)
        // works, every entry point that needs the GPU fails at its hipSetDevice
        c->no_device = true;
        *out = c;
        return JL_OK;
    }
    hipError_t e = H->SetDevice(c->device);
    if (e != hipSuccess) return bail(JL_ERR_HIP, std::string("hipSetDevice: ") + H->GetErrorString(e));
    hipDeviceProp_t prop;
    e = H->GetDeviceProperties(&prop, c->device);
    if (e != hipSuccess) return bail(JL_ERR_HIP, std::string("hipGetDeviceProperties: ") + H->GetErrorString(e));
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return bail(JL_ERR_HIP, std::string("device is ") + prop.gcnArchName + ", this library is gfx950 only");
    c->num_cu = prop.multiProcessorCount;
    c->lds_limit = prop.sharedMemPerBlock;
    {
        // the static workspace's address on this device, looked up once per device with the
        // device current; a failure only disables the entry point that lives on it
        const char* why = "";
        if (jl_static_scratch_get(c->device, &c->static_scratch, &c->static_scratch_bytes, &why) != 0) {
            c->static_scratch = nullptr;
            c->static_scratch_bytes = 0;
            c->static_err = why;
        }
    }
    e = H->StreamCreate(&c->stream);
    if (e != hipSuccess) return bail(JL_ERR_HIP, std::string("hipStreamCreate: ") + H->GetErrorString(e));
    e = H->ModuleLoad(&c->module, path.c_str());
    if (e != hipSuccess)
        return bail(JL_ERR_HIP, "hipModuleLoad(" + path + "): " + H->GetErrorString(e));

    std::vector<std::string> names = {"jl_quantize_act", "jl_dequant", "jl_matvec_q4k_r1_pq", "jl_matvec_q4k_r1_pq_res", "jl_matvec_q8_0_r1_pq", "jl_matvec_q8_0_r1_pq_res", "jl_matvec_q6k_r1_pq", "jl_matvec_q6k_r1_pq_res", "jl_matvec_q8_0p_r1_pq", "jl_matvec_q8_0p_r1_pq_res", "jl_matvec_q4k_r1_res", "jl_matvec_q4k_r1_x4_res", "jl_matvec_q8_0_r1_res", "jl_matvec_q8_0_r1_x4_res", "jl_matvec_q6k_r1_res", "jl_matvec_q6k_r1_x4_res", "jl_matvec_q8_0p_r1_res", "jl_matvec_q8_0p_r1_x4_res", "jl_matvec_q8_0p_r1", "jl_matvec_q8_0p_r2", "jl_matvec_q8_0p_r4", "jl_gemm_prep_q4k", "jl_gemm_prep_q4k_w16", "jl_gemm_q4k_r64", "jl_gemm_q4k_r128", "jl_gemm_q4k_wide", "jl_gemm_prep_q4k_fold", "jl_gemm_q4k_fold_wide", "jl_gemm_q4k_fold_wide4", "jl_gemm_q4k_k2", "jl_gemm_q4k_k2_planes", "jl_gemm_prep_q4k_planes", "jl_gemm_q4k_r64_planes", "jl_gemm_q4k_wide_planes", "jl_gemm_w16_prep_q4k", "jl_gemm_q4k_w16", "jl_gemm_q4k_few32", "jl_moe_route", "jl_moe_route_g2", "jl_moe_route_g4", "jl_moe_logits", "jl_moe_logits_e2", "jl_moe_logits_e2_f16", "jl_moe_logits_e4", "jl_moe_logits_e4_f16", "jl_moe_logits_e8", "jl_moe_logits_e8_f16", "jl_moe_group", "jl_moe_group2", "jl_moe_quant", "jl_moe_matvec_planes_q4k", "jl_moe_combine", "jl_moe_worklist", "jl_moe_gemm_prep", "jl_moe_gemm_prep_planes", "jl_moe_gemm_q4k", "jl_moe_g16_prep", "jl_moe_g16_prep_planes", "jl_moe_g16_c1", "jl_moe_g16_c2", "jl_moe_g16_c3", "jl_moe_g16_f1", "jl_moe_g16_f2", "jl_moe_g16_f3", "jl_moe_g16_g1", "jl_moe_g16_g2", "jl_moe_g16_g3", "jl_moe_g16_d1", "jl_moe_g16_d2", "jl_moe_g16_d3", "jl_moe_g16p_c1", "jl_moe_g16p_c2", "jl_moe_g16p_c3", "jl_moe_g16p_f1", "jl_moe_g16p_f2", "jl_moe_g16p_f3", "jl_moe_g16p_g1", "jl_moe_g16p_g2", "jl_moe_g16p_g3", "jl_moe_g16p_d1", "jl_moe_g16p_d2", "jl_moe_g16p_d3", "jl_moe_gemm_r64", "jl_moe_gemm_r64_planes", "jl_mxfp4_prep", "jl_mxfp4_prep_few", "jl_mxfp4_few_t1", "jl_mxfp4_few_t2", "jl_mxfp4_few_t3", "jl_mxfp4_few_t4", "jl_mxfp4_few_planes_t1", "jl_mxfp4_few_planes_t2", "jl_mxfp4_few_planes_t3", "jl_mxfp4_few_planes_t4", "jl_mxfp4_few_c3", "jl_mxfp4_few_c4", "jl_mxfp4_few_planes_c3", "jl_mxfp4_few_planes_c4", "jl_mxfp4_gemm", "jl_mxfp4_gemm_r96", "jl_mxfp4_matvec", "jl_mxfp4_matvec1_b1", "jl_mxfp4_matvec1_b2", "jl_mxfp4_matvec1_b3", "jl_mxfp4_scaled_prep", "jl_mxfp4_scaled_gemm", "jl_mxfp4_planes_prep", "jl_mxfp4_planes_gemm", "jl_mxfp4_planes_gemm_r96", "jl_mxfp4_matvec_planes_r64", "jl_mxfp4_matvec_planes_r32", "jl_mxfp4_matvec_planes_r16", "jl_unpack_mxfp4", "jl_sum_parts", "jl_silu_mul", "jl_add_rows", "jl_host_in", "jl_host_done", "jl_q4k_fold_range", "jl_probe_read", "jl_probe_empty", "jl_probe_wait", "jl_probe_mfma", "jl_probe_mfma_v5",
                                      "jl_pack_weights", "jl_unpack_q4k", "jl_unpack_q6k", "jl_unpack_q8_0"};
    names.push_back("jl_few_prep");
    for (const char* pl : {"", "planes_"})
        for (int nt = 1; nt <= 4; nt++)
            for (int rt = 1; rt <= 2; rt++) names.push_back(std::string("jl_mxfp4_one_") + pl + "t" + std::to_string(nt) + "r" + std::to_string(rt));
    names.push_back("jl_gemm_i8_prep");
    names.push_back("jl_moe_gemm_i8_prep");
    for (const char* tag : {"q4k", "q8_0", "q8_0p", "q6k", "q6kw"})
        for (const char* act : {"", "_a", "_down"})
            for (const char* lpr : {"_l8", "_l16", "_l32", "_l64"}) names.push_back(std::string("jl_moe_gather_") + tag + act + lpr);
    for (const char* rw : {"16", "32", "64"})
        for (const char* form : {"jl_moe_planes_gather_w", "jl_moe_planes_down_w"}) names.push_back(std::string(form) + rw);
    for (const char* tag : {"q4kf", "q6kw"})
        for (const char* form : {"", "_x2", "_x4", "_l32", "_l16"}) names.push_back(std::string("jl_matvec_multi_") + tag + form);
    for (const char* rw : {"16", "32", "64"}) names.push_back(std::string("jl_matvec_packed_multi_q4kf_w") + rw);
    for (const char* tag : {"q4k", "q4k_planes", "q6k"})
        for (const char* form : {"jl_moe_cols_", "jl_moe_cols_prep_"}) names.push_back(std::string(form) + tag);
    for (const char* tag : {"q8_0", "q4k", "q6k", "q6kw"})
        for (const char* form : {"jl_gemm_i8_%s_r2t4", "jl_moe_gemm_i8_%s_r2t4"}) {
            char nm[64];
            snprintf(nm, sizeof nm, form, tag);
            names.push_back(nm);
        }
    names.push_back("jl_moe_gemm_i8_q6k_r2t2");
    names.push_back("jl_gemm_i8_q8_0_r4t4");
    names.push_back("jl_gemm_i8_q8_0_r4t8");
    names.push_back("jl_moe_gemm_i8_q8_0_r4t4");
    for (const char* tag : {"q4k", "q4kw", "q8_0", "q6k", "q6kw"})
        for (const char* layout : {"rows", "planes"})
            for (const char* size : {"t1r1", "t1r2", "t2r1", "t3r1", "t3r2", "t4r1", "t4r2", "t1r4", "t2r2", "t2r4"})
                if (layout[0] == 'p' || (strcmp(size, "t1r4") && strcmp(size, "t2r2") && strcmp(size, "t2r4"))) names.push_back(std::string("jl_few_") + tag + "_" + layout + "_" + size);
    for (const char* tag : {"q4k", "q8_0", "q6k"})
        for (int rw : {16, 32, 64})
            for (const char* form : {"", "q8_"})
                names.push_back(std::string("jl_matvec_packed_") + form + tag + "_w" + std::to_string(rw));
    for (const char* tag : {"q4k", "q8_0", "q6k"})
        for (int lpr : {4, 8, 16, 32, 64}) names.push_back(std::string("jl_moe_matvec_") + tag + "_l" + std::to_string(lpr));
    const int types[] = {JL_TYPE_Q4_K, JL_TYPE_Q8_0, JL_TYPE_Q6_K};
    for (int t : types)
        for (int rpw : {1, 2, 4}) {
            char nm[64];
            snprintf(nm, sizeof nm, "jl_matvec_%s_r%d", type_info(t)->tag, rpw);
            names.push_back(nm);
            names.push_back(std::string(nm) + "_x2");
            names.push_back(std::string(nm) + "_x4");
        }
    for (int rpw : {1, 2, 4})
        for (const char* xp : {"_x2", "_x4"}) names.push_back("jl_matvec_q8_0p_r" + std::to_string(rpw) + xp);
    for (const char* tag : {"q4k", "q8_0", "q6k", "q8_0p"}) names.push_back(std::string("jl_matvec_") + tag + "_r1_x2_res");
    for (const char* lanes : {"_l32", "_l16"}) {
        for (const char* tag : {"q4k", "q8_0", "q6k", "q8_0p"})
            for (const char* form : {"jl_matvec_%s_r1", "jl_matvec_multi_%s", "jl_matvec_multi_%s_n"}) {
                std::string n(form);
                names.push_back(n.replace(n.find("%s"), 2, tag) + lanes);
            }
        for (const char* pre : {"", "_n"}) names.push_back(std::string("jl_matvec_segments") + pre + lanes);
    }
    for (const char* tag : {"q4k", "q8_0", "q6k", "q8_0p"}) {
        for (const char* res : {"", "_res"}) {
            for (const char* pre : {"", "_n", "_a", "_na"})
                for (const char* xp : {"", "_x2", "_x4"}) names.push_back(std::string("jl_matvec_multi_") + tag + pre + xp + res);
            names.push_back(std::string("jl_matvec_multi_") + tag + "_q" + res);
        }
    }
    for (const char* pre : {"", "_n", "_a", "_na"})
        for (const char* res : {"", "_res"}) names.push_back(std::string("jl_matvec_segments") + pre + res);
    for (const char* tag : {"q4k", "q8_0", "q6k"})
        for (int rw : {16, 32, 64})
            for (const char* form : {"", "act_", "norm_"})
                names.push_back(std::string("jl_matvec_packed_multi_") + form + tag + "_w" + std::to_string(rw));
    for (const auto& n : names) {
        hipFunction_t f;
        e = H->ModuleGetFunction(&f, c->module, n.c_str());
        if (e != hipSuccess)
            return bail(JL_ERR_HIP, "hipModuleGetFunction(" + n + "): " + H->GetErrorString(e));
        c->fn.add(n, f);
    }
    for (int form = 0; form < 5; form++)
        for (int planes = 0; planes < 2; planes++)
            for (int nt = 1; nt <= 4; nt++)
                for (int rt : {1, 2, 4}) {
                    const char* tags[] = {"q4k", "q4kw", "q8_0", "q6k", "q6kw"};   // (few_form)
                    Name n;
                    n << "jl_few_" << tags[form] << (planes ? "_planes" : "_rows") << "_t" << nt << "r" << rt;
                    const hipFunction_t f = c->fn.find(n);
                    int regs = 0;
                    if (!f) continue;
                    e = H->FuncGetAttribute(&regs, HIP_FUNC_ATTRIBUTE_NUM_REGS, f);
                    if (e != hipSuccess) return bail(JL_ERR_HIP, std::string("hipFuncGetAttribute(") + (const char*)n + "): " + H->GetErrorString(e));
                    // (a SIMD's 512 registers a lane, in blocks of eight)
                    c->few_simd[form][planes][nt - 1][rt / 2] = (uint8_t)std::max(1, std::min(8, 512 / std::max(8, (regs + 7) / 8 * 8)));
                }
    {
        uint32_t tab[2 * 17];
        for (uint32_t n = 0; n <= 16; n++) { tab[2 * n] = 0; tab[2 * n + 1] = n; }
        e = H->Malloc((void**)&c->one_group, sizeof tab);
        if (e == hipSuccess) e = H->Memcpy(c->one_group, tab, sizeof tab, hipMemcpyHostToDevice);
        if (e != hipSuccess) return bail(JL_ERR_HIP, std::string("column range table: ") + H->GetErrorString(e));
    }
    *out = c;
    return JL_OK;
}

const char* jl_hip_runtime(void) {
    std::string why;
    const HipApi* h = hip_api(&why);
    return h ? h->path.c_str() : "";
}

void jl_ctx_destroy(jl_ctx* c) {
    if (!c) return;
    if (c->no_device) {
        delete c;
        return;
    }
    (void)H->SetDevice(c->device);
    if (c->stream) (void)H->StreamSynchronize(c->stream);
    (void)H->DeviceSynchronize();   // callers' streams may still read the workspaces
    for (auto& kv : c->resident) (void)H->Free(kv.second.dev);
    if (c->gemm_ws) (void)H->Free(c->gemm_ws);
    if (c->w16_ws) (void)H->Free(c->w16_ws);
    if (c->moe_ws) (void)H->Free(c->moe_ws);
    if (c->unpack_ws) (void)H->Free(c->unpack_ws);
    if (c->flag_ws) (void)H->Free(c->flag_ws);
    if (c->moe_q_ws) (void)H->Free(c->moe_q_ws);
    if (c->act_ws) (void)H->Free(c->act_ws);
    if (c->layer_ws) (void)H->Free(c->layer_ws);
    if (c->moe_route_ws) (void)H->Free(c->moe_route_ws);
    for (auto& kv : c->layers)
        if (kv.second.mem) (void)H->Free(kv.second.mem);
    if (c->one_group) (void)H->Free(c->one_group);
    if (c->mx_ws) (void)H->Free(c->mx_ws);
    if (c->pin) (void)H->HostFree(c->pin);
    if (c->pin_flag) (void)H->HostFree((void*)c->pin_flag);
    if (c->stage_x) (void)H->Free(c->stage_x);
    if (c->stage_out) (void)H->Free(c->stage_out);
    if (c->module) (void)H->ModuleUnload(c->module);
    if (c->stream) (void)H->StreamDestroy(c->stream);
    delete c;
}

const char* jl_last_error(const jl_ctx* c) { return c ? c->err.c_str() : g_create_error.c_str(); }

int jl_set_act_window(jl_ctx* c, int window) {
    if (!c) return JL_ERR_ARG;
    if (window != 32 && window != 64 && window != 128 && window != 256)
        return fail(c, JL_ERR_ARG, "act_window must be 32, 64, 128 or 256, not %d", window);
    c->act_window = window;
    return JL_OK;
}

void* jl_stream(jl_ctx* c) { return c ? (void*)c->stream : nullptr; }

int jl_synchronize(jl_ctx* c) {
    if (!c) return JL_ERR_ARG;
    HIP_TRY(c, H->SetDevice(c->device));
    HIP_TRY(c, H->StreamSynchronize(c->stream));
    return JL_OK;
}

unsigned long long jl_launch_count(const jl_ctx* c) { return c ? c->launches.load() : 0ull; }

int jl_set_tuning(jl_ctx* c, const char* key, int value) {
    if (!c || !key) return JL_ERR_ARG;
    if (!strcmp(key, "matvec.rpw")) c->tune.rpw = value;
    else if (!strcmp(key, "matvec.block")) c->tune.block = value;
    else if (!strcmp(key, "matvec.grid")) c->tune.grid = value;
    else if (!strcmp(key, "packed.rw")) c->tune.packed_rw = value;
    else if (!strcmp(key, "packed.block")) c->tune.packed_block = value;
    else if (!strcmp(key, "moe.group")) c->tune.moe_group = value;
    else if (!strcmp(key, "moe.logits")) c->tune.moe_logits = value;
    else if (!strcmp(key, "moe.q6k_cols")) (void)value;   // (accepted, without effect)
    else if (!strcmp(key, "moe.shares")) c->tune.moe_shares = value;
    else if (!strcmp(key, "moe.form")) c->tune.moe_form = value;
    else if (!strcmp(key, "moe.group16")) c->tune.moe_g16 = value;
    else if (!strcmp(key, "moe.chunk")) c->tune.moe_chunk = value;
    else if (!strcmp(key, "moe.waves")) c->tune.moe_waves = value;
    else if (!strcmp(key, "matvec.lanes")) c->tune.matvec_lanes = value;
    else if (!strcmp(key, "moe.lpr")) c->tune.moe_lpr = value;
    else if (!strcmp(key, "gemm.rows")) c->tune.gemm_rows = value;
    else if (!strcmp(key, "mxfp4.split")) c->tune.mx_split = value;
    else if (!strcmp(key, "mxfp4.few")) c->tune.mx_few = value;
    else if (!strcmp(key, "mxfp4.few_min")) c->tune.mx_few_min = value;
    else if (!strcmp(key, "gemm.tall")) c->tune.gemm_tall = value;
    else if (!strcmp(key, "mxfp4.one")) c->tune.mx_one = value;
    else if (!strcmp(key, "mxfp4.rows")) c->tune.mx_rows = value;
    else if (!strcmp(key, "mxfp4.planes")) c->tune.mx_planes = value;
    else if (!strcmp(key, "mxfp4.scaled")) c->tune.mx_scaled = value;
    else if (!strcmp(key, "matvec.q8pair")) c->tune.q8pair = value;
    else if (!strcmp(key, "matvec.xpre")) c->tune.xpre = value;
    else if (!strcmp(key, "matvec.act_split")) c->tune.act_split = value;
    else if (!strcmp(key, "gemm.form")) c->tune.gemm_form = value;
    else if (!strcmp(key, "gemm.fold")) c->tune.gemm_fold = value;
    else if (!strcmp(key, "gemm.fold_waves")) c->tune.gemm_fold_waves = value;
    else if (!strcmp(key, "gemm.split")) c->tune.gemm_split = value;
    else if (!strcmp(key, "gemm.prep")) c->tune.gemm_prep = value;
    else if (!strcmp(key, "gemm.planes")) c->tune.gemm_planes = value;
    else if (!strcmp(key, "gemm.few")) c->tune.gemm_few = value;
    else if (!strcmp(key, "gemm.i8")) c->tune.gemm_i8 = value;
    else if (!strcmp(key, "few.nt")) c->tune.few_nt = value;
    else if (!strcmp(key, "few.rt")) c->tune.few_rt = value;
    else if (!strcmp(key, "few.waves")) c->tune.few_waves = value;
    else if (!strcmp(key, "gemm.min_tok")) c->gemm_min_tok = value > 0 ? value : 3;
    else return fail(c, JL_ERR_ARG, "unknown tuning key %s", key);
    return JL_OK;
}

/* ------------------------------------------------ device-pointer entry points */

int jl_quantize_act_dev(jl_ctx* c, const float* x, int ntok, int k, int8_t* q, float* as,
                        float* sum16, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!x || !q || !as || !sum16 || ntok <= 0 || k <= 0)
        return fail(c, JL_ERR_ARG, "quantize_act: bad operand");
    if (k % 32 != 0 || !aligned16(x) || !aligned16(q)) return JL_DECLINED;
    if (ntok > 65535) return JL_DECLINED;
    HIP_TRY(c, H->SetDevice(c->device));
    int per = c->act_window / 32;
    const float* no_gate = nullptr;
    void* params[] = {(void*)&x, (void*)&q, (void*)&as, (void*)&sum16, (void*)&k, (void*)&per, (void*)&no_gate};
    unsigned gx = (unsigned)((k / 4 + 255) / 256);  // one thread per four elements
    return launch(c, "jl_quantize_act", gx, (unsigned)ntok, 256, 0, pick_stream(c, stream), params);
}

int jl_dequant_dev(jl_ctx* c, int type, const void* src, float* dst, size_t n, void* stream) {
    if (!c) return JL_ERR_ARG;
    int be;
    switch (type) {
    case JL_TYPE_Q8_0: case JL_TYPE_MXFP4: be = 32; break;
    case JL_TYPE_Q4_K: case JL_TYPE_Q6_K: be = 256; break;
    default: return JL_DECLINED;
    }
    if (!src || !dst) return fail(c, JL_ERR_ARG, "dequant: null operand");
    if (n == 0 || n % (size_t)be != 0) return fail(c, JL_ERR_ARG, "dequant: %zu elements is not whole blocks", n);
    if (type == JL_TYPE_Q4_K && ((uintptr_t)src & 3) != 0) return JL_DECLINED;
    if (type != JL_TYPE_MXFP4 && ((uintptr_t)src & 1) != 0) return JL_DECLINED;
    size_t blocks = (n + 255) / 256;
    if (blocks > 0x7fffffffu) return JL_DECLINED;
    HIP_TRY(c, H->SetDevice(c->device));
    void* params[] = {(void*)&src, (void*)&dst, (void*)&n, (void*)&type};
    return launch(c, "jl_dequant", (unsigned)blocks, 1, 256, 0, pick_stream(c, stream), params);
}

int jl_matvec_dev(jl_ctx* c, float* out, int type, const void* w, const float* x, int nrows, int k,
                  void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!x) return fail(c, JL_ERR_ARG, "matvec: null x");
    HIP_TRY(c, H->SetDevice(c->device));
    return matvec_launch(c, out, type, w, x, nullptr, nullptr, nullptr, nrows, k, pick_stream(c, stream));
}

int jl_matvec_q8_dev(jl_ctx* c, float* out, int type, const void* w, const int8_t* q,
                     const float* as, const float* sum16, int nrows, int k, void* stream) {
    if (!c) return JL_ERR_ARG;
    HIP_TRY(c, H->SetDevice(c->device));
    return matvec_launch(c, out, type, w, nullptr, q, as, sum16, nrows, k, pick_stream(c, stream));
}

int jl_matvec_group_dev(jl_ctx* c, const jl_mv_group* g, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!g || g->n < 1 || g->n > JL_MAX_GROUP || !g->x || g->k <= 0) return fail(c, JL_ERR_ARG, "matvec group: bad group");
    HIP_TRY(c, H->SetDevice(c->device));
    hipStream_t st = pick_stream(c, stream);
    // everything is checked before the first launch: a group is served whole or not at all
    for (int i = 0; i < g->n; i++) {
        const TypeInfo* ti = nullptr;
        int rc = matvec_check(c, g->type[i], g->rows[i], g->k, &ti);
        if (rc != JL_OK) return rc;
        if (!g->out[i] || !g->w[i]) return fail(c, JL_ERR_ARG, "matvec group: null operand");
        if ((g->type[i] == JL_TYPE_Q4_K && !aligned16(g->w[i])) || ((uintptr_t)g->w[i] & 1)) return JL_DECLINED;
    }
    if (!aligned16(g->x) || (g->act_up && !aligned16(g->act_up))) return JL_DECLINED;
    if ((g->norm_w && !aligned16(g->norm_w)) || (g->norm_out && (!g->norm_w || !aligned16(g->norm_out)))) return JL_DECLINED;
    // one launch: the single-type kernel, or the mixed-type one when the formats differ
    // (the reference's MatVecSegments, jit/gpu/kernels/matvec.go:1411-1431)
    bool mixed = false;
    for (int i = 1; i < g->n; i++) mixed = mixed || g->type[i] != g->type[0];
    return matvec_multi_launch(c, g->type[0], g->n, g->out, g->w, g->rows, g->x, 0, g->act_up, g->resid, g->alpha,
                               g->k, st, g->norm_w, g->norm_eps, g->norm_out, mixed ? g->type : nullptr,
                               g->resid_gate);
}

int jl_matvec_packed_multi_dev(jl_ctx* c, float* const* outs, int type, const uint32_t* const* qs,
                               const uint32_t* const* d, const uint32_t* const* sc, const int* row0, int stride,
                               const float* x, size_t xstride, const float* up, float* resid, float alpha,
                               const float* resid_gate, const float* norm_w, float norm_eps, float* norm_out,
                               int nrows, int k, int m, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!outs || !qs || !d || !row0 || m < 1) return fail(c, JL_ERR_ARG, "packed multi: bad operand");
    if (m > JL_MAX_MULTI) return JL_DECLINED;
    HIP_TRY(c, H->SetDevice(c->device));
    PlaneRef pls[JL_MAX_MULTI];
    for (int j = 0; j < m; j++) {
        pls[j].qs = qs[j]; pls[j].d = d[j]; pls[j].sc = sc ? sc[j] : nullptr;
        pls[j].row = row0[j]; pls[j].stride = stride;
    }
    return packed_matvec_multi_launch(c, type, m, outs, pls, x, xstride, up, resid, alpha, resid_gate, norm_w,
                                      norm_eps, norm_out, nrows, k, pick_stream(c, stream));
}

int jl_matvec_multi_dev(jl_ctx* c, float* const* outs, int type, const void* const* ws, const float* x,
                        int nrows, int k, int m, void* stream) {
    return jl_matvec_gather_dev(c, outs, type, ws, x, 0, nullptr, nrows, k, m, stream);
}

int jl_matvec_gather_dev(jl_ctx* c, float* const* outs, int type, const void* const* ws, const float* x,
                         size_t xstride, const float* up, int nrows, int k, int m, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!outs || !ws || m < 1) return fail(c, JL_ERR_ARG, "matvec multi: bad operand");
    if (m > JL_MAX_MULTI) return JL_DECLINED;
    HIP_TRY(c, H->SetDevice(c->device));
    int rows[JL_MAX_MULTI];
    for (int i = 0; i < m; i++) rows[i] = nrows;
    return matvec_multi_launch(c, type, m, outs, ws, rows, x, xstride, up, nullptr, 0.f, k, pick_stream(c, stream));
}

int jl_matmul_dev(jl_ctx* c, float* out, int type, const void* w, const float* x, int nrows, int k,
                  int ntok, void* stream) {
    if (!c) return JL_ERR_ARG;
    HIP_TRY(c, H->SetDevice(c->device));
    return matmul_launch(c, out, type, w, x, nrows, k, ntok, pick_stream(c, stream));
}

int jl_matmul_static_dev(jl_ctx* c, float* out, int type, const void* w, const float* x, int nrows, int k,
                         int ntok, void* stream) {
    if (!c) return JL_ERR_ARG;
    HIP_TRY(c, H->SetDevice(c->device));
    if (!c->static_scratch) return fail(c, JL_ERR_HIP, "the static scratch is not available: %s", c->static_err.c_str());
    // The call runs jl_matmul_dev's own launch path with every context workspace set aside:
    // whatever the path asks for is carved, in order, from the static array (grow() above), and
    // a shape that needs more than the array holds is an error before anything is launched
    // that would use the missing piece.  No hipMalloc, no hipFree, no synchronisation.
    struct Saved { void** buf; size_t* have; void* b; size_t h; };
    Saved saved[] = {{&c->gemm_ws, &c->gemm_ws_bytes, nullptr, 0}, {&c->w16_ws, &c->w16_ws_bytes, nullptr, 0},
                     {&c->mx_ws, &c->mx_ws_bytes, nullptr, 0},     {&c->moe_q_ws, &c->moe_q_ws_bytes, nullptr, 0},
                     {&c->unpack_ws, &c->unpack_ws_bytes, nullptr, 0}};
    for (auto& s : saved) { s.b = *s.buf; s.h = *s.have; *s.buf = nullptr; *s.have = 0; }
    // a dry run first: the sizes are checked against the array before the first real launch
    int rc;
    {
        CallScope no_alloc(c, false, true);
        {
            CallScope dry(c, true, false);
            rc = matmul_launch(c, out, type, w, x, nrows, k, ntok, pick_stream(c, stream));
        }
        if (rc == JL_OK) {
            for (auto& s : saved) { *s.buf = nullptr; *s.have = 0; }
            g_call.static_used = 0;
            rc = matmul_launch(c, out, type, w, x, nrows, k, ntok, pick_stream(c, stream));
        }
    }
    for (auto& s : saved) { *s.buf = s.b; *s.have = s.h; }
    return rc;
}

size_t jl_static_scratch_bytes(void) { return JL_STATIC_SCRATCH_BYTES; }

int jl_packed_words(int type, int nrows, int k, size_t* nq, size_t* nd, size_t* nsc) {
    if (!nq || !nd || !nsc || nrows <= 0) return JL_ERR_ARG;
    return packed_words(type, (size_t)nrows, k, nq, nd, nsc) ? JL_OK : JL_DECLINED;
}

int jl_pack_weights_dev(jl_ctx* c, int type, const void* src, int nrows, int k, uint32_t* qs, uint32_t* d,
                        uint32_t* sc, void* stream) {
    if (!c) return JL_ERR_ARG;
    size_t nq, nd, nsc;
    if (nrows <= 0 || !packed_words(type, (size_t)nrows, k, &nq, &nd, &nsc)) return JL_DECLINED;
    if (!src || !qs || !d || (nsc && !sc)) return fail(c, JL_ERR_ARG, "pack: null operand");
    if (type != JL_TYPE_MXFP4 && ((uintptr_t)src & (type == JL_TYPE_Q4_K ? 3 : 1))) return JL_DECLINED;
    if (((uintptr_t)qs | (uintptr_t)d | (uintptr_t)sc) & 3) return JL_DECLINED;
    const int units = type == JL_TYPE_Q8_0 || type == JL_TYPE_MXFP4 ? k / 32 : k / 256;
    if (units > 65535) return JL_DECLINED;
    HIP_TRY(c, H->SetDevice(c->device));
    hipStream_t st = pick_stream(c, stream);
    PackArgs a;
    a.src = (const uint8_t*)src; a.qs = qs; a.d = d; a.sc = sc; a.nrows = nrows; a.k = k; a.type = type;
    a.flag = nullptr;
    void* params[] = {&a};
    if (type != JL_TYPE_MXFP4)
        return launch(c, "jl_pack_weights", (unsigned)((nrows + 255) / 256), (unsigned)units, 256, 0, st, params);
    // MXFP4: the packer raises a flag for a block whose exponent the D plane cannot hold
    // (mxfp4Refuse, jit/gpu/kernels/pack.go:407-420); the call waits for it, and a refused
    // matrix leaves the planes' contents undefined.
    int rc = ws_ensure(c, &c->flag_ws, &c->flag_ws_bytes, 256);
    if (rc != JL_OK) return rc;
    uint32_t flag = 0;
    HIP_TRY(c, H->Memcpy(c->flag_ws, &flag, 4, hipMemcpyHostToDevice));
    a.flag = (uint32_t*)c->flag_ws;
    rc = launch(c, "jl_pack_weights", (unsigned)((nrows + 255) / 256), (unsigned)units, 256, 0, st, params);
    if (rc != JL_OK) return rc;
    HIP_TRY(c, H->StreamSynchronize(st));
    HIP_TRY(c, H->Memcpy(&flag, c->flag_ws, 4, hipMemcpyDeviceToHost));
    return flag ? JL_DECLINED : JL_OK;
}

int jl_fold_admit_dev(jl_ctx* c, int type, const void* w, int nrows, int k, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (type != JL_TYPE_Q4_K || nrows <= 0 || k <= 0 || k % 256) return JL_DECLINED;
    if (!w) return fail(c, JL_ERR_ARG, "fold admit: null weights");
    if ((uintptr_t)w & 3) return JL_DECLINED;
    {
        std::lock_guard<std::mutex> g(c->forget_mu);
        c->fold_ok.erase((uintptr_t)w);   // whatever an earlier matrix at this address was found to be
    }
    HIP_TRY(c, H->SetDevice(c->device));
    hipStream_t st = pick_stream(c, stream);
    int rc = ws_ensure(c, &c->flag_ws, &c->flag_ws_bytes, 256);
    if (rc != JL_OK) return rc;
    uint32_t flag = 0;
    HIP_TRY(c, H->Memcpy(c->flag_ws, &flag, 4, hipMemcpyHostToDevice));
    FoldRangeArgs a;
    a.w = (const uint8_t*)w; a.nblocks = (size_t)nrows * (size_t)(k / 256); a.flag = (uint32_t*)c->flag_ws;
    void* params[] = {&a};
    rc = launch(c, "jl_q4k_fold_range", (unsigned)((a.nblocks + 255) / 256), 1, 256, 0, st, params);
    if (rc != JL_OK) return rc;
    HIP_TRY(c, H->StreamSynchronize(st));
    HIP_TRY(c, H->Memcpy(&flag, c->flag_ws, 4, hipMemcpyDeviceToHost));
    if (flag) return JL_DECLINED;
    std::lock_guard<std::mutex> g(c->forget_mu);
    c->fold_ok[(uintptr_t)w] = {nrows, k};
    return JL_OK;
}

int jl_unpack_weights_dev(jl_ctx* c, int type, const uint32_t* qs, const uint32_t* d, const uint32_t* sc,
                          int row, int stride, int nrows, int k, void* dst, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (type == JL_TYPE_MXFP4) {
        const PlaneRef mpl = {qs, d, nullptr, row, stride};
        int mrc = mx_planes_check(c, mpl, nrows, k);
        if (mrc != JL_OK) return mrc;
        if (!dst) return fail(c, JL_ERR_ARG, "unpack: null dst");
        HIP_TRY(c, H->SetDevice(c->device));
        return unpack_launch(c, type, mpl, nrows, k, dst, pick_stream(c, stream));
    }
    if (type != JL_TYPE_Q4_K && type != JL_TYPE_Q6_K && type != JL_TYPE_Q8_0) return JL_DECLINED;
    const PlaneRef pl = {qs, d, sc, row, stride};
    const TypeInfo* ti = nullptr;
    int rc = packed_check(c, type, pl, nrows, k, &ti);
    if (rc != JL_OK) return rc;
    if (!dst) return fail(c, JL_ERR_ARG, "unpack: null dst");
    if (((uintptr_t)dst & (type == JL_TYPE_Q4_K ? 3 : 1)) || k / ti->block_elems > 65535) return JL_DECLINED;
    HIP_TRY(c, H->SetDevice(c->device));
    return unpack_launch(c, type, pl, nrows, k, dst, pick_stream(c, stream));
}

int jl_matvec_packed_dev(jl_ctx* c, float* out, int type, const uint32_t* qs, const uint32_t* d,
                         const uint32_t* sc, int row, int stride, const float* x, int nrows, int k,
                         void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!x) return fail(c, JL_ERR_ARG, "packed matvec: null x");
    HIP_TRY(c, H->SetDevice(c->device));
    const PlaneRef pl = {qs, d, sc, row, stride};
    return packed_matvec_launch(c, out, type, pl, x, nullptr, nullptr, nullptr, nrows, k, pick_stream(c, stream));
}

int jl_matvec_packed_q8_dev(jl_ctx* c, float* out, int type, const uint32_t* qs, const uint32_t* d,
                            const uint32_t* sc, int row, int stride, const int8_t* q, const float* as,
                            const float* sum16, int nrows, int k, void* stream) {
    if (!c) return JL_ERR_ARG;
    HIP_TRY(c, H->SetDevice(c->device));
    const PlaneRef pl = {qs, d, sc, row, stride};
    return packed_matvec_launch(c, out, type, pl, nullptr, q, as, sum16, nrows, k, pick_stream(c, stream));
}

int jl_matmul_packed_dev(jl_ctx* c, float* out, int type, const uint32_t* qs, const uint32_t* d,
                         const uint32_t* sc, int row, int stride, const float* x, int nrows, int k,
                         int ntok, void* stream) {
    if (!c) return JL_ERR_ARG;
    HIP_TRY(c, H->SetDevice(c->device));
    const PlaneRef pl = {qs, d, sc, row, stride};
    return packed_matmul_launch(c, out, type, pl, x, nrows, k, ntok, pick_stream(c, stream));
}

int jl_reserve(jl_ctx* c, int max_tok, int max_k) {
    if (!c) return JL_ERR_ARG;
    if (max_tok <= 0 || max_k <= 0 || max_k % 256 != 0) return fail(c, JL_ERR_ARG, "reserve: %d x %d", max_tok, max_k);
    HIP_TRY(c, H->SetDevice(c->device));
    // the k-quant prep's layout and the window-32 prep's (fragments + two scale planes)
    const size_t tok_pad = ((size_t)max_tok + 255) / 256 * 256;
    const size_t w32 = (size_t)(max_k / 128) * (tok_pad / 32) * 8 * 1024 + 2 * (size_t)(max_k / 32) * tok_pad * 4;
    int rc = gemm_ws_ensure(c, std::max(gemm_ws_need(max_tok, max_k), w32));
    if (rc == JL_OK) rc = ws_ensure(c, &c->mx_ws, &c->mx_ws_bytes, slab_reserve(c));
    if (rc != JL_OK) return rc;
    if (!reserved_for(c, max_tok, max_k)) c->reserved.push_back({max_tok, max_k});
    return JL_OK;
}

int jl_reserve_shape(jl_ctx* c, int type, int nrows, int k, int ntok, int packed) {
    if (!c) return JL_ERR_ARG;
    if (nrows <= 0 || k <= 0 || ntok <= 0) return fail(c, JL_ERR_ARG, "reserve shape: %d x %d, %d tokens", nrows, k, ntok);
    HIP_TRY(c, H->SetDevice(c->device));
    // Walk the call's own launch path with launching switched off: every workspace the path
    // would grow is grown now, by the code that sizes it for the real call.
    float* const out = (float*)(uintptr_t)4096;
    const float* const x = (const float*)(uintptr_t)4096;
    const void* const w = (const void*)(uintptr_t)4096;
    CallScope dry(c, true, false);
    int rc;
    if (type == JL_TYPE_MXFP4) {
        rc = packed ? jl_matmul_mxfp4_packed_bf16_dev(c, out, (const uint32_t*)w, (const uint32_t*)w, 0, nrows,
                                                      (const uint16_t*)w, nrows, k, ntok, nullptr)
                    : jl_matmul_mxfp4_bf16_dev(c, out, w, (const uint16_t*)w, nrows, k, ntok, nullptr);
    } else if (packed) {
        const PlaneRef pl = {(const uint32_t*)w, (const uint32_t*)w, (const uint32_t*)w, 0, nrows};
        rc = packed_matmul_launch(c, out, type, pl, x, nrows, k, ntok, c->stream);
    } else {
        rc = matmul_launch(c, out, type, w, x, nrows, k, ntok, c->stream);
    }
    return rc;
}

int jl_moe_route_dev(jl_ctx* c, const float* logits, int rows, int n_expert, int k_used, uint32_t* sel,
                     int sel_stride, float* wt, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!logits || !sel || !wt || rows <= 0 || n_expert <= 0 || k_used <= 0 || sel_stride < k_used)
        return fail(c, JL_ERR_ARG, "moe route: bad operand");
    if (n_expert > 1024 || k_used > 16 || k_used > n_expert) return JL_DECLINED;
    HIP_TRY(c, H->SetDevice(c->device));
    MoeRouteArgs a;
    a.logits = logits; a.sel = sel; a.wt = wt; a.n_expert = n_expert; a.k_used = k_used; a.sel_stride = sel_stride;
    void* params[] = {&a};
    // the form with the fewest experts a lane that holds them all (less code for a lone wavefront to fetch)
    const char* name = n_expert <= 128 ? "jl_moe_route_g2" : n_expert <= 256 ? "jl_moe_route_g4" : "jl_moe_route";
    return launch(c, name, (unsigned)rows, 1, 64, 0, pick_stream(c, stream), params);
}

int jl_moe_logits_dev(jl_ctx* c, float* logits, int wtype, const void* w, const float* x, int n_expert, int k,
                      int ntok, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!logits || !w || !x || n_expert <= 0 || k <= 0 || ntok <= 0)
        return fail(c, JL_ERR_ARG, "moe logits: bad operand");
    if (wtype != JL_TYPE_F32 && wtype != JL_TYPE_F16) return JL_DECLINED;
    if (((uintptr_t)w & (wtype == JL_TYPE_F32 ? 3 : 1)) || ((uintptr_t)x & 3)) return JL_DECLINED;
    if (n_expert > 65535 || (ntok + 7) / 8 > 65535) return JL_DECLINED;
    HIP_TRY(c, H->SetDevice(c->device));
    MoeLogitsArgs a;
    a.w = w; a.x = x; a.logits = logits; a.n_expert = n_expert; a.k = k; a.ntok = ntok;
    a.f16 = wtype == JL_TYPE_F16;
    void* params[] = {&a};
    // Expert rows a workgroup takes: more of them meet an x value loaded once, fewer are more workgroups, whose wavefronts hide each
    // other's dependent adds.  us by 1 / 2 / 4 / 8 rows, x from memory: 128 experts x 2048, 64 tokens 5.3 / 6.0 / 6.7 / 9.4, 128 9.2 /
    // 6.4 / 7.2 / 9.6, 256 13.6 / 9.0 / 7.7 / 10.3, 512 22 / 14.6 / 11.7 / 11.6, 1024 47 / 31 / 23 / 18.9; 64 x 2048, 512 tokens 14.5 /
    // 10.1 / 7.7 / 10.3; 87 x 1024, 1024 tokens 29 / 12.3 / 9.5 / 10.0; 16 x 2816, 1024 tokens 18.6 / 10.8 / 11.5 / 14.1.  Tuning
    // "moe.logits" = 1 / 2 / 4 / 8 forces a form, and 16 or 32 more the order of the grid below: token groups or rows of the router.
    int eb = c->tune.moe_logits % 16;
    if (eb != 1 && eb != 2 && eb != 4 && eb != 8) {
        const auto a_cu = [&](int e) { return (double)((n_expert + e - 1) / e) * ((ntok + 7) / 8) / c->num_cu; };
        eb = a_cu(1) <= 4 ? 1 : a_cu(2) <= 5 ? 2 : a_cu(4) <= std::max(5.75, 11776.0 / k) ? 4 : 8;
    }
    const unsigned groups = (unsigned)(ntok + 7) / 8, blocks = (unsigned)(n_expert + eb - 1) / eb;   // JL_LOGITS_TOK
    // Workgroups go round the XCDs in the order of their numbers.  Token groups side by side bring each its rows of x to one L2, and every
    // row of the router to all; rows of the router side by side bring each to one L2, and x to all.  Many tokens: the first, unless the router is
    // more than an L2 holds (4 MB).  Up to 64: the second where the router is large, in f32 with a row a workgroup only while the workgroups are few.
    // us, token groups / rows: 384 x 7168 in f32, 2048 tokens 334 / 265, 256 x 7168 192 / 181, 128 x 7168 93 / 100; 256 x 7168 in f16, 16 tokens
    // 21.7 / 13.7, 160 x 5120 in f16, 32 tokens 16.3 / 11.2, in f32 16 tokens 8.4 / 7.6; 128 x 7168 in f32, 64 tokens 13.9 / 15.0; 128 x 2048 in
    // f32, 128 tokens 4.8 / 5.2.  (275 shapes: 0.3 % behind the better order.)
    const size_t elems = (size_t)n_expert * k;
    if (c->tune.moe_logits >= 16) a.by_expert = c->tune.moe_logits >= 32;
    else if (ntok <= 64) a.by_expert = elems >= 800000 && (a.f16 || eb > 1 || (long)blocks * groups <= 3L * c->num_cu);
    else a.by_expert = elems * (a.f16 ? 2 : 4) > ((size_t)4 << 20);
    Name name;
    name << "jl_moe_logits";
    if (eb > 1) name << "_e" << eb << (a.f16 ? "_f16" : "");
    if (a.by_expert) return launch(c, name, blocks, groups, 128, 0, pick_stream(c, stream), params);
    return launch(c, name, std::min(8u, groups), blocks, 128, 0, pick_stream(c, stream), params, (groups + 7) / 8);
}

namespace {
int moe_group_launch(jl_ctx* c, const uint32_t* sel, int sel_stride, int rows, int k_used, int n_expert, uint32_t* start, uint32_t* perm,
                     uint32_t* pos, MoeLists* lists, hipStream_t st) {
    if (!sel || !start || !perm || !pos || rows <= 0 || k_used <= 0 || sel_stride < k_used)
        return fail(c, JL_ERR_ARG, "moe group: bad operand");
    if (n_expert <= 0 || n_expert > 1024) return JL_DECLINED;
    HIP_TRY(c, H->SetDevice(c->device));
    MoeGroupArgs a;
    a.sel = sel; a.start = start; a.perm = perm; a.pos = pos;
    a.sel_stride = sel_stride; a.rows = rows; a.k_used = k_used; a.n_expert = n_expert;
    void* params[] = {&a};
    // the linear-time form, a workgroup for 1024 pairs (moe.group = 1 forces the one that compares every pair with every
    // expert)
    const size_t npairs = (size_t)rows * k_used, lds2 = JL_MOE_GROUP2_LDS((size_t)n_expert);
    if (c->tune.moe_group != 1 && lds2 <= c->lds_limit && npairs <= 0x7fffffffu - 8192) {
        if (lists->nslots) { a.wl[0] = lists->wl[0]; a.wl[1] = lists->wl[1]; a.nslots = lists->nslots; }
        const size_t n1024 = (npairs + 1023) / 1024;
        a.chunks = (int)((n1024 + c->num_cu - 1) / c->num_cu);
        return launch(c, "jl_moe_group2", (unsigned)((n1024 + a.chunks - 1) / a.chunks), 1, 1024, (unsigned)lds2, st, params);
    }
    lists->nslots = 0;   // (this form makes none)
    return launch(c, "jl_moe_group", 1, 1, 1024, 0, st, params);
}
}  // namespace

int jl_moe_group_dev(jl_ctx* c, const uint32_t* sel, int sel_stride, int rows, int k_used, int n_expert,
                     uint32_t* start, uint32_t* perm, uint32_t* pos, void* stream) {
    if (!c) return JL_ERR_ARG;
    MoeLists none{};
    return moe_group_launch(c, sel, sel_stride, rows, k_used, n_expert, start, perm, pos, &none, pick_stream(c, stream));
}

int jl_moe_matvec_dev(jl_ctx* c, float* out0, float* out1, int type, const void* bank0, const void* bank1,
                      const float* x, const float* x2, const uint32_t* src, const uint32_t* start,
                      int n_expert, int ncols, int nrows, int k, void* stream) {
    if (!c) return JL_ERR_ARG;
    HIP_TRY(c, H->SetDevice(c->device));
    return moe_matvec_launch(c, out0, out1, type, bank0, bank1, x, x2, src, start, n_expert, ncols, nrows, k,
                             pick_stream(c, stream));
}

int jl_moe_matvec_packed_dev(jl_ctx* c, float* out0, float* out1, int type, const jl_packed_bank* bank0,
                             const jl_packed_bank* bank1, const float* x, const float* x2, const uint32_t* src,
                             const uint32_t* start, int n_expert, int ncols, int nrows, int k, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!bank0) return fail(c, JL_ERR_ARG, "moe matvec: null bank");
    HIP_TRY(c, H->SetDevice(c->device));
    return moe_matvec_launch(c, out0, out1, type, nullptr, nullptr, x, x2, src, start, n_expert, ncols, nrows, k,
                             pick_stream(c, stream), bank0, bank1);
}

namespace {
// last_id: ids past it are no expert's and add nothing.
int moe_combine_launch(jl_ctx* c, float* resid, const float* y, const float* wt, const uint32_t* sel, int sel_stride, const uint32_t* pos,
                       int rows, int k_used, int n_embd, uint32_t last_id, hipStream_t st) {
    if (!resid || !y || !wt || !sel || !pos || rows <= 0 || n_embd <= 0)
        return fail(c, JL_ERR_ARG, "moe combine: bad operand");
    if (k_used <= 0 || k_used > 16 || sel_stride < k_used || rows > 65535) return JL_DECLINED;
    if (n_embd % 4 != 0 || !aligned16(resid) || !aligned16(y)) return JL_DECLINED;   // four columns a thread
    HIP_TRY(c, H->SetDevice(c->device));
    MoeCombineArgs a;
    a.resid = resid; a.y = y; a.wt = wt; a.sel = sel; a.pos = pos;
    a.sel_stride = sel_stride; a.k_used = k_used; a.n_embd = n_embd; a.last_id = last_id;
    void* params[] = {&a};
    return launch(c, "jl_moe_combine", (unsigned)((n_embd / 4 + 255) / 256), (unsigned)rows, 256, 0, st, params);
}
}  // namespace

// (how many experts there are is not known here: every id counts)
int jl_moe_combine_dev(jl_ctx* c, float* resid, const float* y, const float* wt, const uint32_t* sel,
                       int sel_stride, const uint32_t* pos, int rows, int k_used, int n_embd, void* stream) {
    if (!c) return JL_ERR_ARG;
    return moe_combine_launch(c, resid, y, wt, sel, sel_stride, pos, rows, k_used, n_embd, 0xFFFFFFFFu, pick_stream(c, stream));
}

namespace {
// The routed block's workspace: first columns, row of a column, column of a pair, then gate, up
// and down of every column.
struct MoeWs {
    uint32_t *start, *perm, *pos;
    float *g, *u, *y;
    MoeLists lists;
};
int moe_ws(jl_ctx* c, int rows, int k_used, int n_expert, int n_ffn, int n_embd, MoeWs* w) {
    const size_t ncols = (size_t)rows * k_used;
    auto up256 = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t o_start = 0, o_perm = up256((size_t)(n_expert + 1) * 4), o_pos = o_perm + up256(ncols * 4);
    const size_t o_g = o_pos + up256(ncols * 4), o_u = o_g + up256(ncols * n_ffn * 4);
    const size_t o_y = o_u + up256(ncols * n_ffn * 4), o_wl = o_y + up256(ncols * n_embd * 4);
    const size_t nslots = ncols / 32 + n_expert + 1, list = up256((4 + nslots + ncols / 64 + n_expert) * 4);
    int rc = ws_ensure(c, &c->moe_ws, &c->moe_ws_bytes, o_wl + 2 * list);
    if (rc != JL_OK) return rc;
    char* ws = (char*)c->moe_ws;
    w->start = (uint32_t*)(ws + o_start);
    w->perm = (uint32_t*)(ws + o_perm);
    w->pos = (uint32_t*)(ws + o_pos);
    w->g = (float*)(ws + o_g); w->u = (float*)(ws + o_u); w->y = (float*)(ws + o_y);
    w->lists = MoeLists{{(uint32_t*)(ws + o_wl), (uint32_t*)(ws + o_wl + list)}, (int)nslots};
    return JL_OK;
}

// "moe.form" asks for one of the mixture's own kernels
bool moe_dense_wanted(const jl_ctx* c) { return c->tune.moe_form == 0; }

// A dense gated feed-forward block for n rows: y = W_down (silu(W_gate x) * W_up x), resid[r] += wt[r] * y[r]
// (wt null: 1).  g, u: n n_ffn floats each, y: n n_embd.  Up to 64 rows two few-token matmuls -- gate and up in one
// launch, the gated activation formed by down's activation prep, the residual added where the result is made
// when its weight is one -- and above that three prefill GEMMs: nothing is routed, so nothing of the mixture's
// grouping, work lists and column gathers is needed.  (As a mixture of one expert: Q4_K 3584 / 13056 over
// planes, 34 rows 194 us, Q4_K 1536 / 3328, 17 rows 88 us.)  JL_DECLINED when a matmul has no such form.
int dense_ffn(jl_ctx* c, float* resid, int type, int down_type, const void* gate, const void* up, const void* down,
              const PlaneRef* pg, const PlaneRef* pu, const PlaneRef* pd, const float* x, const float* wt, int n, int n_ffn,
              int n_embd, float* g, float* u, float* y, hipStream_t st) {
    const bool planes = pg != nullptr;
    auto few = [&](int t, const void* w, const PlaneRef* p, int nrows, int k) {
        return n <= 64 && few_fits(c, t, planes, nrows, k, n, planes ? p->stride : 0) && (planes || ((uintptr_t)w & (t == JL_TYPE_Q4_K ? 15 : 3)) == 0);
    };
    // (vectors of four floats are read from x and added to resid; rows longer than the decode kernels take are not
    // served whatever the number of tokens)
    if (n > 65535 || n_embd % 4 || n_ffn % 4 || !aligned16(x) || !aligned16(resid)) return JL_DECLINED;
    const TypeInfo* ti = nullptr;
    int rc;
    if (!planes && ((rc = matvec_check(c, type, n_ffn, n_embd, &ti)) != JL_OK || (rc = matvec_check(c, down_type, n_embd, n_ffn, &ti)) != JL_OK))
        return rc;
    // Two to four rows: a decode matvec a row and matrix, two launches (moe_gather_ffn with no selection) where the few-token form's
    // four are slower: 9 us + 0.12 (Q8_0 0.14) a MB of weights and row, against 15.5 + 0.28 a MB less a tenth.  Rows, us, before -> so:
    // Q4_K 1024 / 4096 2, 4 rows 16.3 -> 10.1, 17.1 -> 11.1; 4096 / 14336 2 rows 42.4 -> 33.5, 3 rows 42.5 (48.3 so);
    // Q6_K 2048 / 8192 3 rows 28.4 -> 25.3, 4 rows 29.1 (27.0 so, left); Q8_0 2048 / 8192 2 rows 26.1 -> 18.0; Q4_K planes 1280 / 5120
    // 2 rows 19.1 -> 12.4.  (From five rows on only the smallest blocks gain, 16.9 -> 14.5 at eight rows of 1024 / 4096, and a row's bits
    // there are those of a longer run, tests/test_gpu_layer.py.)
    if (n >= 2 && n <= 4 && moe_dense_wanted(c) && !c->tune.gemm_form && !c->tune.gemm_few && !c->tune.few_nt && !c->tune.few_rt) {
        const TypeInfo *t = type_info(type), *d = type_info(down_type);
        const double mb = 1e-6 * n_ffn * n_embd * (2.0 * t->block_bytes / t->block_elems + (double)d->block_bytes / d->block_elems);
        if (mb * ((type == JL_TYPE_Q8_0 ? 0.14 : 0.12) * n - 0.25) < 4.4) {
            if (!planes && n_ffn % 64 == 0 && n_embd % 64 == 0 && aligned16(gate) && aligned16(up) && aligned16(down)) {
                rc = moe_gather_ffn(c, resid, type, down_type, gate, up, down, x, nullptr, 0, wt, n, 1, 1, n_ffn, n_embd, g, u, st);
                if (rc != JL_DECLINED) return rc;
            } else if (planes && type == JL_TYPE_Q4_K && down_type == JL_TYPE_Q4_K && pg->stride == pu->stride && !pg->row && !pu->row && !pd->row) {
                const jl_packed_bank bg = {pg->qs, pg->d, pg->sc, 0, pg->stride}, bu = {pu->qs, pu->d, pu->sc, 0, pu->stride},
                                     bd = {pd->qs, pd->d, pd->sc, 0, pd->stride};
                rc = moe_planes_gather_ffn(c, resid, &bg, &bu, &bd, x, nullptr, 0, wt, n, 1, 1, n_ffn, n_embd, g, u, st);
                if (rc != JL_DECLINED) return rc;
            }
        }
    }
    if (few(type, gate, pg, n_ffn, n_embd) && few(type, up, pu, n_ffn, n_embd) && (!planes || (pg->row == pu->row && pg->stride == pu->stride))) {
        FewCall f;
        f.type = type; f.nrows = n_ffn; f.k = n_embd; f.ncols = n; f.nmat = 2; f.x = x;
        f.w[0] = gate; f.w[1] = up; f.pl[0] = pg; f.pl[1] = pu; f.out[0] = g; f.out[1] = u;
        rc = few_launch(c, f, st);
    } else {
        rc = planes ? packed_matmul_launch(c, g, type, *pg, x, n_ffn, n_embd, n, st) : matmul_launch(c, g, type, gate, x, n_ffn, n_embd, n, st);
        if (rc == JL_OK)
            rc = planes ? packed_matmul_launch(c, u, type, *pu, x, n_ffn, n_embd, n, st) : matmul_launch(c, u, type, up, x, n_ffn, n_embd, n, st);
    }
    if (rc != JL_OK) return rc;
    if (few(down_type, down, pd, n_embd, n_ffn)) {
        FewCall f;
        f.type = down_type; f.nrows = n_embd; f.k = n_ffn; f.ncols = n; f.x = g; f.x2 = u;
        f.w[0] = down; f.pl[0] = pd;
        if (wt) f.out[0] = y; else f.resid = resid;
        rc = few_launch(c, f, st);
        if (rc != JL_OK || !wt) return rc;
    } else {
        size_t nh = (size_t)n * n_ffn;
        void* ap[] = {&g, &u, &nh};
        rc = launch(c, "jl_silu_mul", (unsigned)((nh / 4 + 255) / 256), 1, 256, 0, st, ap);
        if (rc == JL_OK)
            rc = planes ? packed_matmul_launch(c, y, down_type, *pd, g, n_embd, n_ffn, n, st)
                        : matmul_launch(c, y, down_type, down, g, n_embd, n_ffn, n, st);
        if (rc != JL_OK) return rc;
    }
    void* rp[] = {&resid, &y, (void*)&wt, &n_embd};
    return launch(c, "jl_add_rows", (unsigned)((n_embd / 4 + 255) / 256), (unsigned)n, 256, 0, st, rp);
}

// Everything the steps of a routed block ask of the caller's operands, asked before anything is enqueued and whether or
// not the steps run (a block of one expert has nothing to group or combine).  Reads nothing of the device.
int moe_ffn_check(jl_ctx* c, const float* resid, int type, int down_type, const void* gate_bank, const void* up_bank,
                  const void* down_bank, const jl_packed_bank* pg, const jl_packed_bank* pu, const jl_packed_bank* pd,
                  const float* x, int rows, int k_used, int n_expert, int n_ffn, int n_embd) {
    if (rows <= 0 || k_used <= 0 || n_expert <= 0 || n_ffn <= 0 || n_embd <= 0) return fail(c, JL_ERR_ARG, "moe ffn: bad shape");
    if (!resid || !x) return fail(c, JL_ERR_ARG, "moe ffn: null operand");
    if (n_expert > 1024 || k_used > 16 || n_ffn % 256 != 0 || n_embd % 256 != 0) return JL_DECLINED;
    int rc = moe_banks_check(c, type, pg != nullptr, gate_bank, up_bank, pg, pu, true, n_expert, n_ffn, n_embd);
    if (rc == JL_OK) rc = moe_banks_check(c, down_type, pg != nullptr, down_bank, nullptr, pd, nullptr, false, n_expert, n_embd, n_ffn);
    if (rc != JL_OK) return rc;
    return aligned16(x) && aligned16(resid) && (size_t)rows * k_used <= 65535 ? JL_OK : JL_DECLINED;
}

int moe_ffn(jl_ctx* c, float* resid, int type, int down_type, const void* gate_bank, const void* up_bank,
            const void* down_bank, const jl_packed_bank* pg, const jl_packed_bank* pu, const jl_packed_bank* pd,
            const float* x, const uint32_t* sel, int sel_stride, const float* wt, int rows, int k_used, int n_expert,
            int n_ffn, int n_embd, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!sel || !wt || sel_stride < k_used) return fail(c, JL_ERR_ARG, "moe ffn: bad selection");
    int rc = moe_ffn_check(c, resid, type, down_type, gate_bank, up_bank, down_bank, pg, pu, pd, x, rows, k_used, n_expert, n_ffn, n_embd);
    if (rc != JL_OK) return rc;
    const bool planes = pg != nullptr;
    const size_t ncols = (size_t)rows * k_used;
    HIP_TRY(c, H->SetDevice(c->device));
    const TypeInfo* ti = nullptr;
    if ((rc = matvec_check(c, type, n_ffn, n_embd, &ti)) != JL_OK || (rc = matvec_check(c, down_type, n_embd, n_ffn, &ti)) != JL_OK) return rc;
    hipStream_t st = pick_stream(c, stream);
    MoeWs w;
    rc = moe_ws(c, rows, k_used, n_expert, n_ffn, n_embd, &w);
    if (rc != JL_OK) return rc;
    uint32_t *start = w.start, *perm = w.perm, *pos = w.pos;
    float *g = w.g, *u = w.u, *y = w.y;
    // one expert: every row is its column, nothing to group (and no selection to read: every id is 0)
    if (n_expert == 1 && k_used == 1 && (!planes || (!pg->sheet_bytes && !pd->sheet_bytes)) && moe_dense_wanted(c)) {
        PlaneRef a{}, b{}, d{};
        if (planes) {
            a = PlaneRef{pg->qs, pg->d, pg->sc, 0, pg->stride}; b = PlaneRef{pu->qs, pu->d, pu->sc, 0, pu->stride};
            d = PlaneRef{pd->qs, pd->d, pd->sc, 0, pd->stride};
        }
        rc = dense_ffn(c, resid, type, down_type, gate_bank, up_bank, down_bank, planes ? &a : nullptr, planes ? &b : nullptr,
                       planes ? &d : nullptr, x, wt, rows, n_ffn, n_embd, g, u, y, st);
        if (rc != JL_DECLINED) return rc;
    }
    const bool gather = c->tune.moe_form == 11 || (c->tune.moe_form == 0 && moe_gather_ffn_wanted(c, type, down_type, planes, rows, k_used, n_expert, n_ffn, n_embd));
    if (gather && planes) {
        rc = moe_planes_gather_ffn(c, resid, pg, pu, pd, x, sel, sel_stride, wt, rows, k_used, n_expert, n_ffn, n_embd, g, u, st);
        if (rc != JL_DECLINED) return rc;
    }
    if (gather && !planes) {
        rc = moe_gather_ffn(c, resid, type, down_type, gate_bank, up_bank, down_bank, x, sel, sel_stride, wt, rows, k_used, n_expert, n_ffn,
                            n_embd, g, u, st);
        if (rc != JL_DECLINED) return rc;
    }
    // (the work lists where a matvec may take the int8 tiles)
    if (planes || ncols < 8 * (size_t)n_expert || (type == JL_TYPE_Q4_K && down_type == JL_TYPE_Q4_K && c->act_window == 256)) w.lists.nslots = 0;
    rc = moe_group_launch(c, sel, sel_stride, rows, k_used, n_expert, start, perm, pos, &w.lists, st);
    if (rc != JL_OK) return rc;
    // gate and up: columns read the routed rows of x
    rc = moe_matvec_launch(c, g, u, type, gate_bank, up_bank, x, nullptr, perm, start, n_expert, (int)ncols, n_ffn, n_embd, st,
                           pg, pu, rows, &w.lists);
    if (rc != JL_OK) return rc;
    // down: the activation of column c is silu(g[c]) * u[c]
    rc = moe_matvec_launch(c, y, nullptr, down_type, down_bank, nullptr, g, u, nullptr, start, n_expert, (int)ncols, n_embd, n_ffn, st,
                           pd, nullptr, 0, &w.lists);
    if (rc != JL_OK) return rc;
    return moe_combine_launch(c, resid, y, wt, sel, sel_stride, pos, rows, k_used, n_embd, (uint32_t)n_expert - 1u, st);
}

// The whole block from the hidden state on: router logits, softmax + top-k, the routed
// feed-forward.  (The three router steps as ONE launch -- the workgroup that stores a token
// group's last logit routes it, the one that routes the last group sorts the pairs -- measured
// slower than the launches it replaces, 117 us a 64-row block against 109: every hand-over inside
// a launch is a device-scope store, an atomic and a device-scope load one after the other, which
// costs what a launch boundary costs.)
int moe_block(jl_ctx* c, float* resid, int type, int down_type, const void* gate_bank, const void* up_bank,
              const void* down_bank, const jl_packed_bank* pg, const jl_packed_bank* pu, const jl_packed_bank* pd,
              int rtype, const void* router, const float* x, int rows, int k_used, int n_expert, int n_ffn, int n_embd,
              uint32_t* sel, float* wt, void* stream) {
    if (rows <= 0 || k_used <= 0 || n_expert <= 0 || n_ffn <= 0 || n_embd <= 0 || !router || !x || !resid)
        return fail(c, JL_ERR_ARG, "moe block: bad operand");
    if (k_used > n_expert) return JL_DECLINED;
    int rc = moe_ffn_check(c, resid, type, down_type, gate_bank, up_bank, down_bank, pg, pu, pd, x, rows, k_used, n_expert, n_ffn, n_embd);
    if (rc != JL_OK) return rc;
    HIP_TRY(c, H->SetDevice(c->device));
    hipStream_t st = pick_stream(c, stream);
    const int sel_stride = k_used + 1;
    auto up256 = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t o_sel = up256((size_t)rows * n_expert * 4), o_wt = o_sel + up256((size_t)rows * sel_stride * 4);
    rc = ws_ensure(c, &c->moe_route_ws, &c->moe_route_ws_bytes, o_wt + up256((size_t)rows * k_used * 4));
    if (rc != JL_OK) return rc;
    float* logits = (float*)c->moe_route_ws;
    if (!sel) sel = (uint32_t*)((char*)c->moe_route_ws + o_sel);
    if (!wt) wt = (float*)((char*)c->moe_route_ws + o_wt);
    rc = jl_moe_logits_dev(c, logits, rtype, router, x, n_expert, n_embd, rows, st);
    if (rc != JL_OK) return rc;
    rc = jl_moe_route_dev(c, logits, rows, n_expert, k_used, sel, sel_stride, wt, st);
    if (rc != JL_OK) return rc;
    return moe_ffn(c, resid, type, down_type, gate_bank, up_bank, down_bank, pg, pu, pd, x, sel, sel_stride, wt, rows, k_used,
                   n_expert, n_ffn, n_embd, st);
}
}  // namespace

int jl_moe_block_dev(jl_ctx* c, float* resid, int type, int down_type, const void* gate_bank, const void* up_bank,
                     const void* down_bank, int router_type, const void* router, const float* x, int rows, int k_used,
                     int n_expert, int n_ffn, int n_embd, uint32_t* sel, float* wt, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!gate_bank || !up_bank || !down_bank) return fail(c, JL_ERR_ARG, "moe block: null bank");
    return moe_block(c, resid, type, down_type, gate_bank, up_bank, down_bank, nullptr, nullptr, nullptr, router_type, router,
                     x, rows, k_used, n_expert, n_ffn, n_embd, sel, wt, stream);
}

int jl_moe_block_packed_dev(jl_ctx* c, float* resid, int type, const jl_packed_bank* gate, const jl_packed_bank* up,
                            const jl_packed_bank* down, int router_type, const void* router, const float* x, int rows,
                            int k_used, int n_expert, int n_ffn, int n_embd, uint32_t* sel, float* wt, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!gate || !up || !down) return fail(c, JL_ERR_ARG, "moe block: null bank");
    return moe_block(c, resid, type, type, nullptr, nullptr, nullptr, gate, up, down, router_type, router, x, rows, k_used,
                     n_expert, n_ffn, n_embd, sel, wt, stream);
}

int jl_moe_ffn_types_dev(jl_ctx* c, float* resid, int type, int down_type, const void* gate_bank, const void* up_bank,
                         const void* down_bank, const float* x, const uint32_t* sel, int sel_stride,
                         const float* wt, int rows, int k_used, int n_expert, int n_ffn, int n_embd, void* stream) {
    return moe_ffn(c, resid, type, down_type, gate_bank, up_bank, down_bank, nullptr, nullptr, nullptr, x, sel, sel_stride, wt,
                   rows, k_used, n_expert, n_ffn, n_embd, stream);
}

int jl_moe_ffn_packed_dev(jl_ctx* c, float* resid, int type, const jl_packed_bank* gate, const jl_packed_bank* up,
                          const jl_packed_bank* down, const float* x, const uint32_t* sel, int sel_stride,
                          const float* wt, int rows, int k_used, int n_expert, int n_ffn, int n_embd, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!gate || !up || !down) return fail(c, JL_ERR_ARG, "moe ffn: null bank");
    return moe_ffn(c, resid, type, type, nullptr, nullptr, nullptr, gate, up, down, x, sel, sel_stride, wt, rows, k_used,
                   n_expert, n_ffn, n_embd, stream);
}

int jl_moe_ffn_dev(jl_ctx* c, float* resid, int type, const void* gate_bank, const void* up_bank,
                   const void* down_bank, const float* x, const uint32_t* sel, int sel_stride,
                   const float* wt, int rows, int k_used, int n_expert, int n_ffn, int n_embd, void* stream) {
    return jl_moe_ffn_types_dev(c, resid, type, type, gate_bank, up_bank, down_bank, x, sel, sel_stride, wt, rows,
                                k_used, n_expert, n_ffn, n_embd, stream);
}

// ------------------------------------------------------------------ the block seam
namespace {
size_t up256(size_t v) { return (v + 255) & ~(size_t)255; }

// Bytes of one matrix (or bank of `sheets` sheets) of a plan: GGUF bytes, or its three planes
// (each rounded up to 256 bytes so that every plane starts aligned).
bool layer_matrix_bytes(int type, int packed, size_t nrows, int k, size_t* total, size_t plane[3]) {
    const TypeInfo* ti = type_info(type);
    if (!ti || k % ti->block_elems) return false;
    if (!packed) {
        *total = nrows * (size_t)(k / ti->block_elems) * ti->block_bytes;
        return true;
    }
    size_t nq, nd, nsc;
    if (nrows > 0x7fffffff || !packed_words(type, nrows, k, &nq, &nd, &nsc)) return false;
    plane[0] = nq * 4; plane[1] = nd * 4; plane[2] = nsc * 4;
    *total = up256(plane[0]) + up256(plane[1]) + up256(plane[2]);
    return true;
}
}  // namespace

int jl_prep_layer(jl_ctx* c, int li, const jl_layer_plan* plan) {
    if (!c) return JL_ERR_ARG;
    if (!plan || li < 0) return fail(c, JL_ERR_ARG, "prep layer: bad argument");
    const jl_layer_plan& P = *plan;
    if (P.n_embd <= 0 || P.n_ffn <= 0 || !P.gate || !P.up || !P.down)
        return fail(c, JL_ERR_ARG, "prep layer %d: missing weights or shape", li);
    const bool moe = P.kind == JL_LAYER_MOE;
    if (P.kind != JL_LAYER_DENSE && !moe) return fail(c, JL_ERR_ARG, "prep layer %d: kind %d", li, P.kind);
    if (moe && (P.n_expert < 1 || P.k_used < 1 || P.k_used > P.n_expert || !P.router))
        return fail(c, JL_ERR_ARG, "prep layer %d: mixture without router or experts", li);
    if (moe && (P.n_expert > 1024 || P.k_used > 16 || P.n_ffn % 256 || P.n_embd % 256)) return JL_DECLINED;
    if (moe && P.norm_w) return JL_DECLINED;
    if (P.packed && P.type != P.down_type && moe) return JL_DECLINED;   // packed banks: one type
    const size_t sheets = moe ? (size_t)P.n_expert : 1;
    size_t bg, bd, pg[3], pd[3];
    if (!layer_matrix_bytes(P.type, P.packed, sheets * P.n_ffn, P.n_embd, &bg, pg) ||
        !layer_matrix_bytes(P.down_type, P.packed, sheets * P.n_embd, P.n_ffn, &bd, pd))
        return JL_DECLINED;   // a type or shape without a kernel
    HIP_TRY(c, H->SetDevice(c->device));
    const size_t o_gate = 0, o_up = up256(bg), o_down = o_up + up256(bg), o_norm = o_down + up256(bd);
    const size_t o_router = o_norm + up256(P.norm_w ? (size_t)P.n_embd * 4 : 0);
    const size_t total = o_router + up256(moe ? (size_t)P.n_expert * P.n_embd * 4 : 0);
    jl_release_layers(c, li, li + 1);
    void* mem = nullptr;
    if (H->Malloc(&mem, total) != hipSuccess) {
        (void)H->GetLastError();
        return JL_DECLINED;   // the block does not fit: it stays on the host
    }
    Layer L;
    L.plan = P;
    L.plan.gate = L.plan.up = L.plan.down = nullptr;
    L.plan.norm_w = L.plan.router = nullptr;
    L.mem = mem;
    char* base = (char*)mem;
    auto fail_free = [&](hipError_t e, const char* what) {
        (void)H->Free(mem);
        return fail(c, JL_ERR_HIP, "prep layer %d: %s: %s", li, what, H->GetErrorString(e));
    };
    auto put = [&](size_t off, const void* src, size_t n) { return H->Memcpy(base + off, src, n, hipMemcpyHostToDevice); };
    hipError_t e = hipSuccess;
    if (!P.packed) {
        if ((e = put(o_gate, P.gate, bg)) != hipSuccess || (e = put(o_up, P.up, bg)) != hipSuccess ||
            (e = put(o_down, P.down, bd)) != hipSuccess)
            return fail_free(e, "weight upload");
        L.gate = base + o_gate; L.up = base + o_up; L.down = base + o_down;
    } else {
        auto put_planes = [&](size_t off, const void* hp, const size_t pl[3], const uint32_t* out[3]) {
            const jl_host_planes* h = (const jl_host_planes*)hp;
            const uint32_t* src[3] = {h->qs, h->d, h->sc};
            for (int i = 0; i < 3; i++) {
                out[i] = (const uint32_t*)(base + off);
                if (pl[i]) {
                    if (!src[i]) return hipErrorInvalidValue;
                    hipError_t ee = put(off, src[i], pl[i]);
                    if (ee != hipSuccess) return ee;
                }
                off += up256(pl[i]);
            }
            return hipSuccess;
        };
        if ((e = put_planes(o_gate, P.gate, pg, L.gp)) != hipSuccess || (e = put_planes(o_up, P.up, pg, L.upl)) != hipSuccess ||
            (e = put_planes(o_down, P.down, pd, L.dp)) != hipSuccess)
            return fail_free(e, "plane upload");
    }
    if (P.norm_w) {
        if ((e = put(o_norm, P.norm_w, (size_t)P.n_embd * 4)) != hipSuccess) return fail_free(e, "norm upload");
        L.norm_w = (const float*)(base + o_norm);
    }
    if (moe) {
        if ((e = put(o_router, P.router, (size_t)P.n_expert * P.n_embd * 4)) != hipSuccess) return fail_free(e, "router upload");
        L.router = (const float*)(base + o_router);
    }
    c->layers[li] = L;
    return JL_OK;
}

int jl_release_layers(jl_ctx* c, int lo, int hi) {
    if (!c) return JL_ERR_ARG;
    bool any = false;
    for (auto it = c->layers.lower_bound(lo); it != c->layers.end() && it->first < hi;) {
        if (!any && !c->no_device) {
            // kernels enqueued by earlier runs may still read the block
            (void)H->SetDevice(c->device);
            (void)H->DeviceSynchronize();
            any = true;
        }
        if (it->second.mem) (void)H->Free(it->second.mem);
        it = c->layers.erase(it);
    }
    return JL_OK;
}

int jl_layer_count(jl_ctx* c) { return c ? (int)c->layers.size() : 0; }

int jl_layer_ffn_dev(jl_ctx* c, int li, const float* h, float* resid, int n, void* stream) {
    if (!c) return JL_ERR_ARG;
    auto it = c->layers.find(li);
    if (it == c->layers.end()) return fail(c, JL_ERR_ARG, "layer %d is not prepared", li);
    if (!h || !resid || n <= 0) return fail(c, JL_ERR_ARG, "layer %d: bad operand", li);
    const Layer& L = it->second;
    const jl_layer_plan& P = L.plan;
    HIP_TRY(c, H->SetDevice(c->device));
    hipStream_t st = pick_stream(c, stream);
    const int E = P.n_embd, F = P.n_ffn;
    jl_packed_bank bg, bu, bd;
    if (P.packed) {
        const int sheets = P.kind == JL_LAYER_MOE ? P.n_expert : 1;
        bg = jl_packed_bank{L.gp[0], L.gp[1], L.gp[2], 0, sheets * F};
        bu = jl_packed_bank{L.upl[0], L.upl[1], L.upl[2], 0, sheets * F};
        bd = jl_packed_bank{L.dp[0], L.dp[1], L.dp[2], 0, sheets * E};
    }
    if (P.kind == JL_LAYER_MOE) {
        return moe_block(c, resid, P.type, P.down_type, L.gate, L.up, L.down, P.packed ? &bg : nullptr, P.packed ? &bu : nullptr,
                         P.packed ? &bd : nullptr, JL_TYPE_F32, L.router, h, n, P.k_used, P.n_expert, F, E, nullptr, nullptr, st);
    }
    // dense, more than one row without a norm in front: as matmuls
    if (n > 1 && !L.norm_w && moe_dense_wanted(c)) {
        MoeWs w;
        int rc = moe_ws(c, n, 1, 1, F, E, &w);
        if (rc != JL_OK) return rc;
        const PlaneRef a = {L.gp[0], L.gp[1], L.gp[2], 0, F}, b = {L.upl[0], L.upl[1], L.upl[2], 0, F}, d = {L.dp[0], L.dp[1], L.dp[2], 0, E};
        rc = dense_ffn(c, resid, P.type, P.down_type, L.gate, L.up, L.down, P.packed ? &a : nullptr, P.packed ? &b : nullptr,
                       P.packed ? &d : nullptr, h, nullptr, n, F, E, w.g, w.u, w.y, st);
        if (rc != JL_DECLINED) return rc;
    }
    // one row at a time: gate and up in one launch (the norm riding in front), down over
    // silu(gate) * up with the residual add riding on it
    const size_t fb = up256((size_t)F * 4);
    int rc = grow(c, &c->layer_ws, &c->layer_ws_bytes, 2 * fb + up256((size_t)E * 4));
    if (rc != JL_OK) return rc;
    float* g = (float*)c->layer_ws;
    float* u = (float*)((char*)c->layer_ws + fb);
    float* y = (float*)((char*)c->layer_ws + 2 * fb);   // down's own rows (resid takes them as they are made)
    for (int r = 0; r < n; r++) {
        const float* hr = h + (size_t)r * E;
        float* rr = resid + (size_t)r * E;
        float* gu[2] = {g, u};
        float* yo[1] = {y};
        if (!P.packed) {
            const void* wgu[2] = {L.gate, L.up};
            const int rgu[2] = {F, F};
            rc = matvec_multi_launch(c, P.type, 2, gu, wgu, rgu, hr, 0, nullptr, nullptr, 0.f, E, st, L.norm_w, P.norm_eps);
            if (rc != JL_OK) return rc;
            const void* wd[1] = {L.down};
            const int rd[1] = {E};
            rc = matvec_multi_launch(c, P.down_type, 1, yo, wd, rd, g, 0, u, rr, 1.0f, F, st);
        } else {
            PlaneRef pgu[2] = {{L.gp[0], L.gp[1], L.gp[2], 0, F}, {L.upl[0], L.upl[1], L.upl[2], 0, F}};
            rc = packed_matvec_multi_launch(c, P.type, 2, gu, pgu, hr, 0, nullptr, nullptr, 0.f, nullptr, L.norm_w,
                                            P.norm_eps, nullptr, F, E, st);
            if (rc != JL_OK) return rc;
            PlaneRef pd1[1] = {{L.dp[0], L.dp[1], L.dp[2], 0, E}};
            rc = packed_matvec_multi_launch(c, P.down_type, 1, yo, pd1, g, 0, u, rr, 1.0f, nullptr, nullptr, 0.f, nullptr,
                                            E, F, st);
        }
        if (rc != JL_OK) return rc;
    }
    return JL_OK;
}

namespace {
// Rows a tile: a round of the CUs takes about 1.36 times as long with 96 (measured at k = 1216 to 4512), so 96 where
// that saves the rounds (2880 rows: 512 tokens 21.1 -> 17.4 us, 384 tokens of 5000 rows 19.7 against 23.7).
double mx_tile_rounds(const jl_ctx* c, int nrows, int ntok, int* trows) {
    auto rounds = [&](int rows) {
        return (double)(((long)((ntok + 63) / 64) * ((nrows + rows - 1) / rows) + c->num_cu - 1) / c->num_cu);
    };
    const double r64 = rounds(64), r96 = 1.36 * rounds(96);
    *trows = c->tune.mx_planes == 3 ? 64 : c->tune.mx_planes == 4 ? 96 : r96 < r64 ? 96 : 64;
    return *trows == 96 ? r96 : r64;
}

// More than a handful of tokens over GGUF rows: tiles of 128 tokens x 128 or 96 rows that read them, K split over
// `split` workgroups of `per` stages, or the smaller tiles of the planes with the rows turned into planes on the way; by
// their costs as measured (us; 1100 x 1216 to 5000 x 2048, 64 to 2048 tokens).  The former: a stage of K = 256 takes 2.15
// with 96 rows and 2.9 with 128, a split a launch and its slabs; the latter: 1 a MB of weights and 2.75 a round and 1024
// of K.
struct MxRowsPlan {
    int trows, split, per;
    double rows_us, planes_us;
};
MxRowsPlan mx_rows_plan(const jl_ctx* c, int nrows, int k, int ntok) {
    MxRowsPlan p;
    const int ttok = (ntok + 127) / 128, stages = (k + 255) / 256;
    // rows per tile: 128, or 96 where that takes fewer rounds x rows (2880 rows x 1024 tokens:
    // 184 tiles of 128 rows leave 72 CUs idle for a whole tile, 240 of 96 rows do not)
    auto cost = [&](int rows) {
        const long t = (long)ttok * ((nrows + rows - 1) / rows);
        return ((t + c->num_cu - 1) / c->num_cu) * rows;
    };
    p.trows = c->tune.mx_rows == 96 || c->tune.mx_rows == 128 ? c->tune.mx_rows : (cost(96) < cost(128) ? 96 : 128);
    const long tiles = (long)ttok * ((nrows + p.trows - 1) / p.trows);
    // A grid that leaves most CUs idle is widened along K: each split writes partial sums
    // to a workspace slab and a second kernel adds the slabs in order.
    long split = c->tune.mx_split > 0 ? c->tune.mx_split : (tiles * 2 <= c->num_cu ? c->num_cu / tiles : 1);
    split = std::min(split, std::min(8L, (long)stages));
    p.per = (int)((stages + split - 1) / split);
    p.split = (stages + p.per - 1) / p.per;   // no empty split
    int mtrows;
    const double rounds = mx_tile_rounds(c, nrows, ntok, &mtrows), mb = 1e-6 * nrows * (double)(k / 32 * 17);
    p.planes_us = 6 + mb + 2.75 * k / 1024 * rounds;
    p.rows_us = 7 + (double)cost(p.trows) / p.trows * p.per * (p.trows == 96 ? 2.15 : 2.9) +
                (p.split > 1 ? 3.5 + (double)ntok * nrows * p.split * 4 / 3e6 : 0);
    return p;
}

// Few tokens: 16-row workgroups whose wavefronts split K, in chunks of up to 64 tokens, one launch after a prep
// that lays the activations out in the order the block decode produces.
// (The same tiles in one launch come first, mx_one_rows.)  From where: the kernels for a handful of tokens grow with the
// tokens, this one does not, but it is two launches, which a host that issues calls one after the other cannot do in less
// than 6.7 us.  From three tokens, so, where the one launch is estimated to take more than that and more than this form:
// over rows a token costs what a round of their workgroups does, four rows each, on all CUs, over planes what K and the
// matrix do (fitted to 17 shapes, 512 x 512 to 12288 x 2048,
// 2 to 8 tokens, 6 % each).  Device us, these against this one: rows 2880 x 2880, 3 and 5 tokens 6.5 and 6.8, 8.9 and 6.9,
// 5760 x 2880, 3 tokens 11.3 and 9.3; planes 5760 x 2880, 3 tokens 9.1 and 7.0, 3413 x 1536, 5 and 8 tokens 6.0 and 5.4,
// 7.5 and 5.4.  (By device time alone it would begin earlier: planes 2124 x 1120, 5 tokens 5.5 and 4.7, but call by call
// 5.4 and 6.8.)
// Up to where: 64 tokens are one chunk.  More, up to 128 tokens, or 256 while the chunks are one round of the CUs: over
// rows while that is estimated faster than the tiles -- 4 and 0.48 a token tile and 1024 of K for each round, a tenth
// more with several chunks (2880 x 2880, 128 tokens 16.3 against 17.8; 2880 x 14336, 80 tokens 46 against 28, 5760 x 5760,
// 128 tokens 35 against 27, 512 x 8192, 128 tokens 24.2 against 20.5 for the tiles) --, over planes, whose tiles have
// no rows to turn, only while they are one round (2880 x 2880, 96 tokens 13.0 against 12.8; 512 x 8192, 256 tokens 20.7
// against 24.5; K slices over rows restored from the planes are no match for either: 2880 x 14336, 96 tokens 57 against 36).
bool mx_few_applies(const jl_ctx* c, int nrows, int k, int ntok, bool planes) {
    if (c->tune.mx_rows == 96 || c->tune.mx_rows == 128 || ntok > 65535) return false;
    const int form = c->tune.mx_planes;
    if (form == 3 || form == 4 || (planes && (form == 2 || (form && ntok <= 8)))) return false;
    if (c->tune.mx_few_min > 0) {
        if (ntok < c->tune.mx_few_min) return false;
    } else if (ntok <= 8) {
        const long r4 = ((nrows + 3) / 4 + (long)c->num_cu - 1) / c->num_cu, r16 = ((nrows + 15) / 16 + (long)c->num_cu - 1) / c->num_cu;
        const double one = planes ? 3.25 + ntok * (0.04 + 0.17e-3 * k + 0.062e-6 * nrows * k) : 2 + ntok * (0.1 + 0.13e-3 * k * r4);
        const double two = 3.85 + (planes ? 0.61e-3 : 0.95e-3) * k * r16;
        if (ntok < 3 || one < std::max(6.7, two)) return false;
    }
    if (c->tune.mx_few > 0) return ntok <= c->tune.mx_few;
    if (ntok <= 64) return true;
    const int tiles = (ntok + 15) / 16, chunks = (tiles + 3) / 4, nt = (tiles + chunks - 1) / chunks;
    const long wgs = (long)((nrows + 15) / 16) * ((tiles + nt - 1) / nt), rounds = (wgs + c->num_cu - 1) / c->num_cu;
    if (ntok > 256 || (rounds > 1 && (planes || ntok > 128))) return false;
    if (planes) return true;
    const MxRowsPlan p = mx_rows_plan(c, nrows, k, ntok);
    return 1.1 * (4 + 0.48e-3 * k * nt * rounds) < std::min(p.rows_us, p.planes_us);
}
// The same tiles in one launch that takes the activations as they lie (mx_one_body): how many row tiles a workgroup owns, 0: another
// form.  Its workgroups bring all activations to their CU, so one of more row tiles is worth it where it saves a round; where LDS
// (128 KB from five units of 16 tokens x 1024 of K on) leaves a CU one workgroup, a started round counts whole.  us, fitted to 12
// shapes, 512 x 512 to 12288 x 2048, 2 to 256 tokens (rows 5 %, planes 8), beside what else serves: two launches 5 to 5.8 and a slope, a
// decode matvec a token over rows, tiles.  Two launches -> one: 2880 x 2880 rows, 3 / 16 / 64 tokens 7.5 -> 6.4, 8.2 -> 6.6, 11.0 ->
// 10.0, planes 8.0 -> 5.7, 7.4 -> 5.9, 10.3 -> 9.2; 5760 x 5760 planes, 16 and 64 tokens 12.5 -> 9.9, 21.3 -> 15.6; 1024 x 1024, 16
// tokens 6.2 -> 3.9.  More than 64 tokens while the chunks are one round: 2880 x 2880 rows, 128 tokens 18.0 -> 13.0; two
// rounds lose (5305 x 3520 planes, 128 tokens 16.8 against 21.2).  Two launches stay where the rounds are several and full: 12288 x 2048
// rows, 64 tokens 16.2 against 17.3.
double mx_one_us(const jl_ctx* c, int nrows, int k, int ntok, bool planes, int rt, double* rounds) {
    const int tiles = (ntok + 15) / 16, chunks = (tiles + 3) / 4, nt = (tiles + chunks - 1) / chunks;
    const double wgs = (double)((nrows + 16 * rt - 1) / (16 * rt)) * ((tiles + nt - 1) / nt), full = wgs / c->num_cu, kk = k / 1024.0;
    const bool two = 2 * JL_MX_ONE_LDS(k, nt) <= 160 * 1024;   // workgroups a CU
    *rounds = two ? std::max(1.0, full) : std::ceil(full);
    const double us = planes ? 2.4 + *rounds * (rt == 1 ? 1.1 + kk * (0.62 + 0.4 * (nt - 1)) : 1.0 + kk * (1.0 + 0.435 * (nt - 1)))
                             : rt == 1 ? 2.6 + *rounds * (0.3 + kk * (1.2 + 0.385 * (nt - 1))) : 3.2 + *rounds * (kk * (2.03 + 0.46 * (nt - 1)) - 0.4);
    return !two && full > 1 ? 1.15 * us : us;
}
int mx_one_rows(const jl_ctx* c, int nrows, int k, int ntok, bool planes) {
    const int form = c->tune.mx_one, tiles = (ntok + 15) / 16, chunks = (tiles + 3) / 4, nt = (tiles + chunks - 1) / chunks;
    // (a lane's place among the activations is 32 bits)
    if (form == 1 || ntok < 2 || chunks > 65535 || (size_t)ntok * k >= ((size_t)1 << 31) || (unsigned)JL_MX_ONE_LDS(k, nt) > c->lds_limit) return 0;
    if (form == 11 || form == 12) return form - 10;
    const int pf = c->tune.mx_planes;
    if (c->tune.mx_rows || c->tune.mx_split || c->tune.mx_few > 0 || c->tune.mx_few_min > 0 || pf == 3 || pf == 4) return 0;
    if (planes && (pf == 2 || (pf && ntok <= 8))) return 0;
    double r1, r2;
    const double us1 = mx_one_us(c, nrows, k, ntok, planes, 1, &r1), us2 = mx_one_us(c, nrows, k, ntok, planes, 2, &r2);
    const double us = std::min(us1, us2), kk = k / 1024.0;
    const int rt = us1 <= us2 ? 1 : 2;
    double other;
    if (ntok <= 8 && !mx_few_applies(c, nrows, k, ntok, planes)) {
        if (planes) {
            // Two tokens over many rows: the plane matvec's rounds of 64 rows a workgroup (fitted to 16384 x 1024 to 201088 x 2880, 5 % where it
            // decides), where LDS leaves this form one workgroup a CU.  us, matvec / so: 32768 x 2880 19.6 / 21.3, 65536 x 2880 36.5 / 40.2, 201088 x
            // 2880 100 / 123; 28672 x 4096 26.4 / 25.7, 14336 x 4096 15.2 / 14.1, 8448 x 8192 30.4 / 19.0, 512 x 14336 13.3 / 9.7, and with two
            // workgroups a CU 65536 x 2048 27.6 / 22.0.  From three tokens on this form is never behind (65536 x 2880 44.9 / 40.8).  No guard for long
            // rows: it rounds less at every K (NMSE, 8 tokens, 1024 x 5760 2.7e-15, the matvec 4.6e-15, 4096 x 14336 4.4e-15, 6.5e-15).
            const long r64 = (nrows + 63) / 64;
            if (ntok > 2 || 2 * JL_MX_ONE_LDS(k, nt) <= 160 * 1024 || r64 * 10 < c->num_cu * 7) return rt;
            const double full64 = (double)r64 / c->num_cu;
            return us <= 2.5 + 3.0 * kk * (full64 < 2 ? std::ceil(full64) : 0.5 * (full64 + std::ceil(full64))) ? rt : 0;
        }
        if (k > 4096) return 0;   // (the decode matvec rounds less there: 5760 x 5760, NMSE 2.35e-15 against 2.61)
        const long r4 = ((nrows + 3) / 4 + (long)c->num_cu - 1) / c->num_cu;
        other = (3.2 + ntok * (0.1 + 0.13e-3 * k * r4)) / 1.08;
    } else {
        const double full = std::max(1.0, (double)((nrows + 15) / 16) * ((tiles + nt - 1) / nt) / c->num_cu), r = 0.5 * (full + std::ceil(full));
        const double two = planes ? 5.8 + r * kk * (0.63 + 0.31 * (nt - 1)) : 5.0 + r * kk * (1.21 + 0.31 * (nt - 1));
        other = two;
        if (ntok > 64) {
            if ((rt == 1 ? r1 : r2) > 1) return 0;
            int trows;
            const MxRowsPlan p = mx_rows_plan(c, nrows, k, ntok);
            other = planes ? 6 + 2.75 * kk * mx_tile_rounds(c, nrows, ntok, &trows) : std::min(p.rows_us, p.planes_us);
            if (mx_few_applies(c, nrows, k, ntok, planes)) other = std::min(other, two);
        }
    }
    return us < other ? rt : 0;
}
int mx_one_launch(jl_ctx* c, MxGemmArgs& a, int rt, hipStream_t st) {
    const int tiles = (a.ntok + 15) / 16, chunks = (tiles + 3) / 4, nt = (tiles + chunks - 1) / chunks;
    const unsigned lds = JL_MX_ONE_LDS(a.k, nt);
    void* params[] = {&a};
    Name name;
    name << "jl_mxfp4_one_" << (a.qs ? "planes_t" : "t") << nt << 'r' << rt;
    return launch(c, name, (unsigned)((a.nrows + 16 * rt - 1) / (16 * rt)), (unsigned)((tiles + nt - 1) / nt), 512, lds, st, params);
}
int mx_few_launch(jl_ctx* c, MxGemmArgs& a, const uint16_t* x, hipStream_t st) {
    const int tiles = (a.ntok + 15) / 16, groups = (a.k + 127) / 128, chunks = (tiles + 3) / 4, nt = (tiles + chunks - 1) / chunks;
    int rc = gemm_ws_ensure(c, (size_t)groups * 4 * tiles * 1024);
    if (rc != JL_OK) return rc;
    MxPrepArgs pa;
    pa.x = x; pa.xf = (uint16_t*)c->gemm_ws; pa.ntok = a.ntok; pa.tok_pad = 16 * tiles; pa.k = a.k;
    void* pp[] = {&pa};
    rc = launch(c, "jl_mxfp4_prep_few", (unsigned)groups, (unsigned)tiles, 256, 0, st, pp);
    if (rc != JL_OK) return rc;
    a.x = (const uint16_t*)c->gemm_ws; a.tok_pad = 16 * tiles;
    void* params[] = {&a};
    Name name;
    name << "jl_mxfp4_few_" << (a.qs ? "planes_" : "") << (chunks > 1 ? 'c' : 't') << nt;
    return launch(c, name, (unsigned)((a.nrows + 15) / 16), (unsigned)((tiles + nt - 1) / nt), 512, 0, st, params);
}
// Tiles of 64 tokens x 64 or 96 rows whose wavefronts split K, the weights taken from planes; rows (w) are turned
// into planes in the workspace by the launch that lays the activations out.
size_t mx_tile_xa_bytes(int k, int ntok) { return (size_t)((k + 63) / 64) * ((ntok + 63) / 64 * 2) * 4 * 1024; }
// rows turned into planes: codes and exponents of rows in whole runs of 64
size_t mx_tile_plane_bytes(int nrows, int k) { return (size_t)(k / 32) * 17 * ((nrows + 63) / 64 * 64); }
int mx_tile_launch(jl_ctx* c, MxPlanesGemmArgs& a, const uint8_t* w, const uint16_t* x, hipStream_t st) {
    const int tok_pad = (a.ntok + 63) / 64 * 64, nks = (a.k + 63) / 64, ntt = tok_pad / 32, nblk = a.k / 32;
    int trows;
    (void)mx_tile_rounds(c, a.nrows, a.ntok, &trows);
    const long tiles = (long)(tok_pad / 64) * ((a.nrows + trows - 1) / trows), stride = (a.nrows + 63) / 64 * 64;
    const long nx = (long)((nks + 3) / 4) * ntt, nw = w ? (stride / 64) * ((nblk + 15) / 16) : 0;
    if (tiles > 0x7fffffffL / 2 || nx + nw > 0x7fffffffL) return JL_DECLINED;
    const size_t xa_bytes = mx_tile_xa_bytes(a.k, a.ntok), qs_bytes = (size_t)nblk * 16 * stride;
    int rc = gemm_ws_ensure(c, xa_bytes + (w ? mx_tile_plane_bytes(a.nrows, a.k) : 0));
    if (rc != JL_OK) return rc;
    MxPlanesPrepArgs pa;
    pa.x = x; pa.xa = (uint32_t*)c->gemm_ws; pa.ntok = a.ntok; pa.tok_pad = tok_pad; pa.k = a.k;
    if (w) {
        pa.w = w; pa.qs = (uint32_t*)((char*)c->gemm_ws + xa_bytes); pa.d = (uint32_t*)((char*)pa.qs + qs_bytes);
        pa.nrows = a.nrows; pa.stride = (int)stride;
        a.qs = pa.qs; a.d = pa.d; a.row0 = 0; a.stride = (int)stride;
    }
    void* pp[] = {&pa};
    rc = launch(c, "jl_mxfp4_planes_prep", (unsigned)(nx + nw), 1, 256, 0, st, pp);
    if (rc != JL_OK) return rc;
    a.xa = pa.xa; a.tok_pad = tok_pad;
    void* gp[] = {&a};
    return launch(c, trows == 96 ? "jl_mxfp4_planes_gemm_r96" : "jl_mxfp4_planes_gemm", (unsigned)(8 * ((tiles + 7) / 8)), 1, 256, (unsigned)(trows / 32 * 16384), st, gp);
}
}  // namespace

int jl_matmul_mxfp4_bf16_dev(jl_ctx* c, float* out, const void* w, const uint16_t* x, int nrows, int k,
                             int ntok, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (!out || !w || !x || nrows <= 0 || k <= 0 || ntok <= 0)
        return fail(c, JL_ERR_ARG, "mxfp4 matmul: bad operand");
    if (k % 32 != 0 || k < 32 || !aligned16(x) || (k % 8) != 0) return JL_DECLINED;
    if ((size_t)(k / 32) * 17 > 0x7fffffffu || ntok > 65535 * 128) return JL_DECLINED;
    HIP_TRY(c, H->SetDevice(c->device));
    MxGemmArgs a;
    a.out = out; a.w = (const uint8_t*)w; a.x = x;
    a.nrows = nrows; a.k = k; a.ntok = ntok; a.row_bytes = (k / 32) * 17;
    a.nsplit = 1; a.part = nullptr; a.tok_pad = 0;
    void* params[] = {&a};
    hipStream_t st = pick_stream(c, stream);
    if (ntok == 1 && k <= 3 * 2048 && c->tune.mx_rows != 1) {
        // one token: the activation stays in registers while a wavefront walks its rows
        const int nbi = (k / 32 + 63) / 64;
        Name name;
        name << "jl_mxfp4_matvec1_b" << nbi;
        // (a wavefront a workgroup: four wavefronts a workgroup of four rows each were 180 workgroups for
        // 2880 rows and left 76 CUs without one: 4.65 -> 4.18 us)
        return launch(c, name, (unsigned)((nrows + JL_MX1_RPW - 1) / JL_MX1_RPW), 1, 64, 0, st, params);
    }
    if (const int rt = mx_one_rows(c, nrows, k, ntok, false)) return mx_one_launch(c, a, rt, st);
    if (mx_few_applies(c, nrows, k, ntok, false)) return mx_few_launch(c, a, x, st);
    if (ntok <= 8)  // a handful of tokens: stream the rows once, no tile to fill
        return launch(c, "jl_mxfp4_matvec", (unsigned)((nrows + 3) / 4), 1, 256, 0, st, params);
    // activations into matrix-fragment order (tokens padded to whole tiles, K to whole stages)
    const int tok_pad = (ntok + 127) / 128 * 128, stages = (k + 255) / 256;
    const MxRowsPlan plan = mx_rows_plan(c, nrows, k, ntok);
    const int trows = plan.trows, nsplit = plan.split;
    const char* gemm_name = trows == 96 ? "jl_mxfp4_gemm_r96" : "jl_mxfp4_gemm";
    // (the estimates are good to about 8 %, so planes only where they win by more: 2880 x 2880, 512 tokens 27.9 -> 21.8,
    // 1024 tokens 31.5 against 32.3, 2048 tokens 57 -> 52)
    const unsigned lds = 2u * 128u * 264u * 2u;   // two weight stages [128][264] bf16
    // (the planes of a reserved call have to fit what is there; jl_reserve_shape, a dry run, makes them room)
    const bool room = !reserved_for(c, ntok, k) || call_dry_run(c) || mx_tile_xa_bytes(k, ntok) + mx_tile_plane_bytes(nrows, k) <= c->gemm_ws_bytes;
    if (c->tune.mx_planes == 3 || c->tune.mx_planes == 4 || lds > c->lds_limit ||
        (room && !c->tune.mx_rows && !c->tune.mx_split && 1.08 * plan.planes_us < plan.rows_us)) {
        MxPlanesGemmArgs ga;
        ga.out = out; ga.nrows = nrows; ga.k = k; ga.ntok = ntok;
        return mx_tile_launch(c, ga, (const uint8_t*)w, x, st);
    }
    int rc = gemm_ws_ensure(c, (size_t)stages * (tok_pad / 32) * 16 * 1024);
    if (rc != JL_OK) return rc;
    MxPrepArgs pa;
    pa.x = x; pa.xf = (uint16_t*)c->gemm_ws; pa.ntok = ntok; pa.tok_pad = tok_pad; pa.k = k;
    void* pp[] = {&pa};
    rc = launch(c, "jl_mxfp4_prep", (unsigned)stages, (unsigned)(tok_pad / 32), 256, 0, st, pp);
    if (rc != JL_OK) return rc;
    a.x = (const uint16_t*)c->gemm_ws; a.tok_pad = tok_pad;
    if (nsplit > 1) {
        const size_t n = (size_t)ntok * nrows;
        rc = ws_ensure(c, &c->mx_ws, &c->mx_ws_bytes, n * nsplit * 4);
        if (rc != JL_OK) return rc;
        a.nsplit = nsplit; a.part = (float*)c->mx_ws;
        rc = launch(c, gemm_name, (unsigned)(tok_pad / 128), (unsigned)((nrows + trows - 1) / trows), 512, lds, st,
                    params, (unsigned)nsplit);
        if (rc != JL_OK) return rc;
        SumPartsArgs sa;
        sa.out = out; sa.part = a.part; sa.n = n; sa.nsplit = nsplit;
        void* sp[] = {&sa};
        return launch(c, "jl_sum_parts", (unsigned)((n + 255) / 256), 1, 256, 0, st, sp);
    }
    return launch(c, gemm_name, (unsigned)(tok_pad / 128), (unsigned)((nrows + trows - 1) / trows), 512,
                  lds, st, params);
}

int jl_matmul_mxfp4_packed_bf16_dev(jl_ctx* c, float* out, const uint32_t* qs, const uint32_t* d, int row,
                                    int stride, const uint16_t* x, int nrows, int k, int ntok, void* stream) {
    if (!c) return JL_ERR_ARG;
    const PlaneRef pl = {qs, d, nullptr, row, stride};
    int rc = mx_planes_check(c, pl, nrows, k);
    if (rc != JL_OK) return rc;
    if (!out || !x || ntok <= 0) return fail(c, JL_ERR_ARG, "mxfp4 packed matmul: bad operand");
    if (!aligned16(x)) return JL_DECLINED;
    HIP_TRY(c, H->SetDevice(c->device));
    hipStream_t st = pick_stream(c, stream);
    if (c->tune.mx_scaled == 1) {
        // opt-in: activations to MX fp8, the planes' codes and exponents straight into the
        // block-scaled matrix instruction (about three bits of every activation are lost)
        if (ntok > 65535 * 32 || k % 8 != 0) return JL_DECLINED;
        const int tok_pad = (ntok + 127) / 128 * 128, nks = (k + 63) / 64, ntt = tok_pad / 32;
        const size_t xa_bytes = (size_t)nks * ntt * 64 * 32;
        rc = gemm_ws_ensure(c, xa_bytes + (size_t)nks * ntt * 64);
        if (rc != JL_OK) return rc;
        MxScaledPrepArgs pa;
        pa.x = x; pa.xa = (uint32_t*)c->gemm_ws; pa.xs = (uint8_t*)c->gemm_ws + xa_bytes;
        pa.ntok = ntok; pa.tok_pad = tok_pad; pa.k = k;
        void* pp[] = {&pa};
        rc = launch(c, "jl_mxfp4_scaled_prep", (unsigned)((nks + 3) / 4), (unsigned)ntt, 256, 0, st, pp);
        if (rc != JL_OK) return rc;
        MxScaledGemmArgs ga;
        ga.out = out; ga.qs = qs; ga.d = d; ga.xa = pa.xa; ga.xs = pa.xs;
        ga.nrows = nrows; ga.k = k; ga.ntok = ntok; ga.tok_pad = tok_pad; ga.row0 = row; ga.stride = stride;
        void* gp[] = {&ga};
        if (65536u > c->lds_limit) return JL_DECLINED;
        const long stiles = (long)(tok_pad / 64) * ((nrows + 63) / 64);
        if (stiles > 0x7fffffffL / 2) return JL_DECLINED;
        return launch(c, "jl_mxfp4_scaled_gemm", (unsigned)(8 * ((stiles + 7) / 8)), 1, 256, 65536, st, gp);
    }
    const int one = mx_one_rows(c, nrows, k, ntok, true);
    if (one || mx_few_applies(c, nrows, k, ntok, true)) {
        MxGemmArgs a;
        a.out = out; a.w = nullptr; a.x = x; a.nrows = nrows; a.k = k; a.ntok = ntok; a.row_bytes = 0;
        a.nsplit = 1; a.part = nullptr; a.tok_pad = 0;
        a.qs = qs; a.d = d; a.row0 = row; a.stride = stride;
        if (one) return mx_one_launch(c, a, one, st);
        return mx_few_launch(c, a, x, st);
    }
    if (ntok <= 8 && (c->tune.mx_planes < 2 || c->tune.mx_planes > 4)) {
        // a handful of tokens: the planes are read where they lie, a lane a row
        MxPlanesArgs a;
        a.out = out; a.qs = qs; a.d = d; a.x = (const uint32_t*)x;
        a.nrows = nrows; a.k = k; a.ntok = ntok; a.row0 = row; a.stride = stride;
        a.nwaves = k / 32 < 16 ? k / 32 : 16;
        // rows a workgroup: 64 when that fills the CUs, else 32 or 16 (more, smaller workgroups)
        int rl = c->tune.mx_planes == 64 || c->tune.mx_planes == 32 || c->tune.mx_planes == 16 ? c->tune.mx_planes : 0;
        // (measured: 2880 rows 5.4 us at 16 against 6.8 at 64; 5760 rows 6.3 at 32 against 7.1 and 8.6)
        if (!rl) rl = (nrows + 63) / 64 * 10 >= c->num_cu * 7 ? 64 : ((nrows + 31) / 32 * 10 >= c->num_cu * 7 ? 32 : 16);
        Name name;
        name << "jl_mxfp4_matvec_planes_r" << rl;
        void* params[] = {&a};
        return launch(c, name, (unsigned)((nrows + rl - 1) / rl), 1, (unsigned)(64 * a.nwaves),
                      (unsigned)(a.nwaves * 8 * 64 * 4), st, params);
    }
    // the planes feed the matrix instruction's weight operand as they lie (a plane word is a lane's eight K values)
    if (c->tune.mx_planes != 2 && ntok <= 65535 * 32 && 49152u <= c->lds_limit) {
        MxPlanesGemmArgs ga;
        ga.out = out; ga.qs = qs; ga.d = d; ga.nrows = nrows; ga.k = k; ga.ntok = ntok; ga.row0 = row; ga.stride = stride;
        return mx_tile_launch(c, ga, nullptr, x, st);
    }
    // (asked for by tuning) the forms over GGUF rows: the rows are restored first
    rc = ws_ensure(c, &c->unpack_ws, &c->unpack_ws_bytes, (size_t)nrows * (size_t)(k / 32) * 17);
    if (rc != JL_OK) return rc;
    rc = unpack_launch(c, JL_TYPE_MXFP4, pl, nrows, k, c->unpack_ws, st);
    if (rc != JL_OK) return rc;
    return jl_matmul_mxfp4_bf16_dev(c, out, c->unpack_ws, x, nrows, k, ntok, st);
}

/* ------------------------------------------------------- host-pointer seam */

namespace {
// The three planes of a matrix in host memory as ONE device allocation keyed on the QS pointer
// (uploaded on first use, jl_forget over the QS pointer releases it).  Called with c->mu held.
int resident_planes(jl_ctx* c, int type, const PlaneRef& host, int k, PlaneRef* pl) {
    size_t nq, nd, nsc;
    if (!packed_words(type, (size_t)host.stride, k, &nq, &nd, &nsc)) return JL_DECLINED;
    auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t o_d = up(nq * 4), o_sc = o_d + up(nd * 4), total = o_sc + up(nsc * 4);
    void* dev = nullptr;
    auto it = c->resident.find(host.qs);
    if (it != c->resident.end() && it->second.bytes == total) {
        dev = it->second.dev;
    } else {
        if (it != c->resident.end()) {
            HIP_TRY(c, H->Free(it->second.dev));
            c->resident.erase(it);
        }
        HIP_TRY(c, H->Malloc(&dev, total));
        hipError_t e = H->Memcpy(dev, host.qs, nq * 4, hipMemcpyHostToDevice);
        if (e == hipSuccess) e = H->Memcpy((char*)dev + o_d, host.d, nd * 4, hipMemcpyHostToDevice);
        if (e == hipSuccess && nsc) e = H->Memcpy((char*)dev + o_sc, host.sc, nsc * 4, hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            (void)H->Free(dev);
            return fail(c, JL_ERR_HIP, "plane upload: %s", H->GetErrorString(e));
        }
        c->resident[host.qs] = Resident{dev, total};
    }
    *pl = PlaneRef{(const uint32_t*)dev, (const uint32_t*)((char*)dev + o_d), (const uint32_t*)((char*)dev + o_sc),
                   host.row, host.stride};
    return JL_OK;
}

// ---- a host-pointer call's operands and results.  Up to kPinMost bytes each way they go through pinned host
// memory that kernels read and write in stream order, and the calling thread watches the word jl_host_done
// raises behind them: no copy and no wait through the runtime, whose cost is latency (Q6_K 4096 x 4096 matvec
// of 4.9 us on the device: 31 us a call with copies).  More than that, and whenever pinned memory is not to be
// had, is copied.  Called with c->mu held, in this order: host_io_begin, stage_in for every operand,
// host_io_go, the launches (which write the results to host_results()), host_out for every result, host_io_end.
constexpr size_t kPinMost = (size_t)1 << 20;
struct HostIo {
    bool pinned = false;
    size_t in_bytes = 0, out_bytes = 0;
    struct Out { float* dst; size_t off, n; };
    std::vector<Out> outs;
};
thread_local HostIo g_io;

// Pinned memory of `need` bytes; *ok stays false where there is none to be had.
int host_pin(jl_ctx* c, size_t need, bool* ok) {
    if (!c->pin_flag) {
        void* f = nullptr;
        if (H->HostMalloc(&f, 256, hipHostMallocCoherent) != hipSuccess) { (void)H->GetLastError(); return JL_OK; }
        memset(f, 0, 256);
        c->pin_flag = (volatile uint32_t*)f;
    }
    if (c->pin_bytes < need) {   // (nothing of an earlier call is in flight: each ends when its results are in)
        if (c->pin) {
            HIP_TRY(c, H->StreamSynchronize(c->stream));
            (void)H->HostFree(c->pin);
        }
        c->pin = nullptr;
        c->pin_bytes = 0;
        size_t want = (size_t)64 << 10;
        while (want < need) want <<= 1;
        if (H->HostMalloc(&c->pin, want, hipHostMallocCoherent) != hipSuccess) {
            (void)H->GetLastError();
            c->pin = nullptr;
            return JL_OK;
        }
        c->pin_bytes = want;
    }
    *ok = true;
    return JL_OK;
}

// Device staging for in_floats of operands (c->stage_x), a place for out_floats of results: pinned memory for
// both, or device staging (c->stage_out).
int host_io_begin(jl_ctx* c, size_t in_floats, size_t out_floats) {
    HostIo& io = g_io;
    io.outs.clear();
    io.in_bytes = (in_floats * 4 + 255) & ~(size_t)255;
    io.out_bytes = (out_floats * 4 + 255) & ~(size_t)255;
    io.pinned = false;
    int rc = ensure_stage(c, &c->stage_x, &c->stage_x_bytes, io.in_bytes);
    if (rc != JL_OK) return rc;
    if (io.in_bytes <= kPinMost && io.out_bytes <= kPinMost && (rc = host_pin(c, io.in_bytes + io.out_bytes, &io.pinned)) != JL_OK) return rc;
    return io.pinned ? JL_OK : ensure_stage(c, &c->stage_out, &c->stage_out_bytes, io.out_bytes);
}

float* host_results(jl_ctx* c) { return g_io.pinned ? (float*)((char*)c->pin + g_io.in_bytes) : (float*)c->stage_out; }
// Host floats -> the staging buffer at a float offset.
int stage_in(jl_ctx* c, size_t off, const float* src, size_t n) {
    if (g_io.pinned) {
        memcpy((float*)c->pin + off, src, n * 4);
        return JL_OK;
    }
    HIP_TRY(c, H->MemcpyAsync((float*)c->stage_x + off, src, n * 4, hipMemcpyHostToDevice, c->stream));
    return JL_OK;
}

// The operands, where the launches find them.  read_once: every launch reads an operand's words once (the
// activation prep of a matmul), so they can stay where the caller's were put; a decode matvec reads its
// activation in every workgroup.
int host_io_go(jl_ctx* c, const float** operands, bool read_once = false) {
    *operands = g_io.pinned && read_once ? (const float*)c->pin : (const float*)c->stage_x;
    if (!g_io.pinned || read_once) return JL_OK;
    const void* src = c->pin;
    void* dst = c->stage_x;
    uint32_t n = (uint32_t)(g_io.in_bytes / 16);
    void* pp[] = {&src, &dst, &n};
    return launch(c, "jl_host_in", std::min(64u, (n + 255) / 256), 1, 256, 0, c->stream, pp, 1, false);
}

// A result that is updated in place in device memory (16-byte aligned, n rounded up to four floats readable).
int host_result_copy(jl_ctx* c, size_t off, const float* src, size_t n) {
    void* dst = host_results(c) + off;
    uint32_t n4 = (uint32_t)((n + 3) / 4);
    void* pp[] = {(void*)&src, &dst, &n4};
    return launch(c, "jl_host_in", std::min(64u, (n4 + 255) / 256), 1, 256, 0, c->stream, pp, 1, false);
}
// A result: n floats at a float offset of host_results().
void host_out(size_t off, float* dst, size_t n) { g_io.outs.push_back({dst, off, n}); }

// Waits for the call's results and hands them over.  On an error of the call's (rc): waits for the stream.
int host_io_end(jl_ctx* c, int rc) {
    HostIo& io = g_io;
    if (rc == JL_OK && io.pinned) {
        uint32_t number = ++c->pin_number;
        uint32_t* flag = (uint32_t*)c->pin_flag;
        void* pp[] = {&flag, &number};
        rc = launch(c, "jl_host_done", 1, 1, 64, 0, c->stream, pp, 1, false);
        if (rc == JL_OK) {
            // watch the word for a few milliseconds, then leave the wait (and any error) to the runtime
            bool seen = false;
            for (int i = 0; i < 200000 && !(seen = __atomic_load_n(flag, __ATOMIC_ACQUIRE) == number); i++) __builtin_ia32_pause();
            if (!seen) HIP_TRY(c, H->StreamSynchronize(c->stream));
            const float* r = host_results(c);
            for (const HostIo::Out& o : io.outs) memcpy(o.dst, r + o.off, o.n * 4);
            return JL_OK;
        }
    }
    if (rc == JL_OK)
        for (const HostIo::Out& o : io.outs)
            HIP_TRY(c, H->MemcpyAsync(o.dst, (const float*)c->stage_out + o.off, o.n * 4, hipMemcpyDeviceToHost, c->stream));
    hipError_t e = H->StreamSynchronize(c->stream);
    if (rc == JL_OK && e != hipSuccess) return fail(c, JL_ERR_HIP, "stream: %s", H->GetErrorString(e));
    return rc;
}
size_t up64(size_t n) { return (n + 63) & ~(size_t)63; }   // floats: keeps every staged vector 256-byte aligned
}  // namespace

int jl_matvec(jl_ctx* c, float* out, int type, const void* w, size_t wbytes, const float* x,
              int nrows, int k) {
    return jl_matmul(c, out, type, w, wbytes, x, nrows, k, 1);
}

int jl_matmul(jl_ctx* c, float* out, int type, const void* w, size_t wbytes, const float* x,
              int nrows, int k, int ntok) {
    if (!c) return JL_ERR_ARG;
    CtxLock lock(c);
    drain_forget(c);
    if (c->no_device) return fail(c, JL_ERR_HIP, "this context is bound to no device");
    const TypeInfo* ti = nullptr;
    int rc = matvec_check(c, type, nrows, k, &ti);
    if (rc != JL_OK) return rc;
    if (!out || !w || !x || ntok <= 0) return fail(c, JL_ERR_ARG, "matmul: bad operand");
    size_t need = (size_t)nrows * (size_t)(k / ti->block_elems) * ti->block_bytes;
    if (wbytes < need)
        return fail(c, JL_ERR_ARG, "matmul: weight has %zu bytes, %dx%d needs %zu", wbytes, nrows, k, need);
    HIP_TRY(c, H->SetDevice(c->device));
    void* wd = nullptr;
    rc = resident_weight(c, w, need, &wd);
    if (rc != JL_OK) return rc;
    const size_t nx = (size_t)ntok * k, no = (size_t)ntok * nrows;
    if ((rc = host_io_begin(c, nx, no)) != JL_OK) return rc;
    rc = stage_in(c, 0, x, nx);
    const float* xd = nullptr;
    if (rc == JL_OK) rc = host_io_go(c, &xd, few_applies(c, type, false, nrows, k, ntok, 0) && !tokens_matvec_wanted(c, type, false, nrows, k, ntok, 0));
    if (rc == JL_OK) rc = matmul_launch(c, host_results(c), type, wd, xd, nrows, k, ntok, c->stream);
    host_out(0, out, no);
    return host_io_end(c, rc);
}

int jl_matvec_packed(jl_ctx* c, float* out, int type, const uint32_t* qs, const uint32_t* d,
                     const uint32_t* sc, int row, int stride, const float* x, int nrows, int k) {
    return jl_matmul_packed(c, out, type, qs, d, sc, row, stride, x, nrows, k, 1);
}

int jl_matvec_packed_multi(jl_ctx* c, float* const* outs, int type, const uint32_t* const* qs,
                           const uint32_t* const* d, const uint32_t* const* sc, const int* row0, int stride,
                           const float* x, size_t xstride, const float* up, int act, int nrows, int k, int m) {
    if (!c) return JL_ERR_ARG;
    CtxLock lock(c);
    drain_forget(c);
    // one matrix is not a batch (packedmulti.go:31-33, 109): jl_matvec_packed serves it
    if (m < 2 || nrows <= 0 || k <= 0 || (xstride != 0 && xstride < (size_t)k)) return JL_DECLINED;
    if (up && act != JL_ACT_SILU) return JL_DECLINED;   // the one gated activation the kernels bake in
    if (!outs || !qs || !d || !row0 || !x) return fail(c, JL_ERR_ARG, "packed multi: null operand");
    if (up && xstride == 0) return fail(c, JL_ERR_ARG, "packed multi: a gated activation needs one activation a matrix");
    if (c->no_device) return fail(c, JL_ERR_HIP, "this context is bound to no device");
    const TypeInfo* ti = nullptr;
    for (int j = 0; j < m; j++) {
        if (!outs[j] || !qs[j] || !d[j]) return fail(c, JL_ERR_ARG, "packed multi: null operand of matrix %d", j);
        const PlaneRef host = {qs[j], d[j], sc ? sc[j] : nullptr, row0[j], stride};
        int rc = packed_check(c, type, host, nrows, k, &ti);
        if (rc != JL_OK) return rc;
    }
    HIP_TRY(c, H->SetDevice(c->device));
    std::vector<PlaneRef> pls((size_t)m);
    for (int j = 0; j < m; j++) {
        const PlaneRef host = {qs[j], d[j], sc ? sc[j] : nullptr, row0[j], stride};
        int rc = resident_planes(c, type, host, k, &pls[(size_t)j]);
        if (rc != JL_OK) return rc;
    }
    const size_t nx = xstride ? (size_t)(m - 1) * xstride + (size_t)k : (size_t)k, o_up = up64(nx);
    const size_t orow = up64((size_t)nrows);
    int rc = host_io_begin(c, o_up + (up ? nx : 0), (size_t)m * orow);
    if (rc != JL_OK) return rc;
    rc = stage_in(c, 0, x, nx);
    if (rc == JL_OK && up) rc = stage_in(c, o_up, up, nx);
    const float* xd = nullptr;
    if (rc == JL_OK) rc = host_io_go(c, &xd);
    const float* ud = up ? xd + o_up : nullptr;
    for (int j0 = 0; j0 < m && rc == JL_OK; j0 += JL_MAX_MULTI) {   // sixteen matrices a launch
        const int n = std::min(m - j0, (int)JL_MAX_MULTI);
        float* od[JL_MAX_MULTI];
        for (int j = 0; j < n; j++) od[j] = host_results(c) + (size_t)(j0 + j) * orow;
        rc = packed_matvec_multi_launch(c, type, n, od, &pls[(size_t)j0], xd + (size_t)j0 * xstride, xstride,
                                        ud ? ud + (size_t)j0 * xstride : nullptr, nullptr, 0.f, nullptr, nullptr, 0.f,
                                        nullptr, nrows, k, c->stream);
    }
    for (int j = 0; j < m; j++) host_out((size_t)j * orow, outs[j], (size_t)nrows);
    return host_io_end(c, rc);
}

int jl_moe_grouped(jl_ctx* c, float* resid, int type, const void* gate_bank, const void* up_bank,
                   const void* down_bank, const float* x, const uint32_t* sel, int sel_stride, const float* wt,
                   int rows, int k_used, int n_expert, int n_ffn, int n_embd) {
    if (!c) return JL_ERR_ARG;
    CtxLock lock(c);
    drain_forget(c);
    if (rows <= 0 || k_used <= 0 || n_expert <= 0 || n_ffn <= 0 || n_embd <= 0 || sel_stride < k_used)
        return fail(c, JL_ERR_ARG, "moe grouped: bad shape");
    if (!resid || !gate_bank || !up_bank || !down_bank || !x || !sel || !wt)
        return fail(c, JL_ERR_ARG, "moe grouped: null operand");
    const TypeInfo* ti = type_info(type);
    if (!ti || n_embd % ti->block_elems || n_ffn % ti->block_elems) return JL_DECLINED;
    if (n_expert > 1024 || k_used > 16 || n_ffn % 256 != 0 || n_embd % 256 != 0) return JL_DECLINED;
    if (c->no_device) return fail(c, JL_ERR_HIP, "this context is bound to no device");
    HIP_TRY(c, H->SetDevice(c->device));
    // the three banks stay resident, each keyed on its host pointer
    const size_t bank = (size_t)n_expert * n_ffn * (size_t)(n_embd / ti->block_elems) * ti->block_bytes;
    void *gd = nullptr, *ud = nullptr, *dd = nullptr;
    int rc = resident_weight(c, gate_bank, bank, &gd);
    if (rc == JL_OK) rc = resident_weight(c, up_bank, bank, &ud);
    if (rc == JL_OK) rc = resident_weight(c, down_bank, bank, &dd);
    if (rc != JL_OK) return rc;
    // staged as floats: x, resid, wt, then the selections (32-bit words as well)
    const size_t nx = (size_t)rows * n_embd, o_res = up64(nx), o_wt = o_res + up64(nx),
                 o_sel = o_wt + up64((size_t)rows * k_used), total = o_sel + up64((size_t)rows * sel_stride);
    if ((rc = host_io_begin(c, total, nx)) != JL_OK) return rc;
    rc = stage_in(c, 0, x, nx);
    if (rc == JL_OK) rc = stage_in(c, o_res, resid, nx);
    if (rc == JL_OK) rc = stage_in(c, o_wt, wt, (size_t)rows * k_used);
    if (rc == JL_OK) rc = stage_in(c, o_sel, (const float*)sel, (size_t)rows * sel_stride);
    const float* xd = nullptr;
    if (rc == JL_OK) rc = host_io_go(c, &xd);
    float* base = (float*)c->stage_x;
    if (rc == JL_OK)
        rc = moe_ffn(c, base + o_res, type, type, gd, ud, dd, nullptr, nullptr, nullptr, base, (const uint32_t*)(base + o_sel),
                 sel_stride, base + o_wt, rows, k_used, n_expert, n_ffn, n_embd, c->stream);
    if (rc == JL_OK) rc = host_result_copy(c, 0, base + o_res, nx);
    host_out(0, resid, nx);
    return host_io_end(c, rc);
}

int jl_matvec_packed_group(jl_ctx* c, int n, float* const* outs, const int* types, const uint32_t* const* qs,
                           const uint32_t* const* d, const uint32_t* const* sc, const int* row, const int* stride,
                           const int* rows, const float* x, int k, const float* act_up, int act, float* resid,
                           float alpha) {
    if (!c) return JL_ERR_ARG;
    CtxLock lock(c);
    drain_forget(c);
    if (n < 1 || n > JL_MAX_GROUP || k <= 0) return JL_DECLINED;   // MaxGroup, packedgroup.go:12
    if (act_up && act != JL_ACT_SILU) return JL_DECLINED;
    if (!outs || !types || !qs || !d || !row || !stride || !rows || !x) return fail(c, JL_ERR_ARG, "packed group: null operand");
    if (c->no_device) return fail(c, JL_ERR_HIP, "this context is bound to no device");
    // nothing runs unless every matrix can (packedgroup.go:47-50)
    for (int i = 0; i < n; i++) {
        if (!outs[i] || !qs[i] || !d[i]) return fail(c, JL_ERR_ARG, "packed group: null operand of matrix %d", i);
        if (rows[i] <= 0) return JL_DECLINED;
        const TypeInfo* ti = nullptr;
        const PlaneRef host = {qs[i], d[i], sc ? sc[i] : nullptr, row[i], stride[i] ? stride[i] : rows[i]};
        int rc = packed_check(c, types[i], host, rows[i], k, &ti);
        if (rc != JL_OK) return rc;
    }
    HIP_TRY(c, H->SetDevice(c->device));
    PlaneRef pls[JL_MAX_GROUP];
    for (int i = 0; i < n; i++) {
        const PlaneRef host = {qs[i], d[i], sc ? sc[i] : nullptr, row[i], stride[i] ? stride[i] : rows[i]};
        int rc = resident_planes(c, types[i], host, k, &pls[i]);
        if (rc != JL_OK) return rc;
    }
    // staged: x, the gate's partner, the residual (matrix 0's rows)
    const size_t o_up = up64((size_t)k), o_res = o_up + (act_up ? up64((size_t)k) : 0);
    size_t o_out[JL_MAX_GROUP], total = 0;
    for (int i = 0; i < n; i++) { o_out[i] = total; total += up64((size_t)rows[i]); }
    const size_t o_rd = total;   // the updated residual comes behind the outputs
    if (resid) total += up64((size_t)rows[0]);
    int rc = host_io_begin(c, o_res + (resid ? up64((size_t)rows[0]) : 0), total);
    if (rc != JL_OK) return rc;
    rc = stage_in(c, 0, x, (size_t)k);
    if (rc == JL_OK && act_up) rc = stage_in(c, o_up, act_up, (size_t)k);
    if (rc == JL_OK && resid) rc = stage_in(c, o_res, resid, (size_t)rows[0]);
    const float* xd = nullptr;
    if (rc == JL_OK) rc = host_io_go(c, &xd);
    const float* ud = act_up ? xd + o_up : nullptr;
    float* rd = resid ? (float*)c->stage_x + o_res : nullptr;
    // matrices of one type and row count that follow one another share a launch (a block's gate
    // and up); the residual rides on matrix 0 (MVGroup.Resid, packedgroup.go:32-36)
    for (int i = 0; i < n && rc == JL_OK;) {
        int e = i + 1;
        while (e < n && types[e] == types[i] && rows[e] == rows[i] && pls[e].stride == pls[i].stride) e++;
        float* od[JL_MAX_GROUP];
        for (int j = i; j < e; j++) od[j - i] = host_results(c) + o_out[j];
        rc = packed_matvec_multi_launch(c, types[i], e - i, od, &pls[i], xd, 0, ud, i == 0 ? rd : nullptr, alpha, nullptr,
                                        nullptr, 0.f, nullptr, rows[i], k, c->stream);
        i = e;
    }
    if (rc == JL_OK && resid) rc = host_result_copy(c, o_rd, rd, (size_t)rows[0]);
    for (int i = 0; i < n; i++) host_out(o_out[i], outs[i], (size_t)rows[i]);
    if (resid) host_out(o_rd, resid, (size_t)rows[0]);   // last: the sum is what stays where resid is also an output
    return host_io_end(c, rc);
}

int jl_matmul_packed(jl_ctx* c, float* out, int type, const uint32_t* qs, const uint32_t* d,
                     const uint32_t* sc, int row, int stride, const float* x, int nrows, int k, int ntok) {
    if (!c) return JL_ERR_ARG;
    CtxLock lock(c);
    drain_forget(c);
    if (c->no_device) return fail(c, JL_ERR_HIP, "this context is bound to no device");
    const PlaneRef host = {qs, d, sc, row, stride};
    const TypeInfo* ti = nullptr;
    int rc = packed_check(c, type, host, nrows, k, &ti);
    if (rc != JL_OK) return rc;
    if (!out || !x || ntok <= 0) return fail(c, JL_ERR_ARG, "packed matmul: bad operand");
    HIP_TRY(c, H->SetDevice(c->device));
    PlaneRef pl;
    if ((rc = resident_planes(c, type, host, k, &pl)) != JL_OK) return rc;
    const size_t nx = (size_t)ntok * k, no = (size_t)ntok * nrows;
    if ((rc = host_io_begin(c, nx, no)) != JL_OK) return rc;
    rc = stage_in(c, 0, x, nx);
    const float* xd = nullptr;
    if (rc == JL_OK) rc = host_io_go(c, &xd, few_applies(c, type, true, nrows, k, ntok, pl.stride) && !tokens_matvec_wanted(c, type, true, nrows, k, ntok, pl.stride));
    if (rc == JL_OK) rc = ntok == 1 ? packed_matvec_launch(c, host_results(c), type, pl, xd, nullptr,
                                          nullptr, nullptr, nrows, k, c->stream)
                   : packed_matmul_launch(c, host_results(c), type, pl, xd, nrows, k,
                                          ntok, c->stream);
    host_out(0, out, no);
    return host_io_end(c, rc);
}

int jl_forget(jl_ctx* c, const void* p, size_t n) {
    if (!c) return JL_ERR_ARG;
    if (!p || n == 0) return JL_OK;
    // Queue the range under a lock no launch or upload holds, so this returns from any thread --
    // also from inside a page-in that this context's own weight upload started.  Then, as the
    // reference does (jit/gpu/tier/forget.go:38-49), apply the queue at once if the context is
    // free: the device copies go now and a caller that never makes another host-pointer call
    // still gets its memory back.  A busy context (another thread's call, or this thread's own)
    // applies the queue at the start of its next host-pointer call; jl_ctx_destroy frees the rest.
    {
        std::lock_guard<std::mutex> g(c->forget_mu);
        c->pending_forget.emplace_back((uintptr_t)p, (uintptr_t)p + n);
        // a device range: the matrices admitted to the folded-scale form inside it
        c->fold_ok.erase(c->fold_ok.lower_bound((uintptr_t)p), c->fold_ok.lower_bound((uintptr_t)p + n));
    }
    if (c->mu_owner.load() != std::this_thread::get_id() && c->mu.try_lock()) {
        c->mu_owner.store(std::this_thread::get_id());
        drain_forget(c);
        c->mu_owner.store(std::thread::id());
        c->mu.unlock();
    }
    return JL_OK;
}

int jl_probe_dev(jl_ctx* c, int kind, const void* src, size_t nbytes, int grid, int block, void* stream) {
    if (!c) return JL_ERR_ARG;
    if (kind == 2) {
        // hold the stream: nbytes is microseconds here, at most a tenth of a second
        if (nbytes > 100000) return fail(c, JL_ERR_ARG, "probe: a wait of %zu us", nbytes);
        HIP_TRY(c, H->SetDevice(c->device));
        size_t ticks = nbytes * 100;   // the constant clock runs at 100 MHz
        void* none = nullptr;
        void* wp[] = {(void*)&none, (void*)&ticks, (void*)&none};
        return launch(c, "jl_probe_wait", 1, 1, 64, 0, pick_stream(c, stream), wp);
    }
    if (kind == 3 || kind == 4) {
        // matrix-core ceiling: nbytes is the rounds of four matrix instructions a wavefront issues
        if (nbytes == 0 || nbytes > 1000000) return fail(c, JL_ERR_ARG, "probe: %zu rounds", nbytes);
        if (grid <= 0) grid = c->num_cu;
        if (block <= 0) block = 512;
        if (block % 64 != 0 || block > 1024) return fail(c, JL_ERR_ARG, "probe: block=%d", block);
        HIP_TRY(c, H->SetDevice(c->device));
        void* none = nullptr;
        void* mp[] = {(void*)&none, (void*)&nbytes, (void*)&none};
        return launch(c, kind == 3 ? "jl_probe_mfma" : "jl_probe_mfma_v5", (unsigned)grid, 1, (unsigned)block, 0,
                      pick_stream(c, stream), mp);
    }
    if (kind != 0 && kind != 1) return fail(c, JL_ERR_ARG, "probe: kind %d", kind);
    if (grid <= 0) grid = 2 * c->num_cu;
    if (block <= 0) block = 1024;
    if (block % 64 != 0 || block > 1024) return fail(c, JL_ERR_ARG, "probe: block=%d", block);
    if (kind == 1 && (!src || ((uintptr_t)src & 1) != 0)) return fail(c, JL_ERR_ARG, "probe: src");
    HIP_TRY(c, H->SetDevice(c->device));
    size_t nvec = nbytes / 16;
    void* sink = nullptr;
    void* params[] = {(void*)&src, (void*)&nvec, (void*)&sink};
    return launch(c, kind ? "jl_probe_read" : "jl_probe_empty", (unsigned)grid, 1, (unsigned)block, 0,
                  pick_stream(c, stream), params);
}

int jl_ctx_lock(jl_ctx* c) {
    if (!c) return JL_ERR_ARG;
    c->mu.lock();
    c->mu_owner.store(std::this_thread::get_id());
    return JL_OK;
}

int jl_ctx_unlock(jl_ctx* c) {
    if (!c) return JL_ERR_ARG;
    c->mu_owner.store(std::thread::id());
    c->mu.unlock();
    return JL_OK;
}

size_t jl_resident_count(jl_ctx* c) {
    if (!c) return 0;
    CtxLock lock(c);
    drain_forget(c);
    return c->resident.size();
}

}  // extern "C"
