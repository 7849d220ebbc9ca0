// C-ABI entry points (include/mhc_hip.h): argument validation, workspace
// carving and kernel sequencing.  Host code only; kernels live in the other
// translation units.
#include <math.h>
#include <string.h>

#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "mhc_hip.h"
#ifdef MHC_KERNEL_TIMING
#include "mhc_hip_timing.h"
#endif
#include "mhc_internal.h"

namespace mhc {

// ---------------------------------------------------------------------------
// Errors
// ---------------------------------------------------------------------------
static thread_local std::string g_last_error;

static int fail(int code, const std::string& msg) {
    g_last_error = msg;
    return code;
}

static int hip_status(hipError_t e) {
    if (e == hipSuccess) return MHC_SUCCESS;
    g_last_error = std::string("HIP error: ") + hipGetErrorString(e);
    return (int)e;
}

#define MHC_REQUIRE(cond, msg) \
    do {                       \
        if (!(cond)) return fail(MHC_ERR_INVALID, msg); \
    } while (0)

static bool valid_dtype(int dt) { return dt == kF32 || dt == kBF16; }

// The layer runs its fixed-n kernels for n in {2..8, 16, 32} (n = 3, 5, 6, 7:
// up to kWideMaxC channels) and the generic kernels (generic.hip) for every
// other n up to kGenMaxN, as the reference takes any n up to
// MAX_EXPANSION_RATE = 64 (mhc_types.h:68); the fused wrapper takes n = 2..32.
static bool supported_layer_n(int n) {
    return n == 2 || n == 4 || n == 8 || n == 16 || n == 32 || generic_layer_n(n);
}
static bool supported_dynamic_n(int n) { return supported_layer_n(n); }
// the standalone aggregate / distribute operators
static bool supported_ops_n(int n) {
    return (n >= 1 && n <= 8) || n == 16 || n == 32 || generic_ops_n(n);
}

// ---------------------------------------------------------------------------
// Device properties
// ---------------------------------------------------------------------------
int device_cu_count() {
    static int cache[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cache[dev] == 0) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            cus = 256;
        cache[dev] = cus;
    }
    return cache[dev];
}

// Resident workgroups of a kernel per CU, asked of the runtime once per
// (device, kernel, launch shape): the entries size their grids and workspaces
// with it several times per call.  At most kOccEntries are kept.
int occupancy_per_cu(const void* fn, int threads, size_t lds) {
    struct Entry {
        int dev, threads;
        const void* fn;
        size_t lds;
        int per_cu;
    };
    constexpr size_t kOccEntries = 512;
    static std::mutex mu;
    static std::vector<Entry> cache;
    int dev = 0;
    if (fn == nullptr || hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        return 1;
    }
    std::lock_guard<std::mutex> lk(mu);
    for (const Entry& e : cache) {
        if (e.fn == fn && e.threads == threads && e.lds == lds && e.dev == dev) return e.per_cu;
    }
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, threads, lds) != hipSuccess || per_cu < 1) {
        (void)hipGetLastError();
        return 1;
    }
    if (cache.size() >= kOccEntries) cache.clear();
    cache.push_back(Entry{dev, threads, fn, lds, per_cu});
    return per_cu;
}

// The row kernels are compiled with __launch_bounds__(512) and chunk counts
// VPT in {1, 2, 4, 8}; at most kRowStateBudget floats of row state stay live
// per thread so that a 512-lane workgroup fits in 256 VGPRs without spilling.  The
// score prefers exact coverage of the row, then workgroups near
// pref_threads lanes.
RowTiling choose_row_tiling(int64_t C, int wc, int n_arrays_live, int pref_threads) {
    RowTiling best{0, 0};
    if (C <= 0 || C % wc != 0) return best;
    const int64_t chunks = C / wc;
    double best_score = 1e30;
    for (int vpt = 1; vpt <= 8; vpt *= 2) {
        if (n_arrays_live * vpt * wc > kRowStateBudget) break;  // live row state per thread (floats)
        int64_t threads = (chunks + vpt - 1) / vpt;
        threads = ((threads + 63) / 64) * 64;
        if (threads > 512) continue;
        const double waste = (double)(threads * vpt - chunks) / (double)(threads * vpt);
        const double shape = fabs(log2((double)threads / (double)pref_threads)) * 0.02;
        const double score = waste + shape;
        if (score < best_score) {
            best_score = score;
            best.threads = (int)threads;
            best.vpt = vpt;
        }
    }
    return best;
}

#ifdef MHC_KERNEL_TIMING
// ---------------------------------------------------------------------------
// Kernel timing registry (the benchmark's build only, MHC_KERNEL_TIMING)
// ---------------------------------------------------------------------------
struct TimingRecord {
    std::string name;
    hipEvent_t start = nullptr;
    hipEvent_t stop = nullptr;
    bool pending = false;
    bool launched = false;
};

static std::mutex g_timing_mu;
static bool g_timing_on = false;
static std::vector<TimingRecord> g_records;
static std::unordered_map<std::string, std::pair<double, int64_t>> g_totals;

static thread_local TimingScope t_scope;
static thread_local bool t_scope_open = false;

TimingScope* timing_scope() { return t_scope_open ? &t_scope : nullptr; }

// A timed scope runs alone on the device: kernels of one stream may overlap
// (the next starts while the previous one's last workgroups drain), so the
// scope waits for the stream before its first launch and after its last, and
// its events time its own kernels only, as a profiler's kernel trace does.
// This build exists for the benchmark's per-kernel pass only.
int timing_begin(const char* name, hipStream_t s) {
    {
        std::lock_guard<std::mutex> lk(g_timing_mu);
        if (!g_timing_on) return -1;
    }
    if (hipStreamSynchronize(s) != hipSuccess) return -1;
    std::lock_guard<std::mutex> lk(g_timing_mu);
    int idx = -1;
    for (size_t i = 0; i < g_records.size(); ++i) {
        if (!g_records[i].pending) { idx = (int)i; break; }
    }
    if (idx < 0) {
        TimingRecord r;
        if (hipEventCreate(&r.start) != hipSuccess || hipEventCreate(&r.stop) != hipSuccess) return -1;
        g_records.push_back(r);
        idx = (int)g_records.size() - 1;
    }
    TimingRecord& r = g_records[idx];
    r.name = name;
    r.pending = true;
    r.launched = false;
    t_scope = TimingScope{r.start, r.stop, true};
    t_scope_open = true;
    return idx;
}

void timing_end(int token, hipStream_t s) {
    if (token < 0) return;
    {
        std::lock_guard<std::mutex> lk(g_timing_mu);
        // a scope without a launch (empty batch) records nothing
        g_records[token].launched = t_scope_open && !t_scope.first;
        t_scope_open = false;
    }
    (void)hipStreamSynchronize(s);
}

hipError_t mhc_launch_kernel(const void* fn, dim3 grid, dim3 block, void** args, size_t shm, hipStream_t s) {
    TimingScope* ts = timing_scope();
    if (!ts) return hipLaunchKernel(fn, grid, block, args, shm, s);
    const hipError_t e = hipExtLaunchKernel(fn, grid, block, args, shm, s, ts->first ? ts->start : nullptr, ts->stop, 0);
    ts->first = false;
    return e;
}

static void timing_drain_locked() {
    for (auto& r : g_records) {
        if (!r.pending) continue;
        r.pending = false;
        if (!r.launched) continue;
        float ms = 0.f;
        if (hipEventSynchronize(r.stop) != hipSuccess || hipEventElapsedTime(&ms, r.start, r.stop) != hipSuccess) {
            (void)hipGetLastError();
            continue;
        }
        auto& t = g_totals[r.name];
        t.first += ms;
        t.second += 1;
    }
}

#endif  // MHC_KERNEL_TIMING

}  // namespace mhc

using namespace mhc;

extern "C" {

int mhc_abi_version(void) { return 101; }

const char* mhc_last_error(void) { return g_last_error.c_str(); }

#ifdef MHC_KERNEL_TIMING
int mhc_timing_enable(int enable) {
    std::lock_guard<std::mutex> lk(g_timing_mu);
    g_timing_on = enable != 0;
    return MHC_SUCCESS;
}

int mhc_timing_reset(void) {
    std::lock_guard<std::mutex> lk(g_timing_mu);
    timing_drain_locked();
    g_totals.clear();
    return MHC_SUCCESS;
}

int mhc_timing_query(const char* kernel, double* total_ms, int64_t* launches) {
    if (!kernel || !total_ms || !launches) return fail(MHC_ERR_INVALID, "mhc_timing_query: null argument");
    std::lock_guard<std::mutex> lk(g_timing_mu);
    timing_drain_locked();
    auto it = g_totals.find(kernel);
    *total_ms = it == g_totals.end() ? 0.0 : it->second.first;
    *launches = it == g_totals.end() ? 0 : it->second.second;
    return MHC_SUCCESS;
}

#endif  // MHC_KERNEL_TIMING

// ---- Sinkhorn ---------------------------------------------------------------
int mhc_sinkhorn_knopp_fwd(const float* inp, float* out, int64_t batch, int32_t n, int32_t num_iters, float eps,
                           void* stream) {
    MHC_REQUIRE(batch >= 0, "sinkhorn_knopp_fwd: batch must be >= 0");
    MHC_REQUIRE(n >= 1, "sinkhorn_knopp_fwd: n must be >= 1");
    MHC_REQUIRE(num_iters >= 0, "sinkhorn_knopp_fwd: num_iters must be >= 0");
    if (batch == 0) return MHC_SUCCESS;
    MHC_REQUIRE(inp && out, "sinkhorn_knopp_fwd: null pointer");
    if (n > 64) return fail(MHC_ERR_UNSUPPORTED, "sinkhorn_knopp_fwd: n > 64 is not supported (one matrix row per lane of a wave)");
    return hip_status(launch_sinkhorn_fwd(n, inp, out, batch, num_iters, eps, (hipStream_t)stream));
}

int mhc_sinkhorn_knopp_bwd(const float* grad_out, const float* inp, const float* out, float* grad_inp,
                           int64_t batch, int32_t n, int32_t num_iters, float eps, void* stream) {
    (void)out;
    MHC_REQUIRE(batch >= 0, "sinkhorn_knopp_bwd: batch must be >= 0");
    MHC_REQUIRE(n >= 1, "sinkhorn_knopp_bwd: n must be >= 1");
    MHC_REQUIRE(num_iters >= 0, "sinkhorn_knopp_bwd: num_iters must be >= 0");
    if (batch == 0) return MHC_SUCCESS;
    MHC_REQUIRE(grad_out && inp && grad_inp, "sinkhorn_knopp_bwd: null pointer");
    if (n > 64) return fail(MHC_ERR_UNSUPPORTED, "sinkhorn_knopp_bwd: n > 64 is not supported (one matrix row per lane of a wave)");
    return hip_status(launch_sinkhorn_bwd(n, grad_out, inp, grad_inp, batch, num_iters, eps, (hipStream_t)stream));
}

// ---- static layer -----------------------------------------------------------
static int check_layer_shape(const char* fn, int64_t batch, int32_t n, int32_t hidden, int32_t x_dtype,
                             int32_t num_iters) {
    if (batch < 0) return fail(MHC_ERR_INVALID, std::string(fn) + ": batch must be >= 0");
    if (n < 1) return fail(MHC_ERR_INVALID, std::string(fn) + ": n must be >= 1");
    if (hidden < 1) return fail(MHC_ERR_INVALID, std::string(fn) + ": hidden must be >= 1");
    if (num_iters < 0) return fail(MHC_ERR_INVALID, std::string(fn) + ": num_iters must be >= 0");
    if (!valid_dtype(x_dtype)) return fail(MHC_ERR_INVALID, std::string(fn) + ": x_dtype must be F32 or BF16");
    if (!supported_layer_n(n))
        return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": n=" + std::to_string(n) +
                                             " is not supported (1 <= n <= " + std::to_string(kGenMaxN) + ")");
    // register rows (n <= 8, 4-channel chunks that fit) or the channel-loop
    // kernels; the generic-n kernels take any hidden size
    if (!generic_layer_n(n) && (layer_fwd_is_wide(n, hidden) || layer_bwd_is_wide(n, hidden)) &&
        !wide_supported(n, hidden))
        return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": hidden=" + std::to_string(hidden) +
                                             " is too large for the row kernels at n=" + std::to_string(n));
    return MHC_SUCCESS;
}

size_t mhc_layer_static_saved_size(int32_t n, int32_t hidden) {
    if (n < 1 || hidden < 1) return 0;
    return ((size_t)saved_w_offset(n) + (size_t)hidden) * sizeof(float);
}

int mhc_layer_static_fwd(const void* x, int32_t x_dtype, const void* weight, int32_t weight_dtype,
                         const float* h_pre, const float* h_post, const float* h_res, float* out, float* rms,
                         float* saved, int64_t batch, int32_t n, int32_t hidden, int32_t num_iters,
                         float sinkhorn_eps, float rmsnorm_eps, void* stream) {
    int st = check_layer_shape("layer_static_fwd", batch, n, hidden, x_dtype, num_iters);
    if (st) return st;
    MHC_REQUIRE(valid_dtype(weight_dtype), "layer_static_fwd: weight_dtype must be F32 or BF16");
    MHC_REQUIRE(weight && h_pre && h_post && h_res && saved, "layer_static_fwd: null parameter pointer");
    MHC_REQUIRE(batch == 0 || (x && out), "layer_static_fwd: null x/out");
    hipStream_t s = (hipStream_t)stream;
    if (layer_static_fwd_fused(n, hidden) && rows_aligned(n, {x, weight, saved, out}))
        return hip_status(launch_layer_static_fwd(x_dtype, n, x, weight, weight_dtype, h_pre, h_post, h_res, saved,
                                                  num_iters, sinkhorn_eps, out, rms, batch, hidden, rmsnorm_eps, s));
    hipError_t e = launch_static_coef(n, h_pre, h_post, h_res, weight, weight_dtype, hidden, saved, num_iters,
                                      sinkhorn_eps, s);
    if (e != hipSuccess) return hip_status(e);
    const float* w32 = saved + saved_w_offset(n);
    return hip_status(launch_layer_fwd(x_dtype, n, x, w32, saved, 0, out, kF32, rms, batch, hidden, rmsnorm_eps, s));
}


struct StaticBwdWs {
    int grid;
    size_t dw_off, scal_off, stage_off, hist_off, rows_off, total;
};

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// The static Sinkhorn adjoint keeps its per-iteration state in a workspace
// region (kStaticSkHistBytes) for n >= 16 and the generic n; without it
// those finalize kernels recompute the forward iterations.
static bool static_sk_hist(int32_t n) { return n >= 16 || (generic_layer_n(n) && !odd_row_n(n)); }

// aligned: rows_aligned() of the call's arrays (the row kernels differ)
static StaticBwdWs static_bwd_ws(int64_t batch, int32_t n, int32_t hidden, int32_t x_dtype, bool aligned) {
    StaticBwdWs w{};
    w.grid = batch > 0 ? layer_bwd_grid(x_dtype, n, batch, hidden, aligned) : 1;
    w.dw_off = 0;
    w.scal_off = align256((size_t)w.grid * hidden * sizeof(float));
    w.stage_off = w.scal_off + align256((size_t)w.grid * (n * n + 2 * n) * sizeof(float));
    w.hist_off = w.stage_off + align256(column_sums_stage_floats(hidden) * sizeof(float));
    // Sinkhorn adjoint history
    w.rows_off = w.hist_off + (static_sk_hist(n) ? kStaticSkHistBytes : 0);
    w.total = w.rows_off + align256(batch > 0 ? layer_bwd_scratch_bytes(x_dtype, n, batch, hidden, aligned) : 0);
    return w;
}

size_t mhc_layer_static_bwd_workspace_size(int64_t batch, int32_t n, int32_t hidden, int32_t x_dtype) {
    if (batch < 0 || n < 1 || hidden < 1) return 0;
    const size_t a = static_bwd_ws(batch, n, hidden, x_dtype, true).total;
    const size_t u = odd_row_n(n) ? static_bwd_ws(batch, n, hidden, x_dtype, false).total : 0;
    return a > u ? a : u;
}

static int static_bwd(const float* grad_out, const void* x, int32_t x_dtype, int32_t weight_dtype,
                      const float* h_pre, const float* h_post, const float* h_res, const float* saved, void* grad_x,
                      void* grad_weight, float* grad_h_pre, float* grad_h_post, float* grad_h_res, void* workspace,
                      size_t workspace_bytes, int64_t batch, int32_t n, int32_t hidden, int32_t num_iters,
                      float sinkhorn_eps, float rmsnorm_eps, void* stream, bool aligned) {
    int st = check_layer_shape("layer_static_bwd", batch, n, hidden, x_dtype, num_iters);
    if (st) return st;
    MHC_REQUIRE(valid_dtype(weight_dtype), "layer_static_bwd: weight_dtype must be F32 or BF16");
    MHC_REQUIRE(h_pre && h_post && h_res && saved, "layer_static_bwd: null parameter pointer");
    MHC_REQUIRE(grad_weight && grad_h_pre && grad_h_post && grad_h_res, "layer_static_bwd: null gradient pointer");
    MHC_REQUIRE(batch == 0 || (grad_out && x && grad_x), "layer_static_bwd: null grad_out/x/grad_x");
    hipStream_t s = (hipStream_t)stream;
    const StaticBwdWs w = static_bwd_ws(batch, n, hidden, x_dtype, aligned);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE, "layer_static_bwd: workspace smaller than mhc_layer_static_bwd_workspace_size()");
    float* dw_part = (float*)((char*)workspace + w.dw_off);
    float* scal_part = (float*)((char*)workspace + w.scal_off);
    float* stage = (float*)((char*)workspace + w.stage_off);
    hipError_t e = hipSuccess;
    int rows = w.grid;
    if (batch == 0) {
        // Empty batch: zero partials (fill kernels, not memsets, so the call
        // stays capturable in a HIP graph); the finalize then writes zeros.
        rows = 1;
        e = launch_fill_zero(dw_part, hidden, s);
        if (e == hipSuccess) e = launch_fill_zero(scal_part, n * n + 2 * n, s);
    } else {
        e = launch_layer_bwd(x_dtype, n, 0, grad_out, x, saved + saved_w_offset(n), saved, 0, grad_x, dw_part,
                             scal_part, w.grid, batch, hidden, rmsnorm_eps, (float*)((char*)workspace + w.rows_off),
                             s, nullptr, aligned);
    }
    if (e == hipSuccess)
        e = launch_column_finalize(n, weight_dtype, dw_part, rows, hidden, stage, grad_weight, scal_part, rows, h_pre,
                                  h_post, h_res, grad_h_pre, grad_h_post, grad_h_res, num_iters, sinkhorn_eps, s,
                                  static_sk_hist(n) ? (float*)((char*)workspace + w.hist_off) : nullptr);
    return hip_status(e);
}

int mhc_layer_static_bwd(const float* grad_out, const void* x, int32_t x_dtype, int32_t weight_dtype,
                         const float* h_pre, const float* h_post, const float* h_res, const float* saved,
                         void* grad_x, void* grad_weight, float* grad_h_pre, float* grad_h_post, float* grad_h_res,
                         void* workspace, size_t workspace_bytes, int64_t batch, int32_t n, int32_t hidden,
                         int32_t num_iters, float sinkhorn_eps, float rmsnorm_eps, void* stream) {
    return static_bwd(grad_out, x, x_dtype, weight_dtype, h_pre, h_post, h_res, saved, grad_x, grad_weight, grad_h_pre,
                      grad_h_post, grad_h_res, workspace, workspace_bytes, batch, n, hidden, num_iters, sinkhorn_eps,
                      rmsnorm_eps, stream, rows_aligned(n, {grad_out, x, grad_x, saved, workspace}));
}

// ---- allocation-free static backward ---------------------------------------
// mhc_layer_static_bwd with its workspace in a file-scope device array
// instead of a caller buffer, for callers that cannot allocate (HIP graph
// capture, serving loops).  Each device holds its own copy of the array for
// the life of the process; its address on a device comes from
// hipGetSymbolAddress on that device's first call (the name itself is only a
// host-side handle).  Nothing in it needs clearing: every kernel writes its
// partials before anything reads them.  Calls that overlap on one device
// share the array and race.
constexpr size_t kNoAllocScratchBytes = size_t(16) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

static std::mutex g_scratch_mu;
static void* g_scratch_ptr[64] = {};

static int scratch_on_current_device(void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_status(e);
    if (dev < 0 || dev >= 64) return fail(MHC_ERR_UNSUPPORTED, "scratch: device index out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_status(e);
        if (!p) return fail(MHC_ERR_INVALID, "scratch: hipGetSymbolAddress returned no address");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return MHC_SUCCESS;
}

size_t mhc_noalloc_scratch_bytes(void) { return kNoAllocScratchBytes; }

int mhc_layer_static_bwd_noalloc(const float* grad_out, const void* x, int32_t x_dtype, int32_t weight_dtype,
                                 const float* h_pre, const float* h_post, const float* h_res, const float* saved,
                                 void* grad_x, void* grad_weight, float* grad_h_pre, float* grad_h_post,
                                 float* grad_h_res, int64_t batch, int32_t n, int32_t hidden, int32_t num_iters,
                                 float sinkhorn_eps, float rmsnorm_eps, void* stream) {
    int st = check_layer_shape("layer_static_bwd_noalloc", batch, n, hidden, x_dtype, num_iters);
    if (st) return st;
    // the generic rows of n = 3, 5, 6, 7 where only theirs fit
    bool aligned = rows_aligned(n, {grad_out, x, grad_x, saved});
    size_t need = static_bwd_ws(batch, n, hidden, x_dtype, aligned).total;
    if (need > kNoAllocScratchBytes && odd_row_n(n)) {
        aligned = false;
        need = static_bwd_ws(batch, n, hidden, x_dtype, false).total;
    }
    if (need > kNoAllocScratchBytes)
        return fail(MHC_ERR_UNSUPPORTED, "layer_static_bwd_noalloc: this shape needs " + std::to_string(need) +
                                             " bytes of scratch, more than the library's " +
                                             std::to_string(kNoAllocScratchBytes) +
                                             "; use mhc_layer_static_bwd with a workspace");
    void* ws = nullptr;
    st = scratch_on_current_device(&ws);
    if (st) return st;
    return static_bwd(grad_out, x, x_dtype, weight_dtype, h_pre, h_post, h_res, saved, grad_x, grad_weight, grad_h_pre,
                      grad_h_post, grad_h_res, ws, kNoAllocScratchBytes, batch, n, hidden, num_iters, sinkhorn_eps,
                      rmsnorm_eps, stream, aligned);
}

// ---- standalone operators ---------------------------------------------------
// Rows the register kernels cannot take run the channel-loop kernels, which
// take any width; the RMSNorm backward's keeps its dw row in LDS (dw_row).
static int check_rows(const char* fn, int64_t batch, int64_t hidden, int32_t dtype, int n_arrays,
                      bool dw_row = false) {
    if (batch < 0) return fail(MHC_ERR_INVALID, std::string(fn) + ": batch must be >= 0");
    if (hidden < 1) return fail(MHC_ERR_INVALID, std::string(fn) + ": hidden must be >= 1");
    if (!valid_dtype(dtype)) return fail(MHC_ERR_INVALID, std::string(fn) + ": dtype must be F32 or BF16");
    if (hidden > 0x7fffffff) return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": hidden must be < 2^31");
    const bool regs = choose_row_tiling(hidden, dtype == kBF16 ? 8 : 4, n_arrays).vpt > 0;
    if (!regs && dw_row && hidden > kWideMaxC)
        return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": hidden=" + std::to_string(hidden) +
                                             " is too large for the row kernels");
    return MHC_SUCCESS;
}

static int check_stream_n(const char* fn, int32_t n) {
    if (n < 1) return fail(MHC_ERR_INVALID, std::string(fn) + ": n must be >= 1");
    if (!supported_ops_n(n))
        return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": n=" + std::to_string(n) + " is not compiled in this build");
    return MHC_SUCCESS;
}

int mhc_rmsnorm_fwd(const void* inp, int32_t dtype, const float* weight, void* out, float* rms, int64_t batch,
                    int32_t hidden, float eps, void* stream) {
    int st = check_rows("rmsnorm_fwd", batch, hidden, dtype, 1);
    if (st) return st;
    MHC_REQUIRE(batch == 0 || (inp && weight && out && rms), "rmsnorm_fwd: null pointer");
    return hip_status(launch_rmsnorm_fwd(dtype, inp, weight, out, rms, batch, hidden, eps, (hipStream_t)stream));
}

struct RowsBwdWs {
    int grid;
    size_t part_off, stage_off, total;
};

static RowsBwdWs rmsnorm_bwd_ws(int64_t batch, int32_t hidden, int32_t dtype) {
    RowsBwdWs w{};
    w.grid = batch > 0 ? rmsnorm_bwd_grid(dtype, batch, hidden) : 1;
    w.part_off = 0;
    w.stage_off = align256((size_t)w.grid * hidden * sizeof(float));
    w.total = w.stage_off + align256(column_sums_stage_floats(hidden) * sizeof(float));
    return w;
}

size_t mhc_rmsnorm_bwd_workspace_size(int64_t batch, int32_t hidden, int32_t dtype) {
    if (batch < 0 || hidden < 1) return 0;
    return rmsnorm_bwd_ws(batch, hidden, dtype).total;
}

int mhc_rmsnorm_bwd(const void* grad_out, const void* inp, int32_t dtype, const float* weight, const float* rms,
                    void* grad_inp, float* grad_weight, void* workspace, size_t workspace_bytes, int64_t batch,
                    int32_t hidden, void* stream) {
    int st = check_rows("rmsnorm_bwd", batch, hidden, dtype, 2, true);
    if (st) return st;
    MHC_REQUIRE(weight && grad_weight, "rmsnorm_bwd: null weight/grad_weight");
    MHC_REQUIRE(batch == 0 || (grad_out && inp && rms && grad_inp), "rmsnorm_bwd: null pointer");
    const RowsBwdWs w = rmsnorm_bwd_ws(batch, hidden, dtype);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE, "rmsnorm_bwd: workspace smaller than mhc_rmsnorm_bwd_workspace_size()");
    hipStream_t s = (hipStream_t)stream;
    float* part = (float*)((char*)workspace + w.part_off);
    float* stage = (float*)((char*)workspace + w.stage_off);
    int rows = w.grid;
    hipError_t e;
    if (batch == 0) {
        rows = 1;
        e = launch_fill_zero(part, hidden, s);
    } else {
        e = launch_rmsnorm_bwd(dtype, grad_out, inp, weight, rms, grad_inp, part, w.grid, batch, hidden, s);
    }
    if (e == hipSuccess)
        e = launch_column_finalize(0, kF32, part, rows, hidden, stage, grad_weight, nullptr, 0, nullptr, nullptr, nullptr,
                                  nullptr, nullptr, nullptr, 0, 0.f, s);
    return hip_status(e);
}

int mhc_compute_rms_fwd(const void* inp, int32_t dtype, float* rms, int64_t batch, int64_t k, float eps,
                        void* stream) {
    int st = check_rows("compute_rms_fwd", batch, k, dtype, 1);
    if (st) return st;
    MHC_REQUIRE(batch == 0 || (inp && rms), "compute_rms_fwd: null pointer");
    return hip_status(launch_compute_rms(dtype, inp, rms, batch, k, eps, (hipStream_t)stream));
}

int mhc_stream_aggregate_fwd(const void* inp, int32_t dtype, const float* h_pre_raw, int64_t h_batch_stride,
                             void* out, float* h_pre_act, int64_t batch, int32_t n, int32_t hidden, void* stream) {
    int st = check_stream_n("stream_aggregate_fwd", n);
    if (!st) st = check_rows("stream_aggregate_fwd", batch, hidden, dtype, n + 1);
    if (st) return st;
    MHC_REQUIRE(h_batch_stride == 0 || h_batch_stride == n, "stream_aggregate_fwd: h_batch_stride must be 0 or n");
    MHC_REQUIRE(batch == 0 || (inp && h_pre_raw && out && h_pre_act), "stream_aggregate_fwd: null pointer");
    return hip_status(launch_aggregate_fwd(dtype, n, inp, h_pre_raw, h_batch_stride, out, h_pre_act, batch, hidden,
                                           (hipStream_t)stream));
}

int mhc_stream_aggregate_bwd(const void* grad_out, const void* inp, int32_t dtype, const float* h_pre_act,
                             int64_t h_batch_stride, void* grad_inp, float* grad_h_pre_act, float* grad_h_pre_raw,
                             int64_t batch, int32_t n, int32_t hidden, void* stream) {
    int st = check_stream_n("stream_aggregate_bwd", n);
    if (!st) st = check_rows("stream_aggregate_bwd", batch, hidden, dtype, n + 1);
    if (st) return st;
    MHC_REQUIRE(h_batch_stride == 0 || h_batch_stride == n, "stream_aggregate_bwd: h_batch_stride must be 0 or n");
    MHC_REQUIRE(batch == 0 || (grad_out && inp && h_pre_act && grad_inp), "stream_aggregate_bwd: null pointer");
    return hip_status(launch_aggregate_bwd(dtype, n, grad_out, inp, h_pre_act, h_batch_stride, grad_inp,
                                           grad_h_pre_act, grad_h_pre_raw, batch, hidden, (hipStream_t)stream));
}

int mhc_stream_distribute_mix_add_fwd(const void* y_norm, const float* h_post_raw, int64_t h_batch_stride,
                                      const float* M, int64_t m_batch_stride, const void* x_inp, int32_t dtype,
                                      float* out, float* h_post_act, int64_t batch, int32_t n, int32_t hidden,
                                      void* stream) {
    int st = check_stream_n("stream_distribute_mix_add_fwd", n);
    if (!st) st = check_rows("stream_distribute_mix_add_fwd", batch, hidden, dtype, n + 1);
    if (st) return st;
    MHC_REQUIRE(h_batch_stride == 0 || h_batch_stride == n,
                "stream_distribute_mix_add_fwd: h_batch_stride must be 0 or n");
    MHC_REQUIRE(m_batch_stride == 0 || m_batch_stride == (int64_t)n * n,
                "stream_distribute_mix_add_fwd: m_batch_stride must be 0 or n*n");
    MHC_REQUIRE(batch == 0 || (y_norm && h_post_raw && M && x_inp && out && h_post_act),
                "stream_distribute_mix_add_fwd: null pointer");
    return hip_status(launch_distribute_fwd(dtype, n, y_norm, h_post_raw, h_batch_stride, M, m_batch_stride, x_inp,
                                            out, h_post_act, batch, hidden, (hipStream_t)stream));
}

int mhc_stream_distribute_mix_add_bwd(const float* grad_out, const void* x_inp, const void* y_norm, int32_t dtype,
                                      const float* M, int64_t m_batch_stride, const float* h_post_act,
                                      int64_t h_batch_stride, void* grad_x, void* grad_y, float* grad_M,
                                      float* grad_h_post_act, float* grad_h_post_raw, int64_t batch, int32_t n,
                                      int32_t hidden, void* stream) {
    int st = check_stream_n("stream_distribute_mix_add_bwd", n);
    if (!st) st = check_rows("stream_distribute_mix_add_bwd", batch, hidden, dtype, 2 * n + 1);
    if (st) return st;
    MHC_REQUIRE(h_batch_stride == 0 || h_batch_stride == n,
                "stream_distribute_mix_add_bwd: h_batch_stride must be 0 or n");
    MHC_REQUIRE(m_batch_stride == 0 || m_batch_stride == (int64_t)n * n,
                "stream_distribute_mix_add_bwd: m_batch_stride must be 0 or n*n");
    MHC_REQUIRE(batch == 0 || (grad_out && x_inp && y_norm && M && h_post_act && grad_x && grad_y && grad_M),
                "stream_distribute_mix_add_bwd: null pointer");
    return hip_status(launch_distribute_bwd(dtype, n, grad_out, x_inp, y_norm, M, m_batch_stride, h_post_act,
                                            h_batch_stride, grad_x, grad_y, grad_M, grad_h_post_act, grad_h_post_raw,
                                            batch, hidden, (hipStream_t)stream));
}

// ---- dynamic-H projection operators ------------------------------------------
static size_t align_floats(size_t n) { return (n + 63) & ~(size_t)63; }

struct ProjFwdWs {
    int ks;
    bool stream;  // more than one output tile: the streaming projection
    size_t phib_off, xpl_off, p_off, ss_off, total;
};

// [Phi planes (one 32-row output tile: three bf16 planes) or, with more
//  tiles, fp32 x split into three bf16 planes | P partials [tile][ks][B][32]
//  | sum x^2 partials [ks][B]]
static size_t phi_planes_bytes(int64_t k, int np) { return align256((size_t)proj_tiles(np) * 3 * 32 * k * 2); }

static ProjFwdWs proj_fwd_ws(int64_t batch, int64_t k, int np) {
    ProjFwdWs w{};
    w.ks = batch > 0 ? proj_ksplit(batch, k, np) : 1;
    w.stream = proj_stream_path(np);
    w.phib_off = 0;
    w.xpl_off = w.stream ? 0 : phi_planes_bytes(k, np);
    w.p_off = w.xpl_off + (w.stream ? align256(proj_xplanes_bytes(batch, k)) : 0);
    w.ss_off = w.p_off + align256((size_t)proj_tiles(np) * w.ks * batch * kProjTile * sizeof(float));
    w.total = w.ss_off + align256((size_t)w.ks * batch * sizeof(float));
    return w;
}

// bf16 x with 33..128 projection rows (n = 5..10) and at least 1024 tokens:
// the streaming projection on the Phi planes reads x once for all output
// tiles instead of once per 32-row tile.  Measured at n = 8, C = 4096 (layer
// forward): 1.134 -> 1.035 ms at 16384 tokens, 0.350 -> 0.333 at 4096; at
// 128-256 tokens (C = 1280) no faster in training and 4-5% slower in the
// forward-only entry, so fewer tokens keep the per-tile kernel.
static bool proj_one_pass(int x_dtype, int np, int64_t batch) {
    return x_dtype == kBF16 && np > kProjTile && batch >= 1024;
}

static int check_proj(const char* fn, int64_t batch, int64_t k, int32_t out_dim) {
    if (batch < 0 || k < 1) return fail(MHC_ERR_INVALID, std::string(fn) + ": batch must be >= 0 and k >= 1");
    if (out_dim < 1) return fail(MHC_ERR_INVALID, std::string(fn) + ": out_dim must be >= 1");
    if (out_dim > kMaxProjRows)
        return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": out_dim > " + std::to_string(kMaxProjRows) +
                                             " is not supported");
    if (k % 32 != 0) return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": k must be a multiple of 32");
    if (k > (int64_t(1) << 22)) return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": k > 4194304 is not supported");
    return MHC_SUCCESS;
}

size_t mhc_fused_rmsnorm_matmul_fwd_workspace_size(int64_t batch, int64_t k, int32_t out_dim) {
    if (batch < 0 || k < 1 || out_dim < 1) return 0;
    return proj_fwd_ws(batch, k, out_dim).total;
}

int mhc_fused_rmsnorm_matmul_fwd(const void* inp, int32_t dtype, const float* weight, float* out, void* workspace,
                                 size_t workspace_bytes, int64_t batch, int64_t k, int32_t out_dim, void* stream) {
    int st = check_proj("fused_rmsnorm_matmul_fwd", batch, k, out_dim);
    if (st) return st;
    MHC_REQUIRE(valid_dtype(dtype), "fused_rmsnorm_matmul_fwd: dtype must be F32 or BF16");
    MHC_REQUIRE(weight && (batch == 0 || (inp && out)), "fused_rmsnorm_matmul_fwd: null pointer");
    if (batch == 0) return MHC_SUCCESS;
    const ProjFwdWs w = proj_fwd_ws(batch, k, out_dim);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE, "fused_rmsnorm_matmul_fwd: workspace too small");
    hipStream_t s = (hipStream_t)stream;
    bf16_raw_t* phib = (bf16_raw_t*)((char*)workspace + w.phib_off);
    float* pp = (float*)((char*)workspace + w.p_off);
    float* ss = (float*)((char*)workspace + w.ss_off);
    hipError_t e = hipSuccess;
    if (w.stream) {
        e = launch_proj_stream(dtype, inp, (bf16_raw_t*)((char*)workspace + w.xpl_off), weight, weight, weight,
                               out_dim, nullptr, out_dim, pp, ss, batch, k, w.ks, s);
    } else {
        e = launch_phi_split(weight, weight, weight, out_dim, out_dim, k, phib, s);
        if (e == hipSuccess) e = launch_proj_mfma(dtype, inp, phib, out_dim, pp, ss, batch, k, w.ks, s);
    }
    if (e == hipSuccess) e = launch_proj_reduce(pp, w.ks, batch, out_dim, out, s);
    return hip_status(e);
}

#ifdef MHC_KERNEL_TIMING
// The benchmark build's VALU projection, for the A/B against the MFMA one
// (include/mhc_hip_timing.h).
// [Phi^T [k][32] | P partials [ks][B][32] | sum x^2 partials [ks][B]]
size_t mhc_timing_proj_valu_workspace_size(int64_t batch, int64_t k, int32_t out_dim) {
    (void)out_dim;
    if (batch <= 0 || k <= 0) return 256;
    const int ks = proj_valu_ksplit(batch, k);
    return align256((size_t)k * 32 * 4) + align256((size_t)ks * batch * 32 * 4) + align256((size_t)ks * batch * 4);
}

int mhc_timing_proj_valu(const void* inp, int32_t dtype, const float* weight, float* out, void* workspace,
                         size_t workspace_bytes, int64_t batch, int64_t k, int32_t out_dim, void* stream) {
    MHC_REQUIRE(batch >= 0 && k >= 1 && k % 32 == 0, "timing_proj_valu: batch >= 0 and k a positive multiple of 32");
    MHC_REQUIRE(out_dim >= 1 && out_dim <= 32, "timing_proj_valu: out_dim must be 1..32");
    MHC_REQUIRE(valid_dtype(dtype), "timing_proj_valu: dtype must be F32 or BF16");
    MHC_REQUIRE(weight && (batch == 0 || (inp && out)), "timing_proj_valu: null pointer");
    if (batch == 0) return MHC_SUCCESS;
    if (!workspace || workspace_bytes < mhc_timing_proj_valu_workspace_size(batch, k, out_dim))
        return fail(MHC_ERR_WORKSPACE, "timing_proj_valu: workspace too small");
    const int ks = proj_valu_ksplit(batch, k);
    char* ws = (char*)workspace;
    float* phit = (float*)ws;
    float* pp = (float*)(ws + align256((size_t)k * 32 * 4));
    float* ss = (float*)(ws + align256((size_t)k * 32 * 4) + align256((size_t)ks * batch * 32 * 4));
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = launch_proj_valu(dtype, inp, weight, out_dim, phit, pp, ss, batch, k, ks, s);
    if (e == hipSuccess) e = launch_proj_reduce(pp, ks, batch, out_dim, out, s);
    return hip_status(e);
}
#endif  // MHC_KERNEL_TIMING

struct ProjBwdWs {
    int tiles;
    size_t part_off, stage_off, total;
};

// dPhi partials and column-sum stage for one 32-row output tile at a time
// (the output tiles are reduced one after another through the same buffers).
static int tile_rows(int np) { return np < kProjTile ? np : kProjTile; }

static ProjBwdWs proj_bwd_ws(int64_t batch, int64_t k, int32_t out_dim) {
    ProjBwdWs w{};
    w.tiles = batch > 0 ? proj_bwd_tiles(kF32, batch, k) : 1;
    w.part_off = 0;
    // the partials region also serves the all-tiles path as its dP planes
    size_t part = (size_t)w.tiles * tile_rows(out_dim) * k * sizeof(float);
    if (batch > 0 && proj_bwd_wide_path(kF32, out_dim, batch) && part < proj_bwd_wide_scratch_bytes(out_dim, batch, k))
        part = proj_bwd_wide_scratch_bytes(out_dim, batch, k);
    w.stage_off = align256(part);
    w.total = w.stage_off + align256(column_sums_stage_floats((int64_t)tile_rows(out_dim) * k) * sizeof(float));
    return w;
}

// The projection backward over all output tiles of Phi (rows o0 = 32 t ..):
// dx gets every tile's term (the first tile also s x, or starts from zero
// when !accumulate), and each tile's dPhi partials are column-summed into
// grad_phi rows o0 .. before the next tile reuses the partial buffer.  Many
// tiles with fp32 x and a moderate batch take the two-kernel path instead
// (dx over all tiles in one pass, dPhi written directly).
static hipError_t proj_bwd_all(int x_dtype, const void* x, const float* dp, int dp_stride_, const float* s_tok,
                               const float* phi_pre, const float* phi_post, const float* phi_res, int n_pre, int np,
                               void* dx, bool accumulate, float* part, int tiles, float* stage, float* grad_phi,
                               int64_t batch, int64_t K, hipStream_t s, const int32_t* dx_scale = nullptr,
                               int groups = 0) {
    if (batch > 0 && proj_bwd_wide_path(x_dtype, np, batch))
        return launch_proj_bwd_wide((const float*)x, dp, dp_stride_, s_tok, phi_pre, phi_post, phi_res, n_pre, np,
                                    (float*)dx, accumulate, grad_phi, part, batch, K, s);
    hipError_t e = hipSuccess;
    for (int o0 = 0; o0 < np && e == hipSuccess; o0 += kProjTile) {
        const int rows_t = np - o0 < kProjTile ? np - o0 : kProjTile;
        int rows = tiles;
        if (batch == 0) {
            rows = 1;
            e = launch_fill_zero(part, (int64_t)rows_t * K, s);
        } else {
            e = launch_proj_bwd(x_dtype, x, dp + o0, dp_stride_, o0 == 0 ? s_tok : nullptr, phi_pre, phi_post,
                                phi_res, n_pre, o0, rows_t, dx, accumulate || o0 > 0, part, tiles, batch, K, s,
                                dx_scale, groups);
        }
        if (e == hipSuccess)
            e = launch_column_finalize(0, kF32, part, rows, (int64_t)rows_t * K, stage, grad_phi + (int64_t)o0 * K,
                                      nullptr, 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0.f, s);
    }
    return e;
}

size_t mhc_fused_rmsnorm_matmul_bwd_workspace_size(int64_t batch, int64_t k, int32_t out_dim) {
    if (batch < 0 || k < 1 || out_dim < 1) return 0;
    return proj_bwd_ws(batch, k, out_dim).total;
}

int mhc_fused_rmsnorm_matmul_bwd(const float* grad_out, const float* x_flat, const float* phi, float* grad_x,
                                 float* grad_phi, void* workspace, size_t workspace_bytes, int64_t batch, int64_t k,
                                 int32_t out_dim, void* stream) {
    int st = check_proj("fused_rmsnorm_matmul_bwd", batch, k, out_dim);
    if (st) return st;
    MHC_REQUIRE(phi && grad_phi && (batch == 0 || (grad_out && x_flat && grad_x)),
                "fused_rmsnorm_matmul_bwd: null pointer");
    const ProjBwdWs w = proj_bwd_ws(batch, k, out_dim);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE, "fused_rmsnorm_matmul_bwd: workspace too small");
    hipStream_t s = (hipStream_t)stream;
    float* part = (float*)((char*)workspace + w.part_off);
    float* stage = (float*)((char*)workspace + w.stage_off);
    return hip_status(proj_bwd_all(kF32, x_flat, grad_out, out_dim, nullptr, phi, phi, phi, out_dim, out_dim, grad_x,
                                   false, part, w.tiles, stage, grad_phi, batch, k, s));
}

// ---- fused dynamic-H layer ----------------------------------------------------
// saved (floats): [w32 (C) | coef (B x np) | P (B x np) | r_h (B)], each 64-aligned
struct DynSaved {
    size_t w_off, coef_off, p_off, rh_off, total;
};

static DynSaved dyn_saved(int64_t batch, int32_t n, int32_t hidden) {
    const size_t np = 2 * n + n * n;
    DynSaved d{};
    d.w_off = 0;
    d.coef_off = align_floats(hidden);
    d.p_off = d.coef_off + align_floats(batch * np);
    d.rh_off = d.p_off + align_floats(batch * np);
    d.total = d.rh_off + align_floats(batch);
    return d;
}

size_t mhc_layer_dynamic_saved_size(int64_t batch, int32_t n, int32_t hidden) {
    if (batch < 0 || n < 1 || hidden < 1) return 0;
    return dyn_saved(batch, n, hidden).total * sizeof(float);
}

size_t mhc_layer_dynamic_fwd_workspace_size(int64_t batch, int32_t n, int32_t hidden) {
    if (batch < 0 || n < 1 || hidden < 1) return 0;
    return proj_fwd_ws(batch, (int64_t)n * hidden, 2 * n + n * n).total;
}

static int check_dyn(const char* fn, int64_t batch, int32_t n, int32_t hidden, int32_t x_dtype, int32_t w_dtype,
                     int32_t num_iters) {
    int st = check_layer_shape(fn, batch, n, hidden, x_dtype, num_iters);
    if (st) return st;
    if (!valid_dtype(w_dtype)) return fail(MHC_ERR_INVALID, std::string(fn) + ": weight_dtype must be F32 or BF16");
    if (!supported_dynamic_n(n))
        return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": n=" + std::to_string(n) +
                                             " is not supported (1 <= n <= " + std::to_string(kGenMaxN) + ")");
    if (((int64_t)n * hidden) % 32 != 0)
        return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": n*hidden must be a multiple of 32");
    return MHC_SUCCESS;
}

int mhc_layer_dynamic_fwd(const void* x, int32_t x_dtype, const void* weight, int32_t weight_dtype,
                          const float* phi_pre, const float* phi_post, const float* phi_res, const float* alpha_pre,
                          const float* alpha_post, const float* alpha_res, const float* b_pre, const float* b_post,
                          const float* b_res, float* out, float* saved, void* workspace, size_t workspace_bytes,
                          int64_t batch, int32_t n, int32_t hidden, int32_t num_iters, float sinkhorn_eps,
                          float rmsnorm_eps, void* stream) {
    int st = check_dyn("layer_dynamic_fwd", batch, n, hidden, x_dtype, weight_dtype, num_iters);
    if (st) return st;
    MHC_REQUIRE(weight && phi_pre && phi_post && phi_res && alpha_pre && alpha_post && alpha_res && b_pre &&
                    b_post && b_res && saved,
                "layer_dynamic_fwd: null parameter pointer");
    MHC_REQUIRE(batch == 0 || (x && out), "layer_dynamic_fwd: null x/out");
    hipStream_t s = (hipStream_t)stream;
    const DynSaved d = dyn_saved(batch, n, hidden);
    float* w32 = saved + d.w_off;
    const int64_t K = (int64_t)n * hidden;
    const ProjFwdWs w = proj_fwd_ws(batch, K, 2 * n + n * n);
    hipError_t e = hipSuccess;
    // the weight's fp32 copy: its own launch, or inside the Phi split's
    if (batch == 0 || w.stream) e = launch_weight_f32(weight, weight_dtype, hidden, w32, s);
    if (e != hipSuccess || batch == 0) return hip_status(e);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE, "layer_dynamic_fwd: workspace smaller than mhc_layer_dynamic_fwd_workspace_size()");
    bf16_raw_t* phib = (bf16_raw_t*)((char*)workspace + w.phib_off);
    float* pp = (float*)((char*)workspace + w.p_off);
    float* ss = (float*)((char*)workspace + w.ss_off);
    const int np = 2 * n + n * n;
    if (w.stream) {
        e = launch_proj_stream(x_dtype, x, (bf16_raw_t*)((char*)workspace + w.xpl_off), phi_pre, phi_post, phi_res,
                               n, nullptr, np, pp, ss, batch, K, w.ks, s);
    } else {
        e = launch_phi_split(phi_pre, phi_post, phi_res, n, np, K, phib, s, weight, weight_dtype, hidden, w32);
        if (e == hipSuccess) {
            if (proj_one_pass(x_dtype, np, batch))
                e = launch_proj_stream(x_dtype, x, nullptr, phi_pre, phi_post, phi_res, n, phib, np, pp, ss, batch, K,
                                       w.ks, s);
            else
                e = launch_proj_mfma(x_dtype, x, phib, np, pp, ss, batch, K, w.ks, s);
        }
    }
    if (e == hipSuccess)
        e = launch_dyn_coef_fwd(n, pp, ss, w.ks, batch, K, alpha_pre, alpha_post, alpha_res, b_pre, b_post, b_res,
                                saved + d.coef_off, saved + d.p_off, saved + d.rh_off, num_iters, sinkhorn_eps,
                                rmsnorm_eps, s);
    // the channel-loop forward uses the sum x^2 partials (ks * batch floats,
    // free once the coefficients are formed) as scratch for its row sums
    float* rs = layer_fwd_is_wide(n, hidden) ? ss : nullptr;
    if (e == hipSuccess)
        e = launch_layer_fwd(x_dtype, n, x, w32, saved + d.coef_off, np, out, kF32, rs, batch, hidden, rmsnorm_eps, s,
                             rs ? (int64_t)w.ks * batch : 0);
    return hip_status(e);
}

// ---- forward-only dynamic-H layer ---------------------------------------------
// packed: [w32 (C floats) | Phi as three bf16 planes in fragment order], the
// planes 256-byte aligned.  workspace: [coef (B x np) | projection partials].
static size_t packed_phib_off(int32_t hidden) { return align256((size_t)hidden * sizeof(float)); }

size_t mhc_layer_dynamic_packed_size(int32_t n, int32_t hidden) {
    if (n < 1 || hidden < 1) return 0;
    return packed_phib_off(hidden) + phi_planes_bytes((int64_t)n * hidden, 2 * n + n * n);
}

int mhc_layer_dynamic_pack(const void* weight, int32_t weight_dtype, const float* phi_pre, const float* phi_post,
                           const float* phi_res, void* packed, size_t packed_bytes, int32_t n, int32_t hidden,
                           void* stream) {
    int st = check_dyn("layer_dynamic_pack", 0, n, hidden, kF32, weight_dtype, 0);
    if (st) return st;
    MHC_REQUIRE(weight && phi_pre && phi_post && phi_res && packed, "layer_dynamic_pack: null pointer");
    if (packed_bytes < mhc_layer_dynamic_packed_size(n, hidden))
        return fail(MHC_ERR_WORKSPACE, "layer_dynamic_pack: buffer smaller than mhc_layer_dynamic_packed_size()");
    hipStream_t s = (hipStream_t)stream;
    const int64_t K = (int64_t)n * hidden;
    hipError_t e = launch_weight_f32(weight, weight_dtype, hidden, (float*)packed, s);
    if (e == hipSuccess)
        e = launch_phi_split(phi_pre, phi_post, phi_res, n, 2 * n + n * n, K,
                             (bf16_raw_t*)((char*)packed + packed_phib_off(hidden)), s);
    return hip_status(e);
}

static size_t infer_proj_off(int64_t batch, int32_t n) { return align256((size_t)batch * (2 * n + n * n) * 4); }

size_t mhc_layer_dynamic_infer_workspace_size(int64_t batch, int32_t n, int32_t hidden) {
    if (batch < 0 || n < 1 || hidden < 1) return 0;
    const ProjFwdWs w = proj_fwd_ws(batch, (int64_t)n * hidden, 2 * n + n * n);
    return infer_proj_off(batch, n) + (w.total - w.xpl_off);
}

int mhc_layer_dynamic_infer(const void* x, int32_t x_dtype, const void* packed, const float* alpha_pre,
                            const float* alpha_post, const float* alpha_res, const float* b_pre, const float* b_post,
                            const float* b_res, void* out, int32_t out_dtype, void* workspace, size_t workspace_bytes,
                            int64_t batch, int32_t n, int32_t hidden, int32_t num_iters, float sinkhorn_eps,
                            float rmsnorm_eps, void* stream) {
    int st = check_dyn("layer_dynamic_infer", batch, n, hidden, x_dtype, kF32, num_iters);
    if (st) return st;
    if (!valid_dtype(out_dtype)) return fail(MHC_ERR_INVALID, "layer_dynamic_infer: out_dtype must be F32 or BF16");
    MHC_REQUIRE(packed && alpha_pre && alpha_post && alpha_res && b_pre && b_post && b_res,
                "layer_dynamic_infer: null parameter pointer");
    if (batch == 0) return MHC_SUCCESS;
    MHC_REQUIRE(x && out, "layer_dynamic_infer: null x/out");
    if (!workspace || workspace_bytes < mhc_layer_dynamic_infer_workspace_size(batch, n, hidden))
        return fail(MHC_ERR_WORKSPACE,
                    "layer_dynamic_infer: workspace smaller than mhc_layer_dynamic_infer_workspace_size()");
    hipStream_t s = (hipStream_t)stream;
    const int64_t K = (int64_t)n * hidden;
    const int np = 2 * n + n * n;
    const ProjFwdWs w = proj_fwd_ws(batch, K, np);
    const float* w32 = (const float*)packed;
    const bf16_raw_t* phib = (const bf16_raw_t*)((const char*)packed + packed_phib_off(hidden));
    float* coef = (float*)workspace;
    // [coef | x planes (streaming path) | P partials | sum x^2 partials]
    char* pw = (char*)workspace + infer_proj_off(batch, n);
    float* pp = (float*)(pw + (w.p_off - w.xpl_off));
    float* ss = (float*)(pw + (w.ss_off - w.xpl_off));
    hipError_t e = hipSuccess;
    if (w.stream) {
        e = launch_proj_stream(x_dtype, x, (bf16_raw_t*)pw, nullptr, nullptr, nullptr, n, phib, np, pp, ss, batch, K,
                               w.ks, s);
    } else if (proj_one_pass(x_dtype, np, batch)) {
        e = launch_proj_stream(x_dtype, x, nullptr, nullptr, nullptr, nullptr, n, phib, np, pp, ss, batch, K, w.ks, s);
    } else {
        e = launch_proj_mfma(x_dtype, x, phib, np, pp, ss, batch, K, w.ks, s);
    }
    if (e == hipSuccess)
        e = launch_dyn_coef_fwd(n, pp, ss, w.ks, batch, K, alpha_pre, alpha_post, alpha_res, b_pre, b_post, b_res,
                                coef, nullptr, nullptr, num_iters, sinkhorn_eps, rmsnorm_eps, s);
    float* rs = layer_fwd_is_wide(n, hidden) ? ss : nullptr;  // as in mhc_layer_dynamic_fwd
    if (e == hipSuccess)
        e = launch_layer_fwd(x_dtype, n, x, w32, coef, np, out, out_dtype, rs, batch, hidden, rmsnorm_eps, s,
                             rs ? (int64_t)w.ks * batch : 0);
    return hip_status(e);
}

// dx of bf16 x is rounded to bf16 once, from the fp32 sum of the row pass's
// stream part and the projection's terms, as the reference's fp32 autograd
// does.  With one 32-row projection tile at n = 2 and 4 on the register-row
// kernels and hidden % 128 == 0 the stream part travels as fp16 against a
// power-of-two scale (11 significant bits; one scale exponent per half wave
// of the row kernel and token, in the workspace) and the projection kernel
// rounds the sum: each element's stream part then enters the sum with a
// relative error of at most 2^-11 (an eighth of the bf16 half-ulp) down to
// 2^-28 of its group's largest element, and within 2^-39 of that largest
// element below.  Otherwise (n = 3, n >= 5, rows the channel-loop kernels take,
// other hidden sizes) dx accumulates in fp32 across the kernels, which read x
// itself or an exact fp32 copy of it.
static bool dyn_bwd_f32_acc(int32_t n, int32_t hidden, int32_t x_dtype) {
    return x_dtype == kBF16 &&
           (odd_row_n(n) || 2 * n + n * n > kProjTile || layer_bwd_is_wide(n, hidden) || hidden % 128 != 0);
}

struct DynBwdWs {
    int grid, cblocks, tiles;
    int wdt;     // element type the row and projection kernels run on
    int groups;  // scale groups per token of the bf16 stream part
    size_t dw_off, scal_off, dp_off, s_off, pscale_off, cpart_off, phip_off, stw_off, stp_off, xw_off, dxw_off, hist_off,
        rows_off, total;
};

static DynBwdWs dyn_bwd_ws(int64_t batch, int32_t n, int32_t hidden, int32_t x_dtype, bool aligned) {
    DynBwdWs w{};
    const int64_t np = 2 * n + n * n;
    const int64_t K = (int64_t)n * hidden;
    w.wdt = dyn_bwd_f32_acc(n, hidden, x_dtype) ? kF32 : x_dtype;
    w.grid = batch > 0 ? layer_bwd_grid(w.wdt, n, batch, hidden, aligned) : 1;
    w.cblocks = batch > 0 ? dyn_coef_bwd_blocks(n, batch) : 1;
    w.tiles = batch > 0 ? proj_bwd_tiles(w.wdt, batch, (int64_t)n * hidden) : 1;
    size_t o = 0;
    w.dw_off = o; o += align256((size_t)w.grid * hidden * 4);
    w.scal_off = o; o += align256((size_t)batch * (n * n + 2 * n + 2) * 4);
    w.dp_off = o; o += align256((size_t)batch * dp_stride((int)np) * 4);
    w.s_off = o; o += align256((size_t)batch * 4);
    // scale exponents of the bf16 stream part
    w.groups = w.wdt == kBF16 ? layer_bwd_part_groups(w.wdt, n, hidden) : 0;
    w.pscale_off = o; o += align256((size_t)batch * w.groups * 4);
    w.cpart_off = o; o += align256((size_t)w.cblocks * (np + 3) * 4);
    // projection partials (per-tile path) or dP planes (all-tiles path)
    const bool all = batch > 0 && w.wdt == kF32 && proj_bwd_tiles_path((int)np, batch);
    const int64_t prows = all ? np : tile_rows((int)np);
    size_t phip = (size_t)w.tiles * prows * K * 4;
    if (batch > 0 && proj_bwd_wide_path(w.wdt, (int)np, batch) &&
        phip < proj_bwd_wide_scratch_bytes((int)np, batch, K))
        phip = proj_bwd_wide_scratch_bytes((int)np, batch, K);
    w.phip_off = o; o += align256(phip);
    w.stw_off = o; o += align256(column_sums_stage_floats(hidden) * 4);
    w.stp_off = o; o += align256(column_sums_stage_floats(prows * K) * 4);
    const size_t acc = w.wdt != x_dtype ? (size_t)batch * K * 4 : 0;
    w.xw_off = o; o += align256(acc);
    w.dxw_off = o; o += align256(acc);
    // Sinkhorn adjoint history (fixed n >= 16: kSkHistBytes; generic n: the
    // region dyn_coef_gen_hist_bytes sizes for the batch)
    w.hist_off = o;
    o += n >= 16 && !generic_layer_n(n) && batch > 0 ? kSkHistBytes : align256(dyn_coef_gen_hist_bytes(n, batch));
    w.rows_off = o; o += align256(batch > 0 ? layer_bwd_scratch_bytes(w.wdt, n, batch, hidden, aligned) : 0);
    w.total = o;
    return w;
}

static size_t dyn_bwd_ws_bytes(int64_t batch, int32_t n, int32_t hidden, int32_t x_dtype) {
    const size_t a = dyn_bwd_ws(batch, n, hidden, x_dtype, true).total;
    const size_t u = odd_row_n(n) ? dyn_bwd_ws(batch, n, hidden, x_dtype, false).total : 0;
    return a > u ? a : u;
}

size_t mhc_layer_dynamic_bwd_workspace_size(int64_t batch, int32_t n, int32_t hidden, int32_t x_dtype) {
    if (batch < 0 || n < 1 || hidden < 1) return 0;
    return dyn_bwd_ws_bytes(batch, n, hidden, x_dtype);
}

int mhc_layer_dynamic_bwd(const float* grad_out, const void* x, int32_t x_dtype, int32_t weight_dtype,
                          const float* phi_pre, const float* phi_post, const float* phi_res, const float* alpha_pre,
                          const float* alpha_post, const float* alpha_res, const float* b_pre, const float* b_post,
                          const float* b_res, const float* saved, void* grad_x, void* grad_weight, float* grad_phi,
                          float* grad_alpha, float* grad_b, void* workspace, size_t workspace_bytes, int64_t batch,
                          int32_t n, int32_t hidden, int32_t num_iters, float sinkhorn_eps, float rmsnorm_eps,
                          void* stream) {
    (void)b_pre;
    (void)b_post;
    int st = check_dyn("layer_dynamic_bwd", batch, n, hidden, x_dtype, weight_dtype, num_iters);
    if (st) return st;
    MHC_REQUIRE(phi_pre && phi_post && phi_res && alpha_pre && alpha_post && alpha_res && b_res && saved,
                "layer_dynamic_bwd: null parameter pointer");
    MHC_REQUIRE(grad_weight && grad_phi && grad_alpha && grad_b, "layer_dynamic_bwd: null gradient pointer");
    MHC_REQUIRE(batch == 0 || (grad_out && x && grad_x), "layer_dynamic_bwd: null grad_out/x/grad_x");
    const bool aligned = rows_aligned(n, {grad_out, x, grad_x, saved, workspace});
    const DynBwdWs w = dyn_bwd_ws(batch, n, hidden, x_dtype, aligned);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE, "layer_dynamic_bwd: workspace smaller than mhc_layer_dynamic_bwd_workspace_size()");
    if (n >= 16 && !generic_layer_n(n) && batch > 0 && dyn_coef_bwd_hist_slots(n, batch, num_iters) < 1)
        return fail(MHC_ERR_UNSUPPORTED, "layer_dynamic_bwd: num_iters too large for the Sinkhorn history at n=" +
                                             std::to_string(n));
    hipStream_t s = (hipStream_t)stream;
    char* ws = (char*)workspace;
    float* dw_part = (float*)(ws + w.dw_off);
    float* scal = (float*)(ws + w.scal_off);
    float* dp = (float*)(ws + w.dp_off);
    float* stok = (float*)(ws + w.s_off);
    float* cpart = (float*)(ws + w.cpart_off);
    float* phip = (float*)(ws + w.phip_off);
    float* stw = (float*)(ws + w.stw_off);
    float* stp = (float*)(ws + w.stp_off);
    float* xw = (float*)(ws + w.xw_off);
    float* dxw = (float*)(ws + w.dxw_off);
    int32_t* pscale = w.wdt == kBF16 ? (int32_t*)(ws + w.pscale_off) : nullptr;
    // the tensors the row and projection kernels work on
    // (direct: the pass over all output tiles and the row kernel read bf16 x
    // itself, where x and dx take 16-byte pieces and the rows fit registers:
    // n = 8, 4096 x 2048 bf16 583 us of kernels with the fp32 copy of x, 497
    // without; n = 3 runs that pass for this, one tile)
    const bool bf16_direct = x_dtype == kBF16 && ((uintptr_t)x | (uintptr_t)grad_x) % 16 == 0 &&
                             layer_bwd_f32_dx_ok(n, hidden, aligned);
    const bool all_tiles = batch > 0 && w.wdt == kF32 &&
                           (proj_bwd_tiles_path(2 * n + n * n, batch) || (n == 3 && bf16_direct));
    const bool direct = all_tiles && (w.wdt == x_dtype || bf16_direct);
    const void* xk = w.wdt != x_dtype && !direct ? (const void*)xw : x;
    void* dxk = w.wdt != x_dtype ? (void*)dxw : grad_x;
    const DynSaved d = dyn_saved(batch, n, hidden);
    const int np = 2 * n + n * n;
    const int64_t K = (int64_t)n * hidden;
    const float* w32 = saved + d.w_off;
    hipError_t e = hipSuccess;
    int rows_w = w.grid, rows_p = w.tiles, rows_c = dyn_coef_bwd_rows(n, batch, num_iters, true);
    if (batch == 0) {
        rows_w = rows_c = 1;
        e = launch_fill_zero(dw_part, hidden, s);
        if (e == hipSuccess) e = launch_fill_zero(cpart, np + 3, s);
    } else {
        if (w.wdt != x_dtype && !direct) e = launch_weight_f32(x, x_dtype, batch * K, xw, s);
        if (e == hipSuccess)
            e = launch_layer_bwd(direct ? x_dtype : w.wdt, n, direct && x_dtype == kBF16 ? 2 : 1, grad_out, xk, w32,
                                 saved + d.coef_off, np, dxk, dw_part, scal, w.grid, batch, hidden, rmsnorm_eps,
                                 (float*)(ws + w.rows_off), s, pscale, aligned);
        if (e == hipSuccess)
            e = launch_dyn_coef_bwd(n, scal, saved + d.coef_off, saved + d.p_off, saved + d.rh_off, batch, K,
                                    alpha_pre, alpha_post, alpha_res, b_res, dp, stok, cpart, num_iters, sinkhorn_eps,
                                    (n >= 16 || generic_layer_n(n)) ? (float*)(ws + w.hist_off) : nullptr, s);
    }
    // One projection tile (n <= 4) and few partial rows: the column sums of
    // dPhi, dw and the db / dalpha partials in one launch after the
    // projection backward.
    const bool one_sum = batch > 0 && np <= kProjTile && !proj_bwd_wide_path(w.wdt, np, batch) &&
                         column_sums_direct(rows_p) && column_sums_direct(rows_w) && column_sums_direct(rows_c);
    if (one_sum) {
        if (e == hipSuccess && all_tiles)
            e = launch_proj_bwd_tiles(x_dtype, x, dp, dp_stride(np), stok, phi_pre, phi_post, phi_res, n, np,
                                      (const float*)dxk, grad_x, phip, rows_p, batch, K, s);
        else if (e == hipSuccess)
            e = launch_proj_bwd(w.wdt, xk, dp, dp_stride(np), stok, phi_pre, phi_post, phi_res, n, 0, np, dxk, true,
                                phip, rows_p, batch, K, s, pscale, w.groups);
        if (e == hipSuccess && w.wdt != x_dtype && !direct) e = launch_cast_bf16(dxw, batch * K, grad_x, s);
        if (e == hipSuccess) {
            ColSumJobs jobs{};
            jobs.j[0] = ColSumJob{phip, grad_phi, nullptr, (int64_t)np * K, rows_p, (int)(np * K), 0, 0, 0};
            jobs.j[1] = ColSumJob{dw_part, grad_weight, nullptr, hidden, rows_w, hidden, weight_dtype == kBF16, 0, 0};
            jobs.j[2] = ColSumJob{cpart, grad_b, grad_alpha, np + 3, rows_c, np, 0, 0, 0};
            jobs.count = 3;
            e = launch_multi_column_sum(jobs, s);
        }
        return hip_status(e);
    }
    if (all_tiles) {
        if (e == hipSuccess)
            e = launch_proj_bwd_tiles(direct ? x_dtype : w.wdt, xk, dp, dp_stride(np), stok, phi_pre,
                                      phi_post, phi_res, n, np, (const float*)dxk, direct ? grad_x : dxk, phip, rows_p,
                                      batch, K, s);
        if (e == hipSuccess && !direct) e = launch_cast_bf16(dxw, batch * K, grad_x, s);
        if (e == hipSuccess)
            e = launch_column_finalize(0, kF32, phip, rows_p, (int64_t)np * K, stp, grad_phi, nullptr, 0, nullptr,
                                       nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0.f, s);
    } else {
        if (e == hipSuccess)
            e = proj_bwd_all(w.wdt, xk, dp, dp_stride(np), stok, phi_pre, phi_post, phi_res, n, np, dxk, true, phip,
                             rows_p, stp, grad_phi, batch, K, s, pscale, w.groups);
        if (e == hipSuccess && w.wdt != x_dtype) e = launch_cast_bf16(dxw, batch * K, grad_x, s);
    }
    if (e == hipSuccess)
        e = launch_column_finalize(0, weight_dtype, dw_part, rows_w, hidden, stw, grad_weight, nullptr, 0, nullptr, nullptr,
                                  nullptr, nullptr, nullptr, nullptr, 0, 0.f, s);
    if (e == hipSuccess) e = launch_small_column_sum(cpart, rows_c, np + 3, grad_b, grad_alpha, np, s);
    return hip_status(e);
}

// ---- reference-shaped dynamic-H entries ----------------------------------------
// The calls of the reference's native module as its ops.py makes them (the
// nine-tensor forward, the 23-argument backward), over the fused entries.
//
// forward workspace: [alphas (3 floats) | fused saved state | fused forward workspace]
struct RefFwdWs {
    size_t alpha_off, saved_off, fwd_off, total;
};

static RefFwdWs ref_fwd_ws(int64_t batch, int32_t n, int32_t hidden) {
    RefFwdWs w{};
    w.alpha_off = 0;
    w.saved_off = 256;
    w.fwd_off = w.saved_off + align256(dyn_saved(batch, n, hidden).total * sizeof(float));
    w.total = w.fwd_off + align256(mhc_layer_dynamic_fwd_workspace_size(batch, n, hidden));
    return w;
}

size_t mhc_layer_fwd_dynamic_workspace_size(int64_t batch, int32_t n, int32_t hidden) {
    if (batch < 0 || n < 1 || hidden < 1) return 0;
    return ref_fwd_ws(batch, n, hidden).total;
}

int mhc_layer_fwd_dynamic(const void* x, int32_t x_dtype, const void* weight, int32_t weight_dtype,
                          const float* phi_concat, float alpha_pre, float alpha_post, float alpha_res,
                          const float* b_pre, const float* b_post, const float* b_res, float* output, float* rms,
                          void* x_agg_bf16, float* h_pre_act, float* h_post_act, float* M, void* y_norm_bf16,
                          void* x_flat_bf16, float* rms_h, void* workspace, size_t workspace_bytes, int64_t batch,
                          int32_t n, int32_t hidden, int32_t num_iters, float sinkhorn_eps, float rmsnorm_eps,
                          void* stream) {
    int st = check_dyn("layer_fwd_dynamic", batch, n, hidden, x_dtype, weight_dtype, num_iters);
    if (st) return st;
    MHC_REQUIRE(weight && phi_concat && b_pre && b_post && b_res, "layer_fwd_dynamic: null parameter pointer");
    MHC_REQUIRE(batch == 0 || (x && output && rms && x_agg_bf16 && h_pre_act && h_post_act && M && y_norm_bf16 &&
                               x_flat_bf16 && rms_h),
                "layer_fwd_dynamic: null x or output pointer");
    const RefFwdWs w = ref_fwd_ws(batch, n, hidden);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE, "layer_fwd_dynamic: workspace smaller than mhc_layer_fwd_dynamic_workspace_size()");
    hipStream_t s = (hipStream_t)stream;
    char* ws = (char*)workspace;
    float* alphas = (float*)(ws + w.alpha_off);
    float* saved = (float*)(ws + w.saved_off);
    const int64_t K = (int64_t)n * hidden;
    hipError_t e = launch_set_scalars(alphas, alpha_pre, alpha_post, alpha_res, s);
    if (e != hipSuccess) return hip_status(e);
    st = mhc_layer_dynamic_fwd(x, x_dtype, weight, weight_dtype, phi_concat, phi_concat + n * K,
                               phi_concat + 2 * n * K, alphas, alphas + 1, alphas + 2, b_pre, b_post, b_res, output,
                               saved, ws + w.fwd_off, w.total - w.fwd_off, batch, n, hidden, num_iters, sinkhorn_eps,
                               rmsnorm_eps, stream);
    if (st) return st;
    const DynSaved d = dyn_saved(batch, n, hidden);
    return hip_status(launch_dyn_intermediates(x_dtype, x, saved + d.w_off, saved + d.coef_off, saved + d.rh_off, n,
                                               batch, hidden, rmsnorm_eps, rms, x_agg_bf16, y_norm_bf16, x_flat_bf16,
                                               h_pre_act, h_post_act, M, rms_h, s));
}

// backward workspace: [alphas | grad_alpha (3) + grad_b (np) | fused saved
// state | projection (P recompute), then the fused backward's workspace |
// grad_phi rows when the caller's three blocks are not consecutive]
struct RefBwdWs {
    size_t alpha_off, small_off, saved_off, work_off, gphi_off, total;
};

static RefBwdWs ref_bwd_ws(int64_t batch, int32_t n, int32_t hidden, int32_t x_dtype) {
    const int np = 2 * n + n * n;
    const int64_t K = (int64_t)n * hidden;
    RefBwdWs w{};
    w.alpha_off = 0;
    w.small_off = 256;
    w.saved_off = w.small_off + align256((size_t)(3 + np) * sizeof(float));
    w.work_off = w.saved_off + align256(dyn_saved(batch, n, hidden).total * sizeof(float));
    size_t work = dyn_bwd_ws_bytes(batch, n, hidden, x_dtype);
    const size_t proj = proj_fwd_ws(batch, K, np).total;
    if (proj > work) work = proj;
    w.gphi_off = w.work_off + align256(work);
    w.total = w.gphi_off + align256((size_t)np * K * sizeof(float));
    return w;
}

size_t mhc_layer_bwd_dynamic_workspace_size(int64_t batch, int32_t n, int32_t hidden, int32_t x_dtype) {
    if (batch < 0 || n < 1 || hidden < 1) return 0;
    return ref_bwd_ws(batch, n, hidden, x_dtype).total;
}

int mhc_layer_bwd_dynamic(const float* grad_output, const void* x, int32_t x_dtype, const void* weight,
                          int32_t weight_dtype, const float* rms, const void* x_agg_bf16, const float* h_pre_act,
                          const float* h_post_act, const float* M, const void* y_norm_bf16, const void* x_flat_bf16,
                          const float* rms_h, const float* phi_pre, const float* phi_post, const float* phi_res,
                          float alpha_pre, float alpha_post, float alpha_res, const float* b_pre, const float* b_post,
                          const float* b_res, void* grad_x, float* grad_weight, float* grad_phi_pre,
                          float* grad_phi_post, float* grad_phi_res, float* grad_alpha_pre, float* grad_alpha_post,
                          float* grad_alpha_res, float* grad_b_pre, float* grad_b_post, float* grad_b_res,
                          void* workspace, size_t workspace_bytes, int64_t batch, int32_t n, int32_t hidden,
                          int32_t num_iters, float sinkhorn_eps, float rmsnorm_eps, void* stream) {
    // rms, x_agg, y_norm and x_flat are recomputed in fp32 from x inside the
    // fused row pass; they are accepted for the reference's call shape.
    (void)rms;
    (void)x_agg_bf16;
    (void)y_norm_bf16;
    (void)x_flat_bf16;
    int st = check_dyn("layer_bwd_dynamic", batch, n, hidden, x_dtype, weight_dtype, num_iters);
    if (st) return st;
    MHC_REQUIRE(weight && phi_pre && phi_post && phi_res && b_res, "layer_bwd_dynamic: null parameter pointer");
    MHC_REQUIRE(grad_weight && grad_phi_pre && grad_phi_post && grad_phi_res && grad_alpha_pre && grad_alpha_post &&
                    grad_alpha_res && grad_b_pre && grad_b_post && grad_b_res,
                "layer_bwd_dynamic: null gradient pointer");
    MHC_REQUIRE(batch == 0 || (grad_output && x && grad_x && h_pre_act && h_post_act && M && rms_h),
                "layer_bwd_dynamic: null grad_output / x / saved tensor / grad_x");
    const RefBwdWs w = ref_bwd_ws(batch, n, hidden, x_dtype);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE,
                    "layer_bwd_dynamic: workspace smaller than mhc_layer_bwd_dynamic_workspace_size()");
    hipStream_t s = (hipStream_t)stream;
    char* ws = (char*)workspace;
    const int np = 2 * n + n * n;
    const int64_t K = (int64_t)n * hidden;
    float* alphas = (float*)(ws + w.alpha_off);
    float* galpha = (float*)(ws + w.small_off);
    float* gb = galpha + 3;
    float* saved = (float*)(ws + w.saved_off);
    char* work = ws + w.work_off;
    const DynSaved d = dyn_saved(batch, n, hidden);
    hipError_t e = launch_set_scalars(alphas, alpha_pre, alpha_post, alpha_res, s);
    if (e == hipSuccess) e = launch_weight_f32(weight, weight_dtype, hidden, saved + d.w_off, s);
    if (e == hipSuccess && batch > 0) {
        // P = x_flat . Phi^T again (bindings.cpp:764-766), into the saved state
        const ProjFwdWs p = proj_fwd_ws(batch, K, np);
        float* pp = (float*)(work + p.p_off);
        float* ss = (float*)(work + p.ss_off);
        if (p.stream) {
            e = launch_proj_stream(x_dtype, x, (bf16_raw_t*)(work + p.xpl_off), phi_pre, phi_post, phi_res, n,
                                   nullptr, np, pp, ss, batch, K, p.ks, s);
        } else {
            e = launch_phi_split(phi_pre, phi_post, phi_res, n, np, K, (bf16_raw_t*)(work + p.phib_off), s);
            if (e == hipSuccess)
                e = launch_proj_mfma(x_dtype, x, (const bf16_raw_t*)(work + p.phib_off), np, pp, ss, batch, K, p.ks,
                                     s);
        }
        if (e == hipSuccess) e = launch_proj_reduce(pp, p.ks, batch, np, saved + d.p_off, s);
        if (e == hipSuccess)
            e = launch_dyn_saved_assemble(h_pre_act, h_post_act, M, rms_h, n, batch, saved + d.coef_off,
                                          saved + d.rh_off, s);
    }
    if (e != hipSuccess) return hip_status(e);
    const bool consecutive = grad_phi_post == grad_phi_pre + (int64_t)n * K &&
                             grad_phi_res == grad_phi_post + (int64_t)n * K;
    float* gphi = consecutive ? grad_phi_pre : (float*)(ws + w.gphi_off);
    st = mhc_layer_dynamic_bwd(grad_output, x, x_dtype, kF32, phi_pre, phi_post, phi_res, alphas, alphas + 1,
                               alphas + 2, b_pre, b_post, b_res, saved, grad_x, grad_weight, gphi, galpha, gb, work,
                               w.gphi_off - w.work_off, batch, n, hidden, num_iters, sinkhorn_eps, rmsnorm_eps,
                               stream);
    if (st) return st;
    auto d2d = [&](void* dst, const void* src, size_t bytes) {
        if (e == hipSuccess) e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, s);
    };
    if (!consecutive) {
        d2d(grad_phi_pre, gphi, (size_t)n * K * sizeof(float));
        d2d(grad_phi_post, gphi + (int64_t)n * K, (size_t)n * K * sizeof(float));
        d2d(grad_phi_res, gphi + (int64_t)2 * n * K, (size_t)n * n * K * sizeof(float));
    }
    d2d(grad_alpha_pre, galpha, sizeof(float));
    d2d(grad_alpha_post, galpha + 1, sizeof(float));
    d2d(grad_alpha_res, galpha + 2, sizeof(float));
    d2d(grad_b_pre, gb, (size_t)n * sizeof(float));
    d2d(grad_b_post, gb + n, (size_t)n * sizeof(float));
    d2d(grad_b_res, gb + 2 * n, (size_t)n * n * sizeof(float));
    return hip_status(e);
}

// ---- fused MHCResidualWrapper ------------------------------------------------
// The n = 4 kernels of wrapper.hip: rows of whole 4-channel chunks that the
// register-row kernels hold, 32-channel rows with dynamic H (the
// projection's k step).  Every other accepted shape runs the run-time-n
// kernels of wrapper_gen.hip.
static bool wrap_fused4(int32_t n, int32_t hidden, bool dynamic) {
    return n == 4 && hidden % 4 == 0 && (!dynamic || hidden % 32 == 0) && choose_row_tiling(hidden, 4, 6).vpt > 0;
}

static int check_wrapper(const char* fn, int64_t tokens, int32_t n, int32_t hidden, int32_t dtype, int32_t w_dtype,
                         int32_t mode, int32_t num_iters, bool dynamic) {
    if (tokens < 0) return fail(MHC_ERR_INVALID, std::string(fn) + ": tokens must be >= 0");
    if (hidden < 1) return fail(MHC_ERR_INVALID, std::string(fn) + ": hidden must be >= 1");
    if (num_iters < 0) return fail(MHC_ERR_INVALID, std::string(fn) + ": num_iters must be >= 0");
    if (!valid_dtype(dtype)) return fail(MHC_ERR_INVALID, std::string(fn) + ": dtype must be F32 or BF16");
    // the reference writes stream 1 (layer.py:301), which needs n >= 2
    if (n < 2) return fail(MHC_ERR_INVALID, std::string(fn) + ": n must be >= 2 (stream 1 holds the branch)");
    if (n > kWgMaxN)
        return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": the fused wrapper takes n <= " + std::to_string(kWgMaxN));
    if (hidden % 4 != 0)
        return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": the fused wrapper needs hidden % 4 == 0");
    if (!valid_dtype(w_dtype)) return fail(MHC_ERR_INVALID, std::string(fn) + ": weight_dtype must be F32 or BF16");
    if (mode != MHC_WRAPPER_DECAY && mode != MHC_WRAPPER_ZERO)
        return fail(MHC_ERR_INVALID, std::string(fn) + ": residual_mode must be MHC_WRAPPER_DECAY or MHC_WRAPPER_ZERO");
    if (!wrap_fused4(n, hidden, dynamic)) {
        if (!wgen_supported(n, hidden))
            return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": hidden too large for the wrapper kernels");
        if (dynamic && ((int64_t)n * hidden) % 32 != 0)
            return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": n*hidden must be a multiple of 32");
        if (dynamic && (int64_t)n * hidden > (int64_t(1) << 22))
            return fail(MHC_ERR_UNSUPPORTED, std::string(fn) + ": n*hidden > 4194304 is not supported");
    }
    return MHC_SUCCESS;
}

size_t mhc_wrapper_dynamic_saved_size(int64_t tokens, int32_t n, int32_t hidden) {
    return mhc_layer_dynamic_saved_size(tokens, n, hidden);
}

static bool wrap_res_grad_vanishes(int32_t num_iters, float sinkhorn_eps);

// ---- run-time-n wrapper (wrapper_gen.hip) ---------------------------------------
// The row passes rebuild the streams from r and b, and so does the forward
// projection where hidden % 8 == 0; otherwise, and in the backward's general
// case, the layer's projection kernels take the stream rows X [tokens, n*C]
// from wgen_synth_kernel, and the backward folds their dX over the streams.
//
// dynamic forward workspace: the folded projection's (wfold_ws), or, for
// hidden sizes it does not take (hidden % 8 != 0), [the layer projection's
// workspace (proj_fwd_ws) | X].
struct WgenFwdWs {
    ProjFwdWs p;
    size_t x_off, total;
};

static WgenFwdWs wgen_fwd_ws(int64_t tokens, int32_t n, int32_t hidden) {
    WgenFwdWs w{};
    const int64_t K = (int64_t)n * hidden;
    w.p = proj_fwd_ws(tokens, K, 2 * n + n * n);
    w.x_off = align256(w.p.total);
    w.total = w.x_off + align256((size_t)tokens * K * sizeof(float));
    return w;
}

// The projection folded onto r and b (wrapper_proj.hip): [packed Phi | P
// partials | sum X^2 partials | aligned copies of r and b, for rows at an
// address that is not 16-byte aligned].
struct WfoldWs {
    int ks;
    size_t p_off, ss_off, copy_off, total;
};

static WfoldWs wfold_ws(int32_t dtype, int64_t tokens, int32_t n, int32_t hidden) {
    WfoldWs w{};
    const int np = 2 * n + n * n;
    w.ks = tokens > 0 ? wfold_ksplit(dtype, tokens, hidden, np) : 1;
    w.p_off = align256(wfold_pack_bytes(dtype, n, hidden, np));
    w.ss_off = w.p_off + align256((size_t)proj_tiles(np) * w.ks * tokens * kProjTile * sizeof(float));
    w.copy_off = w.ss_off + align256((size_t)w.ks * tokens * sizeof(float));
    w.total = w.copy_off + 2 * align256((size_t)tokens * hidden * dtype_size(dtype));
    return w;
}

// What a call needs: the copies only for rows that are not 16-byte aligned.
static size_t wgen_fwd_need(int32_t dtype, int32_t n, int32_t hidden, int64_t tokens, bool aligned) {
    if (wfold_ok(n, hidden)) {
        const WfoldWs f = wfold_ws(dtype, tokens, n, hidden);
        return aligned ? f.copy_off : f.total;
    }
    return wgen_fwd_ws(tokens, n, hidden).x_off + align256((size_t)tokens * n * hidden * dtype_size(dtype));
}

// The size queries' answer.  They keep the relation that callers dividing one
// buffer between storage types count on: fp32 rows, and bf16 rows that the
// streaming projection could not rebuild (up to 32 projection rows, fewer than
// 1024 tokens, hidden % 64 != 0), reserve the stream rows in their own dtype.
static size_t wgen_fwd_size(int32_t dtype, int32_t n, int32_t hidden, int64_t tokens) {
    const size_t need = wgen_fwd_need(dtype, n, hidden, tokens, false);
    if (!wfold_ok(n, hidden) || (proj_one_pass(dtype, 2 * n + n * n, tokens) && hidden % 64 == 0)) return need;
    return need + align256((size_t)tokens * n * hidden * dtype_size(dtype));
}

// backward workspace: [per-token factors | dw partials | dw stage | ...]
//   static:  [scalar rows per wave | their sum | Sinkhorn history
//            (static_sk_hist)]
//   dynamic: [per-token scalars | dP | s | coefficient partials | dPhi
//             partials | their stage | X (fp32) | dX (fp32)]
// With dynamic H and wrap_res_grad_vanishes (the default Sinkhorn settings)
// only the 2n pre / post rows of dP are carried, as by the n = 4 kernels;
// on the shapes wgen_fold_ok takes, wgen_dphi_kernel forms their dPhi from
// r and b and wgen_dx_fold_kernel folds dP . Phi into d r / d b, so the
// stream rows never exist in memory.  Otherwise (all 2n + n^2 rows, or the
// 2n rows on other shapes) the layer's projection backward runs on the
// stream rows X and writes dX = dP . Phi, which wgen_dx_kernel folds; the
// size query has no Sinkhorn settings, so X and dX are always reserved.
//
// The dPhi / fold kernels: n <= 8, and n <= kWgFoldMaxN on rows of at least
// 2048 channels (narrower rows leave the fold's 512-channel workgroups too
// few for the per-workgroup fold of Phi over 2n rows and n streams;
// measured at n = 16, 8192 tokens: 1.29 against 1.13 ms per step at 1024
// channels, 3.58 against 4.09 at 4096).
static bool wgen_fold_ok(int32_t n, int32_t hidden) {
    return n <= 8 || (n <= kWgFoldMaxN && hidden >= 2048);
}

struct WgenBwdWs {
    int cblocks, ptiles, dtiles, qtiles, ftiles, wtiles, srows;
    size_t ep_off, dw_off, stw_off, scal_off, ssum_off, hist_off, dp_off, s_off, cpart_off, x_off, dx_off, part_off,
        stp_off, phif_off, total;
};

static WgenBwdWs wgen_bwd_ws(int64_t tokens, int32_t n, int32_t hidden, bool dynamic) {
    WgenBwdWs w{};
    const int np = 2 * n + n * n;
    const int ns = n * n + 2 * n;
    const int64_t K = (int64_t)n * hidden;
    size_t o = 0;
    w.dtiles = tokens > 0 ? wgen_dx_tiles(tokens, hidden) : 1;
    w.ftiles = tokens > 0 ? wgen_fold_tiles(tokens, hidden) : 1;
    w.wtiles = dynamic && tokens > 0 ? wbwd_tiles(n, tokens, hidden) : 1;
    int dw_rows = dynamic && w.ftiles > w.dtiles ? w.ftiles : w.dtiles;
    if (w.wtiles > dw_rows) dw_rows = w.wtiles;
    w.ep_off = o; o += align256((size_t)tokens * kWgEp * 4);
    w.dw_off = o; o += align256((size_t)dw_rows * hidden * 4);
    w.stw_off = o; o += align256(column_sums_stage_floats(hidden) * 4);
    if (!dynamic) {
        w.srows = tokens > 0 ? 4 * wgen_red_static_grid(tokens) : 1;
        w.scal_off = o; o += align256((size_t)w.srows * ns * 4);
        w.ssum_off = o; o += align256((size_t)ns * 4);
        w.hist_off = o; o += static_sk_hist(n) ? kStaticSkHistBytes : 0;
        w.total = o;
        return w;
    }
    w.cblocks = tokens > 0 ? dyn_coef_bwd_blocks(n, tokens) : 1;
    w.ptiles = tokens > 0 ? proj_bwd_tiles(kF32, tokens, K) : 1;
    w.scal_off = o; o += align256((size_t)tokens * (ns + 2) * 4);
    w.dp_off = o; o += align256((size_t)tokens * dp_stride(np) * 4);
    w.s_off = o; o += align256((size_t)tokens * 4);
    w.cpart_off = o; o += align256((size_t)w.cblocks * (np + 3) * 4);
    // dPhi partials: the 2n pre / post rows per wgen_dphi_kernel tile
    // (wgen_fold_ok), or the one-tile projection backward's (np rows when
    // np <= 32, the 2n pre / post rows when 2n <= 32 without the fold; more
    // rows go through launch_proj_bwd_small, which writes dPhi directly)
    w.qtiles = tokens > 0 ? wgen_dphi_tiles(tokens, hidden) : 1;
    size_t part = wgen_fold_ok(n, hidden) ? (size_t)w.qtiles * 2 * n : 0;
    if (np <= kProjTile && (size_t)w.ptiles * np > part) part = (size_t)w.ptiles * np;
    if (!wgen_fold_ok(n, hidden) && 2 * n <= kProjTile && (size_t)w.ptiles * 2 * n > part)
        part = (size_t)w.ptiles * 2 * n;
    // wbwd_kernel's: 2n rows of each stream that it forms
    const size_t wpart = (size_t)w.wtiles * 2 * n * (n <= 8 ? n : 2) * hidden;
    const int64_t srows = np <= kProjTile ? np : 2 * n;
    w.part_off = o; o += align256((part * K > wpart ? part * K : wpart) * 4);
    w.phif_off = o; o += align256(wbwd_fold_bytes(n, hidden));
    w.stp_off = o; o += align256(column_sums_stage_floats(srows * K) * 4);
    w.x_off = o; o += align256((size_t)tokens * K * 4);
    w.dx_off = o; o += align256((size_t)tokens * K * 4);
    w.total = o;
    return w;
}

// The run-time-n backward keeps the stream rows X and dX (the last regions
// of its workspace) only when the H_res rows of dP do not vanish or the
// shape is not one for the fold kernels.
static size_t wgen_bwd_need(const WgenBwdWs& w, int32_t n, int32_t hidden, int32_t num_iters, float sinkhorn_eps,
                            bool one) {
    return one || (wgen_fold_ok(n, hidden) && wrap_res_grad_vanishes(num_iters, sinkhorn_eps)) ? w.x_off : w.total;
}

// wbwd_kernel takes whole 16-byte pieces of aligned rows; bf16 'decay' past
// n = 8, C % 8 != 0 and unaligned rows keep the kernels of wrapper_gen.hip.  dPhi,
// d r and d b at n = 8 (65,536 x 7168 bf16): 1.30 ms against 3.2; fp32 n = 16 (4096
// x 2048): 50 us against 905
static bool wgen_bwd_one(int32_t dtype, int32_t n, bool decay, int32_t hidden, int64_t tokens, int32_t num_iters,
                         float sinkhorn_eps, std::initializer_list<const void*> rows) {
    uintptr_t a = 0;
    for (const void* p : rows) a |= (uintptr_t)p;
    return tokens > 0 && wrap_res_grad_vanishes(num_iters, sinkhorn_eps) && a % 16 == 0 &&
           wbwd_shape_ok(dtype, n, decay, hidden);
}

static int wgen_dynamic_fwd(const void* residual, const void* branch, int32_t dtype, bool decay, const void* weight,
                            int32_t weight_dtype, const float* phi_pre, const float* phi_post, const float* phi_res,
                            const float* alpha_pre, const float* alpha_post, const float* alpha_res,
                            const float* b_pre, const float* b_post, const float* b_res, float* out, float* saved,
                            void* workspace, size_t workspace_bytes, int64_t tokens, int32_t n, int32_t hidden,
                            int32_t num_iters, float sinkhorn_eps, float rmsnorm_eps, hipStream_t s) {
    const DynSaved d = dyn_saved(tokens, n, hidden);
    float* w32 = saved + d.w_off;
    const bool wfold = tokens > 0 && wfold_ok(n, hidden);
    // the weight's fp32 copy: its own launch, or inside the folded pack's
    hipError_t e = wfold ? hipSuccess : launch_weight_f32(weight, weight_dtype, hidden, w32, s);
    if (e != hipSuccess || tokens == 0) return hip_status(e);
    const bool rows16 = ((uintptr_t)residual | (uintptr_t)branch) % 16 == 0;
    if (!workspace || workspace_bytes < wgen_fwd_need(dtype, n, hidden, tokens, rows16))
        return fail(MHC_ERR_WORKSPACE,
                    "wrapper_dynamic_fwd: workspace smaller than mhc_wrapper_dynamic_fwd_workspace_size_for()");
    const int64_t K = (int64_t)n * hidden;
    const int np = 2 * n + n * n;
    char* pw = (char*)workspace;
    float *pp = nullptr, *ss = nullptr;
    int ks = 1;
    if (wfold) {
        const WfoldWs f = wfold_ws(dtype, tokens, n, hidden);
        const void *pres = residual, *pbr = branch;
        if (!rows16) {
            char* c = pw + f.copy_off;
            char* c2 = c + align256((size_t)tokens * hidden * dtype_size(dtype));
            e = launch_wfold_copy(dtype, residual, c, branch, c2, tokens * hidden, s);
            pres = c;
            pbr = c2;
        }
        ks = f.ks;
        pp = (float*)(pw + f.p_off);
        ss = (float*)(pw + f.ss_off);
        if (e == hipSuccess)
            e = launch_wfold_proj(dtype, n, decay, pres, pbr, phi_pre, phi_post, phi_res, weight, weight_dtype, w32, pw,
                                  pp, ss, tokens, hidden, ks, s);
    } else {
        const WgenFwdWs w = wgen_fwd_ws(tokens, n, hidden);
        void* X = pw + w.x_off;
        bf16_raw_t* phib = (bf16_raw_t*)(pw + w.p.phib_off);
        pp = (float*)(pw + w.p.p_off);
        ss = (float*)(pw + w.p.ss_off);
        ks = w.p.ks;
        e = launch_wgen_synth(dtype, dtype, n, decay, residual, branch, X, tokens, hidden, s);
        if (e == hipSuccess && w.p.stream) {
            e = launch_proj_stream(dtype, X, (bf16_raw_t*)(pw + w.p.xpl_off), phi_pre, phi_post, phi_res, n, nullptr,
                                   np, pp, ss, tokens, K, w.p.ks, s);
        } else if (e == hipSuccess) {
            e = launch_phi_split(phi_pre, phi_post, phi_res, n, np, K, phib, s);
            if (e == hipSuccess && proj_one_pass(dtype, np, tokens))
                e = launch_proj_stream(dtype, X, nullptr, phi_pre, phi_post, phi_res, n, phib, np, pp, ss, tokens, K,
                                       w.p.ks, s);
            else if (e == hipSuccess)
                e = launch_proj_mfma(dtype, X, phib, np, pp, ss, tokens, K, w.p.ks, s);
        }
    }
    if (e == hipSuccess)
        e = launch_dyn_coef_fwd(n, pp, ss, ks, tokens, K, alpha_pre, alpha_post, alpha_res, b_pre, b_post, b_res,
                                saved + d.coef_off, saved + d.p_off, saved + d.rh_off, num_iters, sinkhorn_eps,
                                rmsnorm_eps, s);
    if (e == hipSuccess)
        e = launch_wrow_fwd(dtype, n, decay, residual, branch, w32, saved + d.coef_off, np, out, tokens, hidden,
                            rmsnorm_eps, s);
    return hip_status(e);
}

static int wgen_dynamic_bwd(const float* grad_out, const void* residual, const void* branch, int32_t dtype,
                            bool decay, int32_t weight_dtype, const float* phi_pre, const float* phi_post,
                            const float* phi_res, const float* alpha_pre, const float* alpha_post,
                            const float* alpha_res, const float* b_res, const float* saved, void* grad_residual,
                            void* grad_branch, void* grad_weight, float* grad_phi, float* grad_alpha, float* grad_b,
                            void* workspace, size_t workspace_bytes, int64_t tokens, int32_t n, int32_t hidden,
                            int32_t num_iters, float sinkhorn_eps, float rmsnorm_eps, hipStream_t s) {
    const int np = 2 * n + n * n;
    // rows of dP the projection backward carries (the rest of dPhi: zeros)
    const int rows = wrap_res_grad_vanishes(num_iters, sinkhorn_eps) ? 2 * n : np;
    if (rows > kProjTile && rows > proj_bwd_small_max_rows())
        return fail(MHC_ERR_UNSUPPORTED, "wrapper_dynamic_bwd: at n = " + std::to_string(n) +
                                             " the fused wrapper needs num_iters >= 1 and sinkhorn_eps <= 1e-6 "
                                             "(the H_res gradients then vanish)");
    const WgenBwdWs w = wgen_bwd_ws(tokens, n, hidden, true);
    const bool one = wgen_bwd_one(dtype, n, decay, hidden, tokens, num_iters, sinkhorn_eps,
                                  {grad_out, residual, branch, grad_residual, grad_branch});
    if (!workspace || workspace_bytes < wgen_bwd_need(w, n, hidden, num_iters, sinkhorn_eps, one))
        return fail(MHC_ERR_WORKSPACE,
                    "wrapper_dynamic_bwd: workspace smaller than mhc_wrapper_dynamic_bwd_workspace_size_for()");
    char* ws = (char*)workspace;
    float* ep = (float*)(ws + w.ep_off);
    float* dw_part = (float*)(ws + w.dw_off);
    float* stw = (float*)(ws + w.stw_off);
    float* scal = (float*)(ws + w.scal_off);
    float* dp = (float*)(ws + w.dp_off);
    float* stok = (float*)(ws + w.s_off);
    float* cpart = (float*)(ws + w.cpart_off);
    float* X = (float*)(ws + w.x_off);
    float* dX = (float*)(ws + w.dx_off);
    float* part = (float*)(ws + w.part_off);
    float* stp = (float*)(ws + w.stp_off);
    const DynSaved d = dyn_saved(tokens, n, hidden);
    const float* w32 = saved + d.w_off;
    const int64_t K = (int64_t)n * hidden;
    // the fold kernels' shapes carry the pre / post rows without stream rows
    const bool fold = rows < np && wgen_fold_ok(n, hidden);
    hipError_t e = hipSuccess;
    int rows_w = fold ? w.ftiles : w.dtiles, rows_c = dyn_coef_bwd_rows(n, tokens, num_iters, rows == np);
    if (tokens == 0) {
        rows_w = rows_c = 1;
        e = launch_fill_zero(dw_part, hidden, s);
        if (e == hipSuccess) e = launch_fill_zero(cpart, np + 3, s);
        if (e == hipSuccess) e = launch_fill_zero(grad_phi, (int64_t)rows * K, s);
    } else {
        if (rows < np && wrow_red_ok(dtype, n, decay, hidden))
            e = launch_wrow_red(dtype, n, decay, grad_out, residual, branch, w32, saved + d.coef_off, np, scal, ep,
                                tokens, hidden, rmsnorm_eps, s);
        else
            e = launch_wgen_red(dtype, n, decay, false, grad_out, residual, branch, w32, saved + d.coef_off, np, scal,
                                ep, tokens, hidden, rmsnorm_eps, s);
        // with the H_res rows vanishing no Sinkhorn adjoint runs (their dP,
        // db and dalpha are zeros, overwritten with the NaN carry below)
        if (e == hipSuccess)
            e = launch_dyn_coef_bwd(n, scal, saved + d.coef_off, saved + d.p_off, saved + d.rh_off, tokens, K,
                                    alpha_pre, alpha_post, alpha_res, b_res, dp, stok, cpart, num_iters, sinkhorn_eps,
                                    nullptr, s, rows == np);
        if (one) {
            if (e == hipSuccess)
                e = launch_wbwd(dtype, n, decay, grad_out, residual, branch, w32, ep, dp, dp_stride(np), stok, phi_pre,
                                phi_post, (float*)(ws + w.phif_off), grad_residual, grad_branch, dw_part, part,
                                w.wtiles, tokens, hidden, s);
            const int nst = wbwd_streams(dtype, n, decay);
            const bool few = rows_c <= kWrapSumsMaxRows;
            if (e == hipSuccess)
                e = launch_wrap_sums(WrapSums{part, (int64_t)nst * rows * hidden, (int64_t)rows * hidden, hidden,
                                              w.wtiles, nst, rows, n, np, hidden, decay, grad_phi, dw_part, w.wtiles,
                                              weight_dtype == kBF16, grad_weight, few ? cpart : nullptr,
                                              few ? rows_c : 0, grad_b, grad_alpha, 0},
                                     s);
            if (few || e != hipSuccess) return hip_status(e);
        }
        if (!one && fold) {
            if (e == hipSuccess)
                e = launch_wgen_dphi(dtype, n, decay, residual, branch, dp, dp_stride(np), rows, part, w.qtiles, tokens,
                                     hidden, s);
            if (e == hipSuccess)
                e = launch_column_finalize(0, kF32, part, w.qtiles, (int64_t)rows * K, stp, grad_phi, nullptr, 0,
                                           nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0.f, s);
            if (e == hipSuccess)
                e = launch_wgen_dx_fold(dtype, n, decay, grad_out, residual, branch, w32, saved + d.coef_off, np, ep,
                                        dp, dp_stride(np), rows, stok, phi_pre, phi_post, grad_residual,
                                        grad_branch, dw_part, w.ftiles, tokens, hidden, s);
        }
        const bool full = !one && !fold;
        if (full && e == hipSuccess) e = launch_wgen_synth(dtype, kF32, n, decay, residual, branch, X, tokens, hidden, s);
        if (full && e == hipSuccess) {
            if (rows > kProjTile) {  // X and dX once for all output tiles
                e = launch_proj_bwd_small(X, dp, dp_stride(np), nullptr, phi_pre, phi_post, phi_res, n, rows, dX,
                                          false, grad_phi, tokens, K, s);
            } else {
                e = launch_proj_bwd(kF32, X, dp, dp_stride(np), nullptr, phi_pre, phi_post, phi_res, n, 0, rows, dX,
                                    false, part, w.ptiles, tokens, K, s);
                if (e == hipSuccess)
                    e = launch_column_finalize(0, kF32, part, w.ptiles, (int64_t)rows * K, stp, grad_phi, nullptr, 0,
                                               nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0.f, s);
            }
        }
        if (full && e == hipSuccess)
            e = launch_wgen_dx(dtype, n, decay, grad_out, residual, branch, w32, saved + d.coef_off, np, ep, dX, stok,
                               grad_residual, grad_branch, dw_part, w.dtiles, tokens, hidden, s);
    }
    if (!one && e == hipSuccess)
        e = launch_column_finalize(0, weight_dtype, dw_part, rows_w, hidden, stw, grad_weight, nullptr, 0, nullptr,
                                   nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0.f, s);
    if (e == hipSuccess) e = launch_small_column_sum(cpart, rows_c, np + 3, grad_b, grad_alpha, np, s);
    // the H_res rows of dPhi, db and dalpha: zeros, NaN where the alpha
    // gradients (sums over the same tokens) are not finite, as the n = 4
    // path writes them
    if (e == hipSuccess && rows < np)
        e = launch_fill_zero_carry(grad_phi + (int64_t)rows * K, (int64_t)(np - rows) * K, grad_b + rows, np - rows,
                                   grad_alpha, 3, s);
    if (e == hipSuccess && rows < np) e = launch_fill_zero_carry(grad_alpha + 2, 1, nullptr, 0, grad_alpha, 2, s);
    return hip_status(e);
}

static int wgen_static_bwd(const float* grad_out, const void* residual, const void* branch, int32_t dtype, bool decay,
                           int32_t weight_dtype, const float* h_pre, const float* h_post, const float* h_res,
                           const float* saved, void* grad_residual, void* grad_branch, void* grad_weight,
                           float* grad_h_pre, float* grad_h_post, float* grad_h_res, void* workspace,
                           size_t workspace_bytes, int64_t tokens, int32_t n, int32_t hidden, int32_t num_iters,
                           float sinkhorn_eps, float rmsnorm_eps, hipStream_t s) {
    const WgenBwdWs w = wgen_bwd_ws(tokens, n, hidden, false);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE, "wrapper_static_bwd: workspace smaller than mhc_wrapper_static_bwd_workspace_size()");
    char* ws = (char*)workspace;
    float* ep = (float*)(ws + w.ep_off);
    float* dw_part = (float*)(ws + w.dw_off);
    float* stw = (float*)(ws + w.stw_off);
    float* scal = (float*)(ws + w.scal_off);
    float* ssum = (float*)(ws + w.ssum_off);
    const int ns = n * n + 2 * n;
    const float* w32 = saved + saved_w_offset(n);
    hipError_t e = hipSuccess;
    int rows = w.dtiles;
    if (tokens == 0) {
        rows = 1;
        e = launch_fill_zero(dw_part, hidden, s);
        if (e == hipSuccess) e = launch_fill_zero(ssum, ns, s);
    } else {
        e = launch_wgen_red(dtype, n, decay, true, grad_out, residual, branch, w32, saved, 0, scal, ep, tokens, hidden,
                            rmsnorm_eps, s);
        if (e == hipSuccess) e = launch_small_column_sum(scal, w.srows, ns, ssum, ssum, ns, s);
        if (e == hipSuccess)
            e = launch_wgen_dx(dtype, n, decay, grad_out, residual, branch, w32, saved, 0, ep, nullptr, nullptr,
                               grad_residual, grad_branch, dw_part, w.dtiles, tokens, hidden, s);
    }
    if (e == hipSuccess)
        e = launch_column_finalize(n, weight_dtype, dw_part, rows, hidden, stw, grad_weight, ssum, 1, h_pre, h_post,
                                   h_res, grad_h_pre, grad_h_post, grad_h_res, num_iters, sinkhorn_eps, s,
                                   static_sk_hist(n) ? (float*)(ws + w.hist_off) : nullptr);
    // dH_res vanishes as in mhc_wrapper_static_bwd's n = 4 path
    if (e == hipSuccess && wrap_res_grad_vanishes(num_iters, sinkhorn_eps))
        e = launch_fill_zero_carry(grad_h_res, (int64_t)n * n, nullptr, 0, grad_h_pre, n, s);
    return hip_status(e);
}

struct WrapFwdWs {
    int ks;
    size_t phib_off, p_off, ss_off, total;
};

static WrapFwdWs wrap_fwd_ws(int64_t tokens, int32_t n, int32_t hidden) {
    WrapFwdWs w{};
    const int64_t K = (int64_t)n * hidden;
    w.ks = tokens > 0 ? wrap_proj_csplit(tokens, hidden) : 1;
    w.phib_off = 0;
    w.p_off = align256((size_t)3 * 32 * K * 2);
    w.ss_off = w.p_off + align256((size_t)w.ks * tokens * 32 * sizeof(float));
    w.total = w.ss_off + align256((size_t)w.ks * tokens * sizeof(float));
    return w;
}

size_t mhc_wrapper_dynamic_fwd_workspace_size(int64_t tokens, int32_t n, int32_t hidden) {
    if (tokens < 0 || n < 1 || hidden < 1) return 0;
    if (!wrap_fused4(n, hidden, true)) {
        const size_t a = wgen_fwd_size(kF32, n, hidden, tokens), b = wgen_fwd_size(kBF16, n, hidden, tokens);
        return a > b ? a : b;
    }
    return wrap_fwd_ws(tokens, n, hidden).total;
}

size_t mhc_wrapper_dynamic_fwd_workspace_size_for(int64_t tokens, int32_t n, int32_t hidden, int32_t dtype) {
    if (tokens < 0 || n < 1 || hidden < 1 || !valid_dtype(dtype)) return 0;
    if (!wrap_fused4(n, hidden, true))
        return wgen_fwd_size(dtype, n, hidden, tokens);
    return wrap_fwd_ws(tokens, n, hidden).total;
}

size_t mhc_wrapper_dynamic_fwd_workspace_need(const void* residual, const void* branch, int32_t dtype, int64_t tokens,
                                              int32_t n, int32_t hidden) {
    if (tokens < 0 || n < 1 || hidden < 1 || !valid_dtype(dtype)) return 0;
    if (!wrap_fused4(n, hidden, true))
        return wgen_fwd_need(dtype, n, hidden, tokens, ((uintptr_t)residual | (uintptr_t)branch) % 16 == 0);
    return wrap_fwd_ws(tokens, n, hidden).total;
}

int mhc_wrapper_dynamic_fwd(const void* residual, const void* branch, int32_t dtype, int32_t residual_mode,
                            const void* weight, int32_t weight_dtype, const float* phi_pre, const float* phi_post,
                            const float* phi_res, const float* alpha_pre, const float* alpha_post,
                            const float* alpha_res, const float* b_pre, const float* b_post, const float* b_res,
                            float* out, float* saved, void* workspace, size_t workspace_bytes, int64_t tokens,
                            int32_t n, int32_t hidden, int32_t num_iters, float sinkhorn_eps, float rmsnorm_eps,
                            void* stream) {
    int st = check_wrapper("wrapper_dynamic_fwd", tokens, n, hidden, dtype, weight_dtype, residual_mode, num_iters,
                           true);
    if (st) return st;
    MHC_REQUIRE(weight && phi_pre && phi_post && phi_res && alpha_pre && alpha_post && alpha_res && b_pre &&
                    b_post && b_res && saved,
                "wrapper_dynamic_fwd: null parameter pointer");
    MHC_REQUIRE(tokens == 0 || (residual && branch && out), "wrapper_dynamic_fwd: null residual/branch/out");
    hipStream_t s = (hipStream_t)stream;
    if (!wrap_fused4(n, hidden, true))
        return wgen_dynamic_fwd(residual, branch, dtype, residual_mode == MHC_WRAPPER_DECAY, weight, weight_dtype,
                                phi_pre, phi_post, phi_res, alpha_pre, alpha_post, alpha_res, b_pre, b_post, b_res,
                                out, saved, workspace, workspace_bytes, tokens, n, hidden, num_iters, sinkhorn_eps,
                                rmsnorm_eps, s);
    const DynSaved d = dyn_saved(tokens, n, hidden);
    float* w32 = saved + d.w_off;
    hipError_t e = launch_weight_f32(weight, weight_dtype, hidden, w32, s);
    if (e != hipSuccess || tokens == 0) return hip_status(e);
    const WrapFwdWs w = wrap_fwd_ws(tokens, n, hidden);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE, "wrapper_dynamic_fwd: workspace smaller than mhc_wrapper_dynamic_fwd_workspace_size()");
    const bool decay = residual_mode == MHC_WRAPPER_DECAY;
    const int64_t K = (int64_t)n * hidden;
    const int np = 2 * n + n * n;
    bf16_raw_t* phib = (bf16_raw_t*)((char*)workspace + w.phib_off);
    float* pp = (float*)((char*)workspace + w.p_off);
    float* ss = (float*)((char*)workspace + w.ss_off);
    e = launch_wrap_phi_planes(dtype, n, phi_pre, phi_post, phi_res, hidden, phib, s);
    if (e == hipSuccess) e = launch_wrap_proj(dtype, n, decay, residual, branch, phib, pp, ss, tokens, hidden, w.ks, s);
    if (e == hipSuccess)
        e = launch_dyn_coef_fwd(n, pp, ss, w.ks, tokens, K, alpha_pre, alpha_post, alpha_res, b_pre, b_post, b_res,
                                saved + d.coef_off, saved + d.p_off, saved + d.rh_off, num_iters, sinkhorn_eps,
                                rmsnorm_eps, s);
    if (e == hipSuccess)
        e = launch_wrow_fwd(dtype, n, decay, residual, branch, w32, saved + d.coef_off, np, out, tokens, hidden,
                            rmsnorm_eps, s);
    return hip_status(e);
}

struct WrapBwdWs {
    int grid, cblocks, tiles;
    size_t dw_off, scal_off, dp_off, s_off, ep_off, cpart_off, phip_off, stw_off, stp_off, total;
};

// static: [dw partials (grid rows) | stage | per-workgroup scalars];
// dynamic: [dw partials (tiles rows) | stage | per-token scalars | dP | s |
// stream-part factors | coefficient partials | dPhi partials | stage]
static WrapBwdWs wrap_bwd_ws(int64_t tokens, int32_t n, int32_t hidden, int32_t dtype, bool dynamic, bool decay) {
    WrapBwdWs w{};
    const int64_t np = 2 * n + n * n;
    const int64_t K = (int64_t)n * hidden;
    size_t o = 0;
    if (!dynamic) {
        w.grid = tokens > 0 ? wrap_bwd_grid(dtype, n, decay, tokens, hidden) : 1;
        w.dw_off = o; o += align256((size_t)w.grid * hidden * 4);
        w.stw_off = o; o += align256(column_sums_stage_floats(hidden) * 4);
        w.scal_off = o; o += align256((size_t)w.grid * (n * n + 2 * n) * 4);
        w.total = o;
        return w;
    }
    w.cblocks = tokens > 0 ? dyn_coef_bwd_blocks(n, tokens) : 1;
    w.tiles = tokens > 0 ? wrap_proj_bwd_tiles(dtype, tokens, hidden) : 1;
    w.dw_off = o; o += align256((size_t)w.tiles * hidden * 4);
    w.stw_off = o; o += align256(column_sums_stage_floats(hidden) * 4);
    w.scal_off = o; o += align256((size_t)tokens * (n * n + 2 * n + 2) * 4);
    w.dp_off = o; o += align256((size_t)tokens * 32 * 4);
    w.s_off = o; o += align256((size_t)tokens * 4);
    w.ep_off = o; o += align256((size_t)tokens * kWrapEp * 4);
    w.cpart_off = o; o += align256((size_t)w.cblocks * (np + 3) * 4);
    w.phip_off = o; o += align256((size_t)w.tiles * np * K * 4);
    w.stp_off = o; o += align256(column_sums_stage_floats((int64_t)np * K) * 4);
    w.total = o;
    return w;
}

// Whether the wrapper's H_res gradients vanish.  The wrapper's output is the
// mean of the n layer outputs (layer.py:316), so every stream receives the
// same cotangent G / n and dM_ij = (1/n) sum_c G x_j is constant down each
// column j.  The Sinkhorn pass ends with a column normalisation
// (A_ij / (colsum_j + eps)), whose adjoint maps a column-constant cotangent
// v_j to v_j eps / (colsum_j + eps)^2: zero up to eps, and the earlier
// iterations' adjoints shrink it further.  Measured on a float64
// restatement (n = 4, 37 tokens): the largest H_res gradient against the
// largest of its family (dPhi_pre, dH_pre) is 2e-24 / 1e-19 at 20
// iterations and eps = 1e-8, 2e-9 / 2e-8 at one iteration, 2e-7 / 2e-6 at
// one iteration and eps = 1e-6.  With no iterations M = exp(t) and nothing
// cancels; with a large eps the leftover is not negligible (0.015 / 0.18 at
// one iteration and eps = 0.1).  So for num_iters >= 1 and eps <= 1e-6 the H_res rows
// of dP, dPhi_res, dalpha_res and db_res (and the static dH_res) are written
// as exact zeros and their arithmetic is skipped; otherwise the full adjoint
// runs.
static bool wrap_res_grad_vanishes(int32_t num_iters, float sinkhorn_eps) {
    return num_iters >= 1 && sinkhorn_eps >= 0.f && sinkhorn_eps <= 1e-6f;
}

size_t mhc_wrapper_dynamic_bwd_workspace_size(int64_t tokens, int32_t n, int32_t hidden, int32_t dtype,
                                              int32_t residual_mode) {
    if (tokens < 0 || n < 1 || hidden < 1) return 0;
    if (!wrap_fused4(n, hidden, true)) return wgen_bwd_ws(tokens, n, hidden, true).total;
    return wrap_bwd_ws(tokens, n, hidden, dtype, true, residual_mode == MHC_WRAPPER_DECAY).total;
}

size_t mhc_wrapper_dynamic_bwd_workspace_size_for(int64_t tokens, int32_t n, int32_t hidden, int32_t dtype,
                                                  int32_t residual_mode, int32_t num_iters, float sinkhorn_eps) {
    if (tokens < 0 || n < 1 || hidden < 1) return 0;
    if (!wrap_fused4(n, hidden, true))
        return wgen_bwd_need(wgen_bwd_ws(tokens, n, hidden, true), n, hidden, num_iters, sinkhorn_eps, false);
    return wrap_bwd_ws(tokens, n, hidden, dtype, true, residual_mode == MHC_WRAPPER_DECAY).total;
}

size_t mhc_wrapper_dynamic_bwd_workspace_need(const float* grad_out, const void* residual, const void* branch,
                                              const void* grad_residual, const void* grad_branch, int32_t dtype,
                                              int32_t residual_mode, int64_t tokens, int32_t n, int32_t hidden,
                                              int32_t num_iters, float sinkhorn_eps) {
    if (tokens < 0 || n < 1 || hidden < 1) return 0;
    if (!wrap_fused4(n, hidden, true))
        return wgen_bwd_need(wgen_bwd_ws(tokens, n, hidden, true), n, hidden, num_iters, sinkhorn_eps,
                             wgen_bwd_one(dtype, n, residual_mode == MHC_WRAPPER_DECAY, hidden, tokens, num_iters,
                                          sinkhorn_eps, {grad_out, residual, branch, grad_residual, grad_branch}));
    return wrap_bwd_ws(tokens, n, hidden, dtype, true, residual_mode == MHC_WRAPPER_DECAY).total;
}

int mhc_wrapper_dynamic_bwd(const float* grad_out, const void* residual, const void* branch, int32_t dtype,
                            int32_t residual_mode, int32_t weight_dtype, const float* phi_pre, const float* phi_post,
                            const float* phi_res, const float* alpha_pre, const float* alpha_post,
                            const float* alpha_res, const float* b_res, const float* saved, void* grad_residual,
                            void* grad_branch, void* grad_weight, float* grad_phi, float* grad_alpha, float* grad_b,
                            void* workspace, size_t workspace_bytes, int64_t tokens, int32_t n, int32_t hidden,
                            int32_t num_iters, float sinkhorn_eps, float rmsnorm_eps, void* stream) {
    int st = check_wrapper("wrapper_dynamic_bwd", tokens, n, hidden, dtype, weight_dtype, residual_mode, num_iters,
                           true);
    if (st) return st;
    MHC_REQUIRE(phi_pre && phi_post && phi_res && alpha_pre && alpha_post && alpha_res && b_res && saved,
                "wrapper_dynamic_bwd: null parameter pointer");
    MHC_REQUIRE(grad_weight && grad_phi && grad_alpha && grad_b, "wrapper_dynamic_bwd: null gradient pointer");
    MHC_REQUIRE(tokens == 0 || (grad_out && residual && branch && grad_residual && grad_branch),
                "wrapper_dynamic_bwd: null grad_out/residual/branch/grad pointer");
    const bool decay = residual_mode == MHC_WRAPPER_DECAY;
    hipStream_t s = (hipStream_t)stream;
    if (!wrap_fused4(n, hidden, true))
        return wgen_dynamic_bwd(grad_out, residual, branch, dtype, decay, weight_dtype, phi_pre, phi_post, phi_res,
                                alpha_pre, alpha_post, alpha_res, b_res, saved, grad_residual, grad_branch, grad_weight,
                                grad_phi, grad_alpha, grad_b, workspace, workspace_bytes, tokens, n, hidden, num_iters,
                                sinkhorn_eps, rmsnorm_eps, s);
    const WrapBwdWs w = wrap_bwd_ws(tokens, n, hidden, dtype, true, decay);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE, "wrapper_dynamic_bwd: workspace smaller than mhc_wrapper_dynamic_bwd_workspace_size()");
    char* ws = (char*)workspace;
    float* dw_part = (float*)(ws + w.dw_off);
    float* scal = (float*)(ws + w.scal_off);
    float* dp = (float*)(ws + w.dp_off);
    float* stok = (float*)(ws + w.s_off);
    float* cpart = (float*)(ws + w.cpart_off);
    float* phip = (float*)(ws + w.phip_off);
    float* stw = (float*)(ws + w.stw_off);
    float* stp = (float*)(ws + w.stp_off);
    float* ep = (float*)(ws + w.ep_off);
    const DynSaved d = dyn_saved(tokens, n, hidden);
    const int np = 2 * n + n * n;
    const int64_t K = (int64_t)n * hidden;
    const float* w32 = saved + d.w_off;
    // rows of dPhi formed by the projection backward (the rest are zeros)
    const bool res_rows = !wrap_res_grad_vanishes(num_iters, sinkhorn_eps);
    const int npo = res_rows ? np : 2 * n;
    hipError_t e = hipSuccess;
    int rows_p = w.tiles, rows_c = dyn_coef_bwd_rows(n, tokens, num_iters, res_rows);
    if (tokens == 0) {
        rows_p = rows_c = 1;
        e = launch_fill_zero(dw_part, hidden, s);
        if (e == hipSuccess) e = launch_fill_zero(phip, (int64_t)npo * K, s);
        if (e == hipSuccess) e = launch_fill_zero(cpart, np + 3, s);
    } else {
        e = launch_wrap_bwd_red(dtype, n, decay, grad_out, residual, branch, w32, saved + d.coef_off, np, scal, ep,
                                tokens, hidden, rmsnorm_eps, s);
        if (e == hipSuccess)
            e = launch_dyn_coef_bwd(n, scal, saved + d.coef_off, saved + d.p_off, saved + d.rh_off, tokens, K,
                                    alpha_pre, alpha_post, alpha_res, b_res, dp, stok, cpart, num_iters, sinkhorn_eps,
                                    nullptr, s, res_rows);
        if (e == hipSuccess)
            e = launch_wrap_proj_bwd(dtype, n, decay, grad_out, residual, branch, w32, ep, dp, stok, phi_pre,
                                     phi_post, phi_res, grad_residual, grad_branch, dw_part, phip, w.tiles, tokens,
                                     hidden, res_rows, s);
        // one launch instead of four: the sums of small calls were 15 us of gaps
        if (!res_rows && rows_c <= kWrapSumsMaxRows) {
            if (e == hipSuccess)
                e = launch_wrap_sums(WrapSums{phip, (int64_t)npo * K, hidden, K, w.tiles, n, npo, n, np, hidden, decay,
                                              grad_phi, dw_part, w.tiles, weight_dtype == kBF16, grad_weight, cpart,
                                              rows_c, grad_b, grad_alpha, 0},
                                     s);
            return hip_status(e);
        }
    }
    if (e == hipSuccess)
        e = launch_column_finalize(0, weight_dtype, dw_part, rows_p, hidden, stw, grad_weight, nullptr, 0, nullptr,
                                   nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0.f, s);
    if (e == hipSuccess)
        e = launch_column_finalize(0, kF32, phip, rows_p, (int64_t)npo * K, stp, grad_phi, nullptr, 0, nullptr,
                                  nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0.f, s);
    if (e == hipSuccess) e = launch_small_column_sum(cpart, rows_c, np + 3, grad_b, grad_alpha, np, s);
    // the H_res rows: zeros, NaN where the alpha gradients (sums over the
    // same tokens) are not finite, as the reference's would be then
    if (e == hipSuccess && npo < np)
        e = launch_fill_zero_carry(grad_phi + (int64_t)npo * K, (int64_t)(np - npo) * K, grad_b + npo, np - npo,
                                   grad_alpha, 3, s);
    return hip_status(e);
}

int mhc_wrapper_static_fwd(const void* residual, const void* branch, int32_t dtype, int32_t residual_mode,
                           const void* weight, int32_t weight_dtype, const float* h_pre, const float* h_post,
                           const float* h_res, float* out, float* saved, int64_t tokens, int32_t n, int32_t hidden,
                           int32_t num_iters, float sinkhorn_eps, float rmsnorm_eps, void* stream) {
    int st = check_wrapper("wrapper_static_fwd", tokens, n, hidden, dtype, weight_dtype, residual_mode, num_iters,
                           false);
    if (st) return st;
    MHC_REQUIRE(weight && h_pre && h_post && h_res && saved, "wrapper_static_fwd: null parameter pointer");
    MHC_REQUIRE(tokens == 0 || (residual && branch && out), "wrapper_static_fwd: null residual/branch/out");
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = launch_static_coef(n, h_pre, h_post, h_res, weight, weight_dtype, hidden, saved, num_iters,
                                      sinkhorn_eps, s);
    if (e != hipSuccess) return hip_status(e);
    return hip_status(launch_wrow_fwd(dtype, n, residual_mode == MHC_WRAPPER_DECAY, residual, branch,
                                      saved + saved_w_offset(n), saved, 0, out, tokens, hidden, rmsnorm_eps, s));
}

size_t mhc_wrapper_static_bwd_workspace_size(int64_t tokens, int32_t n, int32_t hidden, int32_t dtype,
                                             int32_t residual_mode) {
    if (tokens < 0 || n < 1 || hidden < 1) return 0;
    if (!wrap_fused4(n, hidden, false)) return wgen_bwd_ws(tokens, n, hidden, false).total;
    return wrap_bwd_ws(tokens, n, hidden, dtype, false, residual_mode == MHC_WRAPPER_DECAY).total;
}

int mhc_wrapper_static_bwd(const float* grad_out, const void* residual, const void* branch, int32_t dtype,
                           int32_t residual_mode, int32_t weight_dtype, const float* h_pre, const float* h_post,
                           const float* h_res, const float* saved, void* grad_residual, void* grad_branch,
                           void* grad_weight, float* grad_h_pre, float* grad_h_post, float* grad_h_res,
                           void* workspace, size_t workspace_bytes, int64_t tokens, int32_t n, int32_t hidden,
                           int32_t num_iters, float sinkhorn_eps, float rmsnorm_eps, void* stream) {
    int st = check_wrapper("wrapper_static_bwd", tokens, n, hidden, dtype, weight_dtype, residual_mode, num_iters,
                           false);
    if (st) return st;
    MHC_REQUIRE(h_pre && h_post && h_res && saved, "wrapper_static_bwd: null parameter pointer");
    MHC_REQUIRE(grad_weight && grad_h_pre && grad_h_post && grad_h_res, "wrapper_static_bwd: null gradient pointer");
    MHC_REQUIRE(tokens == 0 || (grad_out && residual && branch && grad_residual && grad_branch),
                "wrapper_static_bwd: null grad_out/residual/branch/grad pointer");
    const bool decay = residual_mode == MHC_WRAPPER_DECAY;
    hipStream_t s = (hipStream_t)stream;
    if (!wrap_fused4(n, hidden, false))
        return wgen_static_bwd(grad_out, residual, branch, dtype, decay, weight_dtype, h_pre, h_post, h_res, saved,
                               grad_residual, grad_branch, grad_weight, grad_h_pre, grad_h_post, grad_h_res, workspace,
                               workspace_bytes, tokens, n, hidden, num_iters, sinkhorn_eps, rmsnorm_eps, s);
    const WrapBwdWs w = wrap_bwd_ws(tokens, n, hidden, dtype, false, decay);
    if (!workspace || workspace_bytes < w.total)
        return fail(MHC_ERR_WORKSPACE, "wrapper_static_bwd: workspace smaller than mhc_wrapper_static_bwd_workspace_size()");
    float* dw_part = (float*)((char*)workspace + w.dw_off);
    float* scal_part = (float*)((char*)workspace + w.scal_off);
    float* stage = (float*)((char*)workspace + w.stw_off);
    hipError_t e = hipSuccess;
    int rows = w.grid;
    if (tokens == 0) {
        rows = 1;
        e = launch_fill_zero(dw_part, hidden, s);
        if (e == hipSuccess) e = launch_fill_zero(scal_part, n * n + 2 * n, s);
    } else {
        e = launch_wrap_bwd(dtype, n, decay, grad_out, residual, branch, saved + saved_w_offset(n), saved, 0,
                            grad_residual, grad_branch, dw_part, scal_part, w.grid, tokens, hidden, rmsnorm_eps, s);
    }
    if (e == hipSuccess)
        e = launch_column_finalize(n, weight_dtype, dw_part, rows, hidden, stage, grad_weight, scal_part, rows, h_pre,
                                  h_post, h_res, grad_h_pre, grad_h_post, grad_h_res, num_iters, sinkhorn_eps, s);
    // dH_res of the wrapper is zero up to eps (wrap_res_grad_vanishes); NaN
    // where dH_pre (a sum over the same tokens) is not finite
    if (e == hipSuccess && wrap_res_grad_vanishes(num_iters, sinkhorn_eps))
        e = launch_fill_zero_carry(grad_h_res, (int64_t)n * n, nullptr, 0, grad_h_pre, n, s);
    return hip_status(e);
}

}  // extern "C"
