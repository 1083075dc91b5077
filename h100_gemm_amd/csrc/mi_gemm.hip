// mi_gemm.hip -- C ABI of libmi_gemm.so (declared in include/mi_gemm.h): the kernel
// configuration table, shape -> kernel dispatch, and the thin HIP layer the harness uses.
//
// The launch path stands where the reference's host launchers stand: runKernel
// (matmul_h100_optimal.cu:32-59) and gpu_gemm (matmul_h100.cu.jinja:927-985).  Those build
// TMA descriptors, set a shared-memory attribute and launch a persistent grid of 128 CTAs;
// here a launch is a plain grid of one workgroup per output tile, the descriptors are
// built inside the kernel from the raw pointers, and nothing is cached between calls (the
// reference keeps descriptors in globals keyed on M alone, matmul_utils.cuh:49-51).
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

#include "../../include/mi_gemm.h"
#include "gemm_kernel.hpp"
#include "pack_kernel.hpp"
#include "splitk_common.hpp"   // splitk_reduce_kernel
#include "kernel_table.hpp"

namespace mi {
hipError_t launch_reference_gpu_gemm(int dtype, int M, int N, int K, const void* A, const void* B,
                                     void* C, float alpha, float beta, int cus, hipStream_t stream);
}

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return code;
}

#define MI_HIP(call)                                                                  \
    do {                                                                              \
        hipError_t e_ = (call);                                                       \
        if (e_ != hipSuccess)                                                         \
            return fail(MI_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
                        __FILE__, __LINE__);                                          \
    } while (0)

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// Preconditions of the decode (split-K streaming) kernels: whole 16-byte chunks and whole
// 64-deep K slabs, 8-byte aligned C rows.
bool shape_is_streamable(int M, int N, int K, const void* A, const void* B, const void* C) {
    (void)M;   // each decode kernel checks M against its own BM
    return N % 4 == 0 && K % 64 == 0 && aligned16(A) && aligned16(B) &&
           (((uintptr_t)C & 7u) == 0);
}
// The small-tile kernels take any M, N and K and store a C of any alignment: A and B on 4-byte
// boundaries are all they need.
bool shape_has_word_rows(int K, const void* A, const void* B) {
    (void)K;
    return (((uintptr_t)A | (uintptr_t)B) & 3u) == 0;
}

// Split-K geometry for a decode launch.  The decode kernel is bound by what one CU can pull
// from HBM (~26 GB/s, whatever it keeps in flight), so it wants a workgroup on every CU: as
// many pieces as fit into one round of the chip (128 x 8192 x 8192: 2 / 3 / 4 pieces 53 / 39.6 /
// 35.5 us), each at least four 64-deep slabs.  Pieces are contiguous ranges of whole slabs;
// the count is re-derived from the rounded-up piece length so that no piece is empty.
// MI_GEMM_SPLITK=<n> overrides (tuning aid).
int choose_splits(int tiles_n, int K, int cus) {
    static const int env = [] { const char* s = getenv("MI_GEMM_SPLITK"); return s ? atoi(s) : 0; }();
    const int slabs = K / 64;
    int splits = env > 0 ? env : cus / tiles_n;
    if (splits > slabs / 4) splits = slabs / 4;
    if (splits < 1) splits = 1;
    if (splits > 64) splits = 64;
    const int per = (slabs + splits - 1) / splits;
    return (slabs + per - 1) / per;
}
bool is_split_k_decode(int kind) { return kind == mi::KIND_DECODE; }

// Split-K for the tiled 16x16x32 kernel: when a shape has so few tiles that most CUs would
// idle (small M x N, long K), the K range is cut into pieces of whole 128-deep steps, one
// workgroup per (tile, piece); fp32 partials go to the workspace and splitk_reduce_kernel
// adds them in order.  The piece count comes from the time model of the kernel table
// (best_splits); the reduction's vector accesses need N % 4 == 0 and an 8-byte aligned C.
// (A trace buffer changes nothing: every workgroup of a split launch writes its record.)
// MI_GEMM_TILE_SPLITK=<n> forces a piece count (1 = never split; tuning aid).
bool shape_is_splittable(int N, const void* C) {
    return N % 4 == 0 && ((uintptr_t)C & 7u) == 0;
}

int choose_tile_splits(const mi::KernelEntry& e, int M, int N, int K, bool splittable, bool ptr_aligned, int cus,
                       int* k_per_split) {
    *k_per_split = K;
    static const int env = [] { const char* s = getenv("MI_GEMM_TILE_SPLITK"); return s ? atoi(s) : 0; }();
    if (!splittable || e.kind != mi::KIND_MFMA16 || e.kg > 1 || env == 1) return 1;   // (K groups split K inside the workgroup)
    if (env > 1) {
        int s = env < K / 512 ? env : K / 512;
        if (s < 2 || (long long)((M + e.BM - 1) / e.BM) * ((N + e.BN - 1) / e.BN) * 256 * 256 * 4 >= 0x7fffffffLL) return 1;
        const int kps = ((K + s - 1) / s + 127) / 128 * 128;
        s = (K + kps - 1) / kps;
        if (s < 2) return 1;
        *k_per_split = kps;
        return s;
    }
    return mi::best_splits(e, M, N, K, true, ptr_aligned, cus, k_per_split, nullptr);
}

// Split-K for the small-tile kernels: an output of a few tiles with a very long K (128 x 384 x
// 13376: 48 tiles of 32x32) leaves most CUs idle however small the tile, so K is cut into pieces
// of whole 64-deep units, one workgroup per (tile, piece), as above.  The piece count comes from
// the kernels' time model (best_wavek_splits).  MI_GEMM_SMALL_SPLITK=<n> forces a piece count
// (1 = never split; tuning aid).
int choose_small_tile_splits(const mi::KernelEntry& e, int M, int N, int K, bool splittable, int cus, int* k_per_split) {
    *k_per_split = K;
    static const int env = [] { const char* s = getenv("MI_GEMM_SMALL_SPLITK"); return s ? atoi(s) : 0; }();
    if (!splittable || e.kind != mi::KIND_WAVEK || env == 1) return 1;
    if (env > 1) {
        int s = env < K / 128 ? env : K / 128;
        if (s < 2 || (long long)s * M * N * 4 >= 0x7fffffffLL) return 1;
        const int kps = ((K + s - 1) / s + 63) / 64 * 64;
        s = (K + kps - 1) / kps;
        if (s < 2) return 1;
        *k_per_split = kps;
        return s;
    }
    return mi::best_wavek_splits(e, M, N, K, true, cus, k_per_split, nullptr);
}

// Split-K for the deep-ring kernels, as for the tiled one (MI_GEMM_TILE_SPLITK forces a piece count here too).
int choose_deep_splits(const mi::KernelEntry& e, int M, int N, int K, bool splittable, int cus, int* k_per_split) {
    *k_per_split = K;
    static const int env = [] { const char* s = getenv("MI_GEMM_TILE_SPLITK"); return s ? atoi(s) : 0; }();
    if (!splittable || env == 1) return 1;
    if (env > 1) {
        int s = env < K / 512 ? env : K / 512;
        if (s < 2 || (long long)M * N * 4 >= 0x7fffffffLL) return 1;
        const int kps = ((K + s - 1) / s + 127) / 128 * 128;
        s = (K + kps - 1) / kps;
        if (s < 2) return 1;
        *k_per_split = kps;
        return s;
    }
    return mi::best_deep_splits(e, M, N, K, true, cus, k_per_split, nullptr);
}

// ---- where the split-K kernels put their fp32 partial sums ----------------------------
// Three sources, chosen by the entry point:
//  * LIBRARY (mi_gemm_bf16 / _ex / _epilogue): one buffer per (device, stream) -- and thread, for
//    hipStreamPerThread, which is one handle for a stream of every thread -- allocated on first
//    use and replaced by a larger one on demand.  Launches already enqueued and captured graphs
//    keep a buffer's address, so a replaced buffer moves to the stream's retired list
//    (sizes are powers of two, so the retired ones together stay below the live one) and
//    nothing is freed behind the caller's back: mi_gemm_release_workspace frees a stream's
//    buffers (after synchronising it), and the table holds at most kMaxStreamWs streams per
//    device -- a further stream takes over an entry once the device is idle.  A stream that is
//    being captured cannot allocate: if it has no buffer that is large enough yet, the launch
//    runs unsplit instead.
//  * CALLER (mi_gemm_epilogue_ws): the caller's buffer, nothing is allocated; too small (or
//    NULL) means the launch runs unsplit.
//  * STATIC (mi_gemm_bf16_noalloc): the file-scope device array below, one copy per GPU the
//    library runs on, of a fixed size; a shape whose partials do not fit is refused.
// The kernels overwrite every partial they later read ([piece][M][N], all of it), so no
// buffer needs clearing between calls.
//
// A call that uses a buffer is two or three launches, which have to follow each other on the
// stream: with another call's launches on the same buffer in between (two threads on one
// stream), a GEMM would read the other call's copy and a reduction the other call's sums.  A
// call therefore holds the buffer's lock (buffer_order) from its first launch to its last;
// launches on different streams use different buffers.
constexpr int kMaxDevices = 64;
constexpr size_t kScratchBytes = MI_GEMM_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

enum WsMode { WS_LIBRARY, WS_CALLER, WS_STATIC };
struct WsSource {
    WsMode mode = WS_LIBRARY;
    void* ptr = nullptr;      // WS_CALLER: the caller's buffer
    size_t bytes = 0;
};
// Whose buffer an entry is.  hipStreamPerThread names another stream on every thread.
struct StreamKey {
    hipStream_t stream;
    uint64_t thread;
    bool operator==(const StreamKey& o) const { return stream == o.stream && thread == o.thread; }
};
StreamKey key_of(hipStream_t stream) {
    static std::atomic<uint64_t> threads{0};
    if (stream != hipStreamPerThread) return {stream, 0};
    static thread_local const uint64_t id = ++threads;        // (never reused, unlike the system's)
    return {stream, id};
}
struct StreamWs {
    StreamKey key;
    float* ptr;
    size_t bytes;
    std::vector<void*> retired;      // buffers this stream outgrew: an enqueued launch or a captured graph may still
                                     // hold their address, so they live until the stream's workspace is released
    size_t retired_bytes;
    int calls;                       // calls that took the buffer and have launches on it still to make (WsHold)
};
struct DeviceState {
    std::vector<std::unique_ptr<StreamWs>> ws;   // one entry per stream that used a workspace (at most kMaxStreamWs)
    unsigned char* scratch = nullptr;   // device address of `scratch` on this device
    int cus = 0;
    size_t refused = 0;                 // size of the last copy's buffer that could not be allocated, and when
    std::chrono::steady_clock::time_point refused_at;
};
// Streams with a buffer of their own per device.  A process that keeps creating streams does not
// grow the table beyond this: the next new stream waits for the device to go idle and takes over
// an entry (see acquire_workspace), so at most this many live buffers exist per device.
constexpr size_t kMaxStreamWs = 16;
// Most a launch takes of it for a copy of its operands (choose_packing); larger ones run on the
// operands as they are.
constexpr size_t kMaxPackedBytes = (size_t)2 << 30;
// The copy is an option and the memory for it is the caller's to use: no buffer is allocated for one
// that would take what the library holds on a device past kMaxCopyHeldBytes (one stream's largest and
// what it outgrew), and a size that could not be had is not asked for again, with hipMalloc's wait for
// the driver, before kRetryAfter.
constexpr size_t kMaxCopyHeldBytes = (size_t)8 << 30;
constexpr std::chrono::seconds kRetryAfter{1};
std::mutex g_ws_mutex;
std::condition_variable g_ws_idle;       // some entry's `calls` has become 0
DeviceState g_dev[kMaxDevices];

// Keeps the entry a call took its buffer from: until the call has launched everything that uses the
// buffer, waiting for the device says nothing about it, and the entry is neither taken over by another
// stream nor released.
class WsHold {
  public:
    WsHold() = default;
    WsHold(const WsHold&) = delete;
    WsHold& operator=(const WsHold&) = delete;
    ~WsHold() {
        if (!entry_) return;
        std::lock_guard<std::mutex> lock(g_ws_mutex);
        if (--entry_->calls == 0) g_ws_idle.notify_all();
    }
    void keep(StreamWs* entry) {         // (g_ws_mutex is held)
        if (entry_ == entry) return;
        if (entry_ && --entry_->calls == 0) g_ws_idle.notify_all();
        ++entry->calls;
        entry_ = entry;
    }

  private:
    StreamWs* entry_ = nullptr;
};

DeviceState& device_state() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) dev = 0;
    return g_dev[dev];
}

// Device address of the static scratch array on the current device.  In host code the
// array's name is only a handle for the runtime: the address a kernel can use comes from
// hipGetSymbolAddress, once per device (each GPU holds its own copy at its own address).
hipError_t static_scratch(unsigned char** out) {
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    DeviceState& st = device_state();
    if (!st.scratch) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        st.scratch = (unsigned char*)p;
    }
    *out = st.scratch;
    return hipSuccess;
}

// The lock over the launches of one call on the buffer that starts at `p`, whichever source it is from.
// (Buffers that share one only wait for a few launches.)
std::unique_lock<std::mutex> buffer_order(const void* p) {
    static std::mutex order[64];
    return std::unique_lock<std::mutex>(order[((uintptr_t)p * 0x9e3779b97f4a7c15ull) >> 58]);
}

void free_entry(StreamWs& w) {
    if (w.ptr) (void)hipFree(w.ptr);
    for (void* r : w.retired) (void)hipFree(r);
    w.ptr = nullptr;
    w.bytes = 0;
    w.retired.clear();
    w.retired_bytes = 0;
}

// 0: *out holds `bytes` of workspace; 1: none to be had without allocating where that is not
// possible (the caller runs the launch unsplit); < 0: MI_ERR_* with the message set.
// `hold` keeps a buffer of the library's in the caller's hands.  `required` false: the caller can
// do without, so no other stream's entry is taken over, little is held (kMaxCopyHeldBytes) and a
// failed allocation is 1.
int acquire_workspace(const WsSource& src, size_t bytes, hipStream_t stream, WsHold& hold, float** out,
                      bool required = true) {
    *out = nullptr;
    if (src.mode == WS_CALLER) {
        if (!src.ptr || src.bytes < bytes) return 1;
        *out = (float*)src.ptr;
        return 0;
    }
    if (src.mode == WS_STATIC) {
        if (bytes > kScratchBytes)
            return fail(MI_ERR_UNSUPPORTED,
                        "this shape's split-K partial sums need %zu bytes, the static scratch array holds %zu",
                        bytes, kScratchBytes);
        unsigned char* p = nullptr;
        hipError_t e = static_scratch(&p);
        if (e != hipSuccess)
            return fail(MI_ERR_HIP, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
        *out = (float*)p;
        return 0;
    }
    const StreamKey key = key_of(stream);
    std::unique_lock<std::mutex> lock(g_ws_mutex);
    DeviceState& st = device_state();
    StreamWs* mine = nullptr;
    for (;;) {
        bool idle = false;
        for (const auto& w : st.ws) {
            if (w->key == key) mine = w.get();
            if (w->calls == 0) idle = true;
        }
        if (mine || !required || st.ws.size() < kMaxStreamWs || idle) break;
        g_ws_idle.wait(lock);      // (every entry's stream is between two launches of a call)
    }
    if (mine && mine->bytes >= bytes) {
        hold.keep(mine);
        *out = mine->ptr;
        return 0;
    }
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) != hipSuccess) {
        (void)hipGetLastError();
        return 1;      // e.g. the null stream while another stream captures: do not allocate
    }
    if (cap != hipStreamCaptureStatusNone) return 1;
    size_t want = (size_t)4 << 20;
    while (want < bytes) want <<= 1;
    if (!required) {
        size_t held = 0;
        for (const auto& w : st.ws) held += w->bytes + w->retired_bytes;
        if (held + want > kMaxCopyHeldBytes) return 1;
        if (st.refused && want >= st.refused && std::chrono::steady_clock::now() - st.refused_at < kRetryAfter) return 1;
    }
    if (!mine && st.ws.size() >= kMaxStreamWs) {
        if (!required) return 1;
        // The table is full (a process that keeps making streams, or never releases): once the
        // device is idle no launch holds any buffer that no call is about to use, so the smallest
        // entry of those changes hands -- its buffer as it is when large enough, else freed here and
        // replaced below.
        hipError_t e = hipDeviceSynchronize();
        if (e != hipSuccess)
            return fail(MI_ERR_HIP, "hipDeviceSynchronize before reusing a split-K workspace failed: %s", hipGetErrorString(e));
        StreamWs* take = nullptr;
        for (const auto& w : st.ws)     // the smallest entry that is already large enough ...
            if (w->calls == 0 && w->bytes >= bytes && (!take || w->bytes < take->bytes)) take = w.get();
        if (!take)
            for (const auto& w : st.ws)   // ... else the smallest of all
                if (w->calls == 0 && (!take || w->bytes < take->bytes)) take = w.get();
        for (void* r : take->retired) (void)hipFree(r);
        take->retired.clear();
        take->retired_bytes = 0;
        take->key = key;
        if (take->bytes >= bytes) {
            hold.keep(take);
            *out = take->ptr;
            return 0;
        }
        if (take->ptr) (void)hipFree(take->ptr);
        take->ptr = nullptr;
        take->bytes = 0;
        mine = take;
    }
    float* p = nullptr;
    // (relaxed for this thread: the allocation concerns no capture another thread has under way)
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool relaxed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    hipError_t e = hipMalloc((void**)&p, want);
    if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess && !required) {
        (void)hipGetLastError();
        st.refused = want;
        st.refused_at = std::chrono::steady_clock::now();
        return 1;
    }
    if (e != hipSuccess)
        return fail(MI_ERR_HIP, "split-K workspace allocation of %zu bytes failed: %s", want, hipGetErrorString(e));
    if (mine) {
        if (mine->ptr) mine->retired.push_back(mine->ptr);
        mine->retired_bytes += mine->bytes;
        mine->ptr = p;
        mine->bytes = want;
    } else {
        st.ws.push_back(std::unique_ptr<StreamWs>(new StreamWs{key, p, want, {}, 0, 0}));
        mine = st.ws.back().get();
    }
    hold.keep(mine);
    *out = p;
    return 0;
}

bool is_capturing(hipStream_t stream) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) != hipSuccess) {
        (void)hipGetLastError();
        return true;       // e.g. the null stream while another stream captures
    }
    return cap != hipStreamCaptureStatusNone;
}

int compute_units() {
    DeviceState& st = device_state();
    if (st.cus == 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
            st.cus = n;
        else
            st.cus = 256;
    }
    return st.cus;
}

// The aligned kernels assume full tiles, K a multiple of two K steps, 16-byte aligned
// rows of A and B and 8-byte aligned rows of C; everything else takes the predicated twin.
bool shape_is_aligned(const mi::KernelEntry& e, int M, int N, int K, const void* A,
                      const void* B, const void* C) {
    return M % e.BM == 0 && N % e.BN == 0 && K % 128 == 0 && aligned16(A) && aligned16(B) &&
           aligned16(C);
}

// Shapes a launch accepts: positive extents, `int` element indices as in the reference
// (reference.h:30,40 index with int) and 32-bit byte offsets inside one tile's row panel.
bool shape_in_range(int M, int N, int K) {
    return M > 0 && N > 0 && K > 0 && (long long)M * K <= 0x7fffffffLL && (long long)N * K <= 0x7fffffffLL &&
           (long long)M * N <= 0x7fffffffLL && (long long)K * 2 * 256 <= 0x7fffffffLL;
}

int check_args(int config, int dtype, int M, int N, int K, const void* A, const void* B,
               const void* C) {
    if (dtype != MI_DTYPE_BF16 && dtype != MI_DTYPE_FP16)
        return fail(MI_ERR_INVALID, "unknown dtype %d", dtype);
    if (M <= 0 || N <= 0 || K <= 0)
        return fail(MI_ERR_INVALID, "M, N, K must be positive (got %d, %d, %d)", M, N, K);
    if (!A || !B || !C) return fail(MI_ERR_INVALID, "null matrix pointer");
    if (config != MI_CONFIG_AUTO && (config < 0 || config >= mi::kNumKernels))
        return fail(MI_ERR_INVALID, "unknown kernel config %d", config);
    // 32-bit byte offsets inside one tile's row panel, and `int` element indices as in the
    // reference (reference.h:30,40 index with int).
    if ((long long)M * K > 0x7fffffffLL || (long long)N * K > 0x7fffffffLL ||
        (long long)M * N > 0x7fffffffLL)
        return fail(MI_ERR_INVALID, "matrix with more than 2^31-1 elements");
    if ((long long)K * 2 * 256 > 0x7fffffffLL) return fail(MI_ERR_INVALID, "K too large");
    return MI_OK;
}

// Tuned shapes from a file: MI_GEMM_TUNED_FILE names a text file with one `M N K config-name`
// per line (# starts a comment), read once, on first use.  A shape listed there skips the
// time model when its configuration can run the call (the decode kernels have preconditions);
// lines that do not parse or name no compiled configuration are ignored.  Keyed on all of
// M, N and K (the reference keys its cached descriptors on M alone, matmul_utils.cuh:49-51).
struct TunedEntry {
    int M, N, K, config;
};
const std::vector<TunedEntry>& tuned_entries() {
    static const std::vector<TunedEntry> table = [] {
        std::vector<TunedEntry> t;
        const char* path = getenv("MI_GEMM_TUNED_FILE");
        FILE* f = path && *path ? fopen(path, "r") : nullptr;
        if (!f) return t;
        char line[256];
        while (fgets(line, sizeof(line), f)) {
            if (char* hash = strchr(line, '#')) *hash = 0;
            int M = 0, N = 0, K = 0;
            char name[128];
            if (sscanf(line, "%d %d %d %127s", &M, &N, &K, name) != 4 || M <= 0 || N <= 0 || K <= 0) continue;
            for (int i = 0; i < mi::kNumKernels; ++i)
                if (strcmp(name, mi::kKernels[i].name) == 0) {
                    t.push_back({M, N, K, i});
                    break;
                }
        }
        fclose(f);
        return t;
    }();
    return table;
}
// config for (M, N, K) from the tuned file, or -1
int tuned_config(int M, int N, int K, bool streamable, bool ptr_aligned, bool small_ok) {
    for (const TunedEntry& t : tuned_entries()) {
        if (t.M != M || t.N != N || t.K != K) continue;
        const mi::KernelEntry& e = mi::kKernels[t.config];
        if ((is_split_k_decode(e.kind) || e.kind == mi::KIND_STREAM) && (!streamable || M > e.BM)) continue;
        if (e.kind == mi::KIND_WAVEK && !small_ok) continue;
        if (e.kind == mi::KIND_DEEP && !mi::deep_runs(K, ptr_aligned)) continue;
        if (e.kg > 1 && K % (128 * e.kg) != 0) continue;      // (the rule mi_gemm_config_supports applies)
        return t.config;
    }
    return -1;
}

// The automatic choice is a pure function of the shape and three flags and costs 1-3 us of
// host time (the time model runs over every candidate and piece count), which shows when
// small GEMMs are launched back to back: the last few answers are kept per thread, keyed on
// all of its inputs.  (No pointer or other per-call state is cached.)
struct Choice {
    int M, N, K, flags, requested, cus;   // key; requested = the caller's config (MI_CONFIG_AUTO or an index)
    int config, splits, k_per_split;
    bool deep;                            // the config's deep-ring kernel runs the call
};
Choice compute_choice(int requested, int M, int N, int K, bool streamable, bool splittable, bool ptr_aligned,
                      bool small_ok) {
    const int flags = (streamable ? 1 : 0) | (splittable ? 2 : 0) | (ptr_aligned ? 4 : 0) | (small_ok ? 8 : 0);
    const int cus = compute_units();
    Choice c{M, N, K, flags, requested, cus, requested, 1, K, false};
    if (requested == MI_CONFIG_AUTO) {
        c.config = tuned_config(M, N, K, streamable, ptr_aligned, small_ok);
        if (c.config < 0) c.config = mi::select_kernel(M, N, K, streamable, splittable, ptr_aligned, small_ok, cus);
    }
    // (a config that has only a deep-ring kernel runs what that cannot on 128x128 tiles)
    if (mi::kKernels[c.config].kind == mi::KIND_DEEP && !mi::deep_runs(K, ptr_aligned)) c.config = mi::kDeepTwin;
    const mi::KernelEntry& e = mi::kKernels[c.config];
    c.deep = mi::deep_takes(e, K, ptr_aligned);
    if (c.deep) {
        c.splits = choose_deep_splits(e, M, N, K, splittable, cus, &c.k_per_split);
    } else if (e.kind == mi::KIND_MFMA16) {
        c.splits = choose_tile_splits(e, M, N, K, splittable, ptr_aligned, cus, &c.k_per_split);
    } else if (is_split_k_decode(e.kind) && streamable && M <= e.BM) {
        const int tiles_n = (N + e.BN - 1) / e.BN;
        c.splits = choose_splits(tiles_n, K, cus);   // no empty split
        c.k_per_split = ((K / 64 + c.splits - 1) / c.splits) * 64;
    } else if (e.kind == mi::KIND_WAVEK) {
        c.splits = choose_small_tile_splits(e, M, N, K, splittable, cus, &c.k_per_split);
    }
    return c;
}
Choice choose(int requested, int M, int N, int K, bool streamable, bool splittable, bool ptr_aligned, bool small_ok) {
    static thread_local Choice memo[4] = {};
    static thread_local int next = 0;
    const int flags = (streamable ? 1 : 0) | (splittable ? 2 : 0) | (ptr_aligned ? 4 : 0) | (small_ok ? 8 : 0);
    const int cus = compute_units();
    for (const Choice& c : memo)
        if (c.M == M && c.N == N && c.K == K && c.flags == flags && c.requested == requested && c.cus == cus &&
            c.splits > 0)
            return c;
    const Choice c = compute_choice(requested, M, N, K, streamable, splittable, ptr_aligned, small_ok);
    memo[next] = c;
    next = (next + 1) & 3;
    return c;
}

// Which operands of a tiled launch are first copied to rows that start on 128-byte lines
// (pack_operands_kernel), a pure function of the choice and the shape.
//
// With K % 64 != 0 the K loop of the 16x16x32 kernel runs at 0.69-0.83 of its rate on whole lines
// (4095 x 6143 with K = 3073 / 3072: 180.7 / 124.6 us; 8191^3 941, 8191 x 8191 x 8192 725).  What
// the copy saves grows with M*N*K and with the rows a tile loads for its area, less what its MFMAs
// hide: in us per product of extents, 3.5e-10 with 256x256 tiles (measured 2.8-4.4e-10), 6.4e-10 with
// 256x192 (5.9-8.9), 9.2e-10 with 192x192 (7.6-11.5), 12e-10 with 128x256 (11-15.8), 15e-10 with
// 192x128 (14.7-18), 21e-10 with 128x128 (15.7-27).  It is less where CUs idle and with a short K (on
// 450 shapes the median factor before 1 / BM + 1 / BN - 0.0062 is 2.2e-7 from memory and 1.3e-7 with the
// operands in the caches for a K of 1000-2000, 2.9e-7 and 1.5e-7 from 4000; half below 2450, 3200
// where two workgroups on a CU hide each other's loads, leaves as little on the table as a smooth fall);
// less where rows start on 32- or 64-byte boundaries and straddle fewer lines, more on odd 2-byte
// ones.  One operand alone: 0.45 of it with 256x256 tiles, and with the others when the copied one is
// much the smaller (9000x1024x9000 223 -> 189 by B; 3000^3 67 -> 74 by A).  The copy costs its launch
// and 7.5e-7 us per element (5 TB/s).
//
// With the operands left in the caches the copy costs the same and saves half, so one line for both
// gives something away on either side.  On 970 shapes of 1000-9000 rows and columns, this rule and the
// same one blind to the rows' boundary against no copy (geometric mean; shapes > 2 % slower, the worst):
//     from memory     -6.0 %,  6, 15 %    (-5.8 %, 12, 15 %)
//     A in the caches -3.1 %, 64, 24 %    (-2.8 %, 79, 24 %)
//     both there      +0.2 %, 143, 45 %   (+0.5 %, 165, 45 %)
// and one drawn to lose little in the caches (1.7e-7; 317 copies instead of 379): -5.3 / -3.0 / -0.3 %,
// 5 / 42 / 91 shapes, but 97 of them slower from memory by 2-32 % than with the copies it leaves out.
// None / A / B / both in us, from memory: 4095x6143x3073 181 / 167 / 168 / 145, 3000^3 67 / 74 / 72 / 63,
// 2100x2100x9000 in two pieces 109 / 118 / 116 / 99, 2048x28672x4100 454 / 408 / 488 / 457,
// 28672x2048x4100 482 / 500 / 454 / 463; none / both: 1435x3790x13542 229 / 173, 2485x1090x5883 89 / 65;
// left as they are: 2100x2100x9000, 2048x2048x2049 29 / 32, 3333x3333x1111 36 / 44,
// 854x3626x2574 32 / 39, 4000x4000x600 31 / 39.
struct PackPlan {
    bool a, b;
    bool any() const { return a || b; }
    size_t bytes(int M, int N, int K) const {
        return ((a ? (size_t)M : 0) + (b ? (size_t)N : 0)) * (size_t)((K + 63) / 64 * 64) * 2;
    }
};
PackPlan choose_packing(const Choice& c, int M, int N, int K) {
    const mi::KernelEntry& e = mi::kKernels[c.config];
    PackPlan best{false, false};
    if (K % 64 == 0 || e.kind != mi::KIND_MFMA16 || e.kg > 1 || c.deep) return best;
    const double mnk = (double)M * N * K;
    double rate = 2.2e-7 * (1.0 / e.BM + 1.0 / e.BN - 0.0062);
    if (K < (e.occ > 1 ? 3200 : 2450)) rate *= 0.5;
    rate *= K % 2 != 0 ? 1.2 : K % 16 != 0 ? 1.0 : K % 32 != 0 ? 0.8 : 0.6;
    const double wgs = (double)((M + e.BM - 1) / e.BM) * ((N + e.BN - 1) / e.BN) * c.splits;
    if (wgs < c.cus) rate *= std::sqrt(wgs / c.cus);
    double best_gain = 3.6e-11 * mnk;                        // 2 % of the launch at 1.1 PFLOP/s
    for (int which = 1; which <= 3; ++which) {
        const PackPlan p{(which & 1) != 0, (which & 2) != 0};
        if (p.bytes(M, N, K) > kMaxPackedBytes) continue;
        if (which != 3 && e.BM + e.BN < 512 && (p.a ? 6LL * M > N : 6LL * N > M)) continue;
        const double gain = (which == 3 ? 1.0 : 0.45) * rate * mnk - 4.0 - 7.5e-7 * ((p.a ? (double)M : 0.0) + (p.b ? (double)N : 0.0)) * K;
        if (gain > best_gain) {
            best = p;
            best_gain = gain;
        }
    }
    return best;
}
size_t choice_workspace(const Choice& c, int M, int N, int K) {
    return choose_packing(c, M, N, K).bytes(M, N, K) + (c.splits > 1 ? (size_t)c.splits * M * N * sizeof(float) : 0);
}

// The cut of a large ragged shape into two GEMMs is a pure function of the shape and four flags
// like the kernel choice, and costs several passes of the time model: the last answer is kept per
// thread.  MI_GEMM_ROW_CUT=0 switches the cut off (measurement aid).
int rows_to_cut(int M, int N, int K, bool streamable, bool splittable, bool ptr_aligned, bool small_ok) {
    static const int env = [] { const char* s = getenv("MI_GEMM_ROW_CUT"); return s ? atoi(s) : 1; }();
    if (env == 0 || (long long)M * N < 4096LL * 4096LL) return 0;
    struct Memo { int M, N, K, flags, cus, m1; };
    static thread_local Memo memo = {0, 0, 0, -1, 0, 0};
    const int flags = (streamable ? 1 : 0) | (splittable ? 2 : 0) | (ptr_aligned ? 4 : 0) | (small_ok ? 8 : 0);
    const int cus = compute_units();
    if (memo.M != M || memo.N != N || memo.K != K || memo.flags != flags || memo.cus != cus)
        memo = {M, N, K, flags, cus, mi::rows_to_split_off(M, N, K, streamable, splittable, ptr_aligned, small_ok, cus)};
    return memo.m1;
}

// Workgroups the main kernel of a launch has (the grid a trace buffer's records are indexed by).
size_t launch_workgroups(const mi::KernelEntry& e, int M, int N, int splits) {
    const size_t tiles_n = (size_t)(N + e.BN - 1) / e.BN;
    if (e.kind == mi::KIND_STREAM || is_split_k_decode(e.kind)) return tiles_n * (size_t)splits;
    return (size_t)((M + e.BM - 1) / e.BM) * tiles_n * (size_t)splits;
}

// ... for a call that names the config, with operands and C on 16-byte boundaries or not (C on 8 bytes: a K in pieces)
size_t config_workgroups(int config, int M, int N, int K, bool ptr_aligned) {
    const Choice c = compute_choice(config, M, N, K, ptr_aligned && N % 4 == 0 && K % 64 == 0, N % 4 == 0, ptr_aligned, true);
    return launch_workgroups(mi::kKernels[c.config], M, N, c.splits);
}

// One GEMM launch (more with split-K and with a copy of the operands): argument checks, kernel choice, aligned / predicated twin.
// `may_cut`: the automatic choice may run the shape as two GEMMs, the first rows and the rest
// (rows_to_split_off in the kernel table); the parts themselves are not cut again.
int run_gemm(int config, int dtype, int M, int N, int K, const void* A, const void* B, void* C,
             int* DB, float alpha, float beta, void* stream, const WsSource& wsrc = WsSource{}, bool may_cut = true) {
    int rc = check_args(config, dtype, M, N, K, A, B, C);
    if (rc != MI_OK) return rc;
    const bool streamable = shape_is_streamable(M, N, K, A, B, C);
    if (may_cut && config == MI_CONFIG_AUTO &&
        tuned_config(M, N, K, streamable, aligned16(A) && aligned16(B) && aligned16(C), shape_has_word_rows(K, A, B)) < 0) {       // (a tuned shape runs as tuned)
        const int m1 = rows_to_cut(M, N, K, streamable, shape_is_splittable(N, C),
                                   aligned16(A) && aligned16(B) && aligned16(C), shape_has_word_rows(K, A, B));
        if (m1 > 0) {
            // Both parts' workspace is settled before anything is launched: a part that could not
            // get its partial sums' room (the static array too small, an allocation that fails)
            // must not leave the other part's rows of C written and the call failed.
            const void* A2 = (const unsigned char*)A + (size_t)m1 * K * 2;
            void* C2 = (unsigned char*)C + (size_t)m1 * N * 2;
            size_t need = 0;
            WsHold hold;                     // (until both parts are launched)
            size_t wgs_first = 0;            // workgroups of the first part: the second part's trace records follow theirs
            for (int part = 0; part < 2; ++part) {
                const int Mp = part ? M - m1 : m1;
                const void* Ap = part ? A2 : A;
                const void* Cp = part ? C2 : C;
                const Choice c = choose(config, Mp, N, K, shape_is_streamable(Mp, N, K, Ap, B, Cp), shape_is_splittable(N, Cp),
                                        aligned16(Ap) && aligned16(B) && aligned16(Cp), shape_has_word_rows(K, Ap, B));
                const size_t b = c.splits > 1 ? (size_t)c.splits * Mp * N * sizeof(float) : 0;
                if (b > need) need = b;
                if (part == 0) wgs_first = launch_workgroups(mi::kKernels[c.config], Mp, N, c.splits);
            }
            if (need > 0) {
                float* unused = nullptr;
                const int wrc = acquire_workspace(wsrc, need, (hipStream_t)stream, hold, &unused);
                if (wrc < 0) return wrc;
            }
            rc = run_gemm(config, dtype, m1, N, K, A, B, C, DB, alpha, beta, stream, wsrc, false);
            if (rc != MI_OK) return rc;
            return run_gemm(config, dtype, M - m1, N, K, A2, B, C2, DB ? DB + 6 * wgs_first : nullptr, alpha, beta, stream,
                            wsrc, false);
        }
    }
    // (a trace buffer does not change the choice: every kernel family writes the records)
    const Choice choice = choose(config, M, N, K, streamable, shape_is_splittable(N, C),
                                 aligned16(A) && aligned16(B) && aligned16(C), shape_has_word_rows(K, A, B));
    config = choice.config;
    const mi::KernelEntry& e = mi::kKernels[config];

    mi::GemmArgs args;
    args.A = A;
    args.B = B;
    args.C = C;
    args.M = M;
    args.N = N;
    args.K = K;
    args.lda = K;
    args.ldb = K;
    args.ldc = N;
    args.tiles_m = (M + e.BM - 1) / e.BM;
    args.tiles_n = (N + e.BN - 1) / e.BN;
    args.c_vec_ok = (N % 4 == 0) && (((uintptr_t)C & 7u) == 0);
    args.DB = DB;
    args.ws = nullptr;
    args.splits = 1;
    args.k_per_split = K;
    args.alpha = alpha;
    args.beta = beta;
    WsHold hold;
    std::unique_lock<std::mutex> order;      // from the call's first launch on a workspace to its last

    if (e.kind == mi::KIND_STREAM) {
        if (!streamable || M > e.BM)
            return fail(MI_ERR_UNSUPPORTED,
                        "config %s needs M <= %d, N %% 4 == 0, K %% 64 == 0 and 16-byte aligned operands",
                        e.name, e.BM);
        hipError_t err = e.launch[dtype][0](args, (hipStream_t)stream);
        if (err != hipSuccess)
            return fail(MI_ERR_HIP, "launch of %s failed: %s", e.name, hipGetErrorString(err));
        return MI_OK;
    }
    if (e.kind == mi::KIND_WAVEK && !choice.deep) {
        if (!shape_has_word_rows(K, A, B))
            return fail(MI_ERR_UNSUPPORTED, "config %s needs 4-byte aligned A and B", e.name);
        args.splits = choice.splits;
        args.k_per_split = choice.k_per_split;
        if (args.splits > 1) {
            const int wrc = acquire_workspace(wsrc, (size_t)args.splits * M * N * sizeof(float), (hipStream_t)stream, hold, &args.ws);
            if (wrc < 0) return wrc;
            if (wrc == 0) order = buffer_order(wsrc.ptr ? wsrc.ptr : args.ws);
            if (wrc > 0) {           // no workspace to be had: every tile walks all of K
                args.splits = 1;
                args.k_per_split = K;
            }
        }
        hipError_t err = e.launch[dtype][0](args, (hipStream_t)stream);
        if (err != hipSuccess)
            return fail(MI_ERR_HIP, "launch of %s failed: %s", e.name, hipGetErrorString(err));
        return MI_OK;
    }
    if (is_split_k_decode(e.kind)) {
        if (!streamable || M > e.BM)
            return fail(MI_ERR_UNSUPPORTED,
                        "config %s needs M <= %d, N %% 4 == 0, K %% 64 == 0 and 16-byte aligned operands",
                        e.name, e.BM);
        args.splits = choice.splits;
        args.k_per_split = choice.k_per_split;
        if (args.splits > 1) {
            const int wrc = acquire_workspace(wsrc, (size_t)args.splits * M * N * sizeof(float), (hipStream_t)stream, hold, &args.ws);
            if (wrc < 0) return wrc;
            if (wrc == 0) order = buffer_order(wsrc.ptr ? wsrc.ptr : args.ws);
            if (wrc > 0) {           // no workspace to be had: one pass over all of K
                args.splits = 1;
                args.k_per_split = K;
            }
        }
        hipError_t err = e.launch[dtype][0](args, (hipStream_t)stream);
        if (err != hipSuccess)
            return fail(MI_ERR_HIP, "launch of %s failed: %s", e.name, hipGetErrorString(err));
        return MI_OK;
    }

    if (e.kg > 1 && K % (128 * e.kg) != 0)
        return fail(MI_ERR_UNSUPPORTED, "config %s splits K over %d groups of waves and needs K %% %d == 0", e.name,
                    e.kg, 128 * e.kg);
    if (e.kind == mi::KIND_MFMA16 || choice.deep) {
        args.splits = choice.splits;
        args.k_per_split = choice.k_per_split;
        const size_t split_bytes = args.splits > 1 ? (size_t)args.splits * M * N * sizeof(float) : 0;
        // The copy of the operands is an option: without room for it (the static array, a caller's
        // workspace that is too small, no memory) the launch runs on the operands as they are, to the
        // same bits.  Not from the library's buffer under capture: a graph of such a launch needed
        // no workspace and may be replayed on any stream.
        PackPlan plan = choose_packing(choice, M, N, K);
        float* room = nullptr;
        WsSource lines = wsrc;                      // from the first 128-byte line of a caller's workspace on
        if (lines.mode == WS_CALLER) {
            const size_t skip = (size_t)(-(uintptr_t)lines.ptr & 127u);
            lines.ptr = lines.ptr && lines.bytes >= skip ? (unsigned char*)lines.ptr + skip : nullptr;
            lines.bytes = lines.ptr ? lines.bytes - skip : 0;
        }
        if (plan.any() && (wsrc.mode == WS_STATIC || (wsrc.mode == WS_LIBRARY && is_capturing((hipStream_t)stream)) ||
                           acquire_workspace(lines, plan.bytes(M, N, K) + split_bytes, (hipStream_t)stream, hold, &room, false) != 0))
            plan = {false, false};
        if (plan.any()) {
            order = buffer_order(wsrc.ptr ? wsrc.ptr : room);
            unsigned char* packed = (unsigned char*)room;
            const int pitch = (K + 63) / 64 * 64;
            mi::PackArgs pa;
            pa.src[0] = (const uint16_t*)(plan.a ? A : B);
            pa.src[1] = (const uint16_t*)B;
            pa.out = (uint16_t*)packed;
            pa.rows_first = (uint32_t)(plan.a ? M : N);
            pa.chunks = (uint32_t)pitch / 8u;
            pa.total = (pa.rows_first + (plan.a && plan.b ? (uint32_t)N : 0u)) * pa.chunks;
            pa.K = K;
            const uint32_t per_block = 256u * mi::kPackChunks;
            hipError_t err = mi::launch_kernel(mi::pack_operands_kernel, dim3((pa.total + per_block - 1) / per_block), dim3(256),
                                               (hipStream_t)stream, pa);
            if (err != hipSuccess) return fail(MI_ERR_HIP, "launch of the operand copy failed: %s", hipGetErrorString(err));
            if (plan.a) { args.A = packed; args.lda = pitch; }
            if (plan.b) { args.B = packed + (plan.a ? (size_t)M * pitch * 2 : 0); args.ldb = pitch; }
            if (plan.a && plan.b) args.K = pitch;       // both end in zeros: no K tail
            if (split_bytes) args.ws = (float*)(packed + plan.bytes(M, N, K));
        } else if (args.splits > 1) {
            const int wrc = acquire_workspace(wsrc, split_bytes, (hipStream_t)stream, hold, &args.ws);
            if (wrc < 0) return wrc;
            if (wrc == 0) order = buffer_order(wsrc.ptr ? wsrc.ptr : args.ws);
            if (wrc > 0) {
                args.splits = 1;
                args.k_per_split = K;
            }
        }
        if (args.splits == 1) args.k_per_split = args.K;
    }
    const bool edge = choice.deep ? K % 64 != 0 : !shape_is_aligned(e, M, N, args.K, args.A, args.B, C);
    mi::LaunchFn fn = choice.deep ? e.deep[dtype][edge ? 1 : 0] : e.launch[dtype][edge ? 1 : 0];
    if (!fn) return fail(MI_ERR_UNSUPPORTED, "config %s has no %s kernel for dtype %d", e.name,
                         edge ? "predicated" : "aligned", dtype);
    hipError_t err = fn(args, (hipStream_t)stream);
    if (err != hipSuccess)
        return fail(MI_ERR_HIP, "launch of %s failed: %s", e.name, hipGetErrorString(err));
    if (args.splits > 1) {
        const size_t quads = ((size_t)M * N + 3) / 4;
        const dim3 rgrid((unsigned)((quads + 255) / 256));
        err = dtype == MI_DTYPE_BF16
                  ? mi::launch_kernel(mi::splitk_reduce_kernel<mi::DT_BF16>, rgrid, dim3(256), (hipStream_t)stream,
                                      args.ws, C, M, N, N, args.splits, alpha, beta)
                  : mi::launch_kernel(mi::splitk_reduce_kernel<mi::DT_FP16>, rgrid, dim3(256), (hipStream_t)stream,
                                      args.ws, C, M, N, N, args.splits, alpha, beta);
        if (err != hipSuccess)
            return fail(MI_ERR_HIP, "launch of the split-K reduction failed: %s", hipGetErrorString(err));
    }
    return MI_OK;
}

}  // namespace

extern "C" {

const char* mi_last_error(void) { return g_err; }

int mi_gemm_num_configs(void) { return mi::kNumKernels; }

const char* mi_gemm_config_name(int config) {
    if (config < 0 || config >= mi::kNumKernels) return nullptr;
    return mi::kKernels[config].name;
}

int mi_gemm_find_config(const char* name) {
    if (!name) return -1;
    for (int i = 0; i < mi::kNumKernels; ++i)
        if (strcmp(name, mi::kKernels[i].name) == 0) return i;
    return -1;
}

int mi_gemm_config_lds_bytes(int config) {
    if (config < 0 || config >= mi::kNumKernels) return 0;
    return mi::kKernels[config].lds_bytes;
}

int mi_gemm_config_supports(int config, int dtype, int M, int N, int K) {
    if (config < 0 || config >= mi::kNumKernels) return 0;
    if (dtype != MI_DTYPE_BF16 && dtype != MI_DTYPE_FP16) return 0;
    if (!shape_in_range(M, N, K)) return 0;
    const mi::KernelEntry& e = mi::kKernels[config];
    if (is_split_k_decode(e.kind) || e.kind == mi::KIND_STREAM)
        return M <= e.BM && N % 4 == 0 && K % 64 == 0;
    if (e.kind == mi::KIND_WAVEK) return 1;
    if (e.kg > 1 && K % (128 * e.kg) != 0) return 0;
    return e.kind == mi::KIND_DEEP || e.launch[dtype][1] != nullptr;
}

int mi_gemm_config_grid(int config, int M, int N, int K) {
    if (config < 0 || config >= mi::kNumKernels || !shape_in_range(M, N, K)) return 0;
    const mi::KernelEntry& e = mi::kKernels[config];
    if (e.kind == mi::KIND_STREAM) return M > e.BM || K % 64 != 0 ? 0 : (N + e.BN - 1) / e.BN;
    if (is_split_k_decode(e.kind)) {
        if (M > e.BM || K % 64 != 0) return 0;
        const int tiles_n = (N + e.BN - 1) / e.BN;
        return tiles_n * choose_splits(tiles_n, K, compute_units());
    }
    // (operands and C on 16-byte boundaries)
    return (int)config_workgroups(config, M, N, K, true);
}

int mi_gemm_select_config(int dtype, int M, int N, int K) {
    (void)dtype;
    if (!shape_in_range(M, N, K)) return -1;
    // pointer alignment is unknown here: assume the usual 256-byte aligned allocations
    const bool streamable = N % 4 == 0 && K % 64 == 0;
    const int tuned = tuned_config(M, N, K, streamable, true, true);
    if (tuned >= 0) return tuned;
    return mi::select_kernel(M, N, K, streamable, N % 4 == 0, true, true, compute_units());
}

int mi_gemm_row_cut(int dtype, int M, int N, int K) {
    (void)dtype;
    if (!shape_in_range(M, N, K)) return 0;
    const bool streamable = N % 4 == 0 && K % 64 == 0;
    if (tuned_config(M, N, K, streamable, true, true) >= 0) return 0;
    return rows_to_cut(M, N, K, streamable, N % 4 == 0, true, true);
}

int mi_gemm_tuned_entries(void) { return (int)tuned_entries().size(); }

size_t mi_gemm_trace_words(int M, int N, int K) {
    // enough for whichever kernel configuration ends up running the shape, with the boundaries of the
    // operands and C as they may be (a config's call on 4- or 8-byte boundaries can be another kernel's, in
    // more pieces) -- or its two parts, one after the other, where the automatic choice cuts the shape's rows
    auto largest = [&](int rows) {
        size_t grid = 0;
        for (int c = 0; c < mi::kNumKernels; ++c)
            for (int aligned = 0; aligned < 2; ++aligned) {
                const size_t g = config_workgroups(c, rows, N, K, aligned != 0);
                if (g > grid) grid = g;
            }
        return grid;
    };
    if (!shape_in_range(M, N, K)) return 1;
    size_t grid = largest(M);
    for (int flags = 0; flags < 16; ++flags) {
        const int m1 = rows_to_cut(M, N, K, (flags & 1) != 0 && N % 4 == 0 && K % 64 == 0, (flags & 2) != 0 && N % 4 == 0,
                                   (flags & 4) != 0, (flags & 8) != 0);
        if (m1 > 0 && largest(m1) + largest(M - m1) > grid) grid = largest(m1) + largest(M - m1);
    }
    return grid * 6 + 1;
}

int mi_gemm_ex(int config, int dtype, int M, int N, int K, const void* A, const void* B,
               void* C, int* DB, void* stream) {
    return run_gemm(config, dtype, M, N, K, A, B, C, DB, 1.0f, 0.0f, stream);
}

int mi_gemm_epilogue(int config, int dtype, int M, int N, int K, const void* A, const void* B,
                     void* C, float alpha, float beta, int c_layout, void* stream) {
    if (c_layout != MI_C_ROW_MAJOR && c_layout != MI_C_COL_MAJOR)
        return fail(MI_ERR_INVALID, "unknown C layout %d", c_layout);
    if (!(alpha == alpha) || !(beta == beta)) return fail(MI_ERR_INVALID, "alpha or beta is NaN");
    // Column-major C (M x N, element (m, n) at C[n*M + m]) is the row-major N x M matrix
    // C^T = B . A^T: the same GEMM with the operands and their extents exchanged.  Every
    // element is still the k-ordered sum the kernels form for the row-major case.
    if (c_layout == MI_C_COL_MAJOR)
        return run_gemm(config, dtype, N, M, K, B, A, C, nullptr, alpha, beta, stream);
    return run_gemm(config, dtype, M, N, K, A, B, C, nullptr, alpha, beta, stream);
}

int mi_gemm_bf16(int M, int N, int K, const uint16_t* A, const uint16_t* B, uint16_t* C, int* DB,
                 void* stream) {
    return mi_gemm_ex(MI_CONFIG_AUTO, MI_DTYPE_BF16, M, N, K, A, B, C, DB, stream);
}

size_t mi_gemm_workspace_bytes(int config, int dtype, int M, int N, int K, int c_layout) {
    if (dtype != MI_DTYPE_BF16 && dtype != MI_DTYPE_FP16) return 0;
    if (!shape_in_range(M, N, K)) return 0;
    if (config != MI_CONFIG_AUTO && (config < 0 || config >= mi::kNumKernels)) return 0;
    if (c_layout == MI_C_COL_MAJOR) {
        const int t = M;
        M = N;
        N = t;
    }
    // The choice also depends on the alignment of the pointers, unknown here: the largest
    // need over the cases a launch can meet -- and over the two parts, where the automatic
    // choice may cut the shape's rows in two.
    auto uncut = [&](int rows) {
        size_t need = 0;
        const bool can_stream = N % 4 == 0 && K % 64 == 0;
        for (int aligned = 0; aligned < 2; ++aligned)
            for (int streamable = 0; streamable < (can_stream && aligned ? 2 : 1); ++streamable)
                // (a launch that cannot use the small-tile kernels -- operands not 4-byte aligned --
                // may split where one that can does not: both cases)
                for (int small = 0; small < 2; ++small) {
                    const Choice c = compute_choice(config, rows, N, K, streamable != 0, N % 4 == 0, aligned != 0, small != 0);
                    const size_t b = choice_workspace(c, rows, N, K);
                    if (b > need) need = b;
                }
        return need;
    };
    size_t need = uncut(M);
    if (config == MI_CONFIG_AUTO && tuned_config(M, N, K, N % 4 == 0 && K % 64 == 0, true, true) < 0)
        for (int flags = 0; flags < 16; ++flags) {
            const int m1 = rows_to_cut(M, N, K, (flags & 1) != 0 && N % 4 == 0 && K % 64 == 0, (flags & 2) != 0 && N % 4 == 0,
                                       (flags & 4) != 0, (flags & 8) != 0);
            if (m1 > 0) {
                const size_t a = uncut(m1), b = uncut(M - m1);
                if (a > need) need = a;
                if (b > need) need = b;
            }
        }
    return need;
}

int mi_gemm_epilogue_ws(int config, int dtype, int M, int N, int K, const void* A, const void* B, void* C,
                        float alpha, float beta, int c_layout, void* ws, size_t ws_bytes, void* stream) {
    if (c_layout != MI_C_ROW_MAJOR && c_layout != MI_C_COL_MAJOR)
        return fail(MI_ERR_INVALID, "unknown C layout %d", c_layout);
    if (!(alpha == alpha) || !(beta == beta)) return fail(MI_ERR_INVALID, "alpha or beta is NaN");
    if (ws && !aligned16(ws)) return fail(MI_ERR_INVALID, "the workspace must be 16-byte aligned");
    WsSource src;
    src.mode = WS_CALLER;
    src.ptr = ws;
    src.bytes = ws ? ws_bytes : 0;
    if (c_layout == MI_C_COL_MAJOR)
        return run_gemm(config, dtype, N, M, K, B, A, C, nullptr, alpha, beta, stream, src);
    return run_gemm(config, dtype, M, N, K, A, B, C, nullptr, alpha, beta, stream, src);
}

int mi_gemm_bf16_noalloc(int M, int N, int K, const uint16_t* A, const uint16_t* B, uint16_t* C, void* stream) {
    WsSource src;
    src.mode = WS_STATIC;
    return run_gemm(MI_CONFIG_AUTO, MI_DTYPE_BF16, M, N, K, A, B, C, nullptr, 1.0f, 0.0f, stream, src);
}

int mi_gemm_reserve_workspace(void* stream, size_t bytes) {
    if (bytes == 0) return MI_OK;
    float* p = nullptr;
    WsHold hold;
    const int rc = acquire_workspace(WsSource{}, bytes, (hipStream_t)stream, hold, &p);
    if (rc > 0) return fail(MI_ERR_UNSUPPORTED, "the stream is being captured: no workspace can be allocated now");
    return rc < 0 ? rc : MI_OK;
}

int mi_gemm_release_workspace(void* stream) {
    // NULL: every stream's buffers on the current device, once the device is idle
    auto wait_for_work = [&] { return stream ? hipStreamSynchronize((hipStream_t)stream) : hipDeviceSynchronize(); };
    MI_HIP(wait_for_work());
    // a call that is between two launches makes the rest of them before its buffer goes: what it
    // launched is waited for again, with no further call able to take a buffer
    std::unique_lock<std::mutex> lock(g_ws_mutex);
    DeviceState& st = device_state();
    auto concerned = [&](const StreamWs& w) { return stream == nullptr || w.key == key_of((hipStream_t)stream); };
    g_ws_idle.wait(lock, [&] {
        for (const auto& w : st.ws)
            if (concerned(*w) && w->calls > 0) return false;
        return true;
    });
    MI_HIP(wait_for_work());
    for (size_t i = 0; i < st.ws.size();) {
        if (concerned(*st.ws[i])) {
            free_entry(*st.ws[i]);
            st.ws.erase(st.ws.begin() + (long)i);
        } else {
            ++i;
        }
    }
    return MI_OK;
}

size_t mi_gemm_library_workspace_bytes(void) {
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    size_t total = 0;
    for (const auto& w : device_state().ws) total += w->bytes;
    return total;
}

int mi_reference_gpu_gemm(int dtype, int M, int N, int K, const void* A, const void* B, void* C,
                          float alpha, float beta, void* stream) {
    int rc = check_args(MI_CONFIG_AUTO, dtype, M, N, K, A, B, C);
    if (rc != MI_OK) return rc;
    hipError_t err =
        mi::launch_reference_gpu_gemm(dtype, M, N, K, A, B, C, alpha, beta, compute_units(), (hipStream_t)stream);
    if (err != hipSuccess)
        return fail(MI_ERR_HIP, "launch of the reference GEMM failed: %s", hipGetErrorString(err));
    return MI_OK;
}

// ---- thin HIP layer -------------------------------------------------------------------

int mi_malloc(void** dptr, size_t bytes) {
    if (!dptr) return fail(MI_ERR_INVALID, "mi_malloc: null out pointer");
    MI_HIP(hipMalloc(dptr, bytes));
    return MI_OK;
}
int mi_free(void* dptr) {
    MI_HIP(hipFree(dptr));
    return MI_OK;
}
int mi_memcpy_h2d(void* dst, const void* src, size_t bytes) {
    MI_HIP(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return MI_OK;
}
int mi_memcpy_d2h(void* dst, const void* src, size_t bytes) {
    MI_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return MI_OK;
}
int mi_memcpy_d2d(void* dst, const void* src, size_t bytes) {
    MI_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToDevice));
    return MI_OK;
}
int mi_memset(void* dst, int value, size_t bytes) {
    MI_HIP(hipMemset(dst, value, bytes));
    return MI_OK;
}
int mi_device_sync(void) {
    MI_HIP(hipDeviceSynchronize());
    return MI_OK;
}
int mi_stream_sync(void* stream) {
    MI_HIP(hipStreamSynchronize((hipStream_t)stream));
    return MI_OK;
}
int mi_event_create(void** ev) {
    if (!ev) return fail(MI_ERR_INVALID, "mi_event_create: null out pointer");
    hipEvent_t e;
    MI_HIP(hipEventCreate(&e));
    *ev = (void*)e;
    return MI_OK;
}
int mi_event_destroy(void* ev) {
    MI_HIP(hipEventDestroy((hipEvent_t)ev));
    return MI_OK;
}
int mi_event_record(void* ev, void* stream) {
    MI_HIP(hipEventRecord((hipEvent_t)ev, (hipStream_t)stream));
    return MI_OK;
}
int mi_event_sync(void* ev) {
    MI_HIP(hipEventSynchronize((hipEvent_t)ev));
    return MI_OK;
}
int mi_event_elapsed_ms(float* ms, void* start, void* stop) {
    if (!ms) return fail(MI_ERR_INVALID, "mi_event_elapsed_ms: null out pointer");
    MI_HIP(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop));
    return MI_OK;
}

int mi_get_device_props(mi_device_props* out) {
    if (!out) return fail(MI_ERR_INVALID, "mi_get_device_props: null out pointer");
    int dev = 0;
    MI_HIP(hipGetDevice(&dev));
    hipDeviceProp_t p;
    MI_HIP(hipGetDeviceProperties(&p, dev));
    memset(out, 0, sizeof *out);
    snprintf(out->name, sizeof out->name, "%s", p.name);
    snprintf(out->arch, sizeof out->arch, "%s", p.gcnArchName);
    out->compute_units = p.multiProcessorCount;
    out->clock_khz = p.clockRate;
    out->mem_clock_khz = p.memoryClockRate;
    out->mem_bus_bits = p.memoryBusWidth;
    out->lds_bytes_per_block = (int)p.sharedMemPerBlock;
    out->l2_bytes = p.l2CacheSize;
    out->wavefront = p.warpSize;
    out->hbm_bytes = p.totalGlobalMem;
    return MI_OK;
}

}  // extern "C"
