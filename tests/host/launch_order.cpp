// The library's host side on a machine without a GPU: this program defines the HIP calls that
// libmi_gemm.so makes (its symbols come before libamdhip64's), so "launching" a kernel runs a few lines
// here.  They follow whose operands a workspace holds: a copy or a GEMM that writes one marks it, the
// GEMM or reduction that reads it passes the mark on to C.  Addresses are made up and never
// dereferenced; the top byte names the call they belong to.  Launches with a trace buffer say how many
// of its records they write.
//
//   launch_order <scenario>         exit code 0, or 1 with the fault on stderr
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "../../include/mi_gemm.h"

namespace {

struct Dim3 { uint32_t x, y, z; };
constexpr uint64_t kWorkspace = 0x70ull << 40, kCaller = 0x71ull << 40, kStatic = 0x72ull << 40;
constexpr int kErrorMemory = 2;

std::mutex m;                                      // of everything below
// host stub -> device name; filled by the library's constructors, ahead of this program's own
std::map<const void*, std::string>& kernels() {
    static auto* k = new std::map<const void*, std::string>;
    return *k;
}
std::map<uint64_t, size_t> allocations;            // live ones
std::map<uint64_t, uint64_t> owner;                // workspace base -> call whose data it holds
std::map<uint64_t, uint64_t> result;               // C -> call whose product it holds
std::map<std::thread::id, std::set<uint64_t>> used;   // workspaces each thread's launches named
std::vector<uint64_t> copies;                      // where operands were copied to
std::vector<std::string> faults;
struct Traced { uint64_t buffer; size_t records; };
std::vector<Traced> traced;                        // launches with a trace buffer: a record per workgroup
uint64_t next_address = kWorkspace;
int allocation_calls = 0, fail_above_mib = 0;      // hipMalloc of more than that fails (0: never)
bool capturing = false;
std::function<void(const std::string&)> after_launch;  // called without the lock

void fault(const std::string& s) { faults.push_back(s); }

// the workspace `p` lies in, or 0
uint64_t base_of(uint64_t p) {
    if (p >> 40 == kCaller >> 40) return p & ~0xffffffffull;
    if (p >> 40 == kStatic >> 40) return kStatic;
    if (p >> 40 != kWorkspace >> 40) return 0;
    auto it = allocations.upper_bound(p);
    if (it == allocations.begin() || p >= (--it)->first + it->second) {
        fault("a launch names a workspace that has been freed");
        return 0;
    }
    return it->first;
}
// the call an operand comes from
uint64_t source_of(uint64_t p) {
    if (p >> 40 < kWorkspace >> 40) return p >> 40;
    const uint64_t b = base_of(p);
    return b ? owner[b] : 0;
}

int launch(const void* stub, Dim3 grid, void** args) {
    std::string name;
    {
        std::lock_guard<std::mutex> lock(m);
        name = kernels()[stub];
        uint64_t w[10];
        memcpy(w, args[0], 24);
        auto use = [&](uint64_t p) {
            const uint64_t b = base_of(p);
            if (b) used[std::this_thread::get_id()].insert(b);
            return b;
        };
        if (name.find("pack_operands_kernel") != std::string::npos) {        // {src[2], out, ...}
            owner[use(w[2])] = source_of(w[0]);
            copies.push_back(w[2]);
        } else if (name.find("splitk_reduce_kernel") != std::string::npos) { // (ws, C, ...)
            uint64_t ws, c;
            memcpy(&ws, args[0], 8);
            memcpy(&c, args[1], 8);
            result[c] = owner[use(ws)];
        } else {                                                             // {A, B, C, ...}
            const bool decode = name.find("DecodeArgs") != std::string::npos;    // (else GemmArgs: the workspace further on)
            memcpy(w, args[0], 80);
            if (const uint64_t db = decode ? w[9] : w[8]) traced.push_back({db, (size_t)grid.x * grid.y * grid.z});
            const uint64_t ws = decode ? w[3] : w[9], src = source_of(w[0]);
            if (src != source_of(w[1])) fault("A and B of different calls are multiplied");
            for (int i = 0; i < 2; ++i)
                if (w[i] >> 40 >= kWorkspace >> 40) use(w[i]);
            if (ws) owner[use(ws)] = src;
            else result[w[2]] = src;
        }
    }
    if (after_launch) after_launch(name);
    return 0;
}

}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* stub, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    std::lock_guard<std::mutex> lock(m);
    kernels()[stub] = name;
}
int hipLaunchKernel(const void* stub, Dim3 grid, Dim3, void** args, size_t, void*) { return launch(stub, grid, args); }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipGetSymbolAddress(void** p, const void*) { *p = (void*)kStatic; return 0; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "stub"; }
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamIsCapturing(void*, int* s) { *s = capturing ? 1 : 0; return 0; }
int hipThreadExchangeStreamCaptureMode(int*) { return 0; }
int hipMalloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> lock(m);
    ++allocation_calls;
    if (fail_above_mib && bytes > (size_t)fail_above_mib << 20) return kErrorMemory;
    next_address = (next_address + 0xffffffull) & ~0xffffffull;
    *p = (void*)next_address;
    allocations[next_address] = bytes;
    next_address += bytes;
    return 0;
}
int hipFree(void* p) {
    std::lock_guard<std::mutex> lock(m);
    if (!allocations.erase((uint64_t)p)) fault("hipFree of an address that is not allocated");
    return 0;
}
}

namespace {

struct Shape { int M, N, K; };
const Shape kCopied = {4095, 6143, 3073}, kSmallCopy = {2560, 3072, 2568};    // copy + GEMM
const Shape kMultiLaunch[] = {kCopied, {2100, 2100, 9001}, {128, 8192, 8192}, {800, 800, 6000}};   // + pieces of K, split-K

const void* A_of(uint64_t call) { return (const void*)(call << 40 | 0x1000); }
const void* B_of(uint64_t call) { return (const void*)(call << 40 | 1ull << 32); }
void* C_of(uint64_t call) { return (void*)(call << 40 | 2ull << 32); }

enum Entry { LIBRARY, CALLER, STATIC };
int call(Entry entry, const Shape& s, uint64_t id, void* stream) {
    const uint16_t *a = (const uint16_t*)A_of(id), *b = (const uint16_t*)B_of(id);
    uint16_t* c = (uint16_t*)C_of(id);
    if (entry == LIBRARY) return mi_gemm_bf16(s.M, s.N, s.K, a, b, c, nullptr, stream);
    if (entry == STATIC) return mi_gemm_bf16_noalloc(s.M, s.N, s.K, a, b, c, stream);
    return mi_gemm_epilogue_ws(-1, 0, s.M, s.N, s.K, a, b, c, 1.0f, 0.0f, 0, (void*)(kCaller + 16), (size_t)3 << 30, stream);
}
void expect(bool ok, const std::string& what) {
    std::lock_guard<std::mutex> lock(m);
    if (!ok) fault(what);
}
void expect_product(const Shape& s, uint64_t id, int rc) {
    char text[160];
    std::lock_guard<std::mutex> lock(m);
    const uint64_t got = result[(uint64_t)C_of(id)];
    snprintf(text, sizeof text, "%d x %d x %d: call %d (status %d) got the product of call %d's operands", s.M, s.N, s.K, (int)id, rc, (int)got);
    if (rc != 0 || got != id) fault(text);
    result.erase((uint64_t)C_of(id));
}
void pause_us(int us) { std::this_thread::sleep_for(std::chrono::microseconds(us)); }

// Two threads on one stream and one buffer: each call's launches follow each other.
void one_stream(Entry entry) {
    after_launch = [](const std::string&) { pause_us(30); };
    for (const Shape& s : kMultiLaunch) {
        if (entry == STATIC && s.N == 2100) continue;              // (its sums do not fit the static array)
        std::vector<std::thread> threads;
        for (uint64_t id = 1; id <= 3; ++id)
            threads.emplace_back([&, id] {
                for (int i = 0; i < 60; ++i) {
                    const int rc = call(entry, s, id, nullptr);
                    expect_product(s, id, rc);
                }
            });
        for (auto& t : threads) t.join();
    }
    // and with calls of different shapes, a copy, sums of pieces or both
    if (entry == STATIC) return;
    std::vector<std::thread> threads;
    for (uint64_t id = 1; id <= 3; ++id)
        threads.emplace_back([&, id] {
            for (uint64_t i = 0; i < 120; ++i) {
                const Shape& s = kMultiLaunch[(i * id + id) % 4];
                const int rc = call(entry, s, id, nullptr);
                expect_product(s, id, rc);
            }
        });
    for (auto& t : threads) t.join();
}

// hipStreamPerThread is one handle for as many streams as there are threads: no buffer in common.
void per_thread_stream() {
    void* const per_thread = (void*)2;
    std::map<std::thread::id, std::set<uint64_t>> by_thread;
    for (const Shape& s : kMultiLaunch) {
        std::vector<std::thread> threads;
        std::atomic<int> arrived{0};
        for (uint64_t id = 1; id <= 3; ++id)
            threads.emplace_back([&, id] {
                expect_product(s, id, call(LIBRARY, s, id, per_thread));
                ++arrived;
                while (arrived < 3) std::this_thread::yield();     // (thread ids are not reused before all have run)
            });
        for (auto& t : threads) t.join();
        std::set<uint64_t> seen;
        for (const auto& t : used)
            for (uint64_t b : t.second) expect(seen.insert(b).second, "two threads' streams share a workspace");
        expect(!seen.empty(), "no launch used a workspace");
        used.clear();
        expect(mi_gemm_release_workspace(nullptr) == 0, "release failed");
    }
}

// While one call is between its copy and its GEMM, `other` runs on another thread; the call's buffer
// neither changes hands nor is freed.
void interrupted(const std::function<void()>& other) {
    for (uint64_t s = 0; s < 16; ++s) expect_product(kSmallCopy, 1, call(LIBRARY, kSmallCopy, 1, (void*)(0x100 + s)));
    std::thread second;
    std::atomic<bool> started{false};
    after_launch = [&](const std::string& name) {
        if (name.find("pack_operands_kernel") == std::string::npos || started.exchange(true)) return;
        second = std::thread(other);
        pause_us(100000);
    };
    expect_product(kSmallCopy, 1, call(LIBRARY, kSmallCopy, 1, (void*)0x100));
    second.join();
    expect(started, "the call made no copy");
}

// Every entry's stream is between two launches: a further stream waits for one of them.
void table_busy() {
    const Shape split = {128, 8192, 8192};
    std::atomic<int> between{0};
    std::atomic<bool> go{false}, waited{false};
    after_launch = [&](const std::string& name) {
        if (name.find("pack_operands_kernel") == std::string::npos) return;
        ++between;
        for (int i = 0; i < 2000 && !go; ++i) pause_us(1000);
    };
    std::vector<std::thread> threads;
    for (uint64_t id = 1; id <= 16; ++id)
        threads.emplace_back([&, id] { expect_product(kSmallCopy, id, call(LIBRARY, kSmallCopy, id, (void*)(0x100 + id))); });
    for (int i = 0; i < 2000 && between < 16; ++i) pause_us(1000);
    expect(between == 16, "sixteen calls on streams of their own hold each other up");
    threads.emplace_back([&] {
        const int rc = call(LIBRARY, split, 17, (void*)0x200);
        waited = go.load();
        expect_product(split, 17, rc);
    });
    pause_us(50000);
    go = true;
    for (auto& t : threads) t.join();
    expect(waited, "a buffer changed hands while its call had launches to make");
}

// A caller's workspace on any 16-byte boundary: the copy's rows start on a 128-byte line inside it, and
// the copy is made when it fits behind that.
void caller_alignment() {
    const Shape& s = kCopied;
    const size_t need = mi_gemm_workspace_bytes(-1, 0, s.M, s.N, s.K, 0);
    for (int offset = 0; offset < 256; offset += 16)
        for (int spare : {0, 112}) {
            copies.clear();
            const uint64_t ws = kCaller + (uint64_t)offset;
            const int rc = mi_gemm_epilogue_ws(-1, 0, s.M, s.N, s.K, A_of(1), B_of(1), C_of(1), 1.0f, 0.0f, 0, (void*)ws, need + spare, nullptr);
            expect_product(s, 1, rc);
            const uint64_t first = (ws + 127) / 128 * 128;
            if (first + need > ws + need + spare) expect(copies.empty(), "a copy that does not fit the caller's workspace");
            else expect(copies.size() == 1 && copies[0] == first, "no copy on the first 128-byte line of the caller's workspace");
        }
}

// What the library allocates of its own accord, for copies, is bounded, and an allocation that failed is
// not asked for again on every call (nor is it given up for good).
void copy_memory() {
    const Shape large = {8191, 8191, 28673}, split = {128, 8192, 8192};      // 0.94 GB copied
    for (uint64_t i = 0; i < 16; ++i) expect_product(large, 1, call(LIBRARY, large, 1, (void*)(0x100 + i)));
    expect(mi_gemm_library_workspace_bytes() == (size_t)8 << 30, "more or less than 8 GiB held for copies");
    expect_product(split, 1, call(LIBRARY, split, 1, (void*)0x200));          // sums of pieces are not optional
    expect(mi_gemm_library_workspace_bytes() == ((size_t)8 << 30) + ((size_t)16 << 20), "no workspace for the pieces' sums");
    expect(mi_gemm_release_workspace(nullptr) == 0 && mi_gemm_library_workspace_bytes() == 0, "release failed");

    fail_above_mib = 512;
    allocation_calls = 0;
    const auto start = std::chrono::steady_clock::now();
    for (int i = 0; i < 200; ++i) expect_product(large, 1, call(LIBRARY, large, 1, (void*)0x100));
    const int seconds = (int)std::chrono::duration_cast<std::chrono::seconds>(std::chrono::steady_clock::now() - start).count();
    expect(allocation_calls >= 1 && allocation_calls <= 2 + seconds, "an allocation that fails is tried on every call");
    expect_product(kCopied, 1, call(LIBRARY, kCopied, 1, (void*)0x100));      // a smaller one that there is room for
    expect(mi_gemm_library_workspace_bytes() == (size_t)64 << 20, "no smaller copy after a larger one failed");
    fail_above_mib = 0;
    copies.clear();
    pause_us(1100000);
    expect_product(large, 1, call(LIBRARY, large, 1, (void*)0x100));
    expect(copies.size() == 1, "no copy once there is memory again");
}

// A trace buffer of mi_gemm_trace_words has room for every call of the shape: each configuration and the
// automatic choice, operands and C on every boundary that changes which kernel runs, in how many pieces.
void trace_room() {
    std::vector<Shape> shapes = {{824, 68, 27976}, {825, 72, 19456}, {160, 1280, 11832}, {232, 432, 10952}, {23, 7208, 13488},
                                 {11, 7296, 13376}, {1000, 780, 64}, {1000, 780, 72}, {513, 257, 136}, {7000, 7000, 4096}};
    uint64_t seed = 1;
    auto draw = [&](double lo, double hi, int step) {
        seed = seed * 6364136223846793005ull + 1442695040888963407ull;
        return std::max(step, (int)(lo * pow(hi / lo, (double)(seed >> 11) / 9007199254740992.0)) / step * step);
    };
    for (int i = 0; i < 400; ++i) {
        const int step = i % 4 == 0 ? 1 : i % 4 == 1 ? 64 : 8;
        shapes.push_back({draw(1, 4096, i % 3 ? 1 : step), draw(64, 8192, step == 1 ? 1 : 4), draw(64, 30000, step)});
    }
    const uint64_t db = 5ull << 40;
    for (const Shape& s : shapes) {
        const size_t room = (mi_gemm_trace_words(s.M, s.N, s.K) - 1) / 6;
        for (int config = -1; config < mi_gemm_num_configs(); ++config)
            for (uint64_t a : {0, 4, 2})
                for (uint64_t c : {0, 8, 2}) {
                    traced.clear();
                    mi_gemm_ex(config, 0, s.M, s.N, s.K, (const char*)A_of(1) + a, B_of(1), (char*)C_of(1) + c, (int*)db, nullptr);
                    size_t end = 0;
                    for (const Traced& t : traced) end = std::max(end, (size_t)(t.buffer - db) / 24 + t.records);
                    char text[200];
                    snprintf(text, sizeof text, "%d x %d x %d on %s, A at +%d, C at +%d: %zu records, room for %zu", s.M, s.N, s.K,
                             config < 0 ? "auto" : mi_gemm_config_name(config), (int)a, (int)c, end, room);
                    expect(end <= room, text);
                    // config_grid: what a call with everything on 16-byte boundaries launches
                    if (config >= 0 && a + c == 0 && !traced.empty()) {
                        snprintf(text, sizeof text, "%d x %d x %d on %s: %zu workgroups, config_grid %d", s.M, s.N, s.K,
                                 mi_gemm_config_name(config), end, mi_gemm_config_grid(config, s.M, s.N, s.K));
                        expect(end == (size_t)mi_gemm_config_grid(config, s.M, s.N, s.K), text);
                    }
                }
    }
}

// Every config's kernel for a call on 16-byte boundaries and for one whose A is 4 bytes off: a line each for the test to read
void which_kernel() {
    std::string kernel;
    after_launch = [&](const std::string& name) { kernel = name; };
    for (int config = 0; config < mi_gemm_num_configs(); ++config)
        for (uint64_t a : {0, 4}) {
            kernel = "-";
            mi_gemm_ex(config, 0, 16, 256, 512, (const char*)A_of(1) + a, B_of(1), C_of(1), nullptr, nullptr);
            printf("%s %d %s\n", mi_gemm_config_name(config), (int)a, kernel.c_str());
        }
}

}  // namespace

int main(int argc, char** argv) {
    const std::string scenario = argc > 1 ? argv[1] : "";
    if (scenario == "one_stream_library") one_stream(LIBRARY);
    else if (scenario == "one_stream_caller") one_stream(CALLER);
    else if (scenario == "one_stream_static") one_stream(STATIC);
    else if (scenario == "per_thread_stream") per_thread_stream();
    else if (scenario == "takeover" || scenario == "takeover_larger") {        // a buffer as it is, one that is too small
        const Shape split = scenario == "takeover" ? Shape{128, 8192, 8192} : Shape{2100, 2100, 9001};
        interrupted([&] { expect_product(split, 2, call(LIBRARY, split, 2, (void*)0x200)); });
    } else if (scenario == "release_all") interrupted([] { expect(mi_gemm_release_workspace(nullptr) == 0, "release failed"); });
    else if (scenario == "release_one") interrupted([] { expect(mi_gemm_release_workspace((void*)0x100) == 0, "release failed"); });
    else if (scenario == "table_busy") table_busy();
    else if (scenario == "caller_alignment") caller_alignment();
    else if (scenario == "copy_memory") copy_memory();
    else if (scenario == "trace_room") trace_room();
    else if (scenario == "which_kernel") which_kernel();
    else return 2;
    for (const std::string& f : std::set<std::string>(faults.begin(), faults.end())) fprintf(stderr, "%s\n", f.c_str());
    return faults.empty() ? 0 : 1;
}
