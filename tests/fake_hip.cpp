// The library's host code over a pretended HIP runtime: this program defines
// the runtime functions that liborc_hip.so calls, so its streams, events,
// captures and launches are only written down. One scenario per run (argv[1]);
// exit status 1 and a line on stderr for the first thing that is wrong.
// Launches are printed as "<stream> <captured 0/1> <grid> <kernel>".
#define __HIP_PLATFORM_AMD__ 1
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "../include/orc.h"

struct Stream {
    std::string name;
    bool capturing = false, joined = false;  // joined: pulled into another stream's capture
    int uses = 0;                            // launches so far
};
struct Event {
    Stream* on = nullptr;
    bool captured = false;
    int uses = 0;  // launches of `on` it follows
};
struct Wait {
    Stream* s;
    Event e;
};
static std::recursive_mutex mu;
static std::vector<Wait> waits;
static std::vector<std::string> launches;
static hipError_t last_error = hipSuccess;
static size_t malloc_limit = ~(size_t)0;
static std::function<void(Stream*)> on_query;  // called after the answer of hipStreamIsCapturing is settled
static thread_local dim3 cfg_g, cfg_b;
static thread_local size_t cfg_l;
static thread_local hipStream_t cfg_s;

static std::vector<hipStream_t> held;  // made beforehand
static void hold_streams(hipStream_t* s, int n) { held.assign(s, s + n); }

static Stream* S(hipStream_t s) { return (Stream*)s; }
#define LOCK std::lock_guard<std::recursive_mutex> lk(mu)

// operator new of the library too: fails while asked to
static std::atomic<bool> no_new{false};
void* operator new(size_t n) {
    if (no_new) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

struct MayNew {  // this program's own notes
    bool was = no_new.exchange(false);
    ~MayNew() { no_new = was; }
};

static hipError_t launch(const void* f, dim3 g, hipStream_t s) {
    LOCK;
    MayNew may;
    Dl_info info{};
    const char* n = dladdr(f, &info) && info.dli_sname ? info.dli_sname : "?";
    char line[600];
    std::snprintf(line, sizeof line, "%s %d %ux%ux%u %s", S(s)->name.c_str(), S(s)->capturing || S(s)->joined, g.x, g.y, g.z, n);
    launches.push_back(line);
    ++S(s)->uses;
    return hipSuccess;
}

extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) {
    cfg_g = g, cfg_b = b, cfg_l = l, cfg_s = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* l, hipStream_t* s) {
    *g = cfg_g, *b = cfg_b, *l = cfg_l, *s = cfg_s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3, void**, size_t, hipStream_t s) { return launch(f, g, s); }
hipError_t hipExtLaunchKernel(const void* f, dim3 g, dim3, void**, size_t, hipStream_t s, hipEvent_t, hipEvent_t, int) {
    return launch(f, g, s);
}
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 160 * 1024 : 0;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    return last_error = hipSuccess, e;
}
const char* hipGetErrorString(hipError_t) { return "pretended error"; }
hipError_t hipGetSymbolAddress(void** p, const void*) { return *p = (void*)0x1000, hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
    if (n > malloc_limit) return last_error = hipErrorOutOfMemory;
    return *p = std::malloc(16), hipSuccess;
}
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    static int n;
    if (!held.empty()) return *s = held.back(), held.pop_back(), hipSuccess;
    return *s = (hipStream_t) new Stream{std::string(1, "0ABCDEFG"[n++ % 8])}, hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return delete S(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    {
        LOCK;
        *st = S(s)->capturing || S(s)->joined ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    }
    if (on_query) on_query(S(s));
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    LOCK;
    if (S(s)->capturing) return hipErrorIllegalState;
    return S(s)->capturing = true, hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
    LOCK;
    return S(s)->capturing = false, *g = nullptr, hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { return *e = nullptr, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = (hipEvent_t) new Event, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return delete (Event*)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    LOCK;
    return *(Event*)e = Event{S(s), S(s)->capturing, S(s)->uses}, hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    LOCK;
    waits.push_back({S(s), *(Event*)e});
    if (((Event*)e)->captured) S(s)->joined = true;
    return hipSuccess;
}
}

#define CHECK(c)                                                     \
    do {                                                             \
        if (!(c)) {                                                  \
            std::fprintf(stderr, "line %d: %s\n", __LINE__, #c);     \
            std::exit(1);                                            \
        }                                                            \
    } while (0)

static float* const X = (float*)0x10000000;  // never read: nothing runs
static int gemm(int type, int n_tok, int n_out, int n_in, orc_stream_t s) {
    return orc_gemm(type, X, n_tok, n_out, n_in, X, n_in, X, n_out, s);
}

// Two library streams; the first has used the workspace. Another thread begins
// a capture of it while a call on the second takes the workspace over.
static void capture_race(bool through_library) {
    orc_stream_t a, b;
    CHECK(!orc_init(0) && !orc_stream_create(&a) && !orc_stream_create(&b));
    CHECK(!gemm(ORC_F16, 300, 2048, 2048, a));
    std::thread t;
    std::atomic<bool> begun{false}, armed{true};
    on_query = [&](Stream* s) {
        if (s != S((hipStream_t)a) || !armed.exchange(false)) return;
        t = std::thread([&] {
            CHECK(!(through_library ? orc_graph_begin(a) : (int)hipStreamBeginCapture((hipStream_t)a, hipStreamCaptureModeThreadLocal)));
            begun = true;
        });
        for (int i = 0; i < 30 && !begun; ++i) std::this_thread::sleep_for(std::chrono::milliseconds(10));
    };
    const size_t n0 = launches.size();
    CHECK(!gemm(ORC_F16, 300, 2048, 2048, b));
    armed = false;
    if (t.joinable()) t.join();
    else CHECK(!orc_graph_begin(a));  // the library asked nothing about the stream
    CHECK(launches.size() > n0);
    for (size_t i = n0; i < launches.size(); ++i) CHECK(launches[i].substr(0, 3) == S((hipStream_t)b)->name + " 0");
    CHECK(!S((hipStream_t)b)->joined);
    orc_graph_t g;
    CHECK(!orc_graph_end(a, &g));
    CHECK(!gemm(ORC_F16, 300, 2048, 2048, a));
    // the call on b had the workspace, or (a capture the library does not know of) went without
    CHECK(!through_library || waits.size());
    if (waits.size()) CHECK(waits.back().s == S((hipStream_t)a) && waits.back().e.on == S((hipStream_t)b));
}

// A use followed by a capture of the same stream is still waited for, and a
// call on another stream during the capture takes the kernels it takes at any
// other time.
static void capture_order() {
    orc_stream_t a, b;
    CHECK(!orc_init(0) && !orc_stream_create(&a) && !orc_stream_create(&b));
    CHECK(!gemm(ORC_F16, 300, 2048, 2048, a));
    const size_t per = launches.size();
    const int used = S((hipStream_t)a)->uses;
    CHECK(!orc_graph_begin(a) && !gemm(ORC_F16, 300, 2048, 2048, a));
    const size_t n0 = launches.size();
    CHECK(!gemm(ORC_F16, 300, 2048, 2048, b));
    CHECK(launches.size() == n0 + per);
    for (size_t i = 0; i < per; ++i) CHECK(launches[n0 + i].substr(2) == launches[i].substr(2));
    CHECK(waits.size() == 1 && waits[0].s == S((hipStream_t)b) && waits[0].e.on == S((hipStream_t)a) && !waits[0].e.captured && waits[0].e.uses >= used);
    orc_graph_t g;
    CHECK(!orc_graph_end(a, &g) && !orc_stream_destroy(a) && !orc_stream_destroy(b));
}

// A device without the memory for the workspace: orc_init and every call work, on the
// kernels that need no workspace.
static void no_memory() {
    malloc_limit = 100 << 20;
    CHECK(!orc_init(0));
    for (int type : {ORC_Q4_K, ORC_Q8_0, ORC_F16}) CHECK(!gemm(type, 300, 2048, 2048, nullptr));
    const int H = 8, KV = 2, hd = 64, ld = (H + 2 * KV) * hd;
    CHECK(!orc_attn_prefill(X, ld, 70, H, KV, hd, 50, X, X, X, 128, X, H * hd, nullptr));
    CHECK(launches.size() >= 4);
    for (const std::string& l : launches) CHECK(l.find("k_pf") == l.npos && l.find("k_kv_split") == l.npos);
}

// gemm type n_tok n_out n_in | attn heads kv head_dim n_tok pos: the call's launches
static void route(int argc, char** argv) {
    CHECK(argc == 6 + (argv[1][0] == 'a'));
    int v[5];
    for (int i = 2; i < argc; ++i) v[i - 2] = std::atoi(argv[i]);
    CHECK(!orc_init(0));
    if (argv[1][0] == 'g') CHECK(!gemm(v[0], v[1], v[2], v[3], nullptr));
    else
        CHECK(!orc_attn_prefill(X, (v[0] + 2 * v[1]) * v[2], v[3], v[0], v[1], v[2], v[4], X, X, X, v[4] + v[3], X, v[0] * v[2], nullptr));
}

// The bytes noted for timed attention calls: K and V once, QKV rows in, rows
// out, over the workspace; k_attn_pf reads K and V once per 16-token block.
static void prof_bytes() {
    const int H = 28, KV = 4, hd = 128, n = 1023, pos = 7168, ld = (H + 2 * KV) * hd;
    CHECK(!orc_init(0));
    auto bytes = [&] {
        int64_t calls = 0;
        double ms = 0, by = 0;
        orc_prof_enable(1);
        CHECK(!orc_attn_prefill(X, ld, n, H, KV, hd, pos, X, X, X, pos + n, X, H * hd, nullptr));
        CHECK(!orc_prof_accumulate() && !orc_prof_read(ORC_PROF_ATTN_PF, n, &calls, &ms, &by) && calls == 1);
        orc_prof_enable(0);
        return by;
    };
    const double rows = 4.0 * n * (ld + H * hd), kv = 8.0 * KV * hd;
    CHECK(bytes() == kv * (pos + n) + rows);
    double all = 0;
    for (int t = 0; t < n; t += 16) all += kv * (pos + (t + 16 < n ? t + 16 : n));
    CHECK(!orc_shutdown());
    malloc_limit = 100 << 20;
    CHECK(!orc_init(0) && bytes() == all + rows);
}

// No exception leaves a C entry point where the host's memory runs out: the
// library's own notes of streams and sampler states are left out.
static void no_host_memory() {
    CHECK(!orc_init(0));
    hipStream_t pre[3];
    for (hipStream_t& s : pre) hipStreamCreateWithFlags(&s, 0);
    hold_streams(pre, 3);
    no_new = true;
    orc_stream_t a = nullptr;
    const int rc = orc_stream_create(&a), rs = orc_sampler_init(X, 0.f, 1.f, 0, 1.f, 0, 1, nullptr, 0, a);
    no_new = false;
    CHECK(!rc && a && !rs);
    CHECK(!gemm(ORC_F16, 300, 2048, 2048, a) && !gemm(ORC_F16, 300, 2048, 2048, nullptr));  // an event after every use
    CHECK(waits.size() == 1 && waits[0].e.on == S((hipStream_t)a));
    CHECK(!orc_sample(X, X, 1000, (int32_t*)X, a) && !orc_stream_destroy(a));
}

int main(int argc, char** argv) {
    CHECK(argc > 1);
    const std::string w = argv[1];
    if (w == "race") capture_race(true);
    else if (w == "race_hip") capture_race(false);
    else if (w == "order") capture_order();
    else if (w == "no_memory") no_memory();
    else if (w == "prof_bytes") prof_bytes();
    else if (w == "no_host_memory") no_host_memory();
    else if (w == "gemm" || w == "attn") route(argc, argv);
    else CHECK(!"a scenario");
    for (const std::string& l : launches) std::puts(l.c_str());
    return 0;
}
