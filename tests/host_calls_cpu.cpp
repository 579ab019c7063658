// The host layer's large blocking calls over a device made of host memory: the shim below does at once, on the calling
// thread, what the HIP side enqueues.  One check per run, named by the argument; ends with 0 or says what is wrong.
#include <dlfcn.h>
#include <pthread.h>
#include <sched.h>
#include <unistd.h>

#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <new>
#include <vector>

#include "rk_hip_shim.h"
#include "rk_npu_hip.h"

static std::atomic<int> g_threads{0};
static std::atomic<int> g_syncs{0};          // waits for the context's stream
static std::atomic<int> g_waits{0};          // of one stream for another: panels
static std::atomic<long> g_allocations{-1};  // allocations that still succeed; -1: all of them
static char g_streams[3];                    // [0]: the context's
static int g_made = 1;

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
    static auto real = (int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*))dlsym(RTLD_NEXT, "pthread_create");
    ++g_threads;
    return real(t, a, f, x);
}
static bool may_allocate() { return g_allocations < 0 || g_allocations-- > 0; }
void* operator new(size_t n) {
    if (void* p = may_allocate() ? std::malloc(n ? n : 1) : nullptr) return p;
    throw std::bad_alloc();
}
void* operator new(size_t n, const std::nothrow_t&) noexcept { return may_allocate() ? std::malloc(n ? n : 1) : nullptr; }
void* operator new[](size_t n) { return operator new(n); }
void* operator new[](size_t n, const std::nothrow_t& t) noexcept { return operator new(n, t); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }
void operator delete[](void* p) noexcept { std::free(p); }
void operator delete[](void* p, size_t) noexcept { std::free(p); }

extern "C" {
int rkh_device_count(void) { return 1; }
int rkh_open(int, void** s, char* name, int, int* cus, int* khz) {
    *s = g_streams;
    name[0] = 0;
    *cus = *khz = 1;
    return RKH_OK;
}
void rkh_close(int, void*) {}
int rkh_malloc(int, void** p, size_t n) { return (*p = std::malloc(n)) ? RKH_OK : RKH_ERR_NOMEM; }
void rkh_free(int, void* p) { std::free(p); }
int rkh_host_alloc(void** p, size_t n) { return rkh_malloc(0, p, n); }
void rkh_host_free(void* p) { std::free(p); }
int rkh_h2d(void*, void* d, const void* s, size_t n) { return std::memcpy(d, s, n), RKH_OK; }
int rkh_d2h(void*, void* d, const void* s, size_t n) { return std::memcpy(d, s, n), RKH_OK; }
int rkh_fill32(void*, void* d, uint32_t v, size_t n) {
    for (size_t i = 0; i < n; ++i) static_cast<uint32_t*>(d)[i] = v;
    return RKH_OK;
}
int rkh_sync(void* s) {
    if (s == g_streams) ++g_syncs;
    return RKH_OK;
}
int rkh_event_create(void** e) { return rkh_malloc(0, e, 1); }
void rkh_event_destroy(void* e) { std::free(e); }
int rkh_event_record(void*, void*) { return RKH_OK; }
int rkh_event_sync(void*) { return RKH_OK; }
int rkh_stream_create(int, void** s) { return *s = g_streams + g_made++, RKH_OK; }
void rkh_stream_destroy(void*) {}
int rkh_stream_wait(void*, void*) { return ++g_waits, RKH_OK; }
int rkh_static_scratch(int, void**, size_t*) { return RKH_ERR_RUNTIME; }
void rkh_set_marker(rkh_marker_fn, void*) {}
size_t rkh_gemm_scratch_bytes(int, int, int, int) { return 0; }
int rkh_pack_w4(void*, const int8_t*, int, int, int, uint8_t*, int*, int32_t*) { return RKH_OK; }
int rkh_pack_w8(void*, const int8_t*, int, int, int, uint8_t*) { return RKH_OK; }
// C[m][n] = A[m][n % K], both fp32
int rkh_quant_gemm(void*, const rkh_quant_args* q, const rkh_gemm_args* g) {
    for (int m = 0; m < q->M; ++m) {
        const float* a = static_cast<const float*>(q->src) + (size_t)m * q->K;
        for (int k = 0; k < q->K; ++k)
            if (q->mode == RKH_Q_W4A8 && !std::isfinite(a[k])) *q->bad_flag = 1;
        for (int n = 0; n < g->N; ++n) static_cast<float*>(g->C)[(size_t)m * g->N + n] = a[n % q->K];
    }
    return RKH_OK;
}
static rkh_quant_args g_quantized; // (the two as launches of their own)
int rkh_quant_rows(void*, const rkh_quant_args* q) { return g_quantized = *q, RKH_OK; }
int rkh_gemm(void* s, const rkh_gemm_args* g) { return rkh_quant_gemm(s, &g_quantized, g); }
}

#define CHECK(x)                                                         \
    do {                                                                 \
        if (!(x)) {                                                      \
            std::fprintf(stderr, "line %d: %s\n", __LINE__, #x);         \
            return 1;                                                    \
        }                                                                \
    } while (0)

static constexpr int M = 1000, K = 1100, N = 2200; // A 4.4 MB, C 8.8 MB

struct Calls {
    rk_npu_ctx* ctx = rk_npu_open(nullptr);
    rk_npu_iommu_domain* domain = rk_npu_iommu_domain_create(ctx, 0);
    std::vector<float> A, C;
    rk_npu_w4a8_weights* w4 = nullptr;
    rk_npu_w4a8_workspace* ws4 = nullptr;
    rk_npu_f32i8f32_weights* w8 = nullptr;
    rk_npu_matmul_workspace* ws8 = nullptr;
    rk_npu_w4a8_config config{};
    rk_npu_matmul_strategy strategy{};
    Calls() : A((size_t)M * K), C((size_t)M * N, 7.0f) {
        for (size_t i = 0; i < A.size(); ++i) A[i] = (float)(i % 9973);
        std::vector<int8_t> B((size_t)K * N, 1);
        std::vector<float> scale(N, 1.0f);
        rk_npu_w4a8_config_init(&config, M, N, K);
        const rk_npu_i4_weight_config i4{K, N, config.k_tile};
        w4 = rk_npu_w4a8_weights_create(domain, &i4, B.data(), scale.data());
        ws4 = rk_npu_w4a8_workspace_create(domain, &config);
        cpu_set_t set;
        sched_getaffinity(0, sizeof(set), &set);
        int cpu = 0;
        while (!CPU_ISSET(cpu, &set)) ++cpu;
        strategy.op_kind = RK_NPU_MATMUL_F32I8F32_DYNAMIC;
        strategy.M = M, strategy.N = N, strategy.K = K, strategy.k_tile = K, strategy.n_tile = 1024;
        strategy.npu_core_mask = 1, strategy.cpu_core_mask = 1ull << cpu, strategy.cpu_threads = 1;
        rk_npu_matmul_weight_config i8{};
        i8.K = K, i8.N = N, i8.k_tile = K;
        w8 = rk_npu_f32i8f32_weights_create(domain, &i8, B.data(), scale.data());
        ws8 = rk_npu_matmul_workspace_create(domain, &strategy);
    }
    bool made() const { return w4 && ws4 && w8 && ws8; }
    int run4() { return rk_npu_w4a8_run_f32(ws4, w4, A.data(), C.data(), nullptr); }
    int run8() { return rk_npu_f32i8f32_run_dynamic(ws8, w8, A.data(), C.data()); }
    bool right() {
        bool ok = true;
        for (int m = 0; m < M; ++m)
            for (int n = 0; n < N; ++n) ok = ok && C[(size_t)m * N + n] == A[(size_t)m * K + n % K];
        C.assign(C.size(), 7.0f);
        return ok;
    }
    bool untouched() const {
        for (float v : C)
            if (v != 7.0f) return false;
        return true;
    }
};

// An earlier device call rejected its input, which nothing has looked at since: the next blocking call says so and
// leaves C alone, the one after it is a good one.
static int rejected_before() {
    Calls c;
    CHECK(c.made());
    std::vector<float> dC((size_t)M * N);
    const float good = c.A[5];
    c.A[5] = std::numeric_limits<float>::infinity();
    CHECK(rk_npu_w4a8_run_f32_device(c.ws4, c.w4, c.A.data(), dC.data()) == RK_NPU_OK);
    c.A[5] = good;
    CHECK(c.run4() == RK_NPU_ERR_PARAM);
    CHECK(c.untouched());
    CHECK(c.run4() == RK_NPU_OK && c.right());
    CHECK(rk_npu_hip_sync(c.ctx) == RK_NPU_OK);
    // (and the call's own input, first and last row)
    for (size_t at : {size_t(3), c.A.size() - 1}) {
        const float keep = c.A[at];
        c.A[at] = std::nanf("");
        CHECK(c.run4() == RK_NPU_ERR_PARAM && c.untouched());
        c.A[at] = keep;
        CHECK(c.run4() == RK_NPU_OK && c.right());
    }
    return 0;
}

// A call waits for its own copies and not for the context's stream, on which other threads go on enqueueing once the
// call has given the submission lock back.
static int own_work_only() {
    Calls c;
    CHECK(c.made());
    g_syncs = 0;
    CHECK(c.run4() == RK_NPU_OK && c.right());
    CHECK(c.run8() == RK_NPU_OK && c.right());
    CHECK(g_syncs == 0);
    return 0;
}

// Memory runs out at any allocation: a handle is not made, a run gives its code, and nothing is thrown at the caller.
static int out_of_memory() {
    Calls c;
    CHECK(c.made());
    int made = 0;
    for (long n = 0; n < 64 && made < 2; ++n) {
        g_allocations = n;
        rk_npu_w4a8_workspace* ws4 = rk_npu_w4a8_workspace_create(c.domain, &c.config);
        g_allocations = n;
        rk_npu_matmul_workspace* ws8 = rk_npu_matmul_workspace_create(c.domain, &c.strategy);
        g_allocations = -1;
        made = (ws4 != nullptr) + (ws8 != nullptr);
        for (int pass = 0; pass < 2; ++pass) { // (with what could be made, the calls work)
            if (ws4) CHECK(rk_npu_w4a8_run_f32(ws4, c.w4, c.A.data(), c.C.data(), nullptr) == RK_NPU_OK && c.right());
            if (ws8) CHECK(rk_npu_f32i8f32_run_dynamic(ws8, c.w8, c.A.data(), c.C.data()) == RK_NPU_OK && c.right());
        }
        rk_npu_w4a8_workspace_free(ws4);
        rk_npu_matmul_workspace_free(ws8);
    }
    CHECK(made == 2);
    for (int (Calls::*run)() : {&Calls::run4, &Calls::run8}) {
        g_allocations = 0;
        const int rc = (c.*run)();
        g_allocations = -1;
        CHECK(rc == RK_NPU_OK && c.right());
    }
    return 0;
}

// Helper threads: three at most, and one processor less than the process may run on; with none no panels.
static int helpers() {
    Calls c;
    CHECK(c.made());
    cpu_set_t all, few;
    CHECK(sched_getaffinity(0, sizeof(all), &all) == 0);
    CPU_ZERO(&few);
    int cpus = 0;
    for (int cpu = 0; cpu < CPU_SETSIZE && cpus < 6; ++cpu) {
        if (!CPU_ISSET(cpu, &all)) continue;
        CPU_SET(cpu, &few);
        ++cpus;
        CHECK(sched_setaffinity(0, sizeof(few), &few) == 0);
        for (int (Calls::*run)() : {&Calls::run4, &Calls::run8}) {
            g_threads = g_waits = 0;
            CHECK((c.*run)() == RK_NPU_OK && c.right());
            CHECK(g_threads == (cpus > 3 ? 3 : cpus - 1));
            CHECK((g_waits > 0) == (cpus > 1));
        }
    }
    return 0;
}

// Which calls go in panels (fp32 in and out): both sides of each line.
static int panelled() {
    Calls c;
    CHECK(c.made());
    const struct { int M, K, N; bool panels; } shapes[] = {
        {1000, 1100, 1040, false},                            // less than 4 MiB out
        {1000, 1013, 1100, false}, {1000, 1014, 1100, true},  // two panels
        {200, 7338, 8192, false},  {200, 7339, 8192, true},   // of which the second is small
        {500, 2228, 6600, false},  {500, 2229, 6600, true},   // four
        {384, 2850, 4224, true},   {385, 2850, 4224, true},   // (the shapes of test_gpu_host_panels.py)
        {387, 2850, 4224, true},   {389, 2850, 4224, true},   {510, 2850, 4224, true}};
    for (const auto& s : shapes) {
        const std::vector<int8_t> B((size_t)s.K * s.N, 1);
        const std::vector<float> scale(s.N, 1.0f), A((size_t)s.M * s.K, 1.0f);
        std::vector<float> C((size_t)s.M * s.N);
        rk_npu_matmul_strategy strategy = c.strategy;
        strategy.M = s.M, strategy.N = s.N, strategy.K = strategy.k_tile = s.K;
        rk_npu_matmul_weight_config i8{};
        i8.K = i8.k_tile = s.K, i8.N = s.N;
        rk_npu_f32i8f32_weights* w = rk_npu_f32i8f32_weights_create(c.domain, &i8, B.data(), scale.data());
        rk_npu_matmul_workspace* ws = rk_npu_matmul_workspace_create(c.domain, &strategy);
        g_waits = 0;
        CHECK(rk_npu_f32i8f32_run_dynamic(ws, w, A.data(), C.data()) == RK_NPU_OK);
        for (float v : C) CHECK(v == 1.0f);
        if ((g_waits > 0) != s.panels) std::fprintf(stderr, "%d x %d x %d\n", s.M, s.K, s.N);
        CHECK((g_waits > 0) == s.panels);
        rk_npu_matmul_workspace_free(ws);
        rk_npu_f32i8f32_weights_free(w);
    }
    return 0;
}

int main(int argc, char** argv) {
    const struct { const char* name; int (*check)(); } checks[] = {{"rejected_before", rejected_before}, {"own_work_only", own_work_only},
                                                                    {"out_of_memory", out_of_memory}, {"helpers", helpers},
                                                                    {"panelled", panelled}};
    for (const auto& c : checks)
        if (argc > 1 && !std::strcmp(argv[1], c.name)) return c.check();
    return 2;
}
