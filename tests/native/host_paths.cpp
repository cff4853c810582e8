// Host paths of the library on a HIP runtime made of host memory: the functions
// below stand in for the runtime's (the executable's definitions come first), so
// allocations can be made to fail, a second device can be current, and what is
// launched, allocated and freed is known.  No kernel runs.  usage: host_paths CASE
#include <hip/hip_runtime_api.h>
#include <dlfcn.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "../../include/qsketch.h"
#include "../../include/qsketch_learned.h"
#include "../../include/qsketch_sf.h"
#include "../../include/qsketch_single.h"

namespace {
struct launch {
    std::string kernel;
    int device;
};
int g_device = 0;                    // current device
uint64_t g_mallocs = 0, g_frees = 0; // device allocations made, live ones freed
uint64_t g_fail_at = 0;              // the allocation of this number fails (0: none)
hipError_t g_last = hipSuccess;      // sticky, as the runtime's
std::map<void *, size_t> g_live;
std::vector<launch> g_launches;
uint64_t g_handles = 0;
bool g_fail_launches = false;
float g_correction = 0.f; // the first moment's bias correction of the last training step
uint32_t g_word = 0; // the first word of every g_word_bytes-byte copy to the host, unless 0
size_t g_word_bytes = 8;
size_t g_bytes = 0, g_budget = ~(size_t)0; // device memory in use and in all
struct routed {
    const void *keys;
    uint64_t n;
};
std::vector<routed> g_routed; // the routing launches' keys

hipError_t fail(hipError_t e)
{
    g_last = e;
    return e;
}

int g_bad = 0;
void expect(bool ok, const char *what)
{
    if (!ok) {
        printf("FAILED: %s\n", what);
        g_bad = 1;
    }
}
} // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t bytes)
{
    *p = nullptr;
    if (++g_mallocs == g_fail_at || bytes > g_budget - g_bytes)
        return fail(hipErrorOutOfMemory);
    *p = calloc(bytes ? bytes : 1, 1);
    g_live[*p] = bytes;
    g_bytes += bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (!p)
        return hipSuccess;
    const auto it = g_live.find(p);
    if (it == g_live.end())
        return fail(hipErrorInvalidValue);
    g_bytes -= it->second;
    g_live.erase(it);
    ++g_frees;
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned int)
{
    *p = calloc(bytes, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind kind)
{
    memcpy(d, s, n);
    if (g_word && n == g_word_bytes && kind == hipMemcpyDeviceToHost)
        memcpy(d, &g_word, 4);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n)
{
    *n = 2;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = g_device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d)
{
    g_device = d;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int)
{
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) // (a macro names the current version of it)
{
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int)
{
    *s = reinterpret_cast<hipStream_t>(++g_handles);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = reinterpret_cast<hipEvent_t>(++g_handles);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
    *g = reinterpret_cast<hipGraph_t>(++g_handles);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    *x = reinterpret_cast<hipGraphExec_t>(++g_handles);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGetLastError()
{
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shared, hipStream_t *s)
{
    *g = dim3(1);
    *b = dim3(1);
    *shared = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t)
{
    Dl_info info;
    g_launches.push_back({dladdr(f, &info) && info.dli_sname ? info.dli_sname : "?", g_device});
    if (g_launches.back().kernel.find("k_grad_sum") != std::string::npos)
        g_correction = *static_cast<float *>(args[12]);
    if (g_launches.back().kernel.find("k_route") != std::string::npos)
        g_routed.push_back({*static_cast<void **>(args[0]), *static_cast<uint64_t *>(args[1])});
    return g_fail_launches ? fail(hipErrorLaunchFailure) : hipSuccess;
}
} // extern "C"

static qs_params params(uint64_t n_low)
{
    qs_params p;
    qs_default_params(&p, 1 << 16, 0.5);
    p.n_low = n_low;
    p.rng_seed = 1;
    return p;
}

static uint32_t s_keys[1]; // stands for device keys: nothing reads them

// While a captured graph lives, nothing may free the scratch it holds: a batch
// that needs more is refused, whichever way it comes.
static void case_graph()
{
    const qs_params p = params(1021);
    qs_sketch *s = nullptr;
    qs_graph *g = nullptr, *g2 = nullptr;
    expect(qs_create(&p, &s) == QS_OK, "create");
    const uint64_t small[2] = {0, 1500}, less[2] = {0, 1000}, more[2] = {0, 1501};
    expect(qs_graph_capture_insert(s, s_keys, small, nullptr, &g) == QS_OK, "capture");
    const uint64_t frees = g_frees;
    expect(qs_graph_capture_insert(s, s_keys, more, nullptr, &g2) == QS_ERR_STATE && !g2, "larger capture refused");
    expect(qs_insert(s, s_keys, 1501) == QS_ERR_STATE, "larger insert refused");
    expect(qs_insert_async(s, s_keys, 1501, nullptr) == QS_ERR_STATE, "larger stream-ordered insert refused");
    expect(qs_insert(s, s_keys, 1ull << 26) == QS_ERR_STATE, "filtered insert refused");
    expect(g_frees == frees, "the graph's scratch is still allocated");
    expect(qs_graph_capture_insert(s, s_keys, less, nullptr, &g2) == QS_OK, "smaller capture");
    expect(qs_insert(s, s_keys, 1500) == QS_OK, "insert that fits");
    qs_graph_destroy(g);
    expect(qs_insert(s, s_keys, 1501) == QS_ERR_STATE, "refused while the second graph lives");
    qs_graph_destroy(g2);
    expect(qs_insert(s, s_keys, 1501) == QS_OK, "accepted without graphs");
    qs_destroy(s);
    expect(g_live.empty(), "everything freed");
}

// An allocation of the hot-key filter that fails leaves nothing half built: the call is
// inserted the ordinary way, and the next one allocates all of the filter, as the first
// call of another sketch does.
static void case_hot_alloc()
{
    const uint64_t n = 1ull << 26;
    const qs_params p = params(1021);
    uint64_t whole = 0; // allocations of a first filtered call
    for (uint64_t k = 0; k <= 7; ++k) { // the k-th of the filter's own fails (0: none)
        qs_sketch *s = nullptr;
        expect(qs_create(&p, &s) == QS_OK, "create");
        expect(qs_insert_async(s, s_keys, n, nullptr) == QS_OK, "the insert's scratch");
        const size_t live = g_live.size();
        if (k) {
            g_fail_at = g_mallocs + k;
            expect(qs_insert(s, s_keys, n) == QS_OK, "the ordinary insert takes over");
            expect(g_live.size() == live, "what was allocated before the failure is freed");
            g_fail_at = 0;
        }
        const uint64_t before = g_mallocs;
        expect(qs_insert(s, s_keys, n) == QS_ERR_HIP, "no kernel publishes the candidates here");
        whole = k ? whole : g_mallocs - before;
        expect(g_mallocs - before == whole, "the next call allocates everything");
        qs_destroy(s);
        expect(g_live.empty(), "everything freed");
    }
}

// the k-th allocation of `call` fails, for every k: reported as such, with no error
// left in the runtime for the next launch check, and the call works when repeated
template <class F> static void each_allocation_fails(const char *what, F call)
{
    for (uint64_t k = 1;; ++k) {
        const uint64_t before = g_mallocs;
        g_fail_at = before + k;
        const int rc = call();
        g_fail_at = 0;
        if (g_mallocs < before + k) { // it makes fewer than k
            expect(k > 1 && rc == QS_OK, what);
            return;
        }
        expect(rc == QS_ERR_NOMEM, what);
        expect(hipGetLastError() == hipSuccess, what);
    }
}

static void case_alloc_errors()
{
    const qs_params p = params(1021);
    qs_sketch *s = nullptr;
    qs_sf *f = nullptr;
    qs_sl *l = nullptr;
    qs_learned *L = nullptr;
    each_allocation_fails("qs_create", [&] { return qs_create(&p, &s); });
    each_allocation_fails("qs_sf_create", [&] { return qs_sf_create(1021, 8, 3, 1, 1021, 4, 1, &f); });
    each_allocation_fails("qs_sl_create", [&] { return qs_sl_create(1021, 8, 1, 1021, 4, 1, &l); });
    each_allocation_fails("qs_learned_create", [&] { return qs_learned_create(&p, 10, 1, &L); });
    each_allocation_fails("qs_insert", [&] { return qs_insert(s, s_keys, 100000); });
    each_allocation_fails("qs_sf_insert", [&] { return qs_sf_insert(f, s_keys, 100000); });
    each_allocation_fails("qs_learned_insert", [&] { return qs_learned_insert(L, s_keys, 1 << 12, nullptr); });
    qs_destroy(s);
    qs_sf_destroy(f);
    qs_sl_destroy(l);
    qs_learned_destroy(L);
    expect(g_live.empty(), "everything freed");
}

// the learned form's device check (error bit 2 of a call): an insert that lost keys
// says so, and so do the following ones until the clear
static void case_learned_error()
{
    const qs_params p = params(1021);
    qs_learned *L = nullptr;
    expect(qs_learned_create(&p, 10, 1, &L) == QS_OK, "create");
    g_word = 2;
    expect(qs_learned_insert(L, s_keys, 1 << 21, nullptr) == QS_ERR_INTERNAL, "the failed check is reported");
    g_word = 0;
    expect(!qs_learned_table_full(L), "the table is not full");
    expect(qs_learned_insert(L, s_keys, 1 << 10, nullptr) == QS_ERR_INTERNAL, "invalid until the clear");
    expect(qs_learned_clear(L) == QS_OK && qs_learned_insert(L, s_keys, 1 << 10, nullptr) == QS_OK, "valid after it");
    qs_learned_destroy(L);
}

// a sketch is cleared on its own device, whichever is current
static void case_clear_device()
{
    const qs_params p = params(1021);
    qs_sketch *s = nullptr;
    expect(qs_create(&p, &s) == QS_OK, "create");
    for (int current = 1; current >= 0; --current) {
        g_device = current;
        g_launches.clear();
        expect(qs_clear(s) == QS_OK && g_launches.size() == 1, "clear");
        for (const launch &l : g_launches)
            expect(l.device == 0, l.kernel.c_str());
        expect(g_device == current, "the current device is the caller's again");
    }
    qs_destroy(s);
}

// a training step whose launches fail is no step: the next one is the first
static void case_failed_step()
{
    const qs_params p = params(1021);
    qs_learned *L = nullptr;
    expect(qs_learned_create(&p, 10, 1, &L) == QS_OK, "create");
    const float t[1] = {0.f};
    g_fail_launches = true;
    expect(qs_mlp_step(L, s_keys, t, 64, 1e-3f, 0.9f, 0.999f, 1e-8f, nullptr, nullptr) == QS_ERR_HIP, "failed launch");
    g_fail_launches = false;
    for (int step = 1; step <= 2; ++step) {
        expect(qs_mlp_step(L, s_keys, t, 64, 1e-3f, 0.9f, 0.999f, 1e-8f, nullptr, nullptr) == QS_OK, "step");
        expect(g_correction == 1.f - powf(0.9f, (float)step), "bias correction");
    }
    qs_learned_destroy(L);
}

// A learned insert needs no more memory than a flag and one copy of each key beside
// the sketch's scratch: with less than its buffers would like, it runs in pieces.
static void case_learned_memory()
{
    const uint64_t n = (1 << 22) + 77;
    static uint32_t keys[n];
    const qs_params p = params(1021);
    qs_sketch *s = nullptr;
    expect(qs_create(&p, &s) == QS_OK, "create");
    const size_t before = g_bytes;
    expect(qs_insert(s, keys, n) == QS_OK, "insert");
    const size_t scratch = g_bytes - before; // of the sketch, for n keys
    qs_destroy(s);
    qs_learned *L = nullptr;
    expect(qs_learned_create(&p, 10, 1, &L) == QS_OK, "create");
    g_budget = g_bytes + n * 5 + 65536;
    for (int call = 0; call < 2; ++call) {
        uint64_t heavy = 0, at = 0;
        g_routed.clear();
        expect(qs_learned_insert(L, keys, n, &heavy) == QS_OK && heavy == n, "insert in pieces");
        for (const routed &r : g_routed) {
            expect(r.keys == keys + at, "a piece starts where the last one ended");
            at += r.n;
        }
        expect(at == n && g_routed.size() > 1, "the pieces make up the call");
    }
    g_budget = ~(size_t)0;
    qs_learned_destroy(L);
    // the sketch's scratch takes the place of buffers that the routing has done with
    expect(qs_learned_create(&p, 10, 1, &L) == QS_OK, "create");
    expect(qs_learned_insert(L, keys, n, nullptr) == QS_OK, "insert in one piece");
    g_budget = g_bytes + scratch - n * 4;
    g_word_bytes = 4;
    g_word = (uint32_t)n; // every key light
    expect(qs_learned_insert(L, keys, n, nullptr) == QS_OK, "room made for the sketch");
    g_word = 0;
    g_word_bytes = 8;
    g_budget = ~(size_t)0;
    qs_learned_destroy(L);
    expect(g_live.empty(), "everything freed");
}

// The filter only saves time: a call for which it does not fit the device is inserted
// the ordinary way.
static void case_filter_memory()
{
    const uint64_t n = 1ull << 26;
    const qs_params p = params(1021);
    qs_sketch *s = nullptr;
    expect(qs_create(&p, &s) == QS_OK && qs_set_hot_filter(s, 0) == QS_OK, "create");
    const size_t before = g_bytes;
    expect(qs_insert(s, s_keys, n) == QS_OK, "insert without the filter");
    const size_t scratch = g_bytes - before;
    qs_destroy(s);
    for (size_t more : {(size_t)0, (size_t)100 << 20, (size_t)n * 9}) { // (the filter takes 8 bytes per key)
        expect(qs_create(&p, &s) == QS_OK, "create");
        g_budget = g_bytes + scratch + more;
        const int want = more < n * 9 ? QS_OK : QS_ERR_HIP; // (QS_ERR_HIP: no kernel publishes the candidates here)
        for (int call = 0; call < 2; ++call)
            expect(qs_insert(s, s_keys, n) == want, "insert in what the ordinary way takes");
        g_budget = g_bytes + 1;
        expect(qs_insert(s, s_keys, 2 * n) == QS_ERR_NOMEM, "not in less");
        g_budget = ~(size_t)0;
        qs_destroy(s);
        expect(g_live.empty(), "everything freed");
    }
}

int main(int argc, char **argv)
{
    const std::map<std::string, void (*)()> cases = {
        {"graph", case_graph},
        {"hot_alloc", case_hot_alloc},
        {"alloc_errors", case_alloc_errors},
        {"learned_error", case_learned_error},
        {"clear_device", case_clear_device},
        {"failed_step", case_failed_step},
        {"learned_memory", case_learned_memory},
        {"filter_memory", case_filter_memory},
    };
    setvbuf(stdout, nullptr, _IONBF, 0);
    const auto c = cases.find(argc > 1 ? argv[1] : "");
    if (c == cases.end())
        return 2;
    c->second();
    return g_bad;
}
