// The library's host code against a stand-in HIP runtime whose device memory
// is host memory with a limit and whose kernels only leave their names: what
// cw_model_prefill and cw_generate launch when the batched prompt phase's
// buffers fit, when they do not, and when room comes back.  No GPU.
//
// Built from the library's objects and this file, without the HIP runtime.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "chat_wgpu.h"

// host stub -> kernel (filled by the objects' static constructors)
static std::map<const void *, std::string> &names() {
    static std::map<const void *, std::string> m;
    return m;
}
static std::vector<std::string> g_launched;
static std::map<void *, size_t> g_mem;
static size_t g_used = 0, g_limit = ~size_t(0);
static hipError_t g_last = hipSuccess;

static hipError_t put(hipError_t e) {
    if (e != hipSuccess) g_last = e;
    return e;
}

extern "C" {
void **__hipRegisterFatBinary(const void *) { return new void *(nullptr); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, dim3 *, dim3 *, int *) {
    names()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st) {
    *g = *b = dim3(1);
    *s = 0;
    *st = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) {
    g_launched.push_back(names()[f]);
    return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t, hipEvent_t,
                              hipEvent_t, int) {
    g_launched.push_back(names()[f]);
    return hipSuccess;
}
hipError_t hipLaunchCooperativeKernel(const void *, dim3, dim3, void **, unsigned, hipStream_t) {
    return put(hipErrorNotSupported);
}
hipError_t hipMalloc(void **p, size_t n) {
    if (n > g_limit - g_used) return put(hipErrorOutOfMemory);
    *p = calloc(1, n);
    g_mem[*p] = n;
    g_used += n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    g_used -= g_mem[p];
    g_mem.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    p->totalGlobalMem = size_t(288) << 30;
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = 100000;
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) {
    memset(a, 0, sizeof *a);
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static char room[1 << 24];
    *p = room;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    *g = reinterpret_cast<hipGraph_t>(1);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    *e = reinterpret_cast<hipGraphExec_t>(1);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
    g_launched.push_back("graph");
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *) { return put(hipErrorNotSupported); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
}

static int count(const char *part) {
    int n = 0;
    for (const auto &s : g_launched) n += s.find(part) != std::string::npos;
    return n;
}

static int g_failed = 0;
static void expect(bool ok, const char *what, int kv, int rc) {
    printf("%s kv %d rc %d gemm %d gemv %d graph %d: %s\n", ok ? "ok  " : "FAIL", kv, rc,
           count("q4_gemm_kernel"), count("q4_gemv_kernel"), count("graph"), what);
    g_failed += !ok;
}

int main() {
    const int L = 2, n = 6;
    for (int kv : {CW_F32, CW_F16}) {
        cw_ctx *ctx = nullptr;
        cw_model *m = nullptr;
        cw_model_config c{};
        c.family.qk_norm = 1;
        c.n_layers = L;
        c.dim = 256;
        c.n_heads = 4;
        c.n_kv_heads = 2;
        c.head_dim = 128;
        c.hidden = 512;
        c.vocab = 300;
        c.eps = 1e-6f;
        c.rope_theta = 1e6f;
        c.max_seq = 64;
        c.kv_dtype = kv;
        int rc = cw_ctx_create(0, &ctx);
        if (rc == CW_OK) rc = cw_model_create(ctx, &c, &m);
        if (rc == CW_OK) rc = cw_model_load_synthetic(m, 7);
        if (rc == CW_OK) rc = cw_model_finalize(m);
        if (rc != CW_OK) {
            printf("FAIL set-up: %d %s\n", rc, cw_last_error());
            return 1;
        }
        const uint32_t prompt[n] = {1, 2, 3, 4, 5, 6};
        uint32_t next = 0, out[4];
        const size_t before = g_used;
        // no room at all, then room for some of the buffers only
        for (size_t room : {size_t(0), size_t(40000)}) {
            g_limit = before + room;
            g_launched.clear();
            rc = cw_model_prefill(m, prompt, n, 0, &next);
            expect(rc == CW_OK && count("q4_gemm") == 0 &&
                       count("q4_gemv_kernel") == n * (4 * L + 1) && g_used == before,
                   "prefill without room goes step by step and keeps nothing", kv, rc);
            g_launched.clear();
            rc = cw_generate(m, prompt, n, 4, 0, CW_STEP_GRAPH, out);
            expect(rc == CW_OK && count("q4_gemm") == 0 && count("graph") == n + 3 &&
                       g_used == before,
                   "generate without room replays the step for the prompt", kv, rc);
        }
        g_limit = ~size_t(0);
        g_launched.clear();
        rc = cw_model_prefill(m, prompt, n, 0, &next);
        expect(rc == CW_OK && count("q4_gemm_kernel") == 4 * L && count("q4_gemv_kernel") == 1,
               "prefill with room runs as one batch", kv, rc);
        g_launched.clear();
        rc = cw_generate(m, prompt, n, 4, 0, CW_STEP_GRAPH, out);
        expect(rc == CW_OK && count("q4_gemm_kernel") == 4 * L && count("graph") == 3,
               "generate with room batches its prompt", kv, rc);
        cw_model_destroy(m);
        cw_ctx_destroy(ctx);
        expect(g_used == 0, "everything is given back", kv, 0);
    }
    return g_failed != 0;
}
