/*
 * Passes that fail between the pair kernel and the totals, on the host alone:
 * the HIP runtime's entry points that the library calls are defined here, and
 * a kernel launch does only what the work queues see of it.  The pair kernel
 * of the half shell finds its work through the queues, which must be zero
 * when it starts and are used up when it ends; the totals clear them.
 */
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

extern "C" {
#include "mdcore.h"
#include "engine_gpu.h"
struct engine *engine_alloc(void);
void engine_free(struct engine *e);
int engine_prepare(struct engine *e);
int engine_nonbond_eval(struct engine *e);
}

#define NQ 8

static std::map<const void *, std::string> &names() {
    static auto *m = new std::map<const void *, std::string>;
    return *m;
}

static int fail_totals, fail_events, failed; /* switches; an error to report */
static int pair_passes, pair_without_work;

extern "C" {
void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    names()[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

static dim3 cfg_grid, cfg_block;
static size_t cfg_shmem;
static hipStream_t cfg_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
    cfg_grid = g;
    cfg_block = b;
    cfg_shmem = s;
    cfg_stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st) {
    *g = cfg_grid;
    *b = cfg_block;
    *s = cfg_shmem;
    *st = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t) {
    const std::string &n = names()[f];
    auto is = [&](const char *s) { return n.find(s) != std::string::npos; };
    if (is("k_nonbond_half")) {
        int *queue = *(int **)args[19];
        int used = 0;
        for (int q = 0; q < NQ; q++) used |= queue[q] != 0;
        pair_passes++;
        pair_without_work += used;
        for (int q = 0; q < NQ; q++) queue[q] = 1000;
    } else if (is("k_reduce_one") || is("k_reduce_b")) {
        if (fail_totals) {
            failed = 1;
            return hipErrorLaunchFailure;
        }
        memset(*(int **)args[7], 0, sizeof(int) * NQ);
    } else if (is("k_clear_queue"))
        memset(*(int **)args[0], 0, sizeof(int) * NQ);
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const int f = failed;
    failed = 0;
    return f ? hipErrorLaunchFailure : hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) { return (*p = calloc(n ? n : 1, 1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) {
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void *d, int v, size_t n) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipMemcpyToSymbol(const void *, const void *, size_t, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = (hipStream_t)8;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = (hipEvent_t)8;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) {
    /* the third event of a timed pass comes after the pair kernel */
    return fail_events && --fail_events == 0 ? hipErrorInvalidHandle : hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) {
    *t = 0.0f;
    return hipSuccess;
}
#undef hipGetDeviceProperties
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 8;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "stub"; }
}

static int pass(struct engine *e) { return engine_prepare(e) < 0 ? -1 : engine_nonbond_eval(e); }

int main() {
    double o[3] = {0, 0, 0}, d[3] = {3, 3, 3}, h[3] = {1, 1, 1}, ms[4];
    const int N = 300;
    std::vector<double> x(3 * N);
    std::vector<int> t(N, 1);
    struct engine *e = engine_alloc();
    struct potential *p;
    srand48(1);
    for (auto &v : x) v = 3 * drand48();
    if (engine_init(e, o, d, h, 1.0, 7, 1, engine_flag_gpu | engine_flag_halfshell) < 0) return 2;
    if (engine_addtype(e, 1.0, 0.0, (char *)"A", (char *)"A") < 0) return 2;
    if ((p = potential_create_LJ126(0.05, 1.0, 1e-6, 1e-3, 1e-3)) == NULL || engine_addpot(e, p, 1, 1) < 0) return 2;
    if (engine_load(e, x.data(), NULL, t.data(), NULL, NULL, NULL, NULL, N) < 0 || engine_start(e, 1, 1) < 0) return 2;
    if (engine_shuffle(e) < 0 || pass(e) < 0 || pass(e) < 0) return 2;
    /* the totals' launch fails */
    fail_totals = 1;
    if (pass(e) >= 0) return 3;
    fail_totals = 0;
    if (pass(e) < 0) return 4;
    /* the event after the pair kernel fails */
    fail_events = 3;
    if (engine_gpu_time(e, 1, 0, ms) >= 0) return 5;
    if (pass(e) < 0 || pass(e) < 0) return 6;
    printf("%d pair passes, %d without work\n", pair_passes, pair_without_work);
    engine_free(e);
    return pair_without_work != 0;
}
