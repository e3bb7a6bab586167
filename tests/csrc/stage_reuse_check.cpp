/*
 * The pinned block of an upload is not written while its copy may still be
 * under way: on the host alone (the stubs of pass_error_check.cpp), with copies
 * that read their source only when the host waits for the stream.  A pass that
 * ends in an error after its upload does not wait.
 */
#include <hip/hip_runtime_api.h>

#define main pass_error_main
#define hipMemcpyAsync copy_at_once
#define hipStreamSynchronize wait_for_nothing
#include "pass_error_check.cpp"
#undef hipMemcpyAsync
#undef hipStreamSynchronize
#undef main

struct copy {
    const char *src;
    std::vector<char> was;
};
static std::vector<copy> pending;
static int changed;

extern "C" hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
    if (k == hipMemcpyHostToDevice) pending.push_back({(const char *)s, {(const char *)s, (const char *)s + n}});
    return copy_at_once(d, s, n, k, st);
}
extern "C" hipError_t hipStreamSynchronize(hipStream_t st) {
    for (const copy &c : pending) changed += memcmp(c.src, c.was.data(), c.was.size()) != 0;
    pending.clear();
    return wait_for_nothing(st);
}

int main() {
    double o[3] = {0, 0, 0}, d[3] = {3, 3, 3}, h[3] = {1, 1, 1};
    const int N = 300;
    std::vector<double> x(3 * N);
    std::vector<int> t(N, 1);
    struct engine *e = engine_alloc();
    struct potential *p;
    srand48(1);
    for (auto &v : x) v = 3 * drand48();
    if (engine_init(e, o, d, h, 0.9, 7, 1, engine_flag_gpu | engine_flag_verlet_pseudo) < 0) return 2;
    if (engine_addtype(e, 1.0, 0.0, (char *)"A", (char *)"A") < 0) return 2;
    if ((p = potential_create_LJ126(0.05, 0.9, 1e-6, 1e-3, 1e-3)) == NULL || engine_addpot(e, p, 1, 1) < 0) return 2;
    if (engine_load(e, x.data(), NULL, t.data(), NULL, NULL, NULL, NULL, N) < 0 || engine_start(e, 1, 1) < 0) return 2;
    if (engine_shuffle(e) < 0) return 2;
    /* sort lists that do not exist yet: an error after the upload */
    e->s.verlet_rebuild = 0;
    if (pass(e) >= 0) return 3;
    /* the program goes on with other positions */
    for (int c = 0; c < e->s.nr_cells; c++)
        for (int k = 0; k < e->s.cells[c].count; k++) e->s.cells[c].parts[k].x[0] *= 0.5;
    e->s.verlet_rebuild = 1;
    if (pass(e) < 0) return 4;
    printf("%d copies changed under way\n", changed);
    engine_free(e);
    return changed != 0;
}
