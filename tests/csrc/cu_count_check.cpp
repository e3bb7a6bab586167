/*
 * What the projected window's rounding rule takes from the launch does not
 * depend on the device's compute units, on the host alone (the stubs of
 * pass_error_check.cpp): prints k_pair's walk_cap for a device of argv[1]
 * compute units and cubic cells of 1 nm, argv[2] along an axis.
 */
#include <hip/hip_runtime_api.h>

#define main pass_error_main
#define hipLaunchKernel queue_launch
#define hipGetDevicePropertiesR0600 properties_of_256
#include "pass_error_check.cpp"
#undef hipGetDevicePropertiesR0600
#undef hipLaunchKernel
#undef main

#include "../../mdcore-history_amd/csrc/nb_params.h"

static int cus, cap = -1;

extern "C" hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d) {
    properties_of_256(p, d);
    p->multiProcessorCount = cus;
    return hipSuccess;
}
extern "C" hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t n, hipStream_t s) {
    if (names()[f].find("k_pair") != std::string::npos) cap = ((const struct nb_params *)args[0])->walk_cap;
    return queue_launch(f, g, b, args, n, s);
}

int main(int argc, char **argv) {
    cus = atoi(argv[1]);
    const double edge = atof(argv[2]);
    double o[3] = {0, 0, 0}, d[3] = {edge, edge, edge}, h[3] = {1, 1, 1};
    const int N = 300;
    std::vector<double> x(3 * N);
    std::vector<int> t(N, 1);
    struct engine *e = engine_alloc();
    struct potential *p;
    srand48(1);
    for (auto &v : x) v = edge * drand48();
    if (engine_init(e, o, d, h, 1.0, 7, 1, engine_flag_gpu | engine_flag_fullshell | engine_flag_projwindow) < 0) return 2;
    if (engine_addtype(e, 1.0, 0.0, (char *)"A", (char *)"A") < 0) return 2;
    if ((p = potential_create_LJ126(0.05, 1.0, 1e-6, 1e-3, 1e-3)) == NULL || engine_addpot(e, p, 1, 1) < 0) return 2;
    if (engine_load(e, x.data(), NULL, t.data(), NULL, NULL, NULL, NULL, N) < 0 || engine_start(e, 1, 1) < 0) return 2;
    if (engine_shuffle(e) < 0 || pass(e) < 0) return 2;
    printf("%d\n", cap);
    engine_free(e);
    return 0;
}
