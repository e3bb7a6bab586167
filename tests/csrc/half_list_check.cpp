/*
 * The half shell's lists as its kernels get them, on the host alone (the
 * stubs of pass_error_check.cpp): per cell the self task and each pair task
 * whose i cell it is, in task order, and the i cells that visit it as a task's
 * j cell, in task order, each task's slot among those in its entry.
 */
#include <hip/hip_runtime_api.h>

#define main pass_error_main
#define hipLaunchKernel queue_launch
#include "pass_error_check.cpp"
#undef hipLaunchKernel
#undef main

struct entry {
    int x, y, z, w;
};
static const entry *nbr;
static const int *nbr_off, *inv_off, *inv_cell;

extern "C" hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t n, hipStream_t s) {
    const std::string &k = names()[f];
    if (k.find("k_nonbond_half") != std::string::npos) {
        nbr = *(const entry **)args[2];
        nbr_off = *(const int **)args[3];
    } else if (k.find("k_fold") != std::string::npos) {
        inv_off = *(const int **)args[7];
        inv_cell = *(const int **)args[8];
    }
    return queue_launch(f, g, b, args, n, s);
}

int main() {
    /* cells of unequal edges: some tasks' offsets lie along their sort axis,
       others do not */
    double o[3] = {0, 0, 0}, d[3] = {4, 5.2, 3.3}, h[3] = {0.5, 1.3, 1.1};
    const int N = 500;
    std::vector<double> x(3 * N);
    std::vector<int> t(N, 1);
    struct engine *e = engine_alloc();
    struct potential *p;
    srand48(1);
    for (int k = 0; k < 3 * N; k++) x[k] = d[k % 3] * drand48();
    if (engine_init(e, o, d, h, 1.0, 7, 1, engine_flag_gpu | engine_flag_halfshell) < 0) return 2;
    if (engine_addtype(e, 1.0, 0.0, (char *)"A", (char *)"A") < 0) return 2;
    if ((p = potential_create_LJ126(0.05, 1.0, 1e-6, 1e-3, 1e-3)) == NULL || engine_addpot(e, p, 1, 1) < 0) return 2;
    if (engine_load(e, x.data(), NULL, t.data(), NULL, NULL, NULL, NULL, N) < 0 || engine_start(e, 1, 1) < 0) return 2;
    if (engine_shuffle(e) < 0 || pass(e) < 0 || nbr == NULL || inv_off == NULL) return 2;
    struct space *s = &e->s;
    std::vector<int> at(nbr_off, nbr_off + s->nr_cells), in(inv_off, inv_off + s->nr_cells);
    int bad = 0, pairs = 0;
    for (int k = 0; k < s->nr_tasks; k++) {
        const struct task *tk = &s->tasks[k];
        if (tk->type == task_type_self) {
            const entry &en = nbr[at[tk->i]++];
            bad += en.x != tk->i || en.y != 1 << 5;
        } else if (tk->type == task_type_pair) {
            const entry &en = nbr[at[tk->i]++];
            const int slot = 1 + in[tk->j] - inv_off[tk->j];
            bad += en.x != tk->j || (en.y & 0x3f) != tk->flags || (int)((unsigned int)en.y >> 9) != slot;
            bad += inv_cell[in[tk->j]++] != tk->i;
            pairs++;
        }
    }
    for (int c = 0; c < s->nr_cells; c++) bad += at[c] != nbr_off[c + 1] || in[c] != inv_off[c + 1];
    printf("%d pair tasks, %d faults\n", pairs, bad);
    engine_free(e);
    return bad != 0 || pairs == 0;
}
