/* Host packing between cells and the device's cell-ordered arrays; see
   hostpack.h.  Each loop runs over cells in parallel; every cell writes its
   own slot range, so the results do not depend on the thread count. */
#include <omp.h>
#include <pthread.h>

#include "hostpack.h"

/* A loop takes a thread per SPACE_PER_THREAD particles.  The threads of a team
   wait for the next loop actively; a team of all 16 cores for every loop used
   up the process's CPU share, and then the whole process stood still for 20
   to 50 ms.  32,000 particles, 25 surrogate steps a call, mean and longest of
   200 calls: 13.5 to 15.1 ms and 64 with 16 threads always, 11.7 and 13.7 with
   one per 8192, 11.6 and 13.2 per 4096, 11.8 and 14.6 per 16384, 11.9 and 15.2
   per 32768.  Passes of 64,000 particles 0.77, 0.76, 0.76, 0.78, 0.90 ms, of
   100,000 0.95, 0.94, 0.96, 0.97, 1.13. */
#define SPACE_PER_THREAD 8192

/* A child forked after a loop of several threads has none of them, and
   libgomp would wait for them: its loops take one. */
static volatile int teams, alone;

static void forked(void) { alone |= teams; }

__attribute__((constructor)) static void watch_forks(void) { (void)pthread_atfork(NULL, NULL, forked); }

int space_threads(int n) {
    const int m = alone ? 1 : omp_get_max_threads();
    int t = 1 + n / SPACE_PER_THREAD;
    t = t < m ? t : m;
    if (t > 1 && !teams) teams = 1;
    return t;
}

int space_pack(const struct space *s, int max_type, int *count, int *offset, int *cnt_off, double *x, int *type,
               int *id, int *maxc, int *maxid) {
    const int nc = s->nr_cells;
    int n = 0, mc = 0, mid = -1, bad = 0;
    for (int cid = 0; cid < nc; cid++) {
        const int c = s->cells[cid].count;
        count[cid] = c;
        offset[cid] = n;
        cnt_off[2 * cid] = c;
        cnt_off[2 * cid + 1] = n;
        if (c > mc) mc = c;
        n += c;
    }
    offset[nc] = n;
#pragma omp parallel for num_threads(space_threads(s->nr_parts)) schedule(static) reduction(max : mid) reduction(| : bad)
    for (int cid = 0; cid < nc; cid++) {
        const struct cell *c = &s->cells[cid];
        for (int k = 0; k < c->count; k++) {
            const int a = offset[cid] + k;
            const struct part *p = &c->parts[k];
            if (p->type < 0 || p->type >= max_type) bad = 1;
            x[3 * a] = p->x[0];
            x[3 * a + 1] = p->x[1];
            x[3 * a + 2] = p->x[2];
            type[a] = p->type;
            id[a] = p->id;
            if (p->id > mid) mid = p->id;
        }
    }
    *maxc = mc;
    *maxid = mid;
    return bad ? -1 : n;
}

void space_pack_v(const struct space *s, const int *offset, double *v) {
#pragma omp parallel for num_threads(space_threads(s->nr_parts)) schedule(static)
    for (int cid = 0; cid < s->nr_cells; cid++) {
        const struct cell *c = &s->cells[cid];
        for (int k = 0; k < c->count; k++)
            for (int m = 0; m < 3; m++) v[3 * (offset[cid] + k) + m] = c->parts[k].v[m];
    }
}

int space_add_forces(struct space *s, const int *ioi, int n, const float *fhi, const float *flo) {
    int bad = 0;
#pragma omp parallel for num_threads(space_threads(s->nr_parts)) schedule(static) reduction(| : bad)
    for (int cid = 0; cid < s->nr_cells; cid++) {
        struct cell *c = &s->cells[cid];
        for (int k = 0; k < c->count; k++) {
            const int a = ioi[c->parts[k].id];
            if (a < 0 || a >= n) {
                bad = 1;
                continue;
            }
            for (int m = 0; m < 3; m++)
                c->parts[k].f[m] += (double)fhi[4 * (size_t)a + m] + (double)flo[4 * (size_t)a + m];
        }
    }
    return bad ? -1 : 0;
}

void space_add_forces_slots(struct space *s, const int *offset, const float *fhi, const float *flo) {
#pragma omp parallel for num_threads(space_threads(s->nr_parts)) schedule(static)
    for (int cid = 0; cid < s->nr_cells; cid++) {
        struct cell *c = &s->cells[cid];
        for (int k = 0; k < c->count; k++) {
            const size_t a = (size_t)(offset[cid] + k);
            for (int m = 0; m < 3; m++) c->parts[k].f[m] += (double)fhi[4 * a + m] + (double)flo[4 * a + m];
        }
    }
}
