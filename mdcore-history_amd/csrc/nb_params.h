/*
 * Parameters of a nonbonded pass, as its kernels get them.  Internal header.
 */
#ifndef NB_PARAMS_H
#define NB_PARAMS_H

struct nb_params {
    int ncells, nparts, nids, max_type, proj;
    int dmaxdist;
    double dscale, bias, cutoff2;
    double dim[3], h[3];
    float rc2f, band;
    double cutoff;
    int tshift, imask; /* packed record: type = w >> tshift, slot = (w >> 16) & imask */
    /* Pseudo-Verlet: per-cell maxdx widening each pair window
       (runner_dopair.c:428), or NULL (no widening: dmaxdist). */
    const double *maxdx;
    int maxn, maxnbr;
    int ptab_bytes, coef_bytes; /* sizes of the table headers and coefficients */
    /* dynamic LDS layout (byte offsets) */
    int lds_own_key, lds_kfl, lds_stage, lds_hit, lds_dense, lds_jf;
    int nsplit; /* neighbour groups per owner cell (work items per cell) */
    const int *order; /* owner cell of each owner position in the work order */
    int window; /* some entries need the reference's window test (pair_tile.h) */
    float filt; /* k_pair's filter threshold on r^2 */
    int walk_cap; /* k_pair, projected window: see pair_tile.h */
};

#endif /* NB_PARAMS_H */
