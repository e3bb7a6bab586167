/*
 * gfx950 nonbonded engine behind the mdcore C API (C-ABI in engine_gpu.h).
 *
 * One nonbonded pass is a chain of launches on one stream:
 *   k_pack      (at the upload, or with the migration of a resident step)
 *               cell-ordered FP64 positions -> float4 (x, y, z, type bits),
 *               id -> slot map, slot -> cell map;
 *   k_sort_rank runner_dosort (runner_dosort.c:97-161) for every cell and
 *               every flagged direction: 16-bit projection keys computed in
 *               FP64 without contraction; particles with a key of their own
 *               are placed by rank, and a list with equal keys is sorted by
 *               the reference's descending quicksort (runner.c:110-174)
 *               replayed, so that the sorted lists, ties included, are the
 *               reference's (k_sort: the same per list in global memory, for
 *               cells of more than 480 particles).  Cells of more than 64
 *               particles get a wave per direction and a wave-parallel
 *               restatement of that quicksort (sort_desc_wave); smaller
 *               cells one wave that sorts all their lists (sort_lists_wave);
 *   k_pair      (pair_tile.h) full shell, table mode: one wave per work item,
 *               an owner cell and a share of its neighbour list (the
 *               reference's self/pair tasks that touch it): matrix-core
 *               distance filter, the hits dealt over the lanes, FP32 table
 *               evaluation (potential_eval.h:67-104).  It accumulates the
 *               forces of its own atoms only (every pair at both its cells),
 *               so no atomics on forces and no cross-wave write conflicts.
 *               Excluded pairs are subtracted afterwards as in
 *               exclusion.c:81-282;
 *   k_nonbond_half
 *               half shell, table mode: persistent waves pull owner cells from
 *               8 device queues (one per XCD slab of cells) and visit each
 *               pair task once, at its i cell.  Lanes are (owner atom,
 *               partition); each neighbour cell is staged in LDS in window
 *               order, each lane walks its share of the sorted window
 *               (runner_dopair.c:455-478) and evaluates its hits; the opposite
 *               forces go into LDS copies of the visited cell and out to a
 *               slot per visit;
 *   k_nonbond_mlp, k_nonbond_mlp_half
 *               the surrogate's pass, full or half shell: the same walk, the
 *               hits evaluated with the network;
 *   k_fold      per atom, the groups' partial forces and the half-shell
 *               slots, added in a fixed order;
 *   k_reduce_one (few items) or k_reduce_a/b
 *               per-item FP64 energies/virials/counts -> totals, fixed order.
 * Staged neighbour records hold their positions moved into the owner's
 * frame (x + shift, once per record), so a candidate's distance is one
 * subtraction per axis.  In the full shell every pair is evaluated by both
 * of its cells (once per owner); the two owners' FP32 distances are opposite
 * to rounding (each side rounds its own shifted position), so the forces sum
 * to zero to FP32 rounding; energy, virial and counts are taken on the task's
 * i side only.
 */
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdlib.h>
#include <string.h>
#include <time.h>

#include "gpu_state.h"
#include "hostpack.h"

/* ------------------------------------------------------------ device helpers */

__device__ __forceinline__ void acc2(float &hi, float &lo, float v) {
    /* hi + lo += v with the rounding error of hi + v kept in lo (two-sum). */
    float s = hi + v;
    float bp = s - hi;
    float err = (hi - (s - bp)) + (v - bp);
    hi = s;
    lo += err;
}

__device__ __forceinline__ double min_image(double s, double dim) {
    if (s * 2 > dim)
        s -= dim;
    else if (s * 2 < -dim)
        s += dim;
    return s;
}

/* Reference r^2 of a pair task (runner_dopair.c:465-486 with fptype.h:275-278):
   pix = x_i - shift, dx = pix - x_j, r2 = dx0^2 + dx1^2 + dx2^2, no FMA. */
__device__ __forceinline__ double r2_task64(const double *xi, const double *xj, double s0, double s1, double s2) {
#pragma clang fp contract(off)
    double p0 = xi[0] - s0, p1 = xi[1] - s1, p2 = xi[2] - s2;
    double d0 = p0 - xj[0], d1 = p1 - xj[1], d2 = p2 - xj[2];
    return d0 * d0 + d1 * d1 + d2 * d2;
}

/* Reference r^2 of an exclusion (exclusion.c:139-147): i is the smaller id. */
__device__ __forceinline__ double r2_excl64(const double *xi, const double *xj, const int *li, const int *lj,
                                            const double *h) {
#pragma clang fp contract(off)
    double r2 = 0.0;
    for (int k = 0; k < 3; k++) {
        int sh = li[k] - lj[k];
        if (sh > 1)
            sh = -1;
        else if (sh < -1)
            sh = 1;
        double d = xi[k] - xj[k] + h[k] * sh;
        r2 += d * d;
    }
    return r2;
}

/* Table evaluation in FP32: e and f = (dE/dr)/r (potential_eval.h:67-104).
   hdr = (alpha0, alpha1, alpha2, bits(n | chunk0 << 9)). */
__device__ __forceinline__ void pot_eval32(const float4 hdr, const float4 *__restrict__ c4, float r2, float &e,
                                           float &f) {
    const float ir = __builtin_amdgcn_rsqf(r2);
    const float r = r2 * ir;
    const float fi = fmaxf(0.0f, hdr.x + r * (hdr.y + r * hdr.z));
    const unsigned int w = __float_as_uint(hdr.w);
    const int n = (int)(w & 511u);
    int ind = (int)fi;
    ind = ind > n ? n : ind;
    const float4 *c = c4 + 2 * ((int)(w >> 9) + ind);
    const float4 a = c[0], b = c[1];
    const float x = (r - a.x) * a.y;
    float ee = a.z * x + a.w;
    float eff = a.z;
    eff = eff * x + ee;
    ee = ee * x + b.x;
    eff = eff * x + ee;
    ee = ee * x + b.y;
    eff = eff * x + ee;
    ee = ee * x + b.z;
    eff = eff * x + ee;
    ee = ee * x + b.w;
    e = ee;
    f = eff * a.y * ir;
}

/* Buffer-resource loads: 32-bit byte offsets instead of 64-bit addresses
   (word 3 of the descriptor as for every gfx9 target); an offset past the
   declared size reads zeros. */
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, bytes, 0x00020000);
}

__device__ __forceinline__ float4 ld_f4(__amdgpu_buffer_rsrc_t r, int byte_off) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, 0);
    float4 out;
    __builtin_memcpy(&out, &v, sizeof(out));
    return out;
}

/* pot_eval32 for two pairs at once, without branches: both coefficient
   rows are requested before either polynomial is evaluated, so the two
   table lookups overlap.  A pair with use_* false (no hit, or no table for
   its types) reads interval 0 of the first table instead and returns
   e = f = 0. */
__device__ __forceinline__ void pot_eval32r2(const float4 ha, const float4 hb, bool use_a, bool use_b,
                                             __amdgpu_buffer_rsrc_t rc, float r2a, float r2b, float &ea,
                                             float &fa, float &eb, float &fb) {
    const float ira = __builtin_amdgcn_rsqf(r2a), irb = __builtin_amdgcn_rsqf(r2b);
    const float ra = r2a * ira, rb = r2b * irb;
    const unsigned int wa = use_a ? __float_as_uint(ha.w) : 0u;
    const unsigned int wb = use_b ? __float_as_uint(hb.w) : 0u;
    int ia = (int)fmaxf(0.0f, ha.x + ra * (ha.y + ra * ha.z));
    int ib = (int)fmaxf(0.0f, hb.x + rb * (hb.y + rb * hb.z));
    ia = ia > (int)(wa & 511u) ? (int)(wa & 511u) : ia;
    ib = ib > (int)(wb & 511u) ? (int)(wb & 511u) : ib;
    const int offa = 32 * ((int)(wa >> 9) + ia), offb = 32 * ((int)(wb >> 9) + ib);
    const float4 a0 = ld_f4(rc, offa), a1 = ld_f4(rc, offa + 16);
    const float4 b0 = ld_f4(rc, offb), b1 = ld_f4(rc, offb + 16);
    auto horner = [](float r, float ir, const float4 c0, const float4 c1, float &e, float &f) {
        const float x = (r - c0.x) * c0.y;
        float ee = c0.z * x + c0.w;
        float eff = c0.z;
        eff = eff * x + ee;
        ee = ee * x + c1.x;
        eff = eff * x + ee;
        ee = ee * x + c1.y;
        eff = eff * x + ee;
        ee = ee * x + c1.z;
        eff = eff * x + ee;
        ee = ee * x + c1.w;
        e = ee;
        f = eff * c0.y * ir;
    };
    float e1, f1, e2, f2;
    horner(ra, ira, a0, a1, e1, f1);
    horner(rb, irb, b0, b1, e2, f2);
    ea = use_a ? e1 : 0.f;
    fa = use_a ? f1 : 0.f;
    eb = use_b ? e2 : 0.f;
    fb = use_b ? f2 : 0.f;
}

/* A wave of the pair kernels shares its LDS with no other, and the LDS executes a
   wavefront's instructions in order: data written by one lane is visible to
   another lane's later read once this wave's LDS operations have completed.
   This waits for LDS only (lgkmcnt(0)) and keeps the compiler from moving
   memory accesses across it; unlike a workgroup barrier it does not drain
   outstanding global loads, so prefetches stay in flight. */
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

/* Packed staged record: key (16 bits) | index in cell (10 bits) | type (6 bits). */
__device__ __forceinline__ unsigned int rec_key(unsigned int w) { return w & 0xffffu; }
__device__ __forceinline__ int rec_idx(unsigned int w, int imask) { return (int)((w >> 16) & (unsigned int)imask); }
__device__ __forceinline__ int rec_type(unsigned int w, int tshift) { return (int)(w >> tshift); }

/* ------------------------------------------------------------ k_pack */

/* One wave per cell.  With dx, also the arrays of an upload from their one
   staging block: with six copies, a cleared flag and the id clearing, the
   device of a pass of 4,000 atoms was busy for 55 us before the sort; with one
   copy and this kernel, and the clearing while the host packs, 12.  (The map
   slot -> cell by a loop over the cell's slots in one thread: water, 125 atoms
   per cell, 19 us; now 5.) */
__global__ __launch_bounds__(256) void k_pack(int ncells, int nparts, const int2 *__restrict__ cnt_off,
                                              const double *__restrict__ x, const int *__restrict__ type,
                                              const int *__restrict__ id, float4 *__restrict__ xf,
                                              int *__restrict__ index_of_id, int *__restrict__ cell_of,
                                              double *__restrict__ dx, int *__restrict__ dtype, int *__restrict__ did,
                                              int *__restrict__ dcount, int *__restrict__ doffset,
                                              int2 *__restrict__ dcnt_off) {
    const int c = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (c >= ncells) return;
    const int2 co = cnt_off[c];
    if (dx && lane == 0) {
        dcount[c] = co.x;
        doffset[c] = co.y;
        dcnt_off[c] = co;
        if (c == 0) doffset[ncells] = nparts;
    }
    for (int k = lane; k < co.x; k += 64) {
        const int a = co.y + k, t = type[a], i = id[a];
        const double x0 = x[3 * (size_t)a], x1 = x[3 * (size_t)a + 1], x2 = x[3 * (size_t)a + 2];
        xf[a] = make_float4((float)x0, (float)x1, (float)x2, __int_as_float(t));
        index_of_id[i] = a;
        cell_of[a] = c;
        if (dx) {
            dx[3 * (size_t)a] = x0;
            dx[3 * (size_t)a + 1] = x1;
            dx[3 * (size_t)a + 2] = x2;
            dtype[a] = t;
            did[a] = i;
        }
    }
}

__global__ __launch_bounds__(256) void k_clear_ids(int nids, int *__restrict__ index_of_id) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nids) index_of_id[k] = -1;
}

__global__ __launch_bounds__(64) void k_clear_queue(int *__restrict__ queue) {
    if (threadIdx.x < MD_NQUEUE) queue[threadIdx.x] = 0;
}

/* ------------------------------------------------------------ k_sort */

#define MD_SORT_STACK 16

/* Descending sort of (index<<16 | key) words by key: the reference's
   quicksort with selection sort below 16 elements and an explicit stack
   (runner.c:110-174).  The partition and push order decide the order of
   equal keys, so they are kept as they are. */
template <typename A, typename S>
__device__ __forceinline__ void sort_desc_t(A a, int N, S st_lo, S st_hi, int *overflow) {
    int qpos = 0;
    st_lo[0] = 0;
    st_hi[0] = N - 1;
    while (qpos >= 0) {
        int lo = st_lo[qpos], hi = st_hi[qpos];
        qpos -= 1;
        if (hi - lo < 15) {
            for (int i = lo; i < hi; i++) {
                int imax = i;
                unsigned int kmax = a[i] & 0xffff;
                for (int j = i + 1; j <= hi; j++) {
                    unsigned int kj = a[j] & 0xffff;
                    if (kj > kmax) {
                        imax = j;
                        kmax = kj;
                    }
                }
                if (imax != i) {
                    unsigned int t = a[imax];
                    a[imax] = a[i];
                    a[i] = t;
                }
            }
        } else {
            unsigned int pivot = a[(lo + hi) / 2] & 0xffff;
            int i = lo, j = hi;
            while (i <= j) {
                while ((a[i] & 0xffff) > pivot) i++;
                while ((a[j] & 0xffff) < pivot) j--;
                if (i <= j) {
                    if (i < j) {
                        unsigned int t = a[i];
                        a[i] = a[j];
                        a[j] = t;
                    }
                    i += 1;
                    j -= 1;
                }
            }
            if (qpos + 2 >= MD_SORT_STACK) {
                *overflow = 1;
                return;
            }
            if (j > (lo + hi) / 2) {
                if (lo < j) { qpos++; st_lo[qpos] = lo; st_hi[qpos] = j; }
                if (i < hi) { qpos++; st_lo[qpos] = i; st_hi[qpos] = hi; }
            } else {
                if (i < hi) { qpos++; st_lo[qpos] = i; st_hi[qpos] = hi; }
                if (lo < j) { qpos++; st_lo[qpos] = lo; st_hi[qpos] = j; }
            }
        }
    }
}

__device__ void sort_desc(unsigned int *a, int N, int *overflow) {
    int st_lo[MD_SORT_STACK], st_hi[MD_SORT_STACK];
    sort_desc_t(a, N, st_lo, st_hi, overflow);
}

__constant__ double c_axis[39];

/* Projection key (runner_dosort.c:146-149): dscale*(bias + x.n) in FP64,
   left to right, no fused multiply-add, truncated to unsigned. */
__device__ __forceinline__ unsigned int sort_key(const double *x, int sid, double dscale, double bias) {
#pragma clang fp contract(off)
    double v = dscale * (bias + x[0] * c_axis[3 * sid] + x[1] * c_axis[3 * sid + 1] + x[2] * c_axis[3 * sid + 2]);
    return (unsigned int)v;
}

__global__ __launch_bounds__(256) void k_sort(struct nb_params P, const int *__restrict__ count,
                                              const int *__restrict__ offset,
                                              const unsigned int *__restrict__ sortflags,
                                              const double *__restrict__ x, unsigned int *__restrict__ sortlist,
                                              unsigned short *__restrict__ keyof,
                                              unsigned short *__restrict__ kminmax, int *__restrict__ flag) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    int cid = t / 13, sid = t - 13 * (t / 13);
    if (cid >= P.ncells) return;
    if (!((sortflags[cid] >> sid) & 1u)) return;
    int n = count[cid];
    if (n == 0) return;
    int off = offset[cid];
    const size_t seg = 13 * (size_t)off + (size_t)sid * n;
    unsigned int *list = sortlist + seg;
    for (int i = 0; i < n; i++) {
        unsigned int key = sort_key(&x[3 * (size_t)(off + i)], sid, P.dscale, P.bias);
        list[i] = ((unsigned int)i << 16) | key;
        keyof[(size_t)sid * P.nparts + off + i] = (unsigned short)key;
    }
    sort_desc(list, n, flag);
    kminmax[26 * (size_t)cid + sid] = (unsigned short)(list[0] & 0xffffu);
    kminmax[26 * (size_t)cid + 13 + sid] = (unsigned short)(list[n - 1] & 0xffffu);
}

/* The quicksort of sort_desc_t, run by a whole wave on one LDS list with the
   same result, element for element.
   - Segments below 16 elements (selection sort): each step takes the first
     maximal key of the rest, the max of key << 6 | (63 - index) over the
     leaf's lanes (a DPP reduction within the first row of 16 lanes), and
     swaps it to the front with lane reads.
   - Partition (pivot p = middle key): the serial scan's k-th swap pairs the
     k-th element from the left with key <= p (ltab[k]) and the k-th from the
     right with key >= p (rtab[k]), for k = 1..K while ltab[k] <= rtab[k];
     both tables come from ballots and prefix counts.  The scan then stops
     with i = ltab[K] + 1, j = rtab[K] - 1 if these have crossed, else at
     i = min(ltab[K+1], rtab[K]), j = max(rtab[K+1], ltab[K]) (the swapped
     elements stop the pointers), without a further swap.
   The stack (same pushes and overflow test as sort_desc_t) lives in LDS and
   is written by lane 0.  ltab / rtab: maxn + 1 entries each. */

/* Largest value over lanes 0..15, wave-uniform: four DPP row shifts (lane l
   takes the max of lanes l-1, l-2..l-3, l-4..l-7, l-8..l-15 of its row;
   lanes shifted in from outside the row read 0), then lane 15. */
__device__ __forceinline__ unsigned int row0_max_u32(unsigned int v) {
    unsigned int u;
    u = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true); /* row_shr:1 */
    v = u > v ? u : v;
    u = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true); /* row_shr:2 */
    v = u > v ? u : v;
    u = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true); /* row_shr:4 */
    v = u > v ? u : v;
    u = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true); /* row_shr:8 */
    v = u > v ? u : v;
    return (unsigned int)__builtin_amdgcn_readlane((int)v, 15);
}

/* One partition step of sort_desc_t on a[lo..hi] (hi - lo >= 15, at most
   64 R elements) by a whole wave, pivot p = the middle key; returns the
   scan's final (i, j).  ltab / rtab: hi - lo + 2 entries each. */
template <int R>
__device__ __forceinline__ int2 part_wave(unsigned int *a, int lo, int hi, unsigned short *ltab,
                                          unsigned short *rtab, int lane) {
    const unsigned long long below = (1ull << lane) - 1ull;
    const unsigned int p = a[(lo + hi) / 2] & 0xffffu;
    unsigned int wv[R];
    bool isl[R], isr[R];
    int nR = 0;
    for (int r = 0; r < R; r++) {
        const int x = lo + lane + 64 * r;
        const bool valid = x <= hi;
        wv[r] = valid ? a[x] : 0u;
        isl[r] = valid && (wv[r] & 0xffffu) <= p;
        isr[r] = valid && (wv[r] & 0xffffu) >= p;
        nR += __builtin_popcountll(__builtin_amdgcn_ballot_w64(isr[r]));
    }
    int cl = 0, cr = 0;
    for (int r = 0; r < R; r++) {
        const int x = lo + lane + 64 * r;
        const unsigned long long ml = __builtin_amdgcn_ballot_w64(isl[r]);
        const unsigned long long mr = __builtin_amdgcn_ballot_w64(isr[r]);
        if (isl[r]) ltab[cl + __builtin_popcountll(ml & below) + 1] = (unsigned short)x;
        if (isr[r]) rtab[nR - cr - __builtin_popcountll(mr & below)] = (unsigned short)x;
        cl += __builtin_popcountll(ml);
        cr += __builtin_popcountll(mr);
    }
    const int nL = cl, m = nL < nR ? nL : nR;
    wave_lds_sync();
    int K = 0;
    int li[R], ri[R];
    for (int r = 0; r < R; r++) {
        const int k = 1 + lane + 64 * r;
        li[r] = k <= m ? ltab[k] : 0;
        ri[r] = k <= m ? rtab[k] : 0;
        K += __builtin_popcountll(__builtin_amdgcn_ballot_w64(k <= m && li[r] <= ri[r]));
    }
    /* the K swaps touch distinct elements, each lane its own */
    for (int r = 0; r < R; r++) {
        const int k = 1 + lane + 64 * r;
        if (k <= K && li[r] < ri[r]) {
            const unsigned int va = a[li[r]], vb = a[ri[r]];
            a[li[r]] = vb;
            a[ri[r]] = va;
        }
    }
    wave_lds_sync();
    const int lK = ltab[K], rK = rtab[K];
    int i = lK + 1, j = rK - 1;
    if (i <= j) {
        const int l1 = K + 1 <= nL ? (int)ltab[K + 1] : 1 << 30;
        const int r1 = K + 1 <= nR ? (int)rtab[K + 1] : -(1 << 30);
        i = l1 < rK ? l1 : rK;
        j = r1 > lK ? r1 : lK;
    }
    return make_int2(i, j);
}

/* Two partition steps of part_wave at once, one per half wave: lanes 32h..
   32h+31 partition a[lo..hi] (16 to 32 elements; lo > hi leaves the half
   idle) with their half's tables ltab / rtab (33 entries each); lo, hi,
   ltab and rtab are the lane's half's.  Returns the half's final (i, j). */
__device__ __forceinline__ int2 part_wave2(unsigned int *a, int lo, int hi, unsigned short *ltab,
                                           unsigned short *rtab, int lane) {
    const unsigned long long half = (lane & 32) ? 0xffffffff00000000ull : 0x00000000ffffffffull;
    const unsigned long long below = ((1ull << lane) - 1ull) & half;
    const int x = lo + (lane & 31);
    const bool valid = x <= hi;
    const unsigned int p = a[(lo + hi) >> 1] & 0xffffu;
    const unsigned int w = valid ? a[x] : 0u;
    const bool isl = valid && (w & 0xffffu) <= p, isr = valid && (w & 0xffffu) >= p;
    const unsigned long long ml = __builtin_amdgcn_ballot_w64(isl) & half;
    const unsigned long long mr = __builtin_amdgcn_ballot_w64(isr) & half;
    const int nL = __builtin_popcountll(ml), nR = __builtin_popcountll(mr);
    if (isl) ltab[__builtin_popcountll(ml & below) + 1] = (unsigned short)x;
    if (isr) rtab[nR - __builtin_popcountll(mr & below)] = (unsigned short)x;
    const int m = nL < nR ? nL : nR;
    wave_lds_sync();
    const int k = 1 + (lane & 31);
    const int li = k <= m ? ltab[k] : 0, ri = k <= m ? rtab[k] : 0;
    const int K = __builtin_popcountll(__builtin_amdgcn_ballot_w64(k <= m && li <= ri) & half);
    if (k <= K && li < ri) {
        const unsigned int va = a[li], vb = a[ri];
        a[li] = vb;
        a[ri] = va;
    }
    wave_lds_sync();
    const int lK = ltab[K], rK = rtab[K];
    int i = lK + 1, j = rK - 1;
    if (i <= j) {
        const int l1 = K + 1 <= nL ? (int)ltab[K + 1] : 1 << 30;
        const int r1 = K + 1 <= nR ? (int)rtab[K + 1] : -(1 << 30);
        i = l1 < rK ? l1 : rK;
        j = r1 > lK ? r1 : lK;
    }
    return make_int2(i, j);
}

/* R: up to 64 R elements per partition. */
template <int R>
__device__ void sort_desc_wave(unsigned int *a, int N, int *st_lo, int *st_hi, unsigned short *ltab,
                               unsigned short *rtab, int *overflow, int lane) {
    int q = 0;
    if (lane == 0) {
        st_lo[0] = 0;
        st_hi[0] = N - 1;
    }
    wave_lds_sync();
    int pops = 0;
    while (q >= 0) {
        const int lo = st_lo[q], hi = st_hi[q];
        q -= 1;
        /* the serial sort pops at most 2N segments, all inside [0, N): anything
           else is reported as a sort failure instead of looping on */
        if (++pops > 2 * N + 2 || lo < 0 || hi >= N || lo > hi) {
            if (lane == 0) *overflow = 1;
            return;
        }
        if (hi - lo < 15) {
            const int len = hi - lo + 1;
            unsigned int w = lane < len ? a[lo + lane] : 0u;
            /* the leaf lies in lanes 0..14: a row-0 max and lane reads */
            for (int i = 0; i < len - 1; i++) {
                const unsigned int pk =
                    (lane >= i && lane < len) ? (((w & 0xffffu) << 6) | (unsigned int)(63 - lane)) : 0u;
                const int im = 63 - (int)(row0_max_u32(pk) & 63u);
                const unsigned int wi = (unsigned int)__builtin_amdgcn_readlane((int)w, i);
                const unsigned int wm = (unsigned int)__builtin_amdgcn_readlane((int)w, im);
                if (lane == i)
                    w = wm;
                else if (lane == im)
                    w = wi;
            }
            if (lane < len) a[lo + lane] = w;
            wave_lds_sync();
            continue;
        }
        const int2 ij = part_wave<R>(a, lo, hi, ltab, rtab, lane);
        const int i = ij.x, j = ij.y;
        if (q + 2 >= MD_SORT_STACK) {
            if (lane == 0) *overflow = 1;
            return;
        }
        const int mid = (lo + hi) / 2;
        const bool left_first = j > mid;
        /* pushes in sort_desc_t's order: [lo, j] then [i, hi] when j > mid */
        const bool pa = left_first ? lo < j : i < hi, pb = left_first ? i < hi : lo < j;
        const int alo = left_first ? lo : i, ahi = left_first ? j : hi;
        const int blo = left_first ? i : lo, bhi = left_first ? hi : j;
        if (pa) {
            q++;
            if (lane == 0) {
                st_lo[q] = alo;
                st_hi[q] = ahi;
            }
        }
        if (pb) {
            q++;
            if (lane == 0) {
                st_lo[q] = blo;
                st_hi[q] = bhi;
            }
        }
        wave_lds_sync();
    }
}

/* Largest value over the lane's row of 16 lanes, in every lane of the row:
   max with the row rotated by 1, 2, 4 and 8 lanes (DPP row_ror). */
__device__ __forceinline__ unsigned int row_max_all(unsigned int v) {
    unsigned int u;
    u = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xf, 0xf, false); /* row_ror:1 */
    v = u > v ? u : v;
    u = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, false); /* row_ror:2 */
    v = u > v ? u : v;
    u = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false); /* row_ror:4 */
    v = u > v ? u : v;
    u = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false); /* row_ror:8 */
    v = u > v ? u : v;
    return v;
}

/* sort_desc_t on every list l of a cell with bit l of tm set (the lists of
   n <= 64 words at a + l * n), by one wave, with the same result.  A
   partition or a selection sort only touches its own segment, so the
   segments are taken in any order:
   - segments of 33 or more elements are partitioned by the whole wave
     (part_wave), those of 16 to 32 two at a time, one per half wave
     (part_wave2); their parts are queued again;
   - segments of 2..15 elements (the serial sort's selection-sort leaves)
     are sorted four at a time, one per row of 16 lanes: each step takes the
     first maximal key of the rest, the row max of
     key << 12 | (15 - row lane) << 8 | particle index
     (particle indices stay below 256), and swaps it with the step's lane,
     whose word every lane of the row gets from a second row max.
   Segment queues: segq (416 words: segments above 32 elements from the
   front, 16 to 32 from the middle) and leafq (leafcap words), lo | hi << 16
   in list-array positions.  Partition tables: tb, 136 entries.  Reports a
   queue overflow or a runaway loop in *overflow (the host turns it into a
   sort failure). */
__device__ void sort_lists_wave(unsigned int *a, int n, unsigned int tm, unsigned int *segq, unsigned int *leafq,
                                int leafcap, unsigned short *tb, unsigned int *__restrict__ out, int *overflow,
                                int lane) {
    constexpr int QHALF = 13 * MD_SORT_STACK;
    int nbig = 0, nsmall = 0, nl = 0;
    bool bad = false;
    auto push = [&](int lo, int hi) {
        const unsigned int w = (unsigned int)lo | ((unsigned int)hi << 16);
        if (hi - lo >= 32) {
            if (nbig < QHALF) {
                if (lane == 0) segq[nbig] = w;
                nbig++;
            } else
                bad = true;
        } else if (hi - lo >= 15) {
            if (nsmall < QHALF) {
                if (lane == 0) segq[QHALF + nsmall] = w;
                nsmall++;
            } else
                bad = true;
        } else if (hi > lo) {
            if (nl < leafcap) {
                if (lane == 0) leafq[nl] = w;
                nl++;
            } else
                bad = true;
        }
    };
    /* Only the marked elements (keys that others of their list share) are
       written from here on; rank placed the others.  A segment without a
       marked element is dropped.  With one, that element's place is the
       segment's start plus the number of greater keys in it (the others'
       keys differ from its own).  With more, the segment is queued, and its
       leaves write all of their elements in the end. */
    auto place = [&](int lo, int hi) {
        const int x = lo + lane;
        const bool valid = x <= hi;
        const unsigned int w = valid ? a[x] : 0u;
        const unsigned long long mk = __builtin_amdgcn_ballot_w64(valid && (w >> 31) != 0u);
        if (mk == 0ull) return;
        if ((mk & (mk - 1ull)) == 0ull) {
            const unsigned int wt = (unsigned int)__builtin_amdgcn_readlane((int)w, (int)__builtin_ctzll(mk));
            const int g = __builtin_popcountll(__builtin_amdgcn_ballot_w64(valid && (w & 0xffffu) > (wt & 0xffffu)));
            if (lane == 0) out[lo + g] = wt & 0x7fffffffu;
            return;
        }
        push(lo, hi);
    };
    /* the elements a partition leaves between its two parts are in place */
    auto settle = [&](int lo, int hi) {
        const int x = lo + lane;
        if (x <= hi) {
            const unsigned int w = a[x];
            if ((w >> 31) != 0u) out[x] = w & 0x7fffffffu;
        }
    };
    for (unsigned int t = tm; t; t &= t - 1) {
        const int l = __builtin_ctz(t);
        push(l * n, l * n + n - 1);
    }
    wave_lds_sync();
    /* each partition splits a segment into two strictly smaller ones */
    int parts = 0;
    while ((nbig > 0 || nsmall > 0) && !bad) {
        if (nbig > 0) {
            nbig--;
            const unsigned int sg = segq[nbig];
            const int lo = (int)(sg & 0xffffu), hi = (int)(sg >> 16);
            if (++parts > 13 * n) {
                bad = true;
                break;
            }
            const int2 ij = part_wave<1>(a, lo, hi, tb, tb + 68, lane);
            wave_lds_sync();
            place(lo, ij.y);
            place(ij.x, hi);
            settle(ij.y + 1, ij.x - 1);
        } else {
            const bool two = nsmall >= 2;
            const unsigned int s0 = segq[QHALF + nsmall - 1];
            const unsigned int s1 = two ? segq[QHALF + nsmall - 2] : 1u;
            nsmall -= two ? 2 : 1;
            parts += two ? 2 : 1;
            if (parts > 13 * n) {
                bad = true;
                break;
            }
            const unsigned int sm = (lane & 32) ? s1 : s0;
            const int lo = (int)(sm & 0xffffu), hi = (int)(sm >> 16);
            unsigned short *lt = tb + ((lane & 32) ? 68 : 0);
            const int2 ij = part_wave2(a, lo, hi, lt, lt + 34, lane);
            const int i0 = __builtin_amdgcn_readlane(ij.x, 0), j0 = __builtin_amdgcn_readlane(ij.y, 0);
            const int i1 = __builtin_amdgcn_readlane(ij.x, 32), j1 = __builtin_amdgcn_readlane(ij.y, 32);
            wave_lds_sync();
            place((int)(s0 & 0xffffu), j0);
            place(i0, (int)(s0 >> 16));
            settle(j0 + 1, i0 - 1);
            if (two) {
                place((int)(s1 & 0xffffu), j1);
                place(i1, (int)(s1 >> 16));
                settle(j1 + 1, i1 - 1);
            }
        }
        wave_lds_sync();
    }
    if (bad) {
        if (lane == 0) *overflow = 1;
        return;
    }
    const int row = lane >> 4, lr = lane & 15;
    for (int b = 0; b < nl; b += 4) {
        const bool has = b + row < nl;
        const unsigned int sg = has ? leafq[b + row] : 0u;
        const int lo = (int)(sg & 0xffffu), len = has ? (int)(sg >> 16) - lo + 1 : 0;
        unsigned int w = lr < len ? a[lo + lr] : 0u;
        int steps = __builtin_amdgcn_readlane(len, 0);
        steps = max(steps, __builtin_amdgcn_readlane(len, 16));
        steps = max(steps, __builtin_amdgcn_readlane(len, 32));
        steps = max(steps, __builtin_amdgcn_readlane(len, 48));
        for (int i = 0; i < steps - 1; i++) {
            const bool in = lr >= i && lr < len;
            const unsigned int pk =
                in ? ((w & 0xffffu) << 12) | ((unsigned int)(15 - lr) << 8) | ((w >> 16) & 0xffu) : 0u;
            const unsigned int mx = row_max_all(pk);
            const unsigned int wi = row_max_all(lr == i ? w : 0u);
            const int im = 15 - (int)((mx >> 8) & 15u);
            const unsigned int wm = ((mx & 0xffu) << 16) | (mx >> 12);
            if (i < len - 1) {
                if (lr == i)
                    w = wm;
                else if (lr == im)
                    w = wi;
            }
        }
        if (lr < len) out[lo + lr] = w & 0x7fffffffu;
    }
}

/* Sort by rank: one workgroup per cell, all 13 directions at once.  A key that no
   other particle of its list shares has exactly (number of greater keys)
   particles before it in any descending order, the reference's quicksort
   included, so those particles are placed by counting.  Only the order of
   equal keys depends on the quicksort's partitions: a list with equal keys
   is sorted again with the reference's algorithm (runner.c:110-174), in LDS,
   and written whole.  Cells of at most MD_SORT_ONEWAVE_MAX particles, more
   than MD_SORT_FEW of them, get one wave, which sorts all such lists of its cell together (sort_lists_wave);
   larger or few cells get 13 waves, wave l sorting list l (sort_desc_wave).  For
   cells of at most MD_SORT_LDS_MAX particles.  LDS: 3 * maxn positions,
   13 * maxn list words, 13 quicksort stacks, 13 pairs of partition tables
   and 136 more entries (the one-wave sort keeps its segment queues there). */
/* Cells up to which every cell gets 13 waves: a cell's sorts are one serial
   chain, which 13 waves shorten while the device has room for them.  us with
   one wave and with 13: argon 64 cells 37, 27; 125 cells 34, 29 (mixture, with
   more equal keys, 50, 33); 512 cells 36, 33; 1331 cells 37, 45; 10648 cells
   69, 177. */
#define MD_SORT_FEW 768
__global__ __launch_bounds__(1024) void k_sort_rank(struct nb_params P, const int *__restrict__ count,
                                                  const int *__restrict__ offset,
                                                  const unsigned int *__restrict__ sortflags,
                                                  const double *__restrict__ x, unsigned int *__restrict__ sortlist,
                                                  unsigned short *__restrict__ keyof,
                                                  unsigned short *__restrict__ kminmax, int *__restrict__ flag,
                                                  int maxn) {
    extern __shared__ double sh_rank[];
    double *xs = sh_rank;
    unsigned int *lists = (unsigned int *)(sh_rank + 3 * maxn);
    int *stk = (int *)(lists + 13 * maxn);
    unsigned short *tabs = (unsigned short *)(stk + 13 * 2 * MD_SORT_STACK);
    __shared__ int tie[13];
    const int c = blockIdx.x, lane = threadIdx.x;
    const int n = count[c];
    if (n == 0 || n > maxn) return; /* a cell that outgrew the launch: the caller repeats it */
    const unsigned int fl = sortflags[c];
    const int off = offset[c];
    const float rn = 1.0f / (float)n;
    if (lane < 13) tie[lane] = 0;
    for (int k = lane; k < 3 * n; k += (int)blockDim.x) xs[k] = x[3 * (size_t)off + k];
    __syncthreads();
    for (int t = lane; t < 13 * n; t += (int)blockDim.x) {
        const int sid = (int)(((float)t + 0.5f) * rn), i = t - sid * n; /* t / n */
        if (!((fl >> sid) & 1u)) continue;
        const unsigned int key = sort_key(&xs[3 * i], sid, P.dscale, P.bias);
        lists[sid * n + i] = ((unsigned int)i << 16) | key;
        keyof[(size_t)sid * P.nparts + off + i] = (unsigned short)key;
    }
    __syncthreads();
    unsigned int *out = sortlist + 13 * (size_t)off;
    for (int t = lane; t < 13 * n; t += (int)blockDim.x) {
        const int sid = (int)(((float)t + 0.5f) * rn), i = t - sid * n; /* t / n */
        if (!((fl >> sid) & 1u)) continue;
        const unsigned int *L = lists + sid * n;
        const unsigned int w = L[i], key = w & 0xffffu;
        int gt = 0, eq = 0;
        for (int j = 0; j < n; j++) {
            const unsigned int kj = L[j] & 0xffffu;
            gt += kj > key;
            eq += kj == key;
        }
        /* largest and smallest key (particles that share one write the same) */
        if (gt == 0) kminmax[26 * (size_t)c + sid] = (unsigned short)key;
        if (gt + eq == n) kminmax[26 * (size_t)c + 13 + sid] = (unsigned short)key;
        if (eq == 1) {
            out[sid * n + gt] = w;
        } else {
            tie[sid] = 1;
            lists[sid * n + i] = w | 0x80000000u; /* marked: shares its key */
        }
    }
    __syncthreads();
    /* Lists with a repeated key: the reference's quicksort, by 13 waves one
       list each, or by the cell's one wave all lists together. */
    const int wave = lane >> 6, nwave = (int)blockDim.x >> 6, wl = lane & 63;
    if (nwave > 1) {
        for (int l = wave; l < 13; l += nwave) {
            if (!((fl >> l) & 1u) || !tie[l]) continue;
            unsigned int *L = lists + l * n;
            int *st = stk + l * 2 * MD_SORT_STACK;
            unsigned short *tb = tabs + (size_t)l * 2 * (maxn + 1);
            if (n <= 192)
                sort_desc_wave<3>(L, n, st, st + MD_SORT_STACK, tb, tb + maxn + 1, flag, wl);
            else
                sort_desc_wave<8>(L, n, st, st + MD_SORT_STACK, tb, tb + maxn + 1, flag, wl);
            for (int i = wl; i < n; i += 64) out[l * n + i] = L[i] & 0x7fffffffu;
        }
    } else {
        unsigned int tm = 0;
        for (int l = 0; l < 13; l++) tm |= (unsigned int)(tie[l] != 0) << l;
        tm &= fl;
        if (tm) {
            /* segment queue: the stacks' space; partition tables and leaf
               queue: the partition tables' space (26 (maxn + 1) + 136
               entries) */
            sort_lists_wave(lists, n, tm, (unsigned int *)stk, (unsigned int *)(tabs + 136), 13 * (maxn + 1), tabs,
                            out, flag, wl);
        }
    }
}

/* ------------------------------------------------------------ k_nonbond */

/* Window bound of a pair task (runner_dopair.c:428): 2 + dscale (cutoff +
   maxdx_i + maxdx_j) in FP64, left to right, no contraction, truncated; i
   and j in task order. */
__device__ __forceinline__ int pair_dmaxdist(double dscale, double cutoff, double mi, double mj) {
#pragma clang fp contract(off)
    return (int)(2 + dscale * (cutoff + mi + mj));
}

struct nb_out {
    float4 *fhi, *flo;
    double *cell_acc;
    unsigned long long *cell_cnt;
    /* half shell: forces on the visited atoms, jpart[slot][atom][3], slot 0 for
       the self task and 1.. for the atom's cell's incoming tasks */
    float *jpart;
    /* split owners (nsplit > 1): group g's forces on atom a at [g * nparts + a] */
    float4 *phi, *plo;
};

/* True if p holds on any lane (scalar test of the wave's ballot mask). */
__device__ __forceinline__ bool wave_any(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0; }

/* Compile-time tag of a visit kind (self / owner is i / owner is j). */
template <int V>
struct visit_kind {
    static constexpr int value = V;
};

/* Exclusive prefix sum of v over the wave. */
__device__ __forceinline__ int wave_excl_scan(int v, int lane) {
    int x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    return x - v;
}

/* Evaluate the dense pair list [0, T) with the network, 16 pairs per tile;
   f = (dE/dr)/r and e of pair q go to dn_f[q], dn_e[q].  dE/dr is the
   network's own r-derivative, so the forces conserve the energies reported.
   The list goes in chunks of 64 pairs: lane l first computes the inputs of
   pair c + l (square root and four divisions, done once per pair instead of
   in all four lanes that carry its column of a tile) and parks them in the
   list's own slots (rn in dn_r2, irn in dn_f, d irn / dr in dn_e; d rn / dr
   stays in lane l's register), then the chunk's tiles run, each leaving y
   (without the output bias) and dy/dr of its pairs in dn_f and dn_e, and
   lane l turns those of pair c + l into its energy and force.  dn_r2 does not keep r^2.  w1s: the wave's
   LDS copy of layer 1's weights (read there, every tile's layer-1 loads
   leave the vector memory path: 40.9 -> 39.9 ms on the 1M mixture).  All
   64 lanes must call this together (T is wave-uniform). */
__device__ __forceinline__ void mlp_dense_eval(const struct mlp_net &N, const float *w1s, float *dn_r2, const int *dn_p,
                                               float *dn_f, float *dn_e, int T, int lane) {
    /* layer 2's operands stay in registers for the whole list: reloading
       them per tile cost 13 % of the 1M mixture's surrogate pass */
    mlp_bf16x8 w2r[8];
    float4 b2r[4];
    mlp_load_layer2(N, lane, w2r, b2r);
    for (int c = 0; c < T; c += 64) {
        const int q = c + lane;
        float r = 1.0f, drn = 0.0f;
        if (q < T) {
            r = sqrtf(dn_r2[q]);
            float rn, irn, dirn;
            mlp_inputs(N.sc[dn_p[q]], r, rn, irn, drn, dirn);
            dn_r2[q] = rn;
            dn_f[q] = irn;
            dn_e[q] = dirn;
        }
        wave_lds_sync();
        const int nt = min(4, (T - c + 15) >> 4);
        for (int t = 0; t < nt; t++) {
            const int qt = c + 16 * t + (lane & 15);
            const int qv = qt < T ? qt : T - 1;
            const float drt = __shfl(drn, qv - c);
            /* keep the network operands' loads inside the loop: hoisting them
               out keeps ~100 registers live through the whole pair kernel */
            asm volatile("" ::: "memory");
            float y, yd;
            mlp_infer16_reg(N, w1s, w2r, b2r, dn_r2[qv], dn_f[qv], drt, dn_e[qv], dn_p[qv], lane, y, yd);
            if (lane < 16 && qt < T) {
                dn_f[qt] = y;
                dn_e[qt] = yd;
            }
        }
        wave_lds_sync();
        if (q < T) {
            const int p = dn_p[q];
            float e, dedr;
            mlp_energy_force(N.sc[p], N.shift[p], r, dn_f[q] + N.b3[p], dn_e[q], e, dedr);
            dn_f[q] = dedr / r;
            dn_e[q] = e;
        }
    }
}

#define MD_SPLIT_ITEMS_PER_CU 32 /* surrogate: work items per CU below which owners are split */
#define MD_SPLIT_MAX 8           /* surrogate: at most this many neighbour groups per owner cell */
#define MD_PAIR_ITEMS_PER_CU 12  /* k_pair: work items per CU that owners are split up to */
#define MD_PAIR_SPLIT_MAX 32     /* k_pair: at most this many groups (of two entries at least) */
#define MD_PAIR_R64_MEAN 32      /* atoms per cell above which k_pair takes 64 owner atoms at a time */
#define MD_WALK_CELLS 16384 /* k_pair, projected window: cells from which walk_cap is 28 (pair_tile.h) */
#define MD_HCAP 32     /* table mode: hits buffered per lane before they are evaluated */
#define MD_HCAP_WIDE 28 /* the same in the 5-wave build: its LDS then allows 20 waves per CU */
#define MD_HCAP_MLP 8  /* MLP mode: hits per lane per compaction round */
#define MD_XCAP_MLP 8  /* MLP mode: excluded partners per lane per round */

/* The body of the kernels that walk the sorted windows, for two modes:
   MLP = false  (half shell only) every hit is evaluated from the FP32 tables
                by its lane;
   MLP = true   hits below the species pair's r_lo (or without a network)
                are evaluated from the tables, the others are compacted
                wave-wide into a dense LDS pair list and evaluated by the
                surrogate network 16 pairs per MFMA tile; each lane then
                adds its own contiguous run of results in order, so the
                result stays deterministic.  Excluded pairs take the same
                route, so a pair and its exclusion cancel exactly. */
template <bool MLP, bool HALF, int HC = MD_HCAP>
__device__ __forceinline__ void nonbond_body(
    unsigned char *smem, struct nb_params P, const int2 *__restrict__ cnt_off, const int4 *__restrict__ nbr,
    const int *__restrict__ nbr_off, const float4 *__restrict__ nbs, const double *__restrict__ origin,
    const int *__restrict__ loc,
    const float4 *__restrict__ xf, const double *__restrict__ x64, const int *__restrict__ pid,
    const unsigned int *__restrict__ sortlist, const unsigned short *__restrict__ keyof,
    const float4 *__restrict__ ptab, const float4 *__restrict__ coeffs4, const int *__restrict__ excl_off,
    const int *__restrict__ excl_list, const int *__restrict__ index_of_id, const int *__restrict__ cell_of,
    struct nb_out O, int *__restrict__ queue, const struct mlp_net &N, const int *__restrict__ ptype) {
    constexpr int HCAP = MLP ? MD_HCAP_MLP : HC;
    float4 *raw = (float4 *)smem;                                        /* [64]        */
    unsigned short *own_key = (unsigned short *)(smem + P.lds_own_key);  /* [13*64]     */
    int *kfl = (int *)(smem + P.lds_kfl);                                /* [26]        */
    float4 *stage = (float4 *)(smem + P.lds_stage);                      /* [maxn]      */
    unsigned short *hitl = (unsigned short *)(smem + P.lds_hit);         /* [HCAP*64]   */
    /* Dense pair list (r^2, species pair) and its results (f, e),
       and the excluded partners of each lane. */
    float *dn_r2 = (float *)(smem + P.lds_dense);                        /* [HCAP*64]   */
    int *dn_p = (int *)(smem + P.lds_dense + 4 * 64 * MD_HCAP_MLP);
    float *dn_f = (float *)(smem + P.lds_dense + 8 * 64 * MD_HCAP_MLP);
    float *dn_e = (float *)(smem + P.lds_dense + 12 * 64 * MD_HCAP_MLP);
    int *exb = (int *)(smem + P.lds_dense + 16 * 64 * MD_HCAP_MLP);      /* [XCAP*64]   */
    /* layer 1's weights [64][2], copied once per wave */
    float *w1s = (float *)(smem + P.lds_dense + 16 * 64 * MD_HCAP_MLP + 4 * 64 * MD_XCAP_MLP);
    /* half-shell mode: forces on the visited cell's records, 3 per record */
    float *jf = (float *)(smem + P.lds_jf);                              /* [4][3*maxn] */
    const int lane = threadIdx.x;
    const int mt = P.max_type;
    if constexpr (MLP) {
        w1s[lane] = N.w1[lane];
        w1s[64 + lane] = N.w1[64 + lane];
        wave_lds_sync();
    }
    /* A candidate beyond rc2hi is out.  rc2hi is rc2f + band rounded down:
       then every kept r2 has r2 - rc2f <= band exactly (the difference of
       two floats this close is exact), so the evaluation's band test
       catches every kept pair that is not certainly inside, and FP64
       decides it.  (Rounded up, a pair at r2 = rc2hi could slip past both.) */
    float rc2hi = P.rc2f + P.band;
    if (rc2hi - P.rc2f > P.band) rc2hi = __uint_as_float(__float_as_uint(rc2hi) - 1u);
    const __amdgpu_buffer_rsrc_t rs_ptab = make_rsrc(ptab, P.ptab_bytes);
    const __amdgpu_buffer_rsrc_t rs_coef = make_rsrc(coeffs4, P.coef_bytes);

    if (HALF) /* the visited cell's force copies start at zero; each visit's write-out clears them again */
        for (int z = lane; z < 4 * 3 * P.maxn; z += 64) jf[z] = 0.f;
    /* Work items: (owner cell, neighbour group), nsplit groups per cell. */
    const int nitems = P.ncells * P.nsplit;
    int q = blockIdx.x % MD_NQUEUE, tried = 0;
    while (tried < MD_NQUEUE) {
        const int lo_q = (int)(((long long)q * nitems) / MD_NQUEUE);
        const int hi_q = (int)(((long long)(q + 1) * nitems) / MD_NQUEUE);
        int it = 0;
        if (lane == 0) it = atomicAdd(&queue[q], 1);
        it = __shfl(it, 0);
        if (lo_q + it >= hi_q) {
            q = (q + 1) % MD_NQUEUE;
            tried++;
            continue;
        }
        /* Wave-uniform from here: the neighbour list is read with scalar loads. */
        const int item = __builtin_amdgcn_readfirstlane(lo_q + it);
        const int ci = item / P.nsplit, grp = item - ci * P.nsplit;
        const int c = P.order[ci];
        const int2 co_c = cnt_off[c];
        const int nc = co_c.x, offc = co_c.y;
        if (nc == 0) {
            /* An empty cell still owns its slots of the per-item sums. */
            if (lane < 3) {
                O.cell_acc[3 * item + lane] = 0.0;
                O.cell_cnt[3 * item + lane] = 0ull;
            }
            continue;
        }
        const double oc0 = origin[3 * c], oc1 = origin[3 * c + 1], oc2 = origin[3 * c + 2];
        /* this item's share of the owner's neighbour entries */
        const int kc = nbr_off[c], nall = nbr_off[c + 1] - kc;
        const int k0 = kc + (grp * nall) / P.nsplit, nn = kc + ((grp + 1) * nall) / P.nsplit - k0;

        /* Owner metadata: first/last key per direction. */
        wave_lds_sync();
        if (lane < 26) {
            const int sid = lane % 13;
            kfl[lane] = (int)(sortlist[13 * (size_t)offc + (size_t)sid * nc + (lane < 13 ? 0 : nc - 1)] & 0xffffu);
        }

        const int nchunk = (nc + 63) / 64;
        for (int ch = 0; ch < nchunk; ch++) {
            const int i0 = (int)(((long long)ch * nc) / nchunk);
            const int nsub = (int)(((long long)(ch + 1) * nc) / nchunk) - i0;
            /* Lane = (atom il, partition part): every lane works.  Atom il has
               NPi = (63 - il) / nsub + 1 partitions (lanes il, il + nsub, ...),
               each walking every NPi-th record of the atom's window. */
            const int il = lane % nsub, part = lane / nsub;
            const int NPi = (63 - il) / nsub + 1;
            const int NPmax = 63 / nsub + 1;
            const bool active = part < NPi;
            const int myidx = i0 + il; /* storage index in the owner cell */
            const int a = offc + myidx;
            const float4 xi = xf[a];
            const int ti = __float_as_int(xi.w);

            wave_lds_sync();
            if (lane < nsub)
                for (int sid = 0; sid < 13; sid++)
                    own_key[sid * 64 + lane] = keyof[(size_t)sid * P.nparts + offc + i0 + lane];
            wave_lds_sync();

            /* Prefetch a visit's first 64 staged positions: lane t holds atom t
               of the neighbour cell (unsorted position) and its window word t. */
            float4 pfx = make_float4(0.f, 0.f, 0.f, 0.f);
            unsigned int pfw = 0;
            auto prefetch = [&](int kv) {
                const int4 en = nbr[k0 + kv];
                const int2 cs = cnt_off[en.x];
                if (lane < cs.x) {
                    pfx = xf[cs.y + lane];
                    if (!(en.y & 32)) {
                        const int sid = en.y & 15, orient = (en.y >> 4) & 1;
                        pfw = sortlist[13 * (size_t)cs.y + (size_t)sid * cs.x + (orient ? lane : cs.x - 1 - lane)];
                    }
                }
            };
            if (nn > 0) prefetch(0);

            float hx = 0.f, hy = 0.f, hz = 0.f, lx = 0.f, ly = 0.f, lz = 0.f;
            double epot = 0.0, vir = 0.0, eexcl = 0.0;
            unsigned int np = 0, nref = 0, nexcl = 0;

            for (int k = 0; k < nn; k++) {
                const int4 en = nbr[k0 + k];
                const int2 cjc = cnt_off[en.x];
                const int cj = en.x, nj = cjc.x, offj = cjc.y;
                const int sid = en.y & 15, orient = (en.y >> 4) & 1, self = (en.y >> 5) & 1;

                /* Shift from the owner cell to the neighbour (minimum image),
                   rounded to FP32 on the host; the FP64 value is recomputed
                   where needed. */
                const float4 sfv = nbs[k0 + k];

                /* Stage the neighbour in the order its window is
                   walked: ascending keys when the owner is the task's i cell,
                   descending otherwise, storage order for the self task.
                   Record = (x + s, y + s, z + s, key' | index << 16 | type << tshift):
                   the position moved into the owner's frame by its cell's
                   shift s, so that a candidate's distance is one subtraction
                   per axis, and key' = key, or 0xffff - key when the owner is
                   the j cell. */
                wave_lds_sync();
                if (lane < nj) raw[lane] = pfx;
                wave_lds_sync();
                for (int t = lane; t < nj; t += 64) {
                    if (self) {
                        const float4 p = t < 64 ? pfx : xf[offj + t];
                        stage[t] = make_float4(p.x + sfv.x, p.y + sfv.y, p.z + sfv.z,
                                               __uint_as_float(((unsigned int)t << 16) |
                                                               ((unsigned int)__float_as_int(p.w) << P.tshift)));
                    } else {
                        const unsigned int w =
                            t < 64 ? pfw : sortlist[13 * (size_t)offj + (size_t)sid * nj + (orient ? t : nj - 1 - t)];
                        const int idx = (int)(w >> 16) < nj ? (int)(w >> 16) : nj - 1;
                        const float4 p = idx < 64 ? raw[idx] : xf[offj + idx];
                        const unsigned int kk = orient ? 0xffffu - (w & 0xffffu) : (w & 0xffffu);
                        stage[t] = make_float4(p.x + sfv.x, p.y + sfv.y, p.z + sfv.z,
                                               __uint_as_float(kk | ((unsigned int)idx << 16) |
                                                               ((unsigned int)__float_as_int(p.w) << P.tshift)));
                    }
                }
                wave_lds_sync();

                /* Prefetch the next visit while this one is processed. */
                if (k + 1 < nn) prefetch(k + 1);
                if (nj == 0) continue;

                int myk = 0, dns = 0;
                bool live_ref = true, run = true;
                if (!self) {
                    dns = P.proj ? en.w : en.z;
                    {
                        const int kr = (int)(__float_as_uint(stage[0].w) & 0xffffu);
                        const int kstage0 = orient ? 0xffff - kr : kr; /* staged keys are complemented when orient */
                        const int s_imax = orient ? kstage0 : kfl[sid];
                        const int s_jmin = orient ? kfl[13 + sid] : kstage0;
                        live_ref = (s_jmin + en.z - s_imax) >= 0;
                        run = P.proj || live_ref;
                    }
                    myk = own_key[sid * 64 + il];
                }
                /* Window (runner_dopair.c:455-478): record t is admitted while
                   key_j + dnshift - key_i < dmaxdist (owner is i) or
                   key_i + dnshift - key_j < dmaxdist (owner is j).  With the
                   staged key k' = key (owner is i) or 0xffff - key (owner is
                   j), both read k' < kmax, and k' ascends along the staged
                   order, so a lane's window ends at its first failing record. */
                /* With pseudo-Verlet sort reuse the window widens by both
                   cells' displacement since the last sort. */
                const int dmd = (P.maxdx != nullptr && !self)
                                    ? pair_dmaxdist(P.dscale, P.cutoff, P.maxdx[orient ? en.x : c],
                                                    P.maxdx[orient ? c : en.x])
                                    : P.dmaxdist;
                const int kmax = orient ? dmd - (myk + dns - 0xffff) : dmd - (dns - myk);

                float lfx = 0.f, lfy = 0.f, lfz = 0.f, le = 0.f, lv = 0.f;
                unsigned int lnp = 0, lnref = 0;

                /* The reference's FP64 cutoff test (runner_dopair.c:465-489) of
                   this lane's atom and the record with word w of cell cn
                   (storage offset on), in the task's own orientation: the
                   owner is the task's i cell (own_i) or its j cell. */
                auto in_cut64 = [&](int cn, int on, unsigned int w, bool own_i) -> bool {
                    const double *xa = &x64[3 * (size_t)a];
                    const double *xb = &x64[3 * (size_t)(on + rec_idx(w, P.imask))];
                    const double *o_own = &origin[3 * c], *o_nb = &origin[3 * cn];
                    const double r2d =
                        own_i ? r2_task64(xa, xb, min_image(o_nb[0] - o_own[0], P.dim[0]),
                                          min_image(o_nb[1] - o_own[1], P.dim[1]),
                                          min_image(o_nb[2] - o_own[2], P.dim[2]))
                              : r2_task64(xb, xa, min_image(o_own[0] - o_nb[0], P.dim[0]),
                                          min_image(o_own[1] - o_nb[1], P.dim[1]),
                                          min_image(o_own[2] - o_nb[2], P.dim[2]));
                    return r2d <= P.cutoff2;
                };

                /* One visit, specialised by kind: 0 self task, 1 owner is the
                   task's i cell (energies, virial and counts are taken here),
                   2 owner is the j cell (forces only). */
                auto visit = [&](auto kind) {
                    constexpr int VK = decltype(kind)::value;
                    int t = part;
                    bool alive = active && run;
                    while (wave_any(alive)) {
                        /* Filter: up to HCAP records per lane, predicated; the
                           wave leaves as soon as no lane is inside its window. */
                        int h = 0;
                        for (int it = 0; it < HCAP; it++) {
                            const float4 pj = stage[t < nj ? t : nj - 1];
                            const unsigned int wj = __float_as_uint(pj.w);
                            alive = alive && t < nj;
                            if (VK != 0) alive = alive && (int)rec_key(wj) < kmax;
                            /* half shell: a self task takes each pair once, j < i */
                            if (HALF && VK == 0) alive = alive && t < myidx;
                            const bool cand = VK == 0 ? (alive && t != myidx) : alive;
                            const float dx = xi.x - pj.x, dy = xi.y - pj.y, dz = xi.z - pj.z;
                            const float r2 = dx * dx + dy * dy + dz * dz;
                            bool hit;
                            if constexpr (MLP) {
                                hit = cand && r2 <= P.rc2f;
                                const bool near = cand && fabsf(r2 - P.rc2f) <= P.band;
                                if (wave_any(near))
                                    if (near) hit = in_cut64(cj, offj, wj, VK != 2);
                            } else {
                                /* keep everything up to the band's upper edge; the
                                   evaluation decides the band's pairs in FP64 */
                                hit = cand && r2 <= rc2hi;
                            }
                            hitl[h * 64 + lane] = (unsigned short)t;
                            h += hit ? 1 : 0;
                            t += NPi;
                            if (!wave_any(alive)) break;
                        }

                        if constexpr (!MLP) {
                            /* Evaluate the kept hits, two per lane per round.  In
                               half-shell mode each lane starts its list at il mod h,
                               so that lanes of one partition (which kept hits from
                               the same records) add to different records at once. */
                            const int rot = (HALF && h > 0) ? il % h : 0;
                            for (int s = 0; wave_any(s < h); s += 2) {
                                const bool va = s < h, vb = s + 1 < h;
                                int sa = s + rot, sb = s + 1 + rot;
                                if (sa >= h) sa -= h;
                                if (sb >= h) sb -= h;
                                const int ta = va ? hitl[sa * 64 + lane] : 0;
                                const int tb = vb ? hitl[sb * 64 + lane] : ta;
                                const float4 pa = stage[ta], pb = stage[tb];
                                const unsigned int wa = __float_as_uint(pa.w), wb = __float_as_uint(pb.w);
                                const float4 ha = ld_f4(rs_ptab, 16 * (ti * mt + rec_type(wa, P.tshift)));
                                const float4 hb = ld_f4(rs_ptab, 16 * (ti * mt + rec_type(wb, P.tshift)));
                                const float dxa = xi.x - pa.x, dya = xi.y - pa.y, dza = xi.z - pa.z;
                                const float dxb = xi.x - pb.x, dyb = xi.y - pb.y, dzb = xi.z - pb.z;
                                const float r2a = dxa * dxa + dya * dya + dza * dza;
                                const float r2b = dxb * dxb + dyb * dyb + dzb * dzb;
                                bool ua = va && __float_as_int(ha.w) != -1;
                                bool ub = vb && __float_as_int(hb.w) != -1;
                                /* pairs within the band of the cutoff: FP64 decides */
                                const bool na = ua && fabsf(r2a - P.rc2f) <= P.band;
                                const bool nb = ub && fabsf(r2b - P.rc2f) <= P.band;
                                if (wave_any(na || nb)) {
                                    if (na) ua = in_cut64(cj, offj, wa, VK != 2);
                                    if (nb) ub = in_cut64(cj, offj, wb, VK != 2);
                                }
                                float ea, fa, eb, fb;
                                pot_eval32r2(ha, hb, ua, ub, rs_coef, r2a, r2b, ea, fa, eb, fb);
                                lfx = fmaf(-fb, dxb, fmaf(-fa, dxa, lfx));
                                lfy = fmaf(-fb, dyb, fmaf(-fa, dya, lfy));
                                lfz = fmaf(-fb, dzb, fmaf(-fa, dza, lfz));
                                if constexpr (HALF) {
                                    /* the opposite force on the record's atom, into this
                                       lane's copy (lane mod 4) of the visit's array */
                                    float *jc = jf + (lane & 3) * 3 * P.maxn;
                                    if (ua) {
                                        atomicAdd(&jc[3 * ta], fa * dxa);
                                        atomicAdd(&jc[3 * ta + 1], fa * dya);
                                        atomicAdd(&jc[3 * ta + 2], fa * dza);
                                    }
                                    if (ub) {
                                        atomicAdd(&jc[3 * tb], fb * dxb);
                                        atomicAdd(&jc[3 * tb + 1], fb * dyb);
                                        atomicAdd(&jc[3 * tb + 2], fb * dzb);
                                    }
                                }
                                if (VK != 2) {
                                    const bool ca = ua && (VK == 1 || myidx > rec_idx(wa, P.imask));
                                    const bool cb = ub && (VK == 1 || myidx > rec_idx(wb, P.imask));
                                    if (ca) {
                                        le += ea;
                                        lv -= fa * r2a;
                                        lnp++;
                                        if (P.proj) lnref += (VK == 0 ||
                                                  (live_ref && ((int)rec_key(wa) + en.z - myk) < dmd)) ? 1u : 0u;
                                    }
                                    if (cb) {
                                        le += eb;
                                        lv -= fb * r2b;
                                        lnp++;
                                        if (P.proj) lnref += (VK == 0 ||
                                                  (live_ref && ((int)rec_key(wb) + en.z - myk) < dmd)) ? 1u : 0u;
                                    }
                                }
                            }
                        } else {
                            /* Below the pair's r_lo: table, by this lane.  Otherwise
                               keep the hit for the dense list. */
                            int nd = 0;
                            for (int s = 0; s < h; s++) {
                                const int ta = hitl[s * 64 + lane];
                                const float4 pa = stage[ta];
                                const unsigned int wa = __float_as_uint(pa.w);
                                const float dxa = xi.x - pa.x, dya = xi.y - pa.y, dza = xi.z - pa.z;
                                const float r2a = dxa * dxa + dya * dya + dza * dza;
                                /* r_lo^2 is +inf for a type pair without potential, so
                                   only the few hits below r_lo load the table header */
                                if (r2a >= N.rlo2[ti * mt + rec_type(wa, P.tshift)]) {
                                    hitl[nd * 64 + lane] = (unsigned short)ta;
                                    nd++;
                                    continue;
                                }
                                const float4 ha = ptab[ti * mt + rec_type(wa, P.tshift)];
                                if (__float_as_int(ha.w) == -1) continue;
                                float ea, fa;
                                pot_eval32(ha, coeffs4, r2a, ea, fa);
                                lfx -= fa * dxa;
                                lfy -= fa * dya;
                                lfz -= fa * dza;
                                if constexpr (HALF) {
                                    float *jc = jf + (lane & 3) * 3 * P.maxn;
                                    atomicAdd(&jc[3 * ta], fa * dxa);
                                    atomicAdd(&jc[3 * ta + 1], fa * dya);
                                    atomicAdd(&jc[3 * ta + 2], fa * dza);
                                }
                                if (VK != 2 && (VK == 1 || myidx > rec_idx(wa, P.imask))) {
                                    le += ea;
                                    lv -= fa * r2a;
                                    lnp++;
                                    if (P.proj) lnref += (VK == 0 ||
                                              (live_ref && ((int)rec_key(wa) + en.z - myk) < dmd)) ? 1u : 0u;
                                }
                            }
                            /* Dense list: this lane's hits at [off, off + nd). */
                            const int off = wave_excl_scan(nd, lane);
                            const int T = __shfl(off + nd, 63);
                            for (int s = 0; s < nd; s++) {
                                const float4 pa = stage[hitl[s * 64 + lane]];
                                const float dxa = xi.x - pa.x, dya = xi.y - pa.y, dza = xi.z - pa.z;
                                dn_r2[off + s] = dxa * dxa + dya * dya + dza * dza;
                                dn_p[off + s] = ptype[ti * mt + rec_type(__float_as_uint(pa.w), P.tshift)];
                            }
                            wave_lds_sync();
                            mlp_dense_eval(N, w1s, dn_r2, dn_p, dn_f, dn_e, T, lane);
                            wave_lds_sync();
                            for (int s = 0; s < nd; s++) {
                                const int ta = hitl[s * 64 + lane];
                                const float4 pa = stage[ta];
                                const unsigned int wa = __float_as_uint(pa.w);
                                const float dxa = xi.x - pa.x, dya = xi.y - pa.y, dza = xi.z - pa.z;
                                const float r2a = dxa * dxa + dya * dya + dza * dza;
                                const float fa = dn_f[off + s], ea = dn_e[off + s];
                                lfx -= fa * dxa;
                                lfy -= fa * dya;
                                lfz -= fa * dza;
                                if constexpr (HALF) {
                                    float *jc = jf + (lane & 3) * 3 * P.maxn;
                                    atomicAdd(&jc[3 * ta], fa * dxa);
                                    atomicAdd(&jc[3 * ta + 1], fa * dya);
                                    atomicAdd(&jc[3 * ta + 2], fa * dza);
                                }
                                if (VK != 2 && (VK == 1 || myidx > rec_idx(wa, P.imask))) {
                                    le += ea;
                                    lv -= fa * r2a;
                                    lnp++;
                                    if (P.proj) lnref += (VK == 0 ||
                                              (live_ref && ((int)rec_key(wa) + en.z - myk) < dmd)) ? 1u : 0u;
                                }
                            }
                            wave_lds_sync();
                        }
                    }
                };
                if (self)
                    visit(visit_kind<0>{});
                else if (orient == 0)
                    visit(visit_kind<1>{});
                else
                    visit(visit_kind<2>{});
                if constexpr (HALF) {
                    /* this visit's forces on the visited atoms, by slot; later
                       chunks of the owner add to the first one's */
                    wave_lds_sync();
                    for (int q = lane; q < nj; q += 64) {
                        const int idx = rec_idx(__float_as_uint(stage[q].w), P.imask);
                        /* sum the 4 copies, and leave them zero for the next visit */
                        float vv[3];
                        for (int m = 0; m < 3; m++) {
                            float *j0 = jf + 3 * q + m;
                            const int s = 3 * P.maxn;
                            vv[m] = (j0[0] + j0[s]) + (j0[2 * s] + j0[3 * s]);
                            j0[0] = j0[s] = j0[2 * s] = j0[3 * s] = 0.f;
                        }
                        float *dst = O.jpart + 3 * ((size_t)((unsigned int)en.y >> 9) * P.nparts + offj + idx);
                        for (int m = 0; m < 3; m++) dst[m] = ch > 0 ? dst[m] + vv[m] : vv[m];
                    }
                }
                acc2(hx, lx, lfx);
                acc2(hy, ly, lfy);
                acc2(hz, lz, lfz);
                epot += (double)le;
                vir += (double)lv;
                np += lnp;
                nref += P.proj ? lnref : lnp;
            }

            /* Excluded pairs: subtract what the pair pass added
               (exclusion.c:139-208), same FP32 arithmetic as the pair pass. */
            if constexpr (!MLP) {
                if (active && part == 0 && grp == 0) {
                    const int myid = pid[a];
                    for (int k = excl_off[myid]; k < excl_off[myid + 1]; k++) {
                        const int oid = excl_list[k];
                        if (oid == myid) continue;
                        const int b = index_of_id[oid];
                        if (b < 0) continue;
                        const int cb = cell_of[b];
                        const float4 pj = xf[b];
                        const float4 hdr = ptab[ti * mt + __float_as_int(pj.w)];
                        if (__float_as_int(hdr.w) == -1) continue;
                        const float ex = (float)min_image(origin[3 * cb] - oc0, P.dim[0]);
                        const float ey = (float)min_image(origin[3 * cb + 1] - oc1, P.dim[1]);
                        const float ez = (float)min_image(origin[3 * cb + 2] - oc2, P.dim[2]);
                        const float dx = (xi.x - pj.x) - ex, dy = (xi.y - pj.y) - ey, dz = (xi.z - pj.z) - ez;
                        const float r2 = dx * dx + dy * dy + dz * dz;
                        bool in = r2 <= P.rc2f;
                        if (fabsf(r2 - P.rc2f) <= P.band) {
                            const bool mine = myid < oid;
                            const int ia = mine ? a : b, ib = mine ? b : a;
                            const int ca = mine ? c : cb, cbb = mine ? cb : c;
                            in = r2_excl64(&x64[3 * (size_t)ia], &x64[3 * (size_t)ib], &loc[3 * ca], &loc[3 * cbb],
                                           P.h) <= P.cutoff2;
                        }
                        if (!in) continue;
                        float e, ff;
                        pot_eval32(hdr, coeffs4, r2, e, ff);
                        acc2(hx, lx, ff * dx);
                        acc2(hy, ly, ff * dy);
                        acc2(hz, lz, ff * dz);
                        if (myid < oid) {
                            eexcl -= (double)e;
                            nexcl++;
                        }
                    }
                }
            } else {
                const bool xl = active && part == 0 && grp == 0;
                const int myid = xl ? pid[a] : 0;
                int kx = xl ? excl_off[myid] : 0;
                const int kend = xl ? excl_off[myid + 1] : 0;
                /* dx and r^2 of this lane's atom to slot b, as in the pair pass. */
                auto excl_geom = [&](int b, float &dx, float &dy, float &dz) {
                    const int cb = cell_of[b];
                    const float4 pj = xf[b];
                    dx = (xi.x - pj.x) - (float)min_image(origin[3 * cb] - oc0, P.dim[0]);
                    dy = (xi.y - pj.y) - (float)min_image(origin[3 * cb + 1] - oc1, P.dim[1]);
                    dz = (xi.z - pj.z) - (float)min_image(origin[3 * cb + 2] - oc2, P.dim[2]);
                    return __float_as_int(pj.w);
                };
                while (__any(kx < kend)) {
                    int nd = 0;
                    while (kx < kend && nd < MD_XCAP_MLP) {
                        const int oid = excl_list[kx++];
                        if (oid == myid) continue;
                        const int b = index_of_id[oid];
                        if (b < 0) continue;
                        float dx, dy, dz;
                        const int tb = excl_geom(b, dx, dy, dz);
                        const float4 hdr = ptab[ti * mt + tb];
                        if (__float_as_int(hdr.w) == -1) continue;
                        const float r2 = dx * dx + dy * dy + dz * dz;
                        bool in = r2 <= P.rc2f;
                        if (fabsf(r2 - P.rc2f) <= P.band) {
                            const int cb = cell_of[b];
                            const bool mine = myid < oid;
                            const int ia = mine ? a : b, ib = mine ? b : a;
                            const int ca = mine ? c : cb, cbb = mine ? cb : c;
                            in = r2_excl64(&x64[3 * (size_t)ia], &x64[3 * (size_t)ib], &loc[3 * ca], &loc[3 * cbb],
                                           P.h) <= P.cutoff2;
                        }
                        if (!in) continue;
                        if (r2 >= N.rlo2[ti * mt + tb]) {
                            exb[nd * 64 + lane] = b;
                            nd++;
                            continue;
                        }
                        float e, ff;
                        pot_eval32(hdr, coeffs4, r2, e, ff);
                        acc2(hx, lx, ff * dx);
                        acc2(hy, ly, ff * dy);
                        acc2(hz, lz, ff * dz);
                        if (myid < oid) {
                            eexcl -= (double)e;
                            nexcl++;
                        }
                    }
                    const int off = wave_excl_scan(nd, lane);
                    const int T = __shfl(off + nd, 63);
                    for (int s = 0; s < nd; s++) {
                        float dx, dy, dz;
                        const int tb = excl_geom(exb[s * 64 + lane], dx, dy, dz);
                        dn_r2[off + s] = dx * dx + dy * dy + dz * dz;
                        dn_p[off + s] = ptype[ti * mt + tb];
                    }
                    wave_lds_sync();
                    mlp_dense_eval(N, w1s, dn_r2, dn_p, dn_f, dn_e, T, lane);
                    wave_lds_sync();
                    for (int s = 0; s < nd; s++) {
                        const int b = exb[s * 64 + lane];
                        float dx, dy, dz;
                        excl_geom(b, dx, dy, dz);
                        const float ff = dn_f[off + s], e = dn_e[off + s];
                        acc2(hx, lx, ff * dx);
                        acc2(hy, ly, ff * dy);
                        acc2(hz, lz, ff * dz);
                        if (myid < pid[b]) {
                            eexcl -= (double)e;
                            nexcl++;
                        }
                    }
                    wave_lds_sync();
                }
            }

            /* Fold the partitions of each atom into partition 0, in order. */
            for (int p = 1; p < NPmax; p++) {
                const int src = (lane + p * nsub) & 63;
                const float ohx = __shfl(hx, src), ohy = __shfl(hy, src), ohz = __shfl(hz, src);
                const float olx = __shfl(lx, src), oly = __shfl(ly, src), olz = __shfl(lz, src);
                if (part == 0 && p < NPi) {
                    acc2(hx, lx, ohx);
                    acc2(hy, ly, ohy);
                    acc2(hz, lz, ohz);
                    lx += olx;
                    ly += oly;
                    lz += olz;
                }
            }
            if (part == 0) {
                if (P.nsplit == 1) {
                    O.fhi[a] = make_float4(hx, hy, hz, 0.0f);
                    O.flo[a] = make_float4(lx, ly, lz, 0.0f);
                } else {
                    O.phi[(size_t)grp * P.nparts + a] = make_float4(hx, hy, hz, 0.0f);
                    O.plo[(size_t)grp * P.nparts + a] = make_float4(lx, ly, lz, 0.0f);
                }
            }
            if (!active) {
                epot = vir = eexcl = 0.0;
                np = nref = nexcl = 0;
            }

            /* Per-item sums; this wave owns the item's slots, chunks add in order. */
            epot = wave_sum(epot);
            vir = wave_sum(vir);
            eexcl = wave_sum(eexcl);
            np = (unsigned int)wave_sum((int)np);
            nref = (unsigned int)wave_sum((int)nref);
            nexcl = (unsigned int)wave_sum((int)nexcl);
            if (lane == 0) {
                if (ch == 0) {
                    O.cell_acc[3 * item] = epot;
                    O.cell_acc[3 * item + 1] = eexcl;
                    O.cell_acc[3 * item + 2] = vir;
                    O.cell_cnt[3 * item] = np;
                    O.cell_cnt[3 * item + 1] = nexcl;
                    O.cell_cnt[3 * item + 2] = nref;
                } else {
                    O.cell_acc[3 * item] += epot;
                    O.cell_acc[3 * item + 1] += eexcl;
                    O.cell_acc[3 * item + 2] += vir;
                    O.cell_cnt[3 * item] += np;
                    O.cell_cnt[3 * item + 1] += nexcl;
                    O.cell_cnt[3 * item + 2] += nref;
                }
            }
        }
    }
}

#include "pair_tile.h"

#define NB_PARAMS                                                                                             \
    struct nb_params P, const int2 *__restrict__ cnt_off, const int4 *__restrict__ nbr,                       \
        const int *__restrict__ nbr_off, const float4 *__restrict__ nbs, const double *__restrict__ origin,   \
        const int *__restrict__ loc,                                                                         \
        const float4 *__restrict__ xf, const double *__restrict__ x64, const int *__restrict__ pid,          \
        const unsigned int *__restrict__ sortlist, const unsigned short *__restrict__ keyof,                \
        const float4 *__restrict__ ptab, const float4 *__restrict__ coeffs4, const int *__restrict__ excl_off, \
        const int *__restrict__ excl_list, const int *__restrict__ index_of_id, const int *__restrict__ cell_of, \
        struct nb_out O, int *__restrict__ queue
#define NB_ARGS                                                                                              \
    P, cnt_off, nbr, nbr_off, nbs, origin, loc, xf, x64, pid, sortlist, keyof, ptab, coeffs4, excl_off, excl_list, \
        index_of_id, cell_of, O, queue

/* Table mode, full shell (pair_tile.h): at most 32 or 64 owner atoms at a
   time, the reference's or the projected window. */
#define PAIR_PARAMS                                                                                           \
    struct nb_params P, const int2 *__restrict__ cnt_off, const int4 *__restrict__ nbr,                       \
        const int *__restrict__ nbr_off, const int *__restrict__ nbr_mid, const float4 *__restrict__ nbs,     \
        const double *__restrict__ origin, const int *__restrict__ loc,                                      \
        const float4 *__restrict__ xf, const double *__restrict__ x64, const int *__restrict__ pid,          \
        const unsigned short *__restrict__ kminmax, const unsigned int *__restrict__ sortlist,                \
        const unsigned short *__restrict__ keyof, const float4 *__restrict__ ptab,                           \
        const float4 *__restrict__ coeffs4, const int *__restrict__ excl_off, const int *__restrict__ excl_list, \
        const int *__restrict__ index_of_id, const int *__restrict__ cell_of, struct nb_out O
#define PAIR_ARGS                                                                                             \
    P, cnt_off, nbr, nbr_off, nbr_mid, nbs, origin, loc, xf, x64, pid, kminmax, sortlist, keyof, ptab, \
        coeffs4, excl_off, excl_list, index_of_id, cell_of, O

template <int R, int TABS, bool PROJ>
__global__ __launch_bounds__(64 * PT_WAVES) __attribute__((amdgpu_waves_per_eu(R == 32 ? 4 : 3, 8))) void k_pair(
    PAIR_PARAMS) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    /* the waves' working sets, then the tables */
    pair_lds<R> *L = (pair_lds<R> *)smem;
    float4 *tab = (float4 *)(L + PT_WAVES);
    if (TABS) {
        const int nh = P.ptab_bytes / 16, nt = nh + (TABS == 2 ? P.coef_bytes / 16 : 0);
        for (int k = threadIdx.x; k < nt; k += 64 * PT_WAVES) tab[k] = k < nh ? ptab[k] : coeffs4[k - nh];
        __syncthreads();
    }
    pair_body<R, TABS, PROJ>(L[threadIdx.x >> 6], (const char *)tab, PAIR_ARGS);
}

/* Surrogate mode (engine_flag_mlp). */
__global__ __launch_bounds__(64) void k_nonbond_mlp(NB_PARAMS, struct mlp_net N, const int *__restrict__ ptype) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    nonbond_body<true, false>(smem, NB_ARGS, N, ptype);
}

/* Surrogate mode on the half shell: each pair's network evaluation once. */
__global__ __launch_bounds__(64) void k_nonbond_mlp_half(NB_PARAMS, struct mlp_net N, const int *__restrict__ ptype) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    nonbond_body<true, true>(smem, NB_ARGS, N, ptype);
}

/* Table mode on the half shell: each pair once, at the i cell of its task.
   The 5-wave build is for many cells. */
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_nonbond_half(NB_PARAMS) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const struct mlp_net N = {};
    nonbond_body<false, true>(smem, NB_ARGS, N, nullptr);
}
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_nonbond_half_wide(NB_PARAMS) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const struct mlp_net N = {};
    nonbond_body<false, true, MD_HCAP_WIDE>(smem, NB_ARGS, N, nullptr);
}

/* Second step of a split and/or half-shell pass, one wave per cell: each
   atom's force = its owner's (hi, lo), or with nsplit > 1 the groups'
   (hi, lo) in group order, plus (half shell) the forces its cell received in
   its own self task (slot 0) and as the j cell of other cells' tasks (slots
   1.. in task order, those of empty i cells left out: nothing writes them),
   all added with two-sum in that order.  Reads as a stream: the slots of
   consecutive atoms are consecutive, and 8 are in flight per lane. */
__global__ __launch_bounds__(64) void k_fold(int ncells, const int2 *__restrict__ cnt_off, int nsplit, int nparts,
                                             const float4 *__restrict__ phi, const float4 *__restrict__ plo, int half,
                                             const int *__restrict__ inv_off, const int *__restrict__ inv_cell,
                                             const float *__restrict__ jpart, float4 *__restrict__ fhi,
                                             float4 *__restrict__ flo) {
    const int c = blockIdx.x, lane = threadIdx.x;
    const int2 co = cnt_off[c];
    const int q0 = half ? inv_off[c] : 0, nq = half ? inv_off[c + 1] - q0 + 1 : 0;
    for (int s = lane; s < co.x; s += 64) {
        const int a = co.y + s;
        const float4 h = nsplit > 1 ? phi[a] : fhi[a], l = nsplit > 1 ? plo[a] : flo[a];
        float hx = h.x, hy = h.y, hz = h.z, lx = l.x, ly = l.y, lz = l.z;
        for (int gp = 1; gp < nsplit; gp++) {
            const float4 oh = phi[(size_t)gp * nparts + a], ol = plo[(size_t)gp * nparts + a];
            acc2(hx, lx, oh.x);
            acc2(hy, ly, oh.y);
            acc2(hz, lz, oh.z);
            lx += ol.x;
            ly += ol.y;
            lz += ol.z;
        }
        for (int q = 0; q < nq; q += 8) {
            float v[8][3];
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const bool in = q + m < nq && (q + m == 0 || cnt_off[inv_cell[q0 + q + m - 1]].x > 0);
                const float *src = jpart + 3 * ((size_t)(q + m) * nparts + a);
                v[m][0] = in ? src[0] : 0.f;
                v[m][1] = in ? src[1] : 0.f;
                v[m][2] = in ? src[2] : 0.f;
            }
#pragma unroll
            for (int m = 0; m < 8; m++) {
                acc2(hx, lx, v[m][0]);
                acc2(hy, ly, v[m][1]);
                acc2(hz, lz, v[m][2]);
            }
        }
        fhi[a] = make_float4(hx, hy, hz, 0.0f);
        flo[a] = make_float4(lx, ly, lz, 0.0f);
    }
}

/* ------------------------------------------------------------ k_reduce */

/* Two steps, both in a fixed order (the totals are bitwise repeatable):
   k_reduce_a: block b sums the slots [b n / B, (b + 1) n / B) of the
   per-item FP64 sums and counts (strided per thread, then a tree);
   k_reduce_b: one block sums the B partials the same way. */
#define MD_RED_BLOCKS 128
__device__ __forceinline__ void block_tree3(double (*sd)[256], unsigned long long (*sc)[256], int t) {
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (t < s)
            for (int m = 0; m < 3; m++) {
                sd[m][t] += sd[m][t + s];
                sc[m][t] += sc[m][t + s];
            }
        __syncthreads();
    }
}

/* The totals of few items in one launch, by one block: 4.4 us at 3,000 items
   against 8 us and another launch for the two above; a block's 256 threads
   load 32 items each at MD_RED_ONE. */
#define MD_RED_ONE 8192
__global__ __launch_bounds__(256) void k_reduce_one(int n, const double *__restrict__ acc,
                                                    const unsigned long long *__restrict__ cnt,
                                                    double *__restrict__ tot,
                                                    unsigned long long *__restrict__ tot_cnt,
                                                    double *__restrict__ htot,
                                                    unsigned long long *__restrict__ htot_cnt,
                                                    int *__restrict__ queue) {
    __shared__ double sd[3][256];
    __shared__ unsigned long long sc[3][256];
    const int t = threadIdx.x;
    double d0 = 0, d1 = 0, d2 = 0;
    unsigned long long c0 = 0, c1 = 0, c2 = 0;
#pragma unroll 4
    for (int k = t; k < n; k += 256) {
        d0 += acc[3 * k];
        d1 += acc[3 * k + 1];
        d2 += acc[3 * k + 2];
        c0 += cnt[3 * k];
        c1 += cnt[3 * k + 1];
        c2 += cnt[3 * k + 2];
    }
    sd[0][t] = d0;
    sd[1][t] = d1;
    sd[2][t] = d2;
    sc[0][t] = c0;
    sc[1][t] = c1;
    sc[2][t] = c2;
    block_tree3(sd, sc, t);
    if (t < 3) {
        tot[t] = htot[t] = sd[t][0];
        tot_cnt[t] = htot_cnt[t] = sc[t][0];
    }
    if (t < MD_NQUEUE) queue[t] = 0; /* for the next pass */
}

__global__ __launch_bounds__(256) void k_reduce_a(int n, const double *__restrict__ acc,
                                                  const unsigned long long *__restrict__ cnt,
                                                  double *__restrict__ pacc, unsigned long long *__restrict__ pcnt) {
    __shared__ double sd[3][256];
    __shared__ unsigned long long sc[3][256];
    const int t = threadIdx.x, b = blockIdx.x;
    const int lo = (int)(((long long)b * n) / gridDim.x), hi = (int)(((long long)(b + 1) * n) / gridDim.x);
    double d0 = 0, d1 = 0, d2 = 0;
    unsigned long long c0 = 0, c1 = 0, c2 = 0;
    for (int k = lo + t; k < hi; k += 256) {
        d0 += acc[3 * k];
        d1 += acc[3 * k + 1];
        d2 += acc[3 * k + 2];
        c0 += cnt[3 * k];
        c1 += cnt[3 * k + 1];
        c2 += cnt[3 * k + 2];
    }
    sd[0][t] = d0;
    sd[1][t] = d1;
    sd[2][t] = d2;
    sc[0][t] = c0;
    sc[1][t] = c1;
    sc[2][t] = c2;
    block_tree3(sd, sc, t);
    if (t < 3) {
        pacc[3 * b + t] = sd[t][0];
        pcnt[3 * b + t] = sc[t][0];
    }
}

__global__ __launch_bounds__(256) void k_reduce_b(int nb, const double *__restrict__ pacc,
                                                  const unsigned long long *__restrict__ pcnt,
                                                  double *__restrict__ tot, unsigned long long *__restrict__ tot_cnt,
                                                  double *__restrict__ htot,
                                                  unsigned long long *__restrict__ htot_cnt,
                                                  int *__restrict__ queue) {
    __shared__ double sd[3][256];
    __shared__ unsigned long long sc[3][256];
    const int t = threadIdx.x;
    for (int m = 0; m < 3; m++) {
        double d = 0;
        unsigned long long c = 0;
        for (int k = t; k < nb; k += 256) {
            d += pacc[3 * k + m];
            c += pcnt[3 * k + m];
        }
        sd[m][t] = d;
        sc[m][t] = c;
    }
    block_tree3(sd, sc, t);
    if (t < 3) {
        tot[t] = htot[t] = sd[t][0];
        tot_cnt[t] = htot_cnt[t] = sc[t][0];
    }
    if (t < MD_NQUEUE) queue[t] = 0; /* for the next pass */
}

/* ------------------------------------------------------------ host side */

static void gpu_free_pass(struct gpu_state *g) {
    (void)hipFree(g->d_count);
    (void)hipFree(g->d_offset);
    (void)hipFree(g->d_x);
    (void)hipFree(g->d_type);
    (void)hipFree(g->d_id);
    (void)hipFree(g->d_cell_of);
    (void)hipFree(g->d_xf);
    (void)hipFree(g->d_fhi);
    (void)hipFree(g->d_stage);
    (void)hipFree(g->d_sortlist);
    (void)hipFree(g->d_keyof);
    (void)hipHostFree(g->h_stage);
    (void)hipHostFree(g->h_fhi);
    (void)hipHostFree(g->h_v);
    g->d_count = g->d_offset = NULL;
    g->d_x = NULL;
    g->d_type = g->d_id = g->d_cell_of = NULL;
    g->d_xf = g->d_fhi = g->d_flo = NULL;
    g->d_sortlist = NULL;
    g->d_keyof = NULL;
    g->h_stage = g->d_stage = NULL;
    g->h_x = NULL;
    g->h_type = g->h_id = NULL;
    g->h_cnt_off = NULL;
    g->h_fhi = g->h_flo = NULL;
    g->h_v = NULL;
    g->nparts_cap = 0;
}

static int gpu_alloc_parts(struct gpu_state *g, int n) {
    size_t N;
    if (n <= g->nparts_cap) return 0;
    gpu_free_pass(g);
    g->sort_valid = 0;
    N = (size_t)n + n / 8 + 64;
    HIPCHECK(hipMalloc(&g->d_x, sizeof(double) * 3 * N));
    HIPCHECK(hipMalloc(&g->d_type, sizeof(int) * N));
    HIPCHECK(hipMalloc(&g->d_id, sizeof(int) * N));
    HIPCHECK(hipMalloc(&g->d_cell_of, sizeof(int) * N));
    HIPCHECK(hipMalloc(&g->d_xf, sizeof(float4) * N));
    HIPCHECK(hipMalloc(&g->d_fhi, sizeof(float4) * 2 * N)); /* and flo */
    HIPCHECK(hipMalloc((void **)&g->d_stage, GPU_STAGE_BYTES(N, g->ncells)));
    HIPCHECK(hipMalloc(&g->d_sortlist, sizeof(unsigned int) * 13 * N));
    HIPCHECK(hipMalloc(&g->d_keyof, sizeof(unsigned short) * 13 * N));
    HIPCHECK(hipMalloc(&g->d_count, sizeof(int) * g->ncells));
    HIPCHECK(hipMalloc(&g->d_offset, sizeof(int) * (g->ncells + 1)));
    HIPCHECK(hipHostMalloc((void **)&g->h_stage, GPU_STAGE_BYTES(N, g->ncells), hipHostMallocDefault));
    HIPCHECK(hipHostMalloc((void **)&g->h_fhi, sizeof(float4) * 2 * N, hipHostMallocDefault)); /* and flo */
    HIPCHECK(hipHostMalloc((void **)&g->h_v, sizeof(double) * 3 * N, hipHostMallocDefault));
    g->nparts_cap = (int)N;
    return 0;
}

static int gpu_alloc_ids(struct gpu_state *g, int nids) {
    if (nids <= g->nids_cap) return 0;
    (void)hipFree(g->d_index_of_id);
    (void)hipHostFree(g->h_ioi);
    g->h_ioi = NULL;
    HIPCHECK(hipMalloc(&g->d_index_of_id, sizeof(int) * (size_t)nids));
    HIPCHECK(hipHostMalloc((void **)&g->h_ioi, sizeof(int) * (size_t)nids, hipHostMallocDefault));
    g->nids_cap = nids;
    return 0;
}

extern "C" int engine_gpu_setdevice(struct engine *e, int id) {
    int n = 0;
    if (e == NULL) return gerror_(engine_err_null, "NULL engine");
    HIPCHECK(hipGetDeviceCount(&n));
    if (id < 0 || id >= n) return gerror_(engine_err_range, "no such HIP device");
    HIPCHECK(hipSetDevice(id));
    if (e->gpu != NULL) ((struct gpu_state *)e->gpu)->device = id;
    return engine_err_ok;
}

extern "C" int engine_gpu_finalize(struct engine *e) {
    struct gpu_state *g;
    if (e == NULL) return gerror_(engine_err_null, "NULL engine");
    g = (struct gpu_state *)e->gpu;
    if (g == NULL) return engine_err_ok;
    (void)hipSetDevice(g->device);
    (void)hipStreamSynchronize(g->stream);
    gpu_free_pass(g);
    gpu_mlp_free(g);
    gpu_steps_free(g);
    (void)hipFree(g->d_ptab);
    (void)hipFree(g->d_coeffs);
    (void)hipFree(g->d_ptype);
    free(g->h_tabof);
    free(g->h_pair_ti);
    free(g->h_pair_tj);
    (void)hipFree(g->d_nbr);
    (void)hipFree(g->d_nbs);
    (void)hipFree(g->d_nbr_off);
    (void)hipFree(g->d_nbr_mid);
    (void)hipFree(g->d_kminmax);
    (void)hipFree(g->d_nbr_h);
    (void)hipFree(g->d_nbs_h);
    (void)hipFree(g->d_nbr_off_h);
    (void)hipFree(g->d_inv_off);
    (void)hipFree(g->d_inv_cell);
    (void)hipFree(g->d_jpart);
    (void)hipFree(g->d_phi);
    (void)hipFree(g->d_plo);
    (void)hipFree(g->d_origin);
    (void)hipFree(g->d_loc);
    (void)hipFree(g->d_sortflags);
    (void)hipFree(g->d_excl_off);
    (void)hipFree(g->d_excl_list);
    (void)hipFree(g->d_index_of_id);
    (void)hipHostFree(g->h_ioi);
    (void)hipFree(g->d_cnt_off);
    (void)hipFree(g->d_cell_acc);
    (void)hipFree(g->d_cell_cnt);
    (void)hipFree(g->d_tot);
    (void)hipFree(g->d_red_acc);
    (void)hipFree(g->d_red_cnt);
    (void)hipFree(g->d_tot_cnt);
    (void)hipFree(g->d_queue);
    (void)hipFree(g->d_order);
    (void)hipHostFree(g->h_count);
    (void)hipFree(g->d_cell_maxdx);
    (void)hipHostFree(g->h_cell_maxdx);
    free(g->h_sort_count);
    (void)hipHostFree(g->h_offset);
    (void)hipHostFree(g->h_tot);
    (void)hipHostFree(g->h_tot_cnt);
    (void)hipHostFree(g->h_flag);
    for (int k = 0; k < 8; k++) (void)hipEventDestroy(g->ev[k]);
    (void)hipStreamDestroy(g->stream);
    free(g);
    e->gpu = NULL;
    return engine_err_ok;
}

/* Minimum-image shift from cell a's origin to cell b's: the same FP64
   arithmetic as min_image() on the device, rounded once to FP32. */
static float4 cell_shift32(const struct space *s, int a, int b) {
    double v[3];
    for (int k = 0; k < 3; k++) {
        double d = s->cells[b].origin[k] - s->cells[a].origin[k];
        if (d * 2 > s->dim[k])
            d -= s->dim[k];
        else if (d * 2 < -s->dim[k])
            d += s->dim[k];
        v[k] = d;
    }
    return make_float4((float)v[0], (float)v[1], (float)v[2], 0.f);
}

/* dnshift of a pair task (runner_dopair.c:426-452): with the reference's
   norm |shift| and with the projection shift.n on the pair's axis. */
static void task_dnshift(const struct space *s, int ti, int tj, int sid, double dscale, int *dns_ref,
                         int *dns_proj) {
    double sh[3], nshift, dot;
    int k;
    for (k = 0; k < 3; k++) {
        sh[k] = s->cells[tj].origin[k] - s->cells[ti].origin[k];
        if (sh[k] * 2 > s->dim[k])
            sh[k] -= s->dim[k];
        else if (sh[k] * 2 < -s->dim[k])
            sh[k] += s->dim[k];
    }
    nshift = sqrt(sh[0] * sh[0] + sh[1] * sh[1] + sh[2] * sh[2]);
    *dns_ref = (int)(dscale * nshift);
    dot = sh[0] * cell_shift[3 * sid] + sh[1] * cell_shift[3 * sid + 1] + sh[2] * cell_shift[3 * sid + 2];
    *dns_proj = (int)(dscale * dot);
}

/* Whether a task needs the window test: the reference window may cut pairs
   within the cutoff.  Not so when the offset lies along the sort axis
   (pair_tile.h), unless dscale rc is so close below an integer that the
   rounding of the keys' FP64 arithmetic (~1e-11) could matter. */
static int task_window(const struct gpu_state *g, const struct space *s, int dns_ref, int dns_proj) {
    const double rcd = g->P.dscale * s->cutoff;
    return dns_ref > dns_proj || rcd - floor(rcd) > 1.0 - 1e-9;
}

extern "C" int engine_gpu_load(struct engine *e) {
    struct gpu_state *g;
    struct space *s;
    int mt, k, i, j, ntab = 0, nchunks = 0, cid;
    if (e == NULL) return gerror_(engine_err_null, "NULL engine");
    if (e->gpu != NULL) engine_gpu_finalize(e);
    s = &e->s;
    mt = e->max_type;
    if (mt > MD_MAX_TYPES) return gerror_(engine_err_nyi, "more than 1024 particle types");
    g = (struct gpu_state *)calloc(1, sizeof(struct gpu_state));
    if (g == NULL) return gerror_(engine_err_malloc, "calloc failed");
    e->gpu = g;
    HIPCHECK(hipGetDevice(&g->device));
    HIPCHECK(hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking));
    for (k = 0; k < 8; k++) HIPCHECK(hipEventCreate(&g->ev[k]));
    g->ncells = s->nr_cells;
    g->max_type = mt;

    /* Tables: one device table per distinct potential, FP32-rounded, and a
       header per type pair.  A distinct potential is a species pair: its
       index (first appearance in type-pair order) is the pair id that the
       MLP surrogate uses. */
    {
        struct potential **uniq = (struct potential **)calloc((size_t)mt * mt, sizeof(*uniq));
        int *tabof = (int *)malloc(sizeof(int) * mt * mt);
        int *chunk0 = (int *)malloc(sizeof(int) * mt * mt);
        float4 *ptab = (float4 *)malloc(sizeof(float4) * mt * mt);
        float *coef = NULL;
        int bad = 0;
        if (uniq == NULL || tabof == NULL || chunk0 == NULL || ptab == NULL) bad = engine_err_malloc;
        for (k = 0; !bad && k < mt * mt; k++) {
            struct potential *p = e->p[k];
            tabof[k] = -1;
            if (p == NULL) continue;
            if (p->n < 1 || p->n > 511) {
                bad = engine_err_potential;
                break;
            }
            for (j = 0; j < ntab; j++)
                if (uniq[j] == p) break;
            if (j == ntab) {
                chunk0[ntab] = nchunks;
                uniq[ntab++] = p;
                nchunks += p->n + 1;
            }
            tabof[k] = j;
        }
        if (!bad && nchunks >= (1 << 22)) bad = engine_err_potential;
        if (!bad && (coef = (float *)malloc(sizeof(float) * 8 * (nchunks > 0 ? nchunks : 1))) == NULL)
            bad = engine_err_malloc;
        if (!bad) {
            for (j = 0; j < ntab; j++) {
                struct potential *p = uniq[j];
                for (k = 0; k < (p->n + 1) * potential_chunk; k++) coef[8 * chunk0[j] + k] = (float)p->c[k];
            }
            for (k = 0; k < mt * mt; k++) {
                if (tabof[k] < 0) {
                    int m1 = -1;
                    ptab[k] = make_float4(0.f, 0.f, 0.f, 0.f);
                    memcpy(&ptab[k].w, &m1, sizeof(int));
                } else {
                    struct potential *p = uniq[tabof[k]];
                    unsigned int w = (unsigned int)p->n | ((unsigned int)chunk0[tabof[k]] << 9);
                    ptab[k] = make_float4((float)p->alpha[0], (float)p->alpha[1], (float)p->alpha[2], 0.f);
                    memcpy(&ptab[k].w, &w, sizeof(unsigned int));
                }
            }
            g->ntab = ntab;
            g->h_tabof = tabof;
            g->h_pair_ti = (int *)malloc(sizeof(int) * (ntab > 0 ? ntab : 1));
            g->h_pair_tj = (int *)malloc(sizeof(int) * (ntab > 0 ? ntab : 1));
            if (g->h_pair_ti == NULL || g->h_pair_tj == NULL) bad = engine_err_malloc;
            for (k = mt * mt - 1; !bad && k >= 0; k--)
                if (tabof[k] >= 0 && k / mt <= k % mt) {
                    g->h_pair_ti[tabof[k]] = k / mt;
                    g->h_pair_tj[tabof[k]] = k % mt;
                }
        }
        if (!bad) {
            if (hipMalloc(&g->d_ptab, sizeof(float4) * mt * mt) != hipSuccess ||
                hipMalloc(&g->d_coeffs, sizeof(float) * 8 * (nchunks > 0 ? nchunks : 1)) != hipSuccess ||
                hipMalloc(&g->d_ptype, sizeof(int) * mt * mt) != hipSuccess ||
                hipMemcpy(g->d_ptab, ptab, sizeof(float4) * mt * mt, hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(g->d_coeffs, coef, sizeof(float) * 8 * (nchunks > 0 ? nchunks : 1),
                          hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(g->d_ptype, tabof, sizeof(int) * mt * mt, hipMemcpyHostToDevice) != hipSuccess)
                bad = engine_err_gpu;
        }
        free(uniq);
        free(chunk0);
        free(ptab);
        free(coef);
        if (bad) {
            if (g->h_tabof != tabof) free(tabof);
            return gerror_(bad, bad == engine_err_potential ? "table with more than 511 intervals or too large"
                                                            : "table upload failed");
        }
    }

    /* Geometry constants of the sorted window (runner_dopair.c:424-428). */
    {
        struct nb_params *P = &g->P;
        memset(P, 0, sizeof(*P));
        P->ptab_bytes = (int)(sizeof(float4) * mt * mt);
        P->coef_bytes = (int)(sizeof(float) * 8 * (nchunks > 0 ? nchunks : 1));
        P->ncells = s->nr_cells;
        P->max_type = mt;
        /* engine_flag_unsorted: the reference's unsorted runner (runner.c:801-804,
           runner_dopair.c:1049-1290) evaluates every pair within the cutoff,
           which is the pair set of the projected window */
        P->proj = (e->flags & (engine_flag_projwindow | engine_flag_unsorted)) ? 1 : 0;
        P->bias = sqrt(s->h[0] * s->h[0] + s->h[1] * s->h[1] + s->h[2] * s->h[2]);
        P->dscale = (double)32767 / (2 * P->bias);
        P->dmaxdist = (int)(2 + P->dscale * (s->cutoff + 0.0 + 0.0));
        P->cutoff = s->cutoff;
        /* Packed record: key (16 bits) | slot (ibits) | type (16 - ibits). */
        {
            int tbits = 6;
            while ((1 << tbits) < mt) tbits += 2;
            P->tshift = 32 - tbits;
            P->imask = (1 << (16 - tbits)) - 1;
            g->maxcell = 1 << (16 - tbits);
        }
        P->maxdx = NULL;
        P->window = 0;
        /* k_pair's filter threshold: above the cutoff band by 16 roundings
           of the largest squared coordinate in an owner's frame (the four
           products, their sum and |x|^2 stay below 8 of them) */
        {
            double r2 = 0.0;
            for (k = 0; k < 3; k++) r2 += (s->span[k] + 2) * s->h[k] * (s->span[k] + 2) * s->h[k];
            P->filt = (float)(s->cutoff * s->cutoff * (1.0 + 2.1e-5) + r2 * 16.0 / 16777216.0);
        }
        P->cutoff2 = s->cutoff * s->cutoff;
        for (k = 0; k < 3; k++) {
            P->dim[k] = s->dim[k];
            P->h[k] = s->h[k];
        }
        P->rc2f = (float)P->cutoff2;
        /* FP32 r^2 of cell-relative coordinates is within ~2e-6 rc^2 of the
           FP64 value; pairs inside this band are decided in FP64. */
        P->band = 2.0e-5f * P->rc2f;
        HIPCHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_axis), cell_shift, sizeof(double) * 39));
    }

    /* Owner neighbour lists from the task list. */
    {
        int *cnt = (int *)calloc(s->nr_cells + 1, sizeof(int));
        int *fill, *off;
        int4 *nbr;
        float4 *nbs;
        int total = 0, maxnbr = 1;
        for (k = 0; k < s->nr_tasks; k++) {
            struct task *t = &s->tasks[k];
            if (t->type == task_type_self)
                cnt[t->i]++;
            else if (t->type == task_type_pair) {
                cnt[t->i]++;
                cnt[t->j]++;
            }
        }
        for (cid = 0; cid < s->nr_cells; cid++) {
            total += cnt[cid];
            if (cnt[cid] > maxnbr) maxnbr = cnt[cid];
        }
        nbr = (int4 *)malloc(sizeof(int4) * (total > 0 ? total : 1));
        fill = (int *)malloc(sizeof(int) * (s->nr_cells + 1));
        off = (int *)malloc(sizeof(int) * (s->nr_cells + 1));
        fill[0] = 0;
        for (cid = 0; cid < s->nr_cells; cid++) fill[cid + 1] = fill[cid] + cnt[cid];
        memcpy(off, fill, sizeof(int) * (s->nr_cells + 1));
        nbs = (float4 *)malloc(sizeof(float4) * (total > 0 ? total : 1));
        /* the cells' distance class of an entry, its square in cells, goes
           along in bits 16 and up */
        const float ih[3] = {(float)(1.0 / s->h[0]), (float)(1.0 / s->h[1]), (float)(1.0 / s->h[2])};
        const int ND = 256;
        int nd = 1; /* distance classes in use */
        for (k = 0; k < s->nr_tasks; k++) {
            struct task *t = &s->tasks[k];
            if (t->type == task_type_self) {
                nbs[fill[t->i]] = make_float4(0.f, 0.f, 0.f, 0.f);
                nbr[fill[t->i]++] = make_int4(t->i, 1 << 5, 0, 0);
            } else if (t->type == task_type_pair) {
                int dr, dp;
                task_dnshift(s, t->i, t->j, t->flags, g->P.dscale, &dr, &dp);
                const int win = task_window(g, s, dr, dp) << 8;
                if (win) g->P.window = 1;
                const float4 sh = cell_shift32(s, t->i, t->j);
                const float d[3] = {sh.x * ih[0], sh.y * ih[1], sh.z * ih[2]};
                const int d2 = (int)(d[0] * d[0] + d[1] * d[1] + d[2] * d[2] + 0.5f);
                const int dc = d2 < ND ? d2 : ND - 1;
                const int y = t->flags | win | (dc << 16);
                if (dc >= nd) nd = dc + 1;
                nbs[fill[t->i]] = sh;
                nbr[fill[t->i]++] = make_int4(t->j, y, dr, dp);
                nbs[fill[t->j]] = make_float4(-sh.x, -sh.y, -sh.z, 0.f);
                nbr[fill[t->j]++] = make_int4(t->i, y | (1 << 4), dr, dp);
            }
        }
        /* Per owner, the entries whose task has it as the i cell (the self
           task the very first), then the others; of both those without a
           window test first (k_pair's chunks then mostly need the test or do
           not), and nearer cells first: a chunk's cells then hold about as
           many hits for every owner atom. */
        {
            int4 *tn = (int4 *)malloc(sizeof(int4) * maxnbr);
            float4 *ts = (float4 *)malloc(sizeof(float4) * maxnbr);
            int *mid = (int *)malloc(sizeof(int) * s->nr_cells);
            int bin[4 * ND];
            if (tn == NULL || ts == NULL || mid == NULL) {
                free(tn);
                free(ts);
                free(mid);
                return gerror_(engine_err_malloc, "malloc failed");
            }
            auto cls = [nd, ND](const int4 &en) {
                return (((en.y >> 4) & 1) * 2 + ((en.y >> 8) & 1)) * nd + ((en.y >> 16) & (ND - 1));
            };
            for (cid = 0; cid < s->nr_cells; cid++) {
                const int b0 = off[cid], n = off[cid + 1] - off[cid];
                memcpy(tn, &nbr[b0], sizeof(int4) * n);
                memcpy(ts, &nbs[b0], sizeof(float4) * n);
                memset(bin, 0, sizeof(int) * 4 * nd);
                for (k = 0; k < n; k++) bin[cls(tn[k])]++;
                for (int b = 0, m = b0; b < 4 * nd; b++) {
                    if (b == 2 * nd) mid[cid] = m;
                    const int c = bin[b];
                    bin[b] = m;
                    m += c;
                }
                for (k = 0; k < n; k++) {
                    const int m = bin[cls(tn[k])]++;
                    nbr[m] = tn[k];
                    nbs[m] = ts[k];
                }
            }
            free(tn);
            free(ts);
            const bool badm =
                hipMalloc(&g->d_nbr_mid, sizeof(int) * s->nr_cells) != hipSuccess ||
                hipMemcpy(g->d_nbr_mid, mid, sizeof(int) * s->nr_cells, hipMemcpyHostToDevice) != hipSuccess;
            free(mid);
            if (badm) return gerror_(engine_err_gpu, "neighbour lists");
        }
        g->maxnbr = maxnbr;
        g->P.maxnbr = maxnbr;
        HIPCHECK(hipMalloc(&g->d_nbr, sizeof(int4) * (total > 0 ? total : 1)));
        HIPCHECK(hipMalloc(&g->d_nbr_off, sizeof(int) * (s->nr_cells + 1)));
        HIPCHECK(hipMemcpy(g->d_nbr, nbr, sizeof(int4) * (total > 0 ? total : 1), hipMemcpyHostToDevice));
        HIPCHECK(hipMalloc(&g->d_nbs, sizeof(float4) * (total > 0 ? total : 1)));
        HIPCHECK(hipMemcpy(g->d_nbs, nbs, sizeof(float4) * (total > 0 ? total : 1), hipMemcpyHostToDevice));
        HIPCHECK(hipMemcpy(g->d_nbr_off, off, sizeof(int) * (s->nr_cells + 1), hipMemcpyHostToDevice));
        free(cnt);
        free(fill);
        free(off);
        free(nbr);
        free(nbs);
    }

    /* Half-shell lists: the self task and each pair task once, at the task's
       i cell, and for each cell the i cells that visit it as the task's j
       cell, all in task order; of the latter each has slot 1 + its position
       (slot 0 is the self task), which the entry carries in its bits 9 and up. */
    {
        const int nc = s->nr_cells;
        int *hcnt = (int *)calloc(nc + 1, sizeof(int)), *icnt = (int *)calloc(nc + 1, sizeof(int));
        int *hoff = (int *)malloc(sizeof(int) * (nc + 1)), *ioff = (int *)malloc(sizeof(int) * (nc + 1));
        int *hfill = (int *)malloc(sizeof(int) * (nc + 1)), *ifill = (int *)malloc(sizeof(int) * (nc + 1));
        int htot = 0, itot = 0, bad = 0;
        int4 *nbr = NULL;
        float4 *nbs = NULL;
        int *icell = NULL;
        if (hcnt == NULL || icnt == NULL || hoff == NULL || ioff == NULL || hfill == NULL || ifill == NULL) bad = 1;
        for (k = 0; !bad && k < s->nr_tasks; k++) {
            const struct task *t = &s->tasks[k];
            if (t->type == task_type_self)
                hcnt[t->i]++;
            else if (t->type == task_type_pair) {
                hcnt[t->i]++;
                icnt[t->j]++;
            }
        }
        if (!bad) {
            hoff[0] = ioff[0] = 0;
            g->nslots = 1;
            for (cid = 0; cid < nc; cid++) {
                hoff[cid + 1] = hoff[cid] + hcnt[cid];
                ioff[cid + 1] = ioff[cid] + icnt[cid];
                if (icnt[cid] + 1 > g->nslots) g->nslots = icnt[cid] + 1;
            }
            htot = hoff[nc];
            itot = ioff[nc];
            memcpy(hfill, hoff, sizeof(int) * (nc + 1));
            memcpy(ifill, ioff, sizeof(int) * (nc + 1));
            nbr = (int4 *)malloc(sizeof(int4) * (htot > 0 ? htot : 1));
            nbs = (float4 *)malloc(sizeof(float4) * (htot > 0 ? htot : 1));
            icell = (int *)malloc(sizeof(int) * (itot > 0 ? itot : 1));
            if (nbr == NULL || nbs == NULL || icell == NULL) bad = 1;
        }
        for (k = 0; !bad && k < s->nr_tasks; k++) {
            const struct task *t = &s->tasks[k];
            if (t->type == task_type_self) {
                const int en = hfill[t->i]++;
                nbs[en] = make_float4(0.f, 0.f, 0.f, 0.f);
                nbr[en] = make_int4(t->i, 1 << 5, 0, 0);
            } else if (t->type == task_type_pair) {
                int dr, dp;
                const int en = hfill[t->i]++;
                const int slot = 1 + ifill[t->j] - ioff[t->j];
                task_dnshift(s, t->i, t->j, t->flags, g->P.dscale, &dr, &dp);
                nbs[en] = cell_shift32(s, t->i, t->j);
                nbr[en] = make_int4(t->j, t->flags | (slot << 9), dr, dp);
                icell[ifill[t->j]++] = t->i;
            }
        }
        if (!bad) {
            if (hipMalloc(&g->d_nbr_h, sizeof(int4) * (htot > 0 ? htot : 1)) != hipSuccess ||
                hipMalloc(&g->d_nbs_h, sizeof(float4) * (htot > 0 ? htot : 1)) != hipSuccess ||
                hipMalloc(&g->d_nbr_off_h, sizeof(int) * (nc + 1)) != hipSuccess ||
                hipMalloc(&g->d_inv_off, sizeof(int) * (nc + 1)) != hipSuccess ||
                hipMalloc(&g->d_inv_cell, sizeof(int) * (itot > 0 ? itot : 1)) != hipSuccess ||
                hipMemcpy(g->d_nbr_h, nbr, sizeof(int4) * (htot > 0 ? htot : 1), hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(g->d_nbs_h, nbs, sizeof(float4) * (htot > 0 ? htot : 1), hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(g->d_nbr_off_h, hoff, sizeof(int) * (nc + 1), hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(g->d_inv_off, ioff, sizeof(int) * (nc + 1), hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(g->d_inv_cell, icell, sizeof(int) * (itot > 0 ? itot : 1), hipMemcpyHostToDevice) !=
                    hipSuccess)
                bad = 2;
        }
        free(hcnt);
        free(icnt);
        free(hoff);
        free(ioff);
        free(hfill);
        free(ifill);
        free(nbr);
        free(nbs);
        free(icell);
        if (bad) return gerror_(bad == 1 ? engine_err_malloc : engine_err_gpu, "half-shell lists");
    }

    /* Cell origins, locations and sort masks. */
    {
        double *org = (double *)malloc(sizeof(double) * 3 * s->nr_cells);
        int *loc = (int *)malloc(sizeof(int) * 3 * s->nr_cells);
        unsigned int *sf = (unsigned int *)malloc(sizeof(unsigned int) * s->nr_cells);
        for (cid = 0; cid < s->nr_cells; cid++) {
            for (k = 0; k < 3; k++) {
                org[3 * cid + k] = s->cells[cid].origin[k];
                loc[3 * cid + k] = s->cells[cid].loc[k];
            }
            sf[cid] = s->cells[cid].sortflags;
        }
        HIPCHECK(hipMalloc(&g->d_origin, sizeof(double) * 3 * s->nr_cells));
        HIPCHECK(hipMalloc(&g->d_loc, sizeof(int) * 3 * s->nr_cells));
        HIPCHECK(hipMalloc(&g->d_sortflags, sizeof(unsigned int) * s->nr_cells));
        HIPCHECK(hipMemcpy(g->d_origin, org, sizeof(double) * 3 * s->nr_cells, hipMemcpyHostToDevice));
        HIPCHECK(hipMemcpy(g->d_loc, loc, sizeof(int) * 3 * s->nr_cells, hipMemcpyHostToDevice));
        HIPCHECK(hipMemcpy(g->d_sortflags, sf, sizeof(unsigned int) * s->nr_cells, hipMemcpyHostToDevice));
        free(org);
        free(loc);
        free(sf);
    }

    /* Exclusions as per-particle partner lists, by particle id. */
    {
        int maxid = -1;
        for (k = 0; k < s->size_parts; k++)
            if (s->partlist[k] != NULL) maxid = k;
        for (k = 0; k < e->nr_exclusions; k++) {
            if (e->exclusions[k].i > maxid) maxid = e->exclusions[k].i;
            if (e->exclusions[k].j > maxid) maxid = e->exclusions[k].j;
        }
        int nids = maxid + 1;
        int *xo = (int *)calloc(nids + 2, sizeof(int));
        int *xl = (int *)malloc(sizeof(int) * (2 * e->nr_exclusions + 1));
        int *fill = (int *)malloc(sizeof(int) * (nids + 1));
        for (k = 0; k < e->nr_exclusions; k++) {
            if (e->exclusions[k].i < 0 || e->exclusions[k].j < 0) continue;
            xo[e->exclusions[k].i + 1]++;
            xo[e->exclusions[k].j + 1]++;
        }
        for (k = 0; k < nids; k++) xo[k + 1] += xo[k];
        memcpy(fill, xo, sizeof(int) * (nids + 1));
        for (k = 0; k < e->nr_exclusions; k++) {
            i = e->exclusions[k].i;
            j = e->exclusions[k].j;
            if (i < 0 || j < 0) continue;
            xl[fill[i]++] = j;
            xl[fill[j]++] = i;
        }
        HIPCHECK(hipMalloc(&g->d_excl_off, sizeof(int) * (nids + 1)));
        HIPCHECK(hipMalloc(&g->d_excl_list, sizeof(int) * (2 * e->nr_exclusions + 1)));
        HIPCHECK(hipMemcpy(g->d_excl_off, xo, sizeof(int) * (nids + 1), hipMemcpyHostToDevice));
        HIPCHECK(hipMemcpy(g->d_excl_list, xl, sizeof(int) * (2 * e->nr_exclusions + 1), hipMemcpyHostToDevice));
        free(xo);
        free(xl);
        free(fill);
        g->nids = nids;
        if (gpu_alloc_ids(g, nids > 0 ? nids : 1) < 0) return engine_err_gpu;
    }

    {
        hipDeviceProp_t prop;
        HIPCHECK(hipGetDeviceProperties(&prop, g->device));
        g->ncu = prop.multiProcessorCount;
    }
    /* Few, densely filled cells: split each owner's neighbour list into
       nsplit groups, so that the pair kernel has ~MD_SPLIT_ITEMS_PER_CU work
       items per CU.  (With few atoms per cell a visit is short and the extra
       items cost more than they spread.) */
    g->nsplit = 1;
    if (!(e->flags & engine_flag_nosplit) && s->nr_cells < MD_SPLIT_ITEMS_PER_CU * g->ncu &&
        (long long)s->nr_parts >= (long long)engine_gpu_half_mean * s->nr_cells) {
        g->nsplit = (MD_SPLIT_ITEMS_PER_CU * g->ncu + s->nr_cells - 1) / s->nr_cells;
        if (g->nsplit > MD_SPLIT_MAX) g->nsplit = MD_SPLIT_MAX;
    }
    /* k_pair: one wave per item, at most MD_PAIR_ITEMS_PER_CU items per CU,
       whatever the cells hold (3 to 4 waves per SIMD are resident: with more
       items a second turn of waves starts).  us at 8, 12, 16, 20 and 28 items
       per CU: argon 1331 cells 66, 53, 52, 52, 60; mixture 125 cells 120, 114,
       137, 136, 138, 729 cells 170, 122, 114, 134, 132; water 512 cells 408,
       329, 414, 375, 395, 729 cells 706, 497, 575, 546, 574; and unsplit: argon
       64 cells 82, now 34, mixture 125 cells 618, now 116.  (The sweep with FP32
       force sums.) */
    g->nsplit_t = 1;
    if (!(e->flags & engine_flag_nosplit)) {
        int cap = g->maxnbr / 2 < MD_PAIR_SPLIT_MAX ? g->maxnbr / 2 : MD_PAIR_SPLIT_MAX;
        g->nsplit_t = MD_PAIR_ITEMS_PER_CU * g->ncu / s->nr_cells;
        if (g->nsplit_t > cap) g->nsplit_t = cap;
        if (g->nsplit_t < 1) g->nsplit_t = 1;
    }
    const int maxsplit = g->nsplit > g->nsplit_t ? g->nsplit : g->nsplit_t;
    {
        /* Owner cells in blocks of 6x6x6, blocks and the cells inside them in
           raster order: the owners a compute die works on at once, and their
           neighbours, stay close together in its L2. */
        int *ord = (int *)malloc(sizeof(int) * (size_t)s->nr_cells);
        if (ord == NULL) return gerror_(engine_err_malloc, "malloc failed");
        const int B = 6, nbx = (s->cdim[0] + B - 1) / B, nby = (s->cdim[1] + B - 1) / B,
                  nbz = (s->cdim[2] + B - 1) / B;
        int q = 0;
        for (int bx = 0; bx < nbx; bx++)
            for (int by = 0; by < nby; by++)
                for (int bz = 0; bz < nbz; bz++)
                    for (int x = bx * B; x < (bx + 1) * B && x < s->cdim[0]; x++)
                        for (int y = by * B; y < (by + 1) * B && y < s->cdim[1]; y++)
                            for (int z = bz * B; z < (bz + 1) * B && z < s->cdim[2]; z++)
                                ord[q++] = space_cellid(s, x, y, z);
        if (q != s->nr_cells) {
            free(ord);
            return gerror_(engine_err_range, "cell order");
        }
        HIPCHECK(hipMalloc(&g->d_order, sizeof(int) * (size_t)s->nr_cells));
        HIPCHECK(hipMemcpy(g->d_order, ord, sizeof(int) * (size_t)s->nr_cells, hipMemcpyHostToDevice));
        free(ord);
        g->P.order = g->d_order;
    }
    HIPCHECK(hipMalloc(&g->d_kminmax, sizeof(unsigned short) * 26 * (size_t)s->nr_cells));
    HIPCHECK(hipMalloc(&g->d_cnt_off, sizeof(int2) * s->nr_cells));
    HIPCHECK(hipMalloc(&g->d_cell_acc, sizeof(double) * 3 * (size_t)s->nr_cells * maxsplit));
    HIPCHECK(hipMalloc(&g->d_cell_cnt, sizeof(unsigned long long) * 3 * (size_t)s->nr_cells * maxsplit));
    HIPCHECK(hipMalloc(&g->d_tot, sizeof(double) * 4));
    HIPCHECK(hipMalloc(&g->d_red_acc, sizeof(double) * 3 * MD_RED_BLOCKS));
    HIPCHECK(hipMalloc(&g->d_red_cnt, sizeof(unsigned long long) * 3 * MD_RED_BLOCKS));
    HIPCHECK(hipMalloc(&g->d_tot_cnt, sizeof(unsigned long long) * 4));
    HIPCHECK(hipMalloc(&g->d_queue, sizeof(int) * MD_NQUEUE));
    g->queue_used = 1;
    HIPCHECK(hipHostMalloc((void **)&g->h_count, sizeof(int) * s->nr_cells, hipHostMallocDefault));
    HIPCHECK(hipMalloc(&g->d_cell_maxdx, sizeof(double) * s->nr_cells));
    HIPCHECK(hipHostMalloc((void **)&g->h_cell_maxdx, sizeof(double) * s->nr_cells, hipHostMallocDefault));
    if ((g->h_sort_count = (int *)calloc(s->nr_cells, sizeof(int))) == NULL)
        return gerror_(engine_err_malloc, "malloc failed");
    g->sort_valid = 0;
    HIPCHECK(hipHostMalloc((void **)&g->h_offset, sizeof(int) * (s->nr_cells + 1), hipHostMallocDefault));
    HIPCHECK(hipHostMalloc((void **)&g->h_flag, sizeof(int), hipHostMallocDefault));
    *g->h_flag = 0;
    HIPCHECK(hipHostMalloc((void **)&g->h_tot, sizeof(double) * 4, hipHostMallocDefault));
    HIPCHECK(hipHostMalloc((void **)&g->h_tot_cnt, sizeof(unsigned long long) * 4, hipHostMallocDefault));

    return engine_err_ok;
}

/* Pack host particles in cell order and upload them; the device arrays of a
   pass are those of the particles afterwards (gpu_launch: packed). */
int gpu_upload(struct engine *e) {
    struct gpu_state *g = (struct gpu_state *)e->gpu;
    struct space *s = &e->s;
    int cid, n = 0, maxc = 0, maxid = -1;
    for (cid = 0; cid < s->nr_cells; cid++) {
        int c = s->cells[cid].count;
        if (c > maxc) maxc = c;
        n += c;
    }
    if (maxc > g->maxcell)
        return gerror_(engine_err_maxparts, "more particles in a cell than the packed record holds (1024 for up to "
                                            "64 types, 256 for up to 256, 64 for up to 1024)");
    /* the copy of an upload whose call ended in an error before its end */
    if (g->staging) HIPCHECK(hipStreamSynchronize(g->stream));
    g->staging = 0;
    if (gpu_alloc_parts(g, n > 0 ? n : 1) < 0) return engine_err_gpu;
    /* the id clearing runs while the host packs */
    if (gpu_clear_ids(g) < 0) return engine_err_gpu;
    /* one block: positions, types, ids, (count, offset) per cell */
    g->h_x = (double *)g->h_stage;
    g->h_type = (int *)(g->h_x + 3 * (size_t)n);
    g->h_id = g->h_type + n;
    g->h_cnt_off = (int2 *)(g->h_id + n);
    g->d_flo = g->d_fhi + n;
    g->h_flo = g->h_fhi + n;
    if (space_pack(s, g->max_type, g->h_count, g->h_offset, (int *)g->h_cnt_off, g->h_x, g->h_type, g->h_id, &maxc,
                   &maxid) < 0)
        return gerror_(engine_err_range, "particle type out of range");
    if (maxid + 1 > g->nids) return gerror_(engine_err_range, "particle id beyond the ids known at engine_gpu_load");
    g->nparts = n;
    g->maxcount = maxc;
    g->paired = !(e->flags & engine_flag_unpaired);
    /* default shell: the full shell, except for densely filled cells that are
       fewer than the device's CUs, or with engine_flag_unpaired.  There too
       k_pair is the faster one now (water, 27, 64 and 125 cells of 111 to 125
       atoms: 244, 166 and 302 us against 261, 234 and 384), but its energy sums
       run in another order than the half shell's: where pair and exclusion
       energies cancel, the total differs by up to 4e-6 of itself. */
    g->half = (e->flags & engine_flag_halfshell)   ? 1
              : (e->flags & engine_flag_fullshell) ? 0
                                                   : (long long)n >= (long long)engine_gpu_half_mean * s->nr_cells &&
                                                         (!g->paired || s->nr_cells < g->ncu);
    /* surrogate mode: the network evaluation dominates a visit, so the half
       shell's single evaluation per pair wins at any occupancy */
    g->mlp_half = !(e->flags & engine_flag_fullshell);
    g->P.nparts = n;
    g->P.nids = g->nids;
    g->P.maxn = maxc > 0 ? maxc : 1;
    g->staging = 1;
    HIPCHECK(hipMemcpyAsync(g->d_stage, g->h_stage, GPU_STAGE_BYTES(n, s->nr_cells), hipMemcpyHostToDevice, g->stream));
    {
        const double *x = (const double *)g->d_stage;
        const int *type = (const int *)(x + 3 * (size_t)n), *id = type + n;
        hipLaunchKernelGGL(k_pack, dim3((s->nr_cells + 3) / 4), dim3(256), 0, g->stream, s->nr_cells, n,
                           (const int2 *)(id + n), x, type, id, g->d_xf, g->d_index_of_id, g->d_cell_of, g->d_x,
                           g->d_type, g->d_id, g->d_count, g->d_offset, g->d_cnt_off);
        HIPCHECK(hipGetLastError());
    }
    return engine_err_ok;
}

/* No slot for any particle id. */
int gpu_clear_ids(struct gpu_state *g) {
    const int nb = (g->nids + 255) / 256;
    if (nb > 0) hipLaunchKernelGGL(k_clear_ids, dim3(nb), dim3(256), 0, g->stream, g->nids, g->d_index_of_id);
    HIPCHECK(hipGetLastError());
    return engine_err_ok;
}

/* Launch the kernels of one pass on the resident particles, with events
   around each when timed (2: around the whole); mlp selects the surrogate mode of the pair kernel.
   sort: 0 keeps the keys and sort lists of the last sort; packed: d_xf and
   the id and cell maps are those of the particles already. */
int gpu_launch(struct gpu_state *g, int timed, int mlp, int sort, int packed) {
    /* 32 owner atoms at a time while most cells fit (argon 108,000 atoms, at
       26 and 32 per cell: 95 and 93 us against 135 and 131 with 64, whose LDS
       share and registers leave 3 waves per SIMD instead of 4); beyond, the
       cell's neighbours would be staged twice (at 39, 49 and 62 per cell 201,
       226 and 213 us with 32, 135, 157 and 149 with 64; water at 125 per cell
       434 and 328; all with FP32 force sums) */
    const int big = (long long)g->nparts > (long long)MD_PAIR_R64_MEAN * g->ncells;
    const int half = mlp ? g->mlp_half : g->half, pair = !mlp && !half;
    /* table mode on the half shell: 5 waves per SIMD where the cells fill
       them (measured equal to 4 at 64 cells per CU, ahead above) */
    const int wide = !mlp && half && g->ncells >= 64 * g->ncu;
    struct nb_params P = g->P;
    P.walk_cap = g->ncells >= MD_WALK_CELLS ? 28 : 32;
    const int nsplit = P.nsplit = pair ? g->nsplit_t : g->nsplit;
    int nb;
    size_t lds = 0;
    const size_t maxn = (size_t)P.maxn;
    if (!pair) {
        lds = sizeof(float4) * 64; /* raw */
        P.lds_own_key = (int)lds;
        lds += sizeof(unsigned short) * 13 * 64;
        lds = (lds + 15) & ~(size_t)15;
        P.lds_kfl = (int)lds;
        lds += sizeof(int) * 32;
        lds = (lds + 15) & ~(size_t)15;
        P.lds_stage = (int)lds;
        lds += sizeof(float4) * maxn;
        P.lds_hit = (int)lds;
        lds += sizeof(unsigned short) * 64 * (mlp ? MD_HCAP_MLP : wide ? MD_HCAP_WIDE : MD_HCAP);
        lds = (lds + 15) & ~(size_t)15;
        P.lds_dense = (int)lds;
        if (mlp) lds += 16 * 64 * MD_HCAP_MLP + 4 * 64 * MD_XCAP_MLP + sizeof(float) * 2 * MLP_H;
        lds = (lds + 15) & ~(size_t)15;
        P.lds_jf = (int)lds;
        if (half) lds += sizeof(float) * 4 * 3 * maxn;
        if (lds > 64 * 1024) return gerror_(engine_err_maxparts, "LDS staging exceeds 64 KiB");
    }
    if (half && g->jcap < (size_t)g->nslots * g->nparts) {
        /* per slot, the forces on every atom; no pending pass may still use
           the old buffer */
        HIPCHECK(hipStreamSynchronize(g->stream));
        (void)hipFree(g->d_jpart);
        g->d_jpart = NULL;
        g->jcap = 0;
        HIPCHECK(hipMalloc(&g->d_jpart, sizeof(float) * 3 * (size_t)g->nslots * g->nparts));
        g->jcap = (size_t)g->nslots * g->nparts;
    }
    if (nsplit > 1 && g->pcap < (size_t)nsplit * g->nparts) {
        /* per neighbour group, the owner forces of every atom; no pending
           pass may still use the old buffers */
        HIPCHECK(hipStreamSynchronize(g->stream));
        (void)hipFree(g->d_phi);
        (void)hipFree(g->d_plo);
        g->d_phi = g->d_plo = NULL;
        g->pcap = 0;
        HIPCHECK(hipMalloc(&g->d_phi, sizeof(float4) * (size_t)nsplit * g->nparts));
        HIPCHECK(hipMalloc(&g->d_plo, sizeof(float4) * (size_t)nsplit * g->nparts));
        g->pcap = (size_t)nsplit * g->nparts;
    }
    const int kern = mlp ? half : 2 + wide; /* kernels that walk the sorted windows */
    if (!pair && lds != g->lds_nb[kern]) {
        /* Persistent grid: as many single-wave blocks as can be resident. */
        const void *const fn[4] = {(const void *)k_nonbond_mlp, (const void *)k_nonbond_mlp_half,
                                   (const void *)k_nonbond_half, (const void *)k_nonbond_half_wide};
        int per_cu = 0;
        HIPCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn[kern], 64, lds));
        if (per_cu < 1) per_cu = 1;
        g->grid_nb[kern] = g->ncu * per_cu;
        g->lds_nb[kern] = lds;
    }
    if (mlp && g->mlp_np == 0) return gerror_(engine_err_range, "engine_flag_mlp without engine_mlp_init");
    if (!sort && !g->sort_valid) return gerror_(engine_err_range, "no sort lists to reuse");

    if (timed) HIPCHECK(hipEventRecord(g->ev[0], g->stream));
    if (!packed && gpu_clear_ids(g) < 0) return engine_err_gpu;
    if (!packed)
        hipLaunchKernelGGL(k_pack, dim3((g->ncells + 3) / 4), dim3(256), 0, g->stream, g->ncells, g->nparts,
                           g->d_cnt_off, g->d_x, g->d_type, g->d_id, g->d_xf, g->d_index_of_id, g->d_cell_of,
                           (double *)NULL, (int *)NULL, (int *)NULL, (int *)NULL, (int *)NULL, (int2 *)NULL);
    if (!sort) {
        /* pseudo-Verlet step between rebuilds: the keys and sort lists of
           the last sort stay (runner.c:773) */
    } else if (g->maxcount <= MD_SORT_LDS_MAX) {
        const int maxn = g->maxcount > 0 ? g->maxcount : 1;
        const size_t sh = sizeof(double) * 3 * maxn + sizeof(unsigned int) * 13 * maxn +
                          sizeof(int) * 13 * 2 * MD_SORT_STACK + sizeof(unsigned short) * (13 * 2 * (maxn + 1) + 136);
        /* one wave per cell; for large cells (frequent repeated keys) and for
           few cells one wave per direction */
        const int bs = maxn > MD_SORT_ONEWAVE_MAX || g->ncells <= MD_SORT_FEW ? 13 * 64 : 64;
        hipLaunchKernelGGL(k_sort_rank, dim3(g->ncells), dim3(bs), sh, g->stream, P, g->d_count, g->d_offset,
                           g->d_sortflags, g->d_x, g->d_sortlist, g->d_keyof, g->d_kminmax, g->h_flag,
                           maxn);
    } else {
        nb = (g->ncells * 13 + 255) / 256;
        hipLaunchKernelGGL(k_sort, dim3(nb), dim3(256), 0, g->stream, P, g->d_count, g->d_offset, g->d_sortflags,
                           g->d_x, g->d_sortlist, g->d_keyof, g->d_kminmax, g->h_flag);
    }
    if (sort) g->sort_valid = 1;
    if (timed == 1) HIPCHECK(hipEventRecord(g->ev[1], g->stream));
    struct nb_out O;
    O.fhi = g->d_fhi;
    O.flo = g->d_flo;
    O.cell_acc = g->d_cell_acc;
    O.cell_cnt = g->d_cell_cnt;
    O.jpart = g->d_jpart;
    O.phi = g->d_phi;
    O.plo = g->d_plo;
    const int nitems = g->ncells * nsplit;
    if (pair) {
        static const decltype(&k_pair<32, 0, false>) kp[2][3][2] = {
            {{k_pair<32, 0, false>, k_pair<32, 0, true>},
             {k_pair<32, 1, false>, k_pair<32, 1, true>},
             {k_pair<32, 2, false>, k_pair<32, 2, true>}},
            {{k_pair<64, 0, false>, k_pair<64, 0, true>},
             {k_pair<64, 1, false>, k_pair<64, 1, true>},
             {k_pair<64, 2, false>, k_pair<64, 2, true>}}};
        /* the tables in LDS as far as PT_TAB bytes hold them: with them 4
           blocks of 4 waves still fit on a CU, and every access kept from the
           L1 counts (argon 864,000 atoms, all in LDS: 622 -> 595 us; 20 types,
           the headers: 4180 -> 3670 us; with FP32 force sums) */
        const int tabs = P.ptab_bytes + P.coef_bytes <= PT_TAB ? 2 : P.ptab_bytes <= PT_TAB ? 1 : 0;
        const size_t plds = PT_WAVES * (big ? sizeof(pair_lds<64>) : sizeof(pair_lds<32>)) +
                            (tabs ? P.ptab_bytes : 0) + (tabs == 2 ? P.coef_bytes : 0);
        /* the same number of blocks for each die */
        const int nblocks = (nitems + PT_WAVES - 1) / PT_WAVES;
        const dim3 grid((nblocks + MD_NQUEUE - 1) / MD_NQUEUE * MD_NQUEUE);
        hipLaunchKernelGGL(kp[big][tabs][P.proj != 0], grid, dim3(64 * PT_WAVES), plds, g->stream, P, g->d_cnt_off,
                           g->d_nbr, g->d_nbr_off,
                           g->d_nbr_mid, g->d_nbs, g->d_origin, g->d_loc, g->d_xf, g->d_x, g->d_id,
                           g->d_kminmax, g->d_sortlist, g->d_keyof, g->d_ptab, (const float4 *)g->d_coeffs,
                           g->d_excl_off, g->d_excl_list, g->d_index_of_id, g->d_cell_of, O);
    } else {
        /* new, or left used up by a pass that ended in an error before its totals */
        if (g->queue_used) hipLaunchKernelGGL(k_clear_queue, dim3(1), dim3(64), 0, g->stream, g->d_queue);
        g->queue_used = 1;
        /* no more waves than work items: the dispatcher then spreads them
           over all compute units */
        const dim3 grid(g->grid_nb[kern] < nitems ? g->grid_nb[kern] : nitems);
        const int4 *nbr = half ? g->d_nbr_h : g->d_nbr;
        const int *off = half ? g->d_nbr_off_h : g->d_nbr_off;
        const float4 *nbs = half ? g->d_nbs_h : g->d_nbs;
        if (mlp)
            hipLaunchKernelGGL(half ? k_nonbond_mlp_half : k_nonbond_mlp, grid, dim3(64), lds, g->stream, P,
                               g->d_cnt_off, nbr, off, nbs, g->d_origin, g->d_loc, g->d_xf, g->d_x, g->d_id,
                               g->d_sortlist, g->d_keyof, g->d_ptab, (const float4 *)g->d_coeffs, g->d_excl_off,
                               g->d_excl_list, g->d_index_of_id, g->d_cell_of, O, g->d_queue, gpu_mlp_net(g),
                               g->d_ptype);
        else
            hipLaunchKernelGGL(wide ? k_nonbond_half_wide : k_nonbond_half, grid, dim3(64), lds, g->stream, P,
                               g->d_cnt_off, nbr, off, nbs, g->d_origin, g->d_loc, g->d_xf, g->d_x, g->d_id,
                               g->d_sortlist, g->d_keyof, g->d_ptab, (const float4 *)g->d_coeffs, g->d_excl_off,
                               g->d_excl_list, g->d_index_of_id, g->d_cell_of, O, g->d_queue);
    }
    if (half || nsplit > 1)
        hipLaunchKernelGGL(k_fold, dim3(g->ncells), dim3(64), 0, g->stream, g->ncells, g->d_cnt_off, nsplit,
                           g->nparts, (const float4 *)g->d_phi, (const float4 *)g->d_plo, half,
                           g->d_inv_off, g->d_inv_cell, g->d_jpart, g->d_fhi, g->d_flo);
    if (timed == 1) HIPCHECK(hipEventRecord(g->ev[2], g->stream));
    if (nitems <= MD_RED_ONE)
        hipLaunchKernelGGL(k_reduce_one, dim3(1), dim3(256), 0, g->stream, nitems, g->d_cell_acc, g->d_cell_cnt,
                           g->d_tot, g->d_tot_cnt, g->h_tot, g->h_tot_cnt, g->d_queue);
    else {
        hipLaunchKernelGGL(k_reduce_a, dim3(MD_RED_BLOCKS), dim3(256), 0, g->stream, nitems, g->d_cell_acc,
                           g->d_cell_cnt, g->d_red_acc, g->d_red_cnt);
        hipLaunchKernelGGL(k_reduce_b, dim3(1), dim3(256), 0, g->stream, MD_RED_BLOCKS, g->d_red_acc, g->d_red_cnt,
                           g->d_tot, g->d_tot_cnt, g->h_tot, g->h_tot_cnt, g->d_queue);
    }
    if (timed) HIPCHECK(hipEventRecord(g->ev[3], g->stream));
    HIPCHECK(hipGetLastError());
    g->queue_used = 0;
    return engine_err_ok;
}

extern "C" int engine_gpu_sync(struct engine *e, unsigned int what) {
    struct gpu_state *g;
    struct space *s;
    int cid;
    if (e == NULL) return gerror_(engine_err_null, "NULL engine");
    g = (struct gpu_state *)e->gpu;
    if (g == NULL) return gerror_(engine_err_nogpu, "engine_gpu_load was not called");
    s = &e->s;
    HIPCHECK(hipSetDevice(g->device));
    if (what & engine_gpu_sync_parts_up) {
        if (gpu_upload(e) < 0) return engine_err_gpu;
        HIPCHECK(hipStreamSynchronize(g->stream));
        g->staging = 0;
    }
    if (what & engine_gpu_sync_sort_down) {
        unsigned int *tmp = (unsigned int *)malloc(sizeof(unsigned int) * 13 * (size_t)(g->nparts > 0 ? g->nparts : 1));
        if (tmp == NULL) return gerror_(engine_err_malloc, "malloc failed");
        if (hipMemcpy(tmp, g->d_sortlist, sizeof(unsigned int) * 13 * (size_t)g->nparts, hipMemcpyDeviceToHost) !=
            hipSuccess) {
            free(tmp);
            return gerror_(engine_err_gpu, "sortlist download failed");
        }
        for (cid = 0; cid < s->nr_cells; cid++) {
            struct cell *c = &s->cells[cid];
            if (c->count != g->h_count[cid]) {
                free(tmp);
                return gerror_(engine_err_range, "cells changed since the last pass");
            }
            memcpy(c->sortlist, &tmp[13 * (size_t)g->h_offset[cid]], sizeof(unsigned int) * 13 * c->count);
        }
        free(tmp);
    }
    if (what & engine_gpu_sync_forces_down) {
        HIPCHECK(hipMemcpyAsync(g->h_fhi, g->d_fhi, sizeof(float4) * 2 * g->nparts, hipMemcpyDeviceToHost, g->stream));
        HIPCHECK(hipMemcpyAsync(g->h_tot, g->d_tot, sizeof(double) * 3, hipMemcpyDeviceToHost, g->stream));
        HIPCHECK(hipMemcpyAsync(g->h_tot_cnt, g->d_tot_cnt, sizeof(unsigned long long) * 3, hipMemcpyDeviceToHost,
                                g->stream));
        HIPCHECK(hipStreamSynchronize(g->stream));
    }
    return engine_err_ok;
}

/* Pseudo-Verlet (engine_flag_verlet*): the pass sorts only on a rebuild
   step (runner.c:773) and widens each pair window by the cells' maxdx
   (runner_dopair.c:428).  Sets *sort and the device per-cell maxdx; a pass
   that reuses the sort lists needs the layout of the last sort. */
static int gpu_verlet(struct engine *e, struct gpu_state *g, int *sort) {
    struct space *s = &e->s;
    int cid;
    if (!(e->flags & engine_flag_verlet)) {
        g->P.maxdx = NULL;
        *sort = 1;
        return engine_err_ok;
    }
    for (cid = 0; cid < s->nr_cells; cid++) g->h_cell_maxdx[cid] = s->cells[cid].maxdx;
    HIPCHECK(hipMemcpyAsync(g->d_cell_maxdx, g->h_cell_maxdx, sizeof(double) * s->nr_cells, hipMemcpyHostToDevice,
                            g->stream));
    g->P.maxdx = g->d_cell_maxdx;
    *sort = s->verlet_rebuild != 0;
    if (!*sort) {
        if (!g->sort_valid) return gerror_(engine_err_range, "no sort lists to reuse");
        for (cid = 0; cid < s->nr_cells; cid++)
            if (s->cells[cid].count != g->h_sort_count[cid])
                return gerror_(engine_err_range, "cells changed since the last sort");
    }
    return engine_err_ok;
}

static double gpu_wall(void) {
    struct timespec ts;
    clock_gettime(CLOCK_MONOTONIC, &ts);
    return (double)ts.tv_sec + 1e-9 * (double)ts.tv_nsec;
}

/* Counts of the layout the sort lists belong to. */
static void gpu_sorted(struct engine *e, struct gpu_state *g) {
    for (int cid = 0; cid < e->s.nr_cells; cid++) g->h_sort_count[cid] = e->s.cells[cid].count;
}

extern "C" int engine_nonbond_gpu(struct engine *e) {
    struct gpu_state *g;
    struct space *s;
    if (e == NULL) return gerror_(engine_err_null, "NULL engine");
    g = (struct gpu_state *)e->gpu;
    if (g == NULL) return gerror_(engine_err_nogpu, "engine_gpu_load was not called");
    s = &e->s;
    HIPCHECK(hipSetDevice(g->device));
    double tw = gpu_wall();
    if (gpu_upload(e) < 0) return engine_err_gpu;
    e->timers[engine_timer_gpu_load] = gpu_wall() - tw;
    int sort = 1;
    if (gpu_verlet(e, g, &sort) < 0) return engine_err_range;
    *g->h_flag = 0; /* nothing is under way that could set it */
    if (gpu_launch(g, 2, (e->flags & engine_flag_mlp) != 0, sort, 1) < 0) return engine_err_gpu;
    HIPCHECK(hipMemcpyAsync(g->h_fhi, g->d_fhi, sizeof(float4) * 2 * g->nparts, hipMemcpyDeviceToHost, g->stream));
    if (sort) gpu_sorted(e, g); /* meanwhile */
    HIPCHECK(hipStreamSynchronize(g->stream));
    g->staging = 0;
    if (*(const volatile int *)g->h_flag) return gerror_(engine_err_range, "sort stack overflow");
    {
        float ms = 0.0f;
        HIPCHECK(hipEventElapsedTime(&ms, g->ev[0], g->ev[3]));
        e->timers[engine_timer_gpu_kernels] = ms * 1e-3;
    }
    tw = gpu_wall();
    space_add_forces_slots(s, g->h_offset, (const float *)g->h_fhi, (const float *)g->h_flo);
    e->timers[engine_timer_gpu_unload] = gpu_wall() - tw;
    s->epot_nonbond += g->h_tot[0];
    s->epot_exclusion += g->h_tot[1];
    s->epot += g->h_tot[0] + g->h_tot[1];
    s->virial += g->h_tot[2];
    s->nr_pairs += (long long)g->h_tot_cnt[0];
    s->nr_excl_evaluated += (long long)g->h_tot_cnt[1];
    return engine_err_ok;
}

extern "C" int engine_gpu_time(struct engine *e, int nsteps, int nwarm, double *ms) {
    struct gpu_state *g;
    double acc[4] = {0, 0, 0, 0};
    float t;
    int k;
    if (e == NULL || ms == NULL) return gerror_(engine_err_null, "NULL argument");
    g = (struct gpu_state *)e->gpu;
    if (g == NULL || g->nparts_cap == 0) return gerror_(engine_err_nogpu, "no resident particles");
    HIPCHECK(hipSetDevice(g->device));
    /* the sort of a pass that engine_step would make, on the resident data */
    const int sort = !(e->flags & engine_flag_verlet) || e->s.verlet_rebuild || !g->sort_valid;
    for (k = 0; k < nwarm; k++)
        if (gpu_launch(g, 0, (e->flags & engine_flag_mlp) != 0, sort, 0) < 0) return engine_err_gpu;
    HIPCHECK(hipStreamSynchronize(g->stream));
    for (k = 0; k < nsteps; k++) {
        if (gpu_launch(g, 1, (e->flags & engine_flag_mlp) != 0, sort, 0) < 0) return engine_err_gpu;
        HIPCHECK(hipEventSynchronize(g->ev[3]));
        HIPCHECK(hipEventElapsedTime(&t, g->ev[0], g->ev[1]));
        acc[0] += t;
        HIPCHECK(hipEventElapsedTime(&t, g->ev[1], g->ev[2]));
        acc[1] += t;
        HIPCHECK(hipEventElapsedTime(&t, g->ev[2], g->ev[3]));
        acc[2] += t;
        HIPCHECK(hipEventElapsedTime(&t, g->ev[0], g->ev[3]));
        acc[3] += t;
    }
    for (k = 0; k < 4; k++) ms[k] = (nsteps > 0) ? acc[k] / nsteps : 0.0;
    HIPCHECK(hipMemcpyAsync(g->h_tot, g->d_tot, sizeof(double) * 3, hipMemcpyDeviceToHost, g->stream));
    HIPCHECK(hipMemcpyAsync(g->h_tot_cnt, g->d_tot_cnt, sizeof(unsigned long long) * 3, hipMemcpyDeviceToHost,
                            g->stream));
    HIPCHECK(hipStreamSynchronize(g->stream));
    return engine_err_ok;
}

extern "C" int engine_gpu_results(struct engine *e, double *out, long long *counts) {
    struct gpu_state *g;
    if (e == NULL) return gerror_(engine_err_null, "NULL engine");
    g = (struct gpu_state *)e->gpu;
    if (g == NULL) return gerror_(engine_err_nogpu, "engine_gpu_load was not called");
    if (out) {
        out[0] = g->h_tot[0];
        out[1] = g->h_tot[1];
        out[2] = g->h_tot[2];
    }
    if (counts) {
        counts[0] = (long long)g->h_tot_cnt[0];
        counts[1] = (long long)g->h_tot_cnt[1];
        counts[2] = (long long)g->h_tot_cnt[2];
    }
    return engine_err_ok;
}
