/*
 * The full-shell table kernel: matrix-core distance filter, hits dealt over
 * the lanes.  Included by engine_gpu.hip (uses its device helpers).
 *
 * One wave works on one owner cell (at most R of its atoms at a time) and a
 * share of the neighbour cells (runner_dopair / runner_doself tasks that
 * touch it): first the entries whose task has the owner as its i cell (and
 * the self task), then those whose task has it as its j cell (and the self
 * task again, its pairs split between the two).  Of each side the entries go
 * 64 at a time; their atoms, each cell padded to a multiple of 4 slots, are
 * concatenated and taken TC slots at a time:
 *   stage   slot t of the chunk: the atom's position in the owner's frame
 *           (x + the entry's shift), its |x|^2, its type, entry and key.  An
 *           i entry's atoms come in the order of the reference's window
 *           (ascending keys);
 *   filter  v_mfma_f32_16x16x4_f32 gives |xi|^2 + |xj|^2 - 2 xi.xj - thr of
 *           16 slots x 16 owner atoms per instruction (operand rows
 *           (x, y, z, |x|^2), columns (-2x, -2y, -2z, 1), |xi|^2 - thr as
 *           the initial accumulator).  Its sign bit is shifted into a
 *           bitmap (one v_alignbit per value): bit b of word (i, k) is slot
 *           32 k + b.  thr lies above the cutoff by the error of this sum,
 *           so no pair within the cutoff is missed;
 *   i side  takes the energy, the virial and the counts.  Atom i's hits
 *           belong to its NPi lanes (i, part), every NPi-th record of an
 *           entry's window to one lane, in window order: a lane's FP32 sums
 *           run over one entry before they go into FP64, so that they are
 *           those of a walk along the sorted window, whatever the chunks;
 *   j side  has forces only, so its order is free: the H set bits are dealt
 *           to the 64 lanes in runs of Q = ceil(H / 64), in atom order.  The
 *           run that begins an atom stores its sum at the atom's slot, one
 *           that goes on with it at its own, and each atom adds them in the
 *           order of the runs.
 * Both evaluate with the same two steps: distance, the reference's window
 * test where it can matter, the FP64 cutoff band and the request of the
 * table's coefficients for one hit, while the hit before is applied.  Forces
 * add up in FP64 from the product on, on both sides, and leave as (hi, lo).
 * With FP32 sums over a lane's hits of a chunk (about 10) and two-sums between
 * chunks, an atom's forces in different cells met in FP32: small ones beside
 * large ones that cancel were lost, and the relative force error of the
 * mixture was 1.381e-6 at 1,048,576 atoms, now 1.373e-6 (FP32 sums over one
 * visited cell: 1.374e-6).  It adds 1.7 % VALU instructions, four conversions
 * per hit less the two-sums, and up to 5 % of the time, since the FP64 ones take
 * more than one issue cycle (1,048,576 atoms, mixture 3650 -> 3830 us, argon
 * 729 -> 770), nearly all of it on the j side.
 *
 * The set of pairs is the reference's.  Its sorted window
 * (runner_dopair.c:455-478) admits (i, j) exactly when
 * key_j + dnshift - key_i < dmaxdist, whatever the order of equal keys, and
 * skips a whole task whose largest key_i exceeds its smallest
 * key_j + dnshift.  The test is skipped for entries whose offset lies along
 * the sort axis (dnshift not above the projected one): there
 * key_j + dnshift - key_i <= dscale (x_j + shift - x_i).n + 1 <= dscale rc + 1
 * < dmaxdist for every pair within the cutoff.
 *
 * What bounds it: the VALU (81 % of its issue cycles filled on 20 types, and the
 * FP64 instructions take longer), 75 instructions per hit and lane on the i
 * side at half the lanes busy (an atom's hits per chunk differ), 64 on the j
 * side at 97 %; with 20 types the coefficients come next, 384 KB of tables read
 * at random through the 32 KB L1.  The L1 serves about a lane a clock, so a
 * lane without a hit asks for nothing (mixture 1,048,576, with FP32 force sums:
 * 3.0e9 accesses, 1.2 a clock, 4360 us; without them 2.3e9, 4180), and the
 * table headers lie in LDS (1.6e9, 3670), copied once per PT_WAVES waves.
 * The filter costs 5/256 VALU instructions per candidate, against 27/64 at
 * 45 % lane use for the walk along the sorted windows that it replaced.
 * Time with that walk and now (HIP events around the kernel and the fold of
 * split owners, perturbed lattices), us: mixture 1,048,576 atoms 4695, 3830;
 * 99,991 atoms 929, 445; 4,000 atoms 618, 116; argon 1,048,576 atoms 1290,
 * 770; 32,000 atoms 190, 56; 4,000 atoms 82, 34; water 64,000 atoms 555, 337.
 * Also measured, mixture 1,048,576, before the headers lay in LDS: both sides
 * dealt evenly (3350 us, but the energies' FP32 sums then run in another
 * order, up to 2e-6 of the total off where it cancels); the j hits levelling
 * the i lanes in one loop 5180; chunks of 192 slots 4570 (12 waves per CU
 * instead of 16); 3 waves per SIMD 4950; two lanes fetching each 32-byte row
 * together: within 4 %.
 */
#ifndef PAIR_TILE_H
#define PAIR_TILE_H

#define PT_TC 128    /* slots per chunk, a multiple of 64 */
#define PT_FSLOT 64  /* j side: sums of owner atoms in pair_lds::F, after those of the 64 runs */
#define PT_NPP 16    /* i side: pieces (16 slots of one entry at most) dealt at a time */
#define PT_LS 18     /* i side: half words of a lane's list; 9 words, so that lanes differ in bank */
#define PT_WAVES 4   /* items per block: they share the LDS copy of the tables */
#define PT_TAB 8192  /* bytes of LDS for table headers and coefficients */
#define PT_FAR 1.8e19f /* coordinates of a slot without an atom: its r^2 is infinite, whatever the
                          length unit, so it passes neither the filter nor the cutoff */

typedef float pt_f4 __attribute__((ext_vector_type(4)));

struct pt_d3 {
    double x, y, z;
};

template <int V>
struct pt_int {
    static constexpr int value = V;
};

template <int R>
struct pair_lds {
    float4 S[PT_TC];          /* x, y, z in the owner's frame; type | entry << 10 | key << 16    */
    float4 own[R];            /* x, y, z, byte offset of the type's table-header row             */
    int2 E[64];               /* per entry: first slot | sid << 17 | count << 21, cell offset    */
    int W[64];                /* per entry: dmaxdist - dnshift                                   */
    unsigned short okey[13 * R];
    union {
        float Q[PT_TC]; /* |x|^2 for the filter                                                  */
        struct {        /* i side */
            unsigned short lst[64 * PT_LS];   /* per lane: its hits in each piece                */
            unsigned int piece[PT_TC / 4];    /* first slot | length << 8 | first record << 13 | entry << 24 */
            unsigned short slot[PT_TC / 4];   /* 16 x first slot                                 */
        };
        struct {        /* j side */
            pt_d3 F[64 + R];        /* sums: of a run for the atom that an earlier run began,
                                       [64 ..] of the run that began each owner atom             */
            int P[R + 1];           /* hits before each owner atom                               */
            unsigned int start[64]; /* per lane: first list entry | bits to skip << 16           */
        };
    };
    uint2 wl[R * PT_TC / 32]; /* bitmap words, then the compacted (word, slot | atom) list       */
};

/* Inclusive sum over the wave by DPP: shifts within the rows of 16 lanes,
   then the rows' last lanes broadcast on (row_bcast:15, row_bcast:31). */
__device__ __forceinline__ unsigned int wave_incl_scan_u32(unsigned int v) {
    v += (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);
    v += (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);
    v += (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);
    v += (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);
    v += (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);
    v += (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);
    return v;
}

/* Table lookup of one pair in two steps, so that the coefficients' load can
   be in flight while another pair is worked on: pot_eval32's arithmetic. */
struct pair_eval {
    float dx, dy, dz, ir, r2;    /* the pair */
    float4 a, b;                 /* its interval's coefficients */
    bool use, inref, odd;        /* evaluated; inside the reference window; see `parity` */
};

/* r - c with r = r2 ir rounded first (every other hit, see `parity`). */
__device__ __forceinline__ float pt_offset(float r2, float ir, float c) {
#pragma clang fp contract(off)
    const float r = r2 * ir;
    return r - c;
}

/* TABS: 1, 2: the table headers (and 2: the coefficients) are in LDS at tab.
   PROJ: the projected window (every pair within the cutoff); the pass also
   counts the pairs that the reference window admits. */
template <int R, int TABS, bool PROJ>
__device__ __forceinline__ void pair_body(pair_lds<R> &L, const char *tab, const struct nb_params &P,
                                          const int2 *__restrict__ cnt_off,
                                          const int4 *__restrict__ nbr, const int *__restrict__ nbr_off,
                                          const int *__restrict__ nbr_mid, const float4 *__restrict__ nbs,
                                          const double *__restrict__ origin,
                                          const int *__restrict__ loc, const float4 *__restrict__ xf,
                                          const double *__restrict__ x64, const int *__restrict__ pid,
                                          const unsigned short *__restrict__ kminmax,
                                          const unsigned int *__restrict__ sortlist,
                                          const unsigned short *__restrict__ keyof, const float4 *__restrict__ ptab,
                                          const float4 *__restrict__ coeffs4, const int *__restrict__ excl_off,
                                          const int *__restrict__ excl_list, const int *__restrict__ index_of_id,
                                          const int *__restrict__ cell_of, const struct nb_out &O) {
    typedef pair_lds<R> pair_lds_t;
    constexpr int NIT = R / 16, KW = (R * PT_TC / 32 + 63) / 64;
    const int lane = threadIdx.x & 63, ln = lane & 15, g = lane >> 4;
    const int mt = P.max_type;
    unsigned int *const raw = (unsigned int *)L.wl;
    unsigned short *const lst = L.lst + lane * PT_LS;
    /* the filter's row operand: component g of slot t, |x|^2 for g = 3 */
    const int aoff = (int)(g == 3 ? offsetof(pair_lds_t, Q) : offsetof(pair_lds_t, S) + 4 * g), astep = g == 3 ? 4 : 16;
    /* as in nonbond_body: a pair with r2 - rc2f <= band is kept, and FP64
       decides those within the band */
    float rc2hi = P.rc2f + P.band;
    if (rc2hi - P.rc2f > P.band) rc2hi = __uint_as_float(__float_as_uint(rc2hi) - 1u);
    const __amdgpu_buffer_rsrc_t rs_ptab = make_rsrc(ptab, P.ptab_bytes);
    const __amdgpu_buffer_rsrc_t rs_coef = make_rsrc(coeffs4, P.coef_bytes);

    /* One item per wave: (owner cell, neighbour group).  Blocks go to the 8
       compute dies in turn, so block b takes the (b / 8)-th block of die
       b % 8's contiguous share of the work order. */
    const int nitems = P.ncells * P.nsplit;
    const int item = __builtin_amdgcn_readfirstlane(
        (((int)blockIdx.x % MD_NQUEUE) * ((int)gridDim.x / MD_NQUEUE) + (int)blockIdx.x / MD_NQUEUE) * PT_WAVES +
        (int)(threadIdx.x >> 6));
    if (item >= nitems) return;
    const int ci = item / P.nsplit, grp = item - ci * P.nsplit;
    const int c = P.order[ci];
    const int2 co_c = cnt_off[c];
    const int nc = co_c.x, offc = co_c.y;
    double epot = 0.0, vir = 0.0, eexcl = 0.0;
    unsigned int np = 0, nref = 0, nexcl = 0;
    const double oc0 = origin[3 * c], oc1 = origin[3 * c + 1], oc2 = origin[3 * c + 2];
    /* the owner's i entries from kc, its j entries from km; on the j side the
       self task, the first of the i side, comes once more before them */
    const int kc = nbr_off[c], km = nbr_mid[c], kn = nbr_off[c + 1];
    const int kself = km > kc && (nbr[kc].y & 32) ? km - 1 : km;
    const int nchunk = (nc + R - 1) / R;
    for (int ch = 0; ch < nchunk; ch++) {
        const int i0 = (int)(((long long)ch * nc) / nchunk);
        const int nsub = (int)(((long long)(ch + 1) * nc) / nchunk) - i0;
        const int nit = (nsub + 15) >> 4;
        const int a = offc + i0 + (lane < nsub ? lane : 0);
        const float4 xo = xf[a];
        const int to = __float_as_int(xo.w);

        /* The lane's atom and partition on the i side.  The cell's atoms go
           64 at a time over the 64 lanes (whatever R is): of n atoms, the
           i-th has the lanes i, i + n, ..., NPi of them. */
        const int il = lane % nsub, part = lane / nsub;
        int NP;
        {
            const int n64 = (nc + 63) / 64;
            int c64 = (int)(((long long)(i0 + il) * n64) / nc);
            /* the group of 64 that holds the atom */
            if (c64 + 1 < n64 && (int)(((long long)(c64 + 1) * nc) / n64) <= i0 + il) c64++;
            const int b64 = (int)(((long long)c64 * nc) / n64);
            const int s64 = (int)(((long long)(c64 + 1) * nc) / n64) - b64;
            NP = (63 - (i0 + il - b64)) / s64 + 1;
        }
        const bool ilane = part < NP;
        const float rNP = __builtin_amdgcn_rcpf((float)NP);
        /* bits b of the lane's records: b mod NP == part, b < 64 */
        unsigned long long recs = 0ull;
        if (ilane)
            for (int b = part; b < 64; b += NP) recs |= 1ull << b;

        /* Owner atoms: records, keys.  The last tile's empty columns hold any
           atoms: nothing reads their bits. */
        wave_lds_sync();
        if (lane < R) {
            const bool in = lane < nsub;
            L.own[lane] = make_float4(xo.x, xo.y, xo.z, __int_as_float(16 * mt * to));
            if (P.window && in)
                for (int sid = 0; sid < 13; sid++) L.okey[sid * R + lane] = keyof[(size_t)sid * P.nparts + a];
        }
        wave_lds_sync();
        /* filter operands: lane (ln, g) carries component g of owner
           atom 16 it + ln */
        float bop[NIT], cop[NIT];
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const float4 o = L.own[16 * it + ln];
            bop[it] = g == 0 ? -2.0f * o.x : g == 1 ? -2.0f * o.y : g == 2 ? -2.0f * o.z : 1.0f;
            cop[it] = (o.x * o.x + o.y * o.y + o.z * o.z) - P.filt;
        }
        double hx = 0.0, hy = 0.0, hz = 0.0; /* force on the lane's atom */

        /* The i side's entries, then the j side's: of each list this group's
           are every nsplit-th, so that the groups share near and far ones. */
        for (int side = 0; side < 2; side++) {
        const int kbeg = side == 0 ? kc : kself, kend = side == 0 ? km : kn;
        for (int k0 = kbeg + grp; k0 < kend; k0 += 64 * P.nsplit) {
            /* Entry headers, one per lane: the cell's slots in the
               concatenated list, its window constants, and whether the
               reference's unsigned break skips the task. */
            int len = 0, esid = 0, eoff = 0, ecnt = 0, ewin = 0, wcst = 0, eself = 0;
            const int kl = k0 + lane * P.nsplit;
            if (kl < kend) {
                const int4 en = nbr[side && kl < km ? kc : kl];
                const int2 co = cnt_off[en.x];
                eself = (en.y >> 5) & 1;
                esid = en.y & 15;
                eoff = co.y;
                ecnt = min(co.x, MD_MAX_CELL); /* more fit no field; their pass is not used */
                ewin = (en.y >> 8) & 1;
                bool live = ecnt > 0;
                if (!eself && ecnt > 0) {
                    const int ko = kminmax[26 * (size_t)c + (side ? 13 : 0) + esid];
                    const int kb = kminmax[26 * (size_t)en.x + (side ? 0 : 13) + esid];
                    const int s_imax = side ? kb : ko, s_jmin = side ? ko : kb;
                    const bool alive = s_jmin + en.z - s_imax >= 0;
                    const int dmd = P.maxdx != nullptr ? pair_dmaxdist(P.dscale, P.cutoff, P.maxdx[side ? en.x : c],
                                                                      P.maxdx[side ? c : en.x])
                                                       : P.dmaxdist;
                    wcst = dmd - en.z;
                    if (!alive) {
                        /* the projected window evaluates it all the same */
                        if (!PROJ) live = false;
                        wcst = -(1 << 24);
                        ewin = 1;
                    }
                }
                if (!ewin) wcst = 1 << 24;
                len = live ? (ecnt + 3) & ~3 : 0;
                if (!live) eoff = 0; /* an empty last cell's is past the atoms */
            }
            const int pin = (int)wave_incl_scan_u32((unsigned int)len), pex = pin - len;
            const int total = __builtin_amdgcn_readlane(pin, 63);
            if (total == 0) continue;
            wave_lds_sync();
            L.E[lane] = make_int2((int)((unsigned int)pex | ((unsigned int)esid << 17) | ((unsigned int)ecnt << 21)), eoff);
            L.W[lane] = wcst;
            /* the self task's entry, if any, and its first slot */
            const unsigned long long selfm = __builtin_amdgcn_ballot_w64(eself && len > 0);
            const int eslf = selfm ? (int)__builtin_ctzll(selfm) : -1;
            const int tself = selfm ? __builtin_amdgcn_readlane(pex, eslf) : 1 << 28;
            wave_lds_sync();

            /* i side: sums of one entry in window order; whether the lane has
               had a hit in the entry of the last piece */
            float le = 0.f, lv = 0.f;
            bool seen = false;
            /* PROJ: in every other hit of a lane's walk_cap records r is
               rounded before the interval's centre is subtracted.  It makes
               no energy more exact; without it the projected window's totals,
               FP64 outputs, would differ by 1e-9 to 3e-9 of themselves from
               those that this library has always given (a kernel that is gone
               evaluated hits two at a time, walk_cap records a round).  The
               rule depends on the number of cells alone. */
            bool parity = false;
            int rnd = 0;
            const float rnd_inv = __builtin_amdgcn_rcpf((float)(P.walk_cap * NP)) * 1.0001f;
            /* chunks of equal size, a multiple of 4 slots */
            const int nck = (total + PT_TC - 1) / PT_TC;
            const int tck = ((total + nck - 1) / nck + 3) & ~3;
            for (int base = 0; base < total; base += tck) {
                const int tn = min(tck, total - base);
                const int nblk = (tn + 63) >> 6; /* blocks of 64 slots: 2 words per owner atom each */
                const int nwi = 2 * nblk;
                const bool win = wave_any(ewin && pin > base && pex < base + tn);
                /* entry of the slots base + 4 lane .. + 3: the number of
                   entries that end at or before them */
                int eg = 0;
                for (int s = 32; s > 0; s >>= 1) {
                    const int v = __shfl(pin, eg + s - 1);
                    if (v <= base + 4 * lane) eg += s;
                }
                eg = eg > 63 ? 63 : eg;
                /* stage: the blocks' loads together, slots without an atom
                   load some atom's */
                {
                    constexpr int NB = PT_TC / 64;
                    int2 E[NB];
                    int e[NB], u[NB];
                    unsigned int key[NB];
                    bool in[NB];
#pragma unroll
                    for (int s = 0; s < NB; s++) {
                        const int t = 64 * s + lane;
                        e[s] = __shfl(eg, t >> 2);
                        E[s] = L.E[e[s]];
                        const int n = (int)((unsigned int)E[s].x >> 21), sid = (E[s].x >> 17) & 15;
                        u[s] = base + t - (E[s].x & 0x1ffff);
                        in[s] = t < tn && u[s] < n;
                        u[s] = in[s] ? u[s] : 0;
                        key[s] = 0u;
                        if (side) {
                            if (win) key[s] = keyof[(size_t)sid * P.nparts + E[s].y + u[s]];
                        } else {
                            /* ascending keys: the list is descending */
                            const bool sorted = in[s] && e[s] != eslf;
                            const unsigned int w = sortlist[13 * (size_t)E[s].y + (sorted ? sid * n + (n - 1 - u[s]) : 0)];
                            if (sorted) {
                                u[s] = min((int)(w >> 16), n - 1);
                                key[s] = w & 0xffffu;
                            }
                        }
                    }
                    float4 x[NB], sh[NB];
#pragma unroll
                    for (int s = 0; s < NB; s++) {
                        const int k = k0 + e[s] * P.nsplit;
                        x[s] = xf[E[s].y + u[s]];
                        sh[s] = nbs[in[s] && !(side && k < km) ? k : kc]; /* the self task's is the first */
                    }
#pragma unroll
                    for (int s = 0; s < NB; s++) {
                        const int t = 64 * s + lane;
                        float4 p = make_float4(PT_FAR, PT_FAR, PT_FAR, 0.f);
                        if (in[s]) {
                            p.x = x[s].x + sh[s].x;
                            p.y = x[s].y + sh[s].y;
                            p.z = x[s].z + sh[s].z;
                            p.w = __uint_as_float((unsigned int)__float_as_int(x[s].w) |
                                                  ((unsigned int)e[s] << 10) | (key[s] << 16));
                        }
                        L.S[t] = p;
                        L.Q[t] = p.x * p.x + p.y * p.y + p.z * p.z;
                    }
                }
                wave_lds_sync();
                /* filter: row m of tile qt is slot 64 blk + 16 (m / 4)
                   + 4 qt + m % 4, so that the lane's four values of the
                   block's four tiles are 16 consecutive bits of its
                   atom's bitmap */
                auto filter = [&](auto tiles) {
                    /* straight-line per block: a branch between an MFMA and
                       the reads of its result has lost its wait states */
                    constexpr int N = decltype(tiles)::value;
                    for (int blk = 0; blk < nblk; blk++) {
                        unsigned int word[N];
                        const int tb = 64 * blk + 16 * (ln >> 2) + (ln & 3);
#pragma unroll
                        for (int qt = 3; qt >= 0; qt--) {
                            const int t = tb + 4 * qt;
                            const float aop = *(const float *)((const char *)&L + aoff + t * astep);
                            pt_f4 d[N];
#pragma unroll
                            for (int it = 0; it < N; it++) {
                                d[it] = (pt_f4){cop[it], cop[it], cop[it], cop[it]};
                                d[it] = __builtin_amdgcn_mfma_f32_16x16x4f32(aop, bop[it], d[it], 0, 0, 0);
                            }
#pragma unroll
                            for (int it = 0; it < N; it++)
#pragma unroll
                                for (int r = 3; r >= 0; r--)
                                    word[it] = qt == 3 && r == 3
                                                   ? __float_as_uint(d[it][r]) >> 31
                                                   : __builtin_amdgcn_alignbit(word[it], __float_as_uint(d[it][r]), 31);
                        }
#pragma unroll
                        for (int it = 0; it < N; it++)
                            ((unsigned short *)raw)[(16 * it + ln) * 2 * nwi + 4 * blk + g] = (unsigned short)word[it];
                    }
                };
                if constexpr (R == 32) {
                    if (nit == 1)
                        filter(pt_int<1>{});
                    else
                        filter(pt_int<2>{});
                } else {
                    if (nit <= 2)
                        filter(pt_int<2>{});
                    else if (nit == 3)
                        filter(pt_int<3>{});
                    else
                        filter(pt_int<4>{});
                }
                wave_lds_sync();
                pair_eval va, vb;
                double fx = 0.0, fy = 0.0, fz = 0.0; /* j side: of the run */
                unsigned int cur = 0u; /* hits left in the lane's word */
                int tb = 0;            /* 16 x its first slot */
                int tt = 0;            /* i side: its first record in the entry */
                /* the pair of hit s of `mine`, owner atom (xi, io):
                   geometry, window and cutoff tests, its coefficients
                   requested */
                auto fetch = [&](bool have, const float4 &xi, int io, pair_eval &v) {
                    const int bit = __builtin_ctz(cur | 0x80000000u); /* no bit left: any slot */
                    cur &= cur - 1u;
                    const float4 pj = *(const float4 *)((const char *)L.S + tb + 16 * bit);
                    const unsigned int w = __float_as_uint(pj.w);
                    /* a lane without a hit loads nothing (past the end): half
                       the lanes on the i side, and the L1 serves a lane a
                       clock */
                    const int ho = __float_as_int(xi.w) + 16 * (int)__builtin_amdgcn_ubfe(w, 0, 10);
                    const float4 hd = TABS ? *(const float4 *)(tab + (have ? ho : 0)) : ld_f4(rs_ptab, have ? ho : -16);
                    v.dx = xi.x - pj.x;
                    v.dy = xi.y - pj.y;
                    v.dz = xi.z - pj.z;
                    v.r2 = v.dx * v.dx + v.dy * v.dy + v.dz * v.dz;
                    v.use = have && v.r2 <= rc2hi;
                    v.odd = false;
                    if (PROJ && !side) {
                        const int b = have ? (int)((float)(tt + bit) * rnd_inv) : rnd;
                        if (b != rnd) parity = false;
                        rnd = b;
                        v.odd = parity;
                        parity = parity != v.use;
                    }
                    v.use = v.use && __float_as_int(hd.w) != -1;
                    v.inref = true;
                    if (win) {
                        const int e = (int)__builtin_amdgcn_ubfe(w, 10, 6);
                        const int ok = L.okey[((L.E[e].x >> 17) & 15) * R + io], kj = (int)(w >> 16);
                        /* key_j + dnshift - key_i < dmaxdist, i and j in task order */
                        v.inref = (side ? kj - ok : ok - kj) + L.W[e] > 0;
                        if (!PROJ) v.use = v.use && v.inref;
                    }
                    if (v.use && fabsf(v.r2 - P.rc2f) <= P.band) {
                        /* the reference's FP64 cutoff test, in the task's
                           orientation */
                        const int e = (int)__builtin_amdgcn_ubfe(w, 10, 6), ks = k0 + e * P.nsplit;
                        const int2 E = L.E[e];
                        const int n = (int)((unsigned int)E.x >> 21), u = base + (tb >> 4) + bit - (E.x & 0x1ffff);
                        int idx = u;
                        if (!side && e != eslf)
                            idx = min((int)(sortlist[13 * (size_t)E.y + (size_t)((E.x >> 17) & 15) * n + (n - 1 - u)] >> 16),
                                      n - 1);
                        const double *xa = &x64[3 * (size_t)(offc + i0 + io)];
                        const double *xb = &x64[3 * (size_t)(E.y + idx)];
                        const double *on = &origin[3 * nbr[side && ks < km ? kc : ks].x];
                        double sh[3];
                        for (int m = 0; m < 3; m++)
                            sh[m] = side ? min_image(origin[3 * c + m] - on[m], P.dim[m])
                                         : min_image(on[m] - origin[3 * c + m], P.dim[m]);
                        v.use = r2_task64(side ? xb : xa, side ? xa : xb, sh[0], sh[1], sh[2]) <=
                                P.cutoff2;
                    }
                    v.ir = __builtin_amdgcn_rsqf(v.r2);
                    const float r = v.r2 * v.ir;
                    const unsigned int hw = __float_as_uint(hd.w);
                    const int n = (int)(hw & 511u);
                    int ind = (int)fmaxf(0.0f, hd.x + r * (hd.y + r * hd.z));
                    ind = ind > n ? n : ind;
                    const unsigned int off = 32u * ((hw >> 9) + (unsigned int)ind);
                    if (TABS == 2) {
                        const float4 *c = (const float4 *)(tab + P.ptab_bytes + (v.use ? off : 0u));
                        v.a = c[0];
                        v.b = c[1];
                    } else {
                        v.a = ld_f4(rs_coef, v.use ? (int)off : -32);
                        v.b = ld_f4(rs_coef, v.use ? (int)off + 16 : -16);
                    }
                };
                /* its polynomial, force and sums */
                auto apply = [&](auto iside, const pair_eval &v) {
                    if (v.use) {
                        float x = fmaf(v.r2, v.ir, -v.a.x);
                        if constexpr (PROJ && decltype(iside)::value == 1)
                            if (v.odd) x = pt_offset(v.r2, v.ir, v.a.x);
                        x *= v.a.y;
                        float ee = v.a.z * x + v.a.w;
                        float eff = v.a.z;
                        eff = eff * x + ee;
                        ee = ee * x + v.b.x;
                        eff = eff * x + ee;
                        ee = ee * x + v.b.y;
                        eff = eff * x + ee;
                        ee = ee * x + v.b.z;
                        eff = eff * x + ee;
                        const float f = eff * v.a.y * v.ir;
                        const double fd = (double)-f;
                        double &gx = decltype(iside)::value ? hx : fx, &gy = decltype(iside)::value ? hy : fy,
                               &gz = decltype(iside)::value ? hz : fz;
                        gx = __builtin_fma(fd, (double)v.dx, gx);
                        gy = __builtin_fma(fd, (double)v.dy, gy);
                        gz = __builtin_fma(fd, (double)v.dz, gz);
                        if constexpr (decltype(iside)::value == 1) {
                            ee = ee * x + v.b.w;
                            le += ee;
                            lv = fmaf(-f, v.r2, lv);
                            np++;
                            if (PROJ && v.inref) nref++;
                        }
                    }
                };
                if (side == 0) {
                    /* the chunk's pieces */
                    int npc;
                    {
                        const int lo = max(pex, base), hi = min(pex + ecnt, base + tn);
                        const int pl = len > 0 && hi > lo ? hi - lo : 0, n = (pl + 15) >> 4;
                        const int inc = (int)wave_incl_scan_u32((unsigned int)n);
                        npc = __builtin_amdgcn_readlane(inc, 63);
                        for (int k = 0; k < n; k++) {
                            L.piece[inc - n + k] = (unsigned int)(lo - base + 16 * k) |
                                                   ((unsigned int)min(16, pl - 16 * k) << 8) |
                                                   ((unsigned int)(lo - pex + 16 * k) << 13) |
                                                   ((unsigned int)lane << 24);
                            L.slot[inc - n + k] = (unsigned short)(16 * (lo - base + 16 * k));
                        }
                    }
                    wave_lds_sync();
                    const float4 xi = L.own[il];
                    const int npass = (npc + PT_NPP - 1) / PT_NPP, per = (npc + npass - 1) / max(npass, 1);
                    for (int q0 = 0; q0 < npc; q0 += per) {
                        const int nq = min(per, npc - q0);
                        /* the lane's hits in each piece; pieces with any, and
                           those of them that begin an entry's sum */
                        int ni = 0;
                        unsigned int pmask = 0u, first = 0u;
                        for (int q = 0; q < nq; q++) {
                            const unsigned int pd = (unsigned int)__builtin_amdgcn_readfirstlane((int)L.piece[q0 + q]);
                            const int s = (int)(pd & 255u), n = (int)((pd >> 8) & 31u), t0 = (int)((pd >> 13) & 0x7ffu);
                            const int e = (int)(pd >> 24), k = s >> 5;
                            const unsigned int *rw = raw + il * nwi + k;
                            const unsigned int w0 = rw[0], w1 = rw[k + 1 < nwi ? 1 : 0];
                            unsigned int m = __builtin_amdgcn_alignbit(w1, w0, s & 31) & ((1u << n) - 1u);
                            if (t0 <= 48)
                                m &= (unsigned int)(recs >> t0);
                            else {
                                /* (t0 - part) mod NP by a float quotient within one */
                                int r = t0 - part - (int)((float)(t0 - part) * rNP) * NP;
                                r = r < 0 ? r + NP : r >= NP ? r - NP : r;
                                m &= r == 0 ? (unsigned int)(recs >> part) : r > NP - 16 ? (unsigned int)(recs >> part) << (NP - r) : 0u;
                            }
                            if (e == eslf) {
                                /* partners before the atom: those after it
                                   are on the j side */
                                const int o = i0 + il - t0;
                                m &= o <= 0 ? 0u : o < 16 ? (1u << o) - 1u : 0xffffu;
                            }
                            lst[q] = (unsigned short)m;
                            if (t0 == 0) seen = false;
                            if (m) {
                                pmask |= 1u << q;
                                first |= seen ? 0u : 1u << q;
                                seen = true;
                            }
                            ni += __builtin_popcount(m);
                        }
                        int nr = ni; /* rounds: the longest lane's hits */
                        for (int o = 32; o > 0; o >>= 1) nr = max(nr, __shfl_xor(nr, o));
                        nr = __builtin_amdgcn_readfirstlane(nr);
                        /* the lane's next piece with hits; the pending pair
                           still belongs to the old one's sums */
                        auto advance = [&](int s) -> bool {
                            if (!(s < ni && cur == 0u)) return false;
                            const int q = __builtin_ctz(pmask);
                            pmask &= pmask - 1u;
                            cur = lst[q];
                            tb = L.slot[q0 + q];
                            const bool begins = (first >> q) & 1u;
                            if (PROJ) {
                                const unsigned int pd = L.piece[q0 + q];
                                tt = (int)((pd >> 13) & 0x7ffu);
                                if (begins) parity = false;
                            }
                            return begins;
                        };
                        auto flush = [&](bool yes) {
                            if (yes) {
                                epot += (double)le;
                                vir += (double)lv;
                                le = lv = 0.f;
                            }
                        };
                        auto step = [&](int s, const pair_eval &pend, pair_eval &next) {
                            const bool fl = advance(s);
                            fetch(s < ni, xi, il, next);
                            apply(pt_int<1>{}, pend);
                            flush(fl);
                        };
                        if (nr > 0) {
                            /* two hits per round, without a branch between a
                               request and the use of the one before (their
                               loads would be waited for together there) */
                            flush(advance(0));
                            fetch(0 < ni, xi, il, va);
                            int s = 1;
                            for (; s + 1 < nr; s += 2) {
                                step(s, va, vb);
                                step(s + 1, vb, va);
                            }
                            if (s < nr) {
                                step(s, va, vb);
                                apply(pt_int<1>{}, vb);
                            } else
                                apply(pt_int<1>{}, va);
                        }
                    }
                    wave_lds_sync();
                    continue;
                }
                /* j side */
                if (tself < base + tn && tself + nc > base) {
                    /* of the self task's slots keep those after the atom's own */
                    const int t0 = tself - base, t1 = t0 + i0 + lane + 1;
                    if (lane < nsub)
                        for (int k = max(t0, 0) >> 5; k < nwi && 32 * k < t1; k++) {
                            const int lo = min(max(t0 - 32 * k, 0), 32), hi = min(t1 - 32 * k, 32);
                            const unsigned int m = (hi < 32 ? (1u << hi) - 1u : ~0u) & (lo < 32 ? ~0u << lo : 0u);
                            raw[lane * nwi + k] &= ~m;
                        }
                    wave_lds_sync();
                }
                /* deal the H set bits in runs of Q */
                const int nw = nsub * nwi, kw = (nw + 63) >> 6;
                unsigned int wv[KW];
                unsigned int sum = 0u; /* bits | non-empty words << 16 */
#pragma unroll
                for (int j = 0; j < KW; j++) {
                    wv[j] = 0u;
                    if (j < kw && lane * kw + j < nw) wv[j] = raw[lane * kw + j];
                    sum += (unsigned int)__builtin_popcount(wv[j]) + (wv[j] ? 65536u : 0u);
                }
                const unsigned int inc = wave_incl_scan_u32(sum);
                const int H = __builtin_amdgcn_readlane((int)inc, 63) & 0xffff;
                const int Q = (H + 63) >> 6;
                const float rq = __builtin_amdgcn_rcpf((float)(Q > 0 ? Q : 1));
                wave_lds_sync();
                {
                    int hp = (int)((inc - sum) & 0xffffu), zp = (int)((inc - sum) >> 16);
                    /* first run that starts at or after hp */
                    int Ln = (int)((float)(hp + Q - 1) * rq);
                    if (Ln * Q < hp) Ln++;
                    if (Ln > 0 && (Ln - 1) * Q >= hp) Ln--;
                    /* atom and word of the lane's first word */
                    int i = lane * kw / nwi, k = lane * kw - i * nwi;
#pragma unroll
                    for (int j = 0; j < KW; j++) {
                        if (j < kw && i < nsub) {
                            if (k == 0) L.P[i] = hp;
                            if (wv[j]) {
                                const int nb = __builtin_popcount(wv[j]);
                                L.wl[zp] = make_uint2(wv[j], ((unsigned int)k << 9) | ((unsigned int)i << 20));
                                while (Ln * Q < hp + nb) {
                                    L.start[Ln] = (unsigned int)zp | ((unsigned int)(Ln * Q - hp) << 16);
                                    Ln++;
                                }
                                hp += nb;
                                zp++;
                            }
                            if (++k == nwi) {
                                k = 0;
                                i++;
                            }
                        }
                    }
                    if (lane == 0) L.P[nsub] = H;
                }
                wave_lds_sync();
                /* eval: lane's run is hits [lane Q, lane Q + mine) */
                const int mine = min(Q, H - lane * Q); /* may be <= 0 */
                const unsigned int st = mine > 0 ? L.start[lane] : 0u;
                int p = (int)(st & 0xffffu);
                uint2 wd = mine > 0 ? L.wl[p] : make_uint2(0u, 0u);
                cur = wd.x;
                {
                    /* drop the first (st >> 16) set bits */
                    int skip = (int)(st >> 16), pos = 0;
#pragma unroll
                    for (int s = 16; s > 0; s >>= 1) {
                        const int nb = __builtin_popcount((cur >> pos) & ((1u << s) - 1u));
                        if (nb <= skip) {
                            skip -= nb;
                            pos += s;
                        }
                    }
                    cur = (cur >> pos) << pos;
                }
                tb = (int)(wd.y & 0xfffffu);
                int io = (int)(wd.y >> 20);
                float4 xi = L.own[io];
                /* where the atom's sum goes: its own slot, or the run's
                   when an earlier run began the atom */
                int fd = lane * Q > L.P[io] ? lane : PT_FSLOT + io;
                wave_lds_sync();
                /* request hit s while the pending pair, hit s - 1, is applied */
                auto step = [&](int s, const pair_eval &pend, pair_eval &next) {
                    /* the next hit's word, and its atom if that changes: the
                       pending pair still belongs to the old one */
                    bool turn = false;
                    if (s < mine && cur == 0u) {
                        wd = L.wl[++p];
                        cur = wd.x;
                        tb = (int)(wd.y & 0xfffffu);
                        const int ion = (int)(wd.y >> 20);
                        turn = ion != io;
                        if (turn) {
                            io = ion;
                            xi = L.own[io];
                        }
                    }
                    fetch(s < mine, xi, io, next);
                    apply(pt_int<0>{}, pend);
                    if (turn) {
                        L.F[fd] = {fx, fy, fz};
                        fx = fy = fz = 0.0;
                        fd = PT_FSLOT + io;
                    }
                };
                if (Q > 0) {
                    /* two hits per round, without a branch between a
                       request and the use of the one before (their loads
                       would be waited for together there) */
                    fetch(0 < mine, xi, io, va);
                    int s = 1;
                    for (; s + 1 < Q; s += 2) {
                        step(s, va, vb);
                        step(s + 1, vb, va);
                    }
                    if (s < Q) {
                        step(s, va, vb);
                        apply(pt_int<0>{}, vb);
                    } else
                        apply(pt_int<0>{}, va);
                }
                if (mine > 0) L.F[fd] = {fx, fy, fz};
                wave_lds_sync();
                /* fold: the sum of the run that began the atom, then
                   those of the runs that went on with it */
                if (lane < nsub) {
                    const int p0 = L.P[lane], p1 = L.P[lane + 1];
                    if (p1 > p0) {
                        const pt_d3 f = L.F[PT_FSLOT + lane];
                        hx += f.x;
                        hy += f.y;
                        hz += f.z;
                        int la = (int)((float)p0 * rq), lb = (int)((float)(p1 - 1) * rq);
                        if (la * Q > p0) la--;
                        if ((la + 1) * Q <= p0) la++;
                        if (lb * Q > p1 - 1) lb--;
                        if ((lb + 1) * Q <= p1 - 1) lb++;
                        for (int l = la + 1; l <= lb; l++) {
                            const pt_d3 v = L.F[l];
                            hx += v.x;
                            hy += v.y;
                            hz += v.z;
                        }
                    }
                }
                wave_lds_sync();
            }
            epot += (double)le;
            vir += (double)lv;
        }
        }

        /* the partitions' sums, in order, into the atoms' */
        double px = 0.0, py = 0.0, pz = 0.0;
        for (int p = 1; p * nsub < 64; p++) {
            const int l = lane + p * nsub;
            const double ax = __shfl(hx, l & 63), ay = __shfl(hy, l & 63), az = __shfl(hz, l & 63);
            if (lane < nsub && l < 64) {
                px += ax;
                py += ay;
                pz += az;
            }
        }
        hx += px;
        hy += py;
        hz += pz;

        /* Excluded pairs: subtract what the pair pass added
           (exclusion.c:139-208), same FP32 arithmetic. */
        if (lane < nsub && grp == 0) {
            const int myid = pid[a];
            for (int k = excl_off[myid]; k < excl_off[myid + 1]; k++) {
                const int oid = excl_list[k];
                if (oid == myid) continue;
                const int b = index_of_id[oid];
                if (b < 0) continue;
                const int cb = cell_of[b];
                const float4 pj = xf[b];
                const float4 hdr = ptab[to * mt + __float_as_int(pj.w)];
                if (__float_as_int(hdr.w) == -1) continue;
                const float ex = (float)min_image(origin[3 * cb] - oc0, P.dim[0]);
                const float ey = (float)min_image(origin[3 * cb + 1] - oc1, P.dim[1]);
                const float ez = (float)min_image(origin[3 * cb + 2] - oc2, P.dim[2]);
                const float dx = (xo.x - pj.x) - ex, dy = (xo.y - pj.y) - ey, dz = (xo.z - pj.z) - ez;
                const float r2 = dx * dx + dy * dy + dz * dz;
                bool in = r2 <= P.rc2f;
                if (fabsf(r2 - P.rc2f) <= P.band) {
                    const bool mine = myid < oid;
                    const int ia = mine ? a : b, ib = mine ? b : a;
                    const int ca = mine ? c : cb, cbb = mine ? cb : c;
                    in = r2_excl64(&x64[3 * (size_t)ia], &x64[3 * (size_t)ib], &loc[3 * ca], &loc[3 * cbb], P.h) <=
                         P.cutoff2;
                }
                if (!in) continue;
                float e, ff;
                pot_eval32(hdr, coeffs4, r2, e, ff);
                hx = __builtin_fma((double)ff, (double)dx, hx);
                hy = __builtin_fma((double)ff, (double)dy, hy);
                hz = __builtin_fma((double)ff, (double)dz, hz);
                if (myid < oid) {
                    eexcl -= (double)e;
                    nexcl++;
                }
            }
        }
        if (lane < nsub) {
            const size_t o = P.nsplit == 1 ? (size_t)a : (size_t)grp * P.nparts + a;
            const float4 hi = make_float4((float)hx, (float)hy, (float)hz, 0.0f);
            (P.nsplit == 1 ? O.fhi : O.phi)[o] = hi;
            (P.nsplit == 1 ? O.flo : O.plo)[o] =
                make_float4((float)(hx - hi.x), (float)(hy - hi.y), (float)(hz - hi.z), 0.0f);
        }
    }
    /* per-item sums */
    epot = wave_sum(epot);
    vir = wave_sum(vir);
    eexcl = wave_sum(eexcl);
    np = (unsigned int)wave_sum((int)np);
    if (PROJ) nref = (unsigned int)wave_sum((int)nref);
    nexcl = (unsigned int)wave_sum((int)nexcl);
    if (lane == 0) {
        O.cell_acc[3 * item] = epot;
        O.cell_acc[3 * item + 1] = eexcl;
        O.cell_acc[3 * item + 2] = vir;
        O.cell_cnt[3 * item] = np;
        O.cell_cnt[3 * item + 1] = nexcl;
        O.cell_cnt[3 * item + 2] = PROJ ? nref : np;
    }
}

#endif /* PAIR_TILE_H */
