/*
 * mpic_tile_bodies.h -- bodies of the kernels between the push and the E
 * update that work on the sorted tiles: the J gather of the FP32 form, the
 * tile scan and the rank pass.  The loop body runs them in launches shared
 * with field kernels (mpic_fdtd.hip), the stage calls on their own
 * (mpic_tiles.hip, mpic_fdtd.hip).
 */
#ifndef MPIC_TILE_BODIES_H
#define MPIC_TILE_BODIES_H

#include "mpic_launch.h"
#include "mpic_tiles.h"

#define SCAN_TPB 256
#define SCAN_WT 64               /* tiles per wavefront of the scan */
#define SB (SCAN_TPB / 64 * SCAN_WT) /* tiles per scan workgroup */
#define JG_TPB 256

/* The tile scan, in one pass: every workgroup takes SB consecutive tiles,
 * sums their per-key counts, scans (markers, tile non-empty, work items)
 * over its tiles, and finds the sum of all earlier tiles by a decoupled
 * look-back (Merrill and Garland, "Single-pass parallel prefix scan with
 * decoupled look-back", NVIDIA technical report NVR-2016-002): it publishes
 * its own totals at once, then adds up its predecessors' published values
 * back to the first one that has published its inclusive prefix, and
 * publishes its own inclusive prefix.  A workgroup only waits for
 * workgroups of lower index, which the hardware has dispatched before it,
 * so every wait ends; the wait is bounded all the same (SCAN_SPIN polls,
 * then an error flag, and the kernel still exits).
 *
 * Published values are 64-bit words (tag << 32 | value), three for a
 * workgroup's totals and three for its inclusive prefix; the tag is the
 * scan's sequence number (+1), so words of earlier scans never match and
 * the words are never cleared.  The last workgroup advances the sequence
 * number after every workgroup has published (its inclusive prefix needs
 * all of them), i.e. after every workgroup has read it.
 *
 * Layout of the counts: a tile's 64 per-key counts are 16 int4; 16 lanes of
 * a wavefront read one tile (coalesced), a wavefront four tiles per load.
 * With LD = SCAN_WT / 4 all its loads are in flight together and stay in
 * registers for the per-key offsets written at the end (130 VGPRs); with
 * fewer, they are read in rounds of LD and again at the end, which costs
 * 1.5 us on a 32^3 box but leaves the launch the J gather's registers: shared
 * with the 130 of the former, the gather of laser-foil took 48 us, with LD = 8
 * 39 (34 and 13 for gather and scan in launches of their own). */
#define NSCAN 3
#define SCAN_SPIN (1 << 20)
struct ScanArgs {
    TileView            tv;
    unsigned long long *flags;        /* [nb][6] published words */
    int                *seq;          /* scan sequence number */
    unsigned           *err;          /* bit 1: a look-back wait ran out */
    int                 nb, parity_next;
};

__device__ static inline unsigned long long scan_word(unsigned tag, int v)
{
    return ((unsigned long long)tag << 32) | (unsigned)v;
}

/* Inclusive sums over a row of 16 lanes and over the wavefront by DPP moves
 * (a few cycles each; the same steps through shuffles go through the LDS
 * unit and took a third of the scan: 9.2 us on a 32^3 box, see below). */
__device__ static inline int row_sum(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);    /* row_shr:1 */
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);    /* row_shr:2 */
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);    /* row_shr:4 */
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);    /* row_shr:8 */
    return x;
}

__device__ static inline int wave_sum(int x)
{
    x = row_sum(x);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);   /* row_bcast:15 to rows 1, 3 */
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);   /* row_bcast:31 to rows 2, 3 */
    return x;
}

template <int LD>
__device__ static inline void scan_pass(const ScanArgs &A, const VBlock &bk)
{
    constexpr int NV = SCAN_WT / 4;                  /* loads of a wavefront */
    const TileView &tv = A.tv;
    __shared__ int wsum[NSCAN][SCAN_TPB / 64];
    __shared__ int spre[NSCAN];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, blk = (int)bk.x;
    const int wt0 = blk * SB + w * SCAN_WT;          /* first tile of the wavefront */
    const int4 *cnt4 = (const int4 *)tv.count;
    const int seq = *A.seq;                          /* with the counts' latency, not after it */
    int c = 0;                                       /* markers of tile wt0 + lane */
    int4 x[LD];
#pragma unroll 1
    for (int v0 = 0; v0 < NV; v0 += LD) {
#pragma unroll
        for (int v = 0; v < LD; ++v) {
            const int t = wt0 + (v0 + v) * 4 + (lane >> 4);
            x[v] = t < tv.ntiles ? cnt4[(long)t * 16 + (lane & 15)] : make_int4(0, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < LD; ++v) {
            const int inc = row_sum(x[v].x + x[v].y + x[v].z + x[v].w);
            const int tot = __shfl(inc, (lane & 3) * 16 + 15, 64);   /* tile 4 (v0 + v) + (lane & 3) */
            if ((lane >> 2) == v0 + v) c = tot;
        }
    }
    const int own[NSCAN] = {c, c > 0, tile_items(c, tv.chm)};
    int inc[NSCAN];
    for (int a = 0; a < NSCAN; ++a) {                /* wavefront inclusive scan */
        inc[a] = wave_sum(own[a]);
        if (lane == 63) wsum[a][w] = inc[a];
    }
    __syncthreads();
    int agg[NSCAN];
    for (int a = 0; a < NSCAN; ++a) {
        agg[a] = 0;
        for (int q = 0; q < SCAN_TPB / 64; ++q) {
            if (q < w) inc[a] += wsum[a][q];
            agg[a] += wsum[a][q];
        }
    }
    if (w == 0) {                                    /* the look-back, one wavefront */
        unsigned long long *F = A.flags;
        const unsigned tag = (unsigned)(seq % 0x7fffffff) + 1u;
        int pre[NSCAN] = {0, 0, 0};
        if (blk > 0) {
            if (lane < NSCAN)
                __hip_atomic_store(F + 6 * blk + lane, scan_word(tag, agg[lane]), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            int end = blk - 1;                       /* the window's nearest predecessor */
            unsigned polls = 0;
            for (;;) {
                const int j = end - lane;
                bool ready = true, incl = false;
                int v[NSCAN] = {0, 0, 0};
                if (j >= 0) {
                    unsigned long long q[NSCAN];
                    bool ok = true;
                    for (int a = 0; a < NSCAN; ++a) {
                        q[a] = __hip_atomic_load(F + 6 * j + 3 + a, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
                        ok = ok && (unsigned)(q[a] >> 32) == tag;
                    }
                    incl = ok;
                    if (!ok) {
                        ok = true;
                        for (int a = 0; a < NSCAN; ++a) {
                            q[a] = __hip_atomic_load(F + 6 * j + a, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
                            ok = ok && (unsigned)(q[a] >> 32) == tag;
                        }
                    }
                    ready = ok;
                    for (int a = 0; a < NSCAN; ++a) v[a] = (int)(unsigned)q[a];
                }
                /* lanes up to the nearest inclusive prefix (or all) are needed */
                const unsigned long long im = __ballot(incl), nr = __ballot(!ready);
                const int L = im ? __ffsll((long long)im) - 1 : 63;
                const unsigned long long need = L == 63 ? ~0ull : ((2ull << L) - 1ull);
                if (nr & need) {
                    if (++polls > SCAN_SPIN) {       /* never expected: give up, flagged */
                        if (lane == 0 && A.err) atomicOr(A.err, 2u);
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                    continue;
                }
                for (int a = 0; a < NSCAN; ++a) {
                    const int y = wave_sum((lane <= L && j >= 0) ? v[a] : 0);
                    pre[a] += __builtin_amdgcn_readlane(y, 63);
                }
                if (im) break;
                end -= 64;                           /* block 0 is always inclusive: end stays >= 0 */
            }
        }
        if (lane < NSCAN) {
            __hip_atomic_store(F + 6 * blk + 3 + lane, scan_word(tag, pre[lane] + agg[lane]),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            spre[lane] = pre[lane];
        }
        if (blk == A.nb - 1 && lane == 0) {          /* totals, then the next sequence number */
            const int tot = pre[0] + agg[0], na = pre[1] + agg[1], ni = pre[2] + agg[2];
            tv.off[tv.ncellp] = tot;
            tv.toff[tv.ntiles] = tot;
            tv.nactive[A.parity_next] = na;
            *tv.nitems = ni;
            tv.nmark[A.parity_next] = tot;
            *A.seq = seq + 1;
        }
    }
    __syncthreads();
    /* tile offsets, the active list, the work items */
    const int base = spre[0] + inc[0] - own[0];
    const int t = wt0 + lane;
    const long po = (long)A.parity_next * tv.ntiles;
    if (lane < SCAN_WT && t < tv.ntiles) {
        tv.toff[t] = base;
        const int is = spre[2] + inc[2] - own[2], nu = own[2];
        if (c > 0) {
            tv.active[po + spre[1] + inc[1] - own[1]] = t;
            /* item u of nu: an even share of the tile's markers */
            for (int u = 0; u < nu; ++u)
                tv.item[is + u] = make_int4(t, base + (int)((long)u * c / nu),
                                            base + (int)((long)(u + 1) * c / nu), 0);
        }
        tv.titem[po + t] = make_int2(is, nu);
    }
    /* per-key offsets and cursors of the non-empty tiles, counters reset
     * (entries of empty tiles are not maintained) */
    int4 *off4 = (int4 *)tv.off, *cur4 = (int4 *)tv.cursor, *cnt4w = (int4 *)tv.count;
#pragma unroll 1
    for (int v0 = 0; v0 < NV; v0 += LD) {
        int tb[LD];
        bool on[LD];
#pragma unroll
        for (int v = 0; v < LD; ++v) {
            const int tt = (v0 + v) * 4 + (lane >> 4);
            tb[v] = __shfl(base, tt, 64);
            on[v] = __shfl(c, tt, 64) > 0;
            if (LD < NV) x[v] = on[v] ? cnt4[(long)(wt0 + tt) * 16 + (lane & 15)] : make_int4(0, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < LD; ++v) {
            const int s = x[v].x + x[v].y + x[v].z + x[v].w, o0 = tb[v] + row_sum(s) - s;
            if (!on[v]) continue;
            const long q = (long)(wt0 + (v0 + v) * 4 + (lane >> 4)) * 16 + (lane & 15);
            const int4 o = make_int4(o0, o0 + x[v].x, o0 + x[v].x + x[v].y,
                                     o0 + x[v].x + x[v].y + x[v].z);
            off4[q] = o;
            cur4[q] = o;
            cnt4w[q] = make_int4(0, 0, 0, 0);
        }
    }
}

template <> struct KernelDef<ScanArgs> {
    static constexpr int kBlock = SCAN_TPB;
    __device__ __forceinline__ static void body(const ScanArgs &a, VBlock b, VBlock)
    {
        scan_pass<SCAN_WT / 4>(a, b);
    }
};

/* The scan in few registers, for a launch shared with the J gather. */
struct ScanLeanArgs : ScanArgs {
};

template <> struct KernelDef<ScanLeanArgs> {
    static constexpr int kBlock = SCAN_TPB;
    __device__ __forceinline__ static void body(const ScanLeanArgs &a, VBlock b, VBlock)
    {
        scan_pass<8>(a, b);
    }
};

static inline ScanArgs scan_args(const TileView &tv, unsigned long long *words, unsigned *err,
                                 int parity_next)
{
    const int nb = (tv.ntiles + SB - 1) / SB;
    ScanArgs a = {tv, words, (int *)(words + 6L * nb), err, nb, parity_next};
    return a;
}

/* The next order: every position p < nmark[parity] with a key (the push's
 * output, or the markers keyed by k_keys32 / k_keys64) takes slot
 * cursor[key]++ among its key's, one atomic per run of equal keys in a
 * wavefront, and perm[slot] = p.  4 B read and 4 B written per marker
 * instead of moving its records (36 B FP32, 60 B FP64).  A
 * workgroup ranks RANK_BATCHES consecutive batches of 256 positions with
 * all their loads, then all their atomics, in flight together: one
 * batch's chain of dependent accesses would leave the pass latency-bound. */
#define RANK_BATCHES 4
struct RankArgs {
    TileView tv;
    long     nbound;
    int      parity;
};

__device__ static inline void rank_pass(const TileView &tv, long nbound, int parity, long b0)
{
    const long n = tv.nmark[parity];
    int key[RANK_BATCHES], start[RANK_BATCHES], base[RANK_BATCHES];
#pragma unroll
    for (int u = 0; u < RANK_BATCHES; ++u) {
        const long p = b0 + 256 * u + threadIdx.x;
        key[u] = p < nbound ? tv.key[p] : -1;    /* not behind the load of n */
    }
#pragma unroll
    for (int u = 0; u < RANK_BATCHES; ++u) {
        int len;
        bool head;
        if (b0 + 256 * u + threadIdx.x >= n) key[u] = -1;
        wave_run(key[u], start[u], len, head);
        base[u] = 0;
        if (head && key[u] >= 0) base[u] = atomicAdd(tv.cursor + key[u], len);
    }
#pragma unroll
    for (int u = 0; u < RANK_BATCHES; ++u) {
        const int bs = __shfl(base[u], start[u], 64);
        if (key[u] >= 0)
            tv.perm[bs + ((int)(threadIdx.x & 63) - start[u])] = (int)(b0 + 256 * u + threadIdx.x);
    }
}

template <> struct KernelDef<RankArgs> {
    static constexpr int kBlock = 256;
    __device__ __forceinline__ static void body(const RankArgs &a, VBlock b, VBlock)
    {
        if (b.x == 0 && threadIdx.x == 0) {
            /* the active list is in tile order, tiles i-major */
            const int nx = a.parity ^ 1, na = a.tv.nactive[nx], tpp = a.tv.nt[1] * a.tv.nt[2];
            const int *act = a.tv.active + (long)nx * a.tv.ntiles;
            a.tv.xr[0] = na > 0 ? 4 * (act[0] / tpp) : 0;
            a.tv.xr[1] = na > 0 ? 4 * (act[na - 1] / tpp) + 5 : -1;
        }
        rank_pass(a.tv, a.nbound, a.parity, (long)b.x * (256 * RANK_BATCHES));
    }
};

/* Workgroups of the rank pass over at most n markers. */
static inline unsigned rank_blocks(long n)
{
    const long per = 256L * RANK_BATCHES;
    return (unsigned)((n + per - 1) / per);
}

/* Range of tiles u (along one axis) whose J block [4u-1, 4u+5] holds node i. */
__device__ static inline void covering(int i, int nt, int &lo, int &hi)
{
    lo = (i - 2 + 1024) / 4 - 256;          /* ceil((i - 5) / 4) = floor((i - 2) / 4), i >= -1022 */
    hi = (i + 1 + 1024) / 4 - 256;          /* floor((i + 1) / 4) */
    lo = lo < 0 ? 0 : lo;
    hi = hi > nt - 1 ? nt - 1 : hi;
}

/* J += sum of the item blocks of the tiles covering each node, in FP64.
 * Every node of an active tile's block is written once, by the first active
 * tile (in tile order) whose block holds it; the sum runs over the covering
 * tiles in tile order and over each tile's items in order, so the gather
 * adds in a fixed order (what a block holds follows the device order of
 * the tile's markers, which the sort's slot reservation by atomics does not
 * fix from run to run).  One thread per node and all three
 * components: a node lies in at most 2 blocks per axis, and the first item
 * of each of the (at most 8) covering tiles is loaded before any is added,
 * so the gather waits for one memory latency per node, not one per block. */
#define TJN3 (TJN * TJN * TJN)
struct JGatherArgs {
    JPtrs        v;
    Grid         g;
    TileView     tv;
    const float *tj;
    int          parity;     /* of the order that was pushed */
};

__device__ __forceinline__ static void jgather32(const JPtrs &v, const Grid &g, const TileView &tv,
                                                const float *tj, int parity,
                                                const VBlock &bk, const VBlock &gd)
{
    __shared__ int nfirst[27], nitem[27];    /* items of the 3x3x3 tiles around t (0: none) */
    const int nact = tv.nactive[parity];
    const int *active = tv.active + (long)parity * tv.ntiles;
    const int2 *titem = tv.titem + (long)parity * tv.ntiles;
    /* the first tile's load does not wait for the number of tiles: entries
     * past it are stale, and not used */
    const int first = active[(int)bk.x < tv.ntiles ? (int)bk.x : tv.ntiles - 1];
    for (int sl = (int)bk.x; sl < nact; sl += (int)gd.x) {
        const int t = sl == (int)bk.x ? first : active[sl];
        int t0, t1, t2;
        tile_coords(tv, t, t0, t1, t2);
        __syncthreads();
        if (threadIdx.x < 27) {
            const int ux = t0 - 1 + threadIdx.x / 9, uy = t1 - 1 + (threadIdx.x / 3) % 3,
                      uz = t2 - 1 + threadIdx.x % 3;
            const bool in = ux >= 0 && uy >= 0 && uz >= 0 && ux < tv.nt[0] && uy < tv.nt[1] &&
                            uz < tv.nt[2];
            const int2 ti = in ? titem[(ux * tv.nt[1] + uy) * tv.nt[2] + uz] : make_int2(0, 0);
            nfirst[threadIdx.x] = ti.x;
            nitem[threadIdx.x] = ti.y;
        }
        __syncthreads();
        /* nodes in reverse order: the nodes an interior tile owns (block
         * positions 3..6 along each axis, the others belong to the tiles
         * below) all fall in the first pass of the workgroup, so a tile
         * inside the plasma waits on memory once */
        for (int pass = threadIdx.x; pass < TJN3; pass += JG_TPB) {
            const int node = TJN3 - 1 - pass;
            const int cc = node % TJN, bb = (node / TJN) % TJN, aa = node / (TJN * TJN);
            const int i = 4 * t0 - 1 + aa, j = 4 * t1 - 1 + bb, k = 4 * t2 - 1 + cc;
            if (i < -2 || j < -2 || k < -2 || i > g.n[0] + 2 || j > g.n[1] + 2 || k > g.n[2] + 2)
                continue;
            int xl, xh, yl, yh, zl, zh;
            covering(i, tv.nt[0], xl, xh);
            covering(j, tv.nt[1], yl, yh);
            covering(k, tv.nt[2], zl, zh);
            /* the covering tiles (2 per axis at most), in tile order */
            int nb[8], off[8];
            bool use[8];
            int own = -1;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int ux = xl + (q >> 2), uy = yl + ((q >> 1) & 1), uz = zl + (q & 1);
                const bool inr = ux <= xh && uy <= yh && uz <= zh;
                const int b = inr ? ((ux - t0 + 1) * 3 + (uy - t1 + 1)) * 3 + (uz - t2 + 1) : 13;
                use[q] = inr && nitem[b] > 0;
                nb[q] = b;
                const int a = i - (4 * ux - 1), bq = j - (4 * uy - 1), cz = k - (4 * uz - 1);
                off[q] = use[q] ? ((a * TJN + bq) * TJN + cz) * 3 : 0;
                if (use[q] && own < 0) own = (ux * tv.nt[1] + uy) * tv.nt[2] + uz;
            }
            if (own != t) continue;
            const long o = gidx(g, i, j, k);
            const double J0 = v.J[0][o], J1 = v.J[1][o], J2 = v.J[2][o];
            float f[8][3];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const float *blk = tj + (long)(use[q] ? nfirst[nb[q]] : 0) * TJB + off[q];
                f[q][0] = blk[0];
                f[q][1] = blk[1];
                f[q][2] = blk[2];
            }
            double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                if (!use[q]) continue;
                s0 += (double)f[q][0];
                s1 += (double)f[q][1];
                s2 += (double)f[q][2];
                const int n_it = nitem[nb[q]];
                for (int w = 1; w < n_it; ++w) {          /* tiles split into several items */
                    const float *blk = tj + (long)(nfirst[nb[q]] + w) * TJB + off[q];
                    s0 += (double)blk[0];
                    s1 += (double)blk[1];
                    s2 += (double)blk[2];
                }
            }
            v.J[0][o] = J0 + s0;
            v.J[1][o] = J1 + s1;
            v.J[2][o] = J2 + s2;
        }
    }
}

template <> struct KernelDef<JGatherArgs> {
    static constexpr int kBlock = JG_TPB;
    __device__ __forceinline__ static void body(const JGatherArgs &a, VBlock b, VBlock gd)
    {
        jgather32(a.v, a.g, a.tv, a.tj, a.parity, b, gd);
    }
};

#endif
