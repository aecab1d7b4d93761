/*
 * mpic_tiles.h -- tile-major cell keys, the per-step counting sort and the
 * work items shared by the FP64 and FP32 push kernels.
 *
 * The grid of cells is cut into 4x4x4-cell tiles; a marker's key is
 *   key = tile * 64 + (li * 4 + lj) * 4 + lk
 * so that sorting by key groups markers by tile and, inside a tile, by
 * cell.  Offsets are int32 (a run holds fewer than 2^31 markers).
 */
#ifndef MPIC_TILES_H
#define MPIC_TILES_H

#include "mpic_internal.h"

#define TILE_CELLS 64

struct TileView {
    int  nt[3];              /* tiles per axis */
    int  ntiles;
    long ncellp;             /* ntiles * 64 */
    int *off;                /* [ncellp + 1] first marker of every cell key of a non-empty
                              * tile (entries of empty tiles are not maintained) */
    int *toff;               /* [ntiles + 1] first marker of every tile */
    int *cursor;             /* [ncellp] scatter cursors */
    int *count;              /* [ncellp] markers per key after the push (zeroed by the scan) */
    int *key;                /* [capacity] new key of every marker, -1 = deleted */
    int *perm;               /* [capacity] the current order as indices into the
                              * current buffer (nmark[parity] of them; tiled runs) */
    /* What the J gather reads of the order is kept for two orders, by parity:
     * the scan then writes the next order's in the gather's launch. */
    int *active;             /* [2][ntiles] tiles holding markers, in tile order */
    int *nactive;            /* [2] */
    int *nmark;              /* [2] markers in the current / next order */
    int *xr;                 /* [2] x planes of nodes that the active tiles' gathers read
                              * (tiled runs: kept by the rank pass; else the whole grid) */
    /* Work items of the push: an active tile's markers, in the FP32 form split
     * evenly into ceil(count / chm) items of at most chm markers (chm = 0:
     * one item per active tile). */
    int  chm;
    int4 *item;              /* [item capacity] work items in tile order: tile, first and last + 1
                              * position in the order (one load tells a workgroup its work: a
                              * chain of lookups costs a memory latency per link) */
    int2 *titem;             /* [2][ntiles] first item and item count of every tile (count 0:
                              * empty), by parity like active */
    int *nitems;             /* [1] */
};

/* Work items of a tile holding c markers. */
__host__ __device__ static inline int tile_items(int c, int chm)
{
    return c <= 0 ? 0 : (chm > 0 ? (c + chm - 1) / chm : 1);
}

__device__ static inline void tile_coords(const TileView &tv, int t, int &t0, int &t1, int &t2)
{
    t2 = t % tv.nt[2];
    const int r = t / tv.nt[2];
    t1 = r % tv.nt[1];
    t0 = r / tv.nt[1];
}

__device__ static inline int cell_key_ijk(const TileView &tv, const Grid &g, int i, int j, int k)
{
    i = i < 0 ? 0 : (i >= g.n[0] ? g.n[0] - 1 : i);
    j = j < 0 ? 0 : (j >= g.n[1] ? g.n[1] - 1 : j);
    k = k < 0 ? 0 : (k >= g.n[2] ? g.n[2] - 1 : k);
    const int t = ((i >> 2) * tv.nt[1] + (j >> 2)) * tv.nt[2] + (k >> 2);
    return t * TILE_CELLS + (((i & 3) * 4 + (j & 3)) * 4 + (k & 3));
}

/* Key of a position: floor(x/h) as the reference's MF_DBL_TO_INT. */
__device__ static inline int cell_key_of(const TileView &tv, const Grid &g, const double r[3])
{
    const int i = (int)(r[0] / g.h[0] + 128.0) - 128;
    const int j = (int)(r[1] / g.h[1] + 128.0) - 128;
    const int k = (int)(r[2] / g.h[2] + 128.0) - 128;
    return cell_key_ijk(tv, g, i, j, k);
}

/* Wave-level run detection on a wave64: lanes holding equal keys in a row
 * form a run; returns (start lane, length) of the caller's run. */
__device__ static inline void wave_run(int key, int &start, int &len, bool &head)
{
    const int lane = threadIdx.x & 63;
    /* DPP wave_shr:1, a VALU move (a shuffle is a trip through the LDS unit) */
    const int prev = __builtin_amdgcn_update_dpp(key, key, 0x138, 0xf, 0xf, false);
    head = (lane == 0) || (key != prev);
    const unsigned long long hm = __ballot(head);
    const unsigned long long le = (lane == 63) ? ~0ull : ((1ull << (lane + 1)) - 1ull);
    start = 63 - __clzll(hm & le);
    const unsigned long long gt = hm & ~le;
    const int end = gt ? (__ffsll((long long)gt) - 1) : 64;
    len = end - start;
}

/* count[key] += run length, one atomic per run (all lanes must call). */
__device__ static inline void wave_run_count(int *count, int key)
{
    int start, len;
    bool head;
    wave_run(key, start, len, head);
    if (head && key >= 0) atomicAdd(count + key, len);
}

/* Row shift of a double by D lanes inside rows of 16 (DPP row_shr on
 * both halves; 0 from outside the row).  Every lane must be active. */
template <int D> __device__ static inline double row_shr(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x110 + D, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x110 + D, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

/* Sums of N values over the lanes' runs (first lane 'start') within each row
 * of 16 lanes: the last lane of a run in a row (run_tail) ends up with that
 * row's part.  fma(y, 1, x) is x + y rounded once, fma(y, 0, x) is x: one
 * instruction instead of a select of y and an add.  All lanes must call. */
template <int N> __device__ static inline void run_sums(double *v, int start)
{
    const int lane = threadIdx.x & 63;
    const double m1 = lane - 1 >= start ? 1.0 : 0.0, m2 = lane - 2 >= start ? 1.0 : 0.0,
                 m4 = lane - 4 >= start ? 1.0 : 0.0, m8 = lane - 8 >= start ? 1.0 : 0.0;
#pragma unroll
    for (int q = 0; q < N; ++q) {
        double x = v[q];
        x = __builtin_fma(row_shr<1>(x), m1, x);
        x = __builtin_fma(row_shr<2>(x), m2, x);
        x = __builtin_fma(row_shr<4>(x), m4, x);
        x = __builtin_fma(row_shr<8>(x), m8, x);
        v[q] = x;
    }
}

__device__ static inline bool run_tail(int start, int len)
{
    const int lane = threadIdx.x & 63, last = start + len - 1;
    return lane == last || ((lane & 15) == 15 && lane < last);
}

/* A marker's charge at its cell's eight nodes, source/core/plasma_rho.c:160-173;
 * node (a, b, c) of the cell is v[4 a + 2 b + c]. */
__device__ static inline void cic_weights(double sx, double sy, double sz, double val, double *v)
{
    v[0] = (1 - sx) * ((1 - sy) * ((1 - sz) * val));
    v[4] = sx * ((1 - sy) * ((1 - sz) * val));
    v[2] = (1 - sx) * (sy * ((1 - sz) * val));
    v[6] = sx * (sy * ((1 - sz) * val));
    v[1] = (1 - sx) * ((1 - sy) * (sz * val));
    v[5] = sx * ((1 - sy) * (sz * val));
    v[3] = (1 - sx) * (sy * (sz * val));
    v[7] = sx * (sy * (sz * val));
}

/* run_sums for values that need not be finite: a lane outside the run is not
 * added at all (0 times infinity would reach the neighbouring runs). */
template <int D> __device__ static inline double run_step(double x, bool in)
{
    const double y = row_shr<D>(x);
    return in ? x + y : x;
}

template <int N> __device__ static inline void run_sums_any(double *v, int start)
{
    const int lane = threadIdx.x & 63;
    const bool m1 = lane - 1 >= start, m2 = lane - 2 >= start, m4 = lane - 4 >= start,
               m8 = lane - 8 >= start;
#pragma unroll
    for (int q = 0; q < N; ++q)
        v[q] = run_step<8>(run_step<4>(run_step<2>(run_step<1>(v[q], m1), m2), m4), m8);
}

/* rho += the lanes' markers (cell: index of the cell's first node, -1 none):
 * markers in cell order are summed over each run of one cell first, so that
 * HBM sees at most four atomics per node and run of a wavefront.  With one per
 * marker and node the atomics were all the time: 96 x 48 x 48 foil (0.3 M
 * markers) 372 us, laser-foil 4.34 ms; now 20 and 248 us.  A marker whose
 * charge is not finite leaves the other cells' sums alone. */
__device__ static inline void rho_run_add(double *rho, const Grid &g, long cell, double *v)
{
    int start, len;
    bool head;
    wave_run((int)cell, start, len, head);
    run_sums_any<8>(v, start);
    if (!run_tail(start, len) || cell < 0) return;
    const long si = (long)g.GY * g.GZ, sj = g.GZ;
#pragma unroll
    for (int q = 0; q < 8; ++q)
        unsafeAtomicAdd(rho + cell + (q >> 2) * si + ((q >> 1) & 1) * sj + (q & 1), v[q]);
}

int launch_keys64(hipStream_t s, const Markers64 &m, long n, const Grid &g, const TileView &tv,
                  int parity);
/* The tile scan's word buffer (zeroed once at allocation) and launcher;
 * err bit 1 is set if a wait of the scan ran out (never expected). */
long tile_scan_words(int ntiles);
int launch_tile_scan(hipStream_t s, const TileView &tv, unsigned long long *words, unsigned *err,
                     int parity_next);
int launch_rank(hipStream_t s, long nbound, const TileView &tv, int parity);
int launch_scatter64(hipStream_t s, const Markers64 &src, const Markers64 &dst, long nbound,
                     const TileView &tv, int parity);
int launch_push64_tiled(hipStream_t s, const Markers64 &m, const Markers64 &dst,
                        const Fields64 &f, const Grid &g, const PushConsts &c,
                        const TileView &tv, double *kin, unsigned *err, int nblocks, int waves);
int launch_counts_natural(hipStream_t s, const TileView &tv, const Grid &g, int32_t *out);

/* J block of one tile: nodes [4t-1, 4t+5] per axis, xyz interleaved. */
#define TJN 7
#define TJB (TJN * TJN * TJN * 3)

/* nblocks workgroups of 'waves' (1, 2, 4 or 8) wavefronts each. */
int launch_push32(hipStream_t s, const Markers32 &m, const Markers32 &dst, const Fields32 &f,
                  const Grid &g, const PushConsts &pc, const float *qm, const TileView &tv,
                  float *tj, double *kin, int nblocks, int waves);
int launch_jgather32(hipStream_t s, const JPtrs &j, const Grid &g, const TileView &tv,
                     const float *tj, int parity, int nblocks);

/* What the loop body's launches between the push and the E update work on. */
struct AfterPush {
    const BoxSet       *updE;          /* the E caps' update boxes */
    const FaceOp       *ops;           /* the walls on the E caps, x then y then z */
    int                 nop;
    JPtrs               jp;
    int                 bc[6];
    const int          *jr;            /* x planes where J may be non-zero */
    const TileView     *tv;
    unsigned long long *scanw;
    unsigned           *err;
    int                 parity, sorted;   /* sorted: a tiled run, ranked here */
    long                nbound;
    const float        *tj;            /* FP32: the J blocks */
    int                 gather_blocks;
    hipEvent_t          after_gather;  /* FP32: the J gather alone, then this (null: not timed) */
    /* the diagnostics ring's row of this step */
    const double       *part, *kin;
    int                 nparts;
    double             *ring;
    const int          *step;
    int                 ringcap;
};
template <class T>
int launch_after_push(hipStream_t s, const FieldsT<T> &f, const Grid &g, const AfterPush &p);
int launch_keys32(hipStream_t s, const Markers32 &m, long n, const TileView &tv, int parity);
int launch_rho32(hipStream_t s, const Markers32 &m, long n, double *rho, const Grid &g,
                 const TileView &tv, int parity);
int launch_cells32(hipStream_t s, const Markers32 &m, long n, const Grid &g, const TileView &tv,
                   int parity, int32_t *cell);

#endif
