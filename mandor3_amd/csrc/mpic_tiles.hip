/*
 * mpic_tiles.hip -- per-step counting sort of the markers by tile-major
 * cell key.
 *
 * Per step: the push kernel writes each marker's new key and bumps
 * count[key] once per run of equal keys in a wavefront; the scan turns the
 * counts into per-key offsets and builds the lists of non-empty tiles and of
 * work items; the rank pass gives every live marker its slot
 * (cursor[key] reserved once per run) and records the marker's position in
 * the next order's permutation, dropping deleted markers.  The next push
 * reads its markers through that permutation and writes them to the other
 * buffer in order, so no pass moves markers only to sort them (the untiled
 * FP64 push, which keeps no order, is compacted by a scatter instead).
 *
 * Roofline (HBM-bound): scan ~ 3 x 4 B per cell key; rank 4 B read and 4 B
 * written per marker; scatter 4 + 60 + 60 B per FP64 marker.
 */
#include "mpic_tile_bodies.h"

/* Keys of the current array, with per-run counting.  Only the first
 * nmark[parity] markers are live; the buffer past them holds records of
 * earlier orders (or of loaded markers that the walls deleted), which must
 * not be counted. */
__global__ void k_keys64(Markers64 m, long n, Grid g, TileView tv, int parity)
{
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long live = tv.nmark[parity];
    int key = -1;
    if (p < n && p < live && m.qm[p] != 0.0f) {
        const double r[3] = {m.x[p], m.y[p], m.z[p]};
        key = cell_key_of(tv, g, r);
    }
    if (p < n) tv.key[p] = key;
    wave_run_count(tv.count, key);
}

int launch_keys64(hipStream_t s, const Markers64 &m, long n, const Grid &g, const TileView &tv,
                  int parity)
{
    if (n <= 0) return MPIC_OK;
    k_keys64<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(m, n, g, tv, parity);
    MPIC_CHECK(hipGetLastError());
    return MPIC_OK;
}

long tile_scan_words(int ntiles)
{
    return 6L * ((ntiles + SB - 1) / SB) + 1;
}

int launch_tile_scan(hipStream_t s, const TileView &tv, unsigned long long *words, unsigned *err,
                     int parity_next)
{
    const ScanArgs a = scan_args(tv, words, err, parity_next);
    return launch_def(s, a, (unsigned)a.nb);
}

int launch_rank(hipStream_t s, long nbound, const TileView &tv, int parity)
{
    if (nbound <= 0) return MPIC_OK;
    RankArgs a = {tv, nbound, parity};
    return launch_def(s, a, rank_blocks(nbound));
}

/* Moves each live marker of src to its slot in dst (the untiled FP64 push's
 * compacting sort). */
struct Scatter64Args {
    Markers64 src, dst;
    long      nbound;
    TileView  tv;
    int       parity;
};

__device__ static inline void scatter64(const Markers64 &src, const Markers64 &dst, long nbound,
                                        const TileView &tv, int parity, long p)
{
    const long n = tv.nmark[parity];
    const int key = (p < n && p < nbound) ? tv.key[p] : -1;
    int start, len;
    bool head;
    wave_run(key, start, len, head);
    int base = 0;
    if (head && key >= 0) base = atomicAdd(tv.cursor + key, len);
    base = __shfl(base, start, 64);
    if (key < 0) return;
    const long d = base + ((int)(threadIdx.x & 63) - start);
    /* every marker is streamed once: nontemporal, so the fields stay cached */
    __builtin_nontemporal_store(__builtin_nontemporal_load(src.x + p), dst.x + d);
    __builtin_nontemporal_store(__builtin_nontemporal_load(src.y + p), dst.y + d);
    __builtin_nontemporal_store(__builtin_nontemporal_load(src.z + p), dst.z + d);
    __builtin_nontemporal_store(__builtin_nontemporal_load(src.ux + p), dst.ux + d);
    __builtin_nontemporal_store(__builtin_nontemporal_load(src.uy + p), dst.uy + d);
    __builtin_nontemporal_store(__builtin_nontemporal_load(src.uz + p), dst.uz + d);
    __builtin_nontemporal_store(__builtin_nontemporal_load(src.w + p), dst.w + d);
    __builtin_nontemporal_store(__builtin_nontemporal_load(src.qm + p), dst.qm + d);
    __builtin_nontemporal_store(__builtin_nontemporal_load(src.id + p), dst.id + d);
}

template <> struct KernelDef<Scatter64Args> {
    static constexpr int kBlock = 256;
    __device__ __forceinline__ static void body(const Scatter64Args &a, VBlock b, VBlock)
    {
        scatter64(a.src, a.dst, a.nbound, a.tv, a.parity, (long)b.x * 256 + threadIdx.x);
    }
};

int launch_scatter64(hipStream_t s, const Markers64 &src, const Markers64 &dst, long nbound,
                     const TileView &tv, int parity)
{
    if (nbound <= 0) return MPIC_OK;
    Scatter64Args a = {src, dst, nbound, tv, parity};
    return launch_def(s, a, (unsigned)((nbound + 255) / 256));
}

/* Per-cell marker counts in natural (i, j, k) order from the offsets. */
__global__ void k_counts_natural(TileView tv, Grid g, int32_t *out)
{
    const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long nc = (long)g.n[0] * g.n[1] * g.n[2];
    if (c >= nc) return;
    const int k = (int)(c % g.n[2]);
    const long r = c / g.n[2];
    const int j = (int)(r % g.n[1]), i = (int)(r / g.n[1]);
    const int key = cell_key_ijk(tv, g, i, j, k), t = key / TILE_CELLS;
    if (tv.toff[t + 1] == tv.toff[t]) {
        out[c] = 0;                       /* empty tile: its key offsets are not kept */
        return;
    }
    const int end = (key % TILE_CELLS == TILE_CELLS - 1) ? tv.toff[t + 1] : tv.off[key + 1];
    out[c] = end - tv.off[key];
}

int launch_counts_natural(hipStream_t s, const TileView &tv, const Grid &g, int32_t *out)
{
    const long nc = (long)g.n[0] * g.n[1] * g.n[2];
    k_counts_natural<<<(unsigned)((nc + 255) / 256), 256, 0, s>>>(tv, g, out);
    MPIC_CHECK(hipGetLastError());
    return MPIC_OK;
}
