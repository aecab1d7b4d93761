/*
 * mpic_readout.hip -- results on their way to the host: node blocks of the
 * fields, J and rho, the Tecplot node values and the marker records, laid out
 * on the device as the host wants them and written straight to pinned host
 * memory (source/type_mesh.c:285-311, source/IO_tecplot.c:131-214,
 * source/core/plasma_IO.c:273-287 hold the layouts).
 *
 * What bounds it is PCIe (57 GB/s measured) and, for large results, the
 * caller's memory: fresh pages cost the host more than the transfer.  A result
 * larger than one slot goes through up to eight host threads, each with two pinned
 * slots, so that packing, transfer, page faults and copies overlap.  The
 * copies component by component into pageable memory and the interleaving on
 * one host thread that this replaces took 30 ms for the E and H of a
 * 256 x 128 x 128 run (208 MB).
 *
 * Built with -ffp-contract=off: values are those of the host expressions.
 */
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <thread>
#include <type_traits>
#include <vector>

#include "mpic_readout.h"

#define TPB 256

static inline unsigned nblk(long n) { return (unsigned)((n + TPB - 1) / TPB); }

/* ---------------- packing kernels ----------------
 * Each writes items [first, first + count) of its result to out[0 .. count):
 * consecutive lanes write consecutive words, since partial lines over PCIe
 * cost as much as whole ones. */

/* Doubles of nc interleaved components on the nodes lo .. lo + d - 1 per axis,
 * k fastest. */
template <class T>
__global__ void k_pack_block(NodeBlock b, const T *F0, const T *F1, const T *F2, long first,
                             long count, double *out)
{
    const long t = (long)blockIdx.x * TPB + threadIdx.x;
    if (t >= count) return;
    const long e = first + t;
    const unsigned long node = (unsigned long)e / (unsigned)b.nc;
    const int c = (int)(e - (long)node * b.nc);
    const unsigned long r = node / (unsigned)b.d[2];
    const int k = (int)(node - r * b.d[2]), i = (int)(r / (unsigned)b.d[1]),
              j = (int)(r - (unsigned long)i * b.d[1]);
    const T *F = c == 0 ? F0 : (c == 1 ? F1 : F2);
    out[t] = (double)F[gidx(b.g, b.lo + i, b.lo + j, b.lo + k)];
}

/* Node values of the Tecplot records (source/IO_tecplot.c:131-153), nodes
 * [0, n]: kind 0 (E, J) the mean of the two values along the component's axis,
 * kind 1 (H) the mean of the four around the node, in the reference's order. */
template <class T>
__global__ void k_pack_nodes(Grid g, int kind, const T *F0, const T *F1, const T *F2, long first,
                             long count, double *out)
{
    const long t = (long)blockIdx.x * TPB + threadIdx.x;
    if (t >= count) return;
    const long e = first + t;
    const unsigned long node = (unsigned long)e / 3u;
    const int c = (int)(e - (long)node * 3);
    const unsigned long r = node / (unsigned)(g.n[2] + 1);
    const int k = (int)(node - r * (g.n[2] + 1)), i = (int)(r / (unsigned)(g.n[1] + 1)),
              j = (int)(r - (unsigned long)i * (g.n[1] + 1));
    const T *F = c == 0 ? F0 : (c == 1 ? F1 : F2);
    const long o = gidx(g, i, j, k), s[3] = {(long)g.GY * g.GZ, g.GZ, 1};
    if (kind == 0) {
        const long a = c == 0 ? s[0] : (c == 1 ? s[1] : s[2]);
        out[t] = 0.5 * ((double)F[o] + (double)F[o + a]);
    } else {
        const long p = c == 0 ? s[1] : s[0], q = c == 2 ? s[1] : s[2];
        out[t] = 0.25 * ((double)F[o] + (double)F[o + p] + (double)F[o + q] + (double)F[o + p + q]);
    }
}

/* Words of marker_t records (source/type_marker.h:12-25): 8 per record of 64
 * bytes (the last: id and zero padding), 7 of 56.  Markers of the order's
 * positions, through its permutation. */
__device__ static inline unsigned long long two_words(float lo, float hi)
{
    return (unsigned long long)__float_as_uint(hi) << 32 | __float_as_uint(lo);
}

/* The record at position u of the order, -1 (reported) if there is none. */
__device__ static inline long order_entry(const MarkerBlock &b, long u)
{
    const int q = b.perm[u];
    if (q >= 0 && q < *b.extent) return q;
    *b.bad = u;
    return -1;
}

__global__ void k_pack_markers32(MarkerBlock b, Markers32 m, long first, long count,
                                 unsigned long long *out)
{
    const long t = (long)blockIdx.x * TPB + threadIdx.x;
    if (t >= count) return;
    const long e = first + t, u = e / b.words;
    const int w = (int)(e - u * b.words);
    const long q = order_entry(b, u);
    if (q < 0) {
        out[t] = 0;
        return;
    }
    if (w == 7) {
        out[t] = (unsigned)m.id[q];
        return;
    }
    if (w >= 3 && w < 6) {
        const float4 v = m.mom[q];
        out[t] = __double_as_longlong((double)(w == 3 ? v.x : (w == 4 ? v.y : v.z)));
        return;
    }
    const float4 p = m.pos[q];
    const int word = __float_as_int(p.x), key = word & ((1 << 29) - 1);
    if (w == 6) {
        out[t] = two_words(m.mom[q].w, b.qm[(unsigned)word >> 29]);
        return;
    }
    const int loc = key & 63, tile = key >> 6;
    const int t2 = tile % b.nt[2], r = tile / b.nt[2], t1 = r % b.nt[1], t0 = r / b.nt[1];
    const int c = w == 0 ? 4 * t0 + (loc >> 4) : (w == 1 ? 4 * t1 + (loc >> 2 & 3) : 4 * t2 + (loc & 3));
    out[t] = __double_as_longlong((c + (double)(w == 0 ? p.y : (w == 1 ? p.z : p.w))) * b.h[w]);
}

__global__ void k_pack_markers64(MarkerBlock b, Markers64 m, long first, long count,
                                 unsigned long long *out)
{
    const long t = (long)blockIdx.x * TPB + threadIdx.x;
    if (t >= count) return;
    const long e = first + t, u = e / b.words;
    const int w = (int)(e - u * b.words);
    const long q = order_entry(b, u);
    if (q < 0) {
        out[t] = 0;
        return;
    }
    if (w == 7) {
        out[t] = (unsigned)m.id[q];
    } else if (w == 6) {
        out[t] = two_words(m.w[q], m.qm[q]);
    } else {
        const double *s = w == 0 ? m.x : (w == 1 ? m.y : (w == 2 ? m.z : (w == 3 ? m.ux : (w == 4 ? m.uy : m.uz))));
        out[t] = __double_as_longlong(s[q]);
    }
}

/* A launch that returns its own status: hipGetLastError would also return (and
 * take away) what a call of the caller's thread has left there. */
template <class... A>
static int start(hipStream_t s, unsigned blocks, void (*kernel)(A...), std::common_type_t<A>... a)
{
    void *args[] = {(void *)&a...};
    MPIC_CHECK(hipLaunchKernel((const void *)kernel, dim3(blocks), dim3(TPB), args, 0, s));
    return MPIC_OK;
}

int Readout::launch(hipStream_t s, long first, long count, void *out) const
{
    const unsigned nb = nblk(count);
    double *d = (double *)out;
    unsigned long long *w = (unsigned long long *)out;
    const float *f0 = (const float *)F[0], *f1 = (const float *)F[1], *f2 = (const float *)F[2];
    const double *d0 = (const double *)F[0], *d1 = (const double *)F[1], *d2 = (const double *)F[2];
    switch (kind) {
    case BLOCK32: return start(s, nb, k_pack_block<float>, block, f0, f1, f2, first, count, d);
    case BLOCK64: return start(s, nb, k_pack_block<double>, block, d0, d1, d2, first, count, d);
    case NODES32: return start(s, nb, k_pack_nodes<float>, block.g, mean, f0, f1, f2, first, count, d);
    case NODES64: return start(s, nb, k_pack_nodes<double>, block.g, mean, d0, d1, d2, first, count, d);
    case MARKERS32: return start(s, nb, k_pack_markers32, markers, m32, first, count, w);
    case MARKERS64: return start(s, nb, k_pack_markers64, markers, m64, first, count, w);
    }
    return MPIC_ERR_ARG;
}

/* ---------------- pinned slots and helper threads ----------------
 * Two sets per process, shared by all runs: two slots for each of at most
 * HELPERS + 1 threads, and two for a caller without helpers, allocated and
 * started when first needed, given back with the last run.  A call takes the
 * first set if it is free and packs behind whatever is in flight on its run's
 * stream.  One that finds it taken, perhaps by a call that waits for a thousand
 * steps, waits for its own stream, then takes the first set if it is free by
 * now and the second if not: that one is never held while steps run.  So a
 * read-out behind queued steps holds up no other run's, and since runs are
 * counted under a lock of their own, no mpic_create or mpic_destroy.  (With
 * every call waiting for its stream first, a read-out behind steps took 20 to
 * 45 us more: its launches were no longer queued while the steps ran.)
 *
 * The threads wait between calls and claim chunks one by one, so that one that
 * wakes late (the caller's process may keep every core busy) only finds less
 * left to do; threads started for each call and dealt fixed chunks took 2.5 ms
 * instead of 0.5 for 13 MB beside spinning OpenMP threads. */
#define SLOT_WORDS (1L << 17)          /* 1 MiB */
#define HELPERS 7

struct Job {
    const Readout *r;
    long           nchunks;
    int            dev;
    hipStream_t    stream;
    std::atomic<long> next{0}, done{0};
    std::atomic<int>  rc{MPIC_OK};
};

struct Slots {
    std::mutex use;                    /* held by the call that packs through them */
    long       words = 0;              /* pinned words allocated */
    void      *mem = nullptr;
};

struct Pool {
    std::mutex life;                   /* guards runs; taken before the sets */
    int        runs = 0;
    Slots      set[2];                 /* with the helpers; for the caller alone */
    std::mutex mu;                     /* guards what follows, the helpers' */
    std::condition_variable wake, finished;
    std::vector<std::thread> threads;
    std::shared_ptr<Job> job;
    long       serial = 0;             /* of the job */
    bool       stop = false;
};

/* Never destroyed: a process that ends with runs still open ends with the
 * helpers waiting, and destroying what they wait on would never return. */
static Pool &g_pool = *new Pool;

/* Chunks of the job through two slots: the next is packed while this one is
 * copied out.  A claimed chunk is always accounted for. */
static void work(Job &J, char *slots)
{
    hipEvent_t ev[2] = {nullptr, nullptr};
    long at[2] = {-1, -1};
    int slot = 0, rc = MPIC_OK;
    const auto finish = [&](int o) {
        const long first = at[o] * SLOT_WORDS, left = J.r->words - first;
        if (rc == MPIC_OK && hipEventSynchronize(ev[o]) != hipSuccess) rc = MPIC_ERR_DEVICE;
        if (rc == MPIC_OK)
            memcpy((char *)J.r->dst + 8 * first, slots + 8 * SLOT_WORDS * o,
                   8 * std::min(SLOT_WORDS, left));
        at[o] = -1;
        if (rc != MPIC_OK) J.rc = rc;
        if (++J.done == J.nchunks) {
            std::lock_guard<std::mutex> lk(g_pool.mu);
            g_pool.finished.notify_all();
        }
    };
    for (;;) {
        const long c = J.next < J.nchunks ? J.next++ : J.nchunks;
        if (c < J.nchunks) {
            if (!ev[slot] && (hipSetDevice(J.dev) != hipSuccess ||
                              hipEventCreateWithFlags(&ev[slot], hipEventDisableTiming) != hipSuccess))
                rc = MPIC_ERR_DEVICE;
            const long first = c * SLOT_WORDS;
            at[slot] = c;
            if (rc == MPIC_OK)
                rc = J.r->launch(J.stream, first, std::min(SLOT_WORDS, J.r->words - first),
                                 slots + 8 * SLOT_WORDS * slot);
            if (rc == MPIC_OK && hipEventRecord(ev[slot], J.stream) != hipSuccess)
                rc = MPIC_ERR_DEVICE;
        }
        slot ^= 1;
        if (at[slot] >= 0) finish(slot);
        if (c >= J.nchunks) {
            if (at[slot ^ 1] >= 0) finish(slot ^ 1);
            break;
        }
    }
    for (hipEvent_t e : ev)
        if (e) hipEventDestroy(e);
}

static void helper(int w)
{
    long seen = 0;
    for (;;) {
        std::shared_ptr<Job> job;
        {
            std::unique_lock<std::mutex> lk(g_pool.mu);
            g_pool.wake.wait(lk, [&] { return g_pool.stop || (g_pool.job && g_pool.serial != seen); });
            if (g_pool.stop) return;
            seen = g_pool.serial;
            job = g_pool.job;
        }
        work(*job, (char *)g_pool.set[0].mem + 8 * SLOT_WORDS * 2 * w);
    }
}

void readout_ref(void)
{
    std::lock_guard<std::mutex> lk(g_pool.life);
    ++g_pool.runs;
}

void readout_unref(void)
{
    std::lock_guard<std::mutex> l0(g_pool.life);
    if (--g_pool.runs > 0) return;
    {
        std::lock_guard<std::mutex> l2(g_pool.mu);
        g_pool.stop = true;
        g_pool.wake.notify_all();
    }
    for (std::thread &t : g_pool.threads) t.join();
    g_pool.threads.clear();
    g_pool.stop = false;
    for (Slots &S : g_pool.set) {
        if (S.mem) hipHostFree(S.mem);
        S.mem = nullptr;
        S.words = 0;
    }
}

/* At least 'words' pinned words; only grows while no helper runs. */
static int slots_reserve(Slots &S, long words)
{
    if (words <= S.words) return MPIC_OK;
    if (S.mem) hipHostFree(S.mem);
    S.mem = nullptr;
    S.words = 0;
    MPIC_CHECK(hipHostMalloc(&S.mem, 8 * words, hipHostMallocPortable));
    S.words = words;
    return MPIC_OK;
}

int readout(const Readout *r, int n, int dev, hipStream_t s)
{
    int k = 0;
    std::unique_lock<std::mutex> lk(g_pool.set[0].use, std::try_to_lock);
    if (!lk) {
        MPIC_CHECK(hipStreamSynchronize(s));
        if (!lk.try_lock()) {
            k = 1;
            lk = std::unique_lock<std::mutex>(g_pool.set[1].use);
        }
    }
    Slots &S = g_pool.set[k];
    long all = 0;
    for (int q = 0; q < n; ++q) all += r[q].words;
    if (all <= SLOT_WORDS) {
        /* everything through one slot, one wait */
        TRY_READOUT(slots_reserve(S, SLOT_WORDS));
        char *at = (char *)S.mem;
        int rc = MPIC_OK;
        for (int q = 0; q < n && rc == MPIC_OK; ++q) {
            if (r[q].words) rc = r[q].launch(s, 0, r[q].words, at);
            at += 8 * r[q].words;
        }
        MPIC_CHECK(hipStreamSynchronize(s));         /* nothing writes the slot any more */
        if (rc != MPIC_OK) return rc;
        at = (char *)S.mem;
        for (int q = 0; q < n; ++q) {
            if (r[q].words) memcpy(r[q].dst, at, 8 * r[q].words);
            at += 8 * r[q].words;
        }
        return MPIC_OK;
    }
    const int helpers = k == 0 ? HELPERS : 0;
    TRY_READOUT(slots_reserve(S, SLOT_WORDS * 2 * (helpers + 1)));
    for (int q = 0; q < n; ++q) {
        const auto job = std::make_shared<Job>();
        job->r = r + q;
        job->nchunks = (r[q].words + SLOT_WORDS - 1) / SLOT_WORDS;
        job->dev = dev;
        job->stream = s;
        if (!job->nchunks) continue;
        while (g_pool.threads.size() < (size_t)std::min<long>(helpers, job->nchunks - 1)) {
            try {
                const int w = (int)g_pool.threads.size() + 1;
                g_pool.threads.emplace_back(helper, w);
            } catch (...) {
                break;                              /* no more threads: fewer do */
            }
        }
        if (helpers) {
            std::lock_guard<std::mutex> l2(g_pool.mu);
            g_pool.job = job;
            ++g_pool.serial;
        }
        if (helpers && job->nchunks > 1) g_pool.wake.notify_all();
        work(*job, (char *)S.mem);
        if (helpers) {
            std::unique_lock<std::mutex> l2(g_pool.mu);
            g_pool.finished.wait(l2, [&] { return job->done == job->nchunks; });
            g_pool.job.reset();
        }
        if (job->rc != MPIC_OK) {
            hipStreamSynchronize(s);                /* nothing writes the slots any more */
            mpic_set_error("a result could not be read back from the device");
            return job->rc;
        }
    }
    return MPIC_OK;
}
