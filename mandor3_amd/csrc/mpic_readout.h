/*
 * mpic_readout.h -- results packed on the device and brought to host memory
 * (mpic_readout.hip).
 */
#ifndef MPIC_READOUT_H
#define MPIC_READOUT_H

#include "mpic_internal.h"

/* nc interleaved components on the nodes lo .. lo + d - 1 of every axis. */
struct NodeBlock {
    Grid g;
    int  lo, d[3], nc;
};

/* Markers of an order, as records of 'words' 8-byte words (8 or 7).  An entry
 * of the order that names none of the buffer's first *extent records is not
 * followed: its position goes to *bad (host memory, set to -1 by the caller). */
struct MarkerBlock {
    const int *perm;
    const int *extent;
    long      *bad;
    int        words;
    int        nt[3];              /* FP32: tiles per axis, mesh steps, q/m per species */
    double     h[3];
    float      qm[8];
};

struct Readout {
    enum Kind { BLOCK32, BLOCK64, NODES32, NODES64, MARKERS32, MARKERS64 } kind;
    long        words;             /* 8-byte words of the result */
    void       *dst;               /* host memory */
    NodeBlock   block;
    int         mean;              /* NODES: 0 along the component's axis, 1 around the node */
    const void *F[3];
    MarkerBlock markers;
    Markers32   m32;
    Markers64   m64;
    int launch(hipStream_t s, long first, long count, void *out) const;
};

#define TRY_READOUT(x)                  \
    do {                                \
        const int rc_ = (x);            \
        if (rc_ != MPIC_OK) return rc_; \
    } while (0)

/* n results, complete when it returns; ordered after the work on s. */
int readout(const Readout *r, int n, int dev, hipStream_t s);
/* A run exists / is gone (the pinned slots live as long as any run). */
void readout_ref(void);
void readout_unref(void);

#endif
