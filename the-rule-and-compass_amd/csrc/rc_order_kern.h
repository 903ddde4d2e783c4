/*
 * Launchers of the row kernels of the order and maximum stages
 * (rc_order_kern.hip) for their host side (rc_order.hip).
 */
#ifndef RC_ORDER_KERN_H
#define RC_ORDER_KERN_H

#include <hip/hip_runtime.h>
#include <stdint.h>

/* One program set as the row kernels see it: its value stream of the fit VM
   (word pairs in `code`) and its post-order records (in `prog`). */
struct OrSet {
    uint32_t t_off; /* value stream: first word, word pairs; 0 pairs: none */
    int t_m;
    uint32_t r_off; /* records: first word, count */
    int m;
};

struct OrRows {
    const double *cols64;
    const double *y64;
    int n, v;
};

/* A tile's share of a maximum scan. */
struct OrMax {
    unsigned long long key; /* bits of max |r| */
    double lo, hi;
    int row;
    int veto;
};

/* Values the record sweep keeps below its top of stack. */
#define OR_SDEPTH 8
/* Rows the row kernels take: a step past the last one stays in an int. */
#define OR_MAX_ROWS 0x7fff0000
/* Words of a value stream (rch_fitvm_compile's limit for 96 nodes). */
#define OR_STREAM_WORDS (2 * 4 * 96)

/* Sort keys of the segments segs[0 .. nlist) over all rows (rank: of the
   prediction, with the rows; else of |prediction - y|). */
void or_launch_keys(bool rank, int nlist, hipStream_t s, const int *segs, const OrSet *sets,
                    const uint32_t *code, const double *c0, int kmax, int ntrials, OrRows rows,
                    unsigned long long *keys, uint32_t *row_of, int *status);

/* Tiles (and their rows) of a maximum scan over n rows and nsegs segments. */
int or_max_tiles(int n, int nsegs, int *tile_rows);

/* Maximum scan of the segments segs[0 .. nlist): level false, the maximum by
   the value stream; true, the maximum and the level's interval by the record
   sweep.  part holds nlist * tiles entries; redo[seg] is set where a row is
   not finite, or a partial of its derivative is not or leads out of the range of
   f64. */
void or_launch_max(bool level, int nlist, hipStream_t s, const int *segs, const OrSet *sets,
                   const uint32_t *code, const uint32_t *prog, const double *c0, int kmax,
                   int ntrials, const int *coords, const double *levels, OrRows rows, OrMax *part,
                   int tiles, int tile_rows, int *redo);

#endif
