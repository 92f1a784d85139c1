/* Run ordering: Morton keys of a batch (cubie_amd/csrc/cubie_layout.hip).
 * Host library only; the generated kernels do not see this header. */
#ifndef CUBIE_ORDER_H
#define CUBIE_ORDER_H

#define CUBIE_ORDER_MAX_COLUMNS 9

#ifdef __cplusplus
extern "C" {
#endif

/* columns: a device matrix of doubles, one row of n_runs values per input
 * column. Key of run i: for each of n_cols rows index[k], the value scaled by
 * (x - lo[k]) / span[k] and quantised to `bits` bits, the bits of the columns
 * interleaved, most significant first, the first column highest; n_cols * bits
 * is at most 63. keys receives n_runs signed 64-bit integers. Enqueued on
 * `stream`. */
int cubie_hip_morton_keys(const double* columns, long long n_runs, int n_cols, int bits,
                          const int* index, const double* lo, const double* span,
                          long long* keys, void* stream);

#ifdef __cplusplus
}
#endif
#endif
