/* OptionPricing: the launch interface between op_entry.c and op_kernels.hip
 * (not exported). */
#ifndef OP_INTERNAL_H
#define OP_INTERNAL_H

#include <stddef.h>
#include <stdint.h>

#define OP_MAX_BITS 32
#define OP_MAX_MODELS 4     /* models that share a pass over the paths */
#define OP_FEW_BLOCKS 1024  /* workgroups at most, contracts 1 and 2 */
#define OP_MANY_BLOCKS 2048 /* and contract 3 */

#ifdef __cplusplus
extern "C" {
#endif

/* Device pointers to the market data and the Brownian-bridge tables, as the
 * entry point received them (row-major), and the sizes. */
typedef struct {
  int32_t bits;        /* direction-vector bits */
  const float *cs, *vols, *drifts, *sts, *detvals, *discts;
  int32_t K, M;        /* discounts per model, models */
  const int32_t *bbi;  /* [3][dates] */
  const float *bbd;    /* [3][dates] */
  int64_t N;           /* paths */
} op_args;

/* Workgroups of the path kernel for N paths: the f64 partial sums it writes
 * are [op_blocks(contract, N)][models of the pass]. */
int op_blocks(int contract, int64_t paths);

/* Bytes of the tables that op_launch makes for a contract (0: none). */
size_t op_table_bytes(int contract);

/* Makes the contract's tables, runs the paths and writes the mean payoff per
 * model to out[M]; every launch on `stream` (a hipStream_t).  dir_vs
 * [dims][bits]; the contract fixes dims (1, 15 or 1101).  Returns 0 or a
 * hipError_t value. */
int op_launch(void *stream, int contract, const op_args *A, const int32_t *dir_vs,
              void *tables, double *partial, float *out);

#ifdef __cplusplus
}
#endif

#endif /* OP_INTERNAL_H */
