/* C ABI of the FP8 linear as a training step calls it: the forward of
 * block_scaled_matmul (fp8.py:50-78) with the FP8 operands of its backward
 * kept, and the FP8 backward (the forward rule applied to g and b, and to a.T
 * and g.T) from the kept operands or from a and b.  block_k is 128; operands
 * are bf16 or f32 (TG_DTYPE_*); row-major device pointers, the stream as
 * void*, TG_OK / TG_EINVAL / TG_EHIP as in tg_fp8.h.  M (tokens) and N need not
 * be multiples of 128: a partial last block is quantized over its valid
 * elements.  Nothing is allocated; buffers are 256-byte aligned. */
#ifndef TG_FP8_TRAIN_H
#define TG_FP8_TRAIN_H
#include <stddef.h>
#include <stdint.h>

#include "tg_fp8.h"

#ifdef __cplusplus
extern "C" {
#endif

#define TG_KEEP_A 1   /* a.T along M, for db */
#define TG_KEEP_B 2   /* b along N, for da */

size_t tg_linear_kept_bytes(int64_t M, int64_t N, int64_t K, int keep);
size_t tg_linear_fwd_workspace(int64_t M, int64_t N, int64_t K);

/* out (M, N) bf16 = a (M, K) . b (K, N) through FP8.  keep (TG_KEEP_*, M and N
 * multiples of 128): the operands written to `kept` for tg_linear_bwd_kept. */
int tg_linear_fwd(const void* a, int a_dtype, const void* b, int b_dtype, void* out, int64_t M, int64_t N,
                  int64_t K, int keep, void* kept, void* workspace, size_t workspace_bytes, void* stream);

size_t tg_linear_bwd_kept_workspace(int64_t M, int64_t N);

/* da (M, K) and db (K, N) from a forward's kept operands.  A null one is not
 * wanted.  A gradient of dtype f32 holds the bf16 result (fp8.py:95-96).  With
 * M == 0 or N == 0 nothing but the gradients is touched: the wanted one that
 * sums over the empty extent (db with M == 0, da with N == 0) is written as
 * zeros. */
int tg_linear_bwd_kept(const void* kept, int keep, const void* g, int g_dtype, void* da, int da_dtype, void* db,
                       int db_dtype, int64_t M, int64_t N, int64_t K, void* workspace, size_t workspace_bytes,
                       void* stream);

size_t tg_linear_bwd_workspace(int64_t M, int64_t N, int64_t K);

/* The same from a (M, K), b (K, N) and g (M, N), empty extents included; da has
 * a's dtype, db b's. */
int tg_linear_bwd(const void* a, int a_dtype, const void* b, int b_dtype, const void* g, int g_dtype, void* da,
                  void* db, int64_t M, int64_t N, int64_t K, void* workspace, size_t workspace_bytes,
                  void* stream);

#ifdef __cplusplus
}
#endif
#endif
