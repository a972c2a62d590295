/* Which tile the FP8 GEMM takes (host arithmetic only, for tests and tuning;
 * every tile gives the same output bits).  Return values as in tg_fp8.h. */
#ifndef TG_FP8_TILES_H
#define TG_FP8_TILES_H
#include <stdint.h>

#include "tg_fp8.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The tile (rows x cols of C) of an M x N product over K (a multiple of 128) on
 * a device of `cus` compute units: scales_km as tg_gemm_fp8_nt_km (1) or
 * tg_gemm_fp8_nt (0), c_dtype TG_DTYPE_BF16 or TG_DTYPE_F32.  Operands past
 * 32-bit offsets take a kernel of their own: rows and cols 0. */
int tg_gemm_fp8_tile(int64_t M, int64_t N, int64_t K, int scales_km, int c_dtype, int cus, int* rows, int* cols);

#ifdef __cplusplus
}
#endif
#endif
