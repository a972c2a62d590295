/* C ABI of the decoder's prefill (decode.FP8Decoder.prefill): what a prompt's
 * layer needs beside the entry points of tg_fp8.h.  Row-major device pointers,
 * the stream as void*, TG_OK / TG_EINVAL / TG_EHIP as there. */
#ifndef TG_FP8_PREFILL_H
#define TG_FP8_PREFILL_H
#include <stdint.h>

#include "tg_fp8.h"

#ifdef __cplusplus
extern "C" {
#endif

/* K[b, h, t] = k, V[b, h, t] = v (model.py:59-65 for a whole prompt) for
 * t = 0 .. T - 1: qkv (B T, 3 H Dh) bf16 rows q | k | v, caches (B, H, S, Dh)
 * bf16, Dh a multiple of 8, all 16-byte aligned. */
int tg_prefill_kv(const void* qkv, void* k_cache, void* v_cache, int64_t B, int64_t T, int64_t H, int64_t S,
                  int64_t head_dim, void* stream);

#ifdef __cplusplus
}
#endif
#endif
