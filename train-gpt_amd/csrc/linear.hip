// block_scaled_matmul as a training step calls it (fp8.py:30-36, 50-98): the
// forward with the FP8 operands of its backward kept, and the FP8 backward from
// those or from the operands themselves, each as one call on caller-provided
// memory.  Any token count and width: a tensor is quantized in both directions
// from one read, a partial last block over its valid elements, straight into
// operands whose contraction is padded to whole blocks, so nothing is copied to
// a padded tensor first (3000 x 2304 x 9216, forward and backward: three fills,
// three copies and two slices, 72 us, and five quantizer launches, 48 us, are
// two launches of 56 us).  f32 operands go through the same tiles.
#include "tg_device.h"
#include "tg_host.h"
#include "../../include/tg_fp8_train.h"

namespace tg {

static inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }
static inline int64_t round128(int64_t x) { return (x + 127) & ~(int64_t)127; }

// A quantized operand (rows x contraction bytes, K-block-major scales) carved from a buffer.
struct FpOperand {
  uint8_t* q = nullptr;
  float* s = nullptr;
};
static size_t operand_bytes(int64_t rows, int64_t k) {
  return align256((size_t)rows * (size_t)k) + align256((size_t)rows * (size_t)(k / 128) * 4);
}
static FpOperand carve(uint8_t*& p, int64_t rows, int64_t k) {
  FpOperand o;
  o.q = p;
  o.s = reinterpret_cast<float*>(p + align256((size_t)rows * (size_t)k));
  p += operand_bytes(rows, k);
  return o;
}

static bool valid_dtype(int d) { return d == TG_DTYPE_BF16 || d == TG_DTYPE_F32; }
static bool aligned_as(const void* p, int dtype) { return aligned(p, dtype == TG_DTYPE_F32 ? 4 : 2); }
static int grad_dtype(int d) { return d == TG_DTYPE_F32 ? kOutF32OfBf16 : TG_DTYPE_BF16; }

// The wanted gradients of an empty M or N, where nothing is summed: zeros.
static int zero_grad(void* d, int dtype, int64_t n, hipStream_t st) {
  return d ? launch_fill_zero_bf16(d, dtype == TG_DTYPE_F32 ? 2 * n : n, st) : TG_OK;
}
static int zero_grads(void* da, int da_dtype, void* db, int db_dtype, int64_t M, int64_t N, int64_t K, hipStream_t st) {
  TG_TRY(zero_grad(da, da_dtype, M * K, st));
  return zero_grad(db, db_dtype, K * N, st);
}

}  // namespace tg

using namespace tg;

extern "C" size_t tg_linear_kept_bytes(int64_t M, int64_t N, int64_t K, int keep) {
  if (M < 0 || N < 0 || K < 0) return 0;
  return (keep & TG_KEEP_A ? operand_bytes(K, M) : 0) + (keep & TG_KEEP_B ? operand_bytes(K, N) : 0);
}

extern "C" size_t tg_linear_fwd_workspace(int64_t M, int64_t N, int64_t K) {
  if (M < 0 || N < 0 || K < 0) return 0;
  return operand_bytes(M, K) + operand_bytes(N, K);
}

extern "C" int tg_linear_fwd(const void* a, int a_dtype, const void* b, int b_dtype, void* out, int64_t M,
                             int64_t N, int64_t K, int keep, void* kept, void* workspace,
                             size_t workspace_bytes, void* stream) {
  TG_TRY(check_gemm_args("linear_fwd", M, N, K, 128, 1));
  if (!valid_dtype(a_dtype) || !valid_dtype(b_dtype)) return einval("linear_fwd: operands must be bf16 or f32");
  if (keep & ~(TG_KEEP_A | TG_KEEP_B)) return einval("linear_fwd: bad keep");
  if (keep && (M % 128 || N % 128)) return einval("linear_fwd: kept operands need M and N in whole blocks of 128");
  if (M == 0 || N == 0) return TG_OK;
  if (!a || !b || !out || !workspace || (keep && !kept)) return einval("linear_fwd: null pointer");
  if (workspace_bytes < tg_linear_fwd_workspace(M, N, K)) return einval("linear_fwd: workspace too small");
  // b by itself along K (beside an f32 a, or where a.T alone is kept) may start at any element
  const bool b_any = b_dtype == TG_DTYPE_F32 || a_dtype == TG_DTYPE_F32 || keep == TG_KEEP_A;
  if (!aligned(a, 16) || !(b_any ? aligned_as(b, b_dtype) : aligned(b, 16)) || !aligned(workspace, 256) ||
      !aligned(kept, 256))
    return einval("linear_fwd: a and b must be 16-byte and the buffers 256-byte aligned");
  hipStream_t st = as_stream(stream);
  uint8_t* p = reinterpret_cast<uint8_t*>(workspace);
  uint8_t* k = reinterpret_cast<uint8_t*>(kept);
  const FpOperand qa = carve(p, M, K), qbt = carve(p, N, K);
  FpOperand qat, qb;
  if (keep & TG_KEEP_A) qat = carve(k, K, M);
  if (keep & TG_KEEP_B) qb = carve(k, K, N);
  const QuantTensor t[2] = {{a, a_dtype, M, K, keep & TG_KEEP_A ? 0 : 1, qa.q, qa.s, qat.q, qat.s},
                            {b, b_dtype, K, N, keep & TG_KEEP_B ? 0 : 2, qb.q, qb.s, qbt.q, qbt.s}};
  TG_TRY(launch_quant_tensors(t, 2, true, st));                                                // fp8.py:66, 68
  return launch_gemm_fp8(qa.q, qa.s, qbt.q, qbt.s, 1, out, TG_DTYPE_BF16, M, N, K, st, true);   // fp8.py:70-78
}

// g along N for dX and g.T along M for dW, from one read of g.
static int g_part(const void* da, const void* db) { return da && db ? 0 : da ? 1 : 2; }

extern "C" size_t tg_linear_bwd_kept_workspace(int64_t M, int64_t N) {
  if (M < 0 || N < 0) return 0;
  return operand_bytes(M, round128(N)) + operand_bytes(N, round128(M));
}

extern "C" int tg_linear_bwd_kept(const void* kept, int keep, const void* g, int g_dtype, void* da, int da_dtype,
                                  void* db, int db_dtype, int64_t M, int64_t N, int64_t K, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  TG_TRY(check_gemm_args("linear_bwd_kept", M, N, K, 128, 1));
  if (!valid_dtype(g_dtype) || !valid_dtype(da_dtype) || !valid_dtype(db_dtype))
    return einval("linear_bwd_kept: gradients must be bf16 or f32");
  if (M % 128 || N % 128) return einval("linear_bwd_kept: M and N must be multiples of 128");
  if ((db && !(keep & TG_KEEP_A)) || (da && !(keep & TG_KEEP_B)))
    return einval("linear_bwd_kept: the operand of a wanted gradient was not kept");
  if (M == 0 || N == 0) return zero_grads(da, da_dtype, db, db_dtype, M, N, K, as_stream(stream));
  if (!da && !db) return TG_OK;
  if (!kept || !g || !workspace) return einval("linear_bwd_kept: null pointer");
  if (workspace_bytes < tg_linear_bwd_kept_workspace(M, N)) return einval("linear_bwd_kept: workspace too small");
  // g.T alone (dW) may be read from any element
  if (!(da ? aligned(g, 16) : aligned_as(g, g_dtype)) || !aligned(workspace, 256) || !aligned(kept, 256))
    return einval("linear_bwd_kept: g must be 16-byte and the buffers 256-byte aligned");
  hipStream_t st = as_stream(stream);
  uint8_t* p = reinterpret_cast<uint8_t*>(workspace);
  uint8_t* k = reinterpret_cast<uint8_t*>(const_cast<void*>(kept));
  FpOperand qat, qb;
  if (keep & TG_KEEP_A) qat = carve(k, K, M);
  if (keep & TG_KEEP_B) qb = carve(k, K, N);
  const FpOperand qg = carve(p, M, N), qgt = carve(p, N, M);
  const QuantTensor t{g, g_dtype, M, N, g_part(da, db), qg.q, qg.s, qgt.q, qgt.s};
  TG_TRY(launch_quant_tensors(&t, 1, true, st));
  if (da) TG_TRY(launch_gemm_fp8(qg.q, qg.s, qb.q, qb.s, 1, da, grad_dtype(da_dtype), M, K, N, st, true));
  if (db) TG_TRY(launch_gemm_fp8(qat.q, qat.s, qgt.q, qgt.s, 1, db, grad_dtype(db_dtype), K, N, M, st, true));
  return TG_OK;
}

extern "C" size_t tg_linear_bwd_workspace(int64_t M, int64_t N, int64_t K) {
  if (M < 0 || N < 0 || K < 0) return 0;
  const int64_t mp = round128(M), np = round128(N);
  return operand_bytes(M, np) + operand_bytes(K, np) + operand_bytes(K, mp) + operand_bytes(N, mp);
}

extern "C" int tg_linear_bwd(const void* a, int a_dtype, const void* b, int b_dtype, const void* g, int g_dtype,
                             void* da, void* db, int64_t M, int64_t N, int64_t K, void* workspace,
                             size_t workspace_bytes, void* stream) {
  TG_TRY(check_gemm_args("linear_bwd", M, N, K, 128, 1));
  if (!valid_dtype(a_dtype) || !valid_dtype(b_dtype) || !valid_dtype(g_dtype))
    return einval("linear_bwd: operands must be bf16 or f32");
  if (M == 0 || N == 0) return zero_grads(da, a_dtype, db, b_dtype, M, N, K, as_stream(stream));
  if (!da && !db) return TG_OK;
  if (!a || !b || !g || !workspace) return einval("linear_bwd: null pointer");
  if (workspace_bytes < tg_linear_bwd_workspace(M, N, K)) return einval("linear_bwd: workspace too small");
  if (!aligned_as(a, a_dtype) || !aligned_as(b, b_dtype) || !aligned_as(g, g_dtype) || !aligned(workspace, 256))
    return einval("linear_bwd: operands must be aligned to their element and the workspace to 256 bytes");
  hipStream_t st = as_stream(stream);
  const int64_t mp = round128(M), np = round128(N);
  uint8_t* p = reinterpret_cast<uint8_t*>(workspace);
  const FpOperand qg = carve(p, M, np), qb = carve(p, K, np), qat = carve(p, K, mp), qgt = carve(p, N, mp);
  QuantTensor t[3];
  int n = 0;
  t[n++] = QuantTensor{g, g_dtype, M, N, g_part(da, db), qg.q, qg.s, qgt.q, qgt.s};
  if (da) t[n++] = QuantTensor{b, b_dtype, K, N, 1, qb.q, qb.s, nullptr, nullptr};       // b along N
  if (db) t[n++] = QuantTensor{a, a_dtype, M, K, 2, nullptr, nullptr, qat.q, qat.s};     // a.T along M
  TG_TRY(launch_quant_tensors(t, n, true, st));
  if (da) TG_TRY(launch_gemm_fp8(qg.q, qg.s, qb.q, qb.s, 1, da, grad_dtype(a_dtype), M, K, np, st, true));
  if (db) TG_TRY(launch_gemm_fp8(qat.q, qat.s, qgt.q, qgt.s, 1, db, grad_dtype(b_dtype), K, N, mp, st, true));
  return TG_OK;
}
