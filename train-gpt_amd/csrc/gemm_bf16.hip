// bf16 GEMM ("NT": both operands K-contiguous, fp32 accumulation, bf16 out)
// and the straight-through backward of block_scaled_matmul built on it.
//
// The reference's backward (/root/reference/fp8.py:85-98) ignores the FP8
// forward and differentiates the plain product in bf16:
//   da = bf16(g) @ bf16(b).T      -> (M, K)      fp8.py:95
//   db = bf16(a).T @ bf16(g)      -> (K, N)      fp8.py:96
// Both dots take bf16 operands, accumulate in fp32 and round once to bf16.
//
// Design (gfx950, wave64):
//   * v_mfma_f32_16x16x32_bf16, accumulating in place: no per-block scales,
//     so the K loop is MFMA work only.
//   * Workgroup tile 256 x 256, 8 waves as 4 (M) x 2 (N), wave tile 64 x 128
//     = 4 x 8 MFMA tiles, 128 fp32 accumulators per lane; 256 x 192 (wave tile
//     64 x 96) where 256-wide tiles would leave more CUs idle (q4_split_of).
//     Four waves of 128 x 128 read a third less LDS per product but are no
//     faster (0.59 against 0.58 us per slice): one wave per SIMD has nothing
//     to run at a wait, and 256 accumulators fill the accumulation registers.
//   * Operands travel HBM -> LDS by buffer_load ... lds through a ring of four
//     K32 stages (one barrier per stage), issued by one wave per SIMD.
//   * dW contracts over the token axis, which is the row axis of both a and
//     g: the contraction-major kernel reads them in place (g from its packed
//     copy where its rows are not 16-byte aligned); only an f32 or unaligned
//     a has a.T and g.T packed for the NT kernel.
//   * Outputs with few tiles split the contraction over workgroups (q4_split_of).
#include "tg_device.h"
#include "tg_host.h"
#include "gemm_tile.h"

namespace tg {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ v4f mfma_bf16_16x16x32(const uint4& a, const uint4& b, const v4f& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a),
                                                 __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// Four-stage pipeline.  A stage is one K32 slice of the workgroup tile: 256
// rows x 64 B of A and of B (192 of B for the narrow tile), 32 KiB; four stages
// ring through 128 KiB of LDS, so three slices (96 KiB per CU) are in flight
// while one is computed.  (With
// two stages of K64, one 64 KiB step in flight, the copy stream was capped by
// the ~1.4 us round trip to L2 / Infinity Cache at ~45 B/ns per CU; the MFMAs
// consume a K64 step in ~0.9 us.)
//   step s: loader waves wait for their copies of slice s (vmcnt(16), narrow
//           14: the copies of slices s+1 and s+2 stay outstanding); barrier
//           (slice s complete, slice s-1 read by every wave); the loader waves
//           issue slice s+3 into slice s-1's stage; every wave computes s.
// Loads: waves 0-3 (one per SIMD) issue all copies, 8 (narrow: 7) per slice
// (a quarter of the rows of A and of B), so the other wave of each SIMD never
// stalls at a DMA issue; loader and compute waves run separate copies of the loop.  The
// copies are issued unconditionally: past the last slice the offset is out of
// range and the loads read zero, which keeps the vmcnt arithmetic exact.  The
// main loop runs whole rounds of four slices with no exit inside (with exits,
// the compiler's wait analysis merges paths at the loop header and drains
// every outstanding copy there).  The barrier is a bare s_barrier (a fence
// would wait for every outstanding copy).
// LDS rows are 64 B, 16-byte chunk c of row r at c ^ ((r >> 1) & 3): the
// fragment reads (16 rows x 4 chunks per instruction) then run without bank
// conflicts on gfx950 (measured: c ^ ((r >> 2) & 3) doubled every read's
// LDS cycles).  Tiles are computed as
// B . A^T so that a lane holds one output row and four consecutive columns
// (8-byte bf16 pieces for the epilogue).
// ---------------------------------------------------------------------------
__shared__ __attribute__((aligned(16))) uint8_t q4_a0[256 * 64];
__shared__ __attribute__((aligned(16))) uint8_t q4_b0[256 * 64];
__shared__ __attribute__((aligned(16))) uint8_t q4_a1[256 * 64];
__shared__ __attribute__((aligned(16))) uint8_t q4_b1[256 * 64];
__shared__ __attribute__((aligned(16))) uint8_t q4_a2[256 * 64];
__shared__ __attribute__((aligned(16))) uint8_t q4_b2[256 * 64];
__shared__ __attribute__((aligned(16))) uint8_t q4_a3[256 * 64];
__shared__ __attribute__((aligned(16))) uint8_t q4_b3[256 * 64];

template <int S> __device__ __forceinline__ uint8_t* q4_a() {
  return S == 0 ? q4_a0 : S == 1 ? q4_a1 : S == 2 ? q4_a2 : q4_a3;
}
template <int S> __device__ __forceinline__ uint8_t* q4_b() {
  return S == 0 ? q4_b0 : S == 1 ? q4_b1 : S == 2 ? q4_b2 : q4_b3;
}

struct Q4Ctx {
  __amdgpu_buffer_rsrc_t ra, rb;
  uint32_t voa, vob;       // NT: loader lane's byte offsets of slice 0, part 0
  uint32_t row16;          // NT: 16 rows in bytes
  int wave, nks;
  uint32_t fa, fb;         // NT: LDS byte offsets of this lane's fragment chunk (tile 0)
  // TN (operands contraction-major, see gemm_bf16_tn_q4_kernel)
  uint32_t voa4[4], vob4[4];   // loader lane's byte offsets of slice 0, part p
  uint32_t sla, slb;           // bytes of one 32-row slice of A and of B
  uint32_t tro[2];             // LDS byte offset of the row of this lane's transpose read h
  uint32_t trx[2];             // chunk XOR of that row
  uint32_t tca, tcb, tin;      // logical chunk of this lane's columns in subtile 0 of A / B, byte within it
};

// TN stage layout: 32 contraction rows of 512 bytes (the tile's 256 output
// indices); 16-byte chunk c of row r sits at chunk c ^ tn_swz(r).  The XOR
// moves whole 32-byte pieces (a transposed fragment read's 4 lanes of one row)
// and differs over the 8 rows that 32 lanes of one read touch.
__device__ __forceinline__ uint32_t tn_swz(uint32_t r) { return ((r & 3u) | (((r >> 3) & 1u) << 2)) << 1; }

// slice ks into the stage at (la, lb).  NT: loader wave w fills rows
// 64w .. 64w+63 of A and its quarter of B's 32 NJ rows, 16 rows per instruction;
// TN: contraction rows 8w .. 8w+7, 2 rows per instruction.
template <bool LOADER, bool TN, int NJ>
__device__ __forceinline__ void q4_issue(const Q4Ctx& c, uint8_t* la, uint8_t* lb, int ks) {
  if (!LOADER) return;
  if constexpr (TN) {
    const bool in = ks < c.nks;
    const uint32_t soa = in ? (uint32_t)ks * c.sla : 0x80000000u;   // out of range: zeros
    const uint32_t sob = in ? (uint32_t)ks * c.slb : 0x80000000u;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(c.ra, la + c.wave * 4096 + p * 1024, 16, c.voa4[p], soa, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(c.rb, lb + c.wave * 4096 + p * 1024, 16, c.vob4[p], sob, 0, 0);
    }
  } else {
    const uint32_t so = ks < c.nks ? (uint32_t)ks * 64u : 0x80000000u;   // out of range: zeros
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(c.ra, la + c.wave * 4096 + p * 1024, 16, c.voa,
                                               so + p * c.row16, 0, 0);
      if (p < NJ / 2)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(c.rb, lb + c.wave * (NJ * 512) + p * 1024, 16, c.vob,
                                                 so + p * c.row16, 0, 0);
    }
  }
}

typedef short v4s_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s_t lds_v4s_t;

// TN fragment of subtile t (16 output indices at column chunk base cb + 2t):
// lane (fr, fg) gets contraction rows 8 fg .. 8 fg + 7 of output index
// (subtile start) + fr, as the NT fragment holds them, from two transposed
// reads (ds_read_b64_tr_b16: in each 16-lane group, lane i receives element
// i % 4 of the 8-byte pieces lanes 4j + i / 4 read, j = 0..3); lane 4j + q
// of a group reads row 8 fg + j (+4) at columns 4q .. 4q+3 of the subtile.
__device__ __forceinline__ uint4 tn_frag(const uint8_t* l, const Q4Ctx& c, uint32_t cb, int t) {
  const uint32_t ch = cb + 2u * (uint32_t)t;
  const v4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_v4s_t*)(l + c.tro[0] + ((ch ^ c.trx[0]) << 4) + c.tin));
  const v4s_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_v4s_t*)(l + c.tro[1] + ((ch ^ c.trx[1]) << 4) + c.tin));
  return make_uint4(((uint32_t)(uint16_t)lo[0]) | ((uint32_t)(uint16_t)lo[1] << 16),
                    ((uint32_t)(uint16_t)lo[2]) | ((uint32_t)(uint16_t)lo[3] << 16),
                    ((uint32_t)(uint16_t)hi[0]) | ((uint32_t)(uint16_t)hi[1] << 16),
                    ((uint32_t)(uint16_t)hi[2]) | ((uint32_t)(uint16_t)hi[3] << 16));
}

// s_waitcnt vmcnt(n) lgkmcnt(0), and lgkmcnt(0) alone, as the builtin (gfx9
// encoding: vmcnt bits 3:0 and 15:14, expcnt not waited), which the compiler's
// own wait insertion takes into account; an inline-asm wait is opaque to it.
// lgkmcnt: a wave's reads of slice ks - 1 have left LDS before a loader, past
// the barrier, refills that stage (the refills past the last slice return their
// zeros at once, without a trip to memory).
constexpr int wait_vm(int n) { return (n & 15) | ((n >> 4) << 14) | (0x7 << 4); }
constexpr int kWaitLds = (3 << 14) | (0x7 << 4) | 0xF;

template <int S, bool LOADER, bool TN, int NJ>
__device__ __forceinline__ void q4_step(const Q4Ctx& c, int ks, v4f (&acc)[4][NJ]) {
  constexpr int kCopies = 4 + NJ / 2;    // a loader wave's per slice
  __builtin_amdgcn_s_waitcnt(LOADER ? wait_vm(2 * kCopies) : kWaitLds);
  __builtin_amdgcn_s_barrier();
  constexpr int kRefill = (S + 3) & 3;   // the stage slice ks - 1 occupied
  q4_issue<LOADER, TN, NJ>(c, q4_a<kRefill>(), q4_b<kRefill>(), ks + 3);
  const uint8_t* la = q4_a<S>();
  const uint8_t* lb = q4_b<S>();
  uint4 af[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    af[i] = TN ? tn_frag(la, c, c.tca, i) : *reinterpret_cast<const uint4*>(la + c.fa + i * 1024);
  uint4 bn = TN ? tn_frag(lb, c, c.tcb, 0) : *reinterpret_cast<const uint4*>(lb + c.fb);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const uint4 bf = bn;
    if (j + 1 < NJ)
      bn = TN ? tn_frag(lb, c, c.tcb, j + 1) : *reinterpret_cast<const uint4*>(lb + c.fb + (j + 1) * 1024);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i][j] = mfma_bf16_16x16x32(bf, af[i], acc[i][j]);
  }
}

template <bool LOADER, bool TN, int NJ>
__device__ __forceinline__ void q4_main_loop(const Q4Ctx& c, v4f (&acc)[4][NJ]) {
  q4_issue<LOADER, TN, NJ>(c, q4_a0, q4_b0, 0);
  q4_issue<LOADER, TN, NJ>(c, q4_a1, q4_b1, 1);
  q4_issue<LOADER, TN, NJ>(c, q4_a2, q4_b2, 2);
  int ks = 0;
  for (; ks + 4 <= c.nks; ks += 4) {
    q4_step<0, LOADER, TN, NJ>(c, ks, acc);
    q4_step<1, LOADER, TN, NJ>(c, ks + 1, acc);
    q4_step<2, LOADER, TN, NJ>(c, ks + 2, acc);
    q4_step<3, LOADER, TN, NJ>(c, ks + 3, acc);
  }
  if (ks < c.nks) {
    q4_step<0, LOADER, TN, NJ>(c, ks, acc);
    if (ks + 1 < c.nks) {
      q4_step<1, LOADER, TN, NJ>(c, ks + 1, acc);
      if (ks + 2 < c.nks) q4_step<2, LOADER, TN, NJ>(c, ks + 2, acc);
    }
  }
}

// R rows of cnt <= 128 bf16 from LDS (256-byte rows, chunk c of row r at c ^
// (r & 15)) to C rows mw + r from column nw on, where they start at any even
// address, by one wave; r0 (a multiple of 16) is the first row.  LW lanes to a
// row: consecutive 4-byte words from its first 4-byte boundary, and a single
// value at either end where one is left over; a lane without a value stores
// past its descriptor's end, which is dropped, so no branch is taken.  Eight
// instructions' words are read from LDS before the first is stored, in a loop
// that is not unrolled: code that runs once waits for its own fetch.
template <int R, int LW>
__device__ __forceinline__ void q4_store_odd_rows(const uint8_t* l, __bf16* __restrict__ C, int M, int N, int mw,
                                                  int nw, int cnt, int lane, int r0) {
  constexpr int RPI = 64 / LW, IT = R / RPI, B = IT < 8 ? IT : 8;   // rows per instruction; instructions; a batch
  constexpr uint32_t kDrop = 0xFFFFFFF0u;
  const int sub = LW == 64 ? 0 : lane / LW, w = lane % LW, w1 = min(w + 1, 63);
  auto word = [&](int r, int i) {
    return *reinterpret_cast<const uint32_t*>(l + r * 256 + (((i >> 2) ^ (r & 15)) * 16) + (i & 3) * 4);
  };
#pragma unroll 1
  for (int i0 = 0; i0 < IT; i0 += B) {
    const int mb = __builtin_amdgcn_readfirstlane(mw + r0 + i0 * RPI), nb = __builtin_amdgcn_readfirstlane(nw);
    if (mb >= M) break;
    const int nrow = min(M - mb, B * RPI);
    const uint8_t* first = reinterpret_cast<const uint8_t*>(C + (int64_t)mb * N + nb);
    const uint32_t base = (uint32_t)(reinterpret_cast<uintptr_t>(first) & 3u);   // 0 or 2
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(first - base, (uint32_t)(((nrow - 1) * (int64_t)N + cnt) * 2) + base);
    const bool singles = (N & 1) || base;   // else every row starts on a word and holds whole words
    uint32_t own[B], next[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int r = r0 + (i0 + u) * RPI + sub;
      own[u] = word(r, w);
      next[u] = word(r, w1);
    }
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int r = u * RPI + sub, o = (int)((base >> 1) + (uint32_t)(r & N)) & 1, n = (cnt - o) >> 1;
      const uint32_t row = base + (uint32_t)r * (uint32_t)N * 2u, off = row + 2u * o + 4u * w;
      const uint32_t v = o ? __builtin_amdgcn_alignbit(next[u], own[u], 16) : own[u];
      const bool in = r < nrow;
      __builtin_amdgcn_raw_buffer_store_b32(v, rc, in && w < n ? off : kDrop, 0, 0);
      const bool tail = in && w == n && ((cnt - o) & 1), head = in && o && w == 0;
      if (singles && LW == 8) {   // one lane may have both (two values in all)
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)v, rc, tail ? off : kDrop, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)own[u], rc, head ? row : kDrop, 0, 0);
      } else if (singles) {
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(head ? own[u] : v), rc, head ? row : tail ? off : kDrop, 0, 0);
      }
    }
  }
}

// The same for columns nw .. nw + W - 1 (W = 16 NJ, those below N) of any C.  Rows of
// N % 8 == 0 go out as 16-byte pieces, W / 8 lanes per row; others as above
// (2-byte stores of whole pieces touched every line eight times).
template <int R, int NJ>
__device__ __forceinline__ void q4_store_rows(const uint8_t* l, __bf16* __restrict__ C, int M, int N, int mw, int nw,
                                              int lane, int r0) {
  constexpr int PITCH = 256, kRow = 2 * NJ;   // 16-byte pieces per row
  if (N % 8 == 0) {
#pragma unroll
    for (int q = 0; q < R * kRow / 64; ++q) {
      const int o = q * 64 + lane;
      const int r = r0 + o / kRow, k = o % kRow;
      const int m = mw + r, n = nw + k * 8;
      const uint4 v = *reinterpret_cast<const uint4*>(l + r * PITCH + ((k ^ (r & 15)) * 16));
      if (m < M && n < N) *reinterpret_cast<uint4*>(C + (int64_t)m * N + n) = v;
    }
    return;
  }
  const int cnt = min(16 * NJ, N - nw);
  if (cnt <= 0) return;
  if (cnt <= 16) q4_store_odd_rows<R, 8>(l, C, M, N, mw, nw, cnt, lane, r0);
  else if (cnt <= 32) q4_store_odd_rows<R, 16>(l, C, M, N, mw, nw, cnt, lane, r0);
  else if (cnt <= 64) q4_store_odd_rows<R, 32>(l, C, M, N, mw, nw, cnt, lane, r0);
  else q4_store_odd_rows<R, 64>(l, C, M, N, mw, nw, cnt, lane, r0);
}

// Epilogue: lane (fr, fg) holds row i * 16 + fr and columns j * 16 + 4 fg .. +3
// of the wave tile; stage it in this wave's 16 KiB (256-byte rows, chunk c of
// row r at c ^ (r & 15)), then store whole rows.
template <int NJ>
__device__ __forceinline__ void q4_store_tile(const v4f (&acc)[4][NJ], __bf16* __restrict__ C, int M, int N, int m0,
                                              int n0, int wm, int wn, int wave, int lane) {
  const int fr = lane & 15, fg = lane >> 4;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  uint8_t* wbuf = wave == 0 ? q4_a0 : wave == 1 ? q4_b0 : wave == 2 ? q4_a1 : wave == 3 ? q4_b1
                : wave == 4 ? q4_a2 : wave == 5 ? q4_b2 : wave == 6 ? q4_a3 : q4_b3;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int r = i * 16 + fr;
      const int chunk = (j * 2 + (fg >> 1)) ^ (r & 15);
      const v4f v = acc[i][j];
      *reinterpret_cast<uint2*>(wbuf + r * 256 + chunk * 16 + (fg & 1) * 8) =
          make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  // odd rows are one instruction each or more: waves without values take a share
  // of the others' rows
  if (N % 8 && (M - m0 <= 64 || N - n0 <= 16 * NJ)) {
    __syncthreads();
    if (M - m0 <= 64)   // waves 0 and 1 hold every row: a quarter each (33 x 50257 over 128: 10.8 -> 9.4 us)
      q4_store_rows<16, NJ>(wn ? q4_b0 : q4_a0, C, M, N, m0, n0 + wn * (16 * NJ), lane, 16 * wm);
    else                // the left waves hold every column: half of the rows each (4500 x 75 over 192: 14.7 -> 11.0 us)
      q4_store_rows<32, NJ>(wm == 0 ? q4_a0 : wm == 1 ? q4_a1 : wm == 2 ? q4_a2 : q4_a3, C, M, N, m0 + wm * 64, n0, lane,
                            32 * wn);
    return;
  }
  q4_store_rows<64, NJ>(wbuf, C, M, N, m0 + wm * 64, n0 + wn * (16 * NJ), lane, 0);
}

// Split-K: the workgroup's f32 tile in register order, one contiguous 8 KiB
// per (i, j), for q4_reduce_kernel.  The copies issued past the last slice
// still write LDS, so they are waited for before the wave ends.
template <int NJ>
__device__ __forceinline__ void q4_store_part(const v4f (&acc)[4][NJ], float* __restrict__ part) {
  float4* p = reinterpret_cast<float4*>(part) + (size_t)blockIdx.x * (4 * NJ * 512) + threadIdx.x;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      p[(i * NJ + j) * 512] = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Sum of the splits' partial tiles in split order, rounded once to bf16.  One
// workgroup per wave tile (8 per workgroup tile): wave i sums the
// fragments of rows 16 i .. +15 as the GEMM's lanes held them, and the bf16
// rows leave through LDS as whole pieces.
template <int NJ>
__global__ __launch_bounds__(256) void q4_reduce_kernel(const float4* __restrict__ part, __bf16* __restrict__ C,
                                                        int M, int N, int tiles_m, int tiles_n, int nsplit) {
  __shared__ __attribute__((aligned(16))) uint8_t rows[64 * 256];
  const int tile = blockIdx.x >> 3, w = blockIdx.x & 7;
  int tmi, tni;
  tile_of(tile, tiles_m, tiles_n, tmi, tni);
  const int mw = tmi * 256 + (w >> 1) * 64, nw = tni * (32 * NJ) + (w & 1) * (16 * NJ);
  if (mw >= M || nw >= N) return;
  const int lane = threadIdx.x & 63, i = threadIdx.x >> 6, fr = lane & 15, fg = lane >> 4;
  const size_t ntiles = (size_t)tiles_m * tiles_n;
  const float4* p = part + ((size_t)tile * (4 * NJ) + i * NJ) * 512 + w * 64 + lane;
  float4 t[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) t[j] = p[j * 512];
  for (int s = 1; s < nsplit; ++s) {
    p += ntiles * (4 * NJ * 512);
    float4 v[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) v[j] = p[j * 512];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      t[j].x += v[j].x; t[j].y += v[j].y; t[j].z += v[j].z; t[j].w += v[j].w;
    }
  }
  const int r = i * 16 + fr;
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    *reinterpret_cast<uint2*>(rows + r * 256 + (((j * 2 + (fg >> 1)) ^ (r & 15)) * 16) + (fg & 1) * 8) =
        make_uint2(pack_bf16x2(t[j].x, t[j].y), pack_bf16x2(t[j].z, t[j].w));
  __syncthreads();
  q4_store_rows<16, NJ>(rows, C, M, N, mw, nw, lane, 16 * i);
}

// The K slices of this workgroup's split: first slice and count (per slices
// each, the last split takes what is left), and the tile slot within it.
__device__ __forceinline__ int q4_split(int nks, int tiles_m, int tiles_n, int nsplit, int per, int& ks0, int& cnt) {
  const int ntiles = tiles_m * tiles_n;
  const int sp = nsplit > 1 ? (int)blockIdx.x / ntiles : 0;
  ks0 = sp * per;
  cnt = (sp == nsplit - 1 ? nks : ks0 + per) - ks0;
  return (int)blockIdx.x - sp * ntiles;
}

template <int NJ>
__global__ __launch_bounds__(512, 1) void gemm_bf16_nt_q4_kernel(const __bf16* __restrict__ A,
                                                                 const __bf16* __restrict__ B,
                                                                 __bf16* __restrict__ C, int M, int N,
                                                                 int K, int tiles_m, int tiles_n, int nsplit,
                                                                 int per, float* __restrict__ part) {
  Q4Ctx c;
  const int tid = threadIdx.x, lane = tid & 63;
  c.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int ks0;
  const int slot = q4_split(K >> 5, tiles_m, tiles_n, nsplit, per, ks0, c.nks);
  const int fr = lane & 15, fg = lane >> 4;
  const int wm = c.wave >> 1, wn = c.wave & 1;
  int tmi, tni;
  tile_of(slot, tiles_m, tiles_n, tmi, tni);
  const int m0 = tmi * 256, n0 = tni * (32 * NJ);
  const uint32_t rowb = 2u * (uint32_t)K;
  c.ra = make_rsrc(A, (uint32_t)M * rowb);
  c.rb = make_rsrc(B, (uint32_t)N * rowb);
  c.row16 = 16u * rowb;
  // DMA lane L lands at byte 16 L of its 1 KiB slot: row slot + L / 4,
  // physical chunk L % 4, which holds logical chunk (L % 4) ^ ((L >> 3) & 3)
  const int lrow = lane >> 2;   // loader waves 0-3
  const uint32_t lch = (uint32_t)((lane & 3) ^ ((lane >> 3) & 3)) * 16u;
  c.voa = (uint32_t)(m0 + c.wave * 64 + lrow) * rowb + lch + (uint32_t)ks0 * 64u;
  c.vob = (uint32_t)(n0 + c.wave * (8 * NJ) + lrow) * rowb + lch + (uint32_t)ks0 * 64u;
  // fragment: lane (fr, fg) reads logical chunk fg (k 8fg .. 8fg+7) of row
  // (wave tile row) + 16 t + fr, at physical chunk fg ^ ((fr >> 1) & 3)
  const uint32_t ch = (uint32_t)(fg ^ ((fr >> 1) & 3)) * 16u;
  c.fa = (uint32_t)(wm * 64 + fr) * 64u + ch;
  c.fb = (uint32_t)(wn * (16 * NJ) + fr) * 64u + ch;

  v4f acc[4][NJ];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  if (c.wave < 4) q4_main_loop<true, false, NJ>(c, acc);
  else q4_main_loop<false, false, NJ>(c, acc);

  if (nsplit > 1) q4_store_part(acc, part);
  else q4_store_tile(acc, C, M, N, m0, n0, wm, wn, c.wave, lane);
}

// C (M, N) = A^T B on contraction-major operands: A (Kc, M) and B (Kc, N)
// row-major with row pitches lda and ldb elements, C[m][n] = sum_c A[c][m] B[c][n].
// This is the straight-through backward's db = a.T @ g (fp8.py:96) read
// straight from a and g, with no transposed copies.  The pipeline, tiles and
// epilogue are the NT kernel's; a stage holds 32 contraction rows of the
// tile's 256 m (A) or n (B) indices, 512 bytes each (stored with tn_swz), and
// the MFMA fragments come from transposed LDS reads (tn_frag).  Contraction
// rows past Kc read zero; tile columns past M or N read neighbouring memory
// that only reaches discarded outputs.
__global__ __launch_bounds__(512, 1) void gemm_bf16_tn_q4_kernel(const __bf16* __restrict__ A,
                                                                 const __bf16* __restrict__ B,
                                                                 __bf16* __restrict__ C, int M, int N, int Kc,
                                                                 int lda, int ldb, int tiles_m, int tiles_n,
                                                                 int nsplit, int per, float* __restrict__ part) {
  Q4Ctx c;
  const int tid = threadIdx.x, lane = tid & 63;
  c.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int ks0;
  const int slot = q4_split((Kc + 31) >> 5, tiles_m, tiles_n, nsplit, per, ks0, c.nks);
  const int fr = lane & 15, fg = lane >> 4;
  const int wm = c.wave >> 1, wn = c.wave & 1;
  int tmi, tni;
  tile_of(slot, tiles_m, tiles_n, tmi, tni);
  const int m0 = tmi * 256, n0 = tni * 256;
  const uint32_t pa = 2u * (uint32_t)lda, pb = 2u * (uint32_t)ldb;
  c.ra = make_rsrc(A, (uint32_t)Kc * pa);
  c.rb = make_rsrc(B, (uint32_t)Kc * pb);
  c.sla = 32u * pa;
  c.slb = 32u * pb;
  // DMA: instruction p of loader wave w fills slice rows r = 8w + 2p + L / 32;
  // lane L lands at physical chunk L % 32 of row r, which holds logical chunk
  // (L % 32) ^ tn_swz(r)
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const uint32_t r = (uint32_t)(8 * c.wave + 2 * p + (lane >> 5));
    const uint32_t lc = (uint32_t)(lane & 31) ^ tn_swz(r);
    c.voa4[p] = ((uint32_t)ks0 * 32u + r) * pa + (uint32_t)m0 * 2u + lc * 16u;
    c.vob4[p] = ((uint32_t)ks0 * 32u + r) * pb + (uint32_t)n0 * 2u + lc * 16u;
  }
  // transposed reads: lane (fr, fg) reads row 8 fg + fr / 4 (+ 4) at columns
  // 4 (fr % 4) .. +3 of a subtile: chunk (fr % 4) / 2 of it, byte 8 (fr % 2)
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t r = (uint32_t)(8 * fg + 4 * h + (fr >> 2));
    c.tro[h] = r * 512u;
    c.trx[h] = tn_swz(r);
  }
  c.tca = (uint32_t)(wm * 8 + ((fr & 3) >> 1));
  c.tcb = (uint32_t)(wn * 16 + ((fr & 3) >> 1));
  c.tin = 8u * (uint32_t)(fr & 1);

  v4f acc[4][8];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  if (c.wave < 4) q4_main_loop<true, true, 8>(c, acc);
  else q4_main_loop<false, true, 8>(c, acc);

  if (nsplit > 1) q4_store_part(acc, part);
  else q4_store_tile(acc, C, M, N, m0, n0, wm, wn, c.wave, lane);
}

// ---------------------------------------------------------------------------
// Packing: y = bf16(x) (RNE for f32 input), optionally transposed, with every
// output row padded with zeros to `pitch` elements.
//   transpose = 0: x (rows, cols) -> y (rows, pitch),  pitch >= cols
//   transpose = 1: x (rows, cols) -> y (cols, pitch),  pitch >= rows
// A 64 x 64 tile goes through LDS so that both the reads and the writes are
// row-contiguous; the LDS tile has one padding element per row.
// ---------------------------------------------------------------------------
template <bool F32_IN, bool TRANSPOSE>
__global__ __launch_bounds__(256) void pack_bf16_kernel(const void* __restrict__ xv,
                                                        __bf16* __restrict__ y, int rows, int cols,
                                                        int pitch) {
  __shared__ uint16_t tile[64][65];
  const int tid = threadIdx.x;
  // tile origin in x coordinates
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  // read 64 x 64 of x: thread covers column c0 + (tid & 63), rows (tid >> 6) + 4t
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int rr = (tid >> 6) + 4 * t, cc = tid & 63;
    const int r = r0 + rr, col = c0 + cc;
    uint16_t v = 0;
    if (r < rows && col < cols) {
      if (F32_IN) {
        const float f = reinterpret_cast<const float*>(xv)[(int64_t)r * cols + col];
        v = __builtin_bit_cast(uint16_t, (__bf16)f);
      } else {
        v = reinterpret_cast<const uint16_t*>(xv)[(int64_t)r * cols + col];
      }
    }
    if (TRANSPOSE) tile[cc][rr] = v; else tile[rr][cc] = v;
  }
  __syncthreads();
  // write: output row (tile row) ty, output column tx; outputs past the
  // data but inside the pitch are the zero padding read above
  const int out_rows = TRANSPOSE ? cols : rows;
  const int or0 = TRANSPOSE ? c0 : r0, oc0 = TRANSPOSE ? r0 : c0;
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int ty = (tid >> 6) + 4 * t, tx = tid & 63;
    const int orow = or0 + ty, ocol = oc0 + tx;
    if (orow < out_rows && ocol < pitch)
      reinterpret_cast<uint16_t*>(y)[(int64_t)orow * pitch + ocol] = tile[ty][tx];
  }
}

// 8 consecutive bf16 at any even byte offset of a buffer: the 20 bytes from the
// 4-byte boundary at or before it (raw buffer loads need no more than 4-byte
// alignment, and what lies past the buffer reads zero), shifted into place.
struct U8Load {
  u32x4_t v;
  uint32_t w;
};
__device__ __forceinline__ U8Load u8_load(const __amdgpu_buffer_rsrc_t& r, uint32_t off) {
  const uint32_t o = off & ~3u;
  return U8Load{__builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0), __builtin_amdgcn_raw_buffer_load_b32(r, o + 16u, 0, 0)};
}
__device__ __forceinline__ uint4 u8_value(const U8Load& l, uint32_t off) {
  const uint32_t sh = (off & 2u) * 8u;   // 0 or 16 bits
  return make_uint4(__builtin_amdgcn_alignbit(l.v.y, l.v.x, sh), __builtin_amdgcn_alignbit(l.v.z, l.v.y, sh),
                    __builtin_amdgcn_alignbit(l.v.w, l.v.z, sh), __builtin_amdgcn_alignbit(l.w, l.v.w, sh));
}
// The first `n` of the 8 values, zeros after them.
__device__ __forceinline__ uint4 u8_first(const uint4& v, int64_t n) {
  uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] &= n >= 2 * i + 2 ? 0xFFFFFFFFu : n == 2 * i + 1 ? 0xFFFFu : 0u;
  return make_uint4(w[0], w[1], w[2], w[3]);
}
// Descriptor of bytes [x, x + bytes) from the 4-byte boundary at or before x,
// and x's offset in it (0 or 2).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t u8_rsrc(const void* x, uint64_t bytes, uint32_t& base) {
  base = (uint32_t)(reinterpret_cast<uintptr_t>(x) & 3u);
  return make_rsrc(reinterpret_cast<const uint8_t*>(x) - base, (uint32_t)((bytes + base + 3u) & ~3ull));
}

// Row copy of bf16 rows at any even address to rows of `pitch` elements, zeros
// past the row (pitch % 8 == 0, y 16-byte aligned): each thread four 16-byte
// pieces of one output row, 256 pieces apart.  HBM-bound (2 bytes read, 2
// written per element): with the 64 x 64 tiles of 2-byte accesses above,
// 2048 x 50257 took 162 us (2.5 TB/s).
constexpr int kRowPieces = 4;
__global__ __launch_bounds__(256) void pack_bf16_rows_kernel(const uint16_t* __restrict__ x,
                                                             uint16_t* __restrict__ y, int rows, int cols,
                                                             int pitch) {
  uint32_t base;
  const __amdgpu_buffer_rsrc_t rx = u8_rsrc(x, (uint64_t)rows * (uint64_t)cols * 2u, base);
  const int np = pitch >> 3;
  for (int r = blockIdx.y; r < rows; r += gridDim.y) {
    const int p0 = blockIdx.x * (256 * kRowPieces) + threadIdx.x;
    const uint32_t ro = base + (uint32_t)r * (uint32_t)cols * 2u;
    U8Load l[kRowPieces];
#pragma unroll
    for (int u = 0; u < kRowPieces; ++u) l[u] = u8_load(rx, ro + (uint32_t)(p0 + 256 * u) * 16u);
#pragma unroll
    for (int u = 0; u < kRowPieces; ++u) {
      const int p = p0 + 256 * u;
      if (p < np)
        *reinterpret_cast<uint4*>(y + (int64_t)r * pitch + p * 8) = u8_first(u8_value(l[u], ro), (int64_t)cols - 8 * p);
    }
  }
}

// The same for rows narrower than a workgroup's 1024 pieces, over the pieces of
// all rows in turn (one workgroup per row left most of its lanes idle: 7782 x 64
// 11.2 us).
__global__ __launch_bounds__(256) void pack_bf16_flat_kernel(const uint16_t* __restrict__ x,
                                                             uint16_t* __restrict__ y, uint32_t total, int rows,
                                                             int cols, uint32_t np) {
  uint32_t base;
  const __amdgpu_buffer_rsrc_t rx = u8_rsrc(x, (uint64_t)rows * (uint64_t)cols * 2u, base);
  const uint32_t i0 = blockIdx.x * (256 * kRowPieces) + threadIdx.x;
  U8Load l[kRowPieces];
  uint32_t off[kRowPieces], p[kRowPieces];
#pragma unroll
  for (int u = 0; u < kRowPieces; ++u) {
    const uint32_t i = min(i0 + 256 * u, total - 1), r = i / np;
    p[u] = i - r * np;
    off[u] = base + r * (uint32_t)cols * 2u + p[u] * 16u;
    l[u] = u8_load(rx, off[u]);
  }
#pragma unroll
  for (int u = 0; u < kRowPieces; ++u) {
    const uint32_t i = i0 + 256 * u;
    if (i < total)
      *reinterpret_cast<uint4*>(y + (int64_t)i * 8) = u8_first(u8_value(l[u], off[u]), (int64_t)cols - 8 * (int64_t)p[u]);
  }
}

// Transposing pack of bf16 rows (16-byte-aligned ones, or with UA rows at any
// even address, such as an odd vocabulary's): a 128 x 128 tile is loaded with 16-byte row loads into LDS
// (pitch 272 B); lane p of a wave reads the column pair 2p, 2p + 1 one 32-bit
// word per row (conflict-free), the tile is re-staged in LDS as output rows
// (pitch 264 B) and 16 lanes write each output row's 256 bytes, so every store
// instruction covers four whole row segments.  (Writing each lane's 16-byte
// pieces straight out left every output line to be assembled from sixteen
// stores of four waves: 2.4 TB/s instead of 4.5 at 8192 x 50304.)  UA at
// 2304 x 50257: 87 us; the 64 x 64 tiles took 164.  NT: non-
// temporal stores, for outputs larger than the Infinity Cache.
template <bool NT, bool UA>
__global__ __launch_bounds__(256) void pack_bf16_t128_kernel(const uint4* __restrict__ x,
                                                             uint16_t* __restrict__ y, int rows,
                                                             int cols, int pitch) {
  __shared__ uint32_t tile[128 * 68];
  const int tid = threadIdx.x;
  const int r0 = blockIdx.y * 128, c0 = blockIdx.x * 128;
  const int ch = tid & 15, rr = tid >> 4;
  const int cchunks = cols >> 3;
  const bool ch_ok = (c0 >> 3) + ch < cchunks;
  if constexpr (UA) {
    // values past a row's end only reach output rows that are not stored, and
    // rows past the last read zero
    uint32_t base;
    const __amdgpu_buffer_rsrc_t rx = u8_rsrc(x, (uint64_t)rows * (uint64_t)cols * 2u, base);
    U8Load l[8];
    uint32_t off[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      off[u] = base + ((uint32_t)(r0 + rr + 16 * u) * (uint32_t)cols + (uint32_t)(c0 + 8 * ch)) * 2u;
      l[u] = u8_load(rx, off[u]);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      *reinterpret_cast<uint4*>(&tile[(rr + 16 * u) * 68 + ch * 4]) =
          u8_first(u8_value(l[u], off[u]), r0 + rr + 16 * u < rows ? 8 : 0);
  } else {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int r = r0 + rr + 16 * u;
      const uint4 v = (ch_ok && r < rows) ? ldg_stream(x + (int64_t)r * cchunks + (c0 >> 3) + ch)
                                          : make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4*>(&tile[(rr + 16 * u) * 68 + ch * 4]) = v;
    }
  }
  __syncthreads();
  // lane p: input columns 2p, 2p + 1 (output rows), input rows 32g + 8c .. +7
  const int p = tid & 63, g = tid >> 6;
  uint32_t lo[4][4], hi[4][4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int rb = 32 * g + 8 * c;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t w0 = tile[(rb + 2 * e) * 68 + p], w1 = tile[(rb + 2 * e + 1) * 68 + p];
      lo[c][e] = (w0 & 0xFFFFu) | (w1 << 16);
      hi[c][e] = (w0 >> 16) | (w1 & 0xFFFF0000u);
    }
  }
  __syncthreads();   // every lane has read the tile: the same memory stages the output rows
  uint32_t* tq = tile;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int rb = 32 * g + 8 * c;
    *reinterpret_cast<uint4*>(&tq[(2 * p) * 66 + rb / 2]) = make_uint4(lo[c][0], lo[c][1], lo[c][2], lo[c][3]);
    *reinterpret_cast<uint4*>(&tq[(2 * p + 1) * 66 + rb / 2]) = make_uint4(hi[c][0], hi[c][1], hi[c][2], hi[c][3]);
  }
  __syncthreads();
  const int k = tid & 15;            // elements 8k .. 8k+7 of output row n
  const int oc = r0 + 8 * k;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int n = (tid >> 4) + 16 * q;
    if (c0 + n < cols && oc < pitch) {
      const uint4 v = *reinterpret_cast<const uint4*>(&tq[n * 66 + 4 * k]);
      uint4* dst = reinterpret_cast<uint4*>(y + (int64_t)(c0 + n) * pitch + oc);
      if (NT) stg_stream(dst, v);
      else *dst = v;
    }
  }
}

int launch_pack_bf16(const void* x, int x_dtype, int64_t rows, int64_t cols, int transpose,
                     __bf16* y, int64_t pitch, hipStream_t st) {
  if (rows == 0 || cols == 0) return TG_OK;
  // the grid covers the padded extent so the zero padding is written too
  const int64_t ext_r = transpose ? pitch : rows, ext_c = transpose ? cols : pitch;
  const dim3 grid((unsigned)((ext_c + 63) / 64), (unsigned)((ext_r + 63) / 64));
  const int r = (int)rows, c = (int)cols, p = (int)pitch;
  // bf16 to 16-byte-aligned output rows: 16-byte stores, and 16-byte loads at
  // any even address (32-bit buffer offsets, the last tile's overhang included);
  // what is left (f32, an unaligned pitch or output) takes the 64 x 64 tiles
  const bool wide = x_dtype == TG_DTYPE_BF16 && pitch % 8 == 0 && aligned(y, 16) && aligned(x, 2);
  const bool off32 = ((uint64_t)rows + 128) * (uint64_t)cols * 2 + 512 < (1ull << 32);
  const bool in16 = cols % 8 == 0 && aligned(x, 16);
  if (transpose && wide && (in16 || off32)) {
    const dim3 g128((unsigned)((cols + 127) / 128), (unsigned)((pitch + 127) / 128));
    auto X = reinterpret_cast<const uint4*>(x);
    auto Y = reinterpret_cast<uint16_t*>(y);
    const bool nt = (uint64_t)cols * (uint64_t)pitch * 2 > (256ull << 20);   // larger than the Infinity Cache
#define TG_PACK_T128(NT, UA) hipLaunchKernelGGL((pack_bf16_t128_kernel<NT, UA>), g128, dim3(256), 0, st, X, Y, r, c, p)
    if (in16) {
      if (nt) TG_PACK_T128(true, false);
      else TG_PACK_T128(false, false);
    } else {
      if (nt) TG_PACK_T128(true, true);
      else TG_PACK_T128(false, true);
    }
#undef TG_PACK_T128
    return check_launch("pack_bf16_t128");
  }
  if (!transpose && wide && off32 && pitch / 8 < 256 * kRowPieces && rows * (pitch / 8) < 0x7FFFF000) {
    const uint32_t np = (uint32_t)(pitch / 8), total = (uint32_t)rows * np;
    hipLaunchKernelGGL(pack_bf16_flat_kernel, dim3((total + 256 * kRowPieces - 1) / (256 * kRowPieces)), dim3(256), 0, st,
                       reinterpret_cast<const uint16_t*>(x), reinterpret_cast<uint16_t*>(y), total, r, c, np);
    return check_launch("pack_bf16_flat");
  }
  if (!transpose && wide && off32) {
    const dim3 gr((unsigned)((pitch / 8 + 256 * kRowPieces - 1) / (256 * kRowPieces)),
                  (unsigned)(rows < 65535 ? rows : 65535));
    hipLaunchKernelGGL(pack_bf16_rows_kernel, gr, dim3(256), 0, st, reinterpret_cast<const uint16_t*>(x),
                       reinterpret_cast<uint16_t*>(y), r, c, p);
    return check_launch("pack_bf16_rows");
  }
  if (x_dtype == TG_DTYPE_F32) {
    if (transpose) hipLaunchKernelGGL((pack_bf16_kernel<true, true>), grid, dim3(256), 0, st, x, y, r, c, p);
    else hipLaunchKernelGGL((pack_bf16_kernel<true, false>), grid, dim3(256), 0, st, x, y, r, c, p);
  } else {
    if (transpose) hipLaunchKernelGGL((pack_bf16_kernel<false, true>), grid, dim3(256), 0, st, x, y, r, c, p);
    else hipLaunchKernelGGL((pack_bf16_kernel<false, false>), grid, dim3(256), 0, st, x, y, r, c, p);
  }
  return check_launch("pack_bf16");
}

__global__ void fill_zero_u16_kernel(uint16_t* __restrict__ p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0;
}

int launch_fill_zero_bf16(void* p, int64_t n, hipStream_t st) {
  if (n == 0) return TG_OK;
  const int64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(fill_zero_u16_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0,
                     st, reinterpret_cast<uint16_t*>(p), n);
  return check_launch("fill_zero_bf16");
}

// Tile width, and the split of a contraction of nks 32-wide slices over
// workgroups, for outputs whose 256 x 256 tiles leave CUs idle (a head's dX at
// 2048 x 2304: 72 tiles on 256 CUs) or fill a last round badly.
struct Q4Split {
  int n, per;   // splits, slices per split
  int nj;       // tile width / 32: 8 (256 columns) or 6 (192, NT operands only)
};
// The choice with the least modelled time, in slices of the 256-wide tile
// (~0.5 us each; one of the 192-wide tile, three quarters of the matrix work but
// ten twelfths of the fragment reads, takes 0.84 of it): rounds of 256 workgroups
// times a split's slices plus 8 for its first round trip and its tile's store,
// and for n > 1 the partial tiles written and read back (8 bytes per output and
// split at ~5 TB/s) and the reduction's launch.  Measured:
//   4096 x 2304 over 6912   144 tiles 134 us, 192 narrow ones 118 (operands in the
//                           caches; 176 and 152 with them from HBM); three splits
//                           would move 226 MB of partial tiles
//   512 x 768 over 3072     55 -> 43 us
//   4096 x 4096 over 4096   256 tiles 109 us, 352 narrow ones 152
//   2048 x 50304 over 2304  1576 tiles 466 us, 2096 narrow ones 492
//   2048 x 2304 over 50304  72 tiles 1219 us, three splits of them 479 + 12
//                           (reduction)
// A function of the shape alone: the workspace size and the launch agree on
// every device, and the split (so the sum's order) is the same on every call.
// The width does not change a result: every output sums its slices in order.
static int64_t q4_tiles(int64_t M, int64_t N, int nj) { return ((M + 255) / 256) * ((N + 32 * nj - 1) / (32 * nj)); }
static Q4Split q4_split_of(int64_t M, int64_t N, int64_t Kc, bool tn, int max_split) {
  const int64_t nks = (Kc + 31) / 32;
  Q4Split best{1, (int)nks, 8};
  double cost = 1e300;
  for (int nj = 8; nj >= (tn ? 8 : 6); nj -= 2) {
    const int64_t tiles = q4_tiles(M, N, nj);
    const double rel = nj == 8 ? 1.0 : 0.84;   // a slice's time
    for (int64_t n = 1; n <= max_split; ++n) {
      const int64_t per = (nks + n - 1) / n;
      if (n > 1 && (per < 16 || (nks + per - 1) / per != n)) continue;
      const double c = (double)((tiles * n + 255) / 256) * ((double)per * rel + 8) +
                       (n > 1 ? 6.0 + (double)(tiles * n) * (8192.0 * nj * 8.0 / 2.5e6) : 0.0);
      if (c < cost * 0.97) {
        cost = c;
        best = Q4Split{(int)n, (int)per, nj};
      }
    }
  }
  return best;
}
static size_t q4_part_bytes(const Q4Split& sp, int64_t M, int64_t N) {
  return sp.n > 1 ? (size_t)sp.n * (size_t)q4_tiles(M, N, sp.nj) * (size_t)(8192 * sp.nj) * 4 : 0;
}

template <int NJ>
static int launch_q4_reduce(const float* part, __bf16* c, int64_t M, int64_t N, int tiles_m, int tiles_n, int n,
                            hipStream_t st) {
  hipLaunchKernelGGL(q4_reduce_kernel<NJ>, dim3((unsigned)(tiles_m * tiles_n * 8)), dim3(256), 0, st,
                     reinterpret_cast<const float4*>(part), c, (int)M, (int)N, tiles_m, tiles_n, n);
  return check_launch("gemm_bf16_reduce");
}

// C (M, N) = A^T B, A (Kc, M) pitch lda, B (Kc, N) pitch ldb (gemm_bf16_tn_q4_kernel);
// part: q4_part_bytes(sp, M, N) bytes, used when sp.n > 1
int launch_gemm_bf16_tn(const __bf16* a, int64_t lda, const __bf16* b, int64_t ldb, __bf16* c, int64_t M,
                        int64_t N, int64_t Kc, const Q4Split& sp, float* part, hipStream_t st) {
  if (M == 0 || N == 0) return TG_OK;
  const int tiles_m = (int)((M + 255) / 256), tiles_n = (int)((N + 255) / 256);
  hipLaunchKernelGGL(gemm_bf16_tn_q4_kernel, dim3((unsigned)(tiles_m * tiles_n * sp.n)), dim3(512), 0, st, a, b, c,
                     (int)M, (int)N, (int)Kc, (int)lda, (int)ldb, tiles_m, tiles_n, sp.n, sp.per, part);
  TG_TRY(check_launch("gemm_bf16_tn"));
  return sp.n > 1 ? launch_q4_reduce<8>(part, c, M, N, tiles_m, tiles_n, sp.n, st) : TG_OK;
}

template <int NJ>
static int launch_q4_nt(const __bf16* a, const __bf16* b, __bf16* c, int64_t M, int64_t N, int64_t K,
                        const Q4Split& sp, float* part, hipStream_t st) {
  const int tiles_m = (int)((M + 255) / 256), tiles_n = (int)((N + 32 * NJ - 1) / (32 * NJ));
  hipLaunchKernelGGL(gemm_bf16_nt_q4_kernel<NJ>, dim3((unsigned)(tiles_m * tiles_n * sp.n)), dim3(512), 0, st,
                     a, b, c, (int)M, (int)N, (int)K, tiles_m, tiles_n, sp.n, sp.per, part);
  TG_TRY(check_launch("gemm_bf16_nt"));
  return sp.n > 1 ? launch_q4_reduce<NJ>(part, c, M, N, tiles_m, tiles_n, sp.n, st) : TG_OK;
}

int launch_gemm_bf16(const __bf16* a, const __bf16* b, __bf16* c, int64_t M, int64_t N, int64_t K,
                     const Q4Split& sp, float* part, hipStream_t st) {
  if (M == 0 || N == 0) return TG_OK;
  return sp.nj == 8 ? launch_q4_nt<8>(a, b, c, M, N, K, sp, part, st) : launch_q4_nt<6>(a, b, c, M, N, K, sp, part, st);
}

}  // namespace tg

using namespace tg;

static inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }
static inline int64_t round64(int64_t x) { return (x + 63) & ~(int64_t)63; }

static int check_bf16_gemm(int64_t M, int64_t N, int64_t K) {
  if (M < 0 || N < 0 || K <= 0) return einval("bad GEMM shape");
  if (K % 64) return einval("gemm_bf16_nt: K must be a multiple of 64");
  // buffer offsets are 32-bit: each operand must stay below 2 GiB
  if ((uint64_t)M * (uint64_t)K * 2 >= (1ull << 31) || (uint64_t)N * (uint64_t)K * 2 >= (1ull << 31))
    return einval("gemm_bf16_nt: operand larger than 2 GiB");
  if (M > 0x7FFFFFFF || N > 0x7FFFFFFF) return einval("GEMM dimension too large");
  return TG_OK;
}

extern "C" int tg_gemm_bf16_nt(const void* a, const void* b, void* c, int64_t M, int64_t N,
                               int64_t K, void* stream) {
  TG_TRY(check_bf16_gemm(M, N, K));
  if (M == 0 || N == 0) return TG_OK;
  if (!a || !b || !c) return einval("gemm_bf16_nt: null pointer");
  if (!aligned(a, 16) || !aligned(b, 16)) return einval("gemm_bf16_nt: operands must be 16-byte aligned");
  return launch_gemm_bf16(reinterpret_cast<const __bf16*>(a), reinterpret_cast<const __bf16*>(b),
                          reinterpret_cast<__bf16*>(c), M, N, K, q4_split_of(M, N, K, false, 1), nullptr,
                          as_stream(stream));
}

extern "C" int tg_pack_bf16(const void* x, int x_dtype, int64_t rows, int64_t cols, int transpose,
                            void* y, int64_t pitch, void* stream) {
  if (x_dtype != TG_DTYPE_BF16 && x_dtype != TG_DTYPE_F32) return einval("pack_bf16: bad x_dtype");
  if (rows < 0 || cols < 0 || rows > 0x7FFFFFFF || cols > 0x7FFFFFFF) return einval("pack_bf16: bad shape");
  if (pitch < (transpose ? rows : cols) || pitch > 0x7FFFFFFF) return einval("pack_bf16: pitch too small");
  if (rows == 0 || cols == 0) return TG_OK;
  if (!x || !y) return einval("pack_bf16: null pointer");
  if ((transpose ? pitch : rows) > 65535LL * 64) return einval("pack_bf16: too many rows");
  return launch_pack_bf16(x, x_dtype, rows, cols, transpose, reinterpret_cast<__bf16*>(y), pitch,
                          as_stream(stream));
}

extern "C" size_t tg_block_scaled_matmul_bwd_bf16_workspace(int64_t M, int64_t N, int64_t K) {
  if (M < 0 || N < 0 || K < 0) return 0;
  const size_t np = (size_t)round64(N), mp = (size_t)round64(M);
  const size_t px = q4_part_bytes(q4_split_of(M, K, (int64_t)np, false, 16), M, K);
  const size_t pw = q4_part_bytes(q4_split_of(K, N, M, true, 16), K, N);
  return align256((size_t)M * np * 2) + align256((size_t)K * np * 2) +   // g, b packed along N
         align256((size_t)K * mp * 2) + align256((size_t)N * mp * 2) +   // a.T, g.T packed along M
         (px > pw ? px : pw);                                            // split-K partial tiles of dX, then of dW
}

extern "C" int tg_block_scaled_matmul_bwd_bf16(const void* a, int a_dtype, const void* b,
                                               int b_dtype, const void* g, int g_dtype, void* da,
                                               void* db, int64_t M, int64_t N, int64_t K,
                                               void* workspace, size_t workspace_bytes,
                                               void* stream) {
  for (int d : {a_dtype, b_dtype, g_dtype})
    if (d != TG_DTYPE_BF16 && d != TG_DTYPE_F32) return einval("block_scaled_matmul_bwd_bf16: bad dtype");
  if (M < 0 || N < 0 || K < 0) return einval("block_scaled_matmul_bwd_bf16: bad shape");
  if (M == 0 || N == 0 || K == 0) {
    // an empty contraction gives zero gradients; an empty output is a no-op
    if ((M * K && !da) || (K * N && !db)) return einval("block_scaled_matmul_bwd_bf16: null pointer");
    TG_TRY(launch_fill_zero_bf16(da, M * K, as_stream(stream)));
    return launch_fill_zero_bf16(db, K * N, as_stream(stream));
  }
  const int64_t np = round64(N), mp = round64(M);
  TG_TRY(check_bf16_gemm(M, K, np));    // dX = g . b.T   contracts N
  TG_TRY(check_bf16_gemm(K, N, mp));    // dW = a.T . g   contracts M
  if (!a || !b || !g || !da || !db || !workspace) return einval("block_scaled_matmul_bwd_bf16: null pointer");
  if (workspace_bytes < tg_block_scaled_matmul_bwd_bf16_workspace(M, N, K))
    return einval("block_scaled_matmul_bwd_bf16: workspace too small");
  if (!aligned(workspace, 256)) return einval("block_scaled_matmul_bwd_bf16: workspace must be 256-byte aligned");
  hipStream_t st = as_stream(stream);
  uint8_t* p = reinterpret_cast<uint8_t*>(workspace);
  __bf16* gp = reinterpret_cast<__bf16*>(p);   p += align256((size_t)M * np * 2);
  __bf16* bp = reinterpret_cast<__bf16*>(p);   p += align256((size_t)K * np * 2);
  __bf16* at = reinterpret_cast<__bf16*>(p);   p += align256((size_t)K * mp * 2);
  __bf16* gt = reinterpret_cast<__bf16*>(p);   p += align256((size_t)N * mp * 2);
  float* part = reinterpret_cast<float*>(p);
  const Q4Split spx = q4_split_of(M, K, np, false, 16), spw = q4_split_of(K, N, M, true, 16);
  // dX operands: used in place when already bf16, 64-aligned along N and 16-byte aligned
  const __bf16* gx = reinterpret_cast<const __bf16*>(g);
  const __bf16* bx = reinterpret_cast<const __bf16*>(b);
  if (g_dtype != TG_DTYPE_BF16 || np != N || !aligned(g, 16)) {
    TG_TRY(launch_pack_bf16(g, g_dtype, M, N, 0, gp, np, st));
    gx = gp;
  }
  if (b_dtype != TG_DTYPE_BF16 || np != N || !aligned(b, 16)) {
    TG_TRY(launch_pack_bf16(b, b_dtype, K, N, 0, bp, np, st));
    bx = bp;
  }
  TG_TRY(launch_gemm_bf16(gx, bx, reinterpret_cast<__bf16*>(da), M, K, np, spx, part, st));   // fp8.py:95
  // db = a.T . g read straight from a and g (contraction-major operands): rows
  // of a and g are read in 16-byte pieces, g's from its packed copy where its
  // own rows are not aligned (an odd vocabulary)
  const bool g_in_place = gx != gp && N % 8 == 0;
  if (a_dtype == TG_DTYPE_BF16 && K % 8 == 0 && aligned(a, 16) && (gx == gp || g_in_place))
    return launch_gemm_bf16_tn(reinterpret_cast<const __bf16*>(a), K, gx, gx == gp ? np : N,
                               reinterpret_cast<__bf16*>(db), K, N, M, spw, part, st);         // fp8.py:96
  TG_TRY(launch_pack_bf16(a, a_dtype, M, K, 1, at, mp, st));
  TG_TRY(launch_pack_bf16(g, g_dtype, M, N, 1, gt, mp, st));
  return launch_gemm_bf16(at, gt, reinterpret_cast<__bf16*>(db), K, N, mp, spw, part, st);      // fp8.py:96
}
