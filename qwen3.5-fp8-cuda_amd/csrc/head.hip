// bf16 lm_head over several rows (gfx950): logits of every kept position of a
// prompt but the last, which the decode head's fused GEMV + argmax takes.
//
// Semantics (main.py:1596-1604 with logits_to_keep != 1): logits[m] =
// bf16(RMSNorm(x[m]) . W^T), the (1+w) norm rounded to bf16 as the decode head
// does.  One launch reads the 1.27 GB of weights once for up to 128 rows,
// where a GEMV per row read them once for each (96 rows: 18.2 ms).
#include "gemm_tile.h"
#include "qh_common.h"
#include "qh_kernels.h"

namespace {

// One K group and the same order of K steps in every shape, so a row's logits
// do not depend on how many rows there are.  Up to 128 rows the weight stream
// bounds it (a plain read of it: 186 us), above that the matrix products.  us
// at 248320 x 2560, the shapes by their row ranges:
//   8 / 32 rows     32 x 128   218 / 233  (64 x 128: 220 / 233)
//   64 rows         64 x 128   253        (128 x 128: 257)
//   95 / 128 rows   128 x 256  264 / 275  (128 x 128: 280 / 299)
//   512 rows        128 x 128  746        (128 x 256: 778; 256 x 128: 764)
using Head32 = qh_tile::Cfg<2, 2, 1, 4, 1, 64, 3, 2>;
using Head64 = qh_tile::Cfg<4, 2, 1, 4, 1, 64, 3, 2>;
using Head128 = qh_tile::Cfg<4, 4, 2, 4, 1, 64, 3, 2>;
using HeadMany = qh_tile::Cfg<4, 4, 2, 2, 1, 64, 2, 2>;

// Workgroup b runs on XCD b % 8, which takes the x-th eighth of the tiles, row
// tile fastest: the row tiles of a column run together and share its weights.
template <typename C>
__global__ __launch_bounds__(C::THREADS, 2) void head_rows_kernel(const uint16_t* x, const uint16_t* w, uint16_t* y,
                                                                  int M, int N, int K, int tiles_m, int tiles_n) {
  extern __shared__ __align__(16) uint8_t smem[];
  const long T = (long)tiles_m * tiles_n, per = (T + 7) / 8;
  const long item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (item >= T) return;
  const int n0 = (int)(item / tiles_m) * C::BN, m0 = (int)(item % tiles_m) * C::BM;
  qh_tile::Work t = {};
  t.x = x + (size_t)m0 * K;
  t.w = (const uint8_t*)(w + (size_t)n0 * K);
  t.rows_m = min(M - m0, C::BM);
  t.rows_n = min(N - n0, C::BN);
  t.K = K;
  t.u1 = K / C::KU;
  f32x4 acc[C::MI][C::NJ];
  qh_tile::mainloop<C, float>(t, smem, acc);
  qh_tile::store_rows<C>(t, smem, acc, y + (size_t)m0 * N + n0, N);
}

template <typename C>
void launch(const uint16_t* x, const uint16_t* w, uint16_t* y, int M, int N, int K, hipStream_t st) {
  const int tiles_m = (M + C::BM - 1) / C::BM, tiles_n = (N + C::BN - 1) / C::BN;
  const long per = ((long)tiles_m * tiles_n + 7) / 8;
  hipLaunchKernelGGL(head_rows_kernel<C>, dim3((unsigned)(8 * per)), dim3(C::THREADS), (size_t)C::LDS, st, x, w, y, M,
                     N, K, tiles_m, tiles_n);
}

}  // namespace

int qh_launch_head_rows(const void* x, const void* w, void* logits, int M, int N, int K, hipStream_t st) {
  // the tiles' buffer ranges (up to 256 rows of K bf16) stay below 2^31 bytes
  if (K <= 0 || K % 64 != 0 || K >= (1 << 22) || (uintptr_t)x % 16 != 0 || (uintptr_t)w % 16 != 0) {
    qh_set_error("lm_head rows: K=%d must be a positive multiple of 64, x and w 16-byte aligned", K);
    return -1;
  }
  const uint16_t *xa = (const uint16_t*)x, *wa = (const uint16_t*)w;
  if (M <= 32) launch<Head32>(xa, wa, (uint16_t*)logits, M, N, K, st);
  else if (M <= 64) launch<Head64>(xa, wa, (uint16_t*)logits, M, N, K, st);
  else if (M <= 128) launch<Head128>(xa, wa, (uint16_t*)logits, M, N, K, st);
  else launch<HeadMany>(xa, wa, (uint16_t*)logits, M, N, K, st);
  return 0;
}
