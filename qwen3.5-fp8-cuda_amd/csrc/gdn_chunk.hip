// Chunked (WY) GatedDeltaNet prefill on the bf16 matrix cores (gfx950).
//
// Semantics: the gated delta rule of the batch prefill from the stored state
// (main.py:1139-1149 calls transformers torch_chunk_gated_delta_rule,
// modeling_qwen3_5.py:249-328, chunk 64), q and k l2-normalised in bf16 steps
// (gdn_norm_gates_kernel) and q scaled by dk^-1/2.  Per value head h and chunk
// of 64 tokens, with G the cumulative log decay inside the chunk and beta the
// write strength:
//   A  = -tril_(-1)(diag(beta) K K^T * exp(G_i - G_j)),   T = (I - A)^-1
//   W  = T diag(beta e^G) K,   U = T diag(beta) V                (prep kernel)
//   V' = U - W S,   O = diag(e^G) Q S + tril(Q K^T * exp(G_i - G_j)) V'
//   S <- e^{G_last} S + K^T diag(e^{G_last - G}) V'               (state kernel)
// core = bf16(O); gdn_gated_norm_kernel then applies the gated RMSNorm.
//
// Products run on v_mfma_f32_16x16x32_bf16: lane l (r = l % 16, g = l / 16)
// holds A[r][8 g + i], B[8 g + i][r], i = 0..7, and D[4 g + q][r], q = 0..3.  k,
// v and the l2-normalised q are bf16 values, so K K^T, Q K^T and the products
// with K, V and K^T take them exactly in one pass.  fp32 operands (T, W, S, V',
// the decays) are split into bf16 hi + lo, x = hi + lo + O(2^-17 |x|), and
// multiplied in two or three passes (lo x lo dropped); accumulation is fp32.
//
// Work split: the prep kernel is one workgroup per (chunk, head), all chunks at
// once (it does not read the state); the state kernel is one workgroup per
// (head, 16 value columns), walking the chunks in order.  The prep kernel hands
// W, U, the masked Q K^T and K^T to the state kernel through a workspace of
// qh_gdn_chunk_ws_bytes(), each as the state kernel's matrix operands: one
// 1 KB run per 16 x 32 block, lane l's 16 bytes at 16 l, the fp32 ones already
// split.  What bounds the state kernel is that serial walk: per chunk one round
// of loads, W S and Q S, a barrier, the state update, a barrier.  With row-major
// fp32 operands (each load 16 rows, every operand split by every wave) and the
// state in fp32 in LDS a chunk took 3.7 us; now 1.9 (3700 tokens, Hv = 32: 216 ->
// 108 us; 122 without the lines touched ahead), 80 KB of operands per workgroup
// and chunk out of L2.
#include "qh_common.h"
#include "qh_prefill.h"

namespace {

constexpr int CH = 64;           // tokens per chunk
constexpr int DK = 128, DV = 128;
constexpr int RS = 136;          // bf16 row stride of the token-major K tile
constexpr int TS = 72;           // bf16 row stride of the dim-major K^T and V^T tiles
constexpr int AS = 68;           // fp32 row stride of A and T
constexpr int NCG = DV / 16;     // state-kernel workgroups per head
constexpr float kQScale = 0.0883883476483184405f;  // 128^-1/2

// Workspace of one (head, chunk) unit, in floats (256 of them: one 1 KB block of
// 64 lanes x 16 bytes):
//   W   [4 row tiles][4 K steps][hi, lo]   W rows as A operands
//   U   [4 row tiles][8 column tiles]      U as D values (fp32)
//   Att [4 row tiles][2 K steps][hi, lo]   the masked, scaled Q K^T (K step 1 of
//                                          row tiles 0, 1 is zero: not stored)
//   KT  [8 d tiles][2 K steps]             K^T rows as A operands
// and the decays per token E = e^(G_last - G), QE = 128^-1/2 e^G, and e^(G_last).
constexpr size_t kBlk = 256;
constexpr size_t kW = 0, kU = kW + 32 * kBlk, kAtt = kU + 32 * kBlk, kKT = kAtt + 16 * kBlk, kE = kKT + 16 * kBlk,
                 kQE = kE + CH, kEL = kQE + CH, kUnitFloats = kEL + 2 * CH;

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f4 mma(u32x4 a, u32x4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}
// x = hi + lo + O(2^-17 |x|), hi and lo bf16 (round to nearest even), packed in
// pairs
struct HiLo {
  uint32_t hi, lo;
};
__device__ __forceinline__ HiLo split2(float x, float y) {
  const uint32_t hi = pack_bf2(x, y);
  return {hi, pack_bf2(x - bf_lo(hi), y - bf_hi(hi))};
}
__device__ __forceinline__ void split4(f4 x, u32x2& hi, u32x2& lo) {
  const HiLo a = split2(x[0], x[1]), b = split2(x[2], x[3]);
  hi = u32x2{a.hi, b.hi};
  lo = u32x2{a.lo, b.lo};
}
__device__ __forceinline__ void split8(f4 x, f4 y, u32x4& hi, u32x4& lo) {
  const HiLo a = split2(x[0], x[1]), b = split2(x[2], x[3]), c = split2(y[0], y[1]), d = split2(y[2], y[3]);
  hi = u32x4{a.hi, b.hi, c.hi, d.hi};
  lo = u32x4{a.lo, b.lo, c.lo, d.lo};
}
__device__ __forceinline__ f4 zero4() { return f4{0.0f, 0.0f, 0.0f, 0.0f}; }
// Barrier that orders LDS only (a __syncthreads would also wait for the global
// loads in flight, the next chunk's operands).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ---- prep: grid (chunks, Hv), 256 threads -----------------------------------
// Two workgroups per CU (71 KB of LDS; with K, Q, T' and both dim-major tiles
// in LDS it was one, and 3700 tokens took 115 us).
__global__ __launch_bounds__(256, 2) void gdn_chunk_prep_kernel(QhGdnScanParams p, float* ws, int nch) {
  __shared__ __align__(16) uint16_t sKV[DV * TS];  // K token-major (stride RS), then V dim-major (stride TS)
  __shared__ __align__(16) uint16_t sKT[DK * TS];
  __shared__ __align__(16) float sA[CH * AS];
  __shared__ __align__(16) float sT[CH * AS];      // T = (I - A)^-1
  __shared__ __align__(16) float sG[CH], sB[CH], sW[CH];  // G, beta, beta e^G
  static_assert(CH * RS <= DV * TS, "K fits its tile");
  uint16_t* sK = sKV;

  const int c = blockIdx.x, h = blockIdx.y, kh = h / (p.Hv / p.Hk);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int t0 = c * CH;
  float* unit = ws + ((size_t)h * nch + c) * kUnitFloats;

  // ---- loads: every wave the 64 tokens' decay and write strength; waves 0-1
  // K, waves 2-3 V (8 tokens x 8 dims per thread); each wave its 16 rows of Q as
  // A operands.  Rows past M count as zeros (padding: no decay, no write).
  const bool tok_ok = t0 + lane < p.M;
  const int tok = tok_ok ? t0 + lane : p.M - 1;
  float G = p.g[(size_t)tok * p.Hv + h];
  float beta = bf2f(p.beta[(size_t)tok * p.Hv + h]);
  const u32x4 zero = {0u, 0u, 0u, 0u};
  const bool is_v = w >= 2;
  const int tg = tid & 7, dg = (tid & 127) >> 3;  // tokens 8 tg .. + 7, dims 8 dg .. + 7
  u32x4 x[8], qf[4];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int t = min(t0 + 8 * tg + j, p.M - 1);
    x[j] = is_v ? *(const u32x4*)(p.y + (size_t)t * p.C + (size_t)2 * p.Hk * DK + (size_t)h * DV + 8 * dg)
                : *(const u32x4*)(p.kn + ((size_t)t * p.Hk + kh) * DK + 8 * dg);
  }
  {
    const int t = t0 + 16 * w + r;
    const uint16_t* qrow = p.qn + ((size_t)min(t, p.M - 1) * p.Hk + kh) * DK;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = *(const u32x4*)(qrow + 32 * s + 8 * g);
    if (t >= p.M) {
#pragma unroll
      for (int s = 0; s < 4; ++s) qf[s] = zero;
    }
  }
  G = tok_ok ? G : 0.0f;
  beta = tok_ok ? beta : 0.0f;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {  // inclusive cumulative sum of the log decays
    const float y = __shfl_up(G, off, 64);
    G = lane >= off ? G + y : G;
  }
  if (w == 0) {
    const float glast = __shfl(G, CH - 1, 64), eg = expf(G);
    sG[lane] = G;
    sB[lane] = beta;
    sW[lane] = beta * eg;
    unit[kE + lane] = expf(glast - G);
    unit[kQE + lane] = kQScale * eg;
    if (lane == 0) unit[kEL] = expf(glast);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (t0 + 8 * tg + j >= p.M) x[j] = zero;
  // dim 8 dg + j, tokens 8 tg .. + 7: pairs of 16-bit halves (v_perm), 16-byte rows
  auto transposed = [&](int j) {
    const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
    u32x4 col;
#pragma unroll
    for (int q = 0; q < 4; ++q) col[q] = __builtin_amdgcn_perm(x[2 * q + 1][j >> 1], x[2 * q][j >> 1], sel);
    return col;
  };
  if (!is_v) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      *(u32x4*)(sK + (8 * tg + j) * RS + 8 * dg) = x[j];
      *(u32x4*)(sKT + (8 * dg + j) * TS + 8 * tg) = transposed(j);
    }
  }
  __syncthreads();

  // ---- rows i = 16 w .. + 15 of A and of Att, columns j <= i ----------------------
  // Column tiles come in pairs a = 0, 1 over the 32 columns of a K step of the
  // state kernel's Att product, column 8 (m / 4) + 4 a + m % 4 in row m of the
  // matrix operand, so that a lane's four values of both tiles are the eight
  // consecutive columns 8 g .. + 7 it hands over.
  const int i = 16 * w + r;  // the lane's row of both
  const float Gi = sG[i], bi = sB[i];
  const int nks = w < 2 ? 1 : 2;  // 32-column steps with a column <= i
  {
    u32x4 ki[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) ki[s] = *(const u32x4*)(sK + i * RS + 32 * s + 8 * g);
    for (int ks = 0; ks < nks; ++ks) {
      f4 kk[2], qk[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        kk[a] = qk[a] = zero4();
        const int jr = 32 * ks + 8 * (r >> 2) + 4 * a + (r & 3);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const u32x4 kj = *(const u32x4*)(sK + jr * RS + 32 * s + 8 * g);
          kk[a] = mma(kj, ki[s], kk[a]);
          qk[a] = mma(kj, qf[s], qk[a]);
        }
      }
      f4 at[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int j0 = 32 * ks + 8 * g + 4 * a;
        const f4 Gj = *(const f4*)(sG + j0);
        f4 av;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float dec = expf(Gi - Gj[q]);  // used for j <= i only (G_i <= G_j)
          av[q] = j0 + q < i ? -bi * kk[a][q] * dec : 0.0f;
          at[a][q] = j0 + q <= i ? qk[a][q] * kQScale * dec : 0.0f;
        }
        *(f4*)(sA + i * AS + j0) = av;
      }
      u32x4 hi, lo;
      split8(at[0], at[1], hi, lo);
      float* dst = unit + kAtt + (size_t)((w * 2 + ks) * 2) * kBlk + lane * 4;
      *(u32x4*)dst = hi;
      *(u32x4*)(dst + kBlk) = lo;
    }
  }
  __syncthreads();  // sA complete; the K tile is no longer read
  if (is_v) {
#pragma unroll
    for (int j = 0; j < 8; ++j) *(u32x4*)(sKV + (8 * dg + j) * TS + 8 * tg) = transposed(j);
  }

  // ---- T = (I - A)^-1, blocked by 16 ---------------------------------------
  // Diagonal blocks T_bb = (I - A_bb)^-1 by forward substitution, one per wave;
  // then block row by block row, T_ij = T_ii sum_{k=j}^{i-1} A_ik T_kj, wave j
  // computing block (i, j) on v_mfma_f32_16x16x4_f32 (fp32 products and sums).
  // The upper blocks of T are zero.
  {
    // lane m (mod 16) holds column m of A_ww; row n reads A[n][m] from lane m
    // into a scalar register (v_readlane)
    float Acol[16], Tc[16];
#pragma unroll
    for (int n = 0; n < 16; ++n) Acol[n] = sA[(16 * w + n) * AS + 16 * w + r];
#pragma unroll
    for (int m = 0; m < 16; ++m) Tc[m] = m == r ? 1.0f : 0.0f;
#pragma unroll
    for (int n = 1; n < 16; ++n) {
      float acc[2] = {0.0f, 0.0f};
      const int an = __builtin_bit_cast(int, Acol[n]);
#pragma unroll
      for (int m = 0; m < n; ++m)
        acc[m & 1] = fmaf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(an, m)), Tc[m], acc[m & 1]);
      Tc[n] = n > r ? acc[0] + acc[1] : Tc[n];
    }
    if (lane < 16) {
#pragma unroll
      for (int n = 0; n < 16; ++n) sT[(16 * w + n) * AS + 16 * w + r] = Tc[n];
    }
    for (int b = w + 1; b < 4; ++b)  // zero upper blocks of block row w
      *(f4*)(sT + (16 * w + r) * AS + 16 * b + 4 * g) = zero4();
  }
  __syncthreads();
  // the matrix step q of a 16 x 16 x 16 product takes k = 4 g + q, so a lane's
  // row operand is one 16-byte read and a product's result, rows 4 g + q, is
  // the column operand of the next as it stands
  for (int bi2 = 1; bi2 < 4; ++bi2) {
    if (w < bi2) {
      f4 xs = zero4();
      for (int k = w; k < bi2; ++k) {
        const f4 a4 = *(const f4*)(sA + (16 * bi2 + r) * AS + 16 * k + 4 * g);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          xs = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[q], sT[(16 * k + 4 * g + q) * AS + 16 * w + r], xs, 0, 0, 0);
      }
      const f4 t4 = *(const f4*)(sT + (16 * bi2 + r) * AS + 16 * bi2 + 4 * g);
      f4 tv = zero4();
#pragma unroll
      for (int q = 0; q < 4; ++q) tv = __builtin_amdgcn_mfma_f32_16x16x4f32(t4[q], xs[q], tv, 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) sT[(16 * bi2 + 4 * g + q) * AS + 16 * w + r] = tv[q];
    }
    __syncthreads();
  }

  // ---- W = T diag(beta e^G) K and U = T diag(beta) V, rows i ----------------------
  u32x4 wh[2], wl[2], uh[2], ul[2];  // the lane's row of both T', split
  for (int s = 0; s < 2; ++s) {
    const f4 ta = *(const f4*)(sT + i * AS + 32 * s + 8 * g), tb = *(const f4*)(sT + i * AS + 32 * s + 8 * g + 4);
    const f4 wa = *(const f4*)(sW + 32 * s + 8 * g), wb = *(const f4*)(sW + 32 * s + 8 * g + 4);
    const f4 ba = *(const f4*)(sB + 32 * s + 8 * g), bb = *(const f4*)(sB + 32 * s + 8 * g + 4);
    split8(ta * wa, tb * wb, wh[s], wl[s]);
    split8(ta * ba, tb * bb, uh[s], ul[s]);
  }
  // W transposed (rows d): tiles a = 0, 1 of 32 dims, dim 8 (m / 4) + 4 a + m % 4
  // in row m, as for Att
#pragma unroll
  for (int ds = 0; ds < 4; ++ds) {
    f4 wv[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      wv[a] = zero4();
      const int d = 32 * ds + 8 * (r >> 2) + 4 * a + (r & 3);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if (s >= nks) continue;
        const u32x4 kt = *(const u32x4*)(sKT + d * TS + 32 * s + 8 * g);
        wv[a] = mma(kt, wh[s], wv[a]);
        wv[a] = mma(kt, wl[s], wv[a]);
      }
    }
    u32x4 hi, lo;
    split8(wv[0], wv[1], hi, lo);
    float* dst = unit + kW + (size_t)((w * 4 + ds) * 2) * kBlk + lane * 4;
    *(u32x4*)dst = hi;
    *(u32x4*)(dst + kBlk) = lo;
  }
#pragma unroll
  for (int tn = 0; tn < 8; ++tn) {
    f4 u = zero4();
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (s >= nks) continue;
      const u32x4 vt = *(const u32x4*)(sKV + (16 * tn + r) * TS + 32 * s + 8 * g);
      u = mma(uh[s], vt, u);
      u = mma(ul[s], vt, u);
    }
    *(f4*)(unit + kU + (size_t)(w * 8 + tn) * kBlk + lane * 4) = u;
  }
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int s = 0; s < 2; ++s)
      *(u32x4*)(unit + kKT + (size_t)((2 * w + tt) * 2 + s) * kBlk + lane * 4) =
          *(const u32x4*)(sKT + (16 * (2 * w + tt) + r) * TS + 32 * s + 8 * g);
}

// ---- state: grid Hv * NCG (head h, value columns 16 cg .. +15), 512 threads --
// Waves 0-3 ("row waves", token rows 16 w .. +15 of the chunk) form V' = U - W S
// and the output O = diag(e^G) Q S + Att V'; waves 4-7 ("state waves", d rows
// 32 (w-4) .. +31) hold the state in fp32 registers and update it from V',
// alongside the row waves' Att V'.  S, V' and diag(E) V' pass through LDS split
// into bf16 hi + lo once, by the wave that computes them.  Per chunk: [row: W S,
// Q S, V'] barrier [row: Att V', O | state: S update] barrier.  Each wave
// requests its next chunk's global operands (two register sets, the chunk loop
// unrolled by two) while the current chunk runs.
struct RowOps {
  u32x4 wh[4], wl[4];    // W
  u32x2 q[8];            // q rows, 32 s + 8 g .. + 7 (two halves)
  u32x4 ah[2], al[2];    // Att
  f4 u, qe, e;           // U, QE and E of tokens 16 w + 4 g + q
};
struct StateOps {
  u32x4 kt[2][2];
  float elast;           // e^(G_last)
  float touch;           // a word of the unit two chunks further on
};

constexpr int kLines = (int)(kUnitFloats / 32);                      // 128-byte lines of a unit
constexpr int kTouch = (kLines + 4 * NCG - 1) / (4 * NCG);           // per state wave of a head's workgroups

__global__ __launch_bounds__(512, 2) void gdn_chunk_state_kernel(QhGdnScanParams p, const float* ws, int nch) {
  constexpr int SST = DK + 8, VST = CH + 8;  // bf16 strides: 16-byte rows, spread over the banks
  __shared__ __align__(16) uint16_t sSh[16 * SST], sSl[16 * SST];  // the state slice [column][d]
  __shared__ __align__(16) uint16_t sVh[16 * VST], sVl[16 * VST];  // V' of the chunk [column][token]
  __shared__ __align__(16) uint16_t sBh[16 * VST], sBl[16 * VST];  // diag(E) V'
  // The NCG workgroups of a head share its chunk operands (W, Att, q, K^T):
  // with Hv % 8 == 0 they are placed on one XCD (workgroup i runs on XCD
  // i % 8), so those operands come from memory once per head, not once per
  // column group.
  const int bid = (int)blockIdx.x;
  const bool xcd = p.Hv % 8 == 0;
  const int h = xcd ? ((bid >> 3) / NCG) * 8 + (bid & 7) : bid / NCG;
  const int cg = xcd ? (bid >> 3) % NCG : bid % NCG;
  const int kh = h / (p.Hv / p.Hk);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const float* units = ws + (size_t)h * nch * kUnitFloats;

  if (w < 4) {
    // ---------------------------------------------------------- row waves
    // the workgroup's 16 output columns of every token (a uniform resource;
    // the lane's column goes in the offset): bytes past row M - 1 are out of
    // the resource's range
    const auto rout = __builtin_amdgcn_make_buffer_rsrc(p.out + (size_t)h * DV + cg * 16, (short)0,
                                                        (int)(((size_t)(p.M - 1) * p.Hv * DV + 16) * 2), 0x00020000);
    const int nks = w < 2 ? 1 : 2;  // 32-token steps of Att that are not zero
    auto load = [&](RowOps& o, int c) {
      const float* unit = units + (size_t)c * kUnitFloats;
      const int t = min(c * CH + 16 * w + r, p.M - 1);  // rows past M: any row (outputs dropped)
      const uint16_t* qrow = p.qn + ((size_t)t * p.Hk + kh) * DK;
      const float* wp = unit + kW + (size_t)(w * 8) * kBlk + lane * 4;
      const float* ap = unit + kAtt + (size_t)(w * 4) * kBlk + lane * 4;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        o.wh[s] = *(const u32x4*)(wp + (2 * s) * kBlk);
        o.wl[s] = *(const u32x4*)(wp + (2 * s + 1) * kBlk);
        const u32x4 qv = *(const u32x4*)(qrow + 32 * s + 8 * g);
        o.q[2 * s] = u32x2{qv.x, qv.y};
        o.q[2 * s + 1] = u32x2{qv.z, qv.w};
      }
      o.u = *(const f4*)(unit + kU + (size_t)(w * 8 + cg) * kBlk + lane * 4);
      o.qe = *(const f4*)(unit + kQE + 16 * w + 4 * g);
      o.e = *(const f4*)(unit + kE + 16 * w + 4 * g);
#pragma unroll
      for (int s = 0; s < 2; ++s) {  // step 1 of row tiles 0, 1: step 0 again (not used)
        o.ah[s] = *(const u32x4*)(ap + (2 * min(s, nks - 1)) * kBlk);
        o.al[s] = *(const u32x4*)(ap + (2 * min(s, nks - 1) + 1) * kBlk);
      }
    };
    auto step = [&](const RowOps& cur, int c) {
      // W S and Q S: two independent sums of W S, so that no product waits for the one before
      f4 wa = zero4(), wb = zero4(), o = zero4();
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const u32x4 sh = *(const u32x4*)(sSh + r * SST + 32 * s + 8 * g);
        const u32x4 sl = *(const u32x4*)(sSl + r * SST + 32 * s + 8 * g);
        const u32x4 q = {cur.q[2 * s].x, cur.q[2 * s].y, cur.q[2 * s + 1].x, cur.q[2 * s + 1].y};
        wa = mma(cur.wh[s], sh, wa);
        wb = mma(cur.wh[s], sl, wb);
        o = mma(q, sh, o);
        wb = mma(cur.wl[s], sh, wb);
        o = mma(q, sl, o);
      }
      // V' = U - W S (rows: tokens 16 w + 4 g + q, column r)
      const f4 v = cur.u - (wa + wb);
      u32x2 hi, lo;
      split4(v, hi, lo);
      *(u32x2*)(sVh + r * VST + 16 * w + 4 * g) = hi;
      *(u32x2*)(sVl + r * VST + 16 * w + 4 * g) = lo;
      split4(v * cur.e, hi, lo);
      *(u32x2*)(sBh + r * VST + 16 * w + 4 * g) = hi;
      *(u32x2*)(sBl + r * VST + 16 * w + 4 * g) = lo;
      o *= cur.qe;
      lds_barrier();  // V' complete; the old state is read
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if (s >= nks) continue;
        const u32x4 vh = *(const u32x4*)(sVh + r * VST + 32 * s + 8 * g);
        const u32x4 vl = *(const u32x4*)(sVl + r * VST + 32 * s + 8 * g);
        o = mma(cur.ah[s], vh, o);
        o = mma(cur.ah[s], vl, o);
        o = mma(cur.al[s], vh, o);
      }
      // range-checked stores: rows past M are dropped without a branch (a
      // guarded store in this loop made the compiler wait for every
      // outstanding load, the next chunk's operands included, at its head)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        __builtin_amdgcn_raw_buffer_store_b16(
            f2bf(o[q]), rout, (uint32_t)(((c * CH + 16 * w + 4 * g + q) * p.Hv * DV + r) * 2), 0, 0);
      lds_barrier();  // V' read; the new state written
    };
    // the next chunk's loads go out before the step (a scheduling barrier
    // keeps the compiler from sinking them into it, where the next step's
    // wait would expose their latency)
    RowOps ra, rb;
    load(ra, 0);
    lds_barrier();  // the initial state is in LDS
    for (int c = 0; c < nch; c += 2) {
      load(rb, min(c + 1, nch - 1));
      __builtin_amdgcn_sched_barrier(0);
      step(ra, c);
      if (c + 1 >= nch) break;
      load(ra, min(c + 2, nch - 1));
      __builtin_amdgcn_sched_barrier(0);
      step(rb, c + 1);
    }
  } else {
    // -------------------------------------------------------- state waves
    const int sw = w - 4;
    float* state = p.state + (size_t)h * DK * DV + (size_t)(32 * sw + 4 * g) * DV + cg * 16 + r;
    f4 S[2];  // rows 32 sw + 16 tt + 4 g + q, column r
    auto publish = [&](int tt) {
      u32x2 hi, lo;
      split4(S[tt], hi, lo);
      *(u32x2*)(sSh + r * SST + 32 * sw + 16 * tt + 4 * g) = hi;
      *(u32x2*)(sSl + r * SST + 32 * sw + 16 * tt + 4 * g) = lo;
    };
    auto load = [&](StateOps& o, int c) {
      const float* unit = units + (size_t)c * kUnitFloats;
      const float* kp = unit + kKT + (size_t)(4 * sw) * kBlk + lane * 4;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int s = 0; s < 2; ++s) o.kt[tt][s] = *(const u32x4*)(kp + (2 * tt + s) * kBlk);
      o.elast = unit[kEL];
      // this workgroup's eighth of the lines of chunk c + 2 (three ahead of the
      // one being computed): the operands were last written by other XCDs, and
      // a chunk's register prefetch covers a read from this XCD's L2 only
      const int line = min((cg * 4 + sw) * kTouch + min(lane, kTouch - 1), kLines - 1);
      o.touch = units[(size_t)min(c + 2, nch - 1) * kUnitFloats + line * 32];
    };
    // S <- e^{G_last} S + K^T diag(e^{G_last - G}) V'
    auto step = [&](const StateOps& cur) {
      lds_barrier();  // V' complete; the old state is read
      u32x4 bh[2], bl[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        bh[s] = *(const u32x4*)(sBh + r * VST + 32 * s + 8 * g);
        bl[s] = *(const u32x4*)(sBl + r * VST + 32 * s + 8 * g);
      }
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        f4 acc = S[tt] * cur.elast;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          acc = mma(cur.kt[tt][s], bh[s], acc);
          acc = mma(cur.kt[tt][s], bl[s], acc);
        }
        S[tt] = acc;
        publish(tt);
      }
      lds_barrier();  // new state visible; V' read
      asm volatile("" ::"v"(cur.touch));
    };
    StateOps sa, sb;
    load(sa, 0);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int q = 0; q < 4; ++q) S[tt][q] = state[(size_t)(16 * tt + q) * DV];
    publish(0);
    publish(1);
    lds_barrier();
    for (int c = 0; c < nch; c += 2) {
      load(sb, min(c + 1, nch - 1));
      __builtin_amdgcn_sched_barrier(0);
      step(sa);
      if (c + 1 >= nch) break;
      load(sa, min(c + 2, nch - 1));
      __builtin_amdgcn_sched_barrier(0);
      step(sb);
    }
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int q = 0; q < 4; ++q) state[(size_t)(16 * tt + q) * DV] = S[tt][q];
  }
}

}  // namespace

size_t qh_gdn_chunk_ws_bytes(int M, int Hv) {
  if (M <= 0 || Hv <= 0) return 0;
  return (size_t)Hv * ((M + CH - 1) / CH) * kUnitFloats * sizeof(float);
}

int qh_launch_gdn_chunk(const QhGdnScanParams& p, float* ws, size_t ws_bytes, hipStream_t st) {
  if (p.dk != DK || p.dv != DV || p.Hk <= 0 || p.Hv <= 0 || p.Hv % p.Hk != 0) {
    qh_set_error("gdn_chunk: unsupported shape (dk=%d dv=%d Hk=%d Hv=%d)", p.dk, p.dv, p.Hk, p.Hv);
    return -1;
  }
  if (p.M <= 0) return 0;
  const size_t need = qh_gdn_chunk_ws_bytes(p.M, p.Hv);
  if (!ws || ws_bytes < need || ((uintptr_t)ws & 15u) != 0) {
    qh_set_error("gdn_chunk: workspace of %zu bytes (16-byte aligned) needed, got %zu", need, ws_bytes);
    return -1;
  }
  const int nch = (p.M + CH - 1) / CH;
  hipLaunchKernelGGL(gdn_chunk_prep_kernel, dim3(nch, p.Hv), dim3(256), 0, st, p, ws, nch);
  hipLaunchKernelGGL(gdn_chunk_state_kernel, dim3(p.Hv * NCG), dim3(512), 0, st, p, (const float*)ws, nch);
  return qh_launch_gdn_gated_norm(p, st);
}
