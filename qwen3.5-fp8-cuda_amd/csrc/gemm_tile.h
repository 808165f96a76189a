// Device side of the tile GEMM (gfx950): one output tile per workgroup, K
// optionally shared out between the workgroup's waves and between workgroups.
//
//   Y[m, n] = sum_k X[m, k] W[n, k]      X bf16; W E4M3 with 128 x 128 block
//                                        scales (WB = 1) or bf16 (WB = 2)
//
// A workgroup is KG K groups of WM x WN waves.  Every group computes the whole
// BM x BN tile over its own contiguous share of K units (KU = 64 or 128 wide),
// through its own ring of DS LDS stages filled by direct-to-LDS loads; the groups' fp32
// sums meet in LDS at the end.
//
// What bounds it, measured on MI355X by leaving parts out (512 x 9216 x 2560 on
// 128 x 160 tiles, 31.5 us): the loads alone take 28 us, the weights' 17 of
// them although their bytes are few (each unit's weight rows are a round trip
// to HBM), the products and LDS reads alone 30; they overlap badly within one
// workgroup.  So the shapes differ in how they find overlap: K groups (a lone
// wave per group needs no barrier), 128-wide units (half the barriers and half
// the scaling of partials of 64-wide ones), two workgroups per CU where LDS
// allows.  Against the 64 x 64 .. 128 x 192 ring kernel, us (weights out of the
// caches): 24 x 2560 x 9216 48 -> 12, 24 x 9216 x 2560 16.7 -> 9.2, 128 x 2560 x
// 4096 22.8 -> 10.2, 128 x 18432 x 2560 29.5 -> 22.3, 512 x 9216 x 2560 38.3 ->
// 31.5, 3700 x 18432 x 2560 387 -> 346 (1010 TFLOP/s), 3700 x 2560 x 9216 244 ->
// 180.  Measured and not kept: separate waves loading X and W with a deeper W
// ring (no faster), K order rotated by workgroup (no effect).
//
// Products run on v_mfma_f32_16x16x32_bf16 with W as the row operand, so a
// lane ends with four consecutive columns n of one row m (lane l: row l % 16
// of X, columns 4 (l / 16) .. + 3 of W).  Both operands take the same
// permuted K order: lane group g = l / 16 reads the 16 W bytes 16 g .. + 15 of
// a 64-wide K half, whose halves p = 0, 1 feed steps p, and X chunk 2 g + p.
//
// LDS rows are unpadded (direct-to-LDS loads fill whole 1 KB runs) and
// XOR-swizzled by row in 16-byte slots.  A 16-byte read serves lanes 0-3,
// 12-15, 20-23 and 24-27 of a half wave together, then the others; with
// 128-wide units the swizzles put each such group in different banks (counted:
// no conflict cycles), with 64-wide ones 38 % of the LDS cycles still are
// conflicts (half of them with slot c ^ (r / 4) for 64-byte rows).
// LDS reads are inline asm, which the compiler does not count against the
// loads in flight; every read is waited for, by count and tied to its
// registers, before use.
#pragma once

#include "qh_common.h"

namespace qh_tile {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef __attribute__((address_space(3))) void* lds_ptr;

template <int MI_, int NJ_, int WM_, int WN_, int KG_, int KU_, int DS_, int WB_ = 1>
struct Cfg {
  static constexpr int MI = MI_, NJ = NJ_, WM = WM_, WN = WN_, KG = KG_, KU = KU_, DS = DS_, WB = WB_;
  static constexpr int BM = 16 * MI * WM, BN = 16 * NJ * WN;
  static constexpr int GW = WM * WN, THREADS = 64 * GW * KG;
  static constexpr int A = BM * KU * 2, B = BN * KU * WB, STAGE = A + B;
  static constexpr int XC = A / 1024, WC = B / 1024;              // 1 KB loads of a stage
  static constexpr int XL = (XC + GW - 1) / GW, WL = (WC + GW - 1) / GW;  // per wave (the last may repeat)
  static constexpr int KS = KU / 32;                              // matrix-core steps per unit
  static constexpr int KH = WB == 1 ? KU / 64 : KU / 32;          // W reads per 16 columns and unit
  static constexpr int SLAB = BM * (BN + 4) * 4;                  // one group's fp32 tile, padded rows
  static constexpr int RED = KG == 1 ? 0 : KG == 2 ? SLAB : KG * SLAB;
  static constexpr int RING = KG * DS * STAGE;
  static constexpr int LDS = RING > RED ? RING : RED;
  static_assert((KU == 64 || KU == 128) && (WB == 1 || WB == 2) && DS >= 2 && THREADS <= 1024, "config");
  static_assert(LDS <= 163840 && 16 * NJ <= 128, "LDS, scale blocks per wave");
};

__device__ __forceinline__ u32x4 lds_read16(uint32_t a) {
  u32x4 v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(a) : "memory");
  return v;
}
template <int N>
__device__ __forceinline__ void lds_wait() {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N > 15 ? 15 : N) : "memory");
}
__device__ __forceinline__ void lds_wait_c(int n) {  // n: a constant once unrolled
  switch (n > 15 ? 15 : n) {
#define QH_W(c) case c: lds_wait<c>(); break;
    QH_W(0) QH_W(1) QH_W(2) QH_W(3) QH_W(4) QH_W(5) QH_W(6) QH_W(7)
    QH_W(8) QH_W(9) QH_W(10) QH_W(11) QH_W(12) QH_W(13) QH_W(14) QH_W(15)
#undef QH_W
  }
}
// Pins every use of v behind the waits before this point.
__device__ __forceinline__ void settle(u32x4& v) { asm volatile("" : "+v"(v)); }

__device__ __forceinline__ v8bf widen(uint32_t lo, uint32_t hi) {
  const qh_bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false);
  const qh_bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
  const qh_bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false);
  const qh_bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
  return v8bf{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// 16-byte slot that holds chunk c of row r, rows of BYTES bytes
template <int BYTES>
__device__ __forceinline__ int slot(int c, int r) {
  if constexpr (BYTES == 64) return c ^ ((0x78 >> (2 * ((r >> 2) & 3))) & 3);
  else if constexpr (BYTES == 128) return c ^ ((r >> 1) & 7);
  else return c ^ (r & 15);
}

// The tile's operands: X rows m0 .. (rows_m of them), W rows n0 .. (rows_n),
// K units u0 .. u1 - 1 of KU.  Rows past rows_m / rows_n read as zeros.
struct Work {
  const uint16_t* x;   // X + m0 K
  const uint8_t* w;    // W + n0 K (bytes: n0 K WB)
  int rows_m, rows_n, K, u0, u1;
  // block scales (WB = 1): the scale array, its K blocks per row, the tile's
  // first column and the array's last block row
  const void* s;
  int kb, n0, nblk_last;
};

// acc[i][j]: rows 16 i + l % 16, columns 16 j + 4 (l / 16) .. + 3 of the wave's
// sub-tile, summed over the wave's group's share of the K units.
template <typename C, typename ScaleT>
__device__ __forceinline__ void mainloop(const Work& t, uint8_t* smem, f32x4 (&acc)[C::MI][C::NJ]) {
// (device pass only: the host pass rejects lambdas over arrays with template bounds)
#ifdef __HIP_DEVICE_COMPILE__
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wv / C::GW, gw = wv % C::GW;
  const int wm = (gw / C::WN) * 16 * C::MI, wn = (gw % C::WN) * 16 * C::NJ;
  const int r = lane & 15, g = lane >> 4;
  uint8_t* ring = smem + grp * C::DS * C::STAGE;
  const uint32_t ring0 = (uint32_t)(uintptr_t)(lds_ptr)ring;

  // this group's units, and the longest group's count (every wave makes the
  // same number of passes over the barriers)
  const int U = t.u1 - t.u0;
  const int ub = t.u0 + (int)((long)U * grp / C::KG), ue = t.u0 + (int)((long)U * (grp + 1) / C::KG);
  const int passes = (U + C::KG - 1) / C::KG;

  // scales of up to two 128-row blocks of W x 128 K blocks, K block l (+ 64)
  // in lane l: the wave's 16 NJ <= 128 columns span at most two
  float sc[2][2] = {};
  const int nblk0 = C::WB == 1 ? min((t.n0 + wn) >> 7, t.nblk_last) : 0;
  if constexpr (C::WB == 1) {
    const ScaleT* s = (const ScaleT*)t.s;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        sc[b][h] = load_scale<ScaleT>(s, min(nblk0 + b, t.nblk_last) * t.kb + min(lane + 64 * h, t.kb - 1));
  }

  const rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(t.x), (short)0, t.rows_m * t.K * 2,
                                                      0x00020000);
  const rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(t.w), (short)0,
                                                      t.rows_n * t.K * C::WB, 0x00020000);
  // load i of wave q of the group fills LDS run min(q + GW i, runs - 1) of the
  // stage (a repeated last run stores the same bytes twice)
  constexpr int XB = C::KU * 2, WBY = C::KU * C::WB;  // row bytes
  uint32_t xo[C::XL], wo[C::WL];
#pragma unroll
  for (int i = 0; i < C::XL; ++i) {
    const int q = min(gw + C::GW * i, C::XC - 1) * 64 + lane;  // 16-byte slot of the stage's X area
    const int row = q / (XB / 16), c = slot<XB>(q % (XB / 16), row);
    xo[i] = (uint32_t)row * (uint32_t)t.K * 2u + (uint32_t)c * 16u;
  }
#pragma unroll
  for (int i = 0; i < C::WL; ++i) {
    const int q = min(gw + C::GW * i, C::WC - 1) * 64 + lane;
    const int row = q / (WBY / 16), c = slot<WBY>(q % (WBY / 16), row);
    wo[i] = (uint32_t)row * (uint32_t)t.K * (uint32_t)C::WB + (uint32_t)c * 16u;
  }
  // (past the group's share the last unit is loaded again, so that every pass
  // has the same loads in flight)
  auto issue = [&](int st, int u) {
    u = min(u, t.u1 - 1);
    uint8_t* stage = ring + st * C::STAGE;
#pragma unroll
    for (int i = 0; i < C::WL; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr)(stage + C::A + min(gw + C::GW * i, C::WC - 1) * 1024), 16,
                                               wo[i], u * WBY, 0, 0);
#pragma unroll
    for (int i = 0; i < C::XL; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr)(stage + min(gw + C::GW * i, C::XC - 1) * 1024), 16,
                                               xo[i], u * XB, 0, 0);
  };

#pragma unroll
  for (int i = 0; i < C::MI; ++i)
#pragma unroll
    for (int j = 0; j < C::NJ; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int s = 0; s < C::DS - 1; ++s) issue(s, ub + s);

  // LDS byte offsets of the lane's operand chunks within a stage
  uint32_t xr[C::KS], wr[C::KH];
#pragma unroll
  for (int k = 0; k < C::KS; ++k) {
    const int c = 8 * (k >> 1) + 2 * g + (k & 1);
    xr[k] = (uint32_t)((wm + r) * XB + slot<XB>(c, r) * 16);
  }
#pragma unroll
  for (int k = 0; k < C::KH; ++k) {
    const int c = C::WB == 1 ? 4 * k + g : 8 * (k >> 1) + 2 * g + (k & 1);
    wr[k] = (uint32_t)(C::A + (wn + r) * WBY + slot<WBY>(c, r) * 16);
  }
  bool second[C::NJ];  // the lane's columns of sub-tile j lie in the second scale block
#pragma unroll
  for (int j = 0; j < C::NJ; ++j) second[j] = ((t.n0 + wn + 16 * j + 4 * g) >> 7) > nblk0;

  int st = 0;
  for (int it = 0; it < passes; ++it) {
    const int u = ub + it;
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((C::XL + C::WL) * (C::DS - 2)) : "memory");
    // every wave is done with the stage of unit u - 1 and has its share of
    // unit u in LDS (a lone wave waited for its own reads of unit u - 1)
    if constexpr (C::GW > 1) __builtin_amdgcn_s_barrier();
    issue(st == 0 ? C::DS - 1 : st - 1, u + C::DS - 1);
    if (C::KG == 1 || u < ue) {
      const uint32_t base = ring0 + st * C::STAGE;
      float s0 = 0.0f, s1 = 0.0f;
      if constexpr (C::WB == 1) {
        const int kblk = u * C::KU >> 7;
        const int hi = kblk >> 6, ln = kblk & 63;
        s0 = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(hi ? sc[0][1] : sc[0][0]), ln));
        s1 = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(hi ? sc[1][1] : sc[1][0]), ln));
      }
      u32x4 wq[C::NJ][C::KH], xa[C::MI][C::KS];
      constexpr int RH = C::KS / C::KH;  // steps per W read
      auto w_op = [&](int j, int k) {
        if constexpr (C::WB == 1) {
          const u32x4 q = wq[j][k / RH];
          return k % RH ? widen(q.z, q.w) : widen(q.x, q.y);
        } else {
          return __builtin_bit_cast(v8bf, wq[j][k]);
        }
      };
      const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
      constexpr int GR = C::NJ + RH * C::MI;  // reads per W read group
#pragma unroll
      for (int h = 0; h < C::KH; ++h) {
#pragma unroll
        for (int j = 0; j < C::NJ; ++j) wq[j][h] = lds_read16(base + wr[h] + j * 16 * WBY);
#pragma unroll
        for (int p = 0; p < RH; ++p)
#pragma unroll
          for (int i = 0; i < C::MI; ++i) xa[i][RH * h + p] = lds_read16(base + xr[RH * h + p] + i * 16 * XB);
      }
      f32x4 tt[C::MI][C::NJ];
#pragma unroll
      for (int k = 0; k < C::KS; ++k) {
        lds_wait_c((C::KH - 1 - k / RH) * GR + (RH - 1 - k % RH) * C::MI);
#pragma unroll
        for (int i = 0; i < C::MI; ++i) settle(xa[i][k]);
        if (k % RH == 0) {
#pragma unroll
          for (int j = 0; j < C::NJ; ++j) settle(wq[j][k / RH]);
        }
#pragma unroll
        for (int j = 0; j < C::NJ; ++j) {
          const v8bf w8 = w_op(j, k);
#pragma unroll
          for (int i = 0; i < C::MI; ++i) {
            const v8bf x8 = __builtin_bit_cast(v8bf, xa[i][k]);
            if constexpr (C::WB == 1)
              tt[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w8, x8, k == 0 ? zero : tt[i][j], 0, 0, 0);
            else
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w8, x8, acc[i][j], 0, 0, 0);
          }
        }
      }
      if constexpr (C::WB == 1) {
#pragma unroll
        for (int j = 0; j < C::NJ; ++j) {
          const float s = second[j] ? s1 : s0;
#pragma unroll
          for (int i = 0; i < C::MI; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = fmaf(tt[i][j][e], s, acc[i][j][e]);
        }
      }
    }
    st = st == C::DS - 1 ? 0 : st + 1;
  }
  // no load may still be writing this workgroup's LDS when it is reused or given back
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
}

// Meets the K groups' sums and hands the tile to put(m, n, v): four
// consecutive columns n .. n + 3 of row m of the tile (n % 4 == 0), for every
// m < rows_m and n < rows_n.
template <typename C, typename F>
__device__ __forceinline__ void finish(const Work& t, uint8_t* smem, f32x4 (&acc)[C::MI][C::NJ], F put) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wv / C::GW, gw = wv % C::GW;
  const int wm = (gw / C::WN) * 16 * C::MI, wn = (gw % C::WN) * 16 * C::NJ;
  const int r = lane & 15, g = lane >> 4;
  constexpr int LD = C::BN + 4;
  float* slab = (float*)smem;
  if constexpr (C::KG <= 2) {
    if constexpr (C::KG == 2) {
      __syncthreads();  // both groups are done with their rings (every load was waited for)
      if (grp == 1) {
#pragma unroll
        for (int i = 0; i < C::MI; ++i)
#pragma unroll
          for (int j = 0; j < C::NJ; ++j) *(f32x4*)(slab + (wm + 16 * i + r) * LD + wn + 16 * j + 4 * g) = acc[i][j];
      }
      __syncthreads();
      if (grp == 1) return;
    }
#pragma unroll
    for (int i = 0; i < C::MI; ++i) {
      const int m = wm + 16 * i + r;
#pragma unroll
      for (int j = 0; j < C::NJ; ++j) {
        const int n = wn + 16 * j + 4 * g;
        f32x4 v = acc[i][j];
        if constexpr (C::KG == 2) v += *(const f32x4*)(slab + m * LD + n);
        if (m < t.rows_m && n < t.rows_n) put(m, n, v);
      }
    }
  } else {
    __syncthreads();
    float* mine = slab + grp * (C::SLAB / 4);
#pragma unroll
    for (int i = 0; i < C::MI; ++i)
#pragma unroll
      for (int j = 0; j < C::NJ; ++j) *(f32x4*)(mine + (wm + 16 * i + r) * LD + wn + 16 * j + 4 * g) = acc[i][j];
    __syncthreads();
    for (int q = tid; q < C::BM * C::BN / 4; q += C::THREADS) {
      const int m = q / (C::BN / 4), n = (q % (C::BN / 4)) * 4;
      if (m >= t.rows_m || n >= t.rows_n) continue;
      f32x4 v = *(const f32x4*)(slab + m * LD + n);
#pragma unroll
      for (int z = 1; z < C::KG; ++z) v += *(const f32x4*)(slab + z * (C::SLAB / 4) + m * LD + n);
      put(m, n, v);
    }
  }
}

// Rows first, first + step, .. < n of a wave's sub-tile (LR elements apart in
// LDS) to y: ld(row) reads the lane's value, put(row pointer, value) stores it.
// Eight reads ahead of their stores.
template <typename L, typename P>
__device__ __forceinline__ void copy_rows(int first, int step, int n, uint16_t* y, int ldy, L ld, P put) {
  int i = first;
  for (; i + 7 * step < n; i += 8 * step) {
    uint32_t v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = ld(i + k * step);
#pragma unroll
    for (int k = 0; k < 8; ++k) put(y + (size_t)(i + k * step) * ldy, v[k]);
  }
  for (; i < n; i += step) put(y + (size_t)i * ldy, ld(i));
}

// The tile as bf16 rows of y (the tile's first element; row stride ldy).  Rows
// whose 4-column groups are 8-byte aligned take one store per group straight
// from the accumulators.  Other rows (ldy % 4 != 0) would need four 2-byte
// stores per group, each over 16 rows of 32 bytes; with one or two K groups
// each wave turns its sub-tile into rows through LDS instead and stores
// aligned pairs of columns, consecutive lanes consecutive pairs, with the
// lanes chosen once for all rows that start on an odd element and once for the
// others: a lone wave issues an instruction per 5 cycles, so a test per row
// costs as much as the stores.  3153 x 5003 x 640 on 128 x 256 tiles: 48.0 us
// with 2-byte stores, 44 with a test per row, 34.9 now (5004 columns: 29.5);
// 3153 x 5003 x 2560: 96 -> 85 (79).
template <typename C>
__device__ __forceinline__ void store_rows(const Work& t, uint8_t* smem, f32x4 (&acc)[C::MI][C::NJ], uint16_t* y,
                                           int ldy) {
  const bool vec = ldy % 4 == 0 && (uintptr_t)y % 8 == 0;
  if constexpr (C::KG <= 2) {
    if (!vec) {
      constexpr int W = 16 * C::NJ, LR = W + 4, H = 16 * C::MI;  // the sub-tile, and its row in LDS
      static_assert((C::KG == 2 ? C::SLAB : 0) + C::GW * H * LR * 2 <= C::LDS && H % 8 == 0, "staged rows");
      const int lane = threadIdx.x & 63;
      const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
      const int wm = (wv / C::WN) * H, wn = (wv % C::WN) * W;
      uint16_t* rows = (uint16_t*)(smem + (C::KG == 2 ? C::SLAB : 0)) + wv * H * LR;
      if constexpr (C::KG == 1) __syncthreads();  // every wave is done with the ring
      finish<C>(t, smem, acc, [&](int m, int n, f32x4 v) {
        *(u32x2*)(rows + (m - wm) * LR + n - wn) = u32x2{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
      });
      if (C::KG == 2 && wv >= C::GW) return;
      const int nr = min(t.rows_m - wm, H), nc = min(t.rows_n - wn, W);
      if (nr <= 0 || nc <= 0) return;
      asm volatile("" ::: "memory");  // the wave's own rows, in order through LDS
      uint16_t* yw = y + (size_t)wm * ldy + wn;
      const int odd0 = (int)((uintptr_t)yw >> 1) & 1, step = 1 + (ldy & 1);
      const uint16_t* mine = rows + 2 * min(lane, W / 2);
      for (int f = 0; f < step; ++f) {
        if (odd0 ^ f) {  // rows that start on an odd element: pairs (2 lane - 1, 2 lane)
          if (lane > 0 && 2 * lane < nc)
            copy_rows(f, step, nr, yw, ldy,
                      [&](int i) {
                        const uint16_t* r = mine + i * LR;
                        return __builtin_amdgcn_alignbyte(*(const uint32_t*)r, *(const uint32_t*)(r - 2), 2);
                      },
                      [&](uint16_t* d, uint32_t v) { *(uint32_t*)(d + 2 * lane - 1) = v; });
          if (lane == 0 || 2 * lane == nc) {  // the first column, and a last one without a partner
            const int c = lane ? nc - 1 : 0;
            copy_rows(f, step, nr, yw, ldy, [&](int i) { return (uint32_t)rows[i * LR + c]; },
                      [&](uint16_t* d, uint32_t v) { d[c] = (uint16_t)v; });
          }
        } else {  // pairs (2 lane, 2 lane + 1)
          if (2 * lane + 1 < nc)
            copy_rows(f, step, nr, yw, ldy, [&](int i) { return *(const uint32_t*)(mine + i * LR); },
                      [&](uint16_t* d, uint32_t v) { *(uint32_t*)(d + 2 * lane) = v; });
          if (2 * lane + 1 == nc)
            copy_rows(f, step, nr, yw, ldy, [&](int i) { return (uint32_t)rows[i * LR + 2 * lane]; },
                      [&](uint16_t* d, uint32_t v) { d[2 * lane] = (uint16_t)v; });
        }
      }
      return;
    }
  }
  finish<C>(t, smem, acc, [&](int m, int n, f32x4 v) {
    uint16_t* d = y + (size_t)m * ldy + n;
    if (vec) {
      *(u32x2*)d = u32x2{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (n + c < t.rows_n) d[c] = f2bf(v[c]);
    }
  });
}

}  // namespace qh_tile
