// Coded dense GEMM on the matrix cores (prefill / many rows):
//   mid[M][OC] f32 = xh[M][IC] f16 @ decode(code[IC/16][OC/16][8K]).
// Replaces msl.dense_gemm_mat (escha_mlx/msl.py:1608-1782), the reference's
// R=16 simdgroup-matrix GEMM.  Tolerance contract, as there: every decoded
// weight is the bit-exact f16 of the format, f16 x f16 products are exact in
// the f32 accumulator, and only the order of the f32 sum differs from the
// scalar kernels.  The result is deterministic run to run.
#pragma once

#include "fast.hpp"

namespace esc {

// Raw buffer resource over [p, p + bytes) (gfx9 descriptor word 3); loads
// through it take a scalar base and a 32-bit lane offset, and read zero past
// the end instead of faulting.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* p, size_t bytes) {
  const int n = bytes > 0xFFFFFFF0u ? (int)0xFFFFFFF0u : (int)bytes;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, n, 0x00020000);
}

// Coded GEMM with the weights decoded straight into MFMA A operands (no LDS
// for weights): mid[M][OC] f32 = xh[M][IC] f16 @ decode(code).  OC an odd
// multiple of 128: the last column block's waves 2 and 3 run tiles clamped into
// the stream and store nothing.
//
// Block = 4 waves, tile 16*NRB rows x 256 columns (16 code tiles); wave w owns
// tiles 4w..4w+3 (64 columns).  K is walked in steps of 4 kt (64 inputs):
//   * each lane decodes its tile-lane of the wave-step (mma_a_operand: 4
//     column groups x 2 input halves = 8 A operands, v_mfma_f32_16x16x32_f16
//     layout, one kt per 16 lanes), so each weight is decoded once per block;
//   * X: the block's rows x 64 inputs are staged through LDS (double
//     buffered, 16-byte chunks XOR-swizzled by row); a B operand is one
//     16-byte read (16 rows x 8 inputs of one kt per 16 lanes) and feeds the
//     4 A operands of its input half;
//   * each A operand meets NRB row blocks: 8 * NRB MFMAs per wave-step, in
//     one straight-line body with the decode of the next wave-step, so the
//     matrix pipe and the VALU overlap (two workgroups per CU).
// The kernel is decode-bound: the host picks NRB for the shape.
// D register r of lane l: output column of tile-lane 4(l/16) + r, row l%16 of
// the row block.
template <int K, int NRB>
struct Mma2 {
  using G = Geo<K>;
  static constexpr int TPS = 16 / G::LPT, GPW = 4 / TPS, NA = GPW * G::NCOL;
  static_assert(NA == 4, "four 16-column groups per wave");
  static_assert(NRB % 2 == 0 && NRB >= 2 && NRB <= 8, "whole x chunks per thread, 2 waves/SIMD");
  static constexpr int BR = 16 * NRB;            // rows per block
  static constexpr int XCH = BR * 8 / 256;       // 16-byte x chunks per thread per stage
};

// Byte offset of the workgroup's x chunk j of thread tid from the start of
// its row: chunk e = tid + 256j of a stage is row e/8, logical chunk
// (e%8)^(row&7) = kt (lc/2) half (lc%2), 128 bytes per row per stage.
__device__ __forceinline__ int mma2_x_row(int tid, int j) { return (tid + 256 * j) >> 3; }
__device__ __forceinline__ uint32_t mma2_x_chunk(int tid, int j) {
  const int e = tid + 256 * j;
  return 16u * ((e & 7) ^ ((e >> 3) & 7));
}

// Where the main loop's A operands come from: 64 columns x 64 inputs a step, as
// four 16-column groups of two operands each (input halves; lane l: column
// l % 16, inputs 16 (l / 16) + 8 half ..).  Coded weights: cbase is the lane's
// code words of the wave's first tile at kt gk (lane / 16).
template <int K>
struct CodedCols {
  using G = Geo<K>;
  static constexpr int TPS = 16 / G::LPT, GPW = 4 / TPS;
  struct Regs {
    LaneWords<K> w[GPW];
  };
  const uint32_t* cbase;
  size_t kstride;
  __device__ __forceinline__ void load(Regs& r, int s) const {
#pragma unroll
    for (int tg = 0; tg < GPW; ++tg)
      r.w[tg] = load_lane_words<K>(cbase + (size_t)tg * TPS * (8 * K) + (size_t)(4 * s) * kstride);
  }
  __device__ __forceinline__ void decode(const Regs& r, u32x4_t (*Ad)[2]) const {
    const int lane = threadIdx.x & 63;
    const int src = (lane & ~(G::LPT - 1)) | ((lane + G::LPT - 1) & (G::LPT - 1));
#pragma unroll
    for (int tg = 0; tg < GPW; ++tg) {
      const uint32_t wprev = __shfl(r.w[tg].w[G::WPL - 1], src);
#pragma unroll
      for (int ci = 0; ci < G::NCOL; ++ci)
#pragma unroll
        for (int P = 0; P < 2; ++P)
          Ad[tg * G::NCOL + ci][P] = mma_a_operand<K>(r.w[tg], wprev, ci, P);
    }
  }
};

// The main loop over steps [s0, s1) (s1 > s0): acc[a][r] += the wave's 64
// columns x row block r, of the first NACT row blocks (even; the others: zero).
// xoff: byte offsets of the thread's x chunks.
template <int NRB, int NACT = NRB, typename Cols>
__device__ __forceinline__ void mma2_loop(const Cols& cols, __amdgpu_buffer_rsrc_t xrs,
                                          const uint32_t* xoff, int s0, int s1,
                                          uint4 (*s_x)[16 * NRB * 8], f32x4_t (*acc)[NRB]) {
  constexpr int NA = 4, XCH = NACT / 2;
  const int tid = threadIdx.x, lane = tid & 63;
  const int gk = lane >> 4, c = lane & 15;
  auto load_x = [&](uint4* xr, int s) {
#pragma unroll
    for (int j = 0; j < XCH; ++j) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(xrs, xoff[j], 128u * s, 0);
      xr[j] = make_uint4(v[0], v[1], v[2], v[3]);
    }
  };
  auto store_x = [&](const uint4* xr, int buf) {
#pragma unroll
    for (int j = 0; j < XCH; ++j) s_x[buf][tid + 256 * j] = xr[j];
  };
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int r = 0; r < NRB; ++r) acc[a][r] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // software pipeline: the MFMAs of step s and the decode of step s+1 sit in
  // one straight-line body (the matrix pipe and the VALU overlap); loads past
  // the last step re-read it (in bounds, never used)
  typename Cols::Regs cw;
  uint4 xr[XCH];
  u32x4_t A[NA][2];
  cols.load(cw, s0);
  load_x(xr, s0);
  store_x(xr, 0);
  cols.decode(cw, A);
  cols.load(cw, min(s0 + 1, s1 - 1));
  lds_barrier();
  for (int s = s0; s < s1; ++s) {
    const int buf = (s - s0) & 1;
    load_x(xr, min(s + 1, s1 - 1));
    typename Cols::Regs cn;
    cols.load(cn, min(s + 2, s1 - 1));
    u32x4_t An[NA][2];
#pragma unroll
    for (int P = 0; P < 2; ++P)
#pragma unroll
      for (int r = 0; r < NACT; ++r) {
        const uint4 bv = s_x[buf][(16 * r + c) * 8 + ((2 * gk + P) ^ (c & 7))];
        const u32x4_t b = __builtin_bit_cast(u32x4_t, bv);
#pragma unroll
        for (int a = 0; a < NA; ++a) acc[a][r] = mma16(A[a][P], b, acc[a][r]);
      }
    cols.decode(cw, An);
    store_x(xr, buf ^ 1);
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      A[a][0] = An[a][0];
      A[a][1] = An[a][1];
    }
    cw = cn;
    lds_barrier();
  }
}

// ---- the 128-point transform of a row block in the accumulators' layout.
// A 128-column block is two waves' 64 columns.  Lane l holds, for row l % 16,
// 16 of its wave's columns in registers and the other columns sit in the lanes
// l ^ 16, l ^ 32, so four butterfly stages are plain adds, two exchange
// registers with another lane (v_permlane16_swap / v_permlane32_swap, which
// swap a pair of registers' halves: the butterfly then pairs registers, and the
// register bit and the lane bit have traded columns) and one exchanges half of
// the registers with the other wave through LDS.  Stages run from column bit 0
// up, each a + b and a - b of the same operands as h128_wave: bit-identical to
// it.  Against transposing each row to one wave (16 scattered LDS writes and
// h128_wave's 60 instructions per row and 128 columns) this is about a third
// of the VALU and a quarter of the LDS traffic.
template <int BIT, int N>
__device__ __forceinline__ void bfly_reg(float (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (!(i & BIT)) {
      const float a = v[i], b = v[i | BIT];
      v[i] = a + b;
      v[i | BIT] = a - b;
    }
}
// column bit of lane bit 4 (X16) or 5, traded with the register bit BIT
template <int BIT, bool X16, int N>
__device__ __forceinline__ void bfly_lane(float (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (!(i & BIT)) {
      const unsigned x = __builtin_bit_cast(unsigned, v[i]);
      const unsigned y = __builtin_bit_cast(unsigned, v[i | BIT]);
      unsigned lo, hi;
      if constexpr (X16) {
        const auto p = __builtin_amdgcn_permlane16_swap(x, y, false, false);
        lo = p[0], hi = p[1];
      } else {
        const auto p = __builtin_amdgcn_permlane32_swap(x, y, false, false);
        lo = p[0], hi = p[1];
      }
      const float a = __builtin_bit_cast(float, lo), b = __builtin_bit_cast(float, hi);
      v[i] = a + b;
      v[i | BIT] = a - b;
    }
}

// The first six stages of one row block's 64 columns.  v[8h + j] is then column
// 32h + 8 chunk + j, chunk = mma2_chunk<K>().
template <int K>
__device__ __forceinline__ int mma2_chunk() {
  const int g = (threadIdx.x & 63) >> 4;
  return K == 2 ? g : 2 * (g & 1) + (g >> 1);
}
template <int K, int NRB>
__device__ __forceinline__ void mma2_h64(const f32x4_t (*acc)[NRB], int r, float (&v)[16]) {
  if constexpr (K == 2) {
    // register index = column % 16 (acc slot ci: bits 0 and 3, D register:
    // bits 1, 2); lane bit 4: column bit 4, lane bit 5: column bit 5
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = acc[(i & 1) + 2 * (i >> 3)][r][(i >> 1) & 3];
    bfly_reg<1>(v);
    bfly_reg<2>(v);
    bfly_reg<4>(v);
    bfly_reg<8>(v);
    bfly_lane<8, true>(v);   // register bit 3: column bit 4, lane bit 4: 3
    bfly_lane<8, false>(v);  // register bit 3: column bit 5, lane bit 5: 4
  } else {
    // register index: column bits 0, 1 (D register), 3 (ci), 5 (tile group);
    // lane bit 4: column bit 2, lane bit 5: column bit 4
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = acc[2 * (i >> 3) + ((i >> 2) & 1)][r][i & 3];
    bfly_reg<1>(v);
    bfly_reg<2>(v);
    bfly_lane<4, true>(v);   // register bit 2: column bit 2, lane bit 4: 3
    bfly_lane<8, true>(v);   // register bit 3: column bit 3, lane bit 4: 5
    bfly_lane<8, false>(v);  // register bit 3: column bit 4, lane bit 5: 3
    bfly_lane<8, true>(v);   // register bit 3: column bit 5, lane bit 4: 4
  }
}

// a or b by value (a conditional between two array elements selects their
// address, which keeps the array in memory)
template <typename T>
__device__ __forceinline__ T pick(bool first, T a, T b) {
  return first ? a : b;
}

// The last stage (column bit 6, the other wave of the pair): wave hw finishes
// the columns of v[8 hw ..], o[8b + j] = column 64b + 32hw + 8 chunk + j.  buf:
// the workgroup's exchange area, float4 [4 waves][2][64 lanes]; the caller
// keeps a barrier between two uses of one area.
constexpr int kMma2Xch = 4 * 2 * 64;  // float4 per exchange area
__device__ __forceinline__ void mma2_h128_last(const float (&v)[16], float4* buf, float (&o)[16]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const bool hw = wave & 1;
  float m[8], t[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    m[j] = pick(hw, v[8 + j], v[j]);
    t[j] = pick(hw, v[j], v[8 + j]);
  }
  float4* w = buf + wave * 128 + lane;
  w[0] = make_float4(t[0], t[1], t[2], t[3]);
  w[64] = make_float4(t[4], t[5], t[6], t[7]);
  lds_barrier();
  const float4* p = buf + (wave ^ 1) * 128 + lane;
  const float4 p0 = p[0], p1 = p[64];
  const float q[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float a = pick(hw, q[j], m[j]), b = pick(hw, m[j], q[j]);
    o[j] = a + b;
    o[8 + j] = a - b;
  }
}

// Output columns h[0..7] at element i, h[8..15] at i + 64 of y, whose element
// type is ydt (kRowsF16 / kRowsBF16 / kRowsF32: the f16 value converted).
__device__ __forceinline__ void mma2_store16(void* y, int ydt, size_t i, const half_t* h) {
  if (ydt == kRowsF32) {
    float* d = static_cast<float*>(y) + i;
#pragma unroll
    for (int j = 0; j < 16; j += 4)
      *reinterpret_cast<float4*>(d + 64 * (j >> 3) + (j & 7)) =
          make_float4((float)h[j], (float)h[j + 1], (float)h[j + 2], (float)h[j + 3]);
    return;
  }
  uint32_t w[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) w[j] = pack2(h[2 * j], h[2 * j + 1]);
  if (ydt == kRowsBF16) {
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = pack2_bf16((float)h[2 * j], (float)h[2 * j + 1]);
  }
  uint16_t* d = static_cast<uint16_t*>(y) + i;
  *reinterpret_cast<uint4*>(d) = make_uint4(w[0], w[1], w[2], w[3]);
  *reinterpret_cast<uint4*>(d + 64) = make_uint4(w[4], w[5], w[6], w[7]);
}

// The output transform of one row block in the accumulators' layout and its
// store: y = (bias +) f16((H128(row) * rs) * ro), ro[8b + j] (and bias) of
// columns col + 64b + j.
template <int K, int NRB>
__device__ __forceinline__ void mma2_out(const f32x4_t (*acc)[NRB], int r, float4* buf, float rs,
                                         const float* ro, const uint16_t* bias, int col, bool ok,
                                         void* y, int ydt, size_t i) {
  float v[16], o[16];
  mma2_h64<K, NRB>(acc, r, v);
  mma2_h128_last(v, buf, o);
  half_t h[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) h[j] = to_f16((o[j] * rs) * ro[j]);
  if (bias) {
#pragma unroll
    for (int j = 0; j < 16; ++j)
      h[j] = to_f16((float)h[j] +
                    (float)__builtin_bit_cast(half_t, bias[col + 64 * (j >> 3) + (j & 7)]));
  }
  if (ok) mma2_store16(y, ydt, i, h);
}

// What the main loop's sums become (MODE):
//   kMmaMid  mid[M][OC] f32;
//   kMmaOut  y = the output transform in the epilogue, in the accumulators'
//            layout (the formula and rounding of k_output_transform, bit-identical
//            to it); mid is not written;
//   kMmaPart the partial sums of split z = blockIdx.y of gridDim.y (steps
//            [z NS / S, (z + 1) NS / S)), as k_mma2_reduce reads them: one
//            float4 per lane and accumulator, 16 KiB per (split, 16-row block,
//            column block), row blocks past M not written.
enum { kMmaMid = 0, kMmaOut = 1, kMmaPart = 2 };

struct MmaArgs {
  const uint16_t* xh;
  const uint32_t* code;
  int M, TK, TN;
  float* mid;          // kMmaMid / kMmaPart
  const float* rout;   // kMmaOut
  const uint16_t* bias;
  float rs;
  void* y;
  int ydt;
};

// float4 index of accumulator a, lane 0 of a partial slice
__device__ __forceinline__ size_t mma2_part_index(int z, int rb16, int nrb16, int cb, int ncb,
                                                  int wave, int a) {
  return ((((size_t)z * nrb16 + rb16) * ncb + cb) * 4 + wave) * 256 + 64 * a;
}

// Two products of the same rows and splits may share a launch (p1 from workgroup
// n0 on): gate and up of 2048 rows hold 4.25 tiles per CU each, 8.5 together, and
// a launch takes what its busiest CU holds.
template <int K, int NRB, int MODE>
__global__ __launch_bounds__(256, 2) void k_gemm_mma2(MmaArgs p0, MmaArgs p1, int n0) {
  using G = Geo<K>;
  using D = Mma2<K, NRB>;
  constexpr int TPS = D::TPS, GPW = D::GPW, NA = D::NA, BR = D::BR, XCH = D::XCH;
  __shared__ uint4 s_x[2][BR * 8];        // [stage][row][chunk ^ (row & 7)]

  const bool second = (int)blockIdx.x >= n0;
  const MmaArgs p = second ? p1 : p0;
  const int b = second ? (int)blockIdx.x - n0 : (int)blockIdx.x;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int M = p.M, TK = p.TK, TN = p.TN;
  const int IC = TK * 16, OC = TN * 16;
  const int ncb = (TN + 15) / 16;
  int rb, cb;
  if (ncb % 8 == 0) {
    const int per = ncb / 8, qq = b / 8, x = b % 8;
    rb = qq / per;
    cb = 8 * (qq % per) + x;
  } else {
    rb = b / ncb;
    cb = b % ncb;
  }
  const int row0 = rb * BR;
  int tile0 = cb * 16 + 4 * wave;
  const bool live = tile0 < TN;
  if (!live) tile0 = TN - 4;
  const int gk = lane >> 4, c = lane & 15, tc = c / G::LPT, q = lane % G::LPT;

  // code: tile group tg of the wave, lane's kt = 4s + gk
  const size_t kstride = (size_t)TN * (8 * K);
  const uint32_t* cbase = p.code + (size_t)(tile0 + tc) * (8 * K) + q * G::WPL + gk * kstride;
  uint32_t xoff[XCH];
#pragma unroll
  for (int j = 0; j < XCH; ++j)
    xoff[j] = 2u * ((uint32_t)min(row0 + mma2_x_row(tid, j), M - 1) * IC) + mma2_x_chunk(tid, j);
  const __amdgpu_buffer_rsrc_t xrs = buf_rsrc(p.xh, (size_t)M * IC * 2);
  const int NS = TK / 4;
  int s0 = 0, s1 = NS;
  if constexpr (MODE == kMmaPart) {
    s0 = NS * (int)blockIdx.y / (int)gridDim.y;
    s1 = NS * ((int)blockIdx.y + 1) / (int)gridDim.y;
  }
  f32x4_t acc[NA][NRB];
  mma2_loop<NRB>(CodedCols<K>{cbase, kstride}, xrs, xoff, s0, s1, s_x, acc);

  if constexpr (MODE == kMmaMid) {
#pragma unroll
    for (int r = 0; r < NRB; ++r) {
      const int row = row0 + 16 * r + c;
      if (row < M && live) {
#pragma unroll
        for (int tg = 0; tg < GPW; ++tg) {
          f32x4_t t[G::NCOL];
#pragma unroll
          for (int ci = 0; ci < G::NCOL; ++ci) t[ci] = acc[tg * G::NCOL + ci][r];
          mma_store<K>(t, gk, p.mid + (size_t)row * OC + 16 * (tile0 + TPS * tg));
        }
      }
    }
  } else if constexpr (MODE == kMmaPart) {
    const int nrb16 = (M + 15) / 16;
    f32x4_t* part = reinterpret_cast<f32x4_t*>(p.mid);
#pragma unroll
    for (int r = 0; r < NRB; ++r)
      if (row0 + 16 * r < M) {
#pragma unroll
        for (int a = 0; a < NA; ++a)
          part[mma2_part_index(blockIdx.y, rb * NRB + r, nrb16, cb, ncb, wave, a) + lane] =
              acc[a][r];
      }
  } else {
    // two exchange areas, one per row-block parity: over x's stages (unused
    // since the loop's last barrier) where they fit
    static_assert(sizeof(s_x) >= 2 * kMma2Xch * sizeof(float4) || NRB < 4, "");
    __shared__ float4 s_o[NRB < 4 ? 2 * kMma2Xch : 1];
    float4* so = NRB < 4 ? s_o : reinterpret_cast<float4*>(&s_x[0][0]);
    // this lane's 16 columns: col + 64b + j (b = 0, 1; j = 0..7)
    const int col = live ? 256 * cb + 128 * (wave >> 1) + 32 * (wave & 1) + 8 * mma2_chunk<K>() : 0;
    float ro[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) ro[j] = p.rout[col + 64 * (j >> 3) + (j & 7)];
#pragma unroll
    for (int r = 0; r < NRB; ++r) {
      const int row = row0 + 16 * r + c;
      mma2_out<K, NRB>(acc, r, so + (r & 1) * kMma2Xch, p.rs, ro, p.bias, col, row < M && live,
                       p.y, p.ydt, (size_t)row * OC + col);
    }
  }
}

// The sum of S splits' partials (kMmaPart) in split order, then the output
// transform and store of k_gemm_mma2's epilogue.  One workgroup per (column
// block, 16 rows): each wave reads its slices back as it wrote them (1 KiB
// contiguous per accumulator), 8 splits' loads in flight.  Latency-bound: 40
// rows x 5120 columns in 24 splits, 20 MB.  grid (ncb, ceil(M / 16)), block 256.
template <int K>
__global__ __launch_bounds__(256) void k_mma2_reduce(MmaArgs p, int S) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int OC = p.TN * 16, cb = blockIdx.x, ncb = gridDim.x, rb16 = blockIdx.y;
  const int nrb16 = gridDim.y;
  __shared__ float4 s_o[kMma2Xch];
  const bool live = cb * 16 + 4 * wave < p.TN;
  const int col = live ? 256 * cb + 128 * (wave >> 1) + 32 * (wave & 1) + 8 * mma2_chunk<K>() : 0;
  const f32x4_t* part = reinterpret_cast<const f32x4_t*>(p.mid) +
                        mma2_part_index(0, rb16, nrb16, cb, ncb, wave, 0) + lane;
  const size_t zs = mma2_part_index(1, 0, nrb16, 0, ncb, 0, 0);
  f32x4_t acc[4][1];
#pragma unroll
  for (int a = 0; a < 4; ++a) acc[a][0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int z0 = 0; z0 < S; z0 += 8) {
    // splits past the last one re-read it and add +0 (a sum from +0 is never -0)
    f32x4_t v[8][4];
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int a = 0; a < 4; ++a) v[j][a] = part[min(z0 + j, S - 1) * zs + 64 * a];
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[a][0][i] = acc[a][0][i] + (z0 + j < S ? v[j][a][i] : 0.f);
  }
  float ro[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) ro[j] = p.rout[col + 64 * (j >> 3) + (j & 7)];
  const int row = 16 * rb16 + (lane & 15);
  mma2_out<K, 1>(acc, 0, s_o, p.rs, ro, p.bias, col, row < p.M && live, p.y, p.ydt,
                 (size_t)row * OC + col);
}

}  // namespace esc
