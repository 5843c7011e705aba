// Dense int8 / f16 GEMV around the routed experts: the w8a16 linears of the
// shared expert and the vocabulary head (escha_mlx/quant.py:1-30, contract
// wf = f16(f32(w8) * f32(scale)), y = f16(f32-accumulated x @ wf^T); CPU
// statement ref.w8a16, escha_mlx/ref.py:308-311), and the f16 router /
// shared-expert gates (y = f16(x @ w^T), escha_mlx/models/qwen3_5_moe.py:257-273).
//
// Weights are [O][K] row-major (one output channel per row), read once from
// HBM with 16-byte loads: LPR lanes share a row (the chunk count rounded up to
// a power of two, at most 64), each owning up to CPL 16-byte chunks of it, so
// a wave-step covers 64/LPR rows.  The
// lane's inputs for its chunks (NR rows of x) stay in VGPRs for the whole
// launch; the rows' partial sums meet through lane exchanges (DPP / permlane).
// Each weight is rounded exactly as the contract says (int8 -> f32, one fma
// with the row scale, RNE to f16) before the f16 x f16 products, which
// v_dot2c_f32_f16 sums in float32 (tolerance contract: reassociated sum).
#pragma once

#include "basic.hpp"
#include "mfma.hpp"

namespace esc {

// partial sum of the lanes of one row group (LPR lanes, LPR a power of two)
template <int LPR>
__device__ __forceinline__ float row_sum(float v) {
  if constexpr (LPR >= 2) v = v + lane_xor<1>(v);
  if constexpr (LPR >= 4) v = v + lane_xor<2>(v);
  if constexpr (LPR >= 8) v = v + lane_xor<4>(v);
  if constexpr (LPR >= 16) v = v + lane_xor<8>(v);
  if constexpr (LPR >= 32) {
    const unsigned x = __builtin_bit_cast(unsigned, v);
    const auto p = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    const unsigned lo = p[0], hi = p[1];
    v = __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
  }
  if constexpr (LPR >= 64) {
    const unsigned x = __builtin_bit_cast(unsigned, v);
    const auto p = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    const unsigned lo = p[0], hi = p[1];
    v = __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
  }
  return v;
}

// 4 int8 weights (one word) -> two packed f16 pairs per the w8a16 contract:
// f32(w8) * f32(scale), RNE to f16.  q = w8 ^ 0x80 is the unsigned byte w8 + 128,
// and fma(q, s, -128 s) rounds the exact (q - 128) * s once, as the product does.
__device__ __forceinline__ void w8_to_f16x4(uint32_t w, float s, float ms, uint32_t& p0,
                                            uint32_t& p1) {
  const uint32_t q = w ^ 0x80808080u;
  const float f0 = __builtin_fmaf((float)(q & 0xFFu), s, ms);
  const float f1 = __builtin_fmaf((float)((q >> 8) & 0xFFu), s, ms);
  const float f2 = __builtin_fmaf((float)((q >> 16) & 0xFFu), s, ms);
  const float f3 = __builtin_fmaf((float)(q >> 24), s, ms);
  p0 = pack2(to_f16(f0), to_f16(f1));
  p1 = pack2(to_f16(f2), to_f16(f3));
}

// y[m][o] (ldy between rows) for m < M <= NR.  Q8: w is int8 [O][K] with
// scale [O]; otherwise w is f16 [O][K] and scale unused.  The row's `chunks`
// 16-byte pieces are spread over LPR lanes x CPL pieces each.  A lane's piece
// sub + LPR*j beyond the row (chunks not a multiple of LPR) has zero inputs
// and reads the row's last piece instead, so every weight load stays
// unconditional; int8 weights convert to finite values, whose products with
// the zero inputs add +0, while f16 weights (which may hold Inf) are replaced
// by zeros.  grid: any; block 256.
template <bool Q8, int NR, int LPR, int CPL>
__global__ __launch_bounds__(256) void k_rows_gemv(const uint16_t* __restrict__ x,
                                                   const void* __restrict__ wv,
                                                   const float* __restrict__ scale, int M, int K,
                                                   int O, uint16_t* __restrict__ y, int ldy) {
  constexpr int RPS = 64 / LPR;                  // rows per wave-step
  constexpr int WB = Q8 ? 1 : 2;                 // bytes per weight
  constexpr int CW = 16 / WB;                    // weights per 16-byte chunk
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int sub = lane % LPR, rsel = lane / LPR;
  const int chunks = K / CW;
  bool has[CPL];
  int coff[CPL];  // byte offset of the lane's piece j within a weight row
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    has[j] = sub + LPR * j < chunks;
    coff[j] = min(sub + LPR * j, chunks - 1) * 16;
  }
  // the lane's inputs: NR rows x CPL chunks x CW halves, as f16 pairs
  uint32_t xr[NR][CPL][CW / 2];
#pragma unroll
  for (int m = 0; m < NR; ++m)
#pragma unroll
    for (int j = 0; j < CPL; ++j)
#pragma unroll
      for (int i = 0; i < CW / 2; ++i) xr[m][j][i] = 0u;
#pragma unroll
  for (int m = 0; m < NR; ++m) {
    if (m >= M) break;
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      if (!has[j]) continue;
      const uint16_t* xp = x + (size_t)m * K + (size_t)(sub + LPR * j) * CW;
#pragma unroll
      for (int i = 0; i < CW / 8; ++i) {
        const uint4 v = *reinterpret_cast<const uint4*>(xp + 8 * i);
        xr[m][j][4 * i] = v.x;
        xr[m][j][4 * i + 1] = v.y;
        xr[m][j][4 * i + 2] = v.z;
        xr[m][j][4 * i + 3] = v.w;
      }
    }
  }
  const uint8_t* w8 = reinterpret_cast<const uint8_t*>(wv);
  const int nwaves = gridDim.x * 4;
  const int steps = (O + RPS - 1) / RPS;
  // the weights (and scale) of the wave's next step are requested before the
  // current step is converted and multiplied
  auto load_step = [&](int st, uint4* wc, float& s) {
    const int oc = min(st * RPS + rsel, O - 1);  // in-bounds reads for a partial last step
    const uint8_t* row = w8 + (size_t)oc * K * WB;
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      wc[j] = *reinterpret_cast<const uint4*>(row + coff[j]);
      if constexpr (!Q8)
        if (!has[j]) wc[j] = make_uint4(0u, 0u, 0u, 0u);
    }
    if constexpr (Q8) s = scale[oc];
  };
  int st = blockIdx.x * 4 + wave;
  uint4 wn[CPL];
  float sn = 0.f;
  if (st < steps) load_step(st, wn, sn);
  for (; st < steps; st += nwaves) {
    const int o = st * RPS + rsel;
    const bool ok = o < O;
    uint4 wc[CPL];
#pragma unroll
    for (int j = 0; j < CPL; ++j) wc[j] = wn[j];
    const float s = sn, ms = -128.f * sn;
    if (st + nwaves < steps) load_step(st + nwaves, wn, sn);
    float acc[NR];
#pragma unroll
    for (int m = 0; m < NR; ++m) acc[m] = 0.f;
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const uint32_t ww[4] = {wc[j].x, wc[j].y, wc[j].z, wc[j].w};
      uint32_t wp[CW / 2];
      if constexpr (Q8) {
#pragma unroll
        for (int i = 0; i < 4; ++i) w8_to_f16x4(ww[i], s, ms, wp[2 * i], wp[2 * i + 1]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) wp[i] = ww[i];
      }
#pragma unroll
      for (int m = 0; m < NR; ++m)
#pragma unroll
        for (int i = 0; i < CW / 2; ++i) acc[m] = dot2(xr[m][j][i], wp[i], acc[m]);
    }
#pragma unroll
    for (int m = 0; m < NR; ++m) acc[m] = row_sum<LPR>(acc[m]);
    if (ok && sub == 0) {
#pragma unroll
      for (int m = 0; m < NR; ++m)
        if (m < M) y[(size_t)m * ldy + o] = __builtin_bit_cast(uint16_t, to_f16(acc[m]));
    }
  }
}

// w8a16 GEMV for 2..16 rows of x on the matrix core: y[m][o] = f16(sum_k
// x[m][k] * wf[o][k]), wf = f16(f32(w8) * scale[o]) (the contract rounding, as
// k_rows_gemv).  A wave owns 16 output channels at a time and walks all of K in
// steps of 64: lane l reads 16 int8 of channel o0 + l % 16 at k0 + 16 (l / 16),
// converts them, and the two halves are the A operands of two
// v_mfma_f32_16x16x32_f16 (A slot 8g + t <-> k0 + 16g + t, second half +8);
// the B operands are the same k of token l % 16 from x staged in LDS (rows at a
// 16-byte-padded pitch, so the 16 tokens of a lane group hit different banks).
// Every product of a channel lands in one accumulator: no lane reduction.  D
// lane l: token l % 16, channels o0 + 4 (l / 16) + r.  K a multiple of 64;
// dynamic LDS = M x (2K + 16) bytes; grid: any; block 256.
__global__ __launch_bounds__(256) void k_rows_w8_mma(const uint16_t* __restrict__ x,
                                                     const int8_t* __restrict__ w8,
                                                     const float* __restrict__ scale, int M,
                                                     int K, int O, uint16_t* __restrict__ y,
                                                     int ldy) {
  extern __shared__ uint4 s_xm[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int pitch = K / 8 + 1;  // 16-byte units per staged row
  for (int i = threadIdx.x; i < M * (K / 8); i += 256) {
    const int r = i / (K / 8), c = i % (K / 8);
    s_xm[r * pitch + c] = *reinterpret_cast<const uint4*>(x + (size_t)r * K + 8 * c);
  }
  __syncthreads();
  const int j = lane & 15, g = lane >> 4;
  const uint4* xb = s_xm + (size_t)min(j, M - 1) * pitch + 2 * g;  // token j, k0 + 16g
  const int ngroups = (O + 15) / 16, nwaves = gridDim.x * 4;
  for (int grp = blockIdx.x * 4 + wave; grp < ngroups; grp += nwaves) {
    const int oc = min(grp * 16 + j, O - 1);  // in-bounds reads for a partial last group
    const float s = scale[oc], ms = -128.f * s;
    const uint4* wr = reinterpret_cast<const uint4*>(w8 + (size_t)oc * K + 16 * g);
    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto step = [&](const uint4 wc, int k0) {
      u32x4_t a0, a1;
      uint32_t p0, p1;
      w8_to_f16x4(wc.x, s, ms, p0, p1);
      a0[0] = p0;
      a0[1] = p1;
      w8_to_f16x4(wc.y, s, ms, p0, p1);
      a0[2] = p0;
      a0[3] = p1;
      w8_to_f16x4(wc.z, s, ms, p0, p1);
      a1[0] = p0;
      a1[1] = p1;
      w8_to_f16x4(wc.w, s, ms, p0, p1);
      a1[2] = p0;
      a1[3] = p1;
      const uint4 b0 = xb[k0 / 8], b1 = xb[k0 / 8 + 1];
      acc = mma16(a0, __builtin_bit_cast(u32x4_t, b0), acc);
      acc = mma16(a1, __builtin_bit_cast(u32x4_t, b1), acc);
    };
    // two 64-k steps per iteration, the next two requested before these are used
    uint4 n0 = wr[0], n1 = wr[K > 64 ? 4 : 0];
    for (int k0 = 0; k0 < K; k0 += 128) {
      const uint4 c0 = n0, c1 = n1;
      if (k0 + 128 < K) {
        n0 = wr[(k0 + 128) / 16];
        n1 = wr[(k0 + 192 < K ? k0 + 192 : k0 + 128) / 16];
      }
      step(c0, k0);
      if (k0 + 64 < K) step(c1, k0 + 64);
    }
    if (j < M) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int o = grp * 16 + 4 * g + r;
        if (o < O) y[(size_t)j * ldy + o] = __builtin_bit_cast(uint16_t, to_f16(acc[r]));
      }
    }
  }
}

// The A operands of 64 weight rows (channels) x 64 k a step, for k_rows_gemm and
// (as mma2_loop's columns) k_rows_gemm_lds: lane l reads 16 weights of channels
// 16a + l % 16 at k 16 (l / 16), converted per the contract (int8) or as they are.
template <bool Q8>
struct RowCols {
  static constexpr int WL = Q8 ? 1 : 2;  // 16-byte loads per lane, channel and step
  struct Regs {
    uint4 w[4][WL];
  };
  const char* wb;
  uint32_t wo[4];
  float sc[4], ms[4];
  __device__ __forceinline__ void load(Regs& r, int s) const {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int i = 0; i < WL; ++i)
        r.w[a][i] = *reinterpret_cast<const uint4*>(wb + (wo[a] + 64u * WL * s + 16u * i));
  }
  __device__ __forceinline__ void decode(const Regs& r, u32x4_t (*A)[2]) const {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      if constexpr (Q8) {
        const uint32_t ww[4] = {r.w[a][0].x, r.w[a][0].y, r.w[a][0].z, r.w[a][0].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t p0, p1;
          w8_to_f16x4(ww[i], sc[a], ms[a], p0, p1);
          A[a][i >> 1][2 * (i & 1)] = p0;
          A[a][i >> 1][2 * (i & 1) + 1] = p1;
        }
      } else {
        A[a][0] = __builtin_bit_cast(u32x4_t, r.w[a][0]);
        A[a][1] = __builtin_bit_cast(u32x4_t, r.w[a][WL - 1]);
      }
    }
  }
  // channels o0 + 64 wave + 16a + l % 16, clamped to the last one
  __device__ __forceinline__ void init(const void* wv, const float* scale, int o0, int K, int O) {
    const int lane = threadIdx.x & 63;
    wb = static_cast<const char*>(wv) + (size_t)o0 * K * WL;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int oc = min(16 * a + (lane & 15), O - 1 - o0);
      wo[a] = (uint32_t)((oc * K + 16 * (lane >> 4)) * WL);
      sc[a] = 0.f;
      if constexpr (Q8) sc[a] = scale[o0 + oc];
      ms[a] = -128.f * sc[a];
    }
  }
};

// Four consecutive channels o .. o + 3 of one row (f16).
__device__ __forceinline__ void rows_store4(uint16_t* y, int row, int o, int O, const f32x4_t& v) {
  uint16_t* d = y + (size_t)row * O + o;
  if (o + 3 < O && O % 4 == 0) {
    *reinterpret_cast<uint2*>(d) =
        make_uint2(pack2(to_f16(v[0]), to_f16(v[1])), pack2(to_f16(v[2]), to_f16(v[3])));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (o + i < O) d[i] = __builtin_bit_cast(uint16_t, to_f16(v[i]));
  }
}

// Many rows on the matrix core: y[m][o] = f16(sum_k x[m][k] * wf[o][k]) for int8
// weights (Q8: wf = f16(f32(w8) * scale[o]), the contract rounding) or f16 ones.
// A workgroup is 16 NRB rows x 64 channels; its four waves split K (in steps of
// 64) and run without a barrier: per step a lane reads 16 weights of each of
// four channels (o0 + 16a + l % 16, k0 + 16 (l / 16)), which become two A operands
// each, and 2 NRB B operands straight from x (row l % 16 of a row block, the same
// k; x is small and shared by every column of workgroups, so it is L2 traffic).
// The waves' sums meet in LDS in wave order, wave a finishing channels o0 + 16a.
// Splitting K inside the workgroup, not the channels, keeps enough workgroups in
// flight for the narrow projections (203 rows x 512 channels: 56 workgroups of
// 8 steps) and needs no x staging.  Bound by the weights' conversion (about 2.5
// VALU per weight and 16 NRB rows) and the matrix pipe.  Measured on MI355X: 1000
// rows x 4096 channels, K = 2048: see rows_gemm.  K a multiple of 64, at most
// 8192; grid ceil(O / 64) * ceil(M / (16 NRB)), column blocks fastest, block 256.
template <int NRB>
using RowsGemmLds = f32x4_t[4][4][NRB < 4 ? NRB : 4][64];  // [channels][wave][row block][lane]

template <bool Q8, int NRB>
__device__ __forceinline__ void rows_gemm_body(const uint16_t* __restrict__ x,
                                               const void* __restrict__ wv,
                                               const float* __restrict__ scale, int M, int K,
                                               int O, uint16_t* __restrict__ y, int cb, int rb,
                                               RowsGemmLds<NRB>& s_acc) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;
  const int o0 = cb * 64, row0 = rb * 16 * NRB;
  const int NS = K / 64, s0 = NS * wave / 4, s1 = NS * (wave + 1) / 4;
  // channels past O and rows past M read the last one and are not stored;
  // uniform bases and 32-bit byte offsets (at most 128 rows of 16 KiB)
  const char* xb = reinterpret_cast<const char*>(x + (size_t)row0 * K);
  uint32_t xo[NRB];
  RowCols<Q8> cols;
  cols.init(wv, scale, o0, K, O);
#pragma unroll
  for (int r = 0; r < NRB; ++r)
    xo[r] = (uint32_t)(min(16 * r + c, M - 1 - row0) * K + 16 * g) * 2u;
  f32x4_t acc[4][NRB];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int r = 0; r < NRB; ++r) acc[a][r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (s0 < s1) {
    typename RowCols<Q8>::Regs w, wn;
    cols.load(w, s0);
    for (int s = s0; s < s1; ++s) {
      constexpr int RB = NRB < 4 ? NRB : 4;  // row blocks whose B operands are held at once
      uint4 b[RB][2];
      auto load_b = [&](int r0) {
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const uint4* p = reinterpret_cast<const uint4*>(xb + (xo[r0 + r] + 128u * s));
          b[r][0] = p[0];
          b[r][1] = p[1];
        }
      };
      load_b(0);
      cols.load(wn, min(s + 1, s1 - 1));
      u32x4_t A[4][2];
      cols.decode(w, A);
#pragma unroll
      for (int r0 = 0; r0 < NRB; r0 += RB) {
        if (r0) load_b(r0);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int a = 0; a < 4; ++a)
              acc[a][r0 + r] =
                  mma16(A[a][h], __builtin_bit_cast(u32x4_t, b[r][h]), acc[a][r0 + r]);
      }
      w = wn;
    }
  }
  // rounds of up to four row blocks: every wave hands the channels of the
  // others over and sums its own
  constexpr int RR = NRB < 4 ? NRB : 4;
#pragma unroll
  for (int r0 = 0; r0 < NRB; r0 += RR) {
    if (r0) __syncthreads();
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int r = 0; r < RR; ++r) s_acc[a][wave][r][lane] = acc[a][r0 + r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RR; ++r) {
      f32x4_t v = s_acc[wave][0][r][lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) {
        const f32x4_t t = s_acc[wave][w][r][lane];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = v[i] + t[i];
      }
      // lane: row c of the block, channels o .. o + 3
      const int row = row0 + 16 * (r0 + r) + c, o = o0 + 16 * wave + 4 * g;
      if (row >= M) continue;
      rows_store4(y, row, o, O, v);
    }
  }
}

template <bool Q8, int NRB>
__global__ __launch_bounds__(256, 2) void k_rows_gemm(const uint16_t* __restrict__ x,
                                                      const void* __restrict__ wv,
                                                      const float* __restrict__ scale, int M,
                                                      int K, int O, uint16_t* __restrict__ y) {
  __shared__ RowsGemmLds<NRB> s_acc;
  const int ncb = (O + 63) / 64;
  rows_gemm_body<Q8, NRB>(x, wv, scale, M, K, O, y, blockIdx.x % ncb, blockIdx.x / ncb, s_acc);
}

// Several projections of the same rows in one launch (an MoE block's router gate,
// shared-expert gate logit, and shared gate and up): each alone leaves most of the
// chip idle.  blk0: the projection's first workgroup.
constexpr int kRowsMultiMax = 4;
struct RowsMulti {
  const void* w[kRowsMultiMax];
  const float* scale[kRowsMultiMax];  // null: f16 weights
  uint16_t* y[kRowsMultiMax];
  int O[kRowsMultiMax], blk0[kRowsMultiMax];
  int n;
};

template <int NRB>
__global__ __launch_bounds__(256, 2) void k_rows_gemm_multi(const uint16_t* __restrict__ x,
                                                            RowsMulti a, int M, int K) {
  __shared__ RowsGemmLds<NRB> s_acc;
  int i = 0;
  while (i + 1 < a.n && (int)blockIdx.x >= a.blk0[i + 1]) ++i;
  const int O = a.O[i], b = blockIdx.x - a.blk0[i], ncb = (O + 63) / 64;
  if (a.scale[i])
    rows_gemm_body<true, NRB>(x, a.w[i], a.scale[i], M, K, O, a.y[i], b % ncb, b / ncb, s_acc);
  else
    rows_gemm_body<false, NRB>(x, a.w[i], nullptr, M, K, O, a.y[i], b % ncb, b / ncb, s_acc);
}

// The same product where there are tiles enough to fill the chip: k_gemm_mma2's
// main loop over int8 / f16 channels, a workgroup's four waves on 64 channels
// each and x staged through LDS once for all of them (in k_rows_gemm every wave
// reads its own x: 16 KiB per wave and step at 128 rows, more than the 64 B per
// clock of a CU's L1).  K a multiple of 64; grid ceil(O / 256) * ceil(M / (16 NRB)),
// column blocks fastest, block 256.
template <bool Q8, int NRB>
__global__ __launch_bounds__(256, 2) void k_rows_gemm_lds(const uint16_t* __restrict__ x,
                                                          const void* __restrict__ wv,
                                                          const float* __restrict__ scale, int M,
                                                          int K, int O,
                                                          uint16_t* __restrict__ y) {
  constexpr int XCH = NRB / 2;
  __shared__ uint4 s_x[2][16 * NRB * 8];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ncb = (O + 255) / 256;
  const int cb = blockIdx.x % ncb, row0 = (blockIdx.x / ncb) * 16 * NRB;
  // a wave past the last channel runs the last one's and stores nothing
  const int o0 = min(cb * 256 + 64 * wave, O - 1);
  RowCols<Q8> cols;
  cols.init(wv, scale, o0, K, O);
  uint32_t xoff[XCH];
#pragma unroll
  for (int j = 0; j < XCH; ++j)
    xoff[j] = 2u * (uint32_t)(min(mma2_x_row(tid, j), M - 1 - row0) * K) + mma2_x_chunk(tid, j);
  const __amdgpu_buffer_rsrc_t xrs =
      buf_rsrc(x + (size_t)row0 * K, (size_t)min(16 * NRB, M - row0) * K * 2);
  f32x4_t acc[4][NRB];
  mma2_loop<NRB>(cols, xrs, xoff, 0, K / 64, s_x, acc);
  if (cb * 256 + 64 * wave >= O) return;
  const int c = lane & 15, g = lane >> 4;
#pragma unroll
  for (int r = 0; r < NRB; ++r) {
    const int row = row0 + 16 * r + c;
    if (row >= M) continue;
#pragma unroll
    for (int a = 0; a < 4; ++a) rows_store4(y, row, o0 + 16 * a + 4 * g, O, acc[a][r]);
  }
}

// Embedding rows of an int8 table (escha_mlx/quant.py:253-266 under the w8a16
// contract): out[t][k] = f16(f32(w8[ids[t]][k]) * f32(scale[ids[t]])), the
// same rounding as the GEMV's weights.  An id outside [0, N) yields a row of
// f16 NaN (0x7E00) instead of a read outside the table.  K a multiple of 16;
// grid (T), block 256, each thread converting 16-byte chunks of the row.
__global__ __launch_bounds__(256) void k_q8_embed(const int32_t* __restrict__ ids,
                                                  const int8_t* __restrict__ w8,
                                                  const float* __restrict__ scale, int N, int K,
                                                  uint16_t* __restrict__ out) {
  const int t = blockIdx.x;
  const int id = ids[t];
  const bool ok = id >= 0 && id < N;
  const float s = ok ? scale[id] : 0.f, ms = -128.f * s;
  uint4* dst = reinterpret_cast<uint4*>(out + (size_t)t * K);
  const uint4* src = reinterpret_cast<const uint4*>(w8 + (size_t)(ok ? id : 0) * K);
  for (int c = threadIdx.x; c < K / 16; c += 256) {
    uint32_t p[8];
    if (ok) {
      const uint4 v = src[c];
      w8_to_f16x4(v.x, s, ms, p[0], p[1]);
      w8_to_f16x4(v.y, s, ms, p[2], p[3]);
      w8_to_f16x4(v.z, s, ms, p[4], p[5]);
      w8_to_f16x4(v.w, s, ms, p[6], p[7]);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = 0x7E007E00u;
    }
    dst[2 * c] = make_uint4(p[0], p[1], p[2], p[3]);
    dst[2 * c + 1] = make_uint4(p[4], p[5], p[6], p[7]);
  }
}

// Shared-expert activation (escha_mlx/ref.py:345): hh = f16((g / (1 + exp(-g))) * u)
// in float32, g and u f16 [m][I].  grid (ceil(I/256), m), block 256.
__global__ __launch_bounds__(256) void k_shared_act(const uint16_t* __restrict__ g,
                                                    const uint16_t* __restrict__ u, int I,
                                                    uint16_t* __restrict__ hh) {
  const int i = blockIdx.x * 256 + threadIdx.x, row = blockIdx.y;
  if (i >= I) return;
  const size_t o = (size_t)row * I + i;
  const float gf = (float)__builtin_bit_cast(half_t, g[o]);
  const float uf = (float)__builtin_bit_cast(half_t, u[o]);
  hh[o] = __builtin_bit_cast(uint16_t, to_f16((gf / (1.0f + expf(-gf))) * uf));
}

// The activation and the down projection's input transform in one pass (the MLP
// of many rows): xh = f16(H128(f32(h) * rin) * rs), h = f16((g / (1 + exp(-g))) * u)
// as k_shared_act, g and u [m][I] read as f16 (bf16 rows rounded to f16 first, as
// the module's cast does; f32 rows hold f16 values).  HBM-bound, and h is never
// written: 2048 x 17408 62 -> 55 us by 8 lanes per block (h128_oct) against one wave.
// grid: oct_place.
template <int DT, int ROWS>
__global__ __launch_bounds__(256) void k_act_transform(const void* __restrict__ g,
                                                       const void* __restrict__ u,
                                                       const float* __restrict__ rin, int m, int I,
                                                       float rs, uint16_t* __restrict__ xh) {
  const OctPlace at = oct_place<ROWS>(m, I / 128);
  float gv[ROWS][16], uv[ROWS][16], r[16];
#pragma unroll
  for (int j = 0; j < ROWS; ++j) {
    const size_t i = (size_t)min(at.row0 + j, m - 1) * I + at.col;
    load_oct<DT>(g, i, gv[j]);
    load_oct<DT>(u, i, uv[j]);
  }
  load_oct<kRowsF32>(rin, at.col, r);
  auto act = [](float gf, float uf) {
    if constexpr (DT != kRowsF16) {
      gf = (float)(half_t)gf;
      uf = (float)(half_t)uf;
    }
    return (float)to_f16((gf / (1.0f + expf(-gf))) * uf);
  };
#pragma unroll
  for (int j = 0; j < ROWS; ++j) {
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = act(gv[j][i], uv[j][i]) * r[i];
    h128_oct(v);
    if (at.row0 + j < m) store_oct(xh, (size_t)(at.row0 + j) * I + at.col, v, rs);
  }
}

// sigmoid of an f16 logit, in float32.
__device__ __forceinline__ float sigmoid16(uint16_t v) {
  return 1.0f / (1.0f + expf(-(float)__builtin_bit_cast(half_t, v)));
}

// One element of the block's output in element type dt: f16(f32(y) + f32(sh) *
// sg), converted.
__device__ __forceinline__ void block_store(void* out, int dt, size_t i, half_t y, half_t sh,
                                            float sg) {
  const half_t v = to_f16((float)y + (float)sh * sg);
  if (dt == kRowsF32)
    static_cast<float*>(out)[i] = (float)v;
  else
    static_cast<uint16_t*>(out)[i] =
        dt == kRowsBF16 ? (uint16_t)pack2_bf16((float)v, 0.f) : __builtin_bit_cast(uint16_t, v);
}

// acc[m] = sum over one weight row (chunks 16-byte pieces, piece lane + 64j by
// lane) of x row m (m < M <= NR) x weight, summed over the wave: k_rows_gemv's
// products and order at 64 lanes per row.
template <bool Q8, int NR, int CPL>
__device__ __forceinline__ void wave_row_dot(const uint16_t* __restrict__ x, int M, int K,
                                             const void* __restrict__ row, float s, float* acc) {
  constexpr int CW = Q8 ? 16 : 8;
  const int lane = threadIdx.x & 63, chunks = K / CW;
  const float ms = -128.f * s;
  uint4 w[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j)
    w[j] = static_cast<const uint4*>(row)[min(lane + 64 * j, chunks - 1)];
  uint4 xv[NR][CPL][CW / 8];
#pragma unroll
  for (int m = 0; m < NR; ++m)
#pragma unroll
    for (int j = 0; j < CPL; ++j)
#pragma unroll
      for (int i = 0; i < CW / 8; ++i)
        xv[m][j][i] = reinterpret_cast<const uint4*>(
            x + (size_t)min(m, M - 1) * K)[min(lane + 64 * j, chunks - 1) * (CW / 8) + i];
#pragma unroll
  for (int m = 0; m < NR; ++m) acc[m] = 0.f;
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    // pieces past the row's end: zero weights (an int8 zero is 128 - 128, so the
    // converted words are cleared)
    const bool has = lane + 64 * j < chunks;
    uint32_t wp[CW / 2];
    const uint32_t ww[4] = {w[j].x, w[j].y, w[j].z, w[j].w};
    if constexpr (Q8) {
#pragma unroll
      for (int i = 0; i < 4; ++i) w8_to_f16x4(ww[i], s, ms, wp[2 * i], wp[2 * i + 1]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) wp[i] = ww[i];
    }
#pragma unroll
    for (int m = 0; m < NR; ++m) {
      float t = acc[m];
#pragma unroll
      for (int i = 0; i < CW / 8; ++i) {
        t = dot2(xv[m][j][i].x, wp[4 * i], t);
        t = dot2(xv[m][j][i].y, wp[4 * i + 1], t);
        t = dot2(xv[m][j][i].z, wp[4 * i + 2], t);
        t = dot2(xv[m][j][i].w, wp[4 * i + 3], t);
      }
      acc[m] = has ? t : acc[m];
    }
  }
#pragma unroll
  for (int m = 0; m < NR; ++m) acc[m] = row_sum<64>(acc[m]);
}

// An MoE block's first projections for up to NR decode tokens, one output channel
// per wave: the router's E logits and the shared expert's gate logit (f16 weights),
// the shared gate and up (int8).  One launch for four: at one token each is a few
// us of latency (1,281 rows of 2 to 4 KiB).  CF = ceil(H / 512).  grid
// ceil((E + 1 + 2 Ish) / 4), block 256.
struct BlockHead {
  const uint16_t *x, *gate_w, *shg_w;
  const int8_t *sg_w, *su_w;
  const float *sg_s, *su_s;
  uint16_t *logits, *shg, *g, *u;  // [T][E], [T], [T][Ish]
  int T, E, H, Ish;
};
template <int NR, int CF>
__global__ __launch_bounds__(256) void k_block_head(BlockHead a) {
  const int lane = threadIdx.x & 63;
  int o = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  float acc[NR];
  uint16_t* y;
  int ldy;
  if (o <= a.E) {
    const uint16_t* row = o < a.E ? a.gate_w + (size_t)o * a.H : a.shg_w;
    wave_row_dot<false, NR, CF>(a.x, a.T, a.H, row, 0.f, acc);
    y = o < a.E ? a.logits + o : a.shg;
    ldy = o < a.E ? a.E : 1;
  } else {
    o -= a.E + 1;
    if (o >= 2 * a.Ish) return;
    const bool up = o >= a.Ish;
    if (up) o -= a.Ish;
    const float s = (up ? a.su_s : a.sg_s)[o];
    wave_row_dot<true, NR, (CF + 1) / 2>(a.x, a.T, a.H, (up ? a.su_w : a.sg_w) + (size_t)o * a.H,
                                         s, acc);
    y = (up ? a.u : a.g) + o;
    ldy = a.Ish;
  }
#pragma unroll
  for (int m = 0; m < NR; ++m)
    if (lane == 0 && m < a.T) y[(size_t)m * ldy] = __builtin_bit_cast(uint16_t, to_f16(acc[m]));
}

// The block's end for up to NR tokens, one output channel per wave: the shared
// expert's activation of its Ish inputs (each wave its own copy: 16 exponentials per
// lane), its down projection, and out = y + sh * sigmoid(shg).  Three launches in
// one.  CQ = ceil(Ish / 1024).  grid ceil(H / 4), block 256.
struct BlockTail {
  const uint16_t *g, *u, *shg, *y;  // y: the routed sum [T][H]
  const int8_t* sd_w;
  const float* sd_s;
  void* out;
  int odt, T, H, Ish;
};
template <int NR, int CQ>
__global__ __launch_bounds__(256) void k_block_tail(BlockTail a) {
  const int lane = threadIdx.x & 63;
  const int o = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (o >= a.H) return;
  const int chunks = a.Ish / 16;
  const float s = a.sd_s[o], ms = -128.f * s;
  uint4 w[CQ];
#pragma unroll
  for (int j = 0; j < CQ; ++j)
    w[j] = reinterpret_cast<const uint4*>(a.sd_w + (size_t)o * a.Ish)[min(lane + 64 * j, chunks - 1)];
  half_t yv = (half_t)0.f;
  uint16_t sg = 0;
  if (lane < a.T) {
    yv = __builtin_bit_cast(half_t, a.y[(size_t)lane * a.H + o]);
    sg = a.shg[lane];
  }
  float acc[NR];
#pragma unroll
  for (int m = 0; m < NR; ++m) {
    acc[m] = 0.f;
    const int row = min(m, a.T - 1);
#pragma unroll
    for (int j = 0; j < CQ; ++j) {
      const size_t at = (size_t)row * a.Ish + 16 * min(lane + 64 * j, chunks - 1);
      const uint4* gp = reinterpret_cast<const uint4*>(a.g + at);
      const uint4* up = reinterpret_cast<const uint4*>(a.u + at);
      const uint4 g0 = gp[0], g1 = gp[1], u0 = up[0], u1 = up[1];
      const uint32_t gw[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
      const uint32_t uw[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
      const uint32_t ww[4] = {w[j].x, w[j].y, w[j].z, w[j].w};
      uint32_t wp[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) w8_to_f16x4(ww[i], s, ms, wp[2 * i], wp[2 * i + 1]);
      float t = acc[m];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        half_t hh[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float gf = (float)__builtin_bit_cast(half_t, (uint16_t)(gw[i] >> (16 * e)));
          const float uf = (float)__builtin_bit_cast(half_t, (uint16_t)(uw[i] >> (16 * e)));
          hh[e] = to_f16((gf / (1.0f + expf(-gf))) * uf);
        }
        t = dot2(pack2(hh[0], hh[1]), wp[i], t);
      }
      acc[m] = lane + 64 * j < chunks ? t : acc[m];
    }
    acc[m] = row_sum<64>(acc[m]);
  }
  // lane m writes token m
#pragma unroll
  for (int m = 0; m < NR; ++m)
    if (lane == m && m < a.T)
      block_store(a.out, a.odt, (size_t)m * a.H + o, yv, to_f16(acc[m]), sigmoid16(sg));
}

// Block output (escha_mlx/ref.py:346-349, models/qwen3_5_moe.py:270-272):
// out = f16(f32(y) + f32(sh) * sigmoid(f32(shg))), y the f16 routed sum, sh
// the shared expert's f16 output, shg [m] the f16 shared gate logit.
// odt: the element type out is written in.  grid (ceil(H/256), m), block 256.
__global__ __launch_bounds__(256) void k_block_out(const uint16_t* __restrict__ yr,
                                                   const uint16_t* __restrict__ sh,
                                                   const uint16_t* __restrict__ shg, int H,
                                                   void* __restrict__ out, int odt) {
  const int c = blockIdx.x * 256 + threadIdx.x, row = blockIdx.y;
  if (c >= H) return;
  const size_t o = (size_t)row * H + c;
  block_store(out, odt, o, __builtin_bit_cast(half_t, yr[o]), __builtin_bit_cast(half_t, sh[o]),
              sigmoid16(shg[row]));
}

}  // namespace esc
