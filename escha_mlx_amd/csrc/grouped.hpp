// Routed experts for many rows: the grouped coded GEMM on the matrix cores with
// both transforms, SwiGLU and the f16 rounding in its epilogues
// (EschaSparseMoeBlock._expert_path, escha_mlx/models/qwen3_5_moe.py:207-253).
//
// Groups are up to 16 NRB routed rows of one expert (build_groups layout).  A
// workgroup is one group x 256 columns and runs k_gemm_mma2's main loop on the
// group's gathered rows, so each weight is decoded once per group:
//   gate_up (GU): 128 gate columns (waves 0, 1) and the matching 128 up
//     columns (waves 2, 3) of h-block hb; the epilogue has both of a row's
//     128-blocks, so it goes straight to the down projection's input
//     (output transform, SwiGLU, down input transform) as f16: no float32
//     partials, no separate middle kernel;
//   down: 256 columns of H, the output transform in the epilogue, f16 rows
//     that k_combine sums in slot order.
// Every rounding point is k_moe_mid's / k_moe_combine's.  A row's result does
// not depend on its place in a group (one B column each).
//
// What bounds it: the decode (about 4.6 VALU per weight) of one pass over the
// experts' code, so the row-block size is chosen for the fewest, smallest groups
// (moe_mma_nrb), against the split-K chain's one pass per 8 rows; the main loop and
// the epilogue run over the row blocks that hold rows, rounded to an even number in
// the loop (one instance of it per size).  256 experts, hidden 2048, intermediate
// 512, top-8, 2048 tokens (64 rows per expert): the whole call 274 us (289 over all
// row blocks of every group), the split-K chain 1200.
#pragma once

#include <type_traits>

#include "mfma.hpp"
#include "moe.hpp"

namespace esc {

struct MoeMmaArgs {
  const uint16_t* xh;      // [M][IC] transformed rows
  const uint32_t* code;    // [E][TK][TN][8K]
  const int* rows_idx;     // [n_groups * 16 NRB], M = padding
  const int* group_expert; // [n_groups], -1 = no group
  const float* rout;       // [E][OC]
  const float* dn_rin;     // GU: [E][OC / 2]
  uint16_t* out;           // GU: xh2 [M][OC / 2]; down: d16 [M][OC]
  int M, TK, TN, n_groups, ncb;  // ncb: column blocks per group
  float rs;
};

// grid: 8 * ceil(n_groups / 8) * ncb, block 256.  The column blocks of one
// group sit on one XCD (blockIdx % 8 = group % 8): they read the same rows.
// Down with an odd number of 128-column blocks: the last workgroup's waves 2
// and 3 run tiles clamped into the stream and store nothing.
template <int K, int NRB, bool GU>
__global__ __launch_bounds__(256, 2) void k_moe_mma(MoeMmaArgs a) {
  using G = Geo<K>;
  using D = Mma2<K, NRB>;
  constexpr int BR = D::BR, XCH = D::XCH;
  __shared__ uint4 s_x[2][BR * 8];
  // the epilogue's exchange areas, over x's stages where they fit
  constexpr int kAreas = GU ? kMma2Xch + 4 * 3 * 64 : 2 * kMma2Xch;  // float4
  constexpr bool kOwn = sizeof(s_x) < kAreas * sizeof(float4);
  __shared__ float4 s_o[kOwn ? kAreas : 1];
  const int per = 8 * a.ncb, q8 = blockIdx.x / per, rem = blockIdx.x % per;
  const int g = 8 * q8 + rem % 8, cb = rem / 8;
  if (g >= a.n_groups) return;
  const int e = a.group_expert[g];
  if (e < 0) return;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int pair = wave >> 1, hw = wave & 1;  // 128-column half, 64-column quarter
  const int M = a.M, TK = a.TK, TN = a.TN;
  const int IC = TK * 16, OC = TN * 16;
  const int gk = lane >> 4, c = lane & 15, tc = c / G::LPT, q = lane % G::LPT;
  // the wave's first tile (4 tiles, 64 columns)
  int tile0 = GU ? pair * (TN / 2) + 8 * cb + 4 * hw : 16 * cb + 4 * wave;
  const bool live = GU || tile0 < TN;
  if (!live) tile0 = TN - 4;
  const size_t kstride = (size_t)TN * (8 * K);
  const uint32_t* cbase = a.code + (size_t)e * TK * kstride + (size_t)(tile0 + tc) * (8 * K) +
                          q * G::WPL + gk * kstride;
  const int* rows = a.rows_idx + (size_t)g * BR;
  uint32_t xoff[XCH];
#pragma unroll
  for (int j = 0; j < XCH; ++j) {
    const int row = rows[mma2_x_row(tid, j)];
    xoff[j] = 2u * ((uint32_t)(row < M ? row : 0) * IC) + mma2_x_chunk(tid, j);
  }
  const __amdgpu_buffer_rsrc_t xrs = buf_rsrc(a.xh, (size_t)M * IC * 2);
  // row blocks that hold rows (a group's rows come first, then padding)
  int nact = 1;
#pragma unroll
  for (int r = 1; r < NRB; ++r) nact += rows[16 * r] < M;
  f32x4_t acc[D::NA][NRB];
  const CodedCols<K> cols{cbase, kstride};
  auto loop = [&](auto n) {
    mma2_loop<NRB, decltype(n)::value>(cols, xrs, xoff, 0, TK / 4, s_x, acc);
  };
  if constexpr (NRB > 6) {
    if (nact <= NRB - 6) loop(std::integral_constant<int, NRB - 6>{});
  }
  if constexpr (NRB > 4) {
    if (nact > NRB - 6 && nact <= NRB - 4) loop(std::integral_constant<int, NRB - 4>{});
  }
  if constexpr (NRB > 2) {
    if (nact > NRB - 4 && nact <= NRB - 2) loop(std::integral_constant<int, NRB - 2>{});
  }
  if (nact > NRB - 2) loop(std::integral_constant<int, NRB>{});

  float4* so = kOwn ? s_o : reinterpret_cast<float4*>(&s_x[0][0]);
  const float rs = a.rs;
  const int chunk = mma2_chunk<K>();
  if constexpr (GU) {
    const int I = OC / 2;
    // gate (pair 0) and up (pair 1) output scales of the lane's 16 columns
    // col + 64b + j; then the lane's 8 columns of h, ch + j
    const int col = 128 * cb + 32 * hw + 8 * chunk;
    float ro[16], ri[8];
#pragma unroll
    for (int j = 0; j < 16; ++j)
      ro[j] = as_global(a.rout + (size_t)e * OC + pair * I)[col + 64 * (j >> 3) + (j & 7)];
#pragma unroll
    for (int j = 0; j < 8; ++j) ri[j] = as_global(a.dn_rin + (size_t)e * I)[col + 64 * pair + j];
    uint4* s_gu = reinterpret_cast<uint4*>(so + kMma2Xch);  // gate / up halves, f16
    float4* s_a = so + kMma2Xch + 256;                      // the two cross-wave stages of h
    float4* s_b = s_a + 256;
#pragma unroll
    for (int r = 0; r < NRB; ++r) {
      if (r >= nact) break;
      const int row = rows[16 * r + c];
      float v[16], o[16];
      mma2_h64<K, NRB>(acc, r, v);
      mma2_h128_last(v, so, o);
      half_t h[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) h[j] = to_f16((o[j] * rs) * ro[j]);
      // gate waves keep columns 64b + .. of b = 0 and get their up values, up
      // waves b = 1 and their gate values: wave (pair, hw) then has the h
      // columns col + 64 pair + j
      uint32_t mine[4], send[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t p0 = pack2(h[2 * j], h[2 * j + 1]), p1 = pack2(h[8 + 2 * j], h[9 + 2 * j]);
        mine[j] = pick(pair, p1, p0);
        send[j] = pick(pair, p0, p1);
      }
      s_gu[wave * 64 + lane] = make_uint4(send[0], send[1], send[2], send[3]);
      lds_barrier();
      const uint4 got4 = s_gu[(wave ^ 2) * 64 + lane];
      const uint32_t got[4] = {got4.x, got4.y, got4.z, got4.w};
      float f[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t gw = pick(pair, got[j >> 1], mine[j >> 1]);
        const uint32_t uw = pick(pair, mine[j >> 1], got[j >> 1]);
        const half_t hv = swiglu1(__builtin_bit_cast(half_t, (uint16_t)(gw >> (16 * (j & 1)))),
                                  __builtin_bit_cast(half_t, (uint16_t)(uw >> (16 * (j & 1)))));
        f[j] = (float)hv * ri[j];
      }
      // H128 of h: column bits 0..2 in registers, 3 and 4 in the lanes (bit 3
      // is lane bit 4 for K = 2, lane bit 5 for K = 3), 5 and 6 across the waves
      bfly_reg<1>(f);
      bfly_reg<2>(f);
      bfly_reg<4>(f);
      bfly_lane<4, K == 2>(f);  // register bit 2: column bit 3
      bfly_lane<4, K != 2>(f);  // register bit 2: column bit 4
      // column bit 5: the other wave of the pair; this wave keeps bit 4 = hw
      float4* x5 = s_a + wave * 64 + lane;
      float t[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) t[j] = pick(hw, f[j], f[4 + j]);
      *x5 = make_float4(t[0], t[1], t[2], t[3]);
      lds_barrier();
      const float4 p5 = s_a[(wave ^ 1) * 64 + lane];
      const float q5[4] = {p5.x, p5.y, p5.z, p5.w};
      float lo[4], hi[4];  // column bit 5 = 0, 1
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float m = pick(hw, f[4 + j], f[j]);
        const float x0 = pick(hw, q5[j], m), x1 = pick(hw, m, q5[j]);
        lo[j] = x0 + x1;
        hi[j] = x0 - x1;
      }
      // column bit 6: the other pair; this wave keeps bit 5 = pair
#pragma unroll
      for (int j = 0; j < 4; ++j) t[j] = pick(pair, lo[j], hi[j]);
      s_b[wave * 64 + lane] = make_float4(t[0], t[1], t[2], t[3]);
      lds_barrier();
      const float4 p6 = s_b[(wave ^ 2) * 64 + lane];
      const float q6[4] = {p6.x, p6.y, p6.z, p6.w};
      half_t y0[4], y1[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float m = pick(pair, hi[j], lo[j]);
        const float x0 = pick(pair, q6[j], m), x1 = pick(pair, m, q6[j]);
        y0[j] = to_f16((x0 + x1) * rs);
        y1[j] = to_f16((x0 - x1) * rs);
      }
      // columns 64b + 32 pair + 16 hw + 8 (bit 3) + 4 (bit 2) + j, the column
      // bits 2 and 3 in the lanes
      if (row < M) {
        const int b2 = K == 2 ? gk & 1 : gk >> 1, b3 = K == 2 ? gk >> 1 : gk & 1;
        uint16_t* d = a.out + (size_t)row * I + 128 * cb + 32 * pair + 16 * hw + 8 * b3 + 4 * b2;
        *reinterpret_cast<uint2*>(d) = make_uint2(pack2(y0[0], y0[1]), pack2(y0[2], y0[3]));
        *reinterpret_cast<uint2*>(d + 64) = make_uint2(pack2(y1[0], y1[1]), pack2(y1[2], y1[3]));
      }
    }
  } else {
    const int col = live ? 256 * cb + 128 * pair + 32 * hw + 8 * chunk : 0;
    float ro[16];
#pragma unroll
    for (int j = 0; j < 16; ++j)
      ro[j] = as_global(a.rout + (size_t)e * OC)[col + 64 * (j >> 3) + (j & 7)];
#pragma unroll
    for (int r = 0; r < NRB; ++r) {
      if (r >= nact) break;
      const int row = rows[16 * r + c];
      mma2_out<K, NRB>(acc, r, so + (r & 1) * kMma2Xch, rs, ro, nullptr, col, row < M && live,
                       a.out, kRowsF16, (size_t)row * OC + col);
    }
  }
}

}  // namespace esc
