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
// (moe_mma_nrb), against the split-K chain's one pass per 8 rows.  256 experts,
// hidden 2048, intermediate 512, top-8, 2048 tokens (64 rows per expert): the
// whole call 357 us, the split-K chain 1200.
#pragma once

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
  constexpr int kPitch = 128 + 4;  // floats per staged row
  __shared__ uint4 s_x[2][BR * 8];
  static_assert(sizeof(s_x) >= 2 * 16 * kPitch * sizeof(float) || NRB < 6, "");
  __shared__ float s_o[NRB < 6 ? 2 * 16 * kPitch : 1];
  const int per = 8 * a.ncb, q8 = blockIdx.x / per, rem = blockIdx.x % per;
  const int g = 8 * q8 + rem % 8, cb = rem / 8;
  if (g >= a.n_groups) return;
  const int e = a.group_expert[g];
  if (e < 0) return;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int pair = wave >> 1, hw = wave & 1;
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
  f32x4_t acc[D::NA][NRB];
  mma2_loop<K, NRB>(cbase, kstride, xrs, xoff, 0, TK / 4, s_x, acc);

  float* so = NRB < 6 ? s_o : reinterpret_cast<float*>(&s_x[0][0]);
  float* sp = so + pair * 16 * kPitch;
  const float rs = a.rs;
  if constexpr (GU) {
    const int I = OC / 2, col = 128 * cb + 2 * lane;
    const float2 rg = ld_global_f2(a.rout + (size_t)e * OC + col);
    const float2 ru = ld_global_f2(a.rout + (size_t)e * OC + I + col);
    const float2 ri = ld_global_f2(a.dn_rin + (size_t)e * I + col);
#pragma unroll
    for (int r = 0; r < NRB; ++r) {
      mma2_to_lds<K, NRB>(acc, r, sp + 64 * hw, kPitch);
      __syncthreads();
#pragma unroll 2
      for (int j = 0; j < 4; ++j) {
        const int rl = 4 * wave + j, row = rows[16 * r + rl];
        if (row >= M) continue;  // wave-uniform: padding follows the group's rows
        const float* sg = so + rl * kPitch + 2 * lane;
        const float* su = sg + 16 * kPitch;
        float g0 = sg[0], g1 = sg[1], u0 = su[0], u1 = su[1];
        h128_wave(g0, g1);
        h128_wave(u0, u1);
        const half_t h0 = swiglu1(to_f16((g0 * rs) * rg.x), to_f16((u0 * rs) * ru.x));
        const half_t h1 = swiglu1(to_f16((g1 * rs) * rg.y), to_f16((u1 * rs) * ru.y));
        float v0 = (float)h0 * ri.x, v1 = (float)h1 * ri.y;
        h128_wave(v0, v1);
        *reinterpret_cast<uint32_t*>(a.out + (size_t)row * I + col) =
            pack2(to_f16(v0 * rs), to_f16(v1 * rs));
      }
      __syncthreads();
    }
  } else {
    const int col = 256 * cb + 128 * pair + 2 * lane;
    const float2 ro = ld_global_f2(a.rout + (size_t)e * OC + (live ? col : 0));
#pragma unroll
    for (int r = 0; r < NRB; ++r) {
      mma2_to_lds<K, NRB>(acc, r, sp + 64 * hw, kPitch);
      __syncthreads();
#pragma unroll 2
      for (int j = 0; j < 8; ++j) {
        const int rl = 8 * hw + j, row = rows[16 * r + rl];
        if (row >= M || !live) continue;
        float v0 = sp[rl * kPitch + 2 * lane], v1 = sp[rl * kPitch + 2 * lane + 1];
        h128_wave(v0, v1);
        *reinterpret_cast<uint32_t*>(a.out + (size_t)row * OC + col) =
            pack2(to_f16((v0 * rs) * ro.x), to_f16((v1 * rs) * ro.y));
      }
      __syncthreads();
    }
  }
}

}  // namespace esc
