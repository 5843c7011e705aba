// Tile decode, 128-point transforms, router top-k, row grouping.
#pragma once

#include "codec.hpp"

namespace esc {

// ---------------------------------------------------------------- decode
// code [TK][TN][8K] -> w [IC][OC] f16 (escha_mlx/msl.py:183-202, ref.py:126-134).
// One 256-thread block per tile, one thread per trellis step.
template <int K, bool LUT>
__global__ __launch_bounds__(256) void k_decode_tiles(const uint32_t* __restrict__ code, int TN,
                                                      int OC, uint16_t* __restrict__ w) {
  const int tile = blockIdx.x;
  const int kt = tile / TN, nt = tile - kt * TN;
  const int t = threadIdx.x;
  const uint32_t* wp = code + (size_t)tile * (8 * K);
  uint32_t s = step_state<K>([&](int i) { return wp[i]; }, t);
  uint16_t v = LUT ? g_lut.v[s] : decode_hash_bits(s);
  w[(size_t)(16 * kt + step_row(t)) * OC + 16 * nt + step_col(t)] = v;
}

// ---------------------------------------------------------------- H128
// One wave owns one 128-block of one row; lane l holds elements 2l and 2l+1.
// Stage s pairs i with i ^ (1 << s), bit 0 first, (a + b, a - b) in float32
// (escha_mlx/ref.py:204-218, msl.py:905-913).  Built with -ffp-contract=off.
// The lane exchanges stay on the VALU: DPP quad permutes for lane ^ 1 and
// ^ 2, two bank-masked DPP row shifts for ^ 4 and ^ 8, and the gfx950 row /
// half-wave swaps (v_permlane16_swap, v_permlane32_swap) for ^ 16 and ^ 32.

// value of lane ^ M (M in {1, 2, 4, 8}: within a row of 16 lanes)
template <int M>
__device__ __forceinline__ float lane_xor(float v) {
  const int x = __builtin_bit_cast(int, v);
  int r;
  if constexpr (M == 1) {
    r = __builtin_amdgcn_update_dpp(x, x, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
  } else if constexpr (M == 2) {
    r = __builtin_amdgcn_update_dpp(x, x, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
  } else {
    // lanes with bit M clear read lane + M (row_shl), the others lane - M
    // (row_shr); each shift writes only its banks of 4 lanes
    constexpr int lo_banks = M == 4 ? 0x5 : 0x3, hi_banks = M == 4 ? 0xA : 0xC;
    r = __builtin_amdgcn_update_dpp(x, x, 0x100 + M, 0xF, lo_banks, false);
    r = __builtin_amdgcn_update_dpp(r, x, 0x110 + M, 0xF, hi_banks, false);
  }
  return __builtin_bit_cast(float, r);
}

__device__ __forceinline__ void h128_wave(float& v0, float& v1) {
  const int lane = threadIdx.x & 63;
  {
    float a = v0, b = v1;
    v0 = a + b;
    v1 = a - b;
  }
  auto stage = [&](float o0, float o1, bool upper) {
    if (upper) {
      v0 = o0 - v0;
      v1 = o1 - v1;
    } else {
      v0 = v0 + o0;
      v1 = v1 + o1;
    }
  };
  stage(lane_xor<1>(v0), lane_xor<1>(v1), lane & 1);
  stage(lane_xor<2>(v0), lane_xor<2>(v1), lane & 2);
  stage(lane_xor<4>(v0), lane_xor<4>(v1), lane & 4);
  stage(lane_xor<8>(v0), lane_xor<8>(v1), lane & 8);
  // ^ 16 and ^ 32: the swap returns the lower partner's value (lo) and the
  // upper partner's (hi) in every lane: a + b below, a - b above
  auto swap_stage = [&](auto swp, bool upper) {
    const auto p0 = swp(__builtin_bit_cast(unsigned, v0));
    const auto p1 = swp(__builtin_bit_cast(unsigned, v1));
    // elements copied out first: __builtin_bit_cast of a vector element
    // reads element 0 with this compiler
    const unsigned l0 = p0[0], h0 = p0[1], l1 = p1[0], h1 = p1[1];
    const float lo0 = __builtin_bit_cast(float, l0), hi0 = __builtin_bit_cast(float, h0);
    const float lo1 = __builtin_bit_cast(float, l1), hi1 = __builtin_bit_cast(float, h1);
    v0 = upper ? lo0 - hi0 : lo0 + hi0;
    v1 = upper ? lo1 - hi1 : lo1 + hi1;
  };
  swap_stage([](unsigned x) { return __builtin_amdgcn_permlane16_swap(x, x, false, false); },
             lane & 16);
  swap_stage([](unsigned x) { return __builtin_amdgcn_permlane32_swap(x, x, false, false); },
             lane & 32);
}

// The same transform with 8 lanes per 128-block, a wave working on 8 blocks at
// once: v[8b + j] is element 64b + 8 oct_chunk() + j, so element bits 0..2 and 6 are
// additions between registers and bits 3..5 one DPP move and one addition each
// (lane ^ 1, ^ 2 and ^ 7 = quad permutes and the half-row mirror; oct_chunk() is the
// lane numbering in which these flip one bit each).  The stages run in h128_wave's
// order on the same operands (a - b of the upper lane as fma(v, -1, other), exact):
// bit-identical to it.  29 VALU instructions per block with its conversions against
// 60, and 16- and 32-byte accesses per lane.
__device__ __forceinline__ int oct_chunk() {
  const int l = threadIdx.x & 7;
  return l < 4 ? l : l ^ 3;
}
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  const int x = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(x, x, CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ void h128_oct(float (&v)[16]) {
  auto pair = [&](int a, int b) {
    const float x = v[a], y = v[b];
    v[a] = x + y;
    v[b] = x - y;
  };
#pragma unroll
  for (int s = 1; s < 8; s *= 2)
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (!(j & s)) pair(j, j | s);
  const int ch = oct_chunk();
  const float s3 = ch & 1 ? -1.f : 1.f, s4 = ch & 2 ? -1.f : 1.f, s5 = ch & 4 ? -1.f : 1.f;
#pragma unroll
  for (int j = 0; j < 16; ++j) v[j] = __builtin_fmaf(v[j], s3, dpp_move<0xB1>(v[j]));   // ^ 1
#pragma unroll
  for (int j = 0; j < 16; ++j) v[j] = __builtin_fmaf(v[j], s4, dpp_move<0x4E>(v[j]));   // ^ 2
#pragma unroll
  for (int j = 0; j < 16; ++j) v[j] = __builtin_fmaf(v[j], s5, dpp_move<0x141>(v[j]));  // ^ 7
#pragma unroll
  for (int j = 0; j < 8; ++j) pair(j, j + 8);
}

// Element types of the rows an input transform reads (esc_input_transform_typed).
enum { kRowsF16 = 0, kRowsBF16 = 1, kRowsF32 = 2 };

// One 16-bit row element as float32 (exact); dt is kRowsF16 or kRowsBF16.
__device__ __forceinline__ float row_value16(uint16_t v, int dt) {
  const float b = __builtin_bit_cast(float, (uint32_t)v << 16);
  const float h = (float)__builtin_bit_cast(half_t, v);
  return dt == kRowsBF16 ? b : h;
}

// Elements c, c + 1 of a row as float32 (exact for every type).
template <int DT>
__device__ __forceinline__ float2 row_pair(const void* rows, size_t i) {
  if constexpr (DT == kRowsF32) {
    return *reinterpret_cast<const float2*>(static_cast<const float*>(rows) + i);
  } else {
    const uint32_t xv = *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(rows) + i);
    if constexpr (DT == kRowsBF16)
      return make_float2(__builtin_bit_cast(float, xv << 16),
                         __builtin_bit_cast(float, xv & 0xFFFF0000u));
    else
      return make_float2((float)__builtin_bit_cast(half_t, (uint16_t)xv),
                         (float)__builtin_bit_cast(half_t, (uint16_t)(xv >> 16)));
  }
}

// 16 bytes at any element alignment (a caller's rows may start at any element).
struct __attribute__((packed, aligned(2))) Bytes16 {
  uint32_t w[4];
};
// Elements i .. i + 7 and i + 64 .. i + 71 of a row as float32 (exact for every type).
template <int DT>
__device__ __forceinline__ void load_oct(const void* rows, size_t i, float (&v)[16]) {
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    if constexpr (DT == kRowsF32) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const Bytes16 q = *reinterpret_cast<const Bytes16*>(static_cast<const float*>(rows) + i +
                                                            64 * b + 4 * h);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[8 * b + 4 * h + j] = __builtin_bit_cast(float, q.w[j]);
      }
    } else {
      const Bytes16 q =
          *reinterpret_cast<const Bytes16*>(static_cast<const uint16_t*>(rows) + i + 64 * b);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t w = q.w[j];
        v[8 * b + 2 * j] = DT == kRowsBF16 ? __builtin_bit_cast(float, w << 16)
                                           : (float)__builtin_bit_cast(half_t, (uint16_t)w);
        v[8 * b + 2 * j + 1] = DT == kRowsBF16
                                   ? __builtin_bit_cast(float, w & 0xFFFF0000u)
                                   : (float)__builtin_bit_cast(half_t, (uint16_t)(w >> 16));
      }
    }
  }
}
// f16(v * rs) to elements i .. i + 7 and i + 64 .. i + 71 of out.
__device__ __forceinline__ void store_oct(uint16_t* out, size_t i, const float (&v)[16], float rs) {
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    Bytes16 q;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      q.w[j] = (uint32_t)__builtin_bit_cast(uint16_t, to_f16(v[8 * b + 2 * j] * rs)) |
               ((uint32_t)__builtin_bit_cast(uint16_t, to_f16(v[8 * b + 2 * j + 1] * rs)) << 16);
    *reinterpret_cast<Bytes16*>(out + i + 64 * b) = q;
  }
}
// The place of this lane's group of 8 in a grid over (ROWS rows, 128-block), the blocks
// fastest (a wave reads 2 KB runs of a row): first row and element column.  Groups past
// the end repeat the last one's reads (row0 = m: nothing is stored).
struct OctPlace {
  int row0, col;
};
template <int ROWS>
__device__ __forceinline__ OctPlace oct_place(int m, int nblk) {
  const unsigned item = (blockIdx.x * blockDim.x + threadIdx.x) >> 3;
  const unsigned rp = item / (unsigned)nblk, blk = item - rp * (unsigned)nblk;
  return {min(ROWS * (int)rp, m), 128 * (int)blk + 8 * oct_chunk()};
}

// Output transform: one wave per (row, 128-block); a 256-thread workgroup
// covers kTransformRows rows of one 128-block (kTransformRows / 4 per wave,
// their loads issued together).  grid (dim/128, ceil(m / kTransformRows)).
constexpr int kTransformRows = 16;

// xh = f16(H128(f32(rows) * rin) * RS); rin is [E][IC] gathered by row_expert,
// or [IC] when row_expert is null (escha_mlx/msl.py:875-916, 1029-1047).
// DT: the rows' element type; f16 rows are the fused kernel's input, bf16 and
// f32 rows the reference's unfused branch (escha_mlx/dense.py:290-292,
// models/qwen3_5_moe.py:108-110), converted exactly to float32 here with no
// f16 rounding before the transform.
// TWO: the rows are read once for two projections (rin / out and rin1 / out1).
// HBM-bound from some hundred rows on, latency-bound below.  2048 x 5120 f16 rows for
// two projections 23 -> 16.6 us by 8 lanes per block against one wave.  grid: oct_place.
template <int DT, int ROWS, bool TWO = false>
__global__ __launch_bounds__(256) void k_input_transform(const void* __restrict__ rows,
                                                         const float* __restrict__ rin,
                                                         const int* __restrict__ row_expert,
                                                         int m, int IC, float rs,
                                                         uint16_t* __restrict__ out,
                                                         const float* __restrict__ rin1 = nullptr,
                                                         uint16_t* __restrict__ out1 = nullptr) {
  const OctPlace at = oct_place<ROWS>(m, IC / 128);
  float xv[ROWS][16], r[16];
#pragma unroll
  for (int j = 0; j < ROWS; ++j)
    load_oct<DT>(rows, (size_t)min(at.row0 + j, m - 1) * IC + at.col, xv[j]);
  if (!row_expert) load_oct<kRowsF32>(rin, at.col, r);
#pragma unroll
  for (int j = 0; j < ROWS; ++j) {
    const int row = at.row0 + j;
    if (row_expert) load_oct<kRowsF32>(rin, (size_t)row_expert[min(row, m - 1)] * IC + at.col, r);
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = xv[j][i] * r[i];
    h128_oct(v);
    if (row < m) store_oct(out, (size_t)row * IC + at.col, v, rs);
  }
  if constexpr (TWO) {
    load_oct<kRowsF32>(rin1, at.col, r);
#pragma unroll
    for (int j = 0; j < ROWS; ++j) {
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = xv[j][i] * r[i];
      h128_oct(v);
      if (at.row0 + j < m) store_oct(out1, (size_t)(at.row0 + j) * IC + at.col, v, rs);
    }
  }
}

// y = f16((H128(mid) * RS) * rout) [+ bias, added in f32 after the f16 round]
// (escha_mlx/msl.py:919-949, 1050-1067; bias per dense.py:358-361).
// EXP: row_expert is given (rout per row's expert).
template <bool EXP>
__global__ __launch_bounds__(256) void k_output_transform(const float* __restrict__ mid,
                                                          const float* __restrict__ rout,
                                                          const int* __restrict__ row_expert,
                                                          const uint16_t* __restrict__ bias,
                                                          int m, int OC, float rs,
                                                          uint16_t* __restrict__ out) {
  constexpr int RPW = kTransformRows / 4;
  const int blk = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c = blk * 128 + 2 * lane;
  const int row0 = blockIdx.y * kTransformRows + RPW * wave;
  // every load unconditional (rows past m re-read row m - 1 and are not
  // stored), the bias (under its branch) first: a load under a branch waits
  // for all the loads before it
  const uint32_t bw = bias ? *reinterpret_cast<const uint32_t*>(bias + c) : 0u;
  float2 v[RPW], r[RPW];
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int row = min(row0 + j, m - 1);
    v[j] = *reinterpret_cast<const float2*>(mid + (size_t)row * OC + c);
    r[j] = *reinterpret_cast<const float2*>(rout + (EXP ? (size_t)row_expert[row] * OC : 0) + c);
  }
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int row = row0 + j;
    float v0 = v[j].x, v1 = v[j].y;
    h128_wave(v0, v1);
    half_t y0 = to_f16((v0 * rs) * r[j].x);
    half_t y1 = to_f16((v1 * rs) * r[j].y);
    if (bias) {
      y0 = to_f16((float)y0 + (float)__builtin_bit_cast(half_t, (uint16_t)(bw & 0xFFFFu)));
      y1 = to_f16((float)y1 + (float)__builtin_bit_cast(half_t, (uint16_t)(bw >> 16)));
    }
    if (row < m)
      *reinterpret_cast<uint32_t*>(out + (size_t)row * OC + c) =
          (uint32_t)__builtin_bit_cast(uint16_t, y0) | ((uint32_t)__builtin_bit_cast(uint16_t, y1) << 16);
  }
}

// ---------------------------------------------------------------- router
// The wave's largest value in every lane (v_max_f32 over DPP moves and the two
// row swaps; no LDS round trip).
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, lane_xor<1>(v));
  v = fmaxf(v, lane_xor<2>(v));
  v = fmaxf(v, lane_xor<4>(v));
  v = fmaxf(v, lane_xor<8>(v));
  const unsigned x = __builtin_bit_cast(unsigned, v);
  const auto p = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  const unsigned p0 = p[0], p1 = p[1];
  v = fmaxf(__builtin_bit_cast(float, p0), __builtin_bit_cast(float, p1));
  const unsigned y = __builtin_bit_cast(unsigned, v);
  const auto q = __builtin_amdgcn_permlane32_swap(y, y, false, false);
  const unsigned q0 = q[0], q1 = q[1];
  return fmaxf(__builtin_bit_cast(float, q0), __builtin_bit_cast(float, q1));
}

// The top_k of one token's E logits by one wave (NPER = ceil(E / 64) values per
// lane, NaN never chosen): lane k holds the k-th id and value, descending, ties to
// the lower id.  Each pick is a lane-local scan, one wave maximum and a ballot of
// the lanes that hold it (a shuffle reduction of (value, id) pairs waits on twelve
// LDS round trips per pick: 9.5 us for 8 of 256, against 3 us).
template <int NPER>
__device__ __forceinline__ void topk_wave(float (&v)[NPER], int E, int top_k, int& my_id,
                                          float& my_v) {
  const int lane = threadIdx.x & 63;
  my_id = 0;
  my_v = 0.f;
  for (int k = 0; k < top_k; ++k) {
    float bv = -__builtin_inff();
    int bi = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < NPER; ++i) {
      const int e = lane + 64 * i;
      // ids grow with i: a tie keeps the earlier one
      if (e < E && (v[i] > bv || (v[i] == bv && bi == 0x7fffffff))) {
        bv = v[i];
        bi = e;
      }
    }
    const float m = wave_max(bv);
    unsigned long long ties = __ballot(bv == m && bi != 0x7fffffff);
    int id = 0x7fffffff;
    while (ties) {  // the lowest id among the lanes that hold the maximum
      const int l = __builtin_ctzll(ties);
      id = min(id, __builtin_amdgcn_readlane(bi, l));
      ties &= ties - 1;
    }
    if (lane == k) {
      my_id = id;
      my_v = m;
    }
#pragma unroll
    for (int i = 0; i < NPER; ++i)
      if (lane + 64 * i == id) v[i] = -__builtin_inff();
  }
}

// logits [T][E] f32 -> ids [T][k] (descending, ties -> lower id), scores [T][k]
// = softmax over the k selected logits (escha_mlx/ref.py:326-331).
// One wave per token; E <= 64 NPER.  LT: float, or half_t (the router's own f16
// logits, the same values as a float32 copy of them).
template <int NPER, typename LT>
__global__ __launch_bounds__(64) void k_route_topk(const LT* __restrict__ logits, int E,
                                                   int top_k, int* __restrict__ ids,
                                                   float* __restrict__ scores) {
  const int tok = blockIdx.x, lane = threadIdx.x;
  const LT* lg = logits + (size_t)tok * E;
  float v[NPER];
#pragma unroll
  for (int i = 0; i < NPER; ++i) v[i] = (float)lg[min(lane + 64 * i, E - 1)];
  int id;
  float val;
  topk_wave(v, E, top_k, id, val);
  const float top0 =
      __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, val), 0));
  const float ex = expf(val - top0);
  // the denominator in slot order
  float den = 0.f;
  for (int k = 0; k < top_k; ++k)
    den += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ex), k));
  if (lane < top_k) {
    ids[(size_t)tok * top_k + lane] = id;
    scores[(size_t)tok * top_k + lane] = ex / den;
  }
}

// ---------------------------------------------------------------- groups
// Device build_groups (escha_mlx/moe.py:30-78): rows sorted stably by expert,
// each expert padded to a multiple of R, padding slots = m (zero sink row),
// groups past the end = expert -1.  Integer only, one block, deterministic.
// Shared memory holds per-expert counts; E <= 4096.
// The body runs in one block of 1024 threads (k_build_groups, or block 0 of
// k_moe_prep).
// Few rows (E * ceil(m / 64) <= kGroupMaskWords): a bit per (expert, row) in
// LDS; a row's rank within its expert is the popcount of its expert's bits
// below it, so every slot is written once and the only serial step is the
// prefix over the experts' padded counts.  Many rows: each of the 16 waves
// owns a contiguous segment and counts per expert (16 E counters, in the
// mask's LDS: E <= kGroupHistE), the prefix gives each (wave, expert) its first
// slot, and the waves place their segments with no barrier between them
// (16,384 rows of 256 experts; ranking each row by a scan of its chunk's earlier
// rows took 264 us there).  Many rows of more experts: the mask form in chunks.
constexpr int kGroupMaskWords = 4096;
constexpr int kGroupHistE = kGroupMaskWords * 8 / (16 * 4);  // 512

// exclusive prefix over the block (1024 threads) of one int per thread; the
// block's total in *total
__device__ __forceinline__ int block_exclusive_scan(int v, int* s_wsum, int* total) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(inc, o);
    if (lane >= o) inc += t;
  }
  if (lane == 63) s_wsum[wave] = inc;
  __syncthreads();
  int before = 0, all = 0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
    before += w < wave ? s_wsum[w] : 0;
    all += s_wsum[w];
  }
  *total = all;
  return before + inc - v;
}

__device__ void build_groups_mask(const int* __restrict__ row_expert, int m, int E, int R,
                                  int n_groups, int* __restrict__ rows_idx,
                                  int* __restrict__ group_expert, int* s_start,
                                  unsigned long long* s_mask, int* s_wsum,
                                  int* __restrict__ n_active) {
  const int tid = threadIdx.x, nt = blockDim.x;
  const int nw = (m + 63) >> 6;
  for (int i = tid; i < E * nw; i += nt) s_mask[i] = 0ull;
  __syncthreads();
  for (int r = tid; r < m; r += nt)
    atomicOr(&s_mask[row_expert[r] * nw + (r >> 6)], 1ull << (r & 63));
  __syncthreads();
  // experts 4 tid .. 4 tid + 3: counts, padded counts, first slots
  int cnt[4], pad[4], sum = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int e = 4 * tid + j;
    cnt[j] = 0;
    if (e < E)
      for (int w = 0; w < nw; ++w) cnt[j] += __popcll(s_mask[e * nw + w]);
    pad[j] = (cnt[j] + R - 1) / R * R;
    sum += pad[j];
  }
  int total;
  int start = block_exclusive_scan(sum, s_wsum, &total);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int e = 4 * tid + j;
    if (e < E) {
      s_start[e] = start;
      // the expert's groups and its padding slots (= m)
      for (int g = start / R; g < (start + pad[j]) / R; ++g) group_expert[g] = e;
      for (int i = cnt[j]; i < pad[j]; ++i) rows_idx[start + i] = m;
    }
    start += pad[j];
  }
  // past the last expert: padding slots and groups of expert -1
  if (n_active && tid == 0) *n_active = total / R;
  for (int i = total + tid; i < n_groups * R; i += nt) rows_idx[i] = m;
  for (int g = total / R + tid; g < n_groups; g += nt) group_expert[g] = -1;
  __syncthreads();
  // each row at its expert's first slot + the rows of its expert before it
  for (int r = tid; r < m; r += nt) {
    const int e = row_expert[r], w0 = r >> 6;
    const unsigned long long* me = s_mask + e * nw;
    int rank = __popcll(me[w0] & ((1ull << (r & 63)) - 1ull));
    for (int w = 0; w < w0; ++w) rank += __popcll(me[w]);
    rows_idx[s_start[e] + rank] = r;
  }
}

// The segment form (E <= kGroupHistE): s_hist[wave][E] holds the wave's rows
// per expert (s_cnt: the wave's own), then the slot of its next row of that
// expert.
__device__ void build_groups_hist(const int* __restrict__ row_expert, int m, int E, int R,
                                  int n_groups, int* __restrict__ rows_idx,
                                  int* __restrict__ group_expert, int* s_hist, int* s_wsum,
                                  int* __restrict__ n_active) {
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int i = tid; i < 16 * E; i += nt) s_hist[i] = 0;
  __syncthreads();
  const int seg = ((m + 15) / 16 + 63) / 64 * 64;
  const int r0 = wave * seg, r1 = min(m, r0 + seg);
  int* s_cnt = s_hist + wave * E;
  for (int r = r0 + lane; r < r1; r += 64) atomicAdd(&s_cnt[row_expert[r]], 1);
  __syncthreads();
  // expert tid: its padded count, first slot, groups and padding slots (= m),
  // and each wave's first slot
  int cnt = 0;
  if (tid < E)
    for (int w = 0; w < 16; ++w) cnt += s_hist[w * E + tid];
  const int pad = (cnt + R - 1) / R * R;
  int total;
  const int start = block_exclusive_scan(pad, s_wsum, &total);
  if (tid < E) {
    int slot = start;
    for (int w = 0; w < 16; ++w) {
      const int k = s_hist[w * E + tid];
      s_hist[w * E + tid] = slot;
      slot += k;
    }
    for (int g = start / R; g < (start + pad) / R; ++g) group_expert[g] = tid;
    for (int i = cnt; i < pad; ++i) rows_idx[start + i] = m;
  }
  if (n_active && tid == 0) *n_active = total / R;
  for (int i = total + tid; i < n_groups * R; i += nt) rows_idx[i] = m;
  for (int g = total / R + tid; g < n_groups; g += nt) group_expert[g] = -1;
  __syncthreads();
  // 64 rows at a time: a row's rank among them is the number of lower lanes
  // with the same expert, found bit by bit
  int e_next = r0 + lane < r1 ? row_expert[r0 + lane] : 0;
  for (int r = r0; r < r1; r += 64) {
    const int e = e_next;
    const bool ok = r + lane < r1;
    if (r + 64 + lane < r1) e_next = row_expert[r + 64 + lane];
    unsigned long long same = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 9; ++b) {
      const unsigned long long bit = __ballot((e >> b) & 1);
      same &= (e >> b) & 1 ? bit : ~bit;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull)), n = __popcll(same);
    if (ok) {
      const int slot = s_cnt[e];
      rows_idx[slot + rank] = r + lane;
      if (rank == n - 1) s_cnt[e] = slot + n;
    }
    // the slots just written are read by the next 64 rows
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

// Places rows row0 .. row0 + n - 1 (row_expert: of row0; n <= 64 nw) from their
// experts' next slots s_cnt; the masks are zero before and after.
__device__ void build_groups_chunk(const int* __restrict__ row_expert, int row0, int n, int E,
                                   int nw, int* __restrict__ rows_idx, int* s_cnt,
                                   unsigned long long* s_mask) {
  const int tid = threadIdx.x, nt = blockDim.x;
  for (int r = tid; r < n; r += nt)
    atomicOr(&s_mask[row_expert[r] * nw + (r >> 6)], 1ull << (r & 63));
  __syncthreads();
  for (int r = tid; r < n; r += nt) {
    const int e = row_expert[r], w0 = r >> 6;
    const unsigned long long* me = s_mask + e * nw;
    int rank = __popcll(me[w0] & ((1ull << (r & 63)) - 1ull));
    for (int w = 0; w < w0; ++w) rank += __popcll(me[w]);
    rows_idx[s_cnt[e] + rank] = row0 + r;
  }
  __syncthreads();
  for (int r = tid; r < n; r += nt) {
    const int e = row_expert[r];
    atomicAdd(&s_cnt[e], 1);
  }
  for (int i = tid; i < E * nw; i += nt) s_mask[i] = 0ull;
  __syncthreads();
}

// n_active (when not null): the number of groups that hold rows.
__device__ void build_groups_block(const int* __restrict__ row_expert, int m, int E, int R,
                                   int n_groups, int* __restrict__ rows_idx,
                                   int* __restrict__ group_expert,
                                   int* __restrict__ n_active = nullptr) {
  // first padded slot of each expert
  __shared__ int s_start[4096];
  __shared__ unsigned long long s_mask[kGroupMaskWords];  // [E][nw]
  __shared__ int s_wsum[16];
  if ((long)E * ((m + 63) >> 6) <= kGroupMaskWords) {
    build_groups_mask(row_expert, m, E, R, n_groups, rows_idx, group_expert, s_start, s_mask,
                      s_wsum, n_active);
    return;
  }
  if (E <= kGroupHistE) {
    build_groups_hist(row_expert, m, E, R, n_groups, rows_idx, group_expert,
                      reinterpret_cast<int*>(s_mask), s_wsum, n_active);
    return;
  }
  const int tid = threadIdx.x, nt = blockDim.x;
  const int nw = kGroupMaskWords / E;  // mask words per expert, 64 rows each
  int* s_cnt = s_start;  // rows per expert, then each expert's next slot
  for (int e = tid; e < E; e += nt) s_cnt[e] = 0;
  for (int i = tid; i < E * nw; i += nt) s_mask[i] = 0ull;
  __syncthreads();
  for (int r = tid; r < m; r += nt) atomicAdd(&s_cnt[row_expert[r]], 1);
  __syncthreads();
  // experts 4 tid .. 4 tid + 3: padded counts, first slots, their groups and
  // their padding slots (= m)
  int cnt[4], sum = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    cnt[j] = 4 * tid + j < E ? s_cnt[4 * tid + j] : 0;
    sum += (cnt[j] + R - 1) / R * R;
  }
  int total;
  int start = block_exclusive_scan(sum, s_wsum, &total);
  for (int j = 0; j < 4; ++j) {
    const int e = 4 * tid + j, pad = (cnt[j] + R - 1) / R * R;
    if (e < E) {
      s_cnt[e] = start;
      for (int g = start / R; g < (start + pad) / R; ++g) group_expert[g] = e;
      for (int i = cnt[j]; i < pad; ++i) rows_idx[start + i] = m;
    }
    start += pad;
  }
  if (n_active && tid == 0) *n_active = total / R;
  for (int i = total + tid; i < n_groups * R; i += nt) rows_idx[i] = m;
  for (int g = total / R + tid; g < n_groups; g += nt) group_expert[g] = -1;
  // stable placement, one chunk of rows at a time
  __syncthreads();
  for (int c0 = 0; c0 < m; c0 += 64 * nw)
    build_groups_chunk(row_expert + c0, c0, min(64 * nw, m - c0), E, nw, rows_idx, s_cnt, s_mask);
}

__global__ __launch_bounds__(1024) void k_build_groups(const int* __restrict__ row_expert, int m,
                                                       int E, int R, int n_groups,
                                                       int* __restrict__ rows_idx,
                                                       int* __restrict__ group_expert) {
  build_groups_block(row_expert, m, E, R, n_groups, rows_idx, group_expert);
}

}  // namespace esc
