// libescha_hip: the C ABI declared in include/escha_hip.h.
// One translation unit so the device decode table is a single symbol.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <atomic>
#include <mutex>
#include <string>

#include "../../include/escha_hip.h"
#include "fused.hpp"
#include "mfma.hpp"
#include "linear.hpp"
#include "q8.hpp"
#include "probe.hpp"
#include "layers.hpp"
#include "proj.hpp"
#include "grouped.hpp"

namespace {

thread_local std::string g_err;

int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}

#define ESC_REQUIRE(cond, ...) \
  do {                         \
    if (!(cond)) return fail(ESC_EINVAL, __VA_ARGS__); \
  } while (0)

int hip_check(hipError_t e, const char* what) {
  if (e != hipSuccess) return fail(ESC_EHIP, "%s: %s", what, hipGetErrorString(e));
  return ESC_OK;
}

int launched(const char* what) { return hip_check(hipGetLastError(), what); }

inline hipStream_t S(void* s) { return reinterpret_cast<hipStream_t>(s); }

constexpr int kMaxDevices = 64;
std::mutex g_init_mu;
bool g_lut_ready[kMaxDevices];

// The decode table is part of the device image; this records that a table
// decode was asked for on the device (esc_moe_expert_path_static asks that
// esc_init or such a call came first).
int ensure_lut() {
  int dev = 0;
  if (int rc = hip_check(hipGetDevice(&dev), "hipGetDevice")) return rc;
  if (dev < 0 || dev >= kMaxDevices) return fail(ESC_EINVAL, "device index %d out of range", dev);
  std::lock_guard<std::mutex> lk(g_init_mu);
  g_lut_ready[dev] = true;
  return ESC_OK;
}

bool lut_ready() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return false;
  std::lock_guard<std::mutex> lk(g_init_mu);
  return g_lut_ready[dev];
}

int ensure_scratch(void** out);
// Device-wide bounded-wait flag of the single persistent expert launch
// (k_moe_fused): one int per device in pinned, coherent host memory, set by a
// workgroup that gave up a wait and read by the host with no synchronisation,
// so a later call can report the failure.  Allocated at set-up (esc_init, or
// the first esc_moe_expert_path call on the device); the allocation-free entry
// point only uses it once it exists.
int* g_wait_flag[kMaxDevices];
int* g_wait_flag_dev[kMaxDevices];
std::atomic<int> g_spin_limit{esc::kSpinLimit};

int ensure_wait_flag() {
  int dev = 0;
  if (int rc = hip_check(hipGetDevice(&dev), "hipGetDevice")) return rc;
  if (dev < 0 || dev >= kMaxDevices) return fail(ESC_EINVAL, "device index %d out of range", dev);
  std::lock_guard<std::mutex> lk(g_init_mu);
  if (g_wait_flag[dev]) return ESC_OK;
  void* h = nullptr;
  if (int rc = hip_check(hipHostMalloc(&h, 64, hipHostMallocMapped | hipHostMallocCoherent),
                         "hipHostMalloc"))
    return rc;
  void* d = nullptr;
  if (int rc = hip_check(hipHostGetDevicePointer(&d, h, 0), "hipHostGetDevicePointer")) {
    (void)hipHostFree(h);
    return rc;
  }
  *static_cast<volatile int*>(h) = 0;
  g_wait_flag_dev[dev] = static_cast<int*>(d);
  g_wait_flag[dev] = static_cast<int*>(h);
  return ESC_OK;
}

// Takes the device's flag: ESC_ETIMEOUT (flag cleared) if a single persistent
// launch on this device gave up a wait since the last take; *dev_flag is the
// flag's device address for the next launch (null before set-up).
int take_wait_error(int** dev_flag) {
  *dev_flag = nullptr;
  int dev = 0;
  if (int rc = hip_check(hipGetDevice(&dev), "hipGetDevice")) return rc;
  if (dev < 0 || dev >= kMaxDevices) return fail(ESC_EINVAL, "device index %d out of range", dev);
  int* h = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_init_mu);
    h = g_wait_flag[dev];
    *dev_flag = g_wait_flag_dev[dev];
  }
  if (h && __atomic_exchange_n(h, 0, __ATOMIC_ACQ_REL) != 0)
    return fail(ESC_ETIMEOUT,
                "an earlier single-launch expert-path call on device %d gave up a bounded wait: "
                "its outputs are NaN (this call did not run)",
                dev);
  return ESC_OK;
}

int check_proj(int K, int IC, int OC) {
  ESC_REQUIRE(K == 2 || K == 3, "escha code implies K=%d; this runtime implements K in [2, 3]", K);
  ESC_REQUIRE(IC > 0 && OC > 0 && IC % 128 == 0 && OC % 128 == 0,
              "escha linear dimensions must be positive multiples of 128, got %dx%d", IC, OC);
  return ESC_OK;
}

// ---- dispatch helpers over compile-time parameters
template <template <int, bool> class F, typename... A>
int by_k_lut(int K, int lut, A... a) {
  if (K == 2) return lut ? F<2, true>::run(a...) : F<2, false>::run(a...);
  return lut ? F<3, true>::run(a...) : F<3, false>::run(a...);
}

template <int K, bool LUT>
struct DecodeF {
  static int run(const uint32_t* code, int IC, int OC, uint16_t* w, hipStream_t s) {
    const int TK = IC / 16, TN = OC / 16;
    hipLaunchKernelGGL((esc::k_decode_tiles<K, LUT>), dim3(TK * TN), dim3(256), 0, s, code, TN,
                       OC, w);
    return launched("k_decode_tiles");
  }
};

template <int K, bool LUT, int MODE>
struct ExactF {
  template <int R>
  static int go(const uint16_t* xh, const uint32_t* code, const int* a, const int* b, int M,
                int n_groups, int TK, int TN, float* mid, hipStream_t s) {
    hipLaunchKernelGGL((esc::k_gemm_exact<K, LUT, R, MODE>), dim3(TN / 8, n_groups), dim3(512),
                       0, s, xh, code, a, b, M, TK, TN, mid);
    return launched("k_gemm_exact");
  }
  static int run(int R, const uint16_t* xh, const uint32_t* code, const int* a, const int* b,
                 int M, int n_groups, int TK, int TN, float* mid, hipStream_t s) {
    switch (R) {
      case 1: return go<1>(xh, code, a, b, M, n_groups, TK, TN, mid, s);
      case 2: return go<2>(xh, code, a, b, M, n_groups, TK, TN, mid, s);
      case 3: return go<3>(xh, code, a, b, M, n_groups, TK, TN, mid, s);
      case 4: return go<4>(xh, code, a, b, M, n_groups, TK, TN, mid, s);
      case 8: return go<8>(xh, code, a, b, M, n_groups, TK, TN, mid, s);
      case 12: return go<12>(xh, code, a, b, M, n_groups, TK, TN, mid, s);
      case 16: return go<16>(xh, code, a, b, M, n_groups, TK, TN, mid, s);
    }
    return fail(ESC_EINVAL, "rows per group R=%d not in {1,2,3,4,8,12,16}", R);
  }
};

template <int MODE>
int exact_dispatch(int K, int lut, int R, const uint16_t* xh, const uint32_t* code,
                   const int* a, const int* b, int M, int n_groups, int TK, int TN, float* mid,
                   hipStream_t s) {
  if (K == 2)
    return lut ? ExactF<2, true, MODE>::run(R, xh, code, a, b, M, n_groups, TK, TN, mid, s)
               : ExactF<2, false, MODE>::run(R, xh, code, a, b, M, n_groups, TK, TN, mid, s);
  return lut ? ExactF<3, true, MODE>::run(R, xh, code, a, b, M, n_groups, TK, TN, mid, s)
             : ExactF<3, false, MODE>::run(R, xh, code, a, b, M, n_groups, TK, TN, mid, s);
}

template <int K, bool LUT>
struct ExactOutF {
  template <int R>
  static int go(const uint16_t* xh, const uint32_t* code, const float* rout, int M, int TK,
                int TN, float rs, uint16_t* out, hipStream_t s) {
    hipLaunchKernelGGL((esc::k_gemm_exact_out<K, LUT, R>), dim3(TN / 8, (M + R - 1) / R),
                       dim3(512), 0, s, xh, code, rout, M, TK, TN, rs, out);
    return launched("k_gemm_exact_out");
  }
  static int run(int R, const uint16_t* xh, const uint32_t* code, const float* rout, int M,
                 int TK, int TN, float rs, uint16_t* out, hipStream_t s) {
    switch (R) {
      case 1: return go<1>(xh, code, rout, M, TK, TN, rs, out, s);
      case 2: return go<2>(xh, code, rout, M, TK, TN, rs, out, s);
      case 4: return go<4>(xh, code, rout, M, TK, TN, rs, out, s);
      case 8: return go<8>(xh, code, rout, M, TK, TN, rs, out, s);
    }
    return fail(ESC_EINVAL, "rows per group R=%d not in {1,2,4,8}", R);
  }
};

// f(std::integral_constant<int, DT>) for the row element type dtype.
template <typename F>
void by_rows_type(int dtype, F f) {
  if (dtype == ESC_ROWS_BF16) f(std::integral_constant<int, esc::kRowsBF16>{});
  else if (dtype == ESC_ROWS_F32) f(std::integral_constant<int, esc::kRowsF32>{});
  else f(std::integral_constant<int, esc::kRowsF16>{});
}

// ---- split-K GEMV geometry: KS kt per block (multiple of 4, divides TK)
int fast_splits(int K, int M, int TK, int TN, int target = 1024) {
  const int tpw = K == 2 ? 16 : 8;
  const int per_split = ((TN + tpw - 1) / tpw) * M;  // blocks per kt split
  int S = 1;
  // aim for >= target blocks of 4 waves while keeping >= 4 kt per block
  while (per_split * S < target && TK % (S * 2 * 4) == 0 && TK / (S * 2) >= 4) S *= 2;
  return S;
}

template <int K, bool LUT>
struct FastF {
  static int run(const uint16_t* xh, const uint32_t* code, const int* row_expert, int M, int TK,
                 int TN, int S, float* part, hipStream_t s) {
    const int tpw = K == 2 ? 16 : 8;
    hipLaunchKernelGGL((esc::k_gemv_fast<K, LUT>), dim3((TN + tpw - 1) / tpw, M, S), dim3(256), 0, s, xh,
                       code, row_expert, M, TK, TN, TK / S, part);
    return launched("k_gemv_fast");
  }
};

template <int K, bool LUT>
struct FastRowsF {
  template <int R>
  static int go(const uint16_t* xh, const uint32_t* code, int M, int TK, int TN, int S,
                float* part, hipStream_t s) {
    const int tpw = K == 2 ? 16 : 8;
    hipLaunchKernelGGL((esc::k_gemv_fast_rows<K, LUT, R>), dim3((TN + tpw - 1) / tpw, (M + R - 1) / R, S),
                       dim3(256), 0, s, xh, code, nullptr, nullptr, M, TK, TN, TK / S, part);
    return launched("k_gemv_fast_rows");
  }
  static int run(int R, const uint16_t* xh, const uint32_t* code, int M, int TK, int TN, int S,
                 float* part, hipStream_t s) {
    switch (R) {
      case 2: return go<2>(xh, code, M, TK, TN, S, part, s);
      case 4: return go<4>(xh, code, M, TK, TN, S, part, s);
      case 8: return go<8>(xh, code, M, TK, TN, S, part, s);
    }
    return fail(ESC_EINVAL, "rows per block R=%d not in {2,4,8}", R);
  }
};

// Compute units of the current device (queried once per device).
int device_cus() {
  static int cus[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cus[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

// The launch of a transform by 8 lanes per 128-block: f(rows per lane group as a
// constant, grid, block).  Two rows per group (the scales read once) in workgroups of
// 256 once those fill eight waves per CU; below that one row, in single waves, for more
// of them in flight.
template <typename F>
void oct_launch(int m, int dim, F f) {
  const long two = (long)(dim / 128) * ((m + 1) / 2);
  if (two >= 64L * device_cus())
    f(std::integral_constant<int, 2>{}, dim3((unsigned)((two + 31) / 32)), dim3(256));
  else
    f(std::integral_constant<int, 1>{}, dim3((unsigned)(((long)(dim / 128) * m + 7) / 8)), dim3(64));
}

// Row blocks of 16 per k_gemm_mma2 workgroup (NRB in {2,4,6,8}) and splits S of
// the K steps (4 kt each).  A step of one workgroup takes about 0.66 + 0.055 NRB
// us of its CU (K = 3; decode, then MFMAs), a lone workgroup on a CU 1.24 times
// that, and no step less than 1.05 + 0.02 NRB us (the code's latency over the two
// steps it is requested ahead).  A launch takes what the busiest CU holds; splits add
// their float32 partials, written and read back at about 4.5 TB/s, and the
// reduction launch.  Measured on MI355X (whole linear, unsplit against the plan's
// choice; a sweep of 19 (NRB, S) pairs finds nothing more than 5 % faster):
// K = 3 17408 -> 5120, 16 / 40 / 256 / 2048 rows 284 / 287 / 291 / 526 us against
// 37 / 42 / 88 / 446; K = 2 5120 -> 5120, 16 / 256 / 2048 rows 90 / 96 / 165
// against 25 / 44 / 155; K = 2 2048 -> 4096, 16 / 600 rows 42 / 53 against 25 /
// 37.  A split keeps at least kMmaMinSteps steps.
constexpr int kMmaMinSteps = 10;
constexpr size_t kMmaPartMax = size_t(128) << 20;
struct MmaPlan {
  int nrb, S;
  size_t part_bytes;
};
size_t mma2_part_bytes(int M, int TN, int S) {
  return (size_t)S * ((M + 15) / 16) * ((TN + 15) / 16) * 16384;
}
// fixed_S > 0: that many splits; ncb2: column blocks of a second product in the
// launch.
MmaPlan mma_plan(int M, int TK, int TN, bool split, int fixed_S = 0, int ncb2 = 0) {
  const int cus = device_cus(), NS = TK / 4, ncb = (TN + 15) / 16 + ncb2;
  MmaPlan best{8, 1, 0};
  double best_cost = 1e30;
  for (int S = 1; S == 1 || (split && S * kMmaMinSteps <= NS); ++S) {
    const size_t part = S > 1 ? mma2_part_bytes(M, TN, S) : 0;
    if (part > kMmaPartMax) break;
    if (fixed_S && S != fixed_S) continue;
    const double extra = S > 1 ? 2.0 * part / 4.5e6 + 5.0 : 0.0;
    for (int nrb = 8; nrb >= 2; nrb -= 2) {
      const long wgs = (long)((M + 16 * nrb - 1) / (16 * nrb)) * ncb * S;
      const long n = (wgs + cus - 1) / cus;
      const double step = std::max((n + (n & 1 ? 0.24 : 0.0)) * (0.66 + 0.055 * nrb),
                                   1.05 + 0.02 * nrb);
      const double cost = step * ((NS + S - 1) / S) + extra;
      // a split has to pay: 5 % over one launch
      if (cost < best_cost * (S > 1 && best.S == 1 ? 0.95 : 0.999)) {
        best_cost = cost;
        best = {nrb, S, part};
      }
    }
  }
  return best;
}

template <int MODE>
int gemm_mma2_launch(int K, int nrb, int S, const esc::MmaArgs& a, hipStream_t s,
                     const esc::MmaArgs* second = nullptr) {
  const int rb = (a.M + 16 * nrb - 1) / (16 * nrb), n0 = rb * ((a.TN + 15) / 16);
  const dim3 grid(n0 + (second ? rb * ((second->TN + 15) / 16) : 0), S);
  const esc::MmaArgs& b = second ? *second : a;
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, a, b, n0); };
  if (K == 2) {
    if (nrb == 2) go(esc::k_gemm_mma2<2, 2, MODE>);
    else if (nrb == 4) go(esc::k_gemm_mma2<2, 4, MODE>);
    else if (nrb == 6) go(esc::k_gemm_mma2<2, 6, MODE>);
    else go(esc::k_gemm_mma2<2, 8, MODE>);
  } else {
    if (nrb == 2) go(esc::k_gemm_mma2<3, 2, MODE>);
    else if (nrb == 4) go(esc::k_gemm_mma2<3, 4, MODE>);
    else if (nrb == 6) go(esc::k_gemm_mma2<3, 6, MODE>);
    else go(esc::k_gemm_mma2<3, 8, MODE>);
  }
  return launched("k_gemm_mma2");
}

// The splits' partials of a summed and output-transformed.
int mma2_reduce(int K, int S, const esc::MmaArgs& a, hipStream_t s) {
  const dim3 grid((a.TN + 15) / 16, (a.M + 15) / 16);
  if (K == 2)
    hipLaunchKernelGGL(esc::k_mma2_reduce<2>, grid, dim3(256), 0, s, a, S);
  else
    hipLaunchKernelGGL(esc::k_mma2_reduce<3>, grid, dim3(256), 0, s, a, S);
  return launched("k_mma2_reduce");
}

// The many-row GEMM with its output transform: one launch, or the splits'
// partials into a.mid (plan.part_bytes) and their reduction.
int gemm_mma2_out(int K, const MmaPlan& plan, const esc::MmaArgs& a, hipStream_t s) {
  if (plan.S == 1) return gemm_mma2_launch<esc::kMmaOut>(K, plan.nrb, 1, a, s);
  if (int rc = gemm_mma2_launch<esc::kMmaPart>(K, plan.nrb, plan.S, a, s)) return rc;
  return mma2_reduce(K, plan.S, a, s);
}

// ---- one-launch linear for M < 16 (linear.hpp)
constexpr int kLinearSmallRows = 16;
constexpr int kLinearSmallRowsLut = 8;

// Linears below kLinearSmallRows rows read 16-bit rows only.
int check_rows_type(int dtype, int M) {
  ESC_REQUIRE(dtype == ESC_ROWS_F16 || dtype == ESC_ROWS_BF16 ||
                  (dtype == ESC_ROWS_F32 && (M >= kLinearSmallRows || M == 0)),
              "row element type %d with %d rows", dtype, M);
  return ESC_OK;
}

// k_proj_rows1: partial slots per 256-column group, at least the workgroups
// a group of TK units can span: every workgroup holds at least 8 units when
// there are several (at most ceil(n / 16) workgroups for n units)
int rows1_maxc(int TK) { return TK / 8 + 2; }
// K=3 step pairs of every 8 that k_proj_rows1 decodes from the table
constexpr int kTablePairs3 = 4;

// One row (M = 1): the persistent table-mix kernel (k_proj_rows1) for a
// projection of at least kRows1MinUnits units (kt x 256-column groups), the
// one-launch split-K kernel (k_linear_small) by hash otherwise, whichever decode was
// asked for (the two decodes give the same weights).  Measured on MI355X, per call:
// K=2 5120 -> 17408 and 17408 -> 5120 (21,760 units) 19.5 and 20.2 us in the
// persistent kernel against 28.1 and 28.9 us, 8192 x 8192 (16,384 units) 16.3
// against 21.1 us; K=3 21.1 and 22.3 against 25.8 and 26.7 us; K=2 5120 x 5120 (6,400
// units, HIP-graph replay) 14.8 against 12.35 us.
constexpr long kRows1MinUnits = 16384;
bool rows1_single(int M, int IC, int OC) {
  return M == 1 && OC % 256 == 0 && (long)(IC / 16) * (OC / 256) >= kRows1MinUnits;
}
size_t rows1_part_bytes(int TK, int TN) { return (size_t)(TN / 16) * rows1_maxc(TK) * 256 * 4; }

struct LinearPlan {
  int R, S, KS, groups, row_groups;
  size_t off_part, off_cnt, off_xh, off_mid, total;
  MmaPlan mma;        // 16 rows and more
  size_t min_total;   // enough without splits
};

// Fewest splits that reach the workgroup target: more splits mean more
// float32 partials through the device-coherent path and a longer last-arriver
// sum; the table path also stages 128 KiB of LDS per workgroup.
LinearPlan linear_plan(int M, int K, int IC, int OC, bool lut) {
  LinearPlan p{};
  const int TK = IC / 16, TN = OC / 16, tpw = K == 2 ? 16 : 8;
  auto al = [](size_t v) { return (v + 255) & ~size_t(255); };
  if (M < kLinearSmallRows) {
    // every row of the group shares each decoded weight (one B column of
    // the matrix-core multiply each); the table path's LDS holds 8 rows
    p.R = std::min(M, lut ? kLinearSmallRowsLut : kLinearSmallRows - 1);
    p.groups = (TN + tpw - 1) / tpw;
    const int nb = TK / 8;  // 128-input blocks
    // fewest splits (largest KS <= 64) that reach `target` workgroups
    auto splits = [&](int row_groups, int target) {
      int best = nb;
      for (int S = 1; S <= std::min(nb, 64); ++S) {
        if (nb % S || 8 * (nb / S) > 64) continue;
        best = S;
        if (p.groups * row_groups * S >= target) break;
      }
      return best;
    };
    // Several rows by hash: each split's float32 partials (written and summed
    // back through the device-coherent level) grow with the rows, so fewer
    // splits than one row wants; and two row groups when one group at its
    // fewest splits leaves the GPU short of workgroups (each group decodes
    // the weights once, the partials halve again).  Measured on MI355X, K=2
    // 5120 x 5120: 4 rows 21.3 us at 200 workgroups against 23.9 us at 400;
    // 15 rows 30.9 us as 8 + 7 rows against 36.0 us as one group.
    if (!lut && M > 1 && p.R > kLinearSmallRowsLut && p.groups * splits(1, 0) < 256)
      p.R = (M + 1) / 2;
    p.row_groups = (M + p.R - 1) / p.R;
    // measured best on MI355X for 2048..17408 shapes
    const int target = lut ? 128 : M > 1 ? 200 : 256;
    p.S = splits(p.row_groups, target);
    p.KS = 8 * (nb / p.S);
    // counters first, sized for the most row groups either plan of this M
    // has (the table plan's 8-row groups), so that neither plan's partials
    // start inside the other's counters: one zero-filled workspace serves the
    // table and the hash plan alike
    const int rg_max = (M + kLinearSmallRowsLut - 1) / kLinearSmallRowsLut;
    p.off_cnt = 0;
    p.off_part = al((size_t)p.groups * std::max(p.row_groups, rg_max) * 4);
    p.total = p.off_part + al((size_t)p.S * M * OC * 4);
    // one row, OC a multiple of 256: room for the persistent kernel
    // (k_proj_rows1, also esc_linear_multi's), whose counters (one per 256
    // columns) fit in the ones above and whose partials start at off_part
    if (M == 1 && TN % 16 == 0)
      p.total = std::max(p.total, p.off_part + al(rows1_part_bytes(TK, TN)));
  } else {
    // the splits' partials, or the M x OC floats that a workspace always had
    p.mma = mma_plan(M, TK, TN, true);
    p.off_xh = 0;
    p.off_mid = al((size_t)M * IC * 2);
    p.min_total = p.off_mid + al((size_t)M * OC * 4);
    p.total = p.off_mid + al(std::max((size_t)M * OC * 4, p.mma.part_bytes));
  }
  return p;
}

esc::LinearSmallArgs small_args(const void* x, const float* rin, const uint32_t* code,
                                const float* rout, const uint16_t* bias, int M, int TK, int TN,
                                const LinearPlan& lp, float rs, char* ws, void* y, int dt,
                                int ydt, const void* x2 = nullptr) {
  return {static_cast<const uint16_t*>(x), rin, code, rout, bias, M, TK, TN, lp.KS, lp.R, lp.S,
          lp.groups, lp.row_groups, rs, reinterpret_cast<float*>(ws + lp.off_part),
          reinterpret_cast<int*>(ws + lp.off_cnt), y, static_cast<const uint16_t*>(x2), dt, ydt};
}

// one row: VALU GEMV; several rows: matrix-core row-blocked GEMM
template <int K, bool ACT>
int linear_small_launch(const esc::LinearSmallArgs& a, hipStream_t s) {
  if (a.R < 1 || a.R > kLinearSmallRows)
    return fail(ESC_EINVAL, "rows per group %d > %d", a.R, kLinearSmallRows);
  const dim3 grid(a.groups, a.row_groups, a.S);
  if (a.R == 1)
    hipLaunchKernelGGL((esc::k_linear_small<K, 1, ACT>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((esc::k_linear_small<K, kLinearSmallRows, ACT>), grid, dim3(256), 0, s, a);
  return launched("k_linear_small");
}

template <int K0, int K1>
int linear_pair_launch(const esc::LinearSmallArgs& a0, const esc::LinearSmallArgs& a1,
                       hipStream_t s) {
  constexpr int RMAX = kLinearSmallRows;
  if (a0.R != a1.R || a0.R < 1 || a0.R > RMAX)
    return fail(ESC_EINVAL, "rows per group %d / %d (max %d)", a0.R, a1.R, RMAX);
  const long n = (long)a0.groups * a0.row_groups * a0.S + (long)a1.groups * a1.row_groups * a1.S;
  if (a0.R == 1)
    hipLaunchKernelGGL((esc::k_linear_pair<K0, K1, 1>), dim3(n), dim3(256), 0, s, a0, a1);
  else
    hipLaunchKernelGGL((esc::k_linear_pair<K0, K1, RMAX>), dim3(n), dim3(256), 0, s, a0, a1);
  return launched("k_linear_pair");
}

int linear_pair_k(int K0, int K1, const esc::LinearSmallArgs& a0, const esc::LinearSmallArgs& a1,
                  hipStream_t s) {
  if (K0 == 2) return K1 == 2 ? linear_pair_launch<2, 2>(a0, a1, s)
                              : linear_pair_launch<2, 3>(a0, a1, s);
  return K1 == 2 ? linear_pair_launch<3, 2>(a0, a1, s) : linear_pair_launch<3, 3>(a0, a1, s);
}

// k_proj_rows1 over a.np projections whose x .. TK, TN are filled: each
// projection's plan from its own shape (one workgroup per CU, or more when a
// wave would run more than kProjMaxP units), its workgroups after the
// previous projection's.  K=2 decodes kTablePairsLayers of 8 pairs from the
// table, K=3 4 of 8, whichever decode was asked for (q, k and v of 5120 inputs in
// one launch, K=2: 18.7 us against 20.8 by hash alone; level at 2048 and 4096).
template <int K, int NT, bool ACT>
int launch_rows1_k(const esc::ProjArgs& a, int grid, hipStream_t s) {
  static std::once_flag once;
  static hipError_t err = hipSuccess;
  std::call_once(once, [] {
    err = hipFuncSetAttribute((const void*)esc::k_proj_rows1<K, NT, ACT>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, 65536 * 2);
  });
  if (int rc = hip_check(err, "hipFuncSetAttribute")) return rc;
  hipLaunchKernelGGL((esc::k_proj_rows1<K, NT, ACT>), dim3(grid), dim3(64 * esc::kProjWaves), 65536 * 2,
                     s, a);
  return launched("k_proj_rows1");
}

// workgroups for n units: wgs, fewer when a wave would get fewer than two
// units, more when it would get more than kProjMaxP.  (Measured on MI355X:
// spreading 6,400 units over 256 workgroups, one or two per wave, is 5 %
// slower than 200 workgroups of two per wave -- more partials per group; 5 to
// 6 units per wave over 256 workgroups beat 6 over 227 by 2 %.)
int rows1_workgroups(long n, long wgs) {
  const long w = esc::kProjWaves;
  return (int)std::max(std::min(wgs, (n + 2 * w - 1) / (2 * w)),
                       (n + w * esc::kProjMaxP - 1) / (w * esc::kProjMaxP));
}

// merged: the workgroups shared out over the projections by their units
// (one round of workgroups for several small projections); otherwise each
// projection's from its own size alone, so that its outputs are those of
// its own launch.  With x2 (one projection) the row is the MLP activation of x
// and x2.
int launch_rows1(esc::ProjArgs& a, int K, hipStream_t s, bool merged = false) {
  const int cus = device_cus();
  long total = 0;
  for (int i = 0; i < a.np; ++i) {
    ESC_REQUIRE((long)(a.pr[i].TN / 16) * a.pr[i].TK < (1L << 28), "projection too large");
    total += (long)(a.pr[i].TN / 16) * a.pr[i].TK;
  }
  long grid = 0;
  for (int i = 0; i < a.np; ++i) {
    esc::ProjOne& q = a.pr[i];
    q.n = (q.TN / 16) * q.TK;
    q.G = rows1_workgroups(q.n, merged ? std::max(1L, (cus * (long)q.n + total / 2) / total) : cus);
    q.maxc = rows1_maxc(q.TK);
    q.wg0 = (int)grid;
    grid += q.G;
  }
  if (a.pr[0].x2)
    return K == 2 ? launch_rows1_k<2, esc::kTablePairsLayers, true>(a, (int)grid, s)
                  : launch_rows1_k<3, kTablePairs3, true>(a, (int)grid, s);
  return K == 2 ? launch_rows1_k<2, esc::kTablePairsLayers, false>(a, (int)grid, s)
                : launch_rows1_k<3, kTablePairs3, false>(a, (int)grid, s);
}

esc::ProjOne rows1_proj(const void* x, const void* x2, const float* rin, const uint32_t* code,
                        const float* rout, const uint16_t* bias, int IC, int OC, char* part,
                        char* cnt, void* y) {
  esc::ProjOne q{};
  q.x = static_cast<const uint16_t*>(x);
  q.rin = rin;
  q.code = code;
  q.rout = rout;
  q.bias = bias;
  q.y = y;
  q.part = reinterpret_cast<float*>(part);
  q.cnt = reinterpret_cast<int*>(cnt);
  q.TK = IC / 16;
  q.TN = OC / 16;
  q.x2 = static_cast<const uint16_t*>(x2);
  return q;
}

// One linear of fewer than kLinearSmallRows rows (or, with x2, of the MLP
// activation of x and x2): one launch.
int linear_few(const void* x, const void* x2, int dt, const float* rin, const uint32_t* code,
               const float* rout, const uint16_t* bias, int M, int K, int IC, int OC, float rs,
               void* y, int ydt, const LinearPlan& lp, char* w, hipStream_t s) {
  if (rows1_single(M, IC, OC)) {
    // one row: the persistent kernel, its counters at off_cnt and its
    // partials at off_part (linear_plan sizes both)
    esc::ProjArgs a{};
    a.np = 1;
    a.rs = rs;
    a.dt = dt;
    a.ydt = ydt;
    a.pr[0] = rows1_proj(x, x2, rin, code, rout, bias, IC, OC, w + lp.off_part, w + lp.off_cnt, y);
    return launch_rows1(a, K, s);
  }
  // the split-K kernel, by hash
  const esc::LinearSmallArgs a = small_args(x, rin, code, rout, bias, M, IC / 16, OC / 16, lp, rs,
                                            w, y, dt, ydt, x2);
  if (x2) return K == 2 ? linear_small_launch<2, true>(a, s) : linear_small_launch<3, true>(a, s);
  return K == 2 ? linear_small_launch<2, false>(a, s) : linear_small_launch<3, false>(a, s);
}

template <typename LT>
int route_rows(const LT* logits, int T, int E, int top_k, int32_t* ids, float* scores,
               hipStream_t s) {
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(T), dim3(64), 0, s, logits, E, top_k, ids, scores);
  };
  if (E <= 256) go(esc::k_route_topk<4, LT>);
  else go(esc::k_route_topk<16, LT>);
  return launched("k_route_topk");
}

// k_combine, 8 columns per thread where the rows allow 16-byte accesses.
int combine_rows(const uint16_t* d16, const float* scores, int T, int top_k, int H, uint16_t* y,
                 hipStream_t s) {
  const bool wide = H % 8 == 0 && (reinterpret_cast<uintptr_t>(d16) |
                                   reinterpret_cast<uintptr_t>(y)) % 16 == 0;
  const int cols = wide ? 8 : 1;
  const dim3 grid((H / cols + 255) / 256, T);
  if (wide)
    hipLaunchKernelGGL(esc::k_combine<8>, grid, dim3(256), 0, s, d16, scores, top_k, H, y);
  else
    hipLaunchKernelGGL(esc::k_combine<1>, grid, dim3(256), 0, s, d16, scores, top_k, H, y);
  return launched("k_combine");
}

}  // namespace

extern "C" {

int esc_version(void) { return 100; }

const char* esc_last_error(void) { return g_err.c_str(); }

int esc_init(void) {
  if (int rc = ensure_lut()) return rc;
  if (int rc = ensure_wait_flag()) return rc;
  void* ptr = nullptr;
  return ensure_scratch(&ptr);
}

int esc_decode_tiles(const uint32_t* code, int K, int IC, int OC, int use_lut, uint16_t* w,
                     void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(code && w, "null pointer");
  if (use_lut)
    if (int rc = ensure_lut()) return rc;
  return by_k_lut<DecodeF>(K, use_lut, code, IC, OC, w, S(stream));
}

int esc_input_transform_typed(const void* rows, int dtype, const float* rin,
                              const int32_t* row_expert, int m, int IC, float rs, uint16_t* out,
                              void* stream) {
  ESC_REQUIRE(rows && rin && out, "null pointer");
  ESC_REQUIRE(IC > 0 && IC % 128 == 0, "Hadamard dimension must be divisible by 128, got %d", IC);
  ESC_REQUIRE(m >= 0, "negative row count");
  ESC_REQUIRE(dtype == ESC_ROWS_F16 || dtype == ESC_ROWS_BF16 || dtype == ESC_ROWS_F32,
              "row element type must be ESC_ROWS_F16, ESC_ROWS_BF16 or ESC_ROWS_F32, got %d",
              dtype);
  if (m == 0) return ESC_OK;
  by_rows_type(dtype, [&](auto dt) {
    oct_launch(m, IC, [&](auto r, dim3 grid, dim3 blk) {
      hipLaunchKernelGGL((esc::k_input_transform<decltype(dt)::value, decltype(r)::value>), grid,
                         blk, 0, S(stream), rows, rin, row_expert, m, IC, rs, out);
    });
  });
  return launched("k_input_transform");
}

int esc_input_transform(const uint16_t* rows, const float* rin, const int32_t* row_expert, int m,
                        int IC, float rs, uint16_t* out, void* stream) {
  return esc_input_transform_typed(rows, ESC_ROWS_F16, rin, row_expert, m, IC, rs, out, stream);
}

int esc_output_transform(const float* mid, const float* rout, const int32_t* row_expert,
                         const uint16_t* bias, int m, int OC, float rs, uint16_t* out,
                         void* stream) {
  ESC_REQUIRE(mid && rout && out, "null pointer");
  ESC_REQUIRE(OC > 0 && OC % 128 == 0, "Hadamard dimension must be divisible by 128, got %d", OC);
  ESC_REQUIRE(m >= 0, "negative row count");
  if (m == 0) return ESC_OK;
  const int ry = (m + esc::kTransformRows - 1) / esc::kTransformRows;
  if (row_expert)
    hipLaunchKernelGGL(esc::k_output_transform<true>, dim3(OC / 128, ry), dim3(256), 0, S(stream),
                       mid, rout, row_expert, bias, m, OC, rs, out);
  else
    hipLaunchKernelGGL(esc::k_output_transform<false>, dim3(OC / 128, ry), dim3(256), 0, S(stream),
                       mid, rout, row_expert, bias, m, OC, rs, out);
  return launched("k_output_transform");
}

int esc_gemv(const uint16_t* xh, const uint32_t* code, const int32_t* row_expert, int M, int K,
             int IC, int OC, int use_lut, float* mid, void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(xh && code && mid, "null pointer");
  ESC_REQUIRE(M >= 0, "negative row count");
  if (M == 0) return ESC_OK;
  if (use_lut)
    if (int rc = ensure_lut()) return rc;
  return exact_dispatch<esc::kPerRow>(K, use_lut, 1, xh, code, row_expert, nullptr, M, M,
                                      IC / 16, OC / 16, mid, S(stream));
}

size_t esc_gemv_fast_workspace(int M, int K, int IC, int OC) {
  if (check_proj(K, IC, OC) || M <= 0) return 0;
  return (size_t)fast_splits(K, M, IC / 16, OC / 16) * M * OC * sizeof(float);
}

int esc_gemv_fast_out(const uint16_t* xh, const uint32_t* code, const int32_t* row_expert,
                      const float* rout, int M, int K, int IC, int OC, int use_lut, float rs,
                      uint16_t* out, void* ws, size_t ws_bytes, void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(xh && code && rout && out, "null pointer");
  ESC_REQUIRE(M >= 0, "negative row count");
  if (M == 0) return ESC_OK;
  const int TK = IC / 16, TN = OC / 16;
  const int Sp = fast_splits(K, M, TK, TN);
  const size_t need = (size_t)Sp * M * OC * sizeof(float);
  if (!ws || ws_bytes < need)
    return fail(ESC_ENOSPACE, "workspace %zu bytes < required %zu", ws_bytes, need);
  if (use_lut)
    if (int rc = ensure_lut()) return rc;
  float* part = static_cast<float*>(ws);
  if (int rc = by_k_lut<FastF>(K, use_lut, xh, code, row_expert, M, TK, TN, Sp, part, S(stream)))
    return rc;
  hipLaunchKernelGGL(esc::k_splitk_out, dim3(OC / 128, M), dim3(64), 0, S(stream), part, Sp, M,
                     OC, rout, row_expert, rs, out);
  return launched("k_splitk_out");
}

size_t esc_linear_workspace(int M, int K, int IC, int OC) {
  if (check_proj(K, IC, OC) || M <= 0) return 0;
  return std::max(linear_plan(M, K, IC, OC, false).total, linear_plan(M, K, IC, OC, true).total);
}

int esc_linear(const uint16_t* x, const float* rin, const uint32_t* code, const float* rout,
               const uint16_t* bias, int M, int K, int IC, int OC, int use_lut, float rs,
               uint16_t* y, void* ws, size_t ws_bytes, void* stream) {
  return esc_linear_typed(x, ESC_ROWS_F16, rin, code, rout, bias, M, K, IC, OC, use_lut, rs, y, ws,
                          ws_bytes, stream);
}

int esc_linear_typed(const void* x, int dtype, const float* rin, const uint32_t* code,
                     const float* rout, const uint16_t* bias, int M, int K, int IC, int OC,
                     int use_lut, float rs, void* y, void* ws, size_t ws_bytes, void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(x && rin && code && rout && y, "null pointer");
  ESC_REQUIRE(M >= 0, "negative row count");
  if (int rc = check_rows_type(dtype, M)) return rc;
  if (M == 0) return ESC_OK;
  (void)use_lut;  // the decode is the kernel's own choice: both give the same weights
  const LinearPlan lp = linear_plan(M, K, IC, OC, rows1_single(M, IC, OC));
  const size_t need = M < kLinearSmallRows ? lp.total : lp.min_total;
  if (!ws || ws_bytes < need)
    return fail(ESC_ENOSPACE, "workspace %zu bytes < required %zu", ws_bytes, need);
  const int TK = IC / 16, TN = OC / 16;
  hipStream_t s = S(stream);
  char* w = static_cast<char*>(ws);
  if (M < kLinearSmallRows)
    return linear_few(x, nullptr, dtype, rin, code, rout, bias, M, K, IC, OC, rs, y, dtype, lp, w,
                      s);
  // many rows: input transform, then the matrix-core GEMM with the output
  // transform in its epilogue, or in its splits' reduction.  A workspace with
  // no room for the partials takes the one launch.
  uint16_t* xh = reinterpret_cast<uint16_t*>(w + lp.off_xh);
  if (int rc = esc_input_transform_typed(x, dtype, rin, nullptr, M, IC, rs, xh, stream)) return rc;
  const MmaPlan plan = ws_bytes < lp.total ? mma_plan(M, TK, TN, false) : lp.mma;
  const esc::MmaArgs a{xh, code, M, TK, TN, reinterpret_cast<float*>(w + lp.off_mid),
                       rout, bias, rs, y, dtype};
  return gemm_mma2_out(K, plan, a, s);
}

int esc_linear_act(const void* g, const void* u, int dtype, const float* rin,
                   const uint32_t* code, const float* rout, const uint16_t* bias, int M, int K,
                   int IC, int OC, float rs, void* y, int y_dtype, void* ws, size_t ws_bytes,
                   void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(g && u && rin && code && rout && y, "null pointer");
  ESC_REQUIRE(M >= 0 && M < kLinearSmallRows, "%d rows (fewer than %d)", M, kLinearSmallRows);
  if (M == 0) return ESC_OK;
  if (int rc = check_rows_type(dtype, M)) return rc;
  if (int rc = check_rows_type(y_dtype, M)) return rc;
  const LinearPlan lp = linear_plan(M, K, IC, OC, rows1_single(M, IC, OC));
  if (!ws || ws_bytes < lp.total)
    return fail(ESC_ENOSPACE, "workspace %zu bytes < required %zu", ws_bytes, lp.total);
  return linear_few(g, u, dtype, rin, code, rout, bias, M, K, IC, OC, rs, y, y_dtype, lp,
                    static_cast<char*>(ws), S(stream));
}

int esc_linear_xh(const uint16_t* xh, const uint32_t* code, const float* rout,
                  const uint16_t* bias, int M, int K, int IC, int OC, float rs, void* y,
                  int y_dtype, void* ws, size_t ws_bytes, void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(xh && code && rout && y, "null pointer");
  ESC_REQUIRE(M >= kLinearSmallRows || M == 0, "%d rows (%d or more)", M, kLinearSmallRows);
  if (int rc = check_rows_type(y_dtype, M)) return rc;
  if (M == 0) return ESC_OK;
  const int TK = IC / 16, TN = OC / 16;
  MmaPlan plan = mma_plan(M, TK, TN, true);
  if (plan.S > 1 && (!ws || ws_bytes < plan.part_bytes)) plan = mma_plan(M, TK, TN, false);
  const esc::MmaArgs a{xh, code, M, TK, TN, static_cast<float*>(ws), rout, bias, rs, y, y_dtype};
  return gemm_mma2_out(K, plan, a, S(stream));
}

int esc_act_transform(const void* g, const void* u, int dtype, const float* rin, int m, int I,
                      float rs, uint16_t* xh, void* stream) {
  ESC_REQUIRE(g && u && rin && xh, "null pointer");
  ESC_REQUIRE(I > 0 && I % 128 == 0, "Hadamard dimension must be divisible by 128, got %d", I);
  ESC_REQUIRE(m >= 0, "negative row count");
  ESC_REQUIRE(dtype == ESC_ROWS_F16 || dtype == ESC_ROWS_BF16 || dtype == ESC_ROWS_F32,
              "row element type must be ESC_ROWS_F16, ESC_ROWS_BF16 or ESC_ROWS_F32, got %d",
              dtype);
  if (m == 0) return ESC_OK;
  by_rows_type(dtype, [&](auto dt) {
    oct_launch(m, I, [&](auto r, dim3 grid, dim3 blk) {
      hipLaunchKernelGGL((esc::k_act_transform<decltype(dt)::value, decltype(r)::value>), grid, blk,
                         0, S(stream), g, u, rin, m, I, rs, xh);
    });
  });
  return launched("k_act_transform");
}

size_t esc_gemm_mfma_out_workspace(int M, int K, int IC, int OC) {
  if (check_proj(K, IC, OC) || M <= 0) return 0;
  return OC % 256 ? (size_t)M * OC * sizeof(float) : 0;
}

int esc_gemm_mfma_out(const uint16_t* xh, const uint32_t* code, const float* rout,
                      const uint16_t* bias, int M, int K, int IC, int OC, float rs, uint16_t* y,
                      void* ws, size_t ws_bytes, void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(xh && code && rout && y, "null pointer");
  ESC_REQUIRE(M >= 0, "negative row count");
  if (M == 0) return ESC_OK;
  const int TK = IC / 16, TN = OC / 16;
  hipStream_t s = S(stream);
  const size_t need = esc_gemm_mfma_out_workspace(M, K, IC, OC);
  if (need && (!ws || ws_bytes < need))
    return fail(ESC_ENOSPACE, "workspace %zu bytes < required %zu", ws_bytes, need);
  const esc::MmaArgs a{xh, code, M, TK, TN, nullptr, rout, bias, rs, y, ESC_ROWS_F16};
  return gemm_mma2_out(K, mma_plan(M, TK, TN, false), a, s);
}


size_t esc_linear_pair_workspace(int M, int K0, int K1, int IC, int OC0, int OC1) {
  const size_t a = esc_linear_workspace(M, K0, IC, OC0), b = esc_linear_workspace(M, K1, IC, OC1);
  if (!a || !b) return 0;
  return ((a + 255) & ~size_t(255)) + b;
}

int esc_linear_pair(const uint16_t* x, int M, int IC, const float* rin0, const uint32_t* code0,
                    const float* rout0, const uint16_t* bias0, int K0, int OC0, const float* rin1,
                    const uint32_t* code1, const float* rout1, const uint16_t* bias1, int K1,
                    int OC1, int use_lut, float rs, uint16_t* y0, uint16_t* y1, void* ws,
                    size_t ws_bytes, void* stream) {
  return esc_linear_pair_typed(x, ESC_ROWS_F16, M, IC, rin0, code0, rout0, bias0, K0, OC0, rin1,
                               code1, rout1, bias1, K1, OC1, use_lut, rs, y0, y1, ws, ws_bytes,
                               stream);
}

int esc_linear_pair_typed(const void* x, int dtype, int M, int IC, const float* rin0,
                          const uint32_t* code0, const float* rout0, const uint16_t* bias0, int K0,
                          int OC0, const float* rin1, const uint32_t* code1, const float* rout1,
                          const uint16_t* bias1, int K1, int OC1, int use_lut, float rs, void* y0v,
                          void* y1v, void* ws, size_t ws_bytes, void* stream) {
  if (int rc = check_proj(K0, IC, OC0)) return rc;
  if (int rc = check_proj(K1, IC, OC1)) return rc;
  ESC_REQUIRE(x && rin0 && code0 && rout0 && y0v && rin1 && code1 && rout1 && y1v, "null pointer");
  ESC_REQUIRE(M >= 0, "negative row count");
  if (int rc = check_rows_type(dtype, M)) return rc;
  if (M == 0) return ESC_OK;
  const size_t need = esc_linear_pair_workspace(M, K0, K1, IC, OC0, OC1);
  if (!ws || ws_bytes < need)
    return fail(ESC_ENOSPACE, "workspace %zu bytes < required %zu", ws_bytes, need);
  // projection 1's workspace follows projection 0's (each as esc_linear's)
  const size_t ws0 = esc_linear_workspace(M, K0, IC, OC0);
  const size_t off1 = (ws0 + 255) & ~size_t(255);
  char* w = static_cast<char*>(ws);
  if (M >= kLinearSmallRows) {
    const int TK = IC / 16;
    const LinearPlan p0 = linear_plan(M, K0, IC, OC0, false);
    const LinearPlan p1 = linear_plan(M, K1, IC, OC1, false);
    if (K0 != K1 || p0.mma.S != p1.mma.S) {
      if (int rc = esc_linear_typed(x, dtype, rin0, code0, rout0, bias0, M, K0, IC, OC0, use_lut,
                                    rs, y0v, w, ws0, stream))
        return rc;
      return esc_linear_typed(x, dtype, rin1, code1, rout1, bias1, M, K1, IC, OC1, use_lut, rs,
                              y1v, w + off1, ws_bytes - off1, stream);
    }
    // both transforms in one pass over x, both products in one launch, with the
    // splits of their own calls (the row blocks do not change a sum's order)
    hipStream_t s = S(stream);
    const int Sp = p0.mma.S;
    char* w1 = w + off1;
    uint16_t* xh0 = reinterpret_cast<uint16_t*>(w + p0.off_xh);
    uint16_t* xh1 = reinterpret_cast<uint16_t*>(w1 + p1.off_xh);
    by_rows_type(dtype, [&](auto dt) {
      oct_launch(M, IC, [&](auto r, dim3 grid, dim3 blk) {
        hipLaunchKernelGGL((esc::k_input_transform<decltype(dt)::value, decltype(r)::value, true>),
                           grid, blk, 0, s, x, rin0, nullptr, M, IC, rs, xh0, rin1, xh1);
      });
    });
    if (int rc = launched("k_input_transform")) return rc;
    const esc::MmaArgs a0{xh0, code0, M, TK, OC0 / 16, reinterpret_cast<float*>(w + p0.off_mid),
                          rout0, bias0, rs, y0v, dtype};
    const esc::MmaArgs a1{xh1, code1, M, TK, OC1 / 16, reinterpret_cast<float*>(w1 + p1.off_mid),
                          rout1, bias1, rs, y1v, dtype};
    const int nrb = mma_plan(M, TK, OC0 / 16, true, Sp, (OC1 + 255) / 256).nrb;
    if (Sp == 1) return gemm_mma2_launch<esc::kMmaOut>(K0, nrb, 1, a0, s, &a1);
    if (int rc = gemm_mma2_launch<esc::kMmaPart>(K0, nrb, Sp, a0, s, &a1)) return rc;
    if (int rc = mma2_reduce(K0, Sp, a0, s)) return rc;
    return mma2_reduce(K0, Sp, a1, s);
  }
  const bool r0 = rows1_single(M, IC, OC0), r1 = rows1_single(M, IC, OC1);
  const int TK = IC / 16;
  const LinearPlan p0 = linear_plan(M, K0, IC, OC0, r0);
  const LinearPlan p1 = linear_plan(M, K1, IC, OC1, r1);
  char* w1 = w + off1;
  if (r0 && r1 && K0 == K1) {
    // one row: both projections in one persistent launch, each with its own
    // plan and workspace, so each output is its own esc_linear call's
    esc::ProjArgs a{};
    a.np = 2;
    a.rs = rs;
    a.dt = a.ydt = dtype;
    a.pr[0] = rows1_proj(x, nullptr, rin0, code0, rout0, bias0, IC, OC0, w + p0.off_part,
                         w + p0.off_cnt, y0v);
    a.pr[1] = rows1_proj(x, nullptr, rin1, code1, rout1, bias1, IC, OC1, w1 + p1.off_part,
                         w1 + p1.off_cnt, y1v);
    return launch_rows1(a, K0, S(stream));
  }
  if (r0 || r1 || p0.R != p1.R) {
    // one row with the projections on different kernels (or K), or row
    // groups of different sizes: each as its own call
    if (int rc = esc_linear_typed(x, dtype, rin0, code0, rout0, bias0, M, K0, IC, OC0, use_lut, rs,
                                  y0v, w, ws0, stream))
      return rc;
    return esc_linear_typed(x, dtype, rin1, code1, rout1, bias1, M, K1, IC, OC1, use_lut, rs, y1v,
                            w1, ws_bytes - off1, stream);
  }
  const esc::LinearSmallArgs a0 = small_args(x, rin0, code0, rout0, bias0, M, TK, OC0 / 16, p0, rs,
                                             w, y0v, dtype, dtype);
  const esc::LinearSmallArgs a1 = small_args(x, rin1, code1, rout1, bias1, M, TK, OC1 / 16, p1, rs,
                                             w1, y1v, dtype, dtype);
  // the split-K pair kernel, by hash
  return linear_pair_k(K0, K1, a0, a1, S(stream));
}

size_t esc_linear_multi_workspace(int M, int n, int K, int IC, const int* OC) {
  if (M <= 0 || n < 1 || n > esc::kProjMax || !OC) return 0;
  size_t total = 0;
  for (int i = 0; i < n; ++i) {
    if (check_proj(K, IC, OC[i])) return 0;
    if (M == 1) {
      if (OC[i] % 256) return 0;
      // this projection's counters, then its partials
      total += ((size_t)(OC[i] / 256) * 4 + 255) / 256 * 256 + rows1_part_bytes(IC / 16, OC[i] / 16);
    } else {
      // this projection's esc_linear workspace
      total += (esc_linear_workspace(M, K, IC, OC[i]) + 255) & ~size_t(255);
    }
  }
  return total;
}

int esc_linear_multi(const uint16_t* x, int M, int IC, int K, int n, const uint32_t* const* code,
                     const float* const* rin, const float* const* rout,
                     const uint16_t* const* bias, const int* OC, int use_lut, float rs,
                     uint16_t* const* y, void* ws, size_t ws_bytes, void* stream) {
  ESC_REQUIRE(y, "null pointer");
  ESC_REQUIRE(n >= 1 && n <= esc::kProjMax, "%d projections (1 to %d)", n, esc::kProjMax);
  void* yv[esc::kProjMax];
  for (int i = 0; i < n; ++i) yv[i] = y[i];
  return esc_linear_multi_typed(x, ESC_ROWS_F16, M, IC, K, n, code, rin, rout, bias, OC, use_lut,
                                rs, yv, ws, ws_bytes, stream);
}

int esc_linear_multi_typed(const void* x, int dtype, int M, int IC, int K, int n,
                           const uint32_t* const* code, const float* const* rin,
                           const float* const* rout, const uint16_t* const* bias, const int* OC,
                           int use_lut, float rs, void* const* y, void* ws, size_t ws_bytes,
                           void* stream) {
  ESC_REQUIRE(x && code && rin && rout && OC && y, "null pointer");
  ESC_REQUIRE(M >= 0, "negative row count");
  ESC_REQUIRE(n >= 1 && n <= esc::kProjMax, "%d projections (1 to %d)", n, esc::kProjMax);
  static_assert(esc::kLinearMultiMax == esc::kProjMax, "projections per launch");
  for (int i = 0; i < n; ++i) {
    if (int rc = check_proj(K, IC, OC[i])) return rc;
    ESC_REQUIRE(code[i] && rin[i] && rout[i] && y[i], "null pointer (projection %d)", i);
    ESC_REQUIRE(M != 1 || OC[i] % 256 == 0, "OC=%d of projection %d is not a multiple of 256",
                OC[i], i);
  }
  if (int rc = check_rows_type(dtype, M)) return rc;
  if (M == 0) return ESC_OK;
  const size_t need = esc_linear_multi_workspace(M, n, K, IC, OC);
  if (!ws || ws_bytes < need)
    return fail(ESC_ENOSPACE, "workspace %zu bytes < required %zu", ws_bytes, need);
  char* w = static_cast<char*>(ws);
  if (M == 1) {
    // one row: one persistent k_proj_rows1 launch, the units of all
    // projections split over its waves
    esc::ProjArgs a{};
    a.np = n;
    a.rs = rs;
    a.dt = a.ydt = dtype;
    for (int i = 0; i < n; ++i) {
      char* cnt = w;
      w += ((size_t)(OC[i] / 256) * 4 + 255) / 256 * 256;
      a.pr[i] = rows1_proj(x, nullptr, rin[i], code[i], rout[i], bias ? bias[i] : nullptr, IC,
                           OC[i], w, cnt, y[i]);
      w += rows1_part_bytes(IC / 16, OC[i] / 16);
    }
    return launch_rows1(a, K, S(stream), true);
  }
  // several rows: each projection's esc_linear plan and workspace, as one
  // k_linear_multi launch when all run the split-K kernel with one row group
  // size, else one call each
  size_t off[esc::kProjMax];
  LinearPlan pl[esc::kProjMax];
  bool one = M < kLinearSmallRows;
  size_t o = 0;
  for (int i = 0; i < n; ++i) {
    off[i] = o;
    o += (esc_linear_workspace(M, K, IC, OC[i]) + 255) & ~size_t(255);
    pl[i] = linear_plan(M, K, IC, OC[i], false);
    one = one && pl[i].R == pl[0].R;
  }
  if (!one) {
    for (int i = 0; i < n; ++i)
      if (int rc = esc_linear_typed(x, dtype, rin[i], code[i], rout[i], bias ? bias[i] : nullptr,
                                    M, K, IC, OC[i], use_lut, rs, y[i], w + off[i],
                                    ws_bytes - off[i], stream))
        return rc;
    return ESC_OK;
  }
  esc::LinearMultiArgs m{};
  m.n = n;
  long nw = 0;
  for (int i = 0; i < n; ++i) {
    m.p[i] = small_args(x, rin[i], code[i], rout[i], bias ? bias[i] : nullptr, M, IC / 16,
                        OC[i] / 16, pl[i], rs, w + off[i], y[i], dtype, dtype);
    nw += (long)pl[i].groups * pl[i].row_groups * pl[i].S;
  }
  ESC_REQUIRE(pl[0].R >= 2 && pl[0].R <= kLinearSmallRows, "rows per group %d", pl[0].R);
  if (K == 2)
    hipLaunchKernelGGL((esc::k_linear_multi<2, kLinearSmallRows>), dim3(nw), dim3(256), 0, S(stream), m);
  else
    hipLaunchKernelGGL((esc::k_linear_multi<3, kLinearSmallRows>), dim3(nw), dim3(256), 0, S(stream), m);
  return launched("k_linear_multi");
}

size_t esc_gemm_rows_fast_workspace(int M, int R, int K, int IC, int OC) {
  if (check_proj(K, IC, OC) || M <= 0 || R <= 0) return 0;
  return (size_t)fast_splits(K, (M + R - 1) / R, IC / 16, OC / 16) * M * OC * sizeof(float);
}

int esc_gemm_rows_fast_out(const uint16_t* xh, const uint32_t* code, const float* rout, int M,
                           int R, int K, int IC, int OC, int use_lut, float rs, uint16_t* out,
                           void* ws, size_t ws_bytes, void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(xh && code && rout && out, "null pointer");
  ESC_REQUIRE(M >= 0, "negative row count");
  ESC_REQUIRE(R == 2 || R == 4 || R == 8, "rows per block R=%d not in {2,4,8}", R);
  if (M == 0) return ESC_OK;
  const int TK = IC / 16, TN = OC / 16;
  const int Sp = fast_splits(K, (M + R - 1) / R, TK, TN);
  const size_t need = (size_t)Sp * M * OC * sizeof(float);
  if (!ws || ws_bytes < need)
    return fail(ESC_ENOSPACE, "workspace %zu bytes < required %zu", ws_bytes, need);
  if (use_lut)
    if (int rc = ensure_lut()) return rc;
  float* part = static_cast<float*>(ws);
  hipStream_t s = S(stream);
  int rc;
  if (K == 2)
    rc = use_lut ? FastRowsF<2, true>::run(R, xh, code, M, TK, TN, Sp, part, s)
                 : FastRowsF<2, false>::run(R, xh, code, M, TK, TN, Sp, part, s);
  else
    rc = use_lut ? FastRowsF<3, true>::run(R, xh, code, M, TK, TN, Sp, part, s)
                 : FastRowsF<3, false>::run(R, xh, code, M, TK, TN, Sp, part, s);
  if (rc) return rc;
  hipLaunchKernelGGL(esc::k_splitk_out, dim3(OC / 128, M), dim3(64), 0, s, part, Sp, M, OC, rout,
                     nullptr, rs, out);
  return launched("k_splitk_out");
}

int esc_gemm_rows(const uint16_t* xh, const uint32_t* code, const int32_t* rows_idx,
                  const int32_t* group_expert, int n_groups, int R, int n_rows, int K, int IC,
                  int OC, int use_lut, float* mid, void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(xh && code && rows_idx && group_expert && mid, "null pointer");
  ESC_REQUIRE(n_groups >= 0 && n_rows >= 0, "negative size");
  if (n_groups == 0) return ESC_OK;
  if (use_lut)
    if (int rc = ensure_lut()) return rc;
  return exact_dispatch<esc::kMoeGroups>(K, use_lut, R, xh, code, rows_idx, group_expert, n_rows,
                                         n_groups, IC / 16, OC / 16, mid, S(stream));
}

int esc_dense_gemm_rows(const uint16_t* xh, const uint32_t* code, int M, int R, int K, int IC,
                        int OC, int use_lut, float* mid, void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(xh && code && mid, "null pointer");
  ESC_REQUIRE(M >= 0, "negative row count");
  ESC_REQUIRE(R == 1 || R == 2 || R == 4 || R == 8 || R == 16, "dense R=%d not in {1,2,4,8,16}", R);
  if (M == 0) return ESC_OK;
  if (use_lut)
    if (int rc = ensure_lut()) return rc;
  return exact_dispatch<esc::kDenseRows>(K, use_lut, R, xh, code, nullptr, nullptr, M,
                                         (M + R - 1) / R, IC / 16, OC / 16, mid, S(stream));
}

int esc_dense_gemm_rows_out(const uint16_t* xh, const uint32_t* code, const float* rout, int M,
                            int R, int K, int IC, int OC, int use_lut, float rs, uint16_t* out,
                            void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(xh && code && rout && out, "null pointer");
  ESC_REQUIRE(M >= 0, "negative row count");
  if (M == 0) return ESC_OK;
  if (use_lut)
    if (int rc = ensure_lut()) return rc;
  const int TK = IC / 16, TN = OC / 16;
  hipStream_t s = S(stream);
  if (K == 2)
    return use_lut ? ExactOutF<2, true>::run(R, xh, code, rout, M, TK, TN, rs, out, s)
                   : ExactOutF<2, false>::run(R, xh, code, rout, M, TK, TN, rs, out, s);
  return use_lut ? ExactOutF<3, true>::run(R, xh, code, rout, M, TK, TN, rs, out, s)
                 : ExactOutF<3, false>::run(R, xh, code, rout, M, TK, TN, rs, out, s);
}

int esc_gemm_mfma(const uint16_t* xh, const uint32_t* code, int M, int K, int IC, int OC,
                  int use_lut, float* mid, void* stream) {
  if (int rc = check_proj(K, IC, OC)) return rc;
  ESC_REQUIRE(xh && code && mid, "null pointer");
  ESC_REQUIRE(M >= 0, "negative row count");
  (void)use_lut;  // the table holds the hash's own values: both decodes give the same bits
  if (M == 0) return ESC_OK;
  const int TK = IC / 16, TN = OC / 16;
  hipStream_t s = S(stream);
  const esc::MmaArgs a{xh, code, M, TK, TN, mid, nullptr, nullptr, 0.f, nullptr, ESC_ROWS_F16};
  return gemm_mma2_launch<esc::kMmaMid>(K, mma_plan(M, TK, TN, false).nrb, 1, a, s);
}

int esc_build_groups(const int32_t* row_expert, int m, int E, int R, int n_groups,
                     int32_t* rows_idx, int32_t* group_expert, void* stream) {
  ESC_REQUIRE(row_expert && rows_idx && group_expert, "null pointer");
  ESC_REQUIRE(E > 0 && E <= 4096, "expert count %d not in [1, 4096]", E);
  ESC_REQUIRE(R >= 1 && m >= 0, "bad R=%d / m=%d", R, m);
  const long bound = ((long)m + (long)E * (R - 1) + R - 1) / R;
  ESC_REQUIRE(n_groups >= bound, "n_groups %d below the bound %ld", n_groups, bound);
  hipLaunchKernelGGL(esc::k_build_groups, dim3(1), dim3(1024), 0, S(stream), row_expert, m, E, R,
                     n_groups, rows_idx, group_expert);
  return launched("k_build_groups");
}

int esc_route_topk(const float* logits, int T, int E, int top_k, int32_t* ids, float* scores,
                   void* stream) {
  ESC_REQUIRE(logits && ids && scores, "null pointer");
  ESC_REQUIRE(E > 0 && E <= 1024, "expert count %d not in [1, 1024]", E);
  ESC_REQUIRE(top_k >= 1 && top_k <= 32 && top_k <= E, "top_k %d not in [1, min(32, E)]", top_k);
  ESC_REQUIRE(T >= 0, "negative token count");
  if (T == 0) return ESC_OK;
  return route_rows(logits, T, E, top_k, ids, scores, S(stream));
}

int esc_swiglu(const uint16_t* gu, int m, int I, uint16_t* h, void* stream) {
  ESC_REQUIRE(gu && h, "null pointer");
  ESC_REQUIRE(m >= 0 && I > 0, "bad m=%d / I=%d", m, I);
  if (m == 0) return ESC_OK;
  hipLaunchKernelGGL(esc::k_swiglu, dim3((I + 255) / 256, m), dim3(256), 0, S(stream), gu, I, h);
  return launched("k_swiglu");
}

int esc_moe_combine(const uint16_t* d16, const float* scores, int T, int top_k, int H,
                    uint16_t* y, void* stream) {
  ESC_REQUIRE(d16 && scores && y, "null pointer");
  ESC_REQUIRE(T >= 0 && top_k >= 1 && H > 0, "bad T=%d / top_k=%d / H=%d", T, top_k, H);
  if (T == 0) return ESC_OK;
  return combine_rows(d16, scores, T, top_k, H, y, S(stream));
}

// ---- dense int8 / f16 GEMV (q8.hpp): shared expert, gates, vocabulary head

}  // extern "C"

namespace {
// k_rows_gemv geometry: LPR lanes per output row (the row's 16-byte chunk
// count rounded up to a power of two, 8..64), CPL chunks per lane (1..8).
// The lanes keep NR rows of x in registers, NR * CPL * XW words (XW = 8 f16
// pairs per int8 chunk, 4 per f16 chunk): rows per launch are capped at 128
// such words.
constexpr int kRowsXWords = 128;
constexpr int kRowsMaxCpl = 8;

struct RowsGeo {
  int lpr, cpl;
};
RowsGeo rows_geo(int chunks) {
  int lpr = 8;
  while (lpr < chunks && lpr < 64) lpr *= 2;
  return {lpr, (chunks + lpr - 1) / lpr};
}
constexpr int rows_x_words(bool q8) { return q8 ? 8 : 4; }
int rows_nr_max(bool q8, int cpl) {
  int nr = 8;
  while (nr > 1 && nr * cpl * rows_x_words(q8) > kRowsXWords) nr /= 2;
  return nr;
}

template <bool Q8, int NR, int LPR, int CPL>
int rows_launch(const uint16_t* x, const void* w, const float* scale, int M, int K, int O,
                uint16_t* y, hipStream_t s) {
  if constexpr (NR * CPL * rows_x_words(Q8) > kRowsXWords) {
    return fail(ESC_EINVAL, "internal: %d rows x %d chunks exceed the register budget", NR, CPL);
  } else {
    const long steps = ((long)O + 64 / LPR - 1) / (64 / LPR);
    // eight workgroups per CU, each wave striding over the row steps (measured
    // on MI355X with the 248320 x 2048 head: 103 us at 8 per CU, 107 us at 4,
    // 16 no better than 8)
    const int blocks = (int)std::min<long>((steps + 3) / 4, 8L * device_cus());
    hipLaunchKernelGGL((esc::k_rows_gemv<Q8, NR, LPR, CPL>), dim3(blocks), dim3(256), 0, s, x, w,
                       scale, M, K, O, y, O);
    return launched("k_rows_gemv");
  }
}

template <bool Q8, int NR>
int rows_by_geo(RowsGeo g, const uint16_t* x, const void* w, const float* scale, int M, int K,
                int O, uint16_t* y, hipStream_t s) {
  switch (g.lpr) {
    case 8: return rows_launch<Q8, NR, 8, 1>(x, w, scale, M, K, O, y, s);
    case 16: return rows_launch<Q8, NR, 16, 1>(x, w, scale, M, K, O, y, s);
    case 32: return rows_launch<Q8, NR, 32, 1>(x, w, scale, M, K, O, y, s);
  }
  switch (g.cpl) {
    case 1: return rows_launch<Q8, NR, 64, 1>(x, w, scale, M, K, O, y, s);
    case 2: return rows_launch<Q8, NR, 64, 2>(x, w, scale, M, K, O, y, s);
    case 3: return rows_launch<Q8, NR, 64, 3>(x, w, scale, M, K, O, y, s);
    case 4: return rows_launch<Q8, NR, 64, 4>(x, w, scale, M, K, O, y, s);
    case 5: return rows_launch<Q8, NR, 64, 5>(x, w, scale, M, K, O, y, s);
    case 6: return rows_launch<Q8, NR, 64, 6>(x, w, scale, M, K, O, y, s);
    case 7: return rows_launch<Q8, NR, 64, 7>(x, w, scale, M, K, O, y, s);
    default: return rows_launch<Q8, NR, 64, 8>(x, w, scale, M, K, O, y, s);
  }
}

// int8 weights and 2..16 rows per launch: k_rows_w8_mma, the rows' products on
// the matrix core (x staged in LDS, at most kW8MmaLds bytes per workgroup)
constexpr int kW8MmaLds = 64 * 1024;
int w8_mma_rows(int M, int K) {
  if (M < 2 || K % 64) return 0;
  return std::min(16, kW8MmaLds / (2 * K + 16));
}

int rows_w8_mma(const uint16_t* x, const void* w, const float* scale, int M, int K, int O,
                uint16_t* y, int nr, hipStream_t s) {
  const int groups = (O + 15) / 16;
  for (int m0 = 0; m0 < M; m0 += nr) {
    const int mr = std::min(nr, M - m0);
    const size_t lds = (size_t)mr * (2 * K + 16);
    const int per_cu = (int)std::max<size_t>(1, std::min<size_t>(8, 160 * 1024 / lds));
    const int blocks = std::min((groups + 3) / 4, per_cu * device_cus());
    hipLaunchKernelGGL(esc::k_rows_w8_mma, dim3(blocks), dim3(256), lds, s, x + (size_t)m0 * K,
                       static_cast<const int8_t*>(w), scale, mr, K, O, y + (size_t)m0 * O, O);
    if (int rc = launched("k_rows_w8_mma")) return rc;
  }
  return ESC_OK;
}

// Whether the matrix-core GEMMs take a shape (K a multiple of 64).  f16 weights:
// from 9 rows, where the GEMV needs a second launch.  int8: where k_rows_w8_mma
// needs a second launch (its rows of x fill a workgroup's LDS), and below that for
// long rows of few channels, which leave its workgroups (16 channels a wave, all of
// K) latency-bound: whole call, K = 5120 to 5120 / 16384 channels, 2 rows 21 / 23 us
// against 16 / 20, 8 rows 44 / 47 against 17 / 21; not for K <= 2048 (4096 channels
// level, 248320 channels 104 us against 135).
bool rows_gemm_takes(bool q8, int M, int K, int O) {
  if (K % 64) return false;
  if (!q8) return M > 8;
  return M >= 2 && (M > w8_mma_rows(M, K) || (K >= 4096 && O <= 32768));
}

// The time of a launch is that of the busiest CU: n workgroups on it take t0 + t1 n
// us per step (fitted to a sweep of 7 kernels over 33 shapes, int8, on MI355X).
// K = 2048, whole call: 203 x 512 14.1 us (16 rows per launch: 153), 1000 x 4096 35
// (852), 2048 x 4096 59 (1743), 64 x 248320 144 (570).
template <bool Q8>
int rows_gemm(const uint16_t* x, const void* w, const float* scale, int M, int K, int O,
              uint16_t* y, hipStream_t s) {
  const int cus = device_cus(), NS = K / 64;
  struct Kern {
    void (*fn)(const uint16_t*, const void*, const float*, int, int, int, uint16_t*);
    int rows, cols, steps;
    double t0, t1;
  };
  // k_rows_gemm's four waves share the steps
  const Kern kerns[] = {{esc::k_rows_gemm<Q8, 2>, 32, 64, (NS + 3) / 4, 0.0, 1.05},
                        {esc::k_rows_gemm<Q8, 4>, 64, 64, (NS + 3) / 4, 0.0, 1.5},
                        {esc::k_rows_gemm_lds<Q8, 4>, 64, 256, NS, 0.4, 0.75},
                        {esc::k_rows_gemm_lds<Q8, 6>, 96, 256, NS, 0.6, 0.8},
                        {esc::k_rows_gemm_lds<Q8, 8>, 128, 256, NS, 0.8, 1.0}};
  const Kern* best = nullptr;
  double best_cost = 0.0;
  long best_blocks = 0;
  for (const Kern& k : kerns) {
    const long blocks = (long)((O + k.cols - 1) / k.cols) * ((M + k.rows - 1) / k.rows);
    const double cost = (k.t0 + k.t1 * ((blocks + cus - 1) / cus)) * k.steps;
    if (!best || cost < best_cost) best = &k, best_cost = cost, best_blocks = blocks;
  }
  ESC_REQUIRE(best_blocks < (1L << 31), "%d rows x %d channels is too large", M, O);
  hipLaunchKernelGGL(best->fn, dim3((unsigned)best_blocks), dim3(256), 0, s, x, w, scale, M, K, O,
                     y);
  return launched("k_rows_gemm");
}

template <bool Q8>
int rows_gemv(const uint16_t* x, const void* w, const float* scale, int M, int K, int O,
              uint16_t* y, hipStream_t s) {
  const int cw = Q8 ? 16 : 8;  // weights per 16-byte chunk
  const int chunks = K / cw;
  ESC_REQUIRE(K > 0 && K % cw == 0 && chunks >= 8 && chunks <= 64 * kRowsMaxCpl,
              "K=%d: need a multiple of %d in [%d, %d]", K, cw, 8 * cw, 64 * kRowsMaxCpl * cw);
  if (rows_gemm_takes(Q8, M, K, O))
    return rows_gemm<Q8>(x, w, scale, M, K, O, y, s);
  if constexpr (Q8) {
    if (const int nr = w8_mma_rows(M, K); nr >= 2) return rows_w8_mma(x, w, scale, M, K, O, y, nr, s);
  }
  const RowsGeo g = rows_geo(chunks);
  const int nr_max = rows_nr_max(Q8, g.cpl);
  for (int m0 = 0; m0 < M; m0 += nr_max) {
    const int mr = std::min(nr_max, M - m0);
    const uint16_t* xm = x + (size_t)m0 * K;
    uint16_t* ym = y + (size_t)m0 * O;
    int rc;
    if (mr == 1) rc = rows_by_geo<Q8, 1>(g, xm, w, scale, mr, K, O, ym, s);
    else if (mr == 2) rc = rows_by_geo<Q8, 2>(g, xm, w, scale, mr, K, O, ym, s);
    else if (mr <= 4) rc = rows_by_geo<Q8, 4>(g, xm, w, scale, mr, K, O, ym, s);
    else rc = rows_by_geo<Q8, 8>(g, xm, w, scale, mr, K, O, ym, s);
    if (rc) return rc;
  }
  return ESC_OK;
}

// Projections of the same rows: one k_rows_gemm_multi launch (32 rows a
// workgroup: a router and a shared expert are narrow) where all are narrow enough
// to share the chip, else each as its own call.
int rows_multi(int n, const uint16_t* x, const void* const* w, const float* const* scale,
               uint16_t* const* y, const int* O, int M, int K, hipStream_t s) {
  long blocks = 0;
  esc::RowsMulti a{};
  a.n = n;
  for (int i = 0; i < n; ++i) {
    a.w[i] = w[i], a.scale[i] = scale[i], a.y[i] = y[i], a.O[i] = O[i];
    a.blk0[i] = (int)blocks;
    blocks += (long)((O[i] + 63) / 64) * ((M + 31) / 32);
  }
  // (K: what the f16 GEMV of a few rows takes too)
  if (K % 64 == 0 && K <= 4096 && blocks <= 4L * device_cus()) {
    hipLaunchKernelGGL(esc::k_rows_gemm_multi<2>, dim3((unsigned)blocks), dim3(256), 0, s, x, a, M, K);
    return launched("k_rows_gemm_multi");
  }
  for (int i = 0; i < n; ++i) {
    const int rc = scale[i] ? rows_gemv<true>(x, w[i], scale[i], M, K, O[i], y[i], s)
                            : rows_gemv<false>(x, w[i], nullptr, M, K, O[i], y[i], s);
    if (rc) return rc;
  }
  return ESC_OK;
}
}  // namespace

extern "C" {

int esc_w8a16(const uint16_t* x, const int8_t* w8, const float* scale, int M, int K, int O,
              uint16_t* y, void* stream) {
  ESC_REQUIRE(x && w8 && scale && y, "null pointer");
  ESC_REQUIRE(M >= 0 && O > 0, "bad M=%d / O=%d", M, O);
  if (M == 0) return ESC_OK;
  return rows_gemv<true>(x, w8, scale, M, K, O, y, S(stream));
}

int esc_gemv_f16w(const uint16_t* x, const uint16_t* w, int M, int K, int O, uint16_t* y,
                  void* stream) {
  ESC_REQUIRE(x && w && y, "null pointer");
  ESC_REQUIRE(M >= 0 && O > 0, "bad M=%d / O=%d", M, O);
  if (M == 0) return ESC_OK;
  return rows_gemv<false>(x, w, nullptr, M, K, O, y, S(stream));
}

int esc_moe_shared_act(const uint16_t* g, const uint16_t* u, int m, int I, uint16_t* hh,
                       void* stream) {
  ESC_REQUIRE(g && u && hh, "null pointer");
  ESC_REQUIRE(m >= 0 && I > 0, "bad m=%d / I=%d", m, I);
  if (m == 0) return ESC_OK;
  hipLaunchKernelGGL(esc::k_shared_act, dim3((I + 255) / 256, m), dim3(256), 0, S(stream), g, u,
                     I, hh);
  return launched("k_shared_act");
}

int esc_moe_block_out(const uint16_t* y, const uint16_t* sh, const uint16_t* shg, int m, int H,
                      uint16_t* out, void* stream) {
  ESC_REQUIRE(y && sh && shg && out, "null pointer");
  ESC_REQUIRE(m >= 0 && H > 0, "bad m=%d / H=%d", m, H);
  if (m == 0) return ESC_OK;
  hipLaunchKernelGGL(esc::k_block_out, dim3((H + 255) / 256, m), dim3(256), 0, S(stream), y, sh,
                     shg, H, static_cast<void*>(out), ESC_ROWS_F16);
  return launched("k_block_out");
}

int esc_q8_embed(const int32_t* ids, int T, const int8_t* w8, const float* scale, int N, int K,
                 uint16_t* out, void* stream) {
  ESC_REQUIRE(ids && w8 && scale && out, "null pointer");
  ESC_REQUIRE(T >= 0 && N > 0 && K > 0 && K % 16 == 0, "bad T=%d / N=%d / K=%d (K a multiple of 16)",
              T, N, K);
  if (T == 0) return ESC_OK;
  hipLaunchKernelGGL(esc::k_q8_embed, dim3(T), dim3(256), 0, S(stream), ids, w8, scale, N, K, out);
  return launched("k_q8_embed");
}

}  // extern "C"

// ---- routed experts: input transform -> gate_up -> swiglu/transform -> down -> combine
namespace {
// Rows per expert group of the split-K chain: once there are as many routed
// rows as experts, rows of one expert share each decoded weight (groups laid
// out by moe.build_groups, one row per B column of the matrix-core multiply,
// so a group costs one decode whatever its row count, up to 16); below that
// almost every expert has one row.  16 rows per group from four rows per expert
// (measured on MI355X, 256 experts, hidden 2048, intermediate 512, top-8, whole
// call, 8 against 16 rows: 48 tokens 112 / 115 us, 128 145 / 140, 200 167 / 150).
int moe_group_rows(int M, int E) { return M >= 4L * E ? 16 : M >= E ? 8 : 0; }

// Whether the grouped chain decodes with the table (k_gemv_rows_table, which
// stages 128 KiB per CU) or by hash, whichever decode was asked for: the weights
// are the same, and the table wins from about 2^28 weights to decode (measured
// as above, hash against table: 256 experts 48 tokens 128 / 115 us, 200 tokens 164
// / 150; 64 experts, 201 M weights, 66 / 73; 64 experts of 1024 x 256 42 / 46).
bool moe_rows_table(int groups, int H, int I) { return (double)groups * 3 * H * I >= (1 << 28); }

int moe_input(const void* x, int dtype, const int32_t* ids, int top_k, const float* rin, int H,
              float rs, uint16_t* xh, int M, hipStream_t s) {
  by_rows_type(dtype, [&](auto dt) {
    hipLaunchKernelGGL(esc::k_moe_input<decltype(dt)::value>, dim3(H / 128, M), dim3(64), 0, s, x,
                       ids, top_k, rin, H, rs, xh);
  });
  return launched("k_moe_input");
}

// Row blocks of 16 per group of the grouped matrix-core GEMM (k_moe_mma), 0:
// the split-K chain.  Measured on MI355X (256 experts, hidden 2048, intermediate
// 512, top-8; whole call, the split-K chain in brackets): 6 rows per expert 175 us
// (150), 9 rows 175 (164), 12 rows 173 (187), 16 rows 171 (218), 64 rows 284 (1200
// in groups of 8); 64 experts, 8 rows 78 (80 by hash), 12 rows 79 (99), 4 rows 78
// (66).  So from 8 rows per expert, or 11 where the experts' weights fill the chip
// (the split-K chain then decodes with the table).  The row-block size is that of the
// least cost: a group multiplies only the row blocks that hold rows, the same ones at
// every size, so a size is paid for in waves per SIMD (its accumulators) and in groups
// (each decodes its expert anew): 2, 4, 6 and 8 row blocks measure 171, 174, 193 and
// 197 us at 16 rows per expert, 248, 227, 223 and 232 at 32, 318, 251, 243 and 257 at
// 47, 387, 324, 284 and 304 at 64, 524, 429, 392 and 354 at 94, which groups of cost
// 0.45, 0.55, 0.54 and 0.60 order alike; an expert with Poisson(M / E) rows takes sum
// over j of P(rows > 16 NRB j) groups.
int moe_mma_nrb(int M, int E, int H, int I) {
  if (E > 4096 || M / E < (moe_rows_table(E, H, I) ? 11 : 8)) return 0;
  // 32-bit byte offsets into the transformed rows
  if ((size_t)M * std::max(H, I) * 2 > 0xFFFFFFF0u) return 0;
  static constexpr double group_cost[] = {0.45, 0.55, 0.54, 0.60};
  const double lam = (double)M / E, dev = std::sqrt(2.0 * lam);
  int best = 8;
  double best_cost = 1e30;
  for (int nrb = 8; nrb >= 2; nrb -= 2) {
    const int br = 16 * nrb;
    // the j whose P is 1 to within rounding, then the others (normal tail)
    int j = std::max(0, (int)((lam - 6 * std::sqrt(lam)) / br));
    double groups = j;
    for (double p = 1.0; p > 1e-4; ++j) {
      p = 0.5 * std::erfc((j * br + 0.5 - lam) / dev);
      groups += p;
    }
    const double cost = groups * group_cost[nrb / 2 - 1];
    if (cost < best_cost * 0.999) {
      best_cost = cost;
      best = nrb;
    }
  }
  return best;
}

struct MoePlan {
  int M, S1, S2, R, n_groups, nrb;
  bool table;  // the grouped chain's decode
  size_t off_xh, off_p1, off_xh2, off_p2, off_rows, off_gexp, off_nact, off_d16, total;
};
// base: bytes at the start of the workspace left to the caller (the
// no-allocation variant keeps its counters there).
MoePlan moe_plan(int T, int top_k, int E, int H, int I, int K_gu, int K_dn, size_t base = 0) {
  MoePlan p;
  p.M = T * top_k;
  // a fixed scratch keeps 8 rows per group, whose row lists are the smaller
  p.R = E <= 4096 ? std::min(moe_group_rows(p.M, E), base ? 8 : 16) : 0;
  p.n_groups = p.R ? (p.M + E * (p.R - 1) + p.R - 1) / p.R : 0;
  // non-empty groups, about: the experts a uniform routing touches, or M/8
  const int eff = p.R ? std::max((p.M + 7) / 8,
                                 (int)(E * (1.0 - std::pow(1.0 - 1.0 / E, (double)p.M))))
                      : p.M;
  p.table = p.R && moe_rows_table(eff, H, I);
  // the grouped GEMVs aim for 2048 blocks: at 32 tokens (E = 256, H = 2048,
  // I = 512, top-8) 1,201 GB/s against 1,171 at 1024, 1,147 at 512 and
  // 1,161 at 4096 on MI355X; below about 16 tokens the kt bound sets S first
  p.S1 = fast_splits(K_gu, eff, H / 16, 2 * I / 16, 2048);
  p.S2 = fast_splits(K_dn, eff, I / 16, H / 16, 2048);
  auto al = [](size_t v) { return (v + 255) & ~size_t(255); };
  p.off_xh = al(base);
  p.off_p1 = al(p.off_xh + (size_t)p.M * H * 2);
  p.off_xh2 = al(p.off_p1 + (size_t)p.S1 * p.M * 2 * I * 4);
  p.off_p2 = al(p.off_xh2 + (size_t)p.M * I * 2);
  p.off_rows = al(p.off_p2 + (size_t)p.S2 * p.M * H * 4);
  p.off_gexp = al(p.off_rows + (size_t)p.n_groups * p.R * 4);
  p.off_nact = al(p.off_gexp + (size_t)p.n_groups * 4);
  p.off_d16 = 0;
  p.total = al(p.off_nact + 4);
  p.nrb = moe_mma_nrb(p.M, E, H, I);
  if (p.nrb) {
    // the grouped GEMM's buffers in the same bytes (fewer: f16 rows in place of
    // the float32 partials), so what a workspace of this size holds, and which
    // shapes a fixed scratch takes, does not depend on the path
    p.R = 16 * p.nrb;
    p.n_groups = (int)(((long)p.M + (long)E * (p.R - 1) + p.R - 1) / p.R);
    p.off_xh2 = al(p.off_xh + (size_t)p.M * H * 2);
    p.off_d16 = al(p.off_xh2 + (size_t)p.M * I * 2);
    p.off_rows = al(p.off_d16 + (size_t)p.M * H * 2);
    p.off_gexp = al(p.off_rows + (size_t)p.n_groups * p.R * 4);
    p.off_nact = al(p.off_gexp + (size_t)p.n_groups * 4);
    p.total = std::max(p.total, al(p.off_nact + 4));
  }
  return p;
}

// The grouped GEMM by hash: short-lived workgroups over every group there may be.
template <int K, int R>
int launch_rows_hash(const uint16_t* xh, const uint32_t* code, const int* rows, const int* gexp,
                     int n_groups, int M, int TK, int TN, int S, float* part, hipStream_t s) {
  const int tpw = K == 2 ? 16 : 8;
  hipLaunchKernelGGL((esc::k_gemv_fast_rows<K, false, R>), dim3((TN + tpw - 1) / tpw, n_groups, S),
                     dim3(256), 0, s, xh, code, rows, gexp, M, TK, TN, TK / S, part);
  return launched("k_gemv_fast_rows");
}

// The grouped GEMM with the table decode: the persistent k_gemv_rows_table
// (one workgroup per CU, the table staged once), its item count from the
// groups build_groups filled (nact, on the device).
template <int K, int R>
int launch_rows_table(const uint16_t* xh, const uint32_t* code, const int* rows, const int* gexp,
                      const int* nact, int M, int TK, int TN, int S, float* part, hipStream_t s) {
  static std::once_flag once;
  static hipError_t err = hipSuccess;
  std::call_once(once, [] {
    err = hipFuncSetAttribute((const void*)esc::k_gemv_rows_table<K, R>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, 65536 * 2);
  });
  if (int rc = hip_check(err, "hipFuncSetAttribute")) return rc;
  hipLaunchKernelGGL((esc::k_gemv_rows_table<K, R>), dim3(device_cus()), dim3(1024), 65536 * 2, s,
                     xh, code, rows, gexp, nact, M, TK, TN, TK / S, S, part);
  return launched("k_gemv_rows_table");
}

template <int K, int R>
int group_rows_k(const uint16_t* xh, const uint32_t* code, const int* rows, const int* gexp,
                 const int* nact, const MoePlan& p, int TK, int TN, int S, float* part,
                 hipStream_t s) {
  return p.table ? launch_rows_table<K, R>(xh, code, rows, gexp, nact, p.M, TK, TN, S, part, s)
                 : launch_rows_hash<K, R>(xh, code, rows, gexp, p.n_groups, p.M, TK, TN, S, part, s);
}

int group_rows(int K, const uint16_t* xh, const uint32_t* code, const int* rows, const int* gexp,
               const int* nact, const MoePlan& p, int TK, int TN, int S, float* part,
               hipStream_t s) {
  if (K == 2)
    return p.R == 16 ? group_rows_k<2, 16>(xh, code, rows, gexp, nact, p, TK, TN, S, part, s)
                     : group_rows_k<2, 8>(xh, code, rows, gexp, nact, p, TK, TN, S, part, s);
  return p.R == 16 ? group_rows_k<3, 16>(xh, code, rows, gexp, nact, p, TK, TN, S, part, s)
                   : group_rows_k<3, 8>(xh, code, rows, gexp, nact, p, TK, TN, S, part, s);
}

template <int K, bool GU>
int moe_mma_k(int nrb, const esc::MoeMmaArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(8 * ((a.n_groups + 7) / 8) * a.ncb)), blk(256);
  switch (nrb) {
    case 2: hipLaunchKernelGGL((esc::k_moe_mma<K, 2, GU>), grid, blk, 0, s, a); break;
    case 4: hipLaunchKernelGGL((esc::k_moe_mma<K, 4, GU>), grid, blk, 0, s, a); break;
    case 6: hipLaunchKernelGGL((esc::k_moe_mma<K, 6, GU>), grid, blk, 0, s, a); break;
    case 8: hipLaunchKernelGGL((esc::k_moe_mma<K, 8, GU>), grid, blk, 0, s, a); break;
    default: return fail(ESC_EINVAL, "internal: %d row blocks", nrb);
  }
  return launched("k_moe_mma");
}

template <bool GU>
int moe_mma(int K, int nrb, const esc::MoeMmaArgs& a, hipStream_t s) {
  return K == 2 ? moe_mma_k<2, GU>(nrb, a, s) : moe_mma_k<3, GU>(nrb, a, s);
}

// k_moe_prep: the input transform of every routed row and the grouping.
int moe_prep(const void* x, int dtype, const int32_t* ids, int T, int top_k, const float* rin,
             int H, float rs, uint16_t* xh, const MoePlan& p, int E, int* rows, int* gexp,
             int* nact, hipStream_t s) {
  // 8 lanes per block once that leaves eight waves per CU
  const long rows8 = (long)(H / 128) * T * ((top_k + esc::kOctSlots - 1) / esc::kOctSlots);
  const bool oct = rows8 >= 64L * device_cus();
  const long waves = oct ? (rows8 + 7) / 8 : (long)(H / 128) * p.M;
  const dim3 grid((unsigned)(1 + (waves + 15) / 16)), blk(1024);
  by_rows_type(dtype, [&](auto dt) {
    constexpr int DT = decltype(dt)::value;
    if (oct)
      hipLaunchKernelGGL((esc::k_moe_prep<true, DT>), grid, blk, 0, s, x, ids, top_k, rin, H, rs,
                         xh, p.M, E, p.R, p.n_groups, rows, gexp, nact);
    else
      hipLaunchKernelGGL((esc::k_moe_prep<false, DT>), grid, blk, 0, s, x, ids, top_k, rin, H, rs,
                         xh, p.M, E, p.R, p.n_groups, rows, gexp, nact);
  });
  return launched("k_moe_prep");
}

// One-launch path (fused.hpp).  Latency mode: small items over the whole GPU
// for one token-layer; throughput mode: large items for many token-layers.
constexpr int kFusedMaxRows = 64;

struct FusedPlan {
  int L, M, NB, NKC, NKB, NCP, nA, nB, grid;
  size_t off_pa, off_pb, off_xh2, off_int, total;
  int n_int;
};

// H/(16*KTA) <= 62: one polling wave reads the counter and every claim flag
// at once; top_k <= 32: the combine stages one row of d16 per slot in LDS.
bool fused_eligible(int T, int top_k, int H, int I) {
  return T * top_k <= kFusedMaxRows && top_k <= 32 && H % 256 == 0 && H / 128 <= 62 &&
         I % 128 == 0;
}

// kt per item of the many-layer two-launch path (gate_up, down)
// (measured on MI355X: 32 kt per item for either kernel is no faster)
constexpr int kKtaLayers = 16, kKtbLayers = 16;
// kt per item of one token-layer (latency-bound); with I == 512 the down
// items are 128-column blocks over all 32 kt (k_moe_down_blocks)
constexpr int kKtaSingle = 16, kKtbSingle = 16;
constexpr int kKtbBlocks = 32;
// kt per gate_up / down item of the single persistent launch: small items
// where it is esc_moe_expert_path's own choice (H or I not a multiple of 512);
// at the shapes that call runs as two launches (H and I multiples of 512),
// esc_moe_expert_path_one_launch takes larger ones (config 3: 22.3 us per
// token-layer against 32.9 us with the small items, 22.7-22.9 us with 16 and
// 8 kt, 24.5-28.0 us with 32 kt gate_up items)
constexpr int kKtaOne = 8, kKtbOne = 4;
constexpr int kKtaOneLarge = 16, kKtbOneLarge = 16;
// waves per gate_up / block down item of one token-layer, and per block
// down item of many token-layers
constexpr int kGateUpWavesSingle = 16, kDownBlockWavesSingle = 16;
constexpr int kDownBlockWavesLayers = 4;

// int_region > 0: the integer counters sit at offset 0 in a region of that
// many bytes and the float data after it, so calls of different shapes on one
// workspace never find another call's floats where their counters are (the
// no-allocation variant; the caller checks n_int * 4 <= int_region).
bool throughput_ok(int H, int I);

FusedPlan fused_plan(int L, int T, int top_k, int H, int I, bool throughput,
                     size_t int_region = 0) {
  // the two-launch path (throughput) uses the large items; the one-launch
  // path the small ones (KTA = 8, KTB = 4), which spread one token-layer wide,
  // or at two-launch shapes the middle ones (KTA = KTB = 16)
  const bool large = throughput;
  const bool layers = large && L > 1;
  const bool one_large = !large && throughput_ok(H, I);
  const int kta = layers ? kKtaLayers : large ? kKtaSingle : one_large ? kKtaOneLarge : kKtaOne;
  const bool blocks = large && I == 16 * kKtbBlocks;
  const int ktb = blocks ? kKtbBlocks
                  : layers ? kKtbLayers
                  : large  ? kKtbSingle
                  : one_large ? kKtbOneLarge : kKtbOne;
  FusedPlan f;
  f.L = L;
  f.M = T * top_k;
  f.NB = I / 128;
  f.NKC = std::max(1, H / (16 * kta));
  f.NKB = std::max(1, I / (16 * ktb));
  // 128-column blocks for the block kernels, 256-column pairs for every
  // other down item (k_moe_down_items, k_moe_fused): keyed on the kernel the
  // plan is for, not on the item's kt count
  f.NCP = blocks ? H / 128 : H / 256;
  f.nA = f.M * f.NB * f.NKC;
  f.nB = f.M * f.NCP * f.NKB;
  f.grid = throughput ? std::min(L * std::max(f.nA, f.nB), 1024)
                      : std::min(std::max(f.nA, f.nB), 2048);
  auto al = [](size_t v) { return (v + 255) & ~size_t(255); };
  f.n_int = L * (f.M * f.NB + f.nA + T * f.NCP) + 3;
  f.off_pa = al(int_region);
  f.off_pb = f.off_pa + al((size_t)L * f.nA * 256 * 4);
  f.off_xh2 = f.off_pb + al((size_t)L * f.nB * 256 * 4);
  const size_t end = f.off_xh2 + al((size_t)L * f.M * I * 2);
  f.off_int = int_region ? 0 : end;
  f.total = int_region ? end : end + al((size_t)f.n_int * 4);
  return f;
}

// Throughput mode needs the item sizes to divide the shapes.
bool throughput_ok(int H, int I) { return H % 512 == 0 && I % 512 == 0; }

esc::FusedMoe fused_args(const FusedPlan& f, void* ws, int T, int top_k, int H, int I) {
  char* w = static_cast<char*>(ws);
  int* ints = reinterpret_cast<int*>(w + f.off_int);
  esc::FusedMoe p{};
  p.partA = reinterpret_cast<float*>(w + f.off_pa);
  p.partB = reinterpret_cast<float*>(w + f.off_pb);
  p.xh2 = reinterpret_cast<uint16_t*>(w + f.off_xh2);
  p.cntA = ints;
  p.claimA = p.cntA + (size_t)f.L * f.M * f.NB;
  p.cntB = p.claimA + (size_t)f.L * f.nA;
  p.done = p.cntB + (size_t)f.L * T * f.NCP;
  p.err = p.done + 1;
  p.status = p.done + 2;
  p.host_err = nullptr;
  p.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
  p.L = f.L;
  p.T = T;
  p.top_k = top_k;
  p.H = H;
  p.I = I;
  p.NB = f.NB;
  p.NKC = f.NKC;
  p.NKB = f.NKB;
  p.NCP = f.NCP;
  p.nA = f.nA;
  p.nB = f.nB;
  return p;
}

template <int KG, int KD, bool TP>
int launch_fused_k(const esc::FusedMoe& p, int grid, hipStream_t s) {
  if constexpr (TP) {
    // two launches: every gate_up item, then every down item (grid unused);
    // the down inputs are precomputed once per (row, h-block) for
    // multi-layer calls
    (void)grid;
    const dim3 ga(p.L * p.nA), gb(p.L * p.nB), blk(esc::kFusedThreads);
    // the plan's down item size: whole-input blocks (I == 512) or split-K
    const int ktb = p.I / (16 * p.NKB);
    // records in a device table (esc_moe_expert_path_layers, any L): the
    // many-layer items; one record in the arguments: the single-layer ones
    if (p.layers) {
      hipLaunchKernelGGL((esc::k_moe_gate_up_items<KG, kKtaLayers, true>), ga, blk, 0, s, p);
      if (int rc = launched("k_moe_gate_up_items")) return rc;
      if (ktb == kKtbBlocks) {
        hipLaunchKernelGGL((esc::k_moe_down_blocks<KG, KD, true, kDownBlockWavesLayers>), gb,
                           dim3(64 * kDownBlockWavesLayers), 0, s, p);
        return launched("k_moe_down_blocks");
      }
      hipLaunchKernelGGL((esc::k_moe_down_items<KG, KD, kKtbLayers, true>), gb, blk, 0, s, p);
      return launched("k_moe_down_items");
    }
    hipLaunchKernelGGL((esc::k_moe_gate_up_items<KG, kKtaSingle, false, kGateUpWavesSingle>), ga,
                       dim3(64 * kGateUpWavesSingle), 0, s, p);
    if (int rc = launched("k_moe_gate_up_items")) return rc;
    if (ktb == kKtbBlocks) {
      hipLaunchKernelGGL((esc::k_moe_down_blocks<KG, KD, false, kDownBlockWavesSingle>), gb,
                         dim3(64 * kDownBlockWavesSingle), 0, s, p);
      return launched("k_moe_down_blocks");
    }
    hipLaunchKernelGGL((esc::k_moe_down_items<KG, KD, kKtbSingle, false>), gb, blk, 0, s, p);
    return launched("k_moe_down_items");
  } else {
    // k_moe_fused's down items are 256-column pairs (16 tiles each)
    ESC_REQUIRE(p.NCP * 256 == p.H, "one-launch plan with %d column groups for H=%d", p.NCP, p.H);
    // the plan's item size (fused_plan: large items at two-launch shapes)
    if (p.H == 16 * kKtaOneLarge * p.NKC)
      hipLaunchKernelGGL((esc::k_moe_fused<KG, KD, kKtaOneLarge, kKtbOneLarge, true>), dim3(grid),
                         dim3(esc::kFusedThreads), 0, s, p);
    else
      hipLaunchKernelGGL((esc::k_moe_fused<KG, KD, kKtaOne, kKtbOne, true>), dim3(grid),
                         dim3(esc::kFusedThreads), 0, s, p);
    return launched("k_moe_fused");
  }
}

template <bool TP>
int launch_fused(const esc::FusedMoe& p, int K_gu, int K_dn, int grid, hipStream_t s) {
  if (K_gu == 2)
    return K_dn == 2 ? launch_fused_k<2, 2, TP>(p, grid, s) : launch_fused_k<2, 3, TP>(p, grid, s);
  return K_dn == 2 ? launch_fused_k<3, 2, TP>(p, grid, s) : launch_fused_k<3, 3, TP>(p, grid, s);
}

// ---- many-layer calls: the table-assisted kernels (K=2 gate_up and down,
// layers.hpp) or the item kernels above (any other K).  One workspace serves
// both: the item kernels' counters at offset 0, the table-assisted kernels'
// group counters after them, and each path's float data after both counter
// regions, so calls of either path on one workspace never find the other's
// floats where their counters are.
struct LayersWs {
  FusedPlan f;  // the item kernels' plan
  size_t off_cnt_gu, off_cnt_dn, off_cnt_cb, off_part, off_xh2, off_rows, total;
};

LayersWs layers_ws(int L, int T, int top_k, int H, int I) {
  auto al = [](size_t v) { return (v + 255) & ~size_t(255); };
  LayersWs w;
  const size_t M = (size_t)T * top_k, NB = I / 128, NKC = H / 128, NCP = H / 256;
  w.off_cnt_gu = al((size_t)fused_plan(L, T, top_k, H, I, true).n_int * 4);
  w.off_cnt_dn = w.off_cnt_gu + al(L * M * NB * 4);
  w.off_cnt_cb = w.off_cnt_dn + al(L * M * NCP * 4);
  const size_t ireg = w.off_cnt_cb + al((size_t)L * T * NCP * 4);
  w.f = fused_plan(L, T, top_k, H, I, true, ireg);
  // partials: at most one slot per item of a group (one item per wave)
  w.off_part = ireg;
  const size_t part = std::max(L * M * NB * NKC, L * M * NCP * esc::kDownEighths) * 1024;
  w.off_xh2 = w.off_part + al(part);
  w.off_rows = w.off_xh2 + al(L * M * I * 2);
  w.total = std::max(w.f.total, w.off_rows + al(L * M * H * 2));
  return w;
}

bool layers_table_ok(int K_gu, int K_dn, int I) {
  return K_gu == 2 && K_dn == 2 && I <= esc::kLayersMaxI;
}

int launch_layers_table(const esc::MoeLayer* layers, const LayersWs& w, void* ws, int L, int T,
                        int top_k, int H, int I, hipStream_t s) {
  if (int rc = ensure_lut()) return rc;
  static std::once_flag attr_once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(attr_once, [] {
    const void* kerns[] = {(const void*)esc::k_moe_layers_gu, (const void*)esc::k_moe_layers_dn<1>,
                           (const void*)esc::k_moe_layers_dn<2>};
    for (const void* k : kerns) {
      const hipError_t e =
          hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 65536 * 2);
      if (e != hipSuccess) attr_err = e;
    }
  });
  if (int rc = hip_check(attr_err, "hipFuncSetAttribute")) return rc;
  esc::LayersMoe p{};
  p.layers = layers;
  p.ws = static_cast<char*>(ws);
  p.off_part = w.off_part;
  p.off_xh2 = w.off_xh2;
  p.off_rows = w.off_rows;
  p.off_cnt_cb = w.off_cnt_cb;
  p.L = L;
  p.T = T;
  p.top_k = top_k;
  p.H = H;
  p.I = I;
  p.M = T * top_k;
  p.NB = I / 128;
  p.NKC = H / 128;
  p.NHB = H / 128;
  const int cus = device_cus();
  const long na = (long)L * p.M * p.NB * p.NKC, nd = (long)L * p.M * (p.NHB / 2) * esc::kDownEighths;
  ESC_REQUIRE(na < (1L << 30) && nd < (1L << 30), "too many items (%ld, %ld)", na, nd);
  // one workgroup per CU, more when a wave would otherwise run more than
  // kLayersMaxRange items (its items' pointers are staged in LDS); each
  // wave runs P consecutive items, so a group of `size` items spans at most
  // (size + P - 2) / P + 1 waves
  auto plan = [&](long n, int size, int& grid) {
    const long wg = esc::kLayersWaves;
    grid = (int)std::max(std::min<long>(cus, (n + wg - 1) / wg),
                         (n + wg * esc::kLayersMaxRange - 1) / (wg * esc::kLayersMaxRange));
    p.P = (int)((n + wg * grid - 1) / (wg * grid));
    p.maxc = std::min(size, (size + p.P - 2) / p.P + 1);
  };
  const dim3 blk(64 * esc::kLayersWaves);
  const size_t lds = 65536 * 2;
  int grid = 0;
  plan(na, p.NKC, grid);
  p.off_cnt = w.off_cnt_gu;
  hipLaunchKernelGGL(esc::k_moe_layers_gu, dim3(grid), blk, lds, s, p);
  if (int rc = launched("k_moe_layers_gu")) return rc;
  plan(nd, esc::kDownEighths, grid);
  p.off_cnt = w.off_cnt_dn;
  // the down items' inputs: I/16 words, one or two registers per lane
  if (I <= 1024)
    hipLaunchKernelGGL(esc::k_moe_layers_dn<1>, dim3(grid), blk, lds, s, p);
  else
    hipLaunchKernelGGL(esc::k_moe_layers_dn<2>, dim3(grid), blk, lds, s, p);
  return launched("k_moe_layers_dn");
}
}  // namespace

extern "C" {
size_t esc_moe_expert_path_workspace(int T, int top_k, int E, int H, int I) {
  if (T <= 0 || top_k <= 0 || H <= 0 || I <= 0) return 0;
  // the plan's sizes depend on K only through the split counts; take the max
  size_t a = moe_plan(T, top_k, E, H, I, 2, 2).total, b = moe_plan(T, top_k, E, H, I, 3, 3).total;
  size_t c = moe_plan(T, top_k, E, H, I, 2, 3).total, d = moe_plan(T, top_k, E, H, I, 3, 2).total;
  size_t m = std::max(std::max(a, b), std::max(c, d));
  if (fused_eligible(T, top_k, H, I)) {
    m = std::max(m, fused_plan(1, T, top_k, H, I, false).total);
    if (throughput_ok(H, I)) m = std::max(m, fused_plan(1, T, top_k, H, I, true).total);
  }
  return m;
}

int esc_moe_status(const void* ws, size_t ws_bytes, int T, int top_k, int H, int I,
                   int32_t* host_flag, void* stream) {
  ESC_REQUIRE(ws && host_flag, "null pointer");
  *host_flag = 0;
  // only the single persistent launch has a bounded wait
  if (!fused_eligible(T, top_k, H, I)) return ESC_OK;
  if (throughput_ok(H, I)) {
    // esc_moe_expert_path runs two launches at this shape; a call through
    // esc_moe_expert_path_one_launch reports a give-up through the
    // device-wide flag (its workspace slot is not read: the same workspace
    // may have served the two-launch plan, whose layout differs)
    int* unused = nullptr;
    if (take_wait_error(&unused) == ESC_ETIMEOUT) *host_flag = 1;
    return ESC_OK;
  }
  const FusedPlan f = fused_plan(1, T, top_k, H, I, false);
  ESC_REQUIRE(ws_bytes >= f.total, "workspace smaller than the plan");
  // the status slot (the last integer): read, then cleared for the next read
  int32_t* st = reinterpret_cast<int32_t*>(static_cast<char*>(const_cast<void*>(ws)) + f.off_int) +
                (f.n_int - 1);
  if (int rc = hip_check(hipMemcpyAsync(host_flag, st, 4, hipMemcpyDeviceToHost, S(stream)),
                         "hipMemcpyAsync"))
    return rc;
  if (int rc = hip_check(hipMemsetAsync(st, 0, 4, S(stream)), "hipMemsetAsync")) return rc;
  if (int rc = hip_check(hipStreamSynchronize(S(stream)), "hipStreamSynchronize")) return rc;
  // the device-wide flag records the same event: taken here too, so a later
  // call does not report it again
  int* unused = nullptr;
  if (take_wait_error(&unused) == ESC_ETIMEOUT) *host_flag = 1;
  return ESC_OK;
}

int esc_moe_set_spin_limit(int polls) {
  g_spin_limit.store(polls < 0 ? esc::kSpinLimit : polls, std::memory_order_relaxed);
  return ESC_OK;
}

}  // extern "C"

namespace {
// The expert path on a given workspace; int_region > 0 puts every counter in
// a fixed region at its start (see fused_plan).
int moe_expert_path(const void* x, int dtype, const int32_t* ids, const float* scores, int T,
                    int top_k, int E, int H, int I, const uint32_t* gu_code, const float* gu_rin,
                    const float* gu_rout, int K_gu, const uint32_t* dn_code, const float* dn_rin,
                    const float* dn_rout, int K_dn, int use_lut, uint16_t* y, void* ws,
                    size_t ws_bytes, size_t int_region, void* stream, bool one_launch = false) {
  ESC_REQUIRE(x && ids && scores && gu_code && gu_rin && gu_rout && dn_code && dn_rin && dn_rout &&
                  y,
              "null pointer");
  ESC_REQUIRE(E > 0 && top_k >= 1 && top_k <= E, "bad E=%d / top_k=%d", E, top_k);
  if (int rc = check_proj(K_gu, H, 2 * I)) return rc;
  if (int rc = check_proj(K_dn, I, H)) return rc;
  ESC_REQUIRE(T >= 0, "negative token count");
  if (T == 0) return ESC_OK;
  // the item kernels read 16-bit rows; float32 rows take the chain
  if (fused_eligible(T, top_k, H, I) && dtype != ESC_ROWS_F32) {
    // throughput_ok: two launches (gate_up items, down items + combine),
    // measured faster than the single persistent launch for one token-layer
    // on gfx950; otherwise (or when the caller asks for it) the single
    // persistent launch
    const bool two = throughput_ok(H, I) && !one_launch;
    const FusedPlan f = fused_plan(1, T, top_k, H, I, two, int_region);
    // a fixed counter region keeps its last word for the status flag
    if (int_region && (size_t)f.n_int * 4 > int_region - 4)
      return fail(ESC_ENOSPACE, "%d counters exceed the %zu-byte counter region", f.n_int,
                  int_region - 4);
    if (!ws || ws_bytes < f.total)
      return fail(ESC_ENOSPACE, "workspace %zu bytes < required %zu", ws_bytes, f.total);
    esc::FusedMoe p = fused_args(f, ws, T, top_k, H, I);
    // Nothing clears the status flag of a fixed counter region (no caller
    // workspace is read by esc_moe_status): it lives in the region's last
    // word, outside every shape's counters, so a give-up of one call never
    // lands in the counters of a later call of another shape.
    if (int_region) p.status = reinterpret_cast<int*>(static_cast<char*>(ws) + int_region) - 1;
    p.xdt = dtype;
    p.l0 = esc::MoeLayer{static_cast<const uint16_t*>(x), ids, scores, gu_code, gu_rin, gu_rout, dn_code, dn_rin, dn_rout, y};
    p.layers = nullptr;
    if (two) return launch_fused<true>(p, K_gu, K_dn, f.grid, S(stream));
    // only the single persistent launch waits across workgroups
    if (int rc = take_wait_error(&p.host_err)) return rc;
    return launch_fused<false>(p, K_gu, K_dn, f.grid, S(stream));
  }
  const MoePlan p = moe_plan(T, top_k, E, H, I, K_gu, K_dn, int_region);
  if (!ws || ws_bytes < p.total)
    return fail(ESC_ENOSPACE, "workspace %zu bytes < required %zu", ws_bytes, p.total);
  if (use_lut)
    if (int rc = ensure_lut()) return rc;
  char* w = static_cast<char*>(ws);
  uint16_t* xh = reinterpret_cast<uint16_t*>(w + p.off_xh);
  float* p1 = reinterpret_cast<float*>(w + p.off_p1);
  uint16_t* xh2 = reinterpret_cast<uint16_t*>(w + p.off_xh2);
  float* p2 = reinterpret_cast<float*>(w + p.off_p2);
  hipStream_t s = S(stream);
  const float rs = esc::kRS;
  int* rows = reinterpret_cast<int*>(w + p.off_rows);
  int* gexp = reinterpret_cast<int*>(w + p.off_gexp);
  int* nact = reinterpret_cast<int*>(w + p.off_nact);
  if (p.R) {
    // input transform and expert grouping in one launch
    if (int rc = moe_prep(x, dtype, ids, T, top_k, gu_rin, H, rs, xh, p, E, rows, gexp, nact, s)) return rc;
    if (p.nrb) {
      uint16_t* d16 = reinterpret_cast<uint16_t*>(w + p.off_d16);
      esc::MoeMmaArgs a{xh, gu_code, rows, gexp, gu_rout, dn_rin, xh2, p.M, H / 16, 2 * I / 16,
                        p.n_groups, I / 128, rs};
      if (int rc = moe_mma<true>(K_gu, p.nrb, a, s)) return rc;
      a = {xh2, dn_code, rows, gexp, dn_rout, nullptr, d16, p.M, I / 16, H / 16, p.n_groups,
           (H + 255) / 256, rs};
      if (int rc = moe_mma<false>(K_dn, p.nrb, a, s)) return rc;
      return combine_rows(d16, scores, T, top_k, H, y, s);
    }
    if (int rc = group_rows(K_gu, xh, gu_code, rows, gexp, nact, p, H / 16, 2 * I / 16, p.S1, p1, s))
      return rc;
  } else if (int rc = moe_input(x, dtype, ids, top_k, gu_rin, H, rs, xh, p.M, s)) {
    return rc;
  } else if (int rc = by_k_lut<FastF>(K_gu, use_lut, xh, gu_code, ids, p.M, H / 16, 2 * I / 16,
                                      p.S1, p1, s)) {
    return rc;
  }
  auto mid = [&](auto sc) {
    hipLaunchKernelGGL((esc::k_moe_mid<decltype(sc)::value>), dim3(I / 128, p.M), dim3(64), 0, s,
                       p1, p.S1, p.M, I, ids, gu_rout, dn_rin, rs, xh2);
  };
  switch (esc::splits_class(p.S1)) {
    case 1: mid(std::integral_constant<int, 1>{}); break;
    case 2: mid(std::integral_constant<int, 2>{}); break;
    case 4: mid(std::integral_constant<int, 4>{}); break;
    default: mid(std::integral_constant<int, 0>{});
  }
  if (int rc = launched("k_moe_mid")) return rc;
  if (p.R) {
    if (int rc = group_rows(K_dn, xh2, dn_code, rows, gexp, nact, p, I / 16, H / 16, p.S2, p2, s))
      return rc;
  } else if (int rc = by_k_lut<FastF>(K_dn, use_lut, xh2, dn_code, ids, p.M, I / 16, H / 16, p.S2,
                                      p2, s)) {
    return rc;
  }
  auto combine = [&](auto sc) {
    hipLaunchKernelGGL((esc::k_moe_combine<decltype(sc)::value>), dim3(H / 128, T), dim3(64), 0, s,
                       p2, p.S2, p.M, H, ids, scores, top_k, dn_rout, rs, y);
  };
  switch (esc::splits_class(p.S2)) {
    case 1: combine(std::integral_constant<int, 1>{}); break;
    case 2: combine(std::integral_constant<int, 2>{}); break;
    case 4: combine(std::integral_constant<int, 4>{}); break;
    default: combine(std::integral_constant<int, 0>{});
  }
  return launched("k_moe_combine");
}

// ---- the whole MoE block: offsets of its scratch
struct BlockScratch {
  size_t logits, shg, g, u, hh, ids, scores, y, sh, total;
};
BlockScratch block_scratch(int T, int top_k, int E, int H, int Ish) {
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t o = at;
    at += (bytes + 255) & ~size_t(255);
    return o;
  };
  BlockScratch b{};
  b.logits = take((size_t)T * E * 2);
  b.shg = take((size_t)T * 2);
  b.g = take((size_t)T * Ish * 2);
  b.u = take((size_t)T * Ish * 2);
  b.hh = take((size_t)T * Ish * 2);
  b.ids = take((size_t)T * top_k * 4);
  b.scores = take((size_t)T * top_k * 4);
  b.y = take((size_t)T * H * 2);
  b.sh = take((size_t)T * H * 2);
  b.total = at;
  return b;
}

// Tokens up to which k_block_head / k_block_tail take the block's projections.
constexpr int kBlockFewTokens = 4;

template <int NR>
int block_head_nr(const esc::BlockHead& a, hipStream_t s) {
  const dim3 grid((a.E + 1 + 2 * a.Ish + 3) / 4), blk(256);
  switch ((a.H + 511) / 512) {
    case 1: hipLaunchKernelGGL((esc::k_block_head<NR, 1>), grid, blk, 0, s, a); break;
    case 2: hipLaunchKernelGGL((esc::k_block_head<NR, 2>), grid, blk, 0, s, a); break;
    case 3: hipLaunchKernelGGL((esc::k_block_head<NR, 3>), grid, blk, 0, s, a); break;
    case 4: hipLaunchKernelGGL((esc::k_block_head<NR, 4>), grid, blk, 0, s, a); break;
    case 5:
    case 6: hipLaunchKernelGGL((esc::k_block_head<NR, 6>), grid, blk, 0, s, a); break;
    default: hipLaunchKernelGGL((esc::k_block_head<NR, 8>), grid, blk, 0, s, a);
  }
  return launched("k_block_head");
}
int block_head(const esc::BlockHead& a, hipStream_t s) {
  return a.T == 1 ? block_head_nr<1>(a, s) : a.T == 2 ? block_head_nr<2>(a, s) : block_head_nr<4>(a, s);
}

template <int NR>
int block_tail_nr(const esc::BlockTail& a, hipStream_t s) {
  const dim3 grid((a.H + 3) / 4), blk(256);
  if (a.Ish <= 1024) hipLaunchKernelGGL((esc::k_block_tail<NR, 1>), grid, blk, 0, s, a);
  else if (a.Ish <= 2048) hipLaunchKernelGGL((esc::k_block_tail<NR, 2>), grid, blk, 0, s, a);
  else hipLaunchKernelGGL((esc::k_block_tail<NR, 4>), grid, blk, 0, s, a);
  return launched("k_block_tail");
}
int block_tail(const esc::BlockTail& a, hipStream_t s) {
  return a.T == 1 ? block_tail_nr<1>(a, s) : a.T == 2 ? block_tail_nr<2>(a, s) : block_tail_nr<4>(a, s);
}

// ---- the expert path without allocation: a file-scope device scratch array
// Its counters sit in the first kStaticIntBytes (zeroed once per device at
// set-up, left zero by every call), the float data after them.
constexpr size_t kStaticScratchBytes = size_t(4) << 20;
constexpr size_t kStaticIntBytes = size_t(128) << 10;
}  // namespace

__device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
// Device address of `scratch` per device (the symbol's host-side name is not
// a device address): looked up once per device, with that device current,
// and its counter region zeroed by a fill kernel.
void* g_scratch_ptr[kMaxDevices];

__global__ void k_zero_words(uint32_t* p, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

int ensure_scratch(void** out) {
  int dev = 0;
  if (int rc = hip_check(hipGetDevice(&dev), "hipGetDevice")) return rc;
  if (dev < 0 || dev >= kMaxDevices) return fail(ESC_EINVAL, "device index %d out of range", dev);
  std::lock_guard<std::mutex> lk(g_init_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    if (int rc = hip_check(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress"))
      return rc;
    if (!ptr) return fail(ESC_EHIP, "hipGetSymbolAddress returned a null scratch address");
    hipLaunchKernelGGL(k_zero_words, dim3(64), dim3(256), 0, 0, static_cast<uint32_t*>(ptr),
                       kStaticIntBytes / 4);
    if (int rc = launched("k_zero_words")) return rc;
    if (int rc = hip_check(hipDeviceSynchronize(), "scratch set-up sync")) return rc;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return ESC_OK;
}

bool scratch_ready() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return false;
  std::lock_guard<std::mutex> lk(g_init_mu);
  return g_scratch_ptr[dev] != nullptr;
}
}  // namespace

extern "C" {
int esc_moe_expert_path(const uint16_t* x, const int32_t* ids, const float* scores, int T,
                        int top_k, int E, int H, int I, const uint32_t* gu_code,
                        const float* gu_rin, const float* gu_rout, int K_gu,
                        const uint32_t* dn_code, const float* dn_rin, const float* dn_rout,
                        int K_dn, int use_lut, uint16_t* y, void* ws, size_t ws_bytes,
                        void* stream) {
  return esc_moe_expert_path_typed(x, ESC_ROWS_F16, ids, scores, T, top_k, E, H, I, gu_code, gu_rin,
                                   gu_rout, K_gu, dn_code, dn_rin, dn_rout, K_dn, use_lut, y, ws,
                                   ws_bytes, stream);
}

int esc_moe_expert_path_typed(const void* x, int dtype, const int32_t* ids, const float* scores,
                              int T, int top_k, int E, int H, int I, const uint32_t* gu_code,
                              const float* gu_rin, const float* gu_rout, int K_gu,
                              const uint32_t* dn_code, const float* dn_rin, const float* dn_rout,
                              int K_dn, int use_lut, uint16_t* y, void* ws, size_t ws_bytes,
                              void* stream) {
  ESC_REQUIRE(dtype == ESC_ROWS_F16 || dtype == ESC_ROWS_BF16 || dtype == ESC_ROWS_F32,
              "row element type must be ESC_ROWS_F16, ESC_ROWS_BF16 or ESC_ROWS_F32, got %d",
              dtype);
  if (int rc = ensure_wait_flag()) return rc;
  return moe_expert_path(x, dtype, ids, scores, T, top_k, E, H, I, gu_code, gu_rin, gu_rout, K_gu,
                         dn_code, dn_rin, dn_rout, K_dn, use_lut, y, ws, ws_bytes, 0, stream);
}

int esc_moe_expert_path_one_launch(const uint16_t* x, const int32_t* ids, const float* scores,
                                   int T, int top_k, int E, int H, int I,
                                   const uint32_t* gu_code, const float* gu_rin,
                                   const float* gu_rout, int K_gu, const uint32_t* dn_code,
                                   const float* dn_rin, const float* dn_rout, int K_dn,
                                   int use_lut, uint16_t* y, void* ws, size_t ws_bytes,
                                   void* stream) {
  ESC_REQUIRE(T >= 0 && top_k >= 1 && H > 0 && I > 0, "bad sizes T=%d top_k=%d H=%d I=%d", T,
              top_k, H, I);
  ESC_REQUIRE(fused_eligible(T, top_k, H, I),
              "one-launch expert path needs T*top_k <= %d, top_k <= 32, H a multiple of 256 "
              "up to 7936 and I a multiple of 128 (got T=%d top_k=%d H=%d I=%d)",
              kFusedMaxRows, T, top_k, H, I);
  if (int rc = ensure_wait_flag()) return rc;
  return moe_expert_path(x, ESC_ROWS_F16, ids, scores, T, top_k, E, H, I, gu_code, gu_rin, gu_rout,
                         K_gu, dn_code, dn_rin, dn_rout, K_dn, use_lut, y, ws, ws_bytes, 0, stream,
                         true);
}

size_t esc_moe_expert_path_static_max(void) { return kStaticScratchBytes; }

int esc_moe_expert_path_static(const uint16_t* x, const int32_t* ids, const float* scores, int T,
                               int top_k, int E, int H, int I, const uint32_t* gu_code,
                               const float* gu_rin, const float* gu_rout, int K_gu,
                               const uint32_t* dn_code, const float* dn_rin,
                               const float* dn_rout, int K_dn, int use_lut, uint16_t* y,
                               void* stream) {
  ESC_REQUIRE(T >= 0 && top_k >= 1 && H > 0 && I > 0, "bad sizes T=%d top_k=%d H=%d I=%d", T,
              top_k, H, I);
  if (T == 0) return ESC_OK;
  // the table, when asked for, is built by esc_init (a kernel, no allocation)
  ESC_REQUIRE(!use_lut || lut_ready(), "use_lut needs esc_init() on this device first");
  // the scratch set-up launches a fill kernel and synchronises, which a
  // stream under graph capture cannot do: such callers run esc_init first
  if (!scratch_ready()) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (int rc = hip_check(hipStreamIsCapturing(S(stream), &cs), "hipStreamIsCapturing"))
      return rc;
    ESC_REQUIRE(cs == hipStreamCaptureStatusNone,
                "the static scratch is not set up on this device: call esc_init() before "
                "capturing esc_moe_expert_path_static");
  }
  void* ptr = nullptr;
  if (int rc = ensure_scratch(&ptr)) return rc;
  return moe_expert_path(x, ESC_ROWS_F16, ids, scores, T, top_k, E, H, I, gu_code, gu_rin, gu_rout,
                         K_gu, dn_code, dn_rin, dn_rout, K_dn, use_lut, y, ptr, kStaticScratchBytes,
                         kStaticIntBytes, stream);
}

size_t esc_moe_block_scratch(int T, int top_k, int E, int H, int Ish) {
  if (T <= 0 || top_k <= 0 || E <= 0 || H <= 0 || Ish <= 0) return 0;
  return block_scratch(T, top_k, E, H, Ish).total;
}

int esc_moe_block(const void* x, int dtype, const uint16_t* xf, int T, int top_k, int E, int H,
                  int I, int Ish, const uint16_t* gate_w, const uint16_t* shg_w,
                  const int8_t* sg_w, const float* sg_s, const int8_t* su_w, const float* su_s,
                  const int8_t* sd_w, const float* sd_s, const uint32_t* gu_code,
                  const float* gu_rin, const float* gu_rout, int K_gu, const uint32_t* dn_code,
                  const float* dn_rin, const float* dn_rout, int K_dn, int use_lut, void* out,
                  void* scratch, size_t scratch_bytes, void* ws, size_t ws_bytes, void* stream) {
  ESC_REQUIRE(x && xf && gate_w && shg_w && sg_w && sg_s && su_w && su_s && sd_w && sd_s && out,
              "null pointer");
  ESC_REQUIRE(dtype == ESC_ROWS_F16 || dtype == ESC_ROWS_BF16 || dtype == ESC_ROWS_F32,
              "row element type must be ESC_ROWS_F16, ESC_ROWS_BF16 or ESC_ROWS_F32, got %d",
              dtype);
  ESC_REQUIRE(T >= 0, "negative token count");
  ESC_REQUIRE(E > 0 && E <= 1024, "expert count %d not in [1, 1024]", E);
  ESC_REQUIRE(top_k >= 1 && top_k <= 32 && top_k <= E, "top_k %d not in [1, min(32, E)]", top_k);
  ESC_REQUIRE(Ish > 0, "bad shared expert width %d", Ish);
  if (T == 0) return ESC_OK;
  const BlockScratch b = block_scratch(T, top_k, E, H, Ish);
  if (!scratch || scratch_bytes < b.total)
    return fail(ESC_ENOSPACE, "scratch %zu bytes < required %zu", scratch_bytes, b.total);
  char* p = static_cast<char*>(scratch);
  auto u16 = [&](size_t off) { return reinterpret_cast<uint16_t*>(p + off); };
  uint16_t *logits = u16(b.logits), *shg = u16(b.shg), *g = u16(b.g), *u = u16(b.u);
  uint16_t *y = u16(b.y), *sh = u16(b.sh);
  int32_t* ids = reinterpret_cast<int32_t*>(p + b.ids);
  float* scores = reinterpret_cast<float*>(p + b.scores);
  hipStream_t s = S(stream);
  // what the separate calls take: 128..4096 inputs of 16
  const bool few = T <= kBlockFewTokens && H % 16 == 0 && H >= 128 && H <= 4096 && Ish % 16 == 0 &&
                   Ish >= 128 && Ish <= 4096;
  if (few) {
    if (int rc = block_head({xf, gate_w, shg_w, sg_w, su_w, sg_s, su_s, logits, shg, g, u, T, E, H,
                             Ish}, s))
      return rc;
  } else {
    const void* w[] = {gate_w, shg_w, sg_w, su_w};
    const float* sc[] = {nullptr, nullptr, sg_s, su_s};
    uint16_t* o[] = {logits, shg, g, u};
    const int O[] = {E, 1, Ish, Ish};
    if (int rc = rows_multi(4, xf, w, sc, o, O, T, H, s)) return rc;
  }
  if (int rc = route_rows(reinterpret_cast<const esc::half_t*>(logits), T, E, top_k, ids, scores, s))
    return rc;
  if (int rc = esc_moe_expert_path_typed(x, dtype, ids, scores, T, top_k, E, H, I, gu_code, gu_rin,
                                         gu_rout, K_gu, dn_code, dn_rin, dn_rout, K_dn, use_lut, y,
                                         ws, ws_bytes, stream))
    return rc;
  if (few) return block_tail({g, u, shg, y, sd_w, sd_s, out, dtype, T, H, Ish}, s);
  if (int rc = esc_moe_shared_act(g, u, T, Ish, u16(b.hh), stream)) return rc;
  if (int rc = esc_w8a16(u16(b.hh), sd_w, sd_s, T, Ish, H, sh, stream)) return rc;
  hipLaunchKernelGGL(esc::k_block_out, dim3((H + 255) / 256, T), dim3(256), 0, s, y, sh, shg, H, out,
                     dtype);
  return launched("k_block_out");
}

size_t esc_moe_layers_workspace(int L, int T, int top_k, int H, int I) {
  if (L <= 0 || T <= 0 || top_k <= 0 || !fused_eligible(T, top_k, H, I) || !throughput_ok(H, I))
    return 0;
  return layers_ws(L, T, top_k, H, I).total;
}

int esc_moe_expert_path_layers(const esc_moe_layer* layers, int L, int T, int top_k, int E, int H,
                               int I, int K_gu, int K_dn, void* ws, size_t ws_bytes,
                               void* stream) {
  static_assert(sizeof(esc_moe_layer) == sizeof(esc::MoeLayer), "layer record layout");
  ESC_REQUIRE(layers, "null pointer");
  ESC_REQUIRE(L >= 0 && T >= 0, "negative size");
  ESC_REQUIRE(E > 0 && top_k >= 1 && top_k <= E, "bad E=%d / top_k=%d", E, top_k);
  if (int rc = check_proj(K_gu, H, 2 * I)) return rc;
  if (int rc = check_proj(K_dn, I, H)) return rc;
  ESC_REQUIRE(fused_eligible(T, top_k, H, I) && throughput_ok(H, I),
              "multi-layer expert path needs T*top_k <= %d, top_k <= 32, H and I multiples of "
              "512, H <= 7936 (got T=%d top_k=%d H=%d I=%d)",
              kFusedMaxRows, T, top_k, H, I);
  if (L == 0 || T == 0) return ESC_OK;
  const LayersWs w = layers_ws(L, T, top_k, H, I);
  if (!ws || ws_bytes < w.total)
    return fail(ESC_ENOSPACE, "workspace %zu bytes < required %zu", ws_bytes, w.total);
  const auto* lr = reinterpret_cast<const esc::MoeLayer*>(layers);
  if (layers_table_ok(K_gu, K_dn, I))
    return launch_layers_table(lr, w, ws, L, T, top_k, H, I, S(stream));
  esc::FusedMoe p = fused_args(w.f, ws, T, top_k, H, I);
  p.layers = lr;
  return launch_fused<true>(p, K_gu, K_dn, w.f.grid, S(stream));
}


// ---- decode-rate probe (measurement only)
size_t esc_decode_probe_words(int steps, int waves_per_cu) {
  if (steps <= 0 || steps % 4 || (waves_per_cu != 16 && waves_per_cu != 32)) return 0;
  return (size_t)device_cus() * waves_per_cu * steps * 64 * 4;
}

int esc_decode_probe(const uint32_t* code, int steps, int nt, int waves_per_cu, int prefetch,
                     float* out, void* stream) {
  ESC_REQUIRE(code && out, "null pointer");
  ESC_REQUIRE(steps > 0 && steps % 4 == 0, "steps must be a positive multiple of 4");
  ESC_REQUIRE(waves_per_cu == 16 || waves_per_cu == 32, "waves per CU must be 16 or 32");
  ESC_REQUIRE(nt == 0 || waves_per_cu == 16, "the table (nt > 0) fits one workgroup per CU");
  ESC_REQUIRE(prefetch >= 1 && prefetch <= 3, "prefetch depth must be 1, 2 or 3");
  if (nt > 0)
    if (int rc = ensure_lut()) return rc;
  const dim3 grid(device_cus() * (waves_per_cu / 16)), blk(1024);
  const size_t lds = nt > 0 ? 131072 : 0;
  auto go = [&](auto kern) -> int {
    if (lds)
      if (int rc = hip_check(hipFuncSetAttribute((const void*)kern,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)lds),
                             "hipFuncSetAttribute"))
        return rc;
    hipLaunchKernelGGL(kern, grid, blk, lds, S(stream), code, steps, out);
    return launched("k_decode_probe");
  };
  auto by_pf = [&](auto k1, auto k2, auto k3) -> int {
    return prefetch == 1 ? go(k1) : prefetch == 2 ? go(k2) : go(k3);
  };
#define ESC_PROBE(NT) \
  by_pf(esc::k_decode_probe<NT, 1>, esc::k_decode_probe<NT, 2>, esc::k_decode_probe<NT, 3>)
  switch (nt) {
    case 0: return ESC_PROBE(0);
    case 2: return ESC_PROBE(2);
    case 3: return ESC_PROBE(3);
    case 4: return ESC_PROBE(4);
    case 5: return ESC_PROBE(5);
    case 6: return ESC_PROBE(6);
    case 8: return ESC_PROBE(8);
  }
#undef ESC_PROBE
  return fail(ESC_EINVAL, "table pairs per 8 must be one of 0, 2, 3, 4, 5, 6, 8 (got %d)", nt);
}

}  // extern "C"
