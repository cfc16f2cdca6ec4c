// qgemm.hip -- tile plans and launches of the dense quantized matmul (the
// kernels: qgemm_tile.hpp).
#include <algorithm>
#include <type_traits>

#include "epilogue.hpp"
#include "imq_device.hpp"
#include "imq_kernels.hpp"
#include "qgemm_plan.hpp"

namespace imq {
namespace {

// What a launch costs, in one unit per model: a round of tiles
// split_steps * step(mt, nt) plus its prologue and output, a split its second
// launch and the workspace traffic (per output and split).
//
// 128-column tiles (one 32-column tile per wave, nt = 1) double the tiles of a
// shape at a given height, so a short M keeps a taller tile (each dequantized
// weight fragment feeds mt MFMAs); they read 1.5x the activation and weight
// bytes per flop of 256-column ones.
//
// kFit (us): fitted to 2300 forced plans (every tile, up to 12 splits, on 75
// shapes of 33 to 4608 rows, weights past the last-level cache): its pick is
// 0.5% slower than the fastest plan on average and 6.5% at worst, where the
// former model's was 3.4% and 33% slower.  The former model (units of about
// 0.36 us) kept 128-column tiles to activation panels under 4 MB and costed a
// split's second launch at a fifth: [1024 x 3072] K = 3072 28.4 us on 64 x 256
// tiles against 23.6 on 128 x 128, [1300 x 1536] K = 4096 31.9 (32 x 256)
// against 24.6 (64 x 128), [3000 x 2048] K = 6144 81.1 (192 x 256 split in
// two) against 70.3 (192 x 128 unsplit).  It stays for outputs whose partial
// sums of even two splits outgrow the static scratch (8.4 M outputs): there
// both pick alike, and the shapes that the allocation-free entry refuses stay
// the same.  Below that size a split's partial sums fit that scratch.
//
// Two charges that the fit, made on plain products of aligned widths, lacks.  Rows
// of partial sums that are not whole 16-byte pieces (N % 4 != 0) are added float by
// float: without ragged_output [62 x 12390] K = 8448 was split in five, 37.9 us a
// call against 31.3 by two splits; [391 x 9998] K = 3712 68.4 / 50.9, [372 x 6779] K =
// 5824 57.3 / 45.6; the other way [711 x 2474] K = 9984 52.3 / 55.1.  A gate/up pair's
// sum reads two rows per split: four encoder layers (19456 rows of weights, K =
// 2560) of 129 / 136 / 144 rows 338.1 / 340.4 / 342.5 us split in three, 330.1 / 330.7 /
// 332.9 in two; at 64 rows, on half the tile height, three stay ahead, 253.9 against
// 257.0.
struct CostModel {
  double step2[9], step1[9];  // per K-step, by mt: 256 and 128 columns
  double round2, round1;      // per round of tiles
  double split2, split1;      // per split launch
  double per_split;           // and per split of it
  double per_output;          // per output and split
  double ragged_output;       // more where rows of partial sums are not whole 16-byte pieces
  double pair_split;          // a gate/up pair's, per split past the second and 32 rows of tile
};
constexpr CostModel kFit = {
    {0, 0.782, 0.967, 0, 1.477, 1.767, 2.102, 2.449, 2.614},
    {0, 0, 0.557, 0, 0.840, 0.978, 1.211, 1.398, 1.512},
    3.878, 2.818, 2.975, 2.975, 0.371, 1.11e-6, 0.7e-6, 0.085};
constexpr CostModel kLarge = {
    {0, 2.5, 3.5, 0, 5.5, 6.5, 7.5, 8.5, 9.5},
    {0, 0, 1.5, 0, 3.35, 4.275, 5.2, 6.125, 7.05},
    12.0, 12.0, 3.0, 6.0, 0.0, 8.0 / 1.4e6, 0.0, 0.0};
constexpr size_t kLargeMaxPanel = (size_t)4 << 20;  // of a 128-column tile's activations

// The encoder layers' residual add (K % 256 == 0) keeps the former model past 128
// rows: an unsplit tile reads its residual behind its last product, where the
// split's second launch streams it, and a layer's weights are often in the
// last-level cache, where more splits pay less than the fit has it.  Four layers,
// fitted against former: 1024 wide, 180 rows 197.9 / 194 us, 511 rows 236.1 / 230.3;
// 2560 wide, 384 rows 510.5 / 489; below the line 128 rows 1024 wide 186 / 192.
constexpr int kResidFitRows = 128;

// Tile and K split of a launch over n weight rows (split: K may be split;
// pair: a gate/up pair, whose wave holds gate and up columns: 256-column tiles
// of 128 rows and more).  Splits are taken only when the tiles leave CUs idle.
// ms: the rows of each of `count` products of one launch.
BigPlan pick_big_plan(const int* ms, int count, int n, int k, int cus, bool split, bool pair,
                      bool resid = false) {
  int m = 0;
  for (int i = 0; i < count; ++i) m += ms[i];
  const int steps = (k + 255) / 256 * 2;  // of 128, whole scale blocks
  const bool tail = k % 256 != 0;
  const bool large = (size_t)m * n * 8 > kStaticScratchBytes ||
                     (resid && !tail && m > kResidFitRows);
  const CostModel& c = large ? kLarge : kFit;
  const double per_output = c.per_output + (n % 4 ? c.ragged_output : 0.0);
  BigPlan best{8, 2, 1, steps};
  double best_cost = 1e30;
  for (int nt : {2, 1}) {
    if (nt == 1 && pair) continue;
    const int tiles_n = (n + 128 * nt - 1) / (128 * nt);
    for (int mt : {8, 7, 6, 5, 4, 2, 1}) {
      // 32 x 128 tiles are not planned: that instantiation spills registers
      // to scratch memory (the 32 x 256 tile or the few-row kernel take
      // those shapes).
      if (nt == 1 && mt == 1) continue;
      // K % 256 != 0 is built for fewer tiles (tile::tile_built).
      if (tail && (nt == 1 ? mt > 4 : mt == 5 || mt == 7)) continue;
      if (count > 1 && !tile::group_built(mt, nt)) continue;
      long tiles = 0;
      for (int i = 0; i < count; ++i) tiles += (long)((ms[i] + 32 * mt - 1) / (32 * mt)) * tiles_n;
      // Up to two rounds of workgroups (the former model: any).
      const int max_splits =
          !split || tiles >= cus ? 1
          : large                ? std::max(1, steps / 2)
                                 : std::max(1, (int)std::min<long>(steps / 2, 2 * cus / tiles));
      for (int sp = 1; sp <= max_splits; ++sp) {
        const int sps = ((steps + sp - 1) / sp + 1) / 2 * 2;  // even
        const int eff = (steps + sps - 1) / sps;
        if (eff != sp || (eff == 1 && mt < 4 && pair)) continue;
        if ((!large || tail) && eff > 1 && (size_t)eff * m * n * 4 > kStaticScratchBytes) break;
        if (large && nt == 1 && (size_t)m * sps * 128 * 2 > kLargeMaxPanel) continue;
        const long rounds = (tiles * eff + cus - 1) / cus;
        double cost = (double)rounds *
                      (sps * (nt == 2 ? c.step2[mt] : c.step1[mt]) + (nt == 2 ? c.round2 : c.round1));
        if (eff > 1)
          cost += (nt == 2 ? c.split2 : c.split1) + eff * (c.per_split + (double)m * n * per_output) +
                  (pair && eff > 2 ? (eff - 2) * mt * c.pair_split : 0.0);
        if (cost < best_cost - 1e-9) {
          best_cost = cost;
          best = BigPlan{mt, nt, eff, sps};
        }
      }
    }
  }
  return best;
}

BigPlan pick_big_plan(int m, int n, int k, int cus, bool split, bool pair = false,
                      bool resid = false) {
  return pick_big_plan(&m, 1, n, k, cus, split, pair, resid);
}

// 16-byte alignment of an output or residual pointer (vector output stores).
bool al16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

int device_cus() {
  static const int cus = [] {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
      return v;
    return 256;
  }();
  return cus;
}

// K % 256 != 0: a short K whose 128 x 256 tiles nearly fill the chip stays on the
// register-staged kernel.  The large-M kernel computes K rounded up to 256, and at
// three to ten groups its prologue and staged output weigh as much as its loop,
// while two 128 x 256 workgroups fit a CU.  Measured against it (us, weights past
// the last-level cache): [4608 x 9216] K = 448 / 576 / 704 55.0 / 66.4 / 77.2 here,
// 59.2 / 71.6 / 74.0 there; [512 x 18432] K = 320 / 448 / 704 13.4 / 16.5 / 24.9 and
// 15.9 / 16.8 / 20.4; with fewer tiles it has no K split and leaves CUs idle: [2048 x
// 2048] K = 320 10.5 and 8.3, [100 x 3072] K = 448 12.2 and 5.6, [333 x 5001]
// K = 2880 84.5 and 24.3, [512 x 2560] K = 2880 69.1 and 17.3.  At one scale block (K
// = 64, 128 or 192) it always stays there.
//
// From 640 to 1700 of K it stays there where the two costs (us) say so: its tiles
// just fill one or more rounds of two per CU while the large-M kernel's last round
// is nearly empty or a quarter of its K is padding.  Both costs are fitted to 430
// ragged shapes (plain, post-scaled and gate/up outputs alike, so that one choice
// serves all of them): [865 x 16768] K = 832 / 1152 / 1600 (462 tiles of 128 x 256)
// 35.9 / 46.7 / 62.0 here, 40.7 / 48.4 / 66.4 there, with post-scaled fp32 outputs 41.7
// / 52.2 / 67.7 and 50.1 / 57.1 / 72.0; [1948 x 19724] K = 832 125 and 141; on the
// other side [495 x 26496] K = 1152 45.0 and 40.9, [4608 x 3072] K = 960 35.5 and 33.3.
// Past 1700 the large-M kernel is level or ahead ([865 x 16768] K = 2112 83.2 and
// 89.5, but 2880 120.8 and 110.8).
bool tail_on_register_kernel(int k, int n, int m) {
  if (k % 256 == 0) return false;
  const size_t tiles = (size_t)((m + 127) / 128) * ((n + 255) / 256);
  if (k < 320 || (k < 640 && tiles >= 192)) return true;
  if (k < 640 || k > 1700) return false;
  const int cus = device_cus();
  const double outputs = (double)m * n;
  const BigPlan p = pick_big_plan(m, n, k, cus, false);
  const size_t big_tiles =
      (size_t)((m + 32 * p.mt - 1) / (32 * p.mt)) * ((n + 128 * p.nt - 1) / (128 * p.nt));
  const double rounds = (double)((big_tiles + cus - 1) / cus);
  const double big =
      rounds * (1.14 * p.split_steps * (p.nt == 2 ? kFit.step2[p.mt] : kFit.step1[p.mt]) +
                2.0 * (p.nt == 2 ? kFit.round2 : kFit.round1)) +
      0.12e-6 * outputs;
  // Rounds of two workgroups a CU; a last round of one a CU is quicker.
  const int groups = k / 64;
  const size_t pairs = tiles / (2 * (size_t)cus), rest = tiles % (2 * (size_t)cus);
  const double reg = (double)(pairs + (rest > (size_t)cus)) * (1.97 * groups + 0.8) +
                     (rest > 0 && rest <= (size_t)cus ? 1.54 * groups + 2.7 : 0.0) +
                     0.55e-6 * outputs;
  return reg < 1.02 * big;
}

// The tile kernels with output stage ep (the large-M one with two groups per
// K-step, 2-stage ring: half the barriers and waits of one group per step,
// measured 3.5% faster at M=4608 K=3072 N=18432).  When the planner splits K
// and ws holds the partial sums, the kernel writes fp32 partials and
// tile::launch_sum adds them and applies ep; otherwise one pass.
template <int T, class EP>
hipError_t launch_big_ep(const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                         const uint16_t* x, const EP& ep, int k, int n, int m, hipStream_t stream,
                         SplitWs ws) {
  // Short ragged K (the DiT's x_embedder, K = 128) or operands past 32-bit
  // offsets: the register-staged kernel, one pass.
  if (!qgemm_big_supported(k, n, m)) {
    if (ws.kernels) ++*ws.kernels;
    return tile::launch_reg<T, EP>(w, scales, biases, x, ep, k, n, m, stream);
  }
  int cols = n;  // weight rows covered
  int width = n, gate_row = 0, up_row = 0;
  if constexpr (EP::kPair) {
    cols = 2 * ep.width;
    width = ep.width;
    gate_row = ep.gate_row;
    up_row = ep.up_row;
  }
  const bool tail = k % 256 != 0;
  const int cus = device_cus();
  constexpr bool kResid = std::is_same_v<EP, EpResidAdd<T>>;
  BigPlan p = pick_big_plan(m, cols, k, cus, ws.p != nullptr, EP::kPair, kResid);
  if (p.splits > 1 && ws.bytes < (size_t)p.splits * m * cols * sizeof(float))
    p = pick_big_plan(m, cols, k, cus, false, EP::kPair, kResid);  // no room for the partial sums
  if (ws.kernels) *ws.kernels += p.splits == 1 ? 1 : 2;
  if (p.splits == 1)
    return tail ? tile::launch_plan<T, EP, true>(p, w, scales, biases, x, ep, k, n, m, stream)
                : tile::launch_plan<T, EP, false>(p, w, scales, biases, x, ep, k, n, m, stream);
  using Part = EpPartial<EP::kPair>;
  const Part part{ws.p, cols, width, gate_row, up_row};
  const hipError_t e =
      tail ? tile::launch_plan<T, Part, true>(p, w, scales, biases, x, part, k, n, m, stream)
           : tile::launch_plan<T, Part, false>(p, w, scales, biases, x, part, k, n, m, stream);
  if (e != hipSuccess) return e;
  return tile::launch_sum<T, EP>(ws, p.splits, m, width, cols, ep, stream);
}

template <int T>
hipError_t launch_t(const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                    const uint16_t* x, uint16_t* y, int k, int n, int m, hipStream_t stream,
                    SplitWs ws) {
  return launch_big_ep<T>(w, scales, biases, x, EpStore<T>{y, n, al16(y) && n % 8 == 0}, k, n, m,
                          stream, ws);
}

}  // namespace

bool qgemm_big_supported(int k, int n, int m) {
  // The buffer-load kernel addresses x and w with 32-bit byte offsets.
  return (size_t)m * k * 2 < ((size_t)1 << 31) && (size_t)n * k / 2 < ((size_t)1 << 31) &&
         !tail_on_register_kernel(k, n, m);
}

hipError_t launch_qgemm(const uint32_t* w, const void* scales, const void* biases, const void* x,
                        void* y, int k, int n, int m, int dtype, hipStream_t stream, SplitWs ws) {
  const auto* s = static_cast<const uint16_t*>(scales);
  const auto* b = static_cast<const uint16_t*>(biases);
  const auto* xx = static_cast<const uint16_t*>(x);
  auto* yy = static_cast<uint16_t*>(y);
  switch (dtype) {
    case kBf16: return launch_t<kBf16>(w, s, b, xx, yy, k, n, m, stream, ws);
    case kF16: return launch_t<kF16>(w, s, b, xx, yy, k, n, m, stream, ws);
    default: return hipErrorInvalidValue;
  }
}

size_t qgemm_split_bytes(int k, int n, int m, bool fused) {
  if (!qgemm_big_supported(k, n, m)) return 0;
  // The most a stage over these rows takes: a fused stage may be a gate/up
  // pair (no 128-column tiles), a residual add or another.
  size_t bytes = 0;
  for (int v = 0; v < (fused ? 3 : 1); ++v) {
    const BigPlan p = pick_big_plan(m, n, k, device_cus(), true, v == 1, v == 2);
    if (p.splits > 1) bytes = std::max(bytes, (size_t)p.splits * m * n * sizeof(float));
  }
  return bytes;
}

QgemmPlan qgemm_plan(int k, int n, int m, bool split, bool pair) {
  if (!qgemm_big_supported(k, n, m)) return QgemmPlan{false, 128, 1, 0, 256};
  const BigPlan p = pick_big_plan(m, n, k, device_cus(), split, pair);
  return QgemmPlan{true, 32 * p.mt, p.splits,
                   p.splits > 1 ? (size_t)p.splits * m * n * sizeof(float) : 0, 128 * p.nt};
}

hipError_t launch_qgemm_postscale(const uint32_t* w, const void* scales, const void* biases,
                                  const void* x, float* y, int k, int n, int m, float scale,
                                  int dtype, hipStream_t stream, SplitWs ws,
                                  const float* scale_dev) {
  const auto* s = static_cast<const uint16_t*>(scales);
  const auto* b = static_cast<const uint16_t*>(biases);
  const auto* xx = static_cast<const uint16_t*>(x);
  const bool vec = al16(y) && n % 4 == 0;
  switch (dtype) {
    case kBf16:
      return launch_big_ep<kBf16>(w, s, b, xx, EpPostscale<kBf16>{y, n, scale, vec, scale_dev}, k,
                                  n, m, stream, ws);
    case kF16:
      return launch_big_ep<kF16>(w, s, b, xx, EpPostscale<kF16>{y, n, scale, vec, scale_dev}, k,
                                 n, m, stream, ws);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_qgemm_postscale_f16(const uint32_t* w, const void* scales, const void* biases,
                                      const void* x, void* y, int k, int n, int m, float scale,
                                      hipStream_t stream, const float* scale_dev) {
  auto* yy = static_cast<uint16_t*>(y);
  const bool vec = al16(y) && n % 8 == 0;
  return launch_big_ep<kF16>(w, static_cast<const uint16_t*>(scales),
                             static_cast<const uint16_t*>(biases), static_cast<const uint16_t*>(x),
                             EpPostscaleF16{yy, n, scale, vec, scale_dev}, k, n, m, stream,
                             SplitWs{});
}

hipError_t launch_qgemm_resid_add(const uint32_t* w, const void* scales, const void* biases,
                                  const void* x, const void* resid, void* y, int k, int n, int m,
                                  int dtype, hipStream_t stream, SplitWs ws) {
  const auto* s = static_cast<const uint16_t*>(scales);
  const auto* b = static_cast<const uint16_t*>(biases);
  const auto* xx = static_cast<const uint16_t*>(x);
  auto* yy = static_cast<uint16_t*>(y);
  const auto* rr = static_cast<const uint16_t*>(resid);
  const bool vec = al16(y) && al16(resid) && n % 8 == 0;
  switch (dtype) {
    case kBf16:
      return launch_big_ep<kBf16>(w, s, b, xx, EpResidAdd<kBf16>{yy, rr, n, vec}, k, n, m, stream,
                                  ws);
    case kF16:
      return launch_big_ep<kF16>(w, s, b, xx, EpResidAdd<kF16>{yy, rr, n, vec}, k, n, m, stream,
                                 ws);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_qgemm_gate_add(const uint32_t* w, const void* scales, const void* biases,
                                 const void* x, const float* residual, const float* gate, float* y,
                                 int k, int n, int m, float scale, int dtype, hipStream_t stream,
                                 SplitWs ws, const float* scale_dev) {
  const auto* s = static_cast<const uint16_t*>(scales);
  const auto* b = static_cast<const uint16_t*>(biases);
  const auto* xx = static_cast<const uint16_t*>(x);
  const bool vec = al16(y) && al16(residual) && al16(gate) && n % 4 == 0;
  switch (dtype) {
    case kBf16:
      return launch_big_ep<kBf16>(
          w, s, b, xx, EpGateAdd<kBf16>{y, residual, gate, n, scale, vec, scale_dev}, k, n, m,
          stream, ws);
    case kF16:
      return launch_big_ep<kF16>(
          w, s, b, xx, EpGateAdd<kF16>{y, residual, gate, n, scale, vec, scale_dev}, k, n, m,
          stream, ws);
    default: return hipErrorInvalidValue;
  }
}

namespace {

// y[row][j] = T(EpSwiGLU(g, u)) from a T product [rows, 2 width] (gate at
// column j, up at width + j): the fused stage's arithmetic on values already
// rounded to T (its round_to is then exact).
template <int T>
__global__ __launch_bounds__(256) void swiglu_t_kernel(const uint16_t* __restrict__ gu, int ld,
                                                       int rows, const EpSwiGLU<T> ep) {
  const long t = (long)blockIdx.x * 256 + threadIdx.x;
  if (t >= (long)rows * ep.width) return;
  const int row = (int)(t / ep.width), j = (int)(t % ep.width);
  const uint16_t* r = gu + (size_t)row * ld;
  ep.emit1(row, j, Elem<T>::out(ep.value2(Elem<T>::param(r[j]), Elem<T>::param(r[ep.width + j]))));
}

}  // namespace

hipError_t launch_swiglu_t(const void* gu, int ld, int rows, int width, void* y, int ldy,
                           float in_scale, float out_scale, int dtype, hipStream_t stream) {
  if (rows <= 0 || width <= 0) return hipSuccess;
  const auto* g = static_cast<const uint16_t*>(gu);
  auto* yy = static_cast<uint16_t*>(y);
  const dim3 grid((unsigned)(((long)rows * width + 255) / 256));
  switch (dtype) {
    case kBf16:
      hipLaunchKernelGGL((swiglu_t_kernel<kBf16>), grid, dim3(256), 0, stream, g, ld, rows,
                         EpSwiGLU<kBf16>{yy, ldy, width, 0, width, in_scale, out_scale, false});
      return hipGetLastError();
    case kF16:
      hipLaunchKernelGGL((swiglu_t_kernel<kF16>), grid, dim3(256), 0, stream, g, ld, rows,
                         EpSwiGLU<kF16>{yy, ldy, width, 0, width, in_scale, out_scale, false});
      return hipGetLastError();
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_reduce_swiglu(const float* ws, int splits, int m, int width, void* y, int ldy,
                                float in_scale, float out_scale, int dtype, hipStream_t stream) {
  auto* yy = static_cast<uint16_t*>(y);
  const bool vec = al16(y) && ldy % 8 == 0;
  const SplitWs sw{const_cast<float*>(ws), 0};
  switch (dtype) {
    case kBf16:
      return tile::launch_sum<kBf16>(
          sw, splits, m, width, 2 * width,
          EpSwiGLU<kBf16>{yy, ldy, width, 0, width, in_scale, out_scale, vec}, stream);
    case kF16:
      return tile::launch_sum<kF16>(
          sw, splits, m, width, 2 * width,
          EpSwiGLU<kF16>{yy, ldy, width, 0, width, in_scale, out_scale, vec}, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_qgemm_swiglu(const uint32_t* w, const void* scales, const void* biases,
                               const void* x, void* y, int ldy, int k, int n, int m, int width,
                               int gate_row, int up_row, float in_scale, float out_scale, int dtype,
                               hipStream_t stream, SplitWs ws) {
  const auto* s = static_cast<const uint16_t*>(scales);
  const auto* b = static_cast<const uint16_t*>(biases);
  const auto* xx = static_cast<const uint16_t*>(x);
  auto* yy = static_cast<uint16_t*>(y);
  const bool vec = al16(y) && ldy % 8 == 0;
  switch (dtype) {
    case kBf16:
      return launch_big_ep<kBf16>(
          w, s, b, xx,
          EpSwiGLU<kBf16>{yy, ldy, width, gate_row, up_row, in_scale, out_scale, vec}, k, n, m,
          stream, ws);
    case kF16:
      return launch_big_ep<kF16>(
          w, s, b, xx,
          EpSwiGLU<kF16>{yy, ldy, width, gate_row, up_row, in_scale, out_scale, vec}, k, n, m,
          stream, ws);
    default: return hipErrorInvalidValue;
  }
}

namespace {

// Stages of a group that may split K: the sums of six q, k and v products would be
// six more launches, and the split form of a pair's shared launch is not built.
// Unsplit they are ahead of the separate, split products at every size measured,
// the smallest blocks too: q, k and v of 256 + 16 rows (dim 1536, 108 tiles on 256
// CUs) and of 64 + 64 (768) 14.4 and 9.3 us, whole steps of such double blocks by
// graph 642 -> 425 us (five blocks) and 400 -> 232 (four).
bool group_splits(QgemmGroup::Stage stage) { return stage == QgemmGroup::kGateAdd; }

bool group_fits(int k, int n, const int* ms, int count) {
  for (int i = 0; i < count; ++i)
    if (!qgemm_big_supported(k, n, ms[i])) return false;
  return true;
}

template <int T>
hipError_t launch_group_t(const QgemmGroup& in, int k, int n, hipStream_t stream, SplitWs ws) {
  const int cus = device_cus();
  int ms[tile::kMaxGroup], m = 0;
  for (int i = 0; i < in.count; ++i) m += ms[i] = in.p[i].m;
  const bool pair = in.stage == QgemmGroup::kSwiGLU;
  const int cols = pair ? 2 * in.width : n;
  auto fill = [&](auto& g) {
    g.count = in.count;
    for (int i = 0; i < in.count; ++i) {
      g.p[i].w = in.p[i].w;
      g.p[i].scales = static_cast<const uint16_t*>(in.p[i].scales);
      g.p[i].biases = static_cast<const uint16_t*>(in.p[i].biases);
      g.p[i].x = static_cast<const uint16_t*>(in.p[i].x);
      g.p[i].m = in.p[i].m;
    }
  };
  BigPlan p = pick_big_plan(ms, in.count, cols, k, cus, group_splits(in.stage) && ws.p, pair);
  if (p.splits > 1 && ws.bytes < (size_t)p.splits * m * cols * sizeof(float))
    p = pick_big_plan(ms, in.count, cols, k, cus, false, pair);
  if (ws.kernels) *ws.kernels += p.splits == 1 ? 1 : 1 + in.count;
  if (in.stage == QgemmGroup::kStore) {
    tile::Group<EpStore<T>> g{};
    fill(g);
    for (int i = 0; i < in.count; ++i) {
      auto* y = static_cast<uint16_t*>(in.p[i].y);
      g.p[i].ep = EpStore<T>{y, n, al16(y) && n % 8 == 0};
    }
    return tile::launch_group<T, EpStore<T>>(p, g, k, n, stream);
  }
  if (pair) {
    tile::Group<EpSwiGLU<T>> g{};
    fill(g);
    for (int i = 0; i < in.count; ++i) {
      auto* y = static_cast<uint16_t*>(in.p[i].y);
      g.p[i].ep = EpSwiGLU<T>{y, in.width, in.width, 0, in.width, 1.0f, 1.0f,
                              al16(y) && in.width % 8 == 0};
    }
    return tile::launch_group<T, EpSwiGLU<T>>(p, g, k, n, stream);
  }
  auto ep = [&](int i) {
    const QgemmGroup::Product& r = in.p[i];
    auto* y = static_cast<float*>(r.y);
    const bool vec = al16(y) && al16(r.residual) && al16(r.gate) && n % 4 == 0;
    return EpGateAdd<T>{y, r.residual, r.gate, n, 1.0f, vec, nullptr};
  };
  if (p.splits == 1) {
    tile::Group<EpGateAdd<T>> g{};
    fill(g);
    for (int i = 0; i < in.count; ++i) g.p[i].ep = ep(i);
    return tile::launch_group<T, EpGateAdd<T>>(p, g, k, n, stream);
  }
  // Partial sums of product i after those of the products before it.
  tile::Group<EpPartial<false>> g{};
  fill(g);
  float* part = ws.p;
  for (int i = 0; i < in.count; ++i) {
    g.p[i].ep = EpPartial<false>{part, n, n, 0, 0};
    part += (size_t)p.splits * ms[i] * n;
  }
  hipError_t e = tile::launch_group<T, EpPartial<false>>(p, g, k, n, stream);
  for (int i = 0; i < in.count && e == hipSuccess; ++i)
    e = tile::launch_sum<T, EpGateAdd<T>>(SplitWs{g.p[i].ep.ws, 0}, p.splits, ms[i], n, n, ep(i),
                                          stream);
  return e;
}

}  // namespace

hipError_t launch_qgemm_group(const QgemmGroup& g, int k, int n, int dtype, hipStream_t stream,
                              SplitWs ws) {
  if (g.count < 1 || g.count > tile::kMaxGroup || k % 256 != 0) return hipErrorInvalidValue;
  int ms[tile::kMaxGroup];
  for (int i = 0; i < g.count; ++i) ms[i] = g.p[i].m;
  if (!group_fits(k, n, ms, g.count)) {  // operands past 32-bit offsets: one after the other
    const SplitWs count_only{nullptr, 0, ws.kernels};
    hipError_t e = hipSuccess;
    for (int i = 0; i < g.count && e == hipSuccess; ++i) {
      const QgemmGroup::Product& p = g.p[i];
      switch (g.stage) {
        case QgemmGroup::kStore:
          e = launch_qgemm(p.w, p.scales, p.biases, p.x, p.y, k, n, p.m, dtype, stream, count_only);
          break;
        case QgemmGroup::kSwiGLU:
          e = launch_qgemm_swiglu(p.w, p.scales, p.biases, p.x, p.y, g.width, k, n, p.m, g.width, 0,
                                  g.width, 1.0f, 1.0f, dtype, stream, count_only);
          break;
        default:
          e = launch_qgemm_gate_add(p.w, p.scales, p.biases, p.x, p.residual, p.gate,
                                    static_cast<float*>(p.y), k, n, p.m, 1.0f, dtype, stream, ws,
                                    nullptr);
      }
    }
    return e;
  }
  switch (dtype) {
    case kBf16: return launch_group_t<kBf16>(g, k, n, stream, ws);
    case kF16: return launch_group_t<kF16>(g, k, n, stream, ws);
    default: return hipErrorInvalidValue;
  }
}

QgemmPlan qgemm_group_plan(QgemmGroup::Stage stage, int k, int n, const int* ms, int count) {
  if (!group_fits(k, n, ms, count)) return QgemmPlan{false, 128, 1, 0, 256};
  int m = 0;
  for (int i = 0; i < count; ++i) m += ms[i];
  const BigPlan p = pick_big_plan(ms, count, n, k, device_cus(), group_splits(stage),
                                  stage == QgemmGroup::kSwiGLU);
  return QgemmPlan{true, 32 * p.mt, p.splits,
                   p.splits > 1 ? (size_t)p.splits * m * n * sizeof(float) : 0, 128 * p.nt};
}

}  // namespace imq
