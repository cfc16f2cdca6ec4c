// qgemm_plan.hpp -- what qgemm.hip (plans, dispatch) and the translation units
// that hold the tile kernels (qgemm_tile.hpp) share.
#pragma once

#include "epilogue.hpp"
#include "imq_kernels.hpp"

namespace imq {

// Tile height (32 mt rows), width (128 nt columns) and K split of a launch of
// the large-M kernel; split_steps K-steps of 128 per split, an even number (whole
// scale blocks, K rounded up to 256).
struct BigPlan {
  int mt, nt, splits, split_steps;
};

namespace tile {

// The register-staged kernel with output stage ep (any K % 64 == 0).
template <int T, class EP>
hipError_t launch_reg(const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                      const uint16_t* x, const EP& ep, int k, int n, int m, hipStream_t stream);
// The large-M kernel by plan p, with output stage ep or (EpPartial) the
// partial sums of p.splits K ranges.  KT: K % 256 != 0.
template <int T, class EP, bool KT>
hipError_t launch_plan(const BigPlan& p, const uint32_t* w, const uint16_t* scales,
                       const uint16_t* biases, const uint16_t* x, const EP& ep, int k, int n,
                       int m, hipStream_t stream);
// The sum of a split launch's partial sums with output stage ep.
template <int T, class EP>
hipError_t launch_sum(const SplitWs& ws, int splits, int m, int ncols, int ldp, const EP& ep,
                      hipStream_t stream);

// Up to kMaxGroup products of one K, N and output stage for one launch:
// activations of m rows, and the tiles' ids from `first` on (launch_group
// fills first and tiles_m).
constexpr int kMaxGroup = 6;
template <class EP>
struct Product {
  const uint32_t* w;
  const uint16_t* scales;
  const uint16_t* biases;
  const uint16_t* x;
  EP ep;
  int m, tiles_m, first;
};
template <class EP>
struct Group {
  Product<EP> p[kMaxGroup];
  int count;
};
// By plan p: every product's tiles of that size in one grid (K % 256 == 0).
// Built for 128 rows and more, 128 columns at 128, 192 and 256 rows.
template <int T, class EP>
hipError_t launch_group(const BigPlan& p, Group<EP>& g, int k, int n, hipStream_t stream);
constexpr bool group_built(int mt, int nt) { return mt >= 4 && (nt == 2 || mt % 2 == 0); }

// Tiles built for stage EP (mt: 32-row units, nt: 128-column units).
template <int T, class EP, bool KT>
constexpr bool tile_built(int mt, int nt) {
  // A gate/up pair: 256 columns and 128 rows or more; its partial sums any height.
  if (EP::kPair && (nt == 1 || (mt < 4 && !EP::kPartial))) return false;
  // K % 256 != 0: fewer heights (the planner's list is the same).
  if (KT) return nt == 1 ? (mt == 2 || mt == 4) : (mt != 5 && mt != 7);
  return true;
}

}  // namespace tile

}  // namespace imq
