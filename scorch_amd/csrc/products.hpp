// Which products of a batch the wavefronts of a workgroup take, and the one each lane reads: the index arithmetic of SpGEMM's
// walk over a row's products (spgemm.hip).  Plain arithmetic, constexpr so that the kernels and a host compiler share it
// (tests/test_spgemm_products.py).
#ifndef SCORCH_AMD_PRODUCTS_HPP_
#define SCORCH_AMD_PRODUCTS_HPP_

namespace scorch {

constexpr int kProductLanes = 64;  // a wavefront

// A wavefront's products of a step: [first, last), slot u being those from first + 64 u on, one to a lane.
struct ProductStep {
  int first, last;
  constexpr bool has(int slot) const { return first + slot * kProductLanes < last; }
  // The product that a lane reads for a slot: its own, or the wavefront's last where it has none.  That one and no later: a
  // wavefront knows the entries up to its own last product only (entries_of_products), and the place of a product in B is its
  // number plus a constant of its own entry: with another entry's constant it lies outside that entry's row, and with entries in
  // any order may lie outside of B.
  constexpr int product(int slot, int lane) const {
    const int x = first + slot * kProductLanes + lane;
    return x < last ? x : last - 1;
  }
};

// The `count` products from x on, count > 0, as few slots to each of `waves` wavefronts as hold them all: the last
// wavefronts may be left with none (first >= last).
constexpr ProductStep product_step(int x, int count, int waves, int wave) {
  const int threads = waves * kProductLanes, each = (count + threads - 1) / threads;
  const int first = x + wave * each * kProductLanes, last = first + each * kProductLanes;
  return {first, last < x + count ? last : x + count};
}

}  // namespace scorch

#endif  // SCORCH_AMD_PRODUCTS_HPP_
