// CSR x CSR -> CSR (SpGEMM) for gfx950, in the usual two phases: a symbolic
// pass that counts the distinct columns of every output row and turns the
// counts into the row pointer, and a numeric pass that fills column indices
// (ascending within a row) and values.  Every structurally reachable column is
// stored, also when its sum happens to be zero -- the reference's rule.
//
// A row of C is the union of the rows of B selected by the row of A.  How a row
// is processed depends on an upper bound of its size, the number of products
// it sums (sum over its entries of the length of the B row they select):
//
//   up to 32 products    a quarter wavefront, hash table of 64 slots in LDS
//   up to 256 products   one wavefront, hash table of up to 512 slots in LDS
//                        (a wavefront takes four consecutive rows: the first kind
//                        all at once, then the second kind one after the other)
//   up to 1024 products  one workgroup, hash table of 2048 slots in LDS
//   up to 4096 products  B of at most 131,072 columns: a bitmap of the columns in LDS
//                        (see below), or, with up to 3,968, a sum to each of them; wider B: one
//                        workgroup, hash table of 8192 slots in LDS
//   more, B of at most 131,072 columns, and the two passes share what they find out
//                        the products sorted by ranges of columns (see "the longest rows by
//                        bins of columns")
//   more, and more than a 128th of all such rows' products
//                        several workgroups (see "rows shared out among workgroups")
//   more                 one workgroup of 1024 threads with a bitmap of the columns
//                        in LDS, 524,288 columns at a time (B of up to 4.2 M
//                        columns is covered in up to eight such ranges, walking the
//                        row's products once more for each); wider B: a bitmap over
//                        all N columns in global memory, one per workgroup of a pool
//
// A bitmap row needs neither hashing nor sorting: one walk over the products
// sets the bits, a prefix sum over the bitmap gives every column its rank in
// the row, and (numeric pass) a second walk adds each product at its column's
// rank.
//
// Hash rows are emitted sorted: the wavefront version ranks every entry by
// counting smaller keys (at most 256 of them), the workgroup version sorts in
// LDS by buckets over the row's column range (a bitonic sort when the columns
// cluster).  Bitmap rows come out sorted by construction.
// Floating-point sums are accumulated with atomics, so their rounding can
// differ from run to run in the last bits; the structure never does, and
// integer results are exact.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "products.hpp"
#include "sync.hpp"

namespace scorch {

constexpr int kTinyProducts = 256;     // wavefront tier (512 slots)
constexpr int kTinySlots = 512;
constexpr int kSmallProducts = 1024;   // workgroup tier 1 (2048 slots)
constexpr int kMediumProducts = 4096;  // workgroup tier 2 (8192 slots)
constexpr int kMediumWorkgroups = 2048;   // where the number of rows is not known
constexpr int kKnownWorkgroups = 65536;
constexpr int kMinHugeWorkgroups = 64;
constexpr int kMaxHugeWorkgroups = 1024;
constexpr size_t kHugeSlabBudget = (size_t)1 << 30;
constexpr int kNarrowColumns = 32 * 4096;              // widest B whose bitmap leaves room for other workgroups in a CU's LDS
constexpr int kLdsBitmapColumns = 8 * 32 * 16384;  // widest B served by the LDS bitmap (in up to 8 ranges of columns)

// Number of bitmap workgroups: as many slabs (N bits and N / 32 ranks) as fit
// the budget, within [kMinHugeWorkgroups, kMaxHugeWorkgroups].
inline int huge_workgroups(int64_t N) {
  const size_t slab = (size_t)(N + 31) / 32 * 8 + 1;
  const size_t fit = kHugeSlabBudget / slab;
  return (int)(fit < (size_t)kMinHugeWorkgroups ? kMinHugeWorkgroups
                                                : (fit > (size_t)kMaxHugeWorkgroups ? kMaxHugeWorkgroups : fit));
}

__device__ __forceinline__ int hash_slot(int key, int mask) {
  return (int)(((unsigned)key * 2654435761u) >> 12) & mask;
}

// Slot of `key` in an open-addressing table (empty = -1); inserts it if absent.
__device__ __forceinline__ int hash_insert(int *keys, int mask, int key, bool &fresh) {
  int s = hash_slot(key, mask);
  for (;;) {
    const int prev = atomicCAS(&keys[s], -1, key);
    fresh = prev == -1;
    if (prev == -1 || prev == key) return s;
    s = (s + 1) & mask;
  }
}

// *addr += v, atomically, in global memory.  Floating-point sums use the hardware's add
// instructions (global_atomic_add_f32 / _f64) rather than a compare-and-swap loop; they are exact
// for ordinary device memory, which is what the workspace must be.
template <typename A>
__device__ __forceinline__ void atomic_accumulate(A *addr, A v) { atomicAdd(addr, v); }
template <>
__device__ __forceinline__ void atomic_accumulate<float>(float *addr, float v) { unsafeAtomicAdd(addr, v); }
template <>
__device__ __forceinline__ void atomic_accumulate<double>(double *addr, double v) { unsafeAtomicAdd(addr, v); }
template <>
__device__ __forceinline__ void atomic_accumulate<uint64_t>(uint64_t *addr, uint64_t v) {
  atomicAdd(reinterpret_cast<unsigned long long *>(addr), (unsigned long long)v);
}

// The same in LDS.  What a CU takes for an instruction of 64 lanes at random addresses, in clocks: reads
// and writes 7, integer or / add 8, compare-and-swap 12, ds_add_f64 21, and ds_add_f32 193, three
// for every lane.  fp32 sums are therefore compare-and-swapped starting
// from the guess that this is the first product of its column, as it mostly is.
template <typename A>
__device__ __forceinline__ void lds_accumulate(A *addr, A v) { atomic_accumulate<A>(addr, v); }
template <>
__device__ __forceinline__ void lds_accumulate<float>(float *addr, float v) {
  unsigned *const bits = reinterpret_cast<unsigned *>(addr);
  for (unsigned seen = 0u;;) {
    const unsigned found = atomicCAS(bits, seen, __builtin_bit_cast(unsigned, __builtin_bit_cast(float, seen) + v));
    if (found == seen) return;
    seen = found;
  }
}

// A workgroup's slab in global memory is private to it: its wavefronts share one
// CU and one L2, so workgroup scope is all the ordering it needs.  (A
// device-scope fence would make the L2 write its dirty lines back, once per
// row and workgroup.)  Read after the atomics of other wavefronts of the
// workgroup, behind a __syncthreads().
template <typename A>
__device__ __forceinline__ A workgroup_load(const A *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <typename A>
__device__ __forceinline__ void workgroup_store(A *p, A v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Prefix sums and maxima over TEAM lanes (16, or the 64 of a wavefront), inclusive: the exchanges are
// carried by the operation itself (DPP: row_shr 1, 2, 4, 8 within rows of 16 lanes, then
// row_bcast 15 and 31 across them).  A shuffle goes through the LDS pipe and is waited for at
// every step.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_or_zero(int x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false);
}
template <int TEAM>
__device__ __forceinline__ int team_inclusive_sum(int x) {
  static_assert(TEAM == 16 || TEAM == kWaveSize, "a row of lanes or a wavefront");
  x += dpp_or_zero<0x111, 0xf>(x);
  x += dpp_or_zero<0x112, 0xf>(x);
  x += dpp_or_zero<0x114, 0xf>(x);
  x += dpp_or_zero<0x118, 0xf>(x);
  if (TEAM == 16) return x;
  x += dpp_or_zero<0x142, 0xa>(x);
  return x + dpp_or_zero<0x143, 0xc>(x);
}
template <int TEAM>  // of numbers from 0 up
__device__ __forceinline__ int team_inclusive_max(int x) {
  static_assert(TEAM == 16 || TEAM == kWaveSize, "a row of lanes or a wavefront");
  x = max(x, dpp_or_zero<0x111, 0xf>(x));
  x = max(x, dpp_or_zero<0x112, 0xf>(x));
  x = max(x, dpp_or_zero<0x114, 0xf>(x));
  x = max(x, dpp_or_zero<0x118, 0xf>(x));
  if (TEAM == 16) return x;
  x = max(x, dpp_or_zero<0x142, 0xa>(x));
  return max(x, dpp_or_zero<0x143, 0xc>(x));
}
// The last lane's value, for every lane of the team.
template <int TEAM>
__device__ __forceinline__ int team_last(int x) {
  if (TEAM == kWaveSize) return __builtin_amdgcn_readlane(x, kWaveSize - 1);
  return __shfl(x, wave_lane() | (TEAM - 1));
}

// Exclusive prefix sum of one int per thread over a workgroup of WAVES
// wavefronts; `total` receives the sum.  `scratch` holds WAVES ints.
template <int WAVES>
__device__ __forceinline__ int block_exclusive_scan_n(int v, int *scratch, int &total) {
  const int lane = wave_lane();
  const int w = threadIdx.x / kWaveSize;
  const int incl = team_inclusive_sum<kWaveSize>(v);
  __syncthreads();  // scratch may still be read from a previous call
  if (lane == kWaveSize - 1) scratch[w] = incl;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    const int part = scratch[i];
    if (i < w) before += part;
    all += part;
  }
  total = all;
  return before + incl - v;
}

__device__ __forceinline__ int block_exclusive_scan(int v, int *scratch, int &total) {
  return block_exclusive_scan_n<kWavesPerBlock>(v, scratch, total);
}

// Exclusive scan of `v` over a workgroup of WAVES wavefronts and, behind the same two
// barriers, the workgroup's minimum of `lo` (from 0 up) and maximum of `hi` (from -1 up).
template <int WAVES>
__device__ __forceinline__ int block_scan_min_max(int v, int &total, int &lo, int &hi, int *scan_scratch,
                                                  int *min_scratch, int *max_scratch) {
  const int lane = wave_lane();
  const int w = threadIdx.x / kWaveSize;
  const int incl = team_inclusive_sum<kWaveSize>(v);
  lo = INT_MAX - team_inclusive_max<kWaveSize>(INT_MAX - lo);
  hi = team_inclusive_max<kWaveSize>(hi + 1) - 1;
  __syncthreads();  // the scratch arrays may still be read from a previous call
  if (lane == kWaveSize - 1) {
    scan_scratch[w] = incl;
    min_scratch[w] = lo;
    max_scratch[w] = hi;
  }
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    const int part = scan_scratch[i];
    if (i < w) before += part;
    all += part;
    lo = i == 0 ? min_scratch[0] : min(lo, min_scratch[i]);
    hi = i == 0 ? max_scratch[0] : max(hi, max_scratch[i]);
  }
  total = all;
  return before + incl - v;
}

// ---- walking the products of one row of C ------------------------------------------------
// The products of a row are the entries of the B rows its A entries select.  B
// rows are often much shorter than a wavefront, so handing one B row to a team
// at a time wastes most lanes and chains three dependent loads per A entry.
// Instead the team (TEAM = 16: a quarter wavefront, 64: one wavefront, 256 or
// 1024: the workgroup) takes
// TEAM entries of A at once -- thread t reads entry t, its B row's start and
// length -- turns the lengths into offsets with a prefix sum, and then walks the
// batch's products flat: product x belongs to the entry e with off[e] <= x <
// off[e + 1].  Teams of up to a wavefront
// mark the first product of every entry that has any and take the running maximum of
// the marks: six vector instructions per product instead of six dependent LDS reads with their
// compares.  The wavefronts of a workgroup take up to 256 products each, mark the first products of
// entries by a bit, and count the bits up to a product's (entries_of_products); entries without products are left
// out of the batch.  All lanes stay busy and consecutive lanes read consecutive entries of a B row.
constexpr int kProductsInFlight = 4;

template <int TEAM, typename A>
struct ProductBatch {  // of the entries that have products, in their order, INT_MAX behind them:
  int first[TEAM];     // first product within the batch
  int start[TEAM];     // where the B row starts, less that
  A a_val[TEAM];
  uint4 begins[TEAM / kWaveSize][2];  // a wavefront's: a bit per product of its step that is an entry's first
};
template <typename A>
struct MarkedBatch {
  int start[kWaveSize];                                 // where entry e's B row starts, less its first product
  A a_val[kWaveSize];
  unsigned mark[kProductsInFlight * kWaveSize / 4];     // a byte per product: the entry it is the first of, or 0
};
template <typename A> struct ProductBatch<kWaveSize, A> : MarkedBatch<A> {};
template <typename A>
struct ProductBatch<16, A> {
  int start[16];
  A a_val[16];
  unsigned mark[kProductsInFlight * 16 / 4];
};

template <int TEAM>
__device__ __forceinline__ int team_exclusive_scan(int v, int &total) {
  const int incl = team_inclusive_sum<TEAM>(v);
  total = team_last<TEAM>(incl);
  return incl - v;
}

// Entries of a batch for a team of wavefronts: thread t's entry has `len` products, its B row starts at `lo`.  Returns
// the number of products.  Two barriers, and one behind which the batch may be read.
template <int TEAM, bool NUMERIC, typename A>
__device__ __forceinline__ int fill_batch(int len, int lo, A av, ProductBatch<TEAM, A> &batch, int *scan_scratch) {
  constexpr int WAVES = TEAM / kWaveSize;
  const int t = threadIdx.x, lane = wave_lane(), w = t / kWaveSize;
  const unsigned long long has = __ballot(len > 0);
  const int incl = team_inclusive_sum<kWaveSize>(len);
  __syncthreads();  // the previous batch has been read by everyone
  if (lane == kWaveSize - 1) {
    scan_scratch[w] = incl;
    batch.begins[w][0].x = (unsigned)__popcll(has);
  }
  __syncthreads();
  int first = incl - len, total = 0, entries = 0;
  int at = __builtin_amdgcn_mbcnt_hi((unsigned)(has >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)has, 0u));
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    if (i == w) first += total, at += entries;
    total += scan_scratch[i];
    entries += (int)batch.begins[i][0].x;
  }
  if (len > 0) {
    batch.first[at] = first;
    batch.start[at] = lo - first;
    if (NUMERIC) batch.a_val[at] = av;
  }
  if (t >= entries) batch.first[t] = INT_MAX;
  __syncthreads();
  return total;
}

// The entries e[u] that the products of a wavefront's step belong to, slot u < U and lane: those of step.product(u, lane), which
// is below the step's end (an entry that begins there or later leaves no bit).  0 <= step.first < step.last.  The entry of the first is looked for by the whole wavefront at once; every entry that begins
// behind it leaves a bit, and an entry's number is the bits up to the product: a third of the LDS reads and half of the vector
// instructions of a bisection for every product.  (131,072 nodes, 16 a row, us: products made and sorted 108 -> 100, rows of up to
// 4,096 products counted 19.6 -> 18.2 and summed 70.3 -> 66.7, of up to 1,024 28.6 -> 26.6 and 79.8 -> 78.2; what is left of the sort
// is the gathers from B and its own writes, 4.4 TB/s.)
template <int TEAM, int U, typename A>
__device__ __forceinline__ void entries_of_products(const ProductStep &step, ProductBatch<TEAM, A> &batch, int (&e)[U]) {
  static_assert(U <= 4 && kProductLanes == kWaveSize, "a bit per product");
  const int xs = step.first, xe = step.last;
  constexpr int S = TEAM / kWaveSize;
  const int lane = wave_lane(), w = uniform((int)threadIdx.x / kWaveSize);
  unsigned *const begins = reinterpret_cast<unsigned *>(batch.begins[w]);
  if (lane < 8) begins[lane] = 0u;
  const int stretch = __popcll(__ballot(batch.first[lane * S] <= xs)) - 1;
  const int e0 = stretch * S + __popcll(__ballot(lane < S && batch.first[stretch * S + lane % S] <= xs)) - 1;
  wave_lds_sync();
  for (int i = e0 + 1 + lane;; i += kWaveSize) {  // (64 of them begin in the step: there may be more)
    const int first = i < TEAM ? batch.first[i] : INT_MAX;
    if (first < xe) atomicOr(&begins[(first - xs) >> 5], 1u << ((first - xs) & 31));
    if (!__all(first < xe)) break;
  }
  wave_lds_sync();
  const uint4 b0 = batch.begins[w][0], b1 = batch.begins[w][1];
  const unsigned words[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
  int before = e0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const unsigned long long m = (unsigned long long)(unsigned)uniform((int)words[2 * u + 1]) << 32 | (unsigned)uniform((int)words[2 * u]);
    const unsigned long long behind = m >> 1;  // bits up to a lane's own: the first, and of these those below it
    e[u] = before + (int)(m & 1u) + __builtin_amdgcn_mbcnt_hi((unsigned)(behind >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)behind, 0u));
    before += __popcll(m);
  }
}

// The same for a team of up to a wavefront, U = kProductsInFlight: `first` and `len` are this lane's entry's
// products, `carried` the last entry that began before the step (its products may go on).
template <int TEAM, bool NUMERIC, typename T, typename A, typename Fn>
__device__ __forceinline__ void marked_step(int x0, int total, int t, int first, int len, int &carried,
                                            const int *__restrict__ b_crd, const T *__restrict__ b_val,
                                            ProductBatch<TEAM, A> &batch, Fn &fn) {
  constexpr int U = kProductsInFlight;
  unsigned char *const marks = reinterpret_cast<unsigned char *>(batch.mark);
  batch.mark[t] = 0u;
  wave_lds_sync();
  // (entries with products start at different ones: no two lanes write one byte)
  if (len > 0 && first >= x0 && first < x0 + U * TEAM) marks[first - x0] = (unsigned char)t;
  wave_lds_sync();
  int e[U], q[U], col[U];
  A b[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u > 0 && x0 + u * TEAM >= total) break;  // uniform over the team
    e[u] = team_inclusive_max<TEAM>(marks[u * TEAM + t]);
    const int last = team_last<TEAM>(e[u]);
    e[u] = max(e[u], carried);
    carried = max(carried, last);
    // (slots beyond the last product read that product again and hand nothing to fn)
    q[u] = min(x0 + u * TEAM + t, total - 1) + batch.start[e[u]];
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u > 0 && x0 + u * TEAM >= total) break;  // uniform over the team
    col[u] = b_crd[q[u]];
    b[u] = NUMERIC ? (A)b_val[q[u]] : (A)0;
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (x0 + u * TEAM + t < total) fn(col[u], NUMERIC ? batch.a_val[e[u]] * b[u] : (A)0);
}

// The columns and products of a wavefront's step, 0 <= step.first < step.last: slot u's are those of step.product(u, lane) if the
// wavefront has any there.
template <int TEAM, bool NUMERIC, typename T, typename A, int U>
__device__ __forceinline__ void products_of_step(const ProductStep &step, const int *__restrict__ b_crd, const T *__restrict__ b_val,
                                                 ProductBatch<TEAM, A> &batch, int (&col)[U], A (&product)[U]) {
  const int lane = wave_lane();
  int e[U], q[U];
  A b[U];
  entries_of_products<TEAM, U, A>(step, batch, e);
#pragma unroll
  for (int u = 0; u < U; ++u) q[u] = step.product(u, lane) + batch.start[e[u]];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u > 0 && !step.has(u)) break;  // uniform over the wavefront
    col[u] = b_crd[q[u]];
    b[u] = NUMERIC ? (A)b_val[q[u]] : (A)0;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u > 0 && !step.has(u)) break;
    product[u] = NUMERIC ? batch.a_val[e[u]] * b[u] : (A)0;
  }
}

// fn(column, product) for every product of A entries [a_lo, a_hi); `t` is the
// thread's number in the team.  Uniform over the team.
template <int TEAM, bool NUMERIC, typename T, typename A, typename Fn>
__device__ __forceinline__ void for_each_product(int a_lo, int a_hi, int t, const int *__restrict__ a_crd,
                                                 const T *__restrict__ a_val, const int *__restrict__ b_pos,
                                                 const int *__restrict__ b_crd, const T *__restrict__ b_val,
                                                 ProductBatch<TEAM, A> &batch, int *scan_scratch, Fn fn) {
  constexpr int U = kProductsInFlight;
  for (int base = a_lo; base < a_hi; base += TEAM) {
    const int p = base + t;
    int lo = 0, len = 0;
    A av = (A)0;
    if (p < a_hi) {
      const int j = a_crd[p];
      lo = b_pos[j];
      len = b_pos[j + 1] - lo;
      if (NUMERIC) av = (A)a_val[p];
    }
    if constexpr (TEAM <= kWaveSize) {
      int total = 0;
      const int first = team_exclusive_scan<TEAM>(len, total);
      wave_lds_sync();  // the previous batch has been read by everyone (LDS operations of a wavefront complete in program order)
      batch.start[t] = lo - first;
      if (NUMERIC) batch.a_val[t] = av;
      int carried = 0;
      for (int x = 0; x < total; x += U * TEAM)
        marked_step<TEAM, NUMERIC, T, A>(x, total, t, first, len, carried, b_crd, b_val, batch, fn);
    } else {
      const int total = fill_batch<TEAM, NUMERIC, A>(len, lo, av, batch, scan_scratch);
      const int lane = wave_lane(), w = uniform(t / kWaveSize);
      for (int x = 0; x < total; x += U * TEAM) {
        const ProductStep step = product_step(x, min(U * TEAM, total - x), TEAM / kWaveSize, w);
        if (step.first >= step.last) break;
        int col[U];
        A product[U];
        products_of_step<TEAM, NUMERIC, T, A>(step, b_crd, b_val, batch, col, product);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (step.first + u * kWaveSize + lane < step.last) fn(col[u], product[u]);
      }
    }
  }
}

// ---- exclusive prefix sum of n ints, in place (counts -> row pointer) ------------------
// Three small kernels: per-tile totals, a one-workgroup scan of the totals, and
// a rescan of every tile from its offset.
constexpr int kScanPerThread = 16;
constexpr int kScanTile = kBlockThreads * kScanPerThread;

// counters: [0] medium rows, [1] huge rows, [2] small rows, [5] giant rows listed; [3], [4] next row to hand out;
// [6] (64 bits) the number of entries of the result; [8] rows shared out, [9] their slices; [10] (64 bits) the giant
// rows' products; [12] (64 bits) the products of all rows beyond kMediumProducts, and [14] their batches of kBinEntries
// entries; [15] workgroups of pass 0 that are through; [16..20] the bins' totals (Bins)
// Every counter has a 128-byte line of its own: atomics on one line follow one another at 12 ns each, whatever
// they address (512 workgroups with eight counts each: 71 us on one line).
constexpr int kSpgemmCounters = 22;
__host__ __device__ constexpr int counter(int i) { return 32 * i; }
constexpr int kBinEntries = 512;

// The symbolic pass is over: the numeric pass hands its longest rows out from the first again, and
// the host thread, if it waits, gets the report (SpgemmReport).
__device__ __forceinline__ void end_of_symbolic(int *counters, unsigned long long entries, int64_t *report, int64_t sequence) {
  if (report) {
    const int64_t words[7] = {entries > (unsigned long long)INT32_MAX ? -1 : (int64_t)entries,
                              counters[counter(2)], counters[counter(0)], counters[counter(1)],
                              counters[counter(5)], counters[counter(8)], counters[counter(9)]};
    sync_publish(report, sequence, words, 7);
  }
  counters[counter(3)] = 0;
}

// A thread's kScanPerThread consecutive elements, four to a request (one at a time, a wavefront's request touches 64 lines
// for 256 bytes: the one-workgroup scan below took 21 us for 21,648 rows and 43 for 45,000); 0 beyond the end.
__device__ __forceinline__ void load_run(const int *data, int64_t first, int64_t n, int (&v)[kScanPerThread]) {
  if (first + kScanPerThread <= n) {
#pragma unroll
    for (int q = 0; q < kScanPerThread / 4; ++q) {
      const Vec<int, 4> x = load_vec<int, 4>(data + first + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * q + e] = x.v[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < kScanPerThread; ++e) v[e] = first + e < n ? data[first + e] : 0;
  }
}
// Their exclusive sums, starting from `running`.
__device__ __forceinline__ void store_run(int *data, int64_t first, int64_t n, int running, const int (&v)[kScanPerThread]) {
  int sums[kScanPerThread];
#pragma unroll
  for (int e = 0; e < kScanPerThread; ++e) {
    sums[e] = running;
    running += v[e];
  }
  if (first + kScanPerThread <= n) {
#pragma unroll
    for (int q = 0; q < kScanPerThread / 4; ++q)
      store_vec<int, 4>(data + first + 4 * q, Vec<int, 4>{{sums[4 * q], sums[4 * q + 1], sums[4 * q + 2], sums[4 * q + 3]}});
  } else {
#pragma unroll
    for (int e = 0; e < kScanPerThread; ++e)
      if (first + e < n) data[first + e] = sums[e];
  }
}

// (*grand_total also receives the sum of all counts in 64 bits: the row pointer is int32,
// and a result of 2^31 entries or more must be reported, not wrapped)
__global__ __launch_bounds__(kBlockThreads) void scan_tile_totals_kernel(const int *__restrict__ data,
                                                                         int64_t n,
                                                                         int *__restrict__ totals,
                                                                         unsigned long long *__restrict__ grand_total) {
  __shared__ int s_scan[kWavesPerBlock + 1];
  const int64_t first = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanPerThread;
  int v[kScanPerThread];
  load_run(data, first, n, v);
  int mine = 0;
  long long wide = 0;
#pragma unroll
  for (int e = 0; e < kScanPerThread; ++e) {
    mine += v[e];
    wide += v[e];
  }
  int total = 0;
  (void)block_exclusive_scan(mine, s_scan, total);
  if (threadIdx.x == 0) totals[blockIdx.x] = total;
#pragma unroll
  for (int off = kWaveSize / 2; off > 0; off >>= 1) wide += __shfl_xor(wide, off);
  if (wave_lane() == 0 && wide > 0) atomicAdd(grand_total, (unsigned long long)wide);
}

// (also, at the end of the symbolic pass: see end_of_symbolic)
__global__ __launch_bounds__(kBlockThreads) void scan_spine_kernel(int *__restrict__ totals,
                                                                   int64_t n_tiles, int *__restrict__ counters,
                                                                   int64_t *__restrict__ report, int64_t sequence) {
  if (threadIdx.x == 0) end_of_symbolic(counters, *reinterpret_cast<const unsigned long long *>(counters + counter(6)), report, sequence);
  __shared__ int s_scan[kWavesPerBlock + 1];
  int carried = 0;
  for (int64_t base = 0; base < n_tiles; base += kBlockThreads) {
    const int64_t i = base + threadIdx.x;
    const int v = i < n_tiles ? totals[i] : 0;
    int total = 0;
    const int before = block_exclusive_scan(v, s_scan, total);
    if (i < n_tiles) totals[i] = carried + before;
    carried += total;
  }
}

// (the last element, the total, becomes -1 when the 64-bit total does not fit an int32)
// SPINE: `totals` has been through scan_spine_kernel; else a workgroup adds up the totals of the tiles before its own,
// and the first one ends the symbolic pass.
constexpr int64_t kScanOwnTotals = 4096;  // most tiles for that
template <bool SPINE>
__global__ __launch_bounds__(kBlockThreads) void scan_apply_kernel(int *__restrict__ data, int64_t n,
                                                                   const int *__restrict__ totals, int *__restrict__ counters,
                                                                   int64_t *__restrict__ report, int64_t sequence) {
  __shared__ int s_scan[kWavesPerBlock + 1];
  const unsigned long long grand_total = *reinterpret_cast<const unsigned long long *>(counters + counter(6));
  if (!SPINE && blockIdx.x == 0 && threadIdx.x == 0) end_of_symbolic(counters, grand_total, report, sequence);
  const int64_t first = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanPerThread;
  int v[kScanPerThread];
  load_run(data, first, n, v);
  int mine = 0, total = 0, before = 0;
#pragma unroll
  for (int e = 0; e < kScanPerThread; ++e) mine += v[e];
  if (SPINE) {
    before = totals[blockIdx.x];
  } else {
    int part = 0;
    for (int i = threadIdx.x; i < (int)blockIdx.x; i += kBlockThreads) part += totals[i];
    (void)block_exclusive_scan(part, s_scan, before);
  }
  const int running = before + block_exclusive_scan(mine, s_scan, total);
  store_run(data, first, n, running, v);
  if (first <= n - 1 && n - 1 < first + kScanPerThread && grand_total > (unsigned long long)INT32_MAX) data[n - 1] = -1;
}

// The same for few rows, in one workgroup and one launch.
constexpr int kScanThreads = 1024;
constexpr int kScanOneGroup = kScanThreads * kScanPerThread;  // one round (more rows: two launches of 4 us)
__global__ __launch_bounds__(kScanThreads) void scan_one_group_kernel(int *__restrict__ data, int n, int *__restrict__ counters,
                                                                      int64_t *__restrict__ report, int64_t sequence) {
  __shared__ int s_scan[kScanThreads / kWaveSize];
  unsigned long long wide = 0;
  const int first = (int)threadIdx.x * kScanPerThread;
  int v[kScanPerThread], mine = 0, total = 0;
  load_run(data, first, n, v);
#pragma unroll
  for (int e = 0; e < kScanPerThread; ++e) {
    mine += v[e];
    wide += (unsigned)v[e];
  }
  store_run(data, first, n, block_exclusive_scan_n<kScanThreads / kWaveSize>(mine, s_scan, total), v);
#pragma unroll
  for (int off = kWaveSize / 2; off > 0; off >>= 1) {
    const unsigned lo = (unsigned)__shfl_xor((int)(unsigned)wide, off), hi = (unsigned)__shfl_xor((int)(unsigned)(wide >> 32), off);
    wide += ((unsigned long long)hi << 32) | lo;
  }
  __shared__ unsigned long long s_wide;
  if (threadIdx.x == 0) s_wide = 0;
  __syncthreads();
  if (wave_lane() == 0) atomicAdd(&s_wide, wide);
  __syncthreads();
  if (threadIdx.x == 0) {
    *reinterpret_cast<unsigned long long *>(counters + counter(6)) = s_wide;
    end_of_symbolic(counters, s_wide, report, sequence);
    if (s_wide > (unsigned long long)INT32_MAX) data[n - 1] = -1;
  }
}

// ---- pass 0: products per row, and the lists of rows too big for a wavefront ----
// A workgroup takes up to kBoundsRows consecutive rows, eight lanes per row; rows
// of A with more than kBoundsLongRow entries are queued in LDS and summed
// afterwards, by a wavefront each or, beyond kBoundsWaveRow entries, by the whole
// workgroup one after the other, so that a hub row does not leave its neighbours'
// lanes waiting on a long dependent chain.  The three row lists are gathered in LDS
// first and appended to the global lists with one atomic per list and
// workgroup: thousands of atomics on one counter would serialise in the L2.
// Rows beyond kMediumProducts products come in two classes: the workgroups that
// take them get them one at a time from a counter, and the longest rows decide
// when that kernel ends, so those of at least kGiantProducts are listed apart
// (from the back of the same array) and handed out first.
constexpr int kGiantProducts = 16384;
constexpr int kBoundsLongRow = 64;
constexpr int kBoundsWaveRow = 2048;
constexpr int kBoundsRows = 256;

// Rows to a workgroup: fewer for matrices that would not fill the chip otherwise
// (their rows tend to be the long ones, which a workgroup takes a few at a time).
inline int bounds_rows_per_group(int64_t M) {
  const int64_t rows = (M / 1024 + 31) / 32 * 32;
  return (int)(rows < 32 ? 32 : rows > kBoundsRows ? kBoundsRows : rows);
}

// Products of entries p, p + stride, ... (N of them, those before hi): all of A's columns are requested before the
// first is used, then all of B's row pointers.
template <int N>
__device__ __forceinline__ long long products_of_entries(int p, int stride, int hi, const int *__restrict__ a_crd,
                                                   const int *__restrict__ b_pos) {
  int j[N];
  long long sum = 0;
#pragma unroll
  for (int u = 0; u < N; ++u) j[u] = a_crd[min(p + u * stride, hi - 1)];
  Vec<int, 2> b[N];
#pragma unroll
  for (int u = 0; u < N; ++u) b[u] = load_vec<int, 2>(b_pos + j[u]);
#pragma unroll
  for (int u = 0; u < N; ++u) sum += p + u * stride < hi ? b[u].v[1] - b[u].v[0] : 0;
  return sum;
}

__global__ __launch_bounds__(kBlockThreads) void spgemm_bounds_kernel(
    int M, int rows_per_group, const int *__restrict__ a_pos, const int *__restrict__ a_crd,
    const int *__restrict__ b_pos, int *__restrict__ products, int *__restrict__ small_rows,
    int *__restrict__ medium_rows, int *__restrict__ huge_rows, int *__restrict__ counters,
    int64_t *__restrict__ report, int64_t sequence) {
  constexpr int G = 8;  // lanes per row
  constexpr int kStep = kBlockThreads / G;
  constexpr int kRowsAtOnce = 4;          // whose loads a lane has in flight together
  __shared__ int s_long[kBoundsRows];
  __shared__ int s_very_long[kBoundsRows];
  __shared__ int s_list[4][kBoundsRows];  // medium, huge, small, giant
  __shared__ int s_n[6];                  // [4], [5]: long and very long rows queued
  __shared__ int s_base[4];
  __shared__ long long s_part[kWavesPerBlock];
  __shared__ unsigned long long s_giant_products, s_big_products;
  __shared__ int s_big_batches;
  if (threadIdx.x < 6) s_n[threadIdx.x] = 0;
  if (threadIdx.x == 0) s_giant_products = s_big_products = 0, s_big_batches = 0;
  __syncthreads();
  auto file_row = [&](int row, long long sum, int entries) {
    const int bound = sum > INT_MAX ? INT_MAX : (int)sum;
    products[row] = bound;
    const int list = bound >= kGiantProducts ? 3 : bound > kMediumProducts ? 1 : bound > kSmallProducts ? 0
                     : bound > kTinyProducts ? 2 : -1;
    if (list >= 0) s_list[list][atomicAdd(&s_n[list], 1)] = row;
    if (list == 3) atomicAdd(&s_giant_products, (unsigned long long)bound);
    if (list & 1 && list > 0) {
      atomicAdd(&s_big_products, (unsigned long long)sum);
      atomicAdd(&s_big_batches, (entries + kBinEntries - 1) / kBinEntries);
    }
  };

  const int t = threadIdx.x % G;
  const int64_t first = (int64_t)blockIdx.x * rows_per_group;
  const int64_t end = min(first + rows_per_group, (int64_t)M);
  for (int64_t base = first + threadIdx.x / G; base < end; base += kRowsAtOnce * kStep) {
    int lo[kRowsAtOnce], hi[kRowsAtOnce], j[kRowsAtOnce][2];
    Vec<int, 2> b[kRowsAtOnce][2];
#pragma unroll
    for (int r = 0; r < kRowsAtOnce; ++r) {
      const int64_t row = min(base + r * kStep, end - 1);
      lo[r] = a_pos[row];
      hi[r] = a_pos[row + 1];
    }
#pragma unroll
    for (int r = 0; r < kRowsAtOnce; ++r)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        j[r][u] = -1;
        if (lo[r] + t + u * G < hi[r]) j[r][u] = a_crd[lo[r] + t + u * G];
      }
#pragma unroll
    for (int r = 0; r < kRowsAtOnce; ++r)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        b[r][u].v[0] = b[r][u].v[1] = 0;
        if (j[r][u] >= 0) b[r][u] = load_vec<int, 2>(b_pos + j[r][u]);
      }
#pragma unroll
    for (int r = 0; r < kRowsAtOnce; ++r) {
      const int64_t row = base + r * kStep;
      if (row >= end) break;
      const int entries = hi[r] - lo[r];
      if (entries > kBoundsLongRow) {
        if (t > 0) continue;
        if (entries > kBoundsWaveRow) s_very_long[atomicAdd(&s_n[5], 1)] = (int)row;
        else s_long[atomicAdd(&s_n[4], 1)] = (int)row;
        continue;
      }
      long long sum = (long long)(b[r][0].v[1] - b[r][0].v[0]) + (b[r][1].v[1] - b[r][1].v[0]);
      for (int p = lo[r] + t + 2 * G; p < hi[r]; p += 4 * G) sum += products_of_entries<4>(p, G, hi[r], a_crd, b_pos);
#pragma unroll
      for (int off = G / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
      if (t == 0) file_row((int)row, sum, entries);
    }
  }
  __syncthreads();

  const int n_long = s_n[4];
  for (int i = threadIdx.x / kWaveSize; i < n_long; i += kWavesPerBlock) {  // uniform over the wavefront
    const int r = s_long[i];
    long long part = 0;
    const int hi = a_pos[r + 1];
    for (int p = a_pos[r] + wave_lane(); p < hi; p += 8 * kWaveSize)
      part += products_of_entries<8>(p, kWaveSize, hi, a_crd, b_pos);
#pragma unroll
    for (int off = kWaveSize / 2; off > 0; off >>= 1) part += __shfl_xor(part, off);
    if (wave_lane() == 0) file_row(r, part, a_pos[r + 1] - a_pos[r]);
  }
  const int n_very_long = s_n[5];
  for (int i = 0; i < n_very_long; ++i) {  // uniform over the workgroup
    const int r = s_very_long[i];
    long long part = 0;
    const int hi = a_pos[r + 1];
    for (int p = a_pos[r] + (int)threadIdx.x; p < hi; p += 16 * kBlockThreads)
      part += products_of_entries<16>(p, kBlockThreads, hi, a_crd, b_pos);
#pragma unroll
    for (int off = kWaveSize / 2; off > 0; off >>= 1) part += __shfl_xor(part, off);
    __syncthreads();
    if (wave_lane() == 0) s_part[threadIdx.x / kWaveSize] = part;
    __syncthreads();
    if (threadIdx.x == 0) {
      long long total = 0;
      for (int w = 0; w < kWavesPerBlock; ++w) total += s_part[w];
      file_row(r, total, a_pos[r + 1] - a_pos[r]);
    }
  }
  __syncthreads();
  if (threadIdx.x < 4 && s_n[threadIdx.x] > 0)
    s_base[threadIdx.x] = atomicAdd(&counters[counter(threadIdx.x < 3 ? threadIdx.x : 5)], s_n[threadIdx.x]);
  if (threadIdx.x == 0 && s_giant_products > 0)
    atomicAdd(reinterpret_cast<unsigned long long *>(counters + counter(10)), s_giant_products);
  if (threadIdx.x == 0 && s_big_batches > 0) {
    atomicAdd(reinterpret_cast<unsigned long long *>(counters + counter(12)), s_big_products);
    atomicAdd(&counters[counter(14)], s_big_batches);
  }
  if (report) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's counts are in memory
  __syncthreads();
  if (report && threadIdx.x == 0 &&  // the last workgroup hands the totals to the host thread
      __hip_atomic_fetch_add(&counters[counter(15)], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1) {
    const auto total = [&](int i) { return __hip_atomic_load(&counters[counter(i)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    const int64_t words[6] = {total(2), total(0), total(1), total(5),
                              (int64_t)__hip_atomic_load(reinterpret_cast<unsigned long long *>(counters + counter(12)),
                                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                              total(14)};
    sync_publish(report, sequence, words, 6);
  }
  int *const lists[3] = {medium_rows, huge_rows, small_rows};
#pragma unroll
  for (int l = 0; l < 3; ++l)
    for (int i = threadIdx.x; i < s_n[l]; i += kBlockThreads) lists[l][s_base[l] + i] = s_list[l][i];
  for (int i = threadIdx.x; i < s_n[3]; i += kBlockThreads) huge_rows[M - 1 - (s_base[3] + i)] = s_list[3][i];
}

// Entry `idx` of the rows beyond kMediumProducts products, the giant ones first.
__device__ __forceinline__ int huge_row(const int *__restrict__ rows, int M, int n_giant, int idx) {
  return idx < n_giant ? rows[M - 1 - idx] : rows[idx - n_giant];
}

// (The bitmaps of the rows that may be shared out start clear)
__global__ __launch_bounds__(kBlockThreads) void spgemm_reset_kernel(int *counters, int *c_pos_last, int64_t clear_words,
                                                                     unsigned *bits) {
  if (blockIdx.x == 0) {
    for (int i = threadIdx.x; i < counter(kSpgemmCounters); i += kBlockThreads) counters[i] = 0;
    if (threadIdx.x == 0 && c_pos_last) *c_pos_last = 0;
  }
  const int64_t stride = (int64_t)gridDim.x * kBlockThreads;
  for (int64_t i = (int64_t)blockIdx.x * kBlockThreads + threadIdx.x; i < clear_words; i += stride) bits[i] = 0u;
}

// ---- rows of at most kMicroProducts products: a quarter wavefront each -----------------
// Most rows of a very sparse product have a few dozen products: a wavefront each
// would mean a wavefront's start-up and its chain of dependent loads (A's row,
// B's row pointers, B's entries) for every such row.  Sixteen lanes do the same
// steps on tables a quarter the size, four rows to a wavefront.  The teams of a
// wavefront take different numbers of steps; all synchronisation is the
// wavefront's own program order, and shuffles and ballots only look at a
// team's own lanes.
constexpr int kMicroTeam = 16;
constexpr int kMicroProducts = 32;
constexpr int kMicroSlots = 64;

// What TEAMS teams keep in LDS for their rows: the hash table (its occupied slots
// are later compacted to the front of the same arrays: less LDS, more wavefronts
// per CU, and these rows are bound by how many are in flight) and the batch of A
// entries being walked.
template <typename A, bool NUMERIC, int TEAM, int TEAMS, int SLOTS, int PRODUCTS>
struct TeamTables {
  alignas(16) int keys[TEAMS][SLOTS];
  alignas(16) A vals[TEAMS][NUMERIC ? SLOTS : 1];
  ProductBatch<TEAM, A> batch[TEAMS];
};

// One row of C by team number `team` of TEAM lanes (a wavefront or an aligned
// part of one; this lane is its number t): hash the row's products, count or
// compact the occupied slots, sort by rank.
// `bound`: the row's products.
// The table is as large as the row asks for, twice its entries (numeric pass: known) or products and
// at least TEAM: most rows of a tier are short, and clearing and going through 512 slots for a
// row of 40 entries cost more than its products.
template <typename T, bool NUMERIC, int TEAM, int TEAMS, int SLOTS, int PRODUCTS>
__device__ __forceinline__ void spgemm_team_row(
    TeamTables<typename Acc<T>::type, NUMERIC, TEAM, TEAMS, SLOTS, PRODUCTS> &lds, int team, int t, int row, int bound,
    const int *__restrict__ a_pos, const int *__restrict__ a_crd, const T *__restrict__ a_val,
    const int *__restrict__ b_pos, const int *__restrict__ b_crd, const T *__restrict__ b_val,
    int *__restrict__ c_pos, int *__restrict__ c_crd, T *__restrict__ c_val) {
  using A = typename Acc<T>::type;
  const int lane = wave_lane();

  const int out = NUMERIC ? c_pos[row] : 0;
  const int n = NUMERIC ? c_pos[row + 1] - out : 0;
  const int most = 2 * (NUMERIC ? n : bound);
  int slots = TEAM;  // uniform over the team
  while (slots < most) slots <<= 1;
  for (int s = 4 * t; s < slots; s += 4 * TEAM) *reinterpret_cast<int4 *>(&lds.keys[team][s]) = make_int4(-1, -1, -1, -1);
  if (NUMERIC) {
    constexpr int kWide = (int)(16 / sizeof(A));
    for (int s = kWide * t; s < slots; s += kWide * TEAM) *reinterpret_cast<uint4 *>(&lds.vals[team][s]) = make_uint4(0u, 0u, 0u, 0u);
  }
  wave_lds_sync();

  int found = 0;

  for_each_product<TEAM, NUMERIC, T, A>(
      a_pos[row], a_pos[row + 1], t, a_crd, a_val, b_pos, b_crd, b_val, lds.batch[team], nullptr,
      [&](int col, A product) {
        bool fresh;
        const int slot = hash_insert(lds.keys[team], slots - 1, col, fresh);
        if (NUMERIC) lds_accumulate<A>(&lds.vals[team][slot], product);
        else found += fresh ? 1 : 0;
      });
  if (!NUMERIC) {
    found = team_inclusive_sum<TEAM>(found);
    if (t == TEAM - 1) c_pos[row] = found;
    return;
  }
  wave_lds_sync();

  // The occupied slots are compacted in place: a step's TEAM slots are read by all
  // lanes before any is written, and entry number `at` never lies beyond the slot it came from.
  int compacted = 0;
  for (int base = 0; base < slots; base += TEAM) {
    const int key = lds.keys[team][base + t];
    const A val = lds.vals[team][base + t];
    unsigned long long occupied = __ballot(key != -1) >> (lane - t);  // the team's lanes from bit 0
    if (TEAM < kWaveSize) occupied &= (1ull << (TEAM % kWaveSize)) - 1ull;
    wave_lds_sync();  // everyone has read this step's slots
    if (key != -1) {
      const int at = compacted + __popcll(occupied & ((1ull << t) - 1ull));
      lds.keys[team][at] = key;
      lds.vals[team][at] = val;
    }
    compacted += __popcll(occupied);
  }
  wave_lds_sync();

  // Whole wavefronts with more than a key per lane sort by buckets: counting
  // ranks below costs n compares per key, half of this tier's time at 256 keys a
  // row.  The keys' range is cut into 2 * TEAM equal power-of-two intervals; a
  // prefix sum of the bucket counts (kept where the batch's indices were) places
  // the buckets, the entries are scattered bucket by bucket into the tables'
  // upper halves (free: n <= PRODUCTS <= SLOTS / 2), and an entry's rank is
  // its bucket's start plus the smaller keys in its bucket.  Crowded buckets
  // (clustered columns) leave the row to the rank count.
  if (TEAM == kWaveSize && 2 * PRODUCTS <= SLOTS && n > TEAM) {
    constexpr int kBuckets = 2 * TEAM;
    constexpr int kPerLane = PRODUCTS / TEAM;
    constexpr int kCrowd = 16;
    static_assert(TEAM < kWaveSize || sizeof(lds.batch[team]) >= kBuckets * sizeof(int), "the counts lie where the batch was");
    int *const cnt = reinterpret_cast<int *>(&lds.batch[team]);
    int key[kPerLane], pos[kPerLane];
    int key_min = INT_MAX, key_max = -1;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      const int e = t + i * TEAM;
      key[i] = e < n ? lds.keys[team][e] : -1;
      if (e < n) {
        key_min = key[i] < key_min ? key[i] : key_min;
        key_max = key[i] > key_max ? key[i] : key_max;
      }
    }
    key_min = INT_MAX - team_last<TEAM>(team_inclusive_max<TEAM>(INT_MAX - key_min));
    key_max = team_last<TEAM>(team_inclusive_max<TEAM>(key_max));  // (every lane has a key)
    int shift = 0;
    while (((key_max - key_min) >> shift) >= kBuckets) ++shift;
    cnt[t] = 0;
    cnt[TEAM + t] = 0;
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < kPerLane; ++i)
      if (t + i * TEAM < n) pos[i] = atomicAdd(&cnt[(key[i] - key_min) >> shift], 1);
    wave_lds_sync();
    const int c0 = cnt[2 * t], c1 = cnt[2 * t + 1];  // lane t places buckets 2t and 2t + 1
    int unused = 0;
    const int before = team_exclusive_scan<TEAM>(c0 + c1, unused);
    int crowd = c0 > c1 ? c0 : c1;
    crowd = team_last<TEAM>(team_inclusive_max<TEAM>(crowd));
    if (crowd <= kCrowd) {  // uniform
      wave_lds_sync();  // everyone has read the counts
      cnt[2 * t] = before;
      cnt[2 * t + 1] = before + c0;
      wave_lds_sync();
#pragma unroll
      for (int i = 0; i < kPerLane; ++i) {
        const int e = t + i * TEAM;
        if (e < n) {
          const int p = PRODUCTS + cnt[(key[i] - key_min) >> shift] + pos[i];
          lds.keys[team][p] = key[i];
          lds.vals[team][p] = lds.vals[team][e];
        }
      }
      wave_lds_sync();
#pragma unroll
      for (int i = 0; i < kPerLane; ++i) {
        const int e = t + i * TEAM;
        if (e < n) {
          const int k = lds.keys[team][PRODUCTS + e];
          const int b = (k - key_min) >> shift;
          const int lo = cnt[b], hi = b + 1 < kBuckets ? cnt[b + 1] : n;
          int rank = lo;
          for (int x = lo; x < hi; ++x) rank += lds.keys[team][PRODUCTS + x] < k ? 1 : 0;
          c_crd[out + rank] = k;
          c_val[out + rank] = (T)lds.vals[team][PRODUCTS + e];
        }
      }
      return;
    }
  }

  // Rank = number of smaller keys (keys are distinct): the sorted position.  Four keys to a read, the
  // last ones padded (n is at most half of the table's slots, or a multiple of four).
  if (t < (-n & 3)) lds.keys[team][n + t] = INT_MAX;
  wave_lds_sync();
  const int4 *const fours = reinterpret_cast<const int4 *>(lds.keys[team]);
  for (int e = t; e < n; e += TEAM) {
    const int key = lds.keys[team][e];
    int rank = 0;
    for (int x = 0; 4 * x < n; ++x) {
      const int4 k = fours[x];
      rank += (k.x < key ? 1 : 0) + (k.y < key ? 1 : 0) + (k.z < key ? 1 : 0) + (k.w < key ? 1 : 0);
    }
    c_crd[out + rank] = key;
    c_val[out + rank] = (T)lds.vals[team][e];
  }
}

// A wavefront takes four consecutive rows: those of at most kMicroProducts
// products by its four quarters at once, then those of up to kTinyProducts one
// after the other with all its lanes (rows beyond that belong to the workgroup
// kernels).  The two kinds of table share the wavefront's LDS.
// (One row per wavefront, for matrices of too few rows to fill the chip four to a wavefront, is
// spgemm_small_matrix_kernel's.)
// One wavefront to a workgroup: rows differ, and of four wavefronts that share a workgroup's LDS the first three wait for the
// last with theirs taken (131,072 nodes, 16 a row: numeric 86 -> 75 us, symbolic 40.7 -> 38.6).
constexpr int kTinyThreads = kWaveSize;
template <typename T, bool NUMERIC>
__global__ __launch_bounds__(kTinyThreads) void spgemm_tiny_kernel(
    int M, const int *__restrict__ a_pos, const int *__restrict__ a_crd, const T *__restrict__ a_val,
    const int *__restrict__ b_pos, const int *__restrict__ b_crd, const T *__restrict__ b_val,
    const int *__restrict__ products, int *__restrict__ c_pos, int *__restrict__ c_crd,
    T *__restrict__ c_val) {
  using A = typename Acc<T>::type;
  constexpr int kQuarters = kWaveSize / kMicroTeam;
  union Tables {
    TeamTables<A, NUMERIC, kWaveSize, 1, kTinySlots, kTinyProducts> wave;
    TeamTables<A, NUMERIC, kMicroTeam, kQuarters, kMicroSlots, kMicroProducts> quarter;
  };
  __shared__ Tables lds[kTinyThreads / kWaveSize];
  const int lane = wave_lane();
  const int w = threadIdx.x / kWaveSize;
  // (the grid is a multiple of 8 workgroups: neighbouring rows, which may well select the same
  // rows of B, go to one XCD)
  const int64_t first = (xcd_contiguous(blockIdx.x, gridDim.x) * (kTinyThreads / kWaveSize) + w) * kQuarters;
  if (first >= M) return;
  const int q = lane / kMicroTeam;
  const int64_t mine = first + q;
  const int bound = mine < M ? products[mine] : INT_MAX;
  if (bound <= kMicroProducts)
    spgemm_team_row<T, NUMERIC, kMicroTeam, kQuarters, kMicroSlots, kMicroProducts>(
        lds[w].quarter, q, lane % kMicroTeam, (int)mine, bound, a_pos, a_crd, a_val, b_pos, b_crd, b_val, c_pos, c_crd,
        c_val);
#pragma unroll
  for (int i = 0; i < kQuarters; ++i) {
    const int b = __shfl(bound, i * kMicroTeam);  // uniform
    if (b > kMicroProducts && b <= kTinyProducts) {
      wave_lds_sync();  // the tables' previous users are done
      spgemm_team_row<T, NUMERIC, kWaveSize, 1, kTinySlots, kTinyProducts>(
          lds[w].wave, 0, lane, (int)(first + i), b, a_pos, a_crd, a_val, b_pos, b_crd, b_val, c_pos, c_crd, c_val);
    }
  }
}

// ---- rows of at most PRODUCTS products: one workgroup each, 2 * PRODUCTS hash slots ----
// THREADS: workgroup size (the tables of the larger form leave room for one workgroup per
// CU: it is given 1024 threads rather than 256).
template <typename A, bool NUMERIC, int PRODUCTS, int THREADS>
struct MediumTables {
  A vals[NUMERIC ? 2 * PRODUCTS : 1];
  union {
    ProductBatch<THREADS, A> batch;
    int cnt[NUMERIC ? PRODUCTS / 2 : 1];  // of the buckets, once the products have been walked
  };
  int keys[2 * PRODUCTS];
  int scan[(THREADS / kWaveSize) + 1];
  int red[2][(THREADS / kWaveSize)];
};

// The rows `block`, block + n_blocks, ... of the list.
template <typename T, bool NUMERIC, int PRODUCTS, int COUNTER, int THREADS>
__device__ __forceinline__ void spgemm_medium_rows(
    MediumTables<typename Acc<T>::type, NUMERIC, PRODUCTS, THREADS> &lds, int block, int n_blocks,
    const int *__restrict__ a_pos, const int *__restrict__ a_crd, const T *__restrict__ a_val,
    const int *__restrict__ b_pos, const int *__restrict__ b_crd, const T *__restrict__ b_val,
    const int *__restrict__ products, const int *__restrict__ rows, const int *__restrict__ counters,
    int *__restrict__ c_pos, int *__restrict__ c_crd, T *__restrict__ c_val) {
  using A = typename Acc<T>::type;
  constexpr int kBuckets = PRODUCTS / 2;
  constexpr int kBucketCrowd = 32;  // a fuller bucket sends the row to the bitonic sort
  auto &s_keys = lds.keys;
  auto &s_vals = lds.vals;
  auto &s_ck = lds.keys;  // (sorted in place: the table's slots pass through registers)
  auto &s_cv = lds.vals;
  auto &s_scan = lds.scan;
  auto &s_red = lds.red;
  auto &s_cnt = lds.cnt;
  auto &s_batch = lds.batch;

  const int tid = threadIdx.x;
  const int n_rows = counters[counter(COUNTER)];

  // (A workgroup to each row where the host knows how many there are: 131,072 nodes, 16 a row, 8,900 such rows 65 -> 52 us
  // against strides of 2,048 workgroups, of which some end long before others.  Handed out one at a time through a counter
  // they measured slower: these rows are short enough for the counter's round trip to show.)
  for (int idx = block; idx < n_rows; idx += n_blocks) {
    const int row = rows[idx];
    const int out = NUMERIC ? c_pos[row] : 0;
    const int most = 2 * (NUMERIC ? c_pos[row + 1] - out : products[row]);
    int slots = THREADS;  // a table as large as the row asks for; uniform
    while (slots < most) slots <<= 1;
    for (int s = tid; s < slots; s += THREADS) {
      s_keys[s] = -1;
      if (NUMERIC) s_vals[s] = (A)0;
    }
    __syncthreads();

    int found = 0;
    for_each_product<THREADS, NUMERIC, T, A>(
        a_pos[row], a_pos[row + 1], tid, a_crd, a_val, b_pos, b_crd, b_val, s_batch, s_scan,
        [&](int col, A product) {
          bool fresh;
          const int slot = hash_insert(s_keys, slots - 1, col, fresh);
          if (NUMERIC) lds_accumulate<A>(&s_vals[slot], product);
          else found += fresh ? 1 : 0;
        });
    if (!NUMERIC) {
      int n = 0;
      (void)block_exclusive_scan_n<THREADS / kWaveSize>(found, s_scan, n);
      if (tid == 0) c_pos[row] = n;
      continue;  // (the scan's barriers have everyone past the table)
    }
    __syncthreads();

    // Each thread takes `run` slots into registers, a workgroup's width apart (neighbouring threads
    // on neighbouring LDS banks); an exclusive scan of the per-thread counts
    // places the occupied ones.  The table is free then, and the row is sorted in its place: 19.6 KB of LDS
    // instead of 29.9, eight workgroups to a CU instead of five (8,900 rows of 256 to 1,024 products: 76 -> 65 us).
    constexpr int kRun = 2 * PRODUCTS / THREADS;
    const int run = slots / THREADS;
    int key[kRun], pos[kRun];
    A val[kRun];
    int mine = 0, key_min = INT_MAX, key_max = -1;
#pragma unroll
    for (int s = 0; s < kRun; ++s) {
      key[s] = -1;
      if (s >= run) continue;  // uniform
      key[s] = s_keys[s * THREADS + tid];
      val[s] = s_vals[s * THREADS + tid];
      if (key[s] != -1) {
        ++mine;
        key_min = key[s] < key_min ? key[s] : key_min;
        key_max = key[s] > key_max ? key[s] : key_max;
      }
    }
    for (int bkt = tid; bkt < kBuckets; bkt += THREADS) s_cnt[bkt] = 0;
    int n = 0;
    int at = block_scan_min_max<THREADS / kWaveSize>(mine, n, key_min, key_max, s_scan, s_red[0], s_red[1]);

    // Sorting the row's (column, value) pairs.  First choice: buckets.  The
    // columns' range [min, max] is cut into kBuckets equal power-of-two intervals
    // (about two entries each when the columns are spread evenly), a prefix sum of
    // the bucket counts places the buckets, the entries are scattered bucket by
    // bucket, and an entry's rank is its bucket's start plus the smaller keys in
    // its bucket.  If some bucket is crowded (clustered columns), a bitonic sort
    // of the whole row takes over.
    int shift = 0;
    while (((key_max - key_min) >> shift) >= kBuckets) ++shift;  // n > 0 here: the row has products
#pragma unroll
    for (int s = 0; s < kRun; ++s)
      if (key[s] != -1) pos[s] = atomicAdd(&s_cnt[(key[s] - key_min) >> shift], 1);
    __syncthreads();
    constexpr int kBucketRun = kBuckets / THREADS;
    int run_total = 0, crowd = 0;
    for (int i = 0; i < kBucketRun; ++i) {
      const int c = s_cnt[tid * kBucketRun + i];
      run_total += c;
      crowd = c > crowd ? c : crowd;
    }
    int unused = 0, unused_min = 0;
    int start = block_scan_min_max<THREADS / kWaveSize>(run_total, unused, unused_min, crowd, s_scan, s_red[0], s_red[1]);
    if (crowd <= kBucketCrowd) {
      for (int i = 0; i < kBucketRun; ++i) {  // counts -> first positions
        const int c = s_cnt[tid * kBucketRun + i];
        s_cnt[tid * kBucketRun + i] = start;
        start += c;
      }
      __syncthreads();
#pragma unroll
      for (int s = 0; s < kRun; ++s)
        if (key[s] != -1) {
          const int p = s_cnt[(key[s] - key_min) >> shift] + pos[s];
          s_ck[p] = key[s];
          s_cv[p] = val[s];
        }
      __syncthreads();
      for (int e = tid; e < n; e += THREADS) {
        const int k = s_ck[e];
        const int bkt = (k - key_min) >> shift;
        const int lo = s_cnt[bkt], hi = bkt + 1 < kBuckets ? s_cnt[bkt + 1] : n;
        int rank = lo;
        for (int x = lo; x < hi; ++x) rank += s_ck[x] < k ? 1 : 0;
        c_crd[out + rank] = k;
        c_val[out + rank] = (T)s_cv[e];
      }
      __syncthreads();
      continue;
    } else {
#pragma unroll
      for (int s = 0; s < kRun; ++s)
        if (key[s] != -1) {
          s_ck[at] = key[s];
          s_cv[at] = val[s];
          ++at;
        }
      int padded = 1;
      while (padded < n) padded <<= 1;
      __syncthreads();
      for (int e = n + tid; e < padded; e += THREADS) s_ck[e] = INT_MAX;
      __syncthreads();
      for (int size = 2; size <= padded; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
          for (int e = tid; e < padded / 2; e += THREADS) {
            const int lo = 2 * e - (e & (stride - 1));
            const int hi = lo + stride;
            const bool ascending = (lo & size) == 0;
            const int klo = s_ck[lo], khi = s_ck[hi];
            if ((klo > khi) == ascending) {
              s_ck[lo] = khi;
              s_ck[hi] = klo;
              const A v = s_cv[lo];
              s_cv[lo] = s_cv[hi];
              s_cv[hi] = v;
            }
          }
          __syncthreads();
        }
      }
    }
    for (int e = tid; e < n; e += THREADS) {
      c_crd[out + e] = s_ck[e];
      c_val[out + e] = (T)s_cv[e];
    }
    __syncthreads();
  }
}

template <typename T, bool NUMERIC, int PRODUCTS, int COUNTER, int THREADS>
__global__ __launch_bounds__(THREADS) void spgemm_medium_kernel(
    const int *__restrict__ a_pos, const int *__restrict__ a_crd, const T *__restrict__ a_val,
    const int *__restrict__ b_pos, const int *__restrict__ b_crd, const T *__restrict__ b_val,
    const int *__restrict__ products, const int *__restrict__ rows, const int *__restrict__ counters,
    int *__restrict__ c_pos, int *__restrict__ c_crd, T *__restrict__ c_val) {
  __shared__ MediumTables<typename Acc<T>::type, NUMERIC, PRODUCTS, THREADS> lds;
  spgemm_medium_rows<T, NUMERIC, PRODUCTS, COUNTER, THREADS>(lds, blockIdx.x, gridDim.x, a_pos, a_crd, a_val, b_pos,
                                                             b_crd, b_val, products, rows, counters, c_pos, c_crd, c_val);
}

// ---- rows beyond that: a bitmap over all columns -------------------------------------------
// Workgroups of 1024 threads: such a row has tens of thousands of products and
// is one workgroup's alone, so its width is the row's parallelism.  The
// symbolic pass sets a bit per product and counts the bits.  The numeric pass
// walks the products twice: first for the bits again, from which it writes the
// row's column indices (ascending by construction), zeroes the row's values and
// notes the rank of every bitmap word's first column; then for the values, each
// product adding itself to the row's output at rank(word) + (bits below its own)
// -- no accumulator over all N columns, whose lines would go through the L2 once
// per product.
constexpr int kHugeThreads = 1024;
constexpr int kHugeWaves = kHugeThreads / kWaveSize;
constexpr int kHugeEmitWords = 256;  // bitmap words emitted per step (at most 8192 columns)

template <typename T, bool NUMERIC>
__global__ __launch_bounds__(kHugeThreads) void spgemm_huge_kernel(
    int M, int N, const int *__restrict__ a_pos, const int *__restrict__ a_crd, const T *__restrict__ a_val,
    const int *__restrict__ b_pos, const int *__restrict__ b_crd, const T *__restrict__ b_val,
    const int *__restrict__ rows, const int *__restrict__ counters, unsigned *__restrict__ bitmaps,
    int *__restrict__ ranks, int *__restrict__ c_pos, int *__restrict__ c_crd, T *__restrict__ c_val) {
  using A = typename Acc<T>::type;
  __shared__ int s_scan[kHugeWaves];
  __shared__ ProductBatch<kHugeThreads, A> s_batch;
  __shared__ int s_cols[NUMERIC ? kHugeEmitWords * 32 : 1];
  const int tid = threadIdx.x;
  const int n_giant = counters[counter(5)];
  const int n_rows = counters[counter(1)] + n_giant;
  if ((int)blockIdx.x >= n_rows) return;

  const int words = (N + 31) / 32;
  unsigned *bitmap = bitmaps + (size_t)blockIdx.x * (size_t)words;
  int *rank = NUMERIC ? ranks + (size_t)blockIdx.x * (size_t)words : nullptr;
  A *acc = reinterpret_cast<A *>(c_val);  // sums wrap (integers) or round (floating point) as T's do
  // This workgroup's bitmap starts clean and is left clean after every row.
  for (int i = tid; i < words; i += kHugeThreads) workgroup_store(&bitmap[i], 0u);
  __syncthreads();

  for (int idx = blockIdx.x; idx < n_rows; idx += gridDim.x) {
    const int row = huge_row(rows, M, n_giant, idx);
    const int a_lo = a_pos[row], a_hi = a_pos[row + 1];
    for_each_product<kHugeThreads, false, T, A>(
        a_lo, a_hi, tid, a_crd, a_val, b_pos, b_crd, b_val, s_batch, s_scan, [&](int k, A) {
          __hip_atomic_fetch_or(&bitmap[k >> 5], 1u << (k & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        });
    __syncthreads();

    if (!NUMERIC) {
      // count the set bits and clear them
      int mine = 0;
      for (int word = tid; word < words; word += kHugeThreads) {
        const unsigned bits = workgroup_load(&bitmap[word]);
        if (bits) {
          mine += __popc(bits);
          workgroup_store(&bitmap[word], 0u);
        }
      }
      int total = 0;
      block_exclusive_scan_n<kHugeWaves>(mine, s_scan, total);
      if (tid == 0) c_pos[row] = total;
    } else {
      // The bitmap in order, kHugeEmitWords words at a time: the set bits of a step
      // are listed in LDS, then written as column indices, coalesced.
      const int out = c_pos[row];
      int emitted = 0;
      for (int base = 0; base < words; base += kHugeEmitWords) {
        const int word = base + tid;
        const bool mine = tid < kHugeEmitWords && word < words;
        unsigned bits = mine ? workgroup_load(&bitmap[word]) : 0u;
        int total = 0;
        int at = block_exclusive_scan_n<kHugeWaves>(__popc(bits), s_scan, total);
        if (mine) workgroup_store(&rank[word], emitted + at);
        while (bits) {
          const int bit = __ffs(bits) - 1;
          bits &= bits - 1;
          s_cols[at++] = word * 32 + bit;
        }
        __syncthreads();
        for (int e = tid; e < total; e += kHugeThreads) {
          c_crd[out + emitted + e] = s_cols[e];
          workgroup_store(&acc[out + emitted + e], (A)0);
        }
        emitted += total;
        // the next step's scan starts with a barrier, which also protects s_cols
      }
      __syncthreads();
      for_each_product<kHugeThreads, true, T, A>(
          a_lo, a_hi, tid, a_crd, a_val, b_pos, b_crd, b_val, s_batch, s_scan, [&](int k, A product) {
            const unsigned bits = workgroup_load(&bitmap[k >> 5]);
            const int at = out + workgroup_load(&rank[k >> 5]) + __popc(bits & ((1u << (k & 31)) - 1u));
            __hip_atomic_fetch_add(&acc[at], product, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          });
      __syncthreads();
      for (int word = tid; word < words; word += kHugeThreads)
        if (workgroup_load(&bitmap[word])) workgroup_store(&bitmap[word], 0u);
    }
    __syncthreads();
  }
}

// ---- the same tier when the bitmap fits LDS ---------------------------------------------------
// Atomics on a bitmap in global memory all land on a few hundred cache lines and
// queue up in the L2's atomic units (the 13.7 M products of a power-law square
// spend 0.4 ms there per walk).  For N up to 32 * WORDS columns the bitmap lives
// in LDS instead, with one rank per four bitmap words, and so do the sums of the
// row's first kAccEntries output entries (the others are added into the output
// with global atomics as above).
constexpr int kLdsBudget = 160 * 1024 - 1024;
// The numeric pass of the tier of up to kMediumProducts products: with 16-bit ranks, and sums of the last hundred of the longest rows
// in the output, four workgroups of eight wavefronts fill a CU (256 threads, four of four, 2,600 rows: 67 us, 512 60).  The symbolic
// pass has neither ranks nor sums in LDS and needs no larger workgroups to fill a CU: kBlockThreads (512: 19.2 us, 256 18.1).
constexpr int kBitmapThreads = 512, kBitmapSums = 3968;

// THREADS: workgroup size.  ACC: LDS sums to provide (0: all the LDS that is left).
// LIST, WORK: which of the counters holds the length of `rows` and the next row to hand out.
template <typename A, bool NUMERIC, int WORDS, int THREADS, int ACC>
struct BitmapTables {
  static constexpr int kGroups = WORDS / 4;
  using Rank = std::conditional_t<(ACC > 0), unsigned short, int>;  // (ACC: of rows with at most kMediumProducts columns)
  static constexpr int kFixed = WORDS * 4 + (NUMERIC ? kGroups * (int)sizeof(Rank) : 0) + (int)sizeof(ProductBatch<THREADS, A>) + 512;
  static constexpr int kAccEntries = !NUMERIC ? 1 : ACC > 0 ? ACC : (kLdsBudget - kFixed) / (int)sizeof(A);
  alignas(16) unsigned bits[WORDS];
  Rank rank[NUMERIC ? kGroups : 1];  // rank of the first column of every group of four words
  A acc[kAccEntries];
  ProductBatch<THREADS, A> batch;
  int scan[THREADS / kWaveSize];
  int next;
};

// Block number `block` of n_blocks.  `narrow_rows`: the list of the tier above (its length in counter 1), whose rows
// of at most kMediumProducts distinct columns -- known in the numeric pass -- are taken here as well; null: none.
template <typename T, bool NUMERIC, int WORDS, int THREADS, int ACC, int LIST, int WORK>
__device__ __forceinline__ void spgemm_lds_bitmap_rows(
    BitmapTables<typename Acc<T>::type, NUMERIC, WORDS, THREADS, ACC> &lds, int block, int n_blocks,
    int M, int N, const int *__restrict__ a_pos, const int *__restrict__ a_crd, const T *__restrict__ a_val,
    const int *__restrict__ b_pos, const int *__restrict__ b_crd, const T *__restrict__ b_val,
    const int *__restrict__ rows, const int *__restrict__ narrow_rows, int *__restrict__ counters,
    int *__restrict__ c_pos, int *__restrict__ c_crd, T *__restrict__ c_val) {
  using A = typename Acc<T>::type;
  using Tables = BitmapTables<A, NUMERIC, WORDS, THREADS, ACC>;
  constexpr int kAccEntries = Tables::kAccEntries;
  constexpr int kWaves = THREADS / kWaveSize;
  constexpr bool kByColumn = NUMERIC && ACC > 0 && 32 * WORDS <= ACC, kHolds = NUMERIC && ACC > 0 && !kByColumn;
  auto &s_bits = lds.bits;
  auto &s_rank = lds.rank;
  auto &s_acc = lds.acc;
  auto &s_batch = lds.batch;
  auto &s_scan = lds.scan;
  int &s_next = lds.next;
  const int tid = threadIdx.x;
  const int n_giant = LIST == 1 ? counters[counter(5)] : 0;  // only the list of the longest rows has the class
  const int n_own = counters[counter(LIST)] + n_giant;
  const int n_rows = n_own + (narrow_rows ? counters[counter(1)] : 0);
  if (block >= n_rows) return;  // more workgroups than rows: no need to queue at the counter
  constexpr int kRangeColumns = 32 * WORDS;
  A *acc = reinterpret_cast<A *>(c_val);
  // B with no more columns than the LDS holds sums: the numeric pass keeps a sum
  // per column and walks the row's products once (bits and sums together)
  // instead of twice (bits, then sums at their ranks).  The tier of up to kMediumProducts products has kernels of its own for it
  // (kByColumn), with a bitmap for as many columns and no registers for held products: fp32 40,000 x 3,000, rows of 2,000 products
  // 832 -> 715 us, 8,000 x 1,000, 1,600 182 -> 139; fp64 1,102 -> 772, 286 -> 153.
  const bool sums_by_column = ACC > 0 ? kByColumn : NUMERIC && N <= kAccEntries && N <= kRangeColumns;

  // The longest rows are handed out through a counter, one at a time, so that the
  // workgroups stay evenly loaded; the rows of the tier below are short enough
  // for the counter's round trip to show, and are taken in fixed strides.
  for (int turn = 0;; ++turn) {
    __syncthreads();  // everyone is done with the previous row (and with s_next)
    int idx;
    if (LIST == 1) {
      if (tid == 0) s_next = atomicAdd(&counters[counter(WORK)], 1);
      __syncthreads();
      idx = s_next;
    } else {
      idx = block + turn * n_blocks;
    }
    if (idx >= n_rows) return;  // the same for every thread
    int row;
    if (LIST == 1) {
      row = huge_row(rows, M, n_giant, idx);
      if (row < 0) continue;  // shared out among workgroups
      // (of few distinct columns: the tier below's, whose smaller workgroups share a compute unit)
      if (NUMERIC && N <= kNarrowColumns && idx >= n_giant && c_pos[row + 1] - c_pos[row] <= kMediumProducts) continue;
    } else if (idx < n_own) {
      row = rows[idx];
    } else {
      row = narrow_rows[idx - n_own];
      if (c_pos[row + 1] - c_pos[row] > kMediumProducts) continue;
    }
    const int a_lo = a_pos[row], a_hi = a_pos[row + 1];
    const int out = NUMERIC ? c_pos[row] : 0;
    int done = 0;  // distinct columns found in the ranges before this one

    // Rows of as many products as the threads hold in registers are walked once (131,072 nodes, 16 a row, 2,600 rows: 60 -> 52 us).
    constexpr int U = kProductsInFlight, kSteps = kHolds ? kMediumProducts / (U * THREADS) : 1;
    static_assert(!kHolds || (kSteps * U * THREADS == kMediumProducts && WORDS * 32 >= kNarrowColumns), "all products of a row of one range");
    int col[kSteps][U];
    A product[kSteps][U];
    ProductStep steps[kSteps] = {};
    bool held = kHolds && a_hi - a_lo <= THREADS;
    if constexpr (kHolds) {
      if (held) {  // uniform
        int start = 0, len = 0;
        A av = (A)0;
        if (a_lo + tid < a_hi) {
          const int j = a_crd[a_lo + tid];
          start = b_pos[j];
          len = b_pos[j + 1] - start;
          av = (A)a_val[a_lo + tid];
        }
        const int total = fill_batch<THREADS, true, A>(len, start, av, s_batch, s_scan);
        held = total <= kMediumProducts;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
          const int x = s * U * THREADS;
          if (!held || x >= total) break;
          steps[s] = product_step(x, min(U * THREADS, total - x), kWaves, uniform(tid / kWaveSize));
          if (steps[s].first < steps[s].last) products_of_step<THREADS, true, T, A>(steps[s], b_crd, b_val, s_batch, col[s], product[s]);
        }
      }
    }

    // B wider than the bitmap: one range of kRangeColumns columns after the other,
    // walking the row's products again for each (ranges ascend, so the row comes
    // out sorted all the same)
    for (int c0 = 0; c0 < N; c0 += kRangeColumns) {
      const int columns = N - c0 < kRangeColumns ? N - c0 : kRangeColumns;
      const int groups = ((columns + 31) / 32 + 3) / 4;
      if (c0 > 0) __syncthreads();  // the previous range's bits, ranks and sums have been used
      for (int i = tid; i < 4 * groups; i += THREADS) s_bits[i] = 0u;
      if (sums_by_column)
        for (int i = tid; i < columns; i += THREADS) s_acc[i] = (A)0;
      __syncthreads();
      if (sums_by_column) {
        for_each_product<THREADS, true, T, A>(
            a_lo, a_hi, tid, a_crd, a_val, b_pos, b_crd, b_val, s_batch, s_scan, [&](int k, A product) {
              if ((unsigned)k >= (unsigned)columns) return;
              atomicOr(&s_bits[k >> 5], 1u << (k & 31));
              lds_accumulate<A>(&s_acc[k], product);
            });
      } else if (held) {
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
#pragma unroll
          for (int u = 0; u < U; ++u) {  // (a column outside of B is left out, as by the walk and by `add` below)
            const unsigned rel = (unsigned)col[s][u];
            if (steps[s].first + u * kWaveSize + wave_lane() < steps[s].last && rel < (unsigned)columns)
              atomicOr(&s_bits[rel >> 5], 1u << (rel & 31));
          }
      } else {
        for_each_product<THREADS, false, T, A>(
            a_lo, a_hi, tid, a_crd, a_val, b_pos, b_crd, b_val, s_batch, s_scan, [&](int k, A) {
              const unsigned rel = (unsigned)(k - c0);
              if (rel < (unsigned)columns) atomicOr(&s_bits[rel >> 5], 1u << (rel & 31));
            });
#pragma unroll
        for (int s = 0; s < kSteps; ++s)  // (nothing is held: no registers for it during the walk)
#pragma unroll
          for (int u = 0; u < U; ++u) col[s][u] = 0, product[s][u] = (A)0;
      }
      __syncthreads();

      // distinct columns of the range, and the rank of each group's first one
      int n = 0;
      for (int base = 0; base < groups; base += THREADS) {
        const int g = base + tid;
        int cnt = 0;
        if (g < groups)
          cnt = __popc(s_bits[4 * g]) + __popc(s_bits[4 * g + 1]) + __popc(s_bits[4 * g + 2]) +
                __popc(s_bits[4 * g + 3]);
        int total = 0;
        const int at = block_exclusive_scan_n<kWaves>(cnt, s_scan, total);
        if (NUMERIC && g < groups) s_rank[g] = (typename Tables::Rank)(n + at);
        n += total;
      }
      if (NUMERIC && n > 0) {  // uniform
        const int first = out + done;  // the range's place in the row's output
        // The first kAccEntries output entries have their sums, and before that their
        // column indices, in LDS; entries beyond go straight to the output: a
        // thread's columns lie far apart there (single 4-byte stores), and sums added
        // with global atomics queue up in the L2's atomic units.
        const int in_lds = n < kAccEntries ? n : kAccEntries;
        __syncthreads();  // s_rank is complete
        for (int g = tid; g < groups; g += THREADS) {
          int at = s_rank[g];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            unsigned bits = s_bits[4 * g + i];
            while (bits) {
              const int bit = __ffs(bits) - 1;
              bits &= bits - 1;
              const int col = c0 + (4 * g + i) * 32 + bit;
              c_crd[first + at] = col;
              if (sums_by_column) c_val[first + at] = (T)s_acc[col];
              ++at;
            }
          }
        }
        if (sums_by_column) break;  // uniform; the only range: the row is complete
        for (int e = in_lds + tid; e < n; e += THREADS) workgroup_store(&acc[first + e], (A)0);
        for (int e = tid; e < in_lds; e += THREADS) s_acc[e] = (A)0;
        __syncthreads();
        const auto add = [&](int k, A product) {
          const unsigned rel = (unsigned)(k - c0);
          if (rel >= (unsigned)columns) return;
          // rank = the group's + the bits below the column's in the group's four words,
          // which come in one read (a loop over the words before the column's
          // would chain up to three more LDS round trips)
          const int w = (int)(rel >> 5), sub = w & 3;
          const uint4 grp = *reinterpret_cast<const uint4 *>(&s_bits[w & ~3]);
          const unsigned below = (1u << (rel & 31)) - 1u;
          const int at = s_rank[w >> 2] + __popc(grp.x & (sub == 0 ? below : ~0u)) +
                         __popc(grp.y & (sub == 1 ? below : sub > 1 ? ~0u : 0u)) +
                         __popc(grp.z & (sub == 2 ? below : sub > 2 ? ~0u : 0u)) +
                         __popc(grp.w & (sub == 3 ? below : 0u));
          if (at < kAccEntries) lds_accumulate<A>(&s_acc[at], product);
          else __hip_atomic_fetch_add(&acc[first + at], product, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        if (held) {
#pragma unroll
          for (int s = 0; s < kSteps; ++s)
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (steps[s].first + u * kWaveSize + wave_lane() < steps[s].last) add(col[s][u], product[s][u]);
        } else {
          for_each_product<THREADS, true, T, A>(a_lo, a_hi, tid, a_crd, a_val, b_pos, b_crd, b_val, s_batch, s_scan, add);
        }
        __syncthreads();
        for (int e = tid; e < in_lds; e += THREADS) c_val[first + e] = (T)s_acc[e];
      }
      done += n;
    }
    if (!NUMERIC && tid == 0) c_pos[row] = done;
  }
}

template <typename T, bool NUMERIC, int WORDS, int THREADS, int ACC, int LIST, int WORK>
__global__ __launch_bounds__(THREADS) void spgemm_lds_bitmap_kernel(
    int M, int N, const int *__restrict__ a_pos, const int *__restrict__ a_crd, const T *__restrict__ a_val,
    const int *__restrict__ b_pos, const int *__restrict__ b_crd, const T *__restrict__ b_val,
    const int *__restrict__ rows, const int *__restrict__ narrow_rows, int *__restrict__ counters,
    int *__restrict__ c_pos, int *__restrict__ c_crd, T *__restrict__ c_val) {
  __shared__ BitmapTables<typename Acc<T>::type, NUMERIC, WORDS, THREADS, ACC> lds;
  spgemm_lds_bitmap_rows<T, NUMERIC, WORDS, THREADS, ACC, LIST, WORK>(lds, blockIdx.x, gridDim.x, M, N, a_pos, a_crd,
                                                                      a_val, b_pos, b_crd, b_val, rows, narrow_rows,
                                                                      counters, c_pos, c_crd, c_val);
}

// ---- a matrix of few rows: the three kinds of work in one launch --------------------------------
// Below 32,768 rows the tiers' kernels are short and what a product costs is launches, 3 to 5 us
// each: workgroups [0, n_bitmap) take bitmap rows, the next n_medium hash rows of up to
// kSmallProducts products, the rest a row of up to kTinyProducts to each wavefront, the longest kinds first.
// The kinds share the workgroup's LDS (40 KB with fp32 sums, four workgroups to a CU).
// THREADS: symbolic 256.  Numeric with sums of 8 bytes, whose tables take the LDS, 512: with 256 half of a CU's wavefronts find no room.
// With sums of 4 bytes 512 for the rows of up to kTinyProducts, and 256 where more than half of the rows have more products (a
// workgroup's barriers are what these wait for).  The product, us, all with 256 and so, M x N with rows of (products): fp32 30,000 x 30,000
// (100) 99, 91; fp64 (100) 135, 104; (400) 474, 439; (2,000) 681, 609; all with 512 and so: fp32 30,000 x 30,000 (400) 376, 296;
// (1,000) 465, 388; (2,000) 515, 455; 8,000 x 3,000 (400) 120, 88.  Graphs of 1,500 nodes of 16 and 25,000 of 10, fp32: 96 and 135 with 256, 92 and 128 so.
template <typename T, bool NUMERIC, int THREADS, int WORDS>
__global__ __launch_bounds__(THREADS) void spgemm_small_matrix_kernel(
    int M, int N, int n_bitmap, int n_medium, const int *__restrict__ a_pos, const int *__restrict__ a_crd,
    const T *__restrict__ a_val, const int *__restrict__ b_pos, const int *__restrict__ b_crd,
    const T *__restrict__ b_val, const int *__restrict__ products, const int *__restrict__ small_rows,
    const int *__restrict__ medium_rows, const int *__restrict__ narrow_rows, int *__restrict__ counters,
    int *__restrict__ c_pos, int *__restrict__ c_crd, T *__restrict__ c_val) {
  using A = typename Acc<T>::type;
  constexpr int kWaves = THREADS / kWaveSize;
  union Tables {
    BitmapTables<A, NUMERIC, WORDS, THREADS, kBitmapSums> bitmap;
    MediumTables<A, NUMERIC, kSmallProducts, THREADS> medium;
    TeamTables<A, NUMERIC, kWaveSize, kWaves, kTinySlots, kTinyProducts> tiny;
  };
  __shared__ Tables lds;
  int block = blockIdx.x;
  if (block < n_bitmap) {
    spgemm_lds_bitmap_rows<T, NUMERIC, WORDS, THREADS, kBitmapSums, 0, 4>(
        lds.bitmap, block, n_bitmap, M, N, a_pos, a_crd, a_val, b_pos, b_crd, b_val, medium_rows, narrow_rows, counters,
        c_pos, c_crd, c_val);
    return;
  }
  block -= n_bitmap;
  if (block < n_medium) {
    spgemm_medium_rows<T, NUMERIC, kSmallProducts, 2, THREADS>(lds.medium, block, n_medium, a_pos, a_crd, a_val, b_pos, b_crd, b_val,
                                                               products, small_rows, counters, c_pos, c_crd, c_val);
    return;
  }
  block -= n_medium;
  const int w = threadIdx.x / kWaveSize;
  const int row = block * kWaves + w;
  const int bound = row < M ? products[row] : INT_MAX;
  if (bound > kTinyProducts) return;
  spgemm_team_row<T, NUMERIC, kWaveSize, kWaves, kTinySlots, kTinyProducts>(
      lds.tiny, w, wave_lane(), row, bound, a_pos, a_crd, a_val, b_pos, b_crd, b_val, c_pos, c_crd, c_val);
}

// ---- rows shared out among workgroups --------------------------------------------------------
// A row is one workgroup's in every tier above, so a tier ends when its longest row does: a hub of
// 50,000 entries in a graph of 131,072 nodes has 850,000 products, 0.31 ms of the symbolic pass
// and 1.25 ms of the numeric one on one CU (its 131,000 sums mostly miss the LDS), while the other
// rows of the tier take a tenth of that on the whole chip.  A giant row with more than a 128th of
// the giant rows' products -- twice a CU's share -- and at least kSplitProducts goes out in slices
// of its A entries instead.  A slice ORs a bitmap of its columns, kept in LDS, into the row's
// bitmap in memory, and adds its products to one sum per column there with device-wide
// atomics: the row's columns are many and its products spread over them, so no address is
// contended (a row with few distinct columns is not in this class: the numeric pass files it
// below).  A pass over bitmap and sums then writes the row.  At most `pool` rows; where more
// qualify there are enough rows to keep the chip busy and the rest stay one workgroup's.
constexpr int kSplitProducts = 32768;
constexpr int kSplitSliceProducts = 8192;   // aimed at: a row of p products gets p / 8192 slices, at most 64
constexpr int kSplitMaxSlices = 64;
constexpr int kSplitMaxRows = 64;
constexpr int kSplitMaxColumns = 32 * 16384;  // the slice's bitmap is in LDS
constexpr int kSplitMinColumns = 4096;        // a narrower B: a hub row has few products, and its sums fit the LDS
constexpr size_t kSplitBudget = (size_t)64 << 20;

inline int split_pool(int64_t N) {
  if (N < kSplitMinColumns || N > kSplitMaxColumns) return 0;
  const size_t fit = kSplitBudget / ((size_t)N * 8);
  return (int)(fit < kSplitMaxRows ? fit : kSplitMaxRows);
}

// split_rows[slot] = row; items[i] = (slot, slice, slices, 0).  One workgroup.
__global__ __launch_bounds__(kBlockThreads) void spgemm_split_select_kernel(
    int M, int pool, const int *__restrict__ a_pos, const int *__restrict__ products, int *__restrict__ huge_rows,
    int *__restrict__ counters, int *__restrict__ split_rows, int4 *__restrict__ items) {
  __shared__ int s_rows, s_items;
  if (threadIdx.x == 0) s_rows = s_items = 0;
  __syncthreads();
  const int n_giant = counters[counter(5)];
  const unsigned long long share = *reinterpret_cast<const unsigned long long *>(counters + counter(10)) / 128;
  for (int i = threadIdx.x; i < n_giant; i += kBlockThreads) {
    const int row = huge_rows[M - 1 - i];
    const int p = products[row];
    if (p < kSplitProducts || (unsigned long long)p < share) continue;
    const int slot = atomicAdd(&s_rows, 1);
    if (slot >= pool) continue;
    huge_rows[M - 1 - i] = -1;
    split_rows[slot] = row;
    const int entries = a_pos[row + 1] - a_pos[row];
    int slices = p / kSplitSliceProducts;
    slices = slices > kSplitMaxSlices ? kSplitMaxSlices : slices;
    slices = slices > entries ? entries : slices;
    const int at = atomicAdd(&s_items, slices);  // at most pool * kSplitMaxSlices in all
    for (int j = 0; j < slices; ++j) items[at + j] = make_int4(slot, j, slices, 0);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    counters[counter(8)] = s_rows < pool ? s_rows : pool;
    counters[counter(9)] = s_items;
  }
}

template <typename A>
__global__ __launch_bounds__(kBlockThreads) void spgemm_split_clear_kernel(int N, const int *__restrict__ counters,
                                                                           A *__restrict__ sums) {
  const int64_t n = (int64_t)counters[counter(8)] * N, stride = (int64_t)gridDim.x * kBlockThreads;
  for (int64_t i = (int64_t)blockIdx.x * kBlockThreads + threadIdx.x; i < n; i += stride) sums[i] = (A)0;
}

// A slice's A entries.
__device__ __forceinline__ void split_slice(const int4 &item, const int *a_pos, int row, int &from, int &to) {
  const int lo = a_pos[row], entries = a_pos[row + 1] - lo;
  from = lo + (int)((int64_t)entries * item.y / item.z);
  to = lo + (int)((int64_t)entries * (item.y + 1) / item.z);
}

template <int WORDS>
__global__ __launch_bounds__(kHugeThreads) void spgemm_split_columns_kernel(
    int words, const int *__restrict__ a_pos, const int *__restrict__ a_crd, const int *__restrict__ b_pos,
    const int *__restrict__ b_crd, const int *__restrict__ counters, const int *__restrict__ split_rows,
    const int4 *__restrict__ items, unsigned *__restrict__ bits) {
  __shared__ unsigned s_bits[WORDS];
  __shared__ ProductBatch<kHugeThreads, float> s_batch;
  __shared__ int s_scan[kHugeWaves];
  const int tid = threadIdx.x;
  const int n_items = counters[counter(9)];
  for (int i = blockIdx.x; i < n_items; i += gridDim.x) {  // uniform
    const int4 item = items[i];
    int from, to;
    split_slice(item, a_pos, split_rows[item.x], from, to);
    for (int w = tid; w < words; w += kHugeThreads) s_bits[w] = 0u;
    __syncthreads();
    for_each_product<kHugeThreads, false, float, float>(from, to, tid, a_crd, nullptr, b_pos, b_crd, nullptr, s_batch, s_scan,
                                                        [&](int k, float) { atomicOr(&s_bits[k >> 5], 1u << (k & 31)); });
    __syncthreads();
    unsigned *row_bits = bits + (size_t)item.x * (size_t)words;
    for (int w = tid; w < words; w += kHugeThreads)
      if (s_bits[w]) atomicOr(&row_bits[w], s_bits[w]);
    __syncthreads();
  }
}

template <typename T>
__global__ __launch_bounds__(kHugeThreads) void spgemm_split_sums_kernel(
    int N, const int *__restrict__ a_pos, const int *__restrict__ a_crd, const T *__restrict__ a_val,
    const int *__restrict__ b_pos, const int *__restrict__ b_crd, const T *__restrict__ b_val,
    const int *__restrict__ counters, const int *__restrict__ split_rows, const int4 *__restrict__ items,
    typename Acc<T>::type *__restrict__ sums) {
  using A = typename Acc<T>::type;
  __shared__ ProductBatch<kHugeThreads, A> s_batch;
  __shared__ int s_scan[kHugeWaves];
  const int n_items = counters[counter(9)];
  for (int i = blockIdx.x; i < n_items; i += gridDim.x) {  // uniform
    const int4 item = items[i];
    int from, to;
    split_slice(item, a_pos, split_rows[item.x], from, to);
    A *row_sums = sums + (size_t)item.x * (size_t)N;
    for_each_product<kHugeThreads, true, T, A>(from, to, threadIdx.x, a_crd, a_val, b_pos, b_crd, b_val, s_batch, s_scan,
                                               [&](int k, A product) { atomic_accumulate<A>(&row_sums[k], product); });
  }
}

struct SplitCount {
  const int *rows;
  const unsigned *bits;
  int words;
};
__global__ __launch_bounds__(kBlockThreads) void spgemm_split_count_kernel(const int *__restrict__ counters, SplitCount split,
                                                                           int *__restrict__ c_pos) {
  __shared__ int s_scan[kWavesPerBlock];
  const int slot = blockIdx.x;
  if (slot >= counters[counter(8)]) return;
  int mine = 0, total = 0;
  for (int w = threadIdx.x; w < split.words; w += kBlockThreads) mine += __popc(split.bits[(size_t)slot * split.words + w]);
  (void)block_exclusive_scan(mine, s_scan, total);
  if (threadIdx.x == 0) c_pos[split.rows[slot]] = total;
}

// Writes the shared-out rows.  grid: (pieces of kEmitWords bitmap words, rows).
constexpr int kEmitWords = 1024;
template <typename T>
__global__ __launch_bounds__(kHugeThreads) void spgemm_split_emit_kernel(
    int N, int words, const int *__restrict__ counters, const int *__restrict__ split_rows,
    const unsigned *__restrict__ bits, const typename Acc<T>::type *__restrict__ sums, const int *__restrict__ c_pos,
    int *__restrict__ c_crd, T *__restrict__ c_val) {
  __shared__ unsigned s_bits[kEmitWords];
  __shared__ int s_rank[kEmitWords];
  __shared__ int s_scan[kHugeWaves];
  const int slot = blockIdx.y;
  if (slot >= counters[counter(8)]) return;
  const int tid = threadIdx.x, lane = wave_lane();
  const unsigned *row_bits = bits + (size_t)slot * (size_t)words;
  const int first = (int)blockIdx.x * kEmitWords;
  int mine = 0, before = 0;
  for (int w = tid; w < first; w += kHugeThreads) mine += __popc(row_bits[w]);
  (void)block_exclusive_scan_n<kHugeWaves>(mine, s_scan, before);
  const unsigned word = first + tid < words ? row_bits[first + tid] : 0u;
  int unused = 0;
  s_rank[tid] = block_exclusive_scan_n<kHugeWaves>(__popc(word), s_scan, unused);
  s_bits[tid] = word;
  __syncthreads();
  const size_t out = (size_t)c_pos[split_rows[slot]] + before;
  const typename Acc<T>::type *row_sums = sums + (size_t)slot * (size_t)N;
  // two bitmap words, 64 columns, per wavefront and step: sums are read and entries written coalesced
  for (int w = 2 * (tid / kWaveSize); w < kEmitWords; w += 2 * kHugeWaves) {
    const int mine_at = w + (lane >> 5), bit = lane & 31;
    const unsigned b = s_bits[mine_at];
    if ((b >> bit) & 1u) {
      const int col = (first + mine_at) * 32 + bit;
      const size_t at = out + s_rank[mine_at] + __popc(b & ((1u << bit) - 1u));
      c_crd[at] = col;
      c_val[at] = (T)row_sums[col];
    }
  }
}

// ---- the longest rows by bins of columns -------------------------------------------------------
// One sum per column of a row beyond kMediumProducts does not fit LDS (131,072 columns), so the kernels
// above walk such a row twice, first for its columns, and a hub's sums are added up in memory (20
// products a nanosecond, however many workgroups do it).  Here the products are made once and
// sorted by ranges of columns: a workgroup turns 2,048 products at a time into runs of equal
// range in LDS and writes them out (a window: 16 bits of column within the range and the value each, 6
// bytes in fp32).  The columns of one range of one row are then counted, and later its sums added up
// in LDS, by a workgroup that reads its runs from all of the row's windows: streams instead of
// gathers, as many workgroups to a row as it has ranges, and a hub shared out by itself.
// Both passes over these rows of a power-law graph squared (131,072 nodes, 16 entries a row, 19 M
// products of this kind), fp32: 240 us (lists 17, sort 80, count 34, sums 111); the numeric pass alone took 512.  The sort is
// bound by the gathers from B (a line for about two entries), the sums by a workgroup's chain of reads.  (Ranges
// without the windows, each item bisecting the rows of B for its piece, fetch those lines once
// per range: 411 us for the numeric pass alone.)
// For products of up to kNarrowColumns columns whose two passes share what they find out.
constexpr int kBinThreads = kBinEntries;
constexpr int kBinProducts = 4 * kBinThreads;  // to a window
constexpr int kBinShare = 4 * kBinProducts;    // products of a batch of entries to a workgroup, where there are many
constexpr int64_t kBinManyProducts = (int64_t)512 * kBinShare;
constexpr int kBinColumns = 8192;              // most columns to a range; a power of two
constexpr int kMaxBins = 32;
constexpr int kHubProducts = 4 * kGiantProducts;
static_assert(kMaxBins * kBinColumns >= kNarrowColumns, "the widest B in ranges of the most columns");
constexpr int64_t kBinBudget = (int64_t)4 << 30;

struct BinWindow {
  int first;                            // its products in `columns` and `values`
  unsigned short at[kMaxBins + 2];      // where its runs begin
};
struct BinRow {
  int row, batches, first_window, first_product, first_item, items;
};
struct BinItem {
  int row, batch, share, shares;  // of the batch's windows this one takes those from `share` on, `shares` apart
};

struct Bins {
  int shift = 0, n = 0;                 // ranges of 2^shift columns, n of them; n 0: not used
  int giant = 0;                        // rows of kGiantProducts products and more: they come first, the longest of them before the others
  int counted_wide = 0;                 // the first rows, whose ranges are counted by a workgroup each, the others' by a wavefront
  int share = kBinShare;                // products of a batch of entries to a workgroup
  int64_t rows = 0, items = 0;
  int *totals;                          // products, windows, items and places handed out to rows so far (counters of pass 0)
  BinRow *row;
  unsigned long long *used;             // per row: windows (upper half) and products written
  BinItem *item;
  BinWindow *window;
  int *counts;                          // [row][n]: distinct columns
  unsigned short *columns;
  void *values;
  size_t total = 0;
};

inline Bins spgemm_bins(char *base, int *counters, int64_t N, size_t elem, int64_t rows, int64_t giant, int64_t products,
                        int64_t batches) {
  Bins b;
  if (rows == 0 || N > kNarrowColumns || products * (int64_t)(2 + elem) > kBinBudget || products > INT32_MAX / 2) return b;
  // Narrow ranges while that makes workgroups the chip has room for, of 512 products and more (45,000 nodes of 11, ranges of
  // 2,048 columns instead of 4,096: sums 29 -> 22 us, counts 21 -> 17; 131,072 nodes of 4, 49 such rows of few
  // products, 4,096 instead of 8,192: 9 -> 12; of 17, 1,074 such rows: 117 -> 186).
  b.shift = 10;
  const auto ranges = [&](int shift) { return rows * ((N + (1 << shift) - 1) >> shift); };
  while ((2 << b.shift) <= kBinColumns &&
         ((kMaxBins << b.shift) < N || ranges(b.shift) > 4096 || ranges(b.shift) * 512 > products))
    ++b.shift;
  b.n = (int)((N + (1 << b.shift) - 1) >> b.shift);
  b.rows = rows;
  b.giant = (int)giant;
  // (Where workgroups for all of them fit the chip, a wavefront's chain is the longer one: 2,500 to 9,800 nodes, the whole product 82 -> 86 us.)
  b.counted_wide = (int)(rows * b.n <= 2048 ? rows : giant);
  // (21,648 rows of 7: 120 workgroups that make four windows one after the other 18 us, of one window each 8.4)
  if (products < kBinManyProducts) b.share = kBinProducts;
  b.items = batches + products / b.share;
  size_t off = 0;
  auto take = [&](size_t bytes) { char *p = base ? base + off : nullptr; off += (bytes + 255) / 256 * 256; return p; };
  b.totals = counters ? counters + counter(16) : nullptr;
  b.row = reinterpret_cast<BinRow *>(take((size_t)rows * sizeof(BinRow)));
  b.used = reinterpret_cast<unsigned long long *>(take((size_t)rows * 8));
  b.item = reinterpret_cast<BinItem *>(take((size_t)b.items * sizeof(BinItem)));
  b.window = reinterpret_cast<BinWindow *>(take((size_t)(products / kBinProducts + batches) * sizeof(BinWindow)));
  b.counts = reinterpret_cast<int *>(take((size_t)(rows * b.n) * 4));
  b.columns = reinterpret_cast<unsigned short *>(take((size_t)products * 2));
  b.values = take((size_t)products * elem);
  b.total = off;
  return b;
}

// Places for the rows' products, windows and work items.
__global__ __launch_bounds__(kBlockThreads) void spgemm_bin_rows_kernel(int M, Bins bins, const int *__restrict__ a_pos,
                                                                        const int *__restrict__ products,
                                                                        const int *__restrict__ huge_rows,
                                                                        const int *__restrict__ counters,
                                                                        int *__restrict__ c_pos) {
  constexpr int kWants = 4;
  __shared__ int s_scan[kWavesPerBlock], s_base[kWants + 1];
  const int64_t i = (int64_t)blockIdx.x * kBlockThreads + threadIdx.x;
  const bool mine = i < bins.rows;
  BinRow r = {};
  int p = 0;
  if (mine) {
    r.row = huge_row(huge_rows, M, counters[counter(5)], (int)i);
    p = products[r.row];
    r.batches = (a_pos[r.row + 1] - a_pos[r.row] + kBinEntries - 1) / kBinEntries;
    r.items = r.batches + p / bins.share;  // at most
  }
  // A workgroup takes a range of a row, and the longest rows decide when the counts and sums end: they go first.
  const bool hub = p >= kHubProducts, giant = i < bins.giant && mine;
  const int want[kWants] = {p, mine ? p / kBinProducts + r.batches : 0, r.items, hub ? 1 << 16 : giant ? 1 : 0};
  int at[kWants];
#pragma unroll
  for (int k = 0; k < kWants; ++k) {
    int total = 0;
    at[k] = block_exclusive_scan(want[k], s_scan, total);
    if (threadIdx.x == (unsigned)k && k < 3) s_base[k] = atomicAdd(bins.totals + counter(k), total);
    if (k == 3 && threadIdx.x == 3) s_base[3] = total >> 16 ? atomicAdd(bins.totals + counter(3), total >> 16) : 0;
    if (k == 3 && threadIdx.x == 4) s_base[4] = total & 0xffff ? atomicAdd(bins.totals + counter(4), total & 0xffff) : 0;
  }
  __syncthreads();
  if (!mine) return;
  r.first_product = s_base[0] + at[0];
  r.first_window = s_base[1] + at[1];
  r.first_item = s_base[2] + at[2];
  const int64_t place = hub ? s_base[3] + (at[3] >> 16) : giant ? bins.giant - 1 - (s_base[4] + (at[3] & 0xffff)) : i;
  bins.row[place] = r;
  bins.used[place] = 0;
  c_pos[r.row] = 0;
}

// A row's work items: a wavefront to a batch of entries.
constexpr int kBinItemThreads = 1024;  // (a row of 50,000 entries is what the launch waits for)
__global__ __launch_bounds__(kBinItemThreads) void spgemm_bin_items_kernel(Bins bins, const int *__restrict__ a_pos,
                                                                           const int *__restrict__ a_crd,
                                                                           const int *__restrict__ b_pos) {
  constexpr int kPer = kBinEntries / kWaveSize;
  __shared__ int s_items;
  if (threadIdx.x == 0) s_items = 0;
  __syncthreads();
  const int lane = wave_lane();
  const BinRow r = bins.row[blockIdx.x];
  const int lo = a_pos[r.row], hi = a_pos[r.row + 1];
  int next[kPer];  // columns of the batch to come
  auto request = [&](int batch) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int p = lo + batch * kBinEntries + i * kWaveSize + lane;
      next[i] = p < hi ? a_crd[p] : -1;
    }
  };
  constexpr int kBatchWaves = kBinItemThreads / kWaveSize;
  int batch = threadIdx.x / kWaveSize;
  if (batch < r.batches) request(batch);
  for (; batch < r.batches; batch += kBatchWaves) {
    Vec<int, 2> b[kPer];
    int total = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      b[i].v[0] = b[i].v[1] = 0;
      if (next[i] >= 0) b[i] = load_vec<int, 2>(b_pos + next[i]);
    }
    if (batch + kBatchWaves < r.batches) request(batch + kBatchWaves);
#pragma unroll
    for (int i = 0; i < kPer; ++i) total += b[i].v[1] - b[i].v[0];
#pragma unroll
    for (int off = kWaveSize / 2; off > 0; off >>= 1) total += __shfl_xor(total, off);
    const int shares = 1 + total / bins.share;
    int first = 0;
    if (lane == 0) first = atomicAdd(&s_items, shares);
    first = r.first_item + uniform(first);
    for (int j = lane; j < shares; j += kWaveSize) bins.item[first + j] = {(int)blockIdx.x, batch, j, shares};
  }
  __syncthreads();
  for (int j = s_items + (int)threadIdx.x; j < r.items; j += kBinItemThreads) bins.item[r.first_item + j] = {0, 0, 0, 0};  // none
}

template <typename T>
__global__ __launch_bounds__(kBinThreads) void spgemm_bin_kernel(
    Bins bins, const int *__restrict__ a_pos, const int *__restrict__ a_crd, const T *__restrict__ a_val,
    const int *__restrict__ b_pos, const int *__restrict__ b_crd, const T *__restrict__ b_val) {
  using A = typename Acc<T>::type;
  constexpr int U = kBinProducts / kBinThreads;
  __shared__ ProductBatch<kBinEntries, A> s_batch;
  __shared__ A s_value[kBinProducts];
  __shared__ unsigned short s_column[kBinProducts];
  __shared__ int s_scan[kBinThreads / kWaveSize], s_count[kMaxBins + 1], s_at[kMaxBins + 1], s_first, s_window;
  if ((int)blockIdx.x >= bins.totals[counter(2)]) return;
  const int tid = threadIdx.x;
  const BinItem item = bins.item[blockIdx.x];
  if (item.shares == 0) return;
  const BinRow r = bins.row[item.row];
  const int lo = a_pos[r.row] + item.batch * kBinEntries, hi = min(lo + kBinEntries, a_pos[r.row + 1]);
  int start = 0, len = 0;
  A av = (A)0;
  if (lo + tid < hi) {
    const int j = a_crd[lo + tid];
    start = b_pos[j];
    len = b_pos[j + 1] - start;
    av = (A)a_val[lo + tid];
  }
  const int total = fill_batch<kBinEntries, true, A>(len, start, av, s_batch, s_scan);
  const int lane = wave_lane(), w = uniform(tid / kWaveSize);
  for (int x0 = item.share * kBinProducts; x0 < total; x0 += item.shares * kBinProducts) {  // uniform
    const int n = min(kBinProducts, total - x0);
    const ProductStep step = product_step(x0, n, kBinThreads / kWaveSize, w);
    int e[U], col[U], rank[U];
    A b[U];
    unsigned long long used = 0;  // (the round trip passes while the products are gathered)
    if (tid == kBinThreads - 1) used = atomicAdd(&bins.used[item.row], (1ull << 32) + (unsigned)n);
    if (step.first < step.last) {
      entries_of_products<kBinEntries, U, A>(step, s_batch, e);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (u > 0 && !step.has(u)) break;  // uniform over the wavefront
        const int q = step.product(u, lane) + s_batch.start[e[u]];
        col[u] = b_crd[q];
        b[u] = (A)b_val[q];
      }
    }
    __syncthreads();  // everyone is done with the previous window
    if (tid <= kMaxBins) s_count[tid] = 0;
    if (tid == kBinThreads - 1) {
      s_first = (int)(unsigned)used;
      s_window = (int)(used >> 32);
    }
    __syncthreads();
    int bin[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (step.first + u * kWaveSize + lane < step.last) {
        bin[u] = col[u] >> bins.shift;
        // The wavefront's products of this range, and one add for all of them: 64 adds to some sixteen counters
        // queue up in the LDS (kernel 99 -> 80 us: vector instructions instead, which had time).
        unsigned long long alike = __ballot(true);
#pragma unroll
        for (int bit = 0; (1 << bit) < kMaxBins; ++bit) {
          if (bins.n <= 1 << bit) break;  // uniform
          const int set = -((bin[u] >> bit) & 1);
          const unsigned long long with = __ballot(set != 0);
          const unsigned lo = (unsigned)alike & ~((unsigned)with ^ (unsigned)set);
          const unsigned hi = (unsigned)(alike >> 32) & ~((unsigned)(with >> 32) ^ (unsigned)set);
          alike = (unsigned long long)hi << 32 | lo;
        }
        const int before = __builtin_amdgcn_mbcnt_hi((unsigned)(alike >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)alike, 0u));
        int base = 0;
        if (before == 0) base = atomicAdd(&s_count[bin[u]], __popcll(alike));
        rank[u] = before + __shfl(base, __ffsll(alike) - 1);
      }
    __syncthreads();
    if (w == 0) {  // (the others wait: a scan by the lanes, not a chain of reads)
      const int count = lane < bins.n ? s_count[lane] : 0, at = team_inclusive_sum<kWaveSize>(count) - count;
      if (lane <= bins.n) {
        s_at[lane] = at;
        bins.window[r.first_window + s_window].at[lane] = (unsigned short)at;
      }
    }
    if (tid == 0) bins.window[r.first_window + s_window].first = r.first_product + s_first;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (step.first + u * kWaveSize + lane < step.last) {
        const int at = s_at[bin[u]] + rank[u];
        s_column[at] = (unsigned short)(col[u] - (bin[u] << bins.shift));
        s_value[at] = s_batch.a_val[e[u]] * b[u];
      }
    __syncthreads();
    const int64_t first = (int64_t)r.first_product + s_first;
    A *values = static_cast<A *>(bins.values) + first;
    for (int i = tid; i < n; i += kBinThreads) {
      bins.columns[first + i] = s_column[i];
      values[i] = s_value[i];
    }
  }
}

// fn(first, last, here) for the products of range `bin` of a row, in columns and values: 64 windows' runs are looked up at a
// time by each of WAVES wavefronts, lane i < here has the i-th's ends.
template <int WAVES, typename Fn>
__device__ __forceinline__ void for_each_runs(const Bins &bins, const BinRow &r, int windows, int bin, Fn fn) {
  const int lane = wave_lane(), w = WAVES == 1 ? 0 : threadIdx.x / kWaveSize;
  for (int base = w; base < windows; base += WAVES * kWaveSize) {
    int first = 0, last = 0;
    if (base + lane * WAVES < windows) {
      const BinWindow &win = bins.window[r.first_window + base + lane * WAVES];
      first = win.first + win.at[bin];
      last = win.first + win.at[bin + 1];
    }
    fn(first, last, min(kWaveSize, (windows - base + WAVES - 1) / WAVES));
  }
}

// fn(place, to) for every product of range `bin` of a row, up to four of them from `place` on, 64 apart and below `to`: a
// wavefront takes a run.
template <int WAVES, typename Fn>
__device__ __forceinline__ void for_each_binned(const Bins &bins, const BinRow &r, int windows, int bin, Fn fn) {
  for_each_runs<WAVES>(bins, r, windows, bin, [&](int first, int last, int here) {
    for (int i = 0; i < here; ++i) {
      const int from = __builtin_amdgcn_readlane(first, i), to = __builtin_amdgcn_readlane(last, i);
      for (int p = from + wave_lane(); p < to; p += 4 * kWaveSize) fn(p, to);
    }
  });
}

// Rows of kGiantProducts products and more: a workgroup to a range; the others: a wavefront to a range, eight of them to a
// workgroup (131,072 nodes, 16 a row: a workgroup of 256 to every range 44 us; with 512 threads for the longest rows, which are
// what the launch waits for, those first, and wavefronts for the others 34).
constexpr int kBinCountThreads = 512;
__global__ __launch_bounds__(kBinCountThreads) void spgemm_bin_count_kernel(Bins bins, int *__restrict__ c_pos) {
  constexpr int kWaves = kBinCountThreads / kWaveSize;
  __shared__ unsigned s_all_bits[kWaves][kBinColumns / 32];
  __shared__ int s_scan[kWaves];
  const int words = (1 << bins.shift) / 32;
  if (blockIdx.x >= (unsigned)bins.counted_wide * (unsigned)bins.n) {
    const unsigned groups = (unsigned)(bins.n + kWaves - 1) / kWaves, at = blockIdx.x - (unsigned)bins.counted_wide * (unsigned)bins.n;
    const int idx = bins.counted_wide + (int)(at / groups), w = uniform((int)threadIdx.x / kWaveSize), bin = (int)(at % groups) * kWaves + w;
    if (bin >= bins.n) return;
    unsigned *const bits = s_all_bits[w];
    const BinRow r = bins.row[idx];
    const int windows = (int)(bins.used[idx] >> 32);
    for (int i = wave_lane(); i < words; i += kWaveSize) bits[i] = 0u;
    wave_lds_sync();
    for_each_binned<1>(bins, r, windows, bin, [&](int p, int to) {
      int c[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) c[u] = p + u * kWaveSize < to ? bins.columns[p + u * kWaveSize] : -1;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (c[u] >= 0) atomicOr(&bits[c[u] >> 5], 1u << (c[u] & 31));
    });
    wave_lds_sync();
    int mine = 0;
    for (int i = wave_lane(); i < words; i += kWaveSize) mine += __popc(bits[i]);
    mine = team_inclusive_sum<kWaveSize>(mine);
    if (wave_lane() == kWaveSize - 1) {
      bins.counts[(size_t)idx * bins.n + bin] = mine;
      if (mine) atomicAdd(&c_pos[r.row], mine);
    }
    return;
  }
  unsigned *const s_bits = s_all_bits[0];
  const int idx = (int)(blockIdx.x / (unsigned)bins.n), bin = (int)(blockIdx.x % (unsigned)bins.n);
  const BinRow r = bins.row[idx];
  const int windows = (int)(bins.used[idx] >> 32);
  for (int i = threadIdx.x; i < words; i += kBinCountThreads) s_bits[i] = 0u;
  __syncthreads();
  // Four runs of a wavefront's at a time, of clamped places (a load behind a condition is waited for before the next, and four
  // runs gain nothing): 131,072 nodes, 16 a row 52 -> 44 us, 45,000, 10 a row 18.0 -> 14.5, with a hub of 50,000 entries 72 -> 63.
  // (The sums: 120 -> 126.)  Not where a wavefront has up to three, many of them of a few products: rows of at most 5,000 entries
  // 28, four at a time 35.
  constexpr int kRuns = 4, kEach = 4;
  if (windows <= 3 * kWaves) {
    for_each_binned<kWaves>(bins, r, windows, bin, [&](int p, int to) {
      int c[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) c[u] = p + u * kWaveSize < to ? bins.columns[p + u * kWaveSize] : -1;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (c[u] >= 0) atomicOr(&s_bits[c[u] >> 5], 1u << (c[u] & 31));
    });
  } else {
    for_each_runs<kWaves>(bins, r, windows, bin, [&](int first, int last, int here) {
      for (int i = 0; i < here; i += kRuns) {
        int p[kRuns], to[kRuns], longest = 0;
#pragma unroll
        for (int j = 0; j < kRuns; ++j) {
          const int run = min(i + j, kWaveSize - 1), from = __builtin_amdgcn_readlane(first, run);
          to[j] = i + j < here ? __builtin_amdgcn_readlane(last, run) : from;
          longest = max(longest, to[j] - from);
          p[j] = from + wave_lane();
        }
        for (int o = 0; o < longest; o += kEach * kWaveSize) {
          int c[kRuns][kEach];
#pragma unroll
          for (int j = 0; j < kRuns; ++j)
#pragma unroll
            for (int u = 0; u < kEach; ++u) c[j][u] = bins.columns[max(min(p[j] + o + u * kWaveSize, to[j] - 1), 0)];
#pragma unroll
          for (int j = 0; j < kRuns; ++j)
#pragma unroll
            for (int u = 0; u < kEach; ++u)
              if (p[j] + o + u * kWaveSize < to[j]) atomicOr(&s_bits[c[j][u] >> 5], 1u << (c[j][u] & 31));
        }
      }
    });
  }
  __syncthreads();
  int mine = 0, total = 0;
  for (int i = threadIdx.x; i < words; i += kBinCountThreads) mine += __popc(s_bits[i]);
  (void)block_exclusive_scan_n<kWaves>(mine, s_scan, total);
  if (threadIdx.x == 0) {
    bins.counts[(size_t)idx * bins.n + bin] = total;
    if (total) atomicAdd(&c_pos[r.row], total);
  }
}

constexpr int kBinSumThreads = 512;
template <typename T>
__global__ __launch_bounds__(kBinSumThreads) void spgemm_bin_sums_kernel(Bins bins, const int *__restrict__ c_pos,
                                                                         int *__restrict__ c_crd, T *__restrict__ c_val) {
  using A = typename Acc<T>::type;
  constexpr int kWaves = kBinSumThreads / kWaveSize, kFour = (int)(16 / sizeof(A));
  static_assert(2 * kBinColumns / 32 <= kBinSumThreads, "a thread to half a word of the bitmap");
  alignas(16) __shared__ A s_sum[kBinColumns];
  __shared__ unsigned s_bits[kBinColumns / 32];
  __shared__ int s_rank[kBinColumns / 32];
  __shared__ int s_scan[kWaves];
  const int tid = threadIdx.x, lane = wave_lane();
  const int idx = (int)(blockIdx.x / (unsigned)bins.n), bin = (int)(blockIdx.x % (unsigned)bins.n);
  const int *counts = bins.counts + (size_t)idx * bins.n;
  const int n = counts[bin];
  const BinRow r = bins.row[idx];
  const int windows = (int)(bins.used[idx] >> 32), columns = 1 << bins.shift, words = columns / 32;
  for (int i = tid; i < columns / kFour; i += kBinSumThreads) reinterpret_cast<uint4 *>(s_sum)[i] = make_uint4(0u, 0u, 0u, 0u);
  for (int i = tid; i < words; i += kBinSumThreads) s_bits[i] = 0u;
  int out = c_pos[r.row];
  for (int i = 0; i < bin; ++i) out += counts[i];
  if (n == 0) return;
  __syncthreads();
  const A *values = static_cast<const A *>(bins.values);
  for_each_binned<kWaves>(bins, r, windows, bin, [&](int p, int to) {
    int c[4];
    A v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int at = p + u * kWaveSize;
      c[u] = at < to ? bins.columns[at] : -1;
      v[u] = at < to ? values[at] : (A)0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (c[u] >= 0) {
        atomicOr(&s_bits[c[u] >> 5], 1u << (c[u] & 31));
        lds_accumulate<A>(&s_sum[c[u]], v[u]);
      }
  });
  __syncthreads();
  int unused = 0;
  const unsigned half = tid < 2 * words ? (s_bits[tid >> 1] >> (16 * (tid & 1))) & 0xffffu : 0u;
  const int rank = block_exclusive_scan_n<kWaves>(__popc(half), s_scan, unused);
  const int first_column = bin << bins.shift;
  if (4 * n < columns) {  // a thread per half word of the bitmap (per word, and cleared four bytes at a time: 120 us, 111)
    int at = out + rank;
    for (unsigned bits = half; bits; bits &= bits - 1, ++at) {
      const int col = tid * 16 + __ffs(bits) - 1;
      c_crd[at] = first_column + col;
      c_val[at] = (T)s_sum[col];
    }
    return;
  }
  if (tid < 2 * words && !(tid & 1)) s_rank[tid >> 1] = rank;
  __syncthreads();
  // two bitmap words, 64 columns, per wavefront and step
  for (int w = 2 * (tid / kWaveSize); w < words; w += 2 * kWaves) {
    const int mine = w + (lane >> 5), bit = lane & 31;
    const unsigned b = s_bits[mine];
    if ((b >> bit) & 1u) {
      const int at = out + s_rank[mine] + __popc(b & ((1u << bit) - 1u));
      c_crd[at] = first_column + mine * 32 + bit;
      c_val[at] = (T)s_sum[mine * 32 + bit];
    }
  }
}

// ---- host side ------------------------------------------------------------------------------
struct SpgemmWorkspace {
  int pool;               // rows that can be shared out among workgroups
  int *split_rows;
  int4 *split_items;
  unsigned *split_bits;
  void *split_sums;
  int *products, *small_rows, *medium_rows, *huge_rows, *counters;
  int huge_pool;
  int *scan_totals;
  unsigned *bitmaps;
  int *ranks;
  size_t total;
};

inline size_t round256(size_t v) { return (v + 255) / 256 * 256; }

inline SpgemmWorkspace spgemm_layout(char *base, int64_t M, int64_t N, size_t elem) {
  SpgemmWorkspace ws;
  size_t off = 0;
  auto take = [&](size_t bytes) { char *p = base ? base + off : nullptr; off += round256(bytes); return p; };
  ws.products = reinterpret_cast<int *>(take((size_t)M * 4));
  ws.small_rows = reinterpret_cast<int *>(take((size_t)M * 4));
  ws.medium_rows = reinterpret_cast<int *>(take((size_t)M * 4));
  ws.huge_rows = reinterpret_cast<int *>(take((size_t)M * 4));
  ws.counters = reinterpret_cast<int *>(take(counter(kSpgemmCounters) * 4));
  ws.pool = split_pool(N);
  ws.split_rows = reinterpret_cast<int *>(take((size_t)ws.pool * 4));
  ws.split_items = reinterpret_cast<int4 *>(take((size_t)ws.pool * kSplitMaxSlices * sizeof(int4)));
  ws.split_bits = reinterpret_cast<unsigned *>(take((size_t)ws.pool * ((size_t)(N + 31) / 32) * 4));
  ws.split_sums = take((size_t)ws.pool * (size_t)N * 8);
  ws.scan_totals = reinterpret_cast<int *>(take(((size_t)(M + 1) / kScanTile + 1) * 4));
  ws.huge_pool = huge_workgroups(N);
  // up to kLdsBitmapColumns columns the bitmap tier lives in LDS and needs no slabs
  const size_t slab_words = N <= kLdsBitmapColumns ? 0 : (size_t)(N + 31) / 32;
  ws.bitmaps = reinterpret_cast<unsigned *>(take((size_t)ws.huge_pool * slab_words * 4));
  ws.ranks = reinterpret_cast<int *>(take((size_t)ws.huge_pool * slab_words * 4));
  (void)elem;  // no part of the workspace depends on the value type
  ws.total = off;
  return ws;
}

inline int spgemm_check(const char *fn, int64_t M, int64_t K, int64_t N, const void *a_pos,
                        const void *a_crd, const void *b_pos, const void *b_crd, const void *c_pos,
                        const void *workspace, size_t workspace_bytes, size_t elem) {
  if (M < 0 || K < 0 || N < 0)
    return fail(SCORCH_HIP_EINVAL, "%s: negative size (M=%lld K=%lld N=%lld)", fn, (long long)M,
                (long long)K, (long long)N);
  if (M >= INT32_MAX || K >= INT32_MAX || N >= INT32_MAX)
    return fail(SCORCH_HIP_EUNSUPPORTED, "%s: sizes must fit int32 indices", fn);
  SCORCH_REQUIRE(a_pos && b_pos && c_pos, "%s: NULL row pointer", fn);
  SCORCH_REQUIRE(aligned_to(a_pos, 4) && aligned_to(a_crd, 4) && aligned_to(b_pos, 4) &&
                     aligned_to(b_crd, 4) && aligned_to(c_pos, 4),
                 "%s: index arrays must be 4-byte aligned", fn);
  const size_t need = spgemm_layout(nullptr, M, N, elem).total;
  if (!workspace || workspace_bytes < need)
    return fail(SCORCH_HIP_EWORKSPACE, "%s: workspace of %zu bytes needed, %zu given", fn, need,
                workspace ? workspace_bytes : (size_t)0);
  SCORCH_REQUIRE(aligned_to(workspace, 256), "%s: workspace must be 256-byte aligned", fn);
  return SCORCH_HIP_OK;
}

// What the symbolic pass found out, for a numeric pass over the same workspace.
struct SpgemmReport {
  int64_t entries;                                         // of the result; -1: 2^31 or more
  int64_t small, medium, huge, giant, split, split_items;  // rows listed per tier; slices of the rows shared out
  int64_t products, batches;                               // of the rows beyond kMediumProducts
};
constexpr int kSpgemmReportWords = 9;
inline SpgemmReport report_of(const int64_t *w) { return {w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7], w[8]}; }

// `known`: the numeric pass finds the row lists of the symbolic pass in the workspace and launches what has rows.
// `sync`: the symbolic pass hands its report over (its short rows' part what pass 0 found, the long rows' part the rest).
// `bins`: the rows beyond kMediumProducts go by bins (the symbolic pass has counted them there already).
constexpr int kShortRows = 1, kLongRows = 2;
template <typename T, bool NUMERIC>
int spgemm_run(int M, int N, const int *a_pos, const int *a_crd, const T *a_val, const int *b_pos,
               const int *b_crd, const T *b_val, int *c_pos, int *c_crd, T *c_val,
               const SpgemmWorkspace &ws, hipStream_t stream, int parts = kShortRows | kLongRows,
               const SpgemmReport *known = nullptr, SyncCall *sync = nullptr, const Bins *bins = nullptr) {
  using A = typename Acc<T>::type;
  const int words = (N + 31) / 32;
  const bool narrow = N <= kNarrowColumns;
  if (parts & kShortRows) {
    if (!known) {
      const int64_t clear_words = (int64_t)ws.pool * words;
      const unsigned clear_blocks = (unsigned)(1 + (clear_words < 1 << 18 ? clear_words : 1 << 18) / 1024);
      spgemm_reset_kernel<<<clear_blocks, kBlockThreads, 0, stream>>>(ws.counters, NUMERIC ? nullptr : c_pos + M, clear_words,
                                                                      ws.split_bits);
      SCORCH_HIP_CHECK(hipGetLastError());
      const int rows_per_group = bounds_rows_per_group(M);
      const unsigned row_groups = (unsigned)(((int64_t)M + rows_per_group - 1) / rows_per_group);
      spgemm_bounds_kernel<<<row_groups, kBlockThreads, 0, stream>>>(M, rows_per_group, a_pos, a_crd, b_pos, ws.products,
                                                                    ws.small_rows, ws.medium_rows,
                                                                    ws.huge_rows, ws.counters,
                                                                    sync ? sync->target() : nullptr, sync ? sync->sequence() : 0);
      SCORCH_HIP_CHECK(hipGetLastError());
    }
    // rows the smaller bitmap kernel goes through; with the result's row pointer known, also those of the tier above
    // that turn out to have few distinct columns
    const int *narrow_rows = NUMERIC && narrow && !bins ? ws.huge_rows : nullptr;
    const bool by_column = NUMERIC && N <= kBitmapSums;  // sums of rows of up to kMediumProducts products (spgemm_lds_bitmap_rows)
    constexpr int kByColumnWords = NUMERIC ? kBitmapSums / 32 : kNarrowColumns / 32;
    const auto blocks_for = [&](int64_t rows) {
      return (unsigned)std::min<int64_t>(rows, known ? kKnownWorkgroups : kMediumWorkgroups);
    };
    const unsigned small_blocks = blocks_for(known ? known->small : M);
    const unsigned bitmap_blocks = blocks_for(known ? known->medium + (narrow_rows ? known->huge : 0) : M);
    if (M < 4 * 8192 && narrow) {
      // (see spgemm_small_matrix_kernel)
      constexpr int kMore = NUMERIC ? kBitmapThreads : kBlockThreads;
      const bool few = known && 2 * (known->small + known->medium) < M;
      const bool more = !by_column && (sizeof(A) > 4 || few);
      const int threads = more ? kMore : kBlockThreads;
      const unsigned tiny_blocks = (unsigned)((M + threads / kWaveSize - 1) / (threads / kWaveSize));
      auto kernel = by_column ? &spgemm_small_matrix_kernel<T, NUMERIC, kBlockThreads, kByColumnWords>
                    : more    ? &spgemm_small_matrix_kernel<T, NUMERIC, kMore, kNarrowColumns / 32>
                              : &spgemm_small_matrix_kernel<T, NUMERIC, kBlockThreads, kNarrowColumns / 32>;
      kernel<<<bitmap_blocks + small_blocks + tiny_blocks, threads, 0, stream>>>(
          M, N, (int)bitmap_blocks, (int)small_blocks, a_pos, a_crd, a_val, b_pos, b_crd, b_val, ws.products, ws.small_rows,
          ws.medium_rows, narrow_rows, ws.counters, c_pos, c_crd, c_val);
      SCORCH_HIP_CHECK(hipGetLastError());
    } else {
      // four rows to a wavefront
      const int64_t rows_per_block = (kTinyThreads / kWaveSize) * (kWaveSize / kMicroTeam);
      const unsigned tiny_blocks = (unsigned)round_up_8(((int64_t)M + rows_per_block - 1) / rows_per_block);
      spgemm_tiny_kernel<T, NUMERIC><<<tiny_blocks, kTinyThreads, 0, stream>>>(
          M, a_pos, a_crd, a_val, b_pos, b_crd, b_val, ws.products, c_pos, c_crd, c_val);
      SCORCH_HIP_CHECK(hipGetLastError());
      if (small_blocks) {
        spgemm_medium_kernel<T, NUMERIC, kSmallProducts, 2, kBlockThreads><<<small_blocks, kBlockThreads, 0, stream>>>(
            a_pos, a_crd, a_val, b_pos, b_crd, b_val, ws.products, ws.small_rows, ws.counters, c_pos, c_crd, c_val);
        SCORCH_HIP_CHECK(hipGetLastError());
      }
      if (bitmap_blocks && narrow) {
        // narrow enough for a bitmap in LDS beside other workgroups: no hashing, nothing to sort
        constexpr int kMore = NUMERIC ? kBitmapThreads : kBlockThreads;
        auto kernel = by_column ? &spgemm_lds_bitmap_kernel<T, NUMERIC, kByColumnWords, kBlockThreads, kBitmapSums, 0, 4>
                                : &spgemm_lds_bitmap_kernel<T, NUMERIC, kNarrowColumns / 32, kMore, kBitmapSums, 0, 4>;
        kernel<<<bitmap_blocks, by_column ? kBlockThreads : kMore, 0, stream>>>(M, N, a_pos, a_crd, a_val, b_pos, b_crd, b_val,
                                                                                ws.medium_rows, narrow_rows, ws.counters, c_pos,
                                                                                c_crd, c_val);
      } else if (bitmap_blocks) {
        // Two workgroups of 512 threads to a CU with sums of 4 bytes, one of 8 wavefronts with 8.  Sorted in the table's place by 1,024
        // threads, with sums of 8 bytes by 256 (as many as had fitted beside separate tables), rows of 1,200 to 2,000 products had lost
        // against those.  20,000 x 200,000, us, separate tables, those threads, now: fp32 (1,200 products) 995, 1,006, 491; (1,600) 1,074,
        // 1,091, 552; (3,600) 1,536, 1,540, 945; fp64 (1,200) 1,204, 1,222, 789; (1,600) 1,404, 1,432, 901; (3,600) 2,547, 2,502, 1,531.
        constexpr int kThreads = kBitmapThreads;
        spgemm_medium_kernel<T, NUMERIC, kMediumProducts, 0, kThreads><<<bitmap_blocks, kThreads, 0, stream>>>(
            a_pos, a_crd, a_val, b_pos, b_crd, b_val, ws.products, ws.medium_rows, ws.counters, c_pos, c_crd, c_val);
      }
      SCORCH_HIP_CHECK(hipGetLastError());
    }
  }
  if (!(parts & kLongRows)) return SCORCH_HIP_OK;
  const int64_t listed = known ? known->huge + known->giant : M;  // rows beyond kMediumProducts, at most
  if (bins) {
    if constexpr (NUMERIC) {
      spgemm_bin_sums_kernel<T><<<(unsigned)(bins->rows * bins->n), kBinSumThreads, 0, stream>>>(*bins, c_pos, c_crd, c_val);
      SCORCH_HIP_CHECK(hipGetLastError());
    }
  } else if (listed > 0) {
    if (ws.pool > 0 && (!known || !NUMERIC || known->split > 0)) {
      A *sums = static_cast<A *>(ws.split_sums);
      if (!NUMERIC || !known) {
        spgemm_split_select_kernel<<<1, kBlockThreads, 0, stream>>>(M, ws.pool, a_pos, ws.products, ws.huge_rows, ws.counters,
                                                                   ws.split_rows, ws.split_items);
        SCORCH_HIP_CHECK(hipGetLastError());
        auto columns_of = words <= 4096 ? &spgemm_split_columns_kernel<4096> : &spgemm_split_columns_kernel<kSplitMaxColumns / 32>;
        columns_of<<<512, kHugeThreads, 0, stream>>>(words, a_pos, a_crd, b_pos, b_crd, ws.counters, ws.split_rows,
                                                     ws.split_items, ws.split_bits);
        SCORCH_HIP_CHECK(hipGetLastError());
      }
      if (NUMERIC) {
        const int64_t n_sums = (int64_t)(known ? (int)known->split : ws.pool) * N;
        spgemm_split_clear_kernel<A><<<(unsigned)(1 + (n_sums < 1 << 20 ? n_sums : 1 << 20) / 1024), kBlockThreads, 0, stream>>>(
            N, ws.counters, sums);
        SCORCH_HIP_CHECK(hipGetLastError());
        const unsigned slices = known ? (unsigned)known->split_items : 512u;
        spgemm_split_sums_kernel<T><<<slices, kHugeThreads, 0, stream>>>(N, a_pos, a_crd, a_val, b_pos, b_crd, b_val, ws.counters,
                                                                        ws.split_rows, ws.split_items, sums);
        SCORCH_HIP_CHECK(hipGetLastError());
        const unsigned pieces = (unsigned)((words + kEmitWords - 1) / kEmitWords);
        spgemm_split_emit_kernel<T><<<dim3(pieces, (unsigned)(known ? known->split : ws.pool)), kHugeThreads, 0, stream>>>(
            N, words, ws.counters, ws.split_rows, ws.split_bits, sums, c_pos, c_crd, c_val);
        SCORCH_HIP_CHECK(hipGetLastError());
      }
    }
    // one workgroup per CU's worth of LDS; more only queue up behind them
    const int64_t huge_rows = listed - (known && NUMERIC ? known->split : 0);
    const unsigned lds_pool = (unsigned)(huge_rows < 512 ? huge_rows : 512);
    if (lds_pool == 0) {
    } else if (narrow) {
      spgemm_lds_bitmap_kernel<T, NUMERIC, kNarrowColumns / 32, kHugeThreads, 0, 1, 3><<<lds_pool, kHugeThreads, 0, stream>>>(
          M, N, a_pos, a_crd, a_val, b_pos, b_crd, b_val, ws.huge_rows, nullptr, ws.counters, c_pos, c_crd, c_val);
    } else if (!NUMERIC && N > 32 * 16384 && N <= 32 * 32768) {
      // the symbolic pass keeps no ranks or sums: its bitmap can be twice as wide, one range instead of two
      spgemm_lds_bitmap_kernel<T, NUMERIC, NUMERIC ? 16384 : 32768, kHugeThreads, 0, 1, 3>
          <<<lds_pool, kHugeThreads, 0, stream>>>(M, N, a_pos, a_crd, a_val, b_pos, b_crd, b_val, ws.huge_rows,
                                                  nullptr, ws.counters, c_pos, c_crd, c_val);
    } else if (N <= kLdsBitmapColumns) {
      spgemm_lds_bitmap_kernel<T, NUMERIC, 16384, kHugeThreads, 0, 1, 3><<<lds_pool, kHugeThreads, 0, stream>>>(
          M, N, a_pos, a_crd, a_val, b_pos, b_crd, b_val, ws.huge_rows, nullptr, ws.counters, c_pos, c_crd, c_val);
    } else {
      spgemm_huge_kernel<T, NUMERIC><<<ws.huge_pool, kHugeThreads, 0, stream>>>(
          M, N, a_pos, a_crd, a_val, b_pos, b_crd, b_val, ws.huge_rows, ws.counters, ws.bitmaps,
          ws.ranks, c_pos, c_crd, c_val);
    }
    SCORCH_HIP_CHECK(hipGetLastError());
  }
  if (!NUMERIC) {
    const int64_t n = (int64_t)M + 1;
    unsigned long long *grand_total = reinterpret_cast<unsigned long long *>(ws.counters + counter(6));
    const SplitCount split = {ws.pool > 0 ? ws.split_rows : nullptr, ws.split_bits, words};
    int64_t *report = sync ? sync->target() : nullptr;
    const int64_t sequence = sync ? sync->sequence() : 0;
    if (ws.pool > 0 && !bins && listed > 0) {
      spgemm_split_count_kernel<<<(unsigned)ws.pool, kBlockThreads, 0, stream>>>(ws.counters, split, c_pos);
      SCORCH_HIP_CHECK(hipGetLastError());
    }
    if (n <= kScanOneGroup) {
      scan_one_group_kernel<<<1, kScanThreads, 0, stream>>>(c_pos, (int)n, ws.counters, report, sequence);
      SCORCH_HIP_CHECK(hipGetLastError());
      return SCORCH_HIP_OK;
    }
    const unsigned tiles = (unsigned)((n + kScanTile - 1) / kScanTile);
    scan_tile_totals_kernel<<<tiles, kBlockThreads, 0, stream>>>(c_pos, n, ws.scan_totals, grand_total);
    SCORCH_HIP_CHECK(hipGetLastError());
    if (tiles <= kScanOwnTotals) {
      scan_apply_kernel<false><<<tiles, kBlockThreads, 0, stream>>>(c_pos, n, ws.scan_totals, ws.counters, report, sequence);
    } else {
      scan_spine_kernel<<<1, kBlockThreads, 0, stream>>>(ws.scan_totals, tiles, ws.counters, report, sequence);
      SCORCH_HIP_CHECK(hipGetLastError());
      scan_apply_kernel<true><<<tiles, kBlockThreads, 0, stream>>>(c_pos, n, ws.scan_totals, ws.counters, report, sequence);
    }
    SCORCH_HIP_CHECK(hipGetLastError());
  }
  return SCORCH_HIP_OK;
}

template <typename T>
int spgemm_numeric_entry(const char *fn, int64_t M, int64_t K, int64_t N, const int32_t *a_pos,
                         const int32_t *a_crd, const T *a_val, const int32_t *b_pos,
                         const int32_t *b_crd, const T *b_val, const int32_t *c_pos, int32_t *c_crd,
                         T *c_val, void *workspace, size_t workspace_bytes, void *stream,
                         const int64_t *report = nullptr, void *bin_memory = nullptr, size_t bin_bytes = 0) {
  if (int rc = spgemm_check(fn, M, K, N, a_pos, a_crd, b_pos, b_crd, c_pos, workspace, workspace_bytes,
                            sizeof(T)))
    return rc;
  if (M == 0 || N == 0 || K == 0) return SCORCH_HIP_OK;
  const SpgemmWorkspace ws = spgemm_layout(static_cast<char *>(workspace), M, N, sizeof(T));
  SpgemmReport known;
  Bins bins;
  if (report) {
    known = report_of(report);
    if (bin_memory) bins = spgemm_bins(static_cast<char *>(bin_memory), ws.counters, N, sizeof(T), known.huge + known.giant,
                                       known.giant, known.products, known.batches);
    if (bins.total > bin_bytes)
      return fail(SCORCH_HIP_EWORKSPACE, "%s: bins of %zu bytes needed, %zu given", fn, bins.total, bin_bytes);
  }
  return spgemm_run<T, true>((int)M, (int)N, a_pos, a_crd, a_val, b_pos, b_crd, b_val,
                             const_cast<int32_t *>(c_pos), c_crd, c_val, ws,
                             static_cast<hipStream_t>(stream), kShortRows | kLongRows, report ? &known : nullptr, nullptr,
                             bins.n > 0 ? &bins : nullptr);
}

// The second half of the symbolic pass.
template <typename T>
int spgemm_symbolic_entry(const char *fn, int64_t M, int64_t K, int64_t N, const int32_t *a_pos,
                          const int32_t *a_crd, const T *a_val, const int32_t *b_pos, const int32_t *b_crd, const T *b_val,
                          int32_t *c_pos, void *workspace, size_t workspace_bytes, void *bin_memory, size_t bin_bytes,
                          int64_t *report, void *stream) {
  if (int rc = spgemm_check(fn, M, K, N, a_pos, a_crd, b_pos, b_crd, c_pos, workspace, workspace_bytes,
                            sizeof(T)))
    return rc;
  SCORCH_REQUIRE(report != nullptr, "%s: report is NULL", fn);
  if (M == 0) return SCORCH_HIP_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  SpgemmReport known = report_of(report);
  const SpgemmWorkspace ws = spgemm_layout(static_cast<char *>(workspace), M, N, sizeof(T));
  Bins bins;
  if (bin_memory) bins = spgemm_bins(static_cast<char *>(bin_memory), ws.counters, N, sizeof(T), known.huge + known.giant,
                                     known.giant, known.products, known.batches);
  if (bins.total > bin_bytes)
    return fail(SCORCH_HIP_EWORKSPACE, "%s: bins of %zu bytes needed, %zu given", fn, bins.total, bin_bytes);
  SyncCall sync;
  if (sync.null()) return fail(SCORCH_HIP_ERUNTIME, "%s: no memory for the report", fn);
  if (bins.n > 0) {
    spgemm_bin_rows_kernel<<<(unsigned)((bins.rows + kBlockThreads - 1) / kBlockThreads), kBlockThreads, 0, s>>>(
        (int)M, bins, a_pos, ws.products, ws.huge_rows, ws.counters, c_pos);
    SCORCH_HIP_CHECK(hipGetLastError());
    spgemm_bin_items_kernel<<<(unsigned)bins.rows, kBinItemThreads, 0, s>>>(bins, a_pos, a_crd, b_pos);
    SCORCH_HIP_CHECK(hipGetLastError());
    spgemm_bin_kernel<T><<<(unsigned)bins.items, kBinThreads, 0, s>>>(bins, a_pos, a_crd, a_val, b_pos, b_crd, b_val);
    SCORCH_HIP_CHECK(hipGetLastError());
    constexpr int kWaves = kBinCountThreads / kWaveSize;
    const int64_t count_blocks = (int64_t)bins.counted_wide * bins.n + (bins.rows - bins.counted_wide) * ((bins.n + kWaves - 1) / kWaves);
    spgemm_bin_count_kernel<<<(unsigned)count_blocks, kBinCountThreads, 0, s>>>(bins, c_pos);
    SCORCH_HIP_CHECK(hipGetLastError());
  }
  if (int rc = spgemm_run<float, false>((int)M, (int)N, a_pos, a_crd, nullptr, b_pos, b_crd, nullptr, c_pos, nullptr, nullptr, ws,
                                        s, kLongRows, &known, &sync, bins.n > 0 ? &bins : nullptr))
    return rc;
  return sync.wait(fn, s, report, 7);
}

}  // namespace scorch

extern "C" {

size_t scorch_hip_spgemm_csr_workspace_bytes(int64_t M, int64_t N, size_t elem_size) {
  if (M < 0 || N < 0 || M >= INT32_MAX || elem_size == 0) return 0;
  return scorch::spgemm_layout(nullptr, M, N, elem_size).total;
}

int scorch_hip_spgemm_csr_symbolic(int64_t M, int64_t K, int64_t N, const int32_t *a_row_ptr,
                                   const int32_t *a_col_idx, const int32_t *b_row_ptr,
                                   const int32_t *b_col_idx, int32_t *c_row_ptr, void *workspace,
                                   size_t workspace_bytes, void *stream) {
  using namespace scorch;
  const char *fn = "scorch_hip_spgemm_csr_symbolic";
  if (int rc = spgemm_check(fn, M, K, N, a_row_ptr, a_col_idx, b_row_ptr, b_col_idx, c_row_ptr,
                            workspace, workspace_bytes, 1))
    return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (M == 0) {
    spgemm_reset_kernel<<<1, kBlockThreads, 0, s>>>(static_cast<int *>(workspace), c_row_ptr, 0, nullptr);
    SCORCH_HIP_CHECK(hipGetLastError());
    return SCORCH_HIP_OK;
  }
  const SpgemmWorkspace ws = spgemm_layout(static_cast<char *>(workspace), M, N, 1);
  return spgemm_run<float, false>((int)M, (int)N, a_row_ptr, a_col_idx, nullptr, b_row_ptr, b_col_idx,
                                  nullptr, c_row_ptr, nullptr, nullptr, ws, s);
}

int scorch_hip_spgemm_csr_symbolic_planned_begin(int64_t M, int64_t K, int64_t N, const int32_t *a_row_ptr,
                                                 const int32_t *a_col_idx, const int32_t *b_row_ptr,
                                                 const int32_t *b_col_idx, int32_t *c_row_ptr, void *workspace,
                                                 size_t workspace_bytes, size_t elem_size, int64_t *report,
                                                 size_t *bin_bytes, void *stream) {
  using namespace scorch;
  const char *fn = "scorch_hip_spgemm_csr_symbolic_planned_begin";
  if (int rc = spgemm_check(fn, M, K, N, a_row_ptr, a_col_idx, b_row_ptr, b_col_idx, c_row_ptr,
                            workspace, workspace_bytes, 1))
    return rc;
  SCORCH_REQUIRE(report != nullptr && bin_bytes != nullptr, "%s: report or bin_bytes is NULL", fn);
  SCORCH_REQUIRE(elem_size == 4 || elem_size == 8, "%s: values of %zu bytes", fn, elem_size);
  hipStream_t s = static_cast<hipStream_t>(stream);
  for (int i = 0; i < kSpgemmReportWords; ++i) report[i] = 0;
  *bin_bytes = 0;
  if (M == 0) {
    spgemm_reset_kernel<<<1, kBlockThreads, 0, s>>>(static_cast<int *>(workspace), c_row_ptr, 0, nullptr);
    SCORCH_HIP_CHECK(hipGetLastError());
    return SCORCH_HIP_OK;
  }
  SyncCall sync;
  if (sync.null()) return fail(SCORCH_HIP_ERUNTIME, "%s: no memory for the report", fn);
  const SpgemmWorkspace ws = spgemm_layout(static_cast<char *>(workspace), M, N, elem_size);
  if (int rc = spgemm_run<float, false>((int)M, (int)N, a_row_ptr, a_col_idx, nullptr, b_row_ptr, b_col_idx, nullptr,
                                        c_row_ptr, nullptr, nullptr, ws, s, kShortRows, nullptr, &sync))
    return rc;
  int64_t words[6];
  if (int rc = sync.wait(fn, s, words, 6)) return rc;  // (the short rows' kernels are still at work)
  for (int i = 0; i < 4; ++i) report[1 + i] = words[i];
  report[7] = words[4], report[8] = words[5];
  *bin_bytes = spgemm_bins(nullptr, nullptr, N, elem_size, words[2] + words[3], words[3], words[4], words[5]).total;
  return SCORCH_HIP_OK;
}

#define SCORCH_DEFINE_SPGEMM(SUFFIX, T)                                                             \
  int scorch_hip_spgemm_csr_numeric_##SUFFIX(                                                        \
      int64_t M, int64_t K, int64_t N, const int32_t *a_row_ptr, const int32_t *a_col_idx,           \
      const T *a_vals, const int32_t *b_row_ptr, const int32_t *b_col_idx, const T *b_vals,          \
      const int32_t *c_row_ptr, int32_t *c_col_idx, T *c_vals, void *workspace,                      \
      size_t workspace_bytes, void *stream) {                                                        \
    return scorch::spgemm_numeric_entry<T>("scorch_hip_spgemm_csr_numeric_" #SUFFIX, M, K, N,       \
                                           a_row_ptr, a_col_idx, a_vals, b_row_ptr, b_col_idx,      \
                                           b_vals, c_row_ptr, c_col_idx, c_vals, workspace,         \
                                           workspace_bytes, stream);                                \
  }                                                                                                 \
  int scorch_hip_spgemm_csr_symbolic_planned_##SUFFIX(                                               \
      int64_t M, int64_t K, int64_t N, const int32_t *a_row_ptr, const int32_t *a_col_idx,           \
      const T *a_vals, const int32_t *b_row_ptr, const int32_t *b_col_idx, const T *b_vals,          \
      int32_t *c_row_ptr, void *workspace, size_t workspace_bytes, void *bins, size_t bin_bytes,     \
      int64_t *report, void *stream) {                                                               \
    return scorch::spgemm_symbolic_entry<T>("scorch_hip_spgemm_csr_symbolic_planned_" #SUFFIX, M, K, \
                                            N, a_row_ptr, a_col_idx, a_vals, b_row_ptr, b_col_idx,   \
                                            b_vals, c_row_ptr, workspace, workspace_bytes, bins,     \
                                            bin_bytes, report, stream);                              \
  }                                                                                                 \
  int scorch_hip_spgemm_csr_numeric_planned_##SUFFIX(                                                \
      int64_t M, int64_t K, int64_t N, const int32_t *a_row_ptr, const int32_t *a_col_idx,           \
      const T *a_vals, const int32_t *b_row_ptr, const int32_t *b_col_idx, const T *b_vals,          \
      const int32_t *c_row_ptr, int32_t *c_col_idx, T *c_vals, void *workspace,                      \
      size_t workspace_bytes, void *bins, size_t bin_bytes, const int64_t *report, void *stream) {   \
    SCORCH_REQUIRE(report && report[0] >= 0, "scorch_hip_spgemm_csr_numeric_planned_" #SUFFIX         \
                   ": no report of a symbolic pass");                                               \
    return scorch::spgemm_numeric_entry<T>("scorch_hip_spgemm_csr_numeric_planned_" #SUFFIX, M, K, N, \
                                           a_row_ptr, a_col_idx, a_vals, b_row_ptr, b_col_idx,      \
                                           b_vals, c_row_ptr, c_col_idx, c_vals, workspace,         \
                                           workspace_bytes, stream, report, bins, bin_bytes);       \
  }

SCORCH_DEFINE_SPGEMM(f32, float)
SCORCH_DEFINE_SPGEMM(f64, double)
SCORCH_DEFINE_SPGEMM(i32, int32_t)
SCORCH_DEFINE_SPGEMM(i64, int64_t)

}  // extern "C"

SCORCH_DEFINE_PRELOAD(spgemm)
