// CSR matrix x vector for a matrix that is multiplied many times and whose vector does not fit an
// L2: a copy of the entries, ordered so that the whole chip reads x from one end to the other.
//
// Why.  Every entry gathers one element of x.  With x beyond 4 MB half of those gathers miss their
// XCD's L2, and each miss moves a line of 128 bytes for the 8 (or 4) that are wanted: 1 M rows, 17.8 M
// entries, fp64: 10.9 M misses, 1.4 GB at the fabric's 7.0 TB/s, 198 us for a matrix of 214 MB.
// Passes over parts of the columns read the matrix again for every part and lose what they save.
//
// Copy.  The merged sequence of entries and rows (an entry counts kSweptEntryItems, a row one: bands of
// equal entries, few of which are cut in many short rows) is cut into kSweptBands bands, one for each SIMD
// of the chip.  A band's entries are ordered by windows of columns, half a megabyte of x each, and
// within a window as the matrix has them: 32 bits of row within the band and column, and the value.
// Rows of more than 1 / kSweptCut of a band may be cut by its ends; the parts get every n-th sixteen of the
// row's entries, not a stretch of its columns.
//
// Kernel.  A wavefront reads its band's list from front to back and adds the products up in LDS, a
// double for each of its rows.  All wavefronts start together and have the same number of entries, so
// they are in the same few windows of x at any time, and those are in every L2: x is fetched once
// per XCD.  Nothing waits for anything; a wavefront that falls behind costs misses.
//   The sums are LDS atomics (ds_add_f64: 22 clocks for 64 random rows; ds_add_f32 takes 196) into memory
// that one wavefront alone uses: its instructions add in program order, and the lanes of one
// instruction in the order in which LDS serves them, which has not been seen to change: results repeat
// bit for bit (tested).  fp32 products are added up in fp64.
//   Bound: the L2s' rate for gathered lines, 250 G/s, 71 us of the case above, and the lists' bytes, 40, in part under
// them (a CU's loads return in order: a line from memory holds up those from the L2).  Measured, us, before and after,
// several matrices in turn: fp64, 1 M rows, 17.8 M entries power-law 203 -> 105; 30 M uniform 327 -> 160; 600,000 rows, 12 M
// 95 -> 70; fp32, 17.8 M 129 -> 92.  One matrix again and again: 198 -> 90, 2 M rows, 10 M entries 151 -> 59, fp32 115 -> 78.
// A band to a wavefront, U entries of a lane in flight, one matrix: 4 wavefronts to a SIMD 114, 3: 102, 2: 94, 1: 86 (fp64,
// U = 4, 4, 4, 8; U = 16: 100): more requests in flight spread the wavefronts over more windows and push lines out of
// the L2s.  Lists marked non-temporal: 121 instead of 104 (4 wavefronts).  Rows counted as much as 8 entries: 122 instead
// of 103, bands of unequal entries drift apart.
#include "spmm.hpp"

namespace scorch {

constexpr int kSweptBands = 1024;               // wavefronts, one to a SIMD
constexpr int kSweptSlots = 2048;               // rows whose sums a wavefront holds: 16 KB of LDS
constexpr int kSweptEntryItems = 8;
constexpr int kSweptCut = 16;
constexpr int kSweptColumnBits = 21;            // of an entry's word; the rest is its row within the band
constexpr int kSweptWindows = 64;
constexpr int64_t kSweptMost = 1 << 30;         // entries, rows: sums of an index and a batch stay below 2^31
constexpr int kSweptInFlight = 8;               // consecutive entries that a lane requests together
static_assert(kSweptSlots <= 1 << (32 - kSweptColumnBits), "a row has to fit its bits");

// Columns of a window: a power of two, half a megabyte of x, more where there would be too many of them.
inline int swept_window_shift(int64_t K, size_t elem) {
  int shift = elem == 8 ? 16 : 17;
  while (((K - 1) >> shift) >= kSweptWindows) ++shift;
  return shift;
}

struct SweptShape {
  int64_t items, bands;
};
inline SweptShape swept_shape(int64_t M, int64_t nnz) {
  const int64_t total = M + kSweptEntryItems * nnz;
  int64_t items = (total + kSweptBands - 1) / kSweptBands;
  if (items < 512 * kSweptEntryItems) items = 512 * kSweptEntryItems;
  return {items, (total + items - 1) / items};
}

// The copy's parts within the caller's buffer.
struct Swept {
  Boundary *bands;     // [bands + 1]: first row, first entry
  int *carry_row;      // [bands]: the row that a band leaves unfinished, or -1
  unsigned *entries;   // the bands' lists, one after the other, each from a multiple of four entries (list_start)
  void *vals;
};
inline size_t swept_layout(Swept &s, void *buffer, int64_t M, int64_t nnz, size_t elem) {
  char *p = static_cast<char *>(buffer);
  const int64_t bands = swept_shape(M, nnz).bands;
  const size_t at_rows = align_up((size_t)(bands + 1) * sizeof(Boundary), 256);
  const size_t at_entries = at_rows + align_up((size_t)bands * sizeof(int), 256);
  const size_t listed = (size_t)nnz + 4 * (size_t)bands + 4;  // list_start of a band beyond the last
  const size_t at_vals = at_entries + align_up(listed * sizeof(unsigned), 256);
  s = {reinterpret_cast<Boundary *>(p), reinterpret_cast<int *>(p + at_rows), reinterpret_cast<unsigned *>(p + at_entries), p + at_vals};
  return at_vals + align_up(listed * elem, 256);
}

// ---- the copy -------------------------------------------------------------------------------
// Where band `b` begins.  A boundary inside a row of up to 1 / kSweptCut of a band moves to the row's start.
__global__ __launch_bounds__(kBlockThreads) void spmv_swept_bands_kernel(int M, int64_t nnz, const int *__restrict__ row_ptr,
                                                                         int64_t items, int64_t bands, Boundary *__restrict__ out) {
  const int64_t b = (int64_t)blockIdx.x * kBlockThreads + threadIdx.x;
  if (b > bands) return;
  const int64_t d = b * items;
  int lo = 0, hi = M;  // rows that end at or before d
  while (lo < hi) {
    const int mid = lo + (hi - lo) / 2;
    if ((int64_t)kSweptEntryItems * row_ptr[mid + 1] + mid + 1 <= d) lo = mid + 1;
    else hi = mid;
  }
  Boundary at = {M, (int)nnz};
  if (b < bands && lo < M) {
    const int begin = row_ptr[lo], end = row_ptr[lo + 1];
    const int64_t off = (d - ((int64_t)kSweptEntryItems * begin + lo)) / kSweptEntryItems;  // >= 0: the row before ends at or before d
    if (b == 0) at = {0, 0};
    else if (off >= end - begin) at = {lo + 1, end};
    else if (end - begin <= items / (kSweptCut * kSweptEntryItems)) at = {lo, begin};
    else at = {lo, begin + (int)off};
  }
  out[b] = at;
}

// Where the list of a band lies whose first entry is y0: at a multiple of four entries.
__device__ __forceinline__ int64_t list_start(int64_t band, int y0) { return (((int64_t)y0 + 3) & ~(int64_t)3) + 4 * band; }

// Where the i-th of a list's n elements lies: a lane takes U consecutive ones from a whole batch, W to a request, and the lanes of a
// request read one stretch (a stretch of every second 16 bytes would ask for its lines twice).
template <int W>
__device__ __forceinline__ int swept_place(int i, int n) {
  constexpr int U = kSweptInFlight, kBatch = U * kWaveSize;
  const int base = i / kBatch * kBatch, j = i - base;
  return base + kBatch <= n ? base + (j % U / W * kWaveSize + j / U) * W + j % W : i;
}

// The entry at position p of a row of `len` entries that bands may share: sixteen at a time, every n-th sixteen of the row after one
// another, so that the part of every band spans the row's columns from end to end.
__device__ __forceinline__ int strided_entry(int p, int len) {
  const int groups = len / 16, g = p / 16;
  if (g >= groups) return p;
  const int n = (groups + 7) / 8;                                         // strides, of eight groups
  const int most = (groups + n - 1) / n, rest = groups - (most - 1) * n;  // `rest` of `most` groups, then one less
  int at;
  if (g < rest * most) at = g % most * n + g / most;
  else at = (g - rest * most) % (most - 1) * n + rest + (g - rest * most) / (most - 1);
  return at * 16 + p % 16;
}

// A workgroup to a band, an eighth of its entries to each wavefront: counted by window, then put in their places, in the order they have.
constexpr int kSweptFillWaves = 8;
template <typename T>
__global__ __launch_bounds__(kSweptFillWaves *kWaveSize) void spmv_swept_fill_kernel(
    int M, int64_t items, int shift, const int *__restrict__ row_ptr, const int *__restrict__ col_idx, const T *__restrict__ vals,
    const Boundary *__restrict__ from, int *__restrict__ carry_row, unsigned *__restrict__ entries, T *__restrict__ out_vals) {
  constexpr int kThreads = kSweptFillWaves * kWaveSize;
  __shared__ int s_rp[kSweptSlots + 2];
  __shared__ int s_next[kSweptFillWaves][kSweptWindows];
  static_assert(kSweptWindows == kWaveSize, "a lane to a window");
  const int lane = wave_lane(), w = uniform((int)threadIdx.x / kWaveSize);
  const int64_t band = blockIdx.x;
  const Boundary b0 = load_boundary(from, band), b1 = load_boundary(from, band + 1);
  const int64_t to = list_start(band, b0.y) - b0.y;
  for (int x0 = b0.x; x0 <= b1.x; x0 += kSweptSlots) {  // a part: the rows whose sums fit LDS
    const int n_rows = min(kSweptSlots, b1.x - x0);
    const bool last = x0 + kSweptSlots > b1.x;  // and the row that goes on in the next band
    __syncthreads();
    // s_rp[r]: first entry of the row x0 + r; row n_rows is the one that goes on in the next band
    for (int r = threadIdx.x; r <= n_rows + 1; r += kThreads) s_rp[r] = row_ptr[min(x0 + r, M)];
    s_next[w][lane] = 0;
    __syncthreads();
    const int y0 = max(b0.y, s_rp[0]), y1 = last ? b1.y : s_rp[n_rows];
    if (last && threadIdx.x == 0) carry_row[band] = y1 > max(s_rp[n_rows], y0) ? b1.x : -1;
    auto entry_of = [&](int p, int &row) {  // of position p, and its row within the band
      int lo = 0, hi = n_rows;              // the last row that begins at or before p
      while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (s_rp[mid] <= p) lo = mid;
        else hi = mid - 1;
      }
      row = lo;
      const int begin = s_rp[lo], len = s_rp[lo + 1] - begin;
      return len <= items / (kSweptCut * kSweptEntryItems) ? p : begin + strided_entry(p - begin, len);
    };
    const int each = (y1 - y0 + kThreads - 1) / kThreads * kWaveSize;
    const int mine = min(y0 + w * each, y1), end = min(mine + each, y1);
    for (int p = mine + lane; p < end; p += kWaveSize) {
      int row;
      atomicAdd(&s_next[w][col_idx[entry_of(p, row)] >> shift], 1);
    }
    __syncthreads();
    if (w == 0) {  // counts to places
      int all = 0;
      for (int i = 0; i < kSweptFillWaves; ++i) all += s_next[i][lane];
      int sum = all;
#pragma unroll
      for (int off = 1; off < kWaveSize; off <<= 1) {
        const int other = __shfl_up(sum, off);
        if (lane >= off) sum += other;
      }
      int at = sum - all;
      for (int i = 0; i < kSweptFillWaves; ++i) {
        const int count = s_next[i][lane];
        s_next[i][lane] = at;
        at += count;
      }
    }
    __syncthreads();
    for (int base = mine; base < end; base += kWaveSize) {
      const bool live = base + lane < end;
      int row = 0, k = y0;
      if (live) k = entry_of(base + lane, row);
      const int col = col_idx[k];
      const int window = live ? col >> shift : -1;
      int at = 0;
      for (unsigned long long left = __ballot(live); left;) {  // the windows among the 64, one after the other
        const int one = __shfl(window, __ffsll(left) - 1);
        const unsigned long long same = __ballot(window == one);
        if (window == one) at = s_next[w][one] + __popcll(same & ((1ull << lane) - 1));
        wave_lds_sync();
        if (lane == 0) s_next[w][one] += __popcll(same);
        wave_lds_sync();
        left &= ~same;
      }
      if (live) {
        entries[to + y0 + swept_place<4>(at, y1 - y0)] = (unsigned)row << kSweptColumnBits | (unsigned)col;
        out_vals[to + y0 + swept_place<16 / sizeof(T)>(at, y1 - y0)] = vals[k];
      }
    }
  }
}

// ---- the product ----------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kBlockThreads, 1) void spmv_swept_kernel(int64_t bands, const Boundary *__restrict__ from,
                                                                      const int *__restrict__ row_ptr, const unsigned *__restrict__ entries,
                                                                      const T *__restrict__ vals, const T *__restrict__ x,
                                                                      T *__restrict__ y, double *__restrict__ carry_val) {
  constexpr int U = kSweptInFlight, kWide = 16 / (int)sizeof(T);
  __shared__ double s_y[kWavesPerBlock][kSweptSlots];
  const int lane = wave_lane(), w = threadIdx.x / kWaveSize;
  // (an XCD's bands are neighbours: rows whose columns are neighbours too then share an L2)
  const int64_t band = xcd_contiguous(blockIdx.x, gridDim.x) * kWavesPerBlock + w;
  if (band >= bands) return;  // no workgroup barriers
  const Boundary b0 = load_boundary(from, band), b1 = load_boundary(from, band + 1);
  double *const sums = s_y[w];
  entries += list_start(band, b0.y) - b0.y;
  vals += list_start(band, b0.y) - b0.y;
  int y0 = b0.y;
  for (int x0 = b0.x;; x0 += kSweptSlots) {  // a part (one, unless most rows are empty)
    const bool last = x0 + kSweptSlots > b1.x;
    const int n_rows = last ? b1.x - x0 : kSweptSlots, y1 = last ? b1.y : uniform(row_ptr[x0 + kSweptSlots]);
    if (y0 == y1) {  // rows without entries
      for (int r = lane; r < n_rows; r += kWaveSize) y[x0 + r] = (T)0;
      if (last) return;  // (no row is cut here: carry_row is -1)
      continue;
    }
    for (int r = lane; r <= n_rows && r < kSweptSlots; r += kWaveSize) sums[r] = 0.0;
    wave_lds_sync();
    {
      auto request = [&](int k, unsigned (&e)[U], T (&v)[U]) {  // a lane's U entries follow one another
        if (k + U * kWaveSize <= y1) {
#pragma unroll
          for (int u = 0; u < U; u += 4) *reinterpret_cast<Vec<unsigned, 4> *>(e + u) = load_vec<unsigned, 4>(entries + k + u * kWaveSize + lane * 4);
#pragma unroll
          for (int u = 0; u < U; u += kWide) *reinterpret_cast<Vec<T, kWide> *>(v + u) = load_vec<T, kWide>(vals + k + u * kWaveSize + lane * kWide);
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int at = min(k + lane * U + u, y1 - 1);
            e[u] = entries[at];
            v[u] = vals[at];
          }
        }
      };
      // Entries k .. of the list, which `e` and `v` hold; those behind them are requested into the other two.
      auto step = [&](int k, const unsigned (&e)[U], const T (&v)[U], unsigned (&next_e)[U], T (&next_v)[U]) {
        T xv[U];
        // (whether the list or x is asked for first, us, lists from memory / from the cache in front of it: fp64 17.8 M entries
        // 104 / 88 and 109 / 85, 30 M 161 and 178, fp32 91 / 81 and 90 / 77)
        constexpr bool kListFirst = sizeof(T) == 8;
        if (kListFirst && k + U * kWaveSize < y1) request(k + U * kWaveSize, next_e, next_v);
#pragma unroll
        for (int u = 0; u < U; ++u) xv[u] = x[e[u] & ((1u << kSweptColumnBits) - 1u)];
        if (!kListFirst && k + U * kWaveSize < y1) request(k + U * kWaveSize, next_e, next_v);
        // those of a row are added up before they go to LDS; a lane beyond the list's end has fewer, or none
        const int n = y1 - k - lane * U;
        unsigned r = e[0] >> kSweptColumnBits;
        double sum = (double)v[0] * (double)xv[0];
#pragma unroll
        for (int u = 1; u < U; ++u) {
          if (u >= n) break;
          const unsigned row = e[u] >> kSweptColumnBits;
          const double p = (double)v[u] * (double)xv[u];
          if (row == r) {
            sum += p;
          } else {
            unsafeAtomicAdd(&sums[r], sum);
            r = row;
            sum = p;
          }
        }
        const unsigned first = (unsigned)uniform((int)r);
        if (__all(r == first && n > 0)) {  // a long row's stretch
#pragma unroll
          for (int off = kWaveSize / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
          if (lane == 0) unsafeAtomicAdd(&sums[first], sum);
        } else if (n > 0) {
          unsafeAtomicAdd(&sums[r], sum);
        }
      };
      unsigned e0[U], e1[U];
      T v0[U], v1[U];
      request(y0, e0, v0);
      for (int k = y0;;) {
        step(k, e0, v0, e1, v1);
        if ((k += U * kWaveSize) >= y1) break;
        step(k, e1, v1, e0, v0);
        if ((k += U * kWaveSize) >= y1) break;
      }
    }
    wave_lds_sync();
    for (int r = lane; r < n_rows; r += kWaveSize) y[x0 + r] = (T)sums[r];
    if (last) {
      if (lane == 0) carry_val[band] = sums[n_rows];
      return;
    }
    wave_lds_sync();
    y0 = y1;
  }
}

// What the bands leave of rows that go on in the next one, added to what the row's last band has put into y: a thread to a band, the sums of
// runs of bands that share a row by doubling distances.
template <typename T>
__global__ __launch_bounds__(kSweptBands) void spmv_swept_fold_kernel(int bands, const int *__restrict__ carry_row,
                                                                      const double *__restrict__ carry_val, T *__restrict__ y) {
  __shared__ int s_row[kSweptBands];
  __shared__ double s_sum[kSweptBands];
  const int b = threadIdx.x;
  const int row = b < bands ? carry_row[b] : -1;
  double sum = row >= 0 ? carry_val[b] : 0.0;  // (a band that leaves none has not written one)
  s_row[b] = row;
  for (int off = 1; off < kSweptBands; off <<= 1) {
    s_sum[b] = sum;
    __syncthreads();
    if (row >= 0 && b >= off && s_row[b - off] == row) sum += s_sum[b - off];
    __syncthreads();
  }
  if (row >= 0 && (b + 1 == kSweptBands || s_row[b + 1] != row)) y[row] = (T)((double)y[row] + sum);
}

// Where the copy pays: x beyond what an L2 keeps beside the matrix (fp64, 300,000 columns, 2.4 M entries: 17.0 and 16.9 us; 400,000,
// 2.8 M: 25.1 -> 22.5), and entries enough (500,000 columns, 2 to a row: 12.9 -> 12.0).
inline int swept_recommended(int64_t M, int64_t K, int64_t nnz, size_t elem) {
  return M > 0 && K > 0 && K <= (int64_t)1 << kSweptColumnBits && K * (int64_t)elem > (3 << 20) && nnz >= 2 * K && nnz >= M &&
         nnz <= kSweptMost && M <= kSweptMost;
}

template <typename T>
int swept_args(const char *fn, int64_t M, int64_t K, int64_t nnz, const void *copy, size_t copy_bytes, Swept &s) {
  SCORCH_REQUIRE(M > 0 && K > 0 && nnz > 0 && M < INT32_MAX && nnz <= INT32_MAX, "%s: sizes M=%lld K=%lld nnz=%lld", fn, (long long)M,
                 (long long)K, (long long)nnz);
  if (K > (int64_t)1 << kSweptColumnBits || M > kSweptMost || nnz > kSweptMost)
    return fail(SCORCH_HIP_EUNSUPPORTED, "%s: more than %d columns, or %lld rows or entries", fn, 1 << kSweptColumnBits, (long long)kSweptMost);
  SCORCH_REQUIRE(copy != nullptr && aligned_to(copy, 256), "%s: the copy is NULL or not 256-byte aligned", fn);
  const size_t need = swept_layout(s, const_cast<void *>(copy), M, nnz, sizeof(T));
  if (copy_bytes < need) return fail(SCORCH_HIP_EWORKSPACE, "%s: the copy takes %zu bytes, %zu given", fn, need, copy_bytes);
  return SCORCH_HIP_OK;
}

template <typename T>
int spmv_swept_copy(const char *fn, int64_t M, int64_t K, int64_t nnz, const int32_t *row_ptr, const int32_t *col_idx, const T *vals,
                    void *copy, size_t copy_bytes, void *stream) {
  if (int rc = check_csr_args(fn, M, K, nnz, row_ptr, col_idx, vals)) return rc;
  Swept to;
  if (int rc = swept_args<T>(fn, M, K, nnz, copy, copy_bytes, to)) return rc;
  SCORCH_REQUIRE(aligned_to(vals, sizeof(T)), "%s: values must be aligned to their size", fn);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const SweptShape shape = swept_shape(M, nnz);
  spmv_swept_bands_kernel<<<dim3((unsigned)(shape.bands / kBlockThreads + 1)), kBlockThreads, 0, s>>>((int)M, nnz, row_ptr, shape.items,
                                                                                                     shape.bands, to.bands);
  SCORCH_HIP_CHECK(hipGetLastError());
  spmv_swept_fill_kernel<T><<<dim3((unsigned)shape.bands), kSweptFillWaves * kWaveSize, 0, s>>>(
      (int)M, shape.items, swept_window_shift(K, sizeof(T)), row_ptr, col_idx, vals, to.bands, to.carry_row, to.entries,
      static_cast<T *>(to.vals));
  SCORCH_HIP_CHECK(hipGetLastError());
  return SCORCH_HIP_OK;
}

template <typename T>
int spmv_swept(const char *fn, int64_t M, int64_t K, int64_t nnz, const int32_t *row_ptr, const void *copy, size_t copy_bytes, const T *x, T *y, void *workspace,
               size_t workspace_bytes, int64_t longest_row, void *stream) {
  Swept from;
  if (int rc = swept_args<T>(fn, M, K, nnz, copy, copy_bytes, from)) return rc;
  SCORCH_REQUIRE(x != nullptr && y != nullptr && aligned_to(x, sizeof(T)) && aligned_to(y, sizeof(T)), "%s: x or y is NULL or misaligned", fn);
  const SweptShape shape = swept_shape(M, nnz);
  if (!workspace || workspace_bytes < (size_t)shape.bands * sizeof(double))
    return fail(SCORCH_HIP_EWORKSPACE, "%s: workspace of %zu bytes needed, %zu given", fn, (size_t)shape.bands * sizeof(double),
                workspace ? workspace_bytes : (size_t)0);
  SCORCH_REQUIRE(aligned_to(workspace, sizeof(double)), "%s: the workspace is misaligned", fn);
  hipStream_t s = static_cast<hipStream_t>(stream);
  double *carry_val = static_cast<double *>(workspace);
  mark_launch(s);
  spmv_swept_kernel<T><<<dim3((unsigned)round_up_8((shape.bands + kWavesPerBlock - 1) / kWavesPerBlock)), kBlockThreads, 0, s>>>(
      shape.bands, from.bands, row_ptr, from.entries, static_cast<const T *>(from.vals), x, y, carry_val);
  SCORCH_HIP_CHECK(hipGetLastError());
  mark_launch(s);
  if (longest_row > 0 && longest_row <= shape.items / (kSweptCut * kSweptEntryItems)) return SCORCH_HIP_OK;  // no band ends inside a row
  spmv_swept_fold_kernel<T><<<1, kSweptBands, 0, s>>>((int)shape.bands, from.carry_row, carry_val, y);
  SCORCH_HIP_CHECK(hipGetLastError());
  mark_launch(s);
  return SCORCH_HIP_OK;
}

}  // namespace scorch

extern "C" {

int scorch_hip_spmv_csr_listed_recommended(int64_t M, int64_t K, int64_t nnz, size_t elem_size) {
  return scorch::swept_recommended(M, K, nnz, elem_size);
}
size_t scorch_hip_spmv_csr_listed_bytes(int64_t M, int64_t nnz, size_t elem_size) {
  if (M <= 0 || nnz <= 0 || (elem_size != 4 && elem_size != 8)) return 0;
  scorch::Swept s;
  return scorch::swept_layout(s, nullptr, M, nnz, elem_size);
}
size_t scorch_hip_spmv_csr_listed_workspace_bytes(int64_t M, int64_t nnz) {
  return M <= 0 || nnz <= 0 ? 0 : (size_t)scorch::swept_shape(M, nnz).bands * sizeof(double);
}

#define SCORCH_SWEPT(SUFFIX, T)                                                                                                       \
  int scorch_hip_spmv_csr_listed_copy_##SUFFIX(int64_t M, int64_t K, int64_t nnz, const int32_t *row_ptr, const int32_t *col_idx,        \
                                              const T *vals, void *copy, size_t copy_bytes, void *stream) {                             \
    return scorch::spmv_swept_copy<T>("scorch_hip_spmv_csr_listed_copy_" #SUFFIX, M, K, nnz, row_ptr, col_idx, vals, copy, copy_bytes,   \
                                      stream);                                                                                          \
  }                                                                                                                                     \
  int scorch_hip_spmv_csr_listed_##SUFFIX(int64_t M, int64_t K, int64_t nnz, const int32_t *row_ptr, const void *copy, size_t copy_bytes, const T *x, T *y,      \
                                         void *workspace, size_t workspace_bytes, int64_t longest_row, void *stream) {                  \
    return scorch::spmv_swept<T>("scorch_hip_spmv_csr_listed_" #SUFFIX, M, K, nnz, row_ptr, copy, copy_bytes, x, y, workspace, workspace_bytes,   \
                                 longest_row, stream);                                                                                  \
  }
SCORCH_SWEPT(f32, float)
SCORCH_SWEPT(f64, double)
#undef SCORCH_SWEPT

}  // extern "C"

SCORCH_DEFINE_PRELOAD(spmv_swept)
