// SDDMM for gfx950: out[p] = mask[p] * <A[row_p, :], B[col_p, :]>.
//
// A wavefront takes its mask entries 64 at a time: lane L fetches the coordinates and the mask value
// of entry L (coalesced).  The wavefront is then split into 64 / GS groups of GS lanes; in step s,
// group g computes the dot product of entry g * GS + s, whose two vectors its lanes read in P pieces
// of 16 bytes each (lane t: chunks t, t + GS, ...).  After GS steps lane L keeps the result of entry L
// and the batch is written with one coalesced store.
//
// What bounds it is the rate at which the L2s answer requests for lines (250 G lines a second when a
// table fits an L2, measured with a load-only kernel; 118 G at twice that size, 55 to 58 G beyond), as
// long as enough of them are in flight and the vector ALU does not fall behind:
//  - eight lanes of 16 bytes ask for exactly one line, and a step of eight entries shares its coordinate
//    exchange, its address arithmetic and its reduction among eight entries instead of four;
//  - a request of 64 lanes x 16 bytes occupies a CU's address unit for sixteen cycles however few of its
//    lanes ask for something: A's rows are fetched once per run of entries, into LDS (batch_dots);
//  - B is requested a chunk of steps ahead, coordinates reach a group's lanes by DPP (no LDS pipe), and
//    sums leave it the same way.
// Before (sixteen lanes a row of 64, A's row held in registers, 256 entries to every wavefront), now, us:
// 65,536^2, 64 per row, K = 64, by lists 89.4 -> 65.5; 92,212 x 684, 54 per row, K = 128, coordinates 132 -> 99
// (its 23 M requests for lines at the L2s' 230 G/s); 30,000^2, 16 per row, K = 256 112 -> 66; 20,000^2, 32 per row,
// K = 50 91.6 -> 17.8; 961 x 10,754, 25 per row, K = 64 15.9 -> 4.5.
#include "common.hpp"

namespace scorch {

constexpr int kEntriesPerWave = 256;
constexpr int kBatches = kEntriesPerWave / kWaveSize;

// x of lane s of every lane's group of GS lanes (s a constant once the caller's loop is unrolled).
template <int GS>
__device__ __forceinline__ int group_broadcast(int x, int s) {
#define SCORCH_BROADCAST_CASE(S)                                                                   \
  case S:                                                                                          \
    if constexpr (GS == 16) return __builtin_amdgcn_update_dpp(0, x, 0x150 + S, 0xf, 0xf, false);  \
    if constexpr (GS == 8 && S < 8) {                                                              \
      int low; /* every lane of it is written by one of the two */                                 \
      asm volatile("" : "=v"(low));                                                                         \
      low = __builtin_amdgcn_update_dpp(low, x, 0x150 + (S & 7), 0xf, 0x3, false);                 \
      return __builtin_amdgcn_update_dpp(low, x, 0x158 + (S & 7), 0xf, 0xc, false);                \
    }                                                                                              \
    if constexpr (GS == 4 && S < 4) return __builtin_amdgcn_update_dpp(0, x, (S & 3) * 0x55, 0xf, 0xf, false); \
    return x;
  switch (s) {
    SCORCH_BROADCAST_CASE(0) SCORCH_BROADCAST_CASE(1) SCORCH_BROADCAST_CASE(2) SCORCH_BROADCAST_CASE(3)
    SCORCH_BROADCAST_CASE(4) SCORCH_BROADCAST_CASE(5) SCORCH_BROADCAST_CASE(6) SCORCH_BROADCAST_CASE(7)
    SCORCH_BROADCAST_CASE(8) SCORCH_BROADCAST_CASE(9) SCORCH_BROADCAST_CASE(10) SCORCH_BROADCAST_CASE(11)
    SCORCH_BROADCAST_CASE(12) SCORCH_BROADCAST_CASE(13) SCORCH_BROADCAST_CASE(14) SCORCH_BROADCAST_CASE(15)
  }
#undef SCORCH_BROADCAST_CASE
  return x;
}

template <int CTRL>
__device__ __forceinline__ float dpp_moved(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}

// Sum over the GS lanes of a group, every lane receiving it: exchanges inside a row of 16 lanes only.
template <int GS>
__device__ __forceinline__ float short_group_sum(float x) {
  if constexpr (GS == 16) return group_sum<16>(x);
  x += dpp_moved<0xb1>(x);                          // lane i ^ 1
  x += dpp_moved<0x4e>(x);                          // lane i ^ 2
  if constexpr (GS == 8) x += dpp_moved<0x141>(x);  // the other four lanes of the eight, mirrored
  return x;
}

// LDS of a wavefront for the rows of A that its 64 entries name.
constexpr int kStageFloats = 2048;

// Dot products of 64 entries, one per lane: (row, col) are the lane's entry, the result is its dot
// product.  Every lane's row and col must name existing rows.  4 <= K <= 4 GS P, and more than
// 4 GS (P - 1), or P = 0 for K below 4; TAIL: K is not 4 GS P, the lanes behind the end of a row read
// its last 16 bytes and count what is not theirs as 0 on both sides.
//
// Consecutive entries mostly share their row of A.  The distinct rows of the 64 entries (runs of equal
// rows) are fetched into LDS once, eight to a request, and read from there: a request made for the one
// group whose row changes occupies the address unit as long as one for eight groups, and those requests
// were as many as B's (mask of 65,536^2, 64 per row, K = 64, by lists: 77 us with the row held in
// registers, 66 so; 55 if there were no rows of A to fetch at all).  Where the runs are more than LDS has
// places for every entry fetches its own, as it does where a row is 64 bytes and sixteen entries share a
// step (10 M entries, K = 16: 97 us, staged 109).
template <int GS, int P, bool TAIL>
__device__ __forceinline__ float batch_dots(int row, int col, const float *__restrict__ A, const float *__restrict__ B,
                                            int K, float *__restrict__ stage) {
  const int lane = wave_lane();
  const int t = lane % GS;
  float mine = 0.0f;
  if constexpr (P == 0) {  // K below 4: an element to a lane
#pragma unroll
    for (int s = 0; s < GS; ++s) {
      const int r = group_broadcast<GS>(row, s), c = group_broadcast<GS>(col, s);
      float dot = t < K ? A[(size_t)(unsigned)r * (size_t)(unsigned)K + t] * B[(size_t)(unsigned)c * (size_t)(unsigned)K + t] : 0.0f;
      dot = short_group_sum<GS>(dot);
      if (t == s) mine = dot;
    }
  } else {
    using V4 = Vec<float, 4>;
    constexpr int kWidth = 4 * GS * P;            // floats of a place in LDS
    constexpr int kPlaces = kStageFloats / kWidth < kWaveSize ? kStageFloats / kWidth : kWaveSize;
    constexpr int kGroups = kWaveSize / GS;
    // steps whose rows of B are requested together
    constexpr int kWanted = P == 1 ? 4 : P == 2 ? 2 : 1;
    constexpr int kFlight = kWanted < GS ? kWanted : GS;
    constexpr int kSums = P == 1 ? 1 : P == 2 ? 2 : 4;
    int at[P];
#pragma unroll
    for (int p = 0; p < P; ++p) at[p] = 4 * (t + GS * p);
    int first_own = 0;  // of the last piece's four elements
    if constexpr (TAIL) {
      const int last = K - 4;
      if (at[P - 1] > last) {
        first_own = at[P - 1] - last;
        at[P - 1] = last;
      }
    }
    auto owned = [&](V4 &x) {
      if constexpr (TAIL)
#pragma unroll
        for (int v = 0; v < 4; ++v) x.v[v] = v >= first_own ? x.v[v] : 0.0f;
    };
    auto row_of = [&](const float *X, int r, V4(&x)[P]) {
      const float *from = X + (size_t)(unsigned)r * (size_t)(unsigned)K;
#pragma unroll
      for (int p = 0; p < P; ++p) x[p] = load_vec<float, 4>(from + at[p]);
    };

    constexpr int kChunks = GS / kFlight;
    V4 b[2][kFlight][P];
    auto request = [&](int c) {
#pragma unroll
      for (int u = 0; u < kFlight; ++u) row_of(B, group_broadcast<GS>(col, c * kFlight + u), b[c & 1][u]);
    };
    request(0);

    const int before = __shfl_up(row, 1);  // (by all lanes: lane 1 reads lane 0's)
    const bool head = lane == 0 || row != before;
    const unsigned long long heads = __ballot(head);
    const int runs = __popcll(heads);
    const int run = __builtin_amdgcn_mbcnt_hi((unsigned)(heads >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)heads, 0u)) + (head ? 0 : -1);
    const bool staged = GS > 4 && runs <= kPlaces;
    if (staged) {
      const int run_row = __builtin_amdgcn_ds_permute(run * 4, row);  // lane i: the row of run i
#pragma unroll 2
      for (int first = 0; first < runs; first += kGroups) {
        const int place = first + lane / GS;
        const int r = __shfl(run_row, place);
        if (place < runs) {
          V4 a[P];
          row_of(A, r, a);
          owned(a[P - 1]);
#pragma unroll
          for (int p = 0; p < P; ++p) *reinterpret_cast<V4 *>(stage + place * kWidth + 4 * (t + GS * p)) = a[p];
        }
      }
      wave_lds_sync();
    }
    auto steps = [&](auto from_stage) {
      const int key = from_stage ? run * kWidth : row;
#pragma unroll
      for (int c = 0; c < kChunks; ++c) {
        if (c + 1 < kChunks) request(c + 1);
        V4 a[kFlight][P];
#pragma unroll
        for (int u = 0; u < kFlight; ++u) {
          const int k = group_broadcast<GS>(key, c * kFlight + u);
          if constexpr (from_stage) {
#pragma unroll
            for (int p = 0; p < P; ++p) a[u][p] = *reinterpret_cast<const V4 *>(stage + k + 4 * (t + GS * p));
          } else {
            row_of(A, k, a[u]);
            owned(a[u][P - 1]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);  // (else all chunks' requests move up here, at the price of wavefronts)
#pragma unroll
        for (int u = 0; u < kFlight; ++u) {
          V4(&mine_b)[P] = b[c & 1][u];
          owned(mine_b[P - 1]);
          // (as many roundings deep as a lane of four elements and a wider group: P sums side by side)
          float sum[kSums];
#pragma unroll
          for (int v = 0; v < kSums; ++v) sum[v] = 0.0f;
#pragma unroll
          for (int p = 0; p < P; ++p)
#pragma unroll
            for (int v = 0; v < 4; ++v) sum[v % kSums] = fmaf(a[u][p].v[v], mine_b[p].v[v], sum[v % kSums]);
          float dot = kSums == 1 ? sum[0] : kSums == 2 ? sum[0] + sum[1 % kSums] : (sum[0] + sum[1 % kSums]) + (sum[2 % kSums] + sum[3 % kSums]);
          dot = short_group_sum<GS>(dot);
          if (t == c * kFlight + u) mine = dot;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (staged) steps(std::true_type{}); else steps(std::false_type{});
    wave_lds_sync();
  }
  return mine;
}

// Row of entry p, known to lie in [lo, hi].
__device__ __forceinline__ int sddmm_entry_row(const int *__restrict__ row_ptr, int row_lo, int row_hi, int64_t p) {
  int lo = row_lo, hi = row_hi;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if ((int64_t)row_ptr[mid + 1] <= p) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// A wavefront owns `per_wave` (a multiple of 64, at most kEntriesPerWave) consecutive entries.
//
// With a CSR mask the row of each entry is found by bisection of row_ptr; the wavefront first narrows
// the range to the rows its entries span, so the per-lane search is a few steps.  The same pass can
// write the row of every entry (the coordinate array of the result).
template <int GS, int P, bool TAIL, bool COO>
__global__ __launch_bounds__(kBlockThreads) __attribute__((amdgpu_waves_per_eu(4))) void sddmm_kernel(
    int M, int K, int64_t nnz, int per_wave, const int *__restrict__ rows /* row_idx (COO) or row_ptr (CSR) */,
    const int *__restrict__ col_idx, const float *__restrict__ mask_vals, const float *__restrict__ A,
    const float *__restrict__ B, float *__restrict__ out_vals, int *__restrict__ out_row_idx, int64_t batch_stride_a,
    int64_t batch_stride_b) {
  __shared__ __attribute__((aligned(16))) float s_stage[kWavesPerBlock][P ? kStageFloats : 1];
  const int lane = wave_lane();
  // grid.y > 1: several products over one mask (one per attention head); problem h has its own A,
  // B and result values, the mask's values are shared and the row coordinates are written once
  if (blockIdx.y > 0) {
    A += blockIdx.y * batch_stride_a;
    B += blockIdx.y * batch_stride_b;
    out_vals += blockIdx.y * nnz;
    out_row_idx = nullptr;
  }
  // the grid is a multiple of 8 workgroups; every XCD takes a contiguous eighth of the entries
  const int64_t wave = xcd_contiguous(blockIdx.x, gridDim.x) * kWavesPerBlock + threadIdx.x / kWaveSize;
  const int64_t first = wave * per_wave;
  if (first >= nnz) return;
  const int64_t last = first + per_wave < nnz ? first + per_wave : nnz;

  // everything the piece's entries need to know is requested at once
  int row[kBatches], col[kBatches];
  float scale[kBatches];
#pragma unroll
  for (int i = 0; i < kBatches; ++i) {
    const int64_t p = first + i * kWaveSize + lane;
    const bool valid = p < last;
    col[i] = valid ? col_idx[p] : 0;
    scale[i] = valid && mask_vals ? mask_vals[p] : 1.0f;  // (no value array: every stored entry is 1)
    row[i] = COO && valid ? rows[p] : 0;
  }
  if (!COO) {
    // rows spanned by this wavefront's entries: row(p) = #{i : row_ptr[i+1] <= p}
    auto end_key = [&](int i) { return (int64_t)rows[i + 1]; };
    const int row_lo = wave_count_below(M, first + 1, end_key);
    const int row_hi = row_lo + wave_count_below(M - row_lo, last, [&](int i) { return end_key(row_lo + i); });
#pragma unroll
    for (int i = 0; i < kBatches; ++i) {
      const int64_t p = first + i * kWaveSize + lane;
      if (p < last) row[i] = sddmm_entry_row(rows, row_lo, row_hi, p);
    }
  }
#pragma unroll
  for (int i = 0; i < kBatches; ++i) {
    const int64_t p = first + i * kWaveSize + lane;
    if (p - lane >= last) break;
    const float dot = batch_dots<GS, P, TAIL>(row[i], col[i], A, B, K, s_stage[threadIdx.x / kWaveSize]);
    if (p < last) {
      out_vals[p] = scale[i] * dot;
      if (!COO && out_row_idx) out_row_idx[p] = row[i];
    }
  }
}

// K above 256: all 64 lanes read the vectors of one entry, in pieces of 64 * VEC elements, four at a time,
// all eight loads requested before the first product.
template <int VEC, bool COO>
__global__ __launch_bounds__(kBlockThreads) void sddmm_deep_kernel(
    int M, int K, int64_t nnz, const int *__restrict__ rows, const int *__restrict__ col_idx,
    const float *__restrict__ mask_vals, const float *__restrict__ A, const float *__restrict__ B,
    float *__restrict__ out_vals, int *__restrict__ out_row_idx, int64_t batch_stride_a, int64_t batch_stride_b) {
  using VecT = Vec<float, VEC>;
  const int lane = wave_lane();
  if (blockIdx.y > 0) {
    A += blockIdx.y * batch_stride_a;
    B += blockIdx.y * batch_stride_b;
    out_vals += blockIdx.y * nnz;
    out_row_idx = nullptr;
  }
  const int64_t wave = xcd_contiguous(blockIdx.x, gridDim.x) * kWavesPerBlock + threadIdx.x / kWaveSize;
  const int64_t first = wave * kEntriesPerWave;
  if (first >= nnz) return;
  const int64_t last = first + kEntriesPerWave < nnz ? first + kEntriesPerWave : nnz;

  int row_lo = 0, row_hi = 0;
  if (!COO) {
    auto end_key = [&](int i) { return (int64_t)rows[i + 1]; };
    row_lo = wave_count_below(M, first + 1, end_key);
    row_hi = wave_count_below(M, last, end_key);  // row of entry last - 1
  }

  for (int64_t base = first; base < last; base += kWaveSize) {
    const int64_t p = base + lane;
    const bool valid = p < last;
    int row = 0, col = 0;
    float scale = 0.0f;
    if (valid) {
      col = col_idx[p];
      scale = mask_vals ? mask_vals[p] : 1.0f;
      row = COO ? rows[p] : sddmm_entry_row(rows, row_lo, row_hi, p);
    }

    float mine = 0.0f;
#pragma unroll 4
    for (int s = 0; s < kWaveSize; ++s) {
      const float *a = A + (size_t)__shfl(row, s) * (size_t)K;
      const float *b = B + (size_t)__shfl(col, s) * (size_t)K;
      float dot = 0.0f;
      constexpr int kPieces = 4, kStep = kWaveSize * VEC;
      for (int k0 = lane * VEC; k0 < K; k0 += kPieces * kStep) {
        VecT av[kPieces], bv[kPieces];
#pragma unroll
        for (int u = 0; u < kPieces; ++u) {
          const int k = k0 + u * kStep;
          if (k < K) {
            av[u] = *reinterpret_cast<const VecT *>(a + k);
            bv[u] = *reinterpret_cast<const VecT *>(b + k);
          } else {
#pragma unroll
            for (int v = 0; v < VEC; ++v) av[u].v[v] = bv[u].v[v] = 0.0f;
          }
        }
#pragma unroll
        for (int u = 0; u < kPieces; ++u)
#pragma unroll
          for (int v = 0; v < VEC; ++v) dot += av[u].v[v] * bv[u].v[v];
      }
      dot = group_sum<kWaveSize>(dot);
      if (lane == s) mine = dot;
    }

    if (valid) {
      out_vals[p] = scale * mine;
      if (!COO && out_row_idx) out_row_idx[p] = row;
    }
  }
}

// ---- a mask that is used again and again: its entries listed per XCD ------------------------
// With B larger than one L2 (4 MB per XCD) most of the gathered B rows come over
// the fabric, although all of B would fit the eight L2s together.  For a mask
// whose pattern stays (an attention mask serves every head, layer and step) the
// entries are therefore listed once by the column range they fall in, one range
// per XCD: XCD x then only ever gathers rows of B from its eighth of B, which
// stays in its L2, at the price of every XCD streaming all of A once.
//
// sddmm_bucket_count_kernel / sddmm_bucket_fill_kernel build the lists: each
// wavefront takes kEntriesPerWave consecutive entries (so that a row's entries
// stay together in the lists and its row of A is reused from the vector cache),
// counts them per range (sddmm_bucket_count_kernel), a scan over the wavefronts'
// counts gives every wavefront its place in every list (sddmm_bucket_scan_kernel),
// and the wavefront writes (entry number, row, column) there
// (sddmm_bucket_fill_kernel).  No atomics: the lists come out in entry order, the
// same on every build.
constexpr int kBuckets = 8;  // one per XCD
// Workgroups per XCD of the kernel that walks the lists: a grid that is resident as a whole (four
// wavefronts to a SIMD), workgroup id & 7 being the XCD it runs on (checked against the hardware's
// XCC_ID register: no workgroup of 102,400 was elsewhere).  65,536^2 mask, 64 per row, K = 64: 128 per
// XCD 66 us, 256 (a second half that starts when the first ends) 69; five or six wavefronts to a SIMD with
// fewer registers 77 and 68.
constexpr int kListedWorkgroupsPerXcd = 128;

// counts[b][wave] = entries of the wavefront's piece whose column lies in range b; columns
// outside [0, n_cols) count for no range
__global__ __launch_bounds__(kBlockThreads) void sddmm_bucket_count_kernel(int64_t nnz, int cols_per_bucket,
                                                                           const int *__restrict__ col_idx,
                                                                           int64_t stride, int *__restrict__ counts) {
  const int lane = wave_lane();
  const int64_t wave = (int64_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWaveSize;
  const int64_t first = wave * kEntriesPerWave;
  if (first >= nnz) return;
  const int64_t last = first + kEntriesPerWave < nnz ? first + kEntriesPerWave : nnz;
  int mine[kBuckets] = {0};
  for (int64_t p = first + lane; p < last; p += kWaveSize) {
    const unsigned b = (unsigned)col_idx[p] / (unsigned)cols_per_bucket;
#pragma unroll
    for (int k = 0; k < kBuckets; ++k) mine[k] += b == (unsigned)k;
  }
  int total = 0;  // lane k < kBuckets ends up with range k's count
#pragma unroll
  for (int k = 0; k < kBuckets; ++k) {
    int sum = mine[k];
#pragma unroll
    for (int off = kWaveSize / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if (lane == k) total = sum;
  }
  if (lane < kBuckets) counts[lane * stride + wave] = total;
}

// One workgroup per range: counts[b][piece] becomes the number of range-b entries in the pieces before,
// and totals[b] their number.  A thread takes sixteen consecutive pieces at a time.
// (One workgroup for all ranges, 1,024 pieces at a time, took 130 us for 16,384 pieces; this takes 5.)
constexpr int kScanThreads = 1024;
constexpr int kScanPieces = 16;

__global__ __launch_bounds__(kScanThreads) void sddmm_bucket_scan_kernel(int64_t n_pieces, int64_t stride, int *__restrict__ counts,
                                                                        int *__restrict__ totals) {
  constexpr int kScanWaves = kScanThreads / kWaveSize;
  __shared__ int s_wave_total[kScanWaves];
  const int lane = wave_lane();
  const int w = threadIdx.x / kWaveSize;
  int *mine = counts + blockIdx.x * stride;
  int running = 0;
  for (int64_t base = 0; base < n_pieces; base += kScanThreads * kScanPieces) {
    const int64_t first = base + threadIdx.x * kScanPieces;  // (stride is a multiple of kScanPieces)
    int4 c[kScanPieces / 4];
    int sum = 0;
#pragma unroll
    for (int q = 0; q < kScanPieces / 4; ++q) {
      c[q] = first < n_pieces ? reinterpret_cast<const int4 *>(mine + first)[q] : int4{0, 0, 0, 0};
      if (first + 4 * q + 0 >= n_pieces) c[q].x = 0;
      if (first + 4 * q + 1 >= n_pieces) c[q].y = 0;
      if (first + 4 * q + 2 >= n_pieces) c[q].z = 0;
      if (first + 4 * q + 3 >= n_pieces) c[q].w = 0;
      sum += c[q].x + c[q].y + c[q].z + c[q].w;
    }
    int upto = sum;
#pragma unroll
    for (int off = 1; off < kWaveSize; off <<= 1) {
      const int from_below = __shfl_up(upto, off);
      if (lane >= off) upto += from_below;
    }
    if (lane == kWaveSize - 1) s_wave_total[w] = upto;
    __syncthreads();
    int before = running + upto - sum;
#pragma unroll
    for (int j = 0; j < kScanWaves; ++j) {
      if (j < w) before += s_wave_total[j];
      running += s_wave_total[j];
    }
    __syncthreads();
    if (first < n_pieces) {
#pragma unroll
      for (int q = 0; q < kScanPieces / 4; ++q) {
        int4 at;
        at.x = before;
        at.y = at.x + c[q].x;
        at.z = at.y + c[q].y;
        at.w = at.z + c[q].z;
        before = at.w + c[q].w;
        reinterpret_cast<int4 *>(mine + first)[q] = at;
      }
    }
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = running;
}

// The entries of every piece go to their places in the lists: range b's part of piece `wave`
// starts at list_ptr[b] + offsets[b][wave] (from the scan above), list_ptr[b] being the entries of the
// ranges before; the first workgroup writes list_ptr down (list_ptr[kBuckets] = entries listed).
__global__ __launch_bounds__(kBlockThreads) void sddmm_bucket_fill_kernel(
    int M, int64_t nnz, int cols_per_bucket, const int *__restrict__ row_ptr, const int *__restrict__ col_idx,
    const int *__restrict__ offsets, int64_t stride, const int *__restrict__ totals, int *__restrict__ list_ptr,
    int *__restrict__ entry_pos, int *__restrict__ entry_row, int *__restrict__ entry_col) {
  const int lane = wave_lane();
  const int64_t wave = (int64_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWaveSize;
  const int64_t first = wave * kEntriesPerWave;
  if (first >= nnz) return;
  const int64_t last = first + kEntriesPerWave < nnz ? first + kEntriesPerWave : nnz;
  auto end_key = [&](int i) { return (int64_t)row_ptr[i + 1]; };
  const int row_lo = wave_count_below(M, first + 1, end_key);
  const int row_hi = wave_count_below(M, last, end_key);

  constexpr int kRounds = kEntriesPerWave / kWaveSize;
  int col[kRounds], row[kRounds];
  unsigned bucket[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int64_t p = first + r * kWaveSize + lane;
    bucket[r] = ~0u;
    col[r] = row[r] = 0;
    if (p < last) {
      col[r] = col_idx[p];
      row[r] = sddmm_entry_row(row_ptr, row_lo, row_hi, p);
      bucket[r] = (unsigned)col[r] / (unsigned)cols_per_bucket;
    }
  }
  // every entry's slot: the wavefront's entries keep their order inside a list, so that a row's
  // entries stay next to each other there (its row of A is then staged in LDS once for all of them,
  // and the entry's mask value and result lie next to its neighbours')
  int base[kBuckets];
  int start = 0;
#pragma unroll
  for (int k = 0; k < kBuckets; ++k) {
    if (wave == 0 && lane == 0) list_ptr[k] = start;
    base[k] = start + offsets[k * stride + wave];
    start += totals[k];
  }
  if (wave == 0 && lane == 0) list_ptr[kBuckets] = start;
  const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (kWaveSize - lane));
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
#pragma unroll
    for (int k = 0; k < kBuckets; ++k) {
      const unsigned long long members = __ballot(bucket[r] == (unsigned)k);
      if (bucket[r] == (unsigned)k) {
        const int at = base[k] + __popcll(members & below);
        entry_pos[at] = (int)(first + r * kWaveSize + lane);
        entry_row[at] = row[r];
        entry_col[at] = col[r];
      }
      base[k] += __popcll(members);
    }
  }
}

// The SDDMM proper over such lists.  Workgroup ids are dealt to the XCDs round robin, so
// workgroup id & 7 is the XCD and the range; the XCD's workgroups share out its list in
// pieces of kEntriesPerWave entries.  Everything else as in sddmm_kernel.
template <int GS, int P, bool TAIL>
__global__ __launch_bounds__(kBlockThreads) __attribute__((amdgpu_waves_per_eu(4))) void sddmm_listed_kernel(
    int K, const int *__restrict__ list_ptr, const int *__restrict__ entry_pos,
    const int *__restrict__ entry_row, const int *__restrict__ entry_col,
    const float *__restrict__ mask_vals, const float *__restrict__ listed_vals, const float *__restrict__ A,
    const float *__restrict__ B, float *__restrict__ out_vals, int *__restrict__ out_row_idx, int64_t nnz,
    int64_t batch_stride_a, int64_t batch_stride_b) {
  __shared__ __attribute__((aligned(16))) float s_stage[kWavesPerBlock][P ? kStageFloats : 1];
  if (blockIdx.y > 0) {  // problem blockIdx.y of a batch over one mask
    A += blockIdx.y * batch_stride_a;
    B += blockIdx.y * batch_stride_b;
    out_vals += blockIdx.y * nnz;
    out_row_idx = nullptr;
  }
  const int lane = wave_lane();
  const int xcd = blockIdx.x & 7;
  const int64_t begin = list_ptr[xcd], end = list_ptr[xcd + 1];
  const int64_t batches = (end - begin + kWaveSize - 1) / kWaveSize;
  const int64_t waves = (int64_t)(gridDim.x >> 3) * kWavesPerBlock;
  const int64_t wave = (int64_t)(blockIdx.x >> 3) * kWavesPerBlock + threadIdx.x / kWaveSize;
  const int64_t stop = uniform((int)(batches * (wave + 1) / waves));
  int64_t batch = uniform((int)(batches * wave / waves));
  if (batch >= stop) return;

  const float *vals = listed_vals ? listed_vals : mask_vals;
  struct Entry { int pos, row, col; } now, next;
  auto place = [&](int64_t b) {
    const int64_t e = begin + b * kWaveSize + lane;
    return e < end ? e : end - 1;
  };
  auto request = [&](int64_t b) {
    const int64_t e = place(b);
    return Entry{entry_pos[e], entry_row[e], entry_col[e]};
  };
  auto value = [&](int64_t b, int pos) { return vals ? vals[listed_vals ? place(b) : (int64_t)pos] : 1.0f; };

  now = request(batch);
  next = request(batch + 1 < stop ? batch + 1 : batch);
  float scale = value(batch, now.pos);
  for (; batch < stop; ++batch) {
    const int64_t after = batch + 2 < stop ? batch + 2 : stop - 1, one = batch + 1 < stop ? batch + 1 : batch;
    const Entry later = request(after);
    const float next_scale = value(one, next.pos);
    const float dot = batch_dots<GS, P, TAIL>(now.row, now.col, A, B, K, s_stage[threadIdx.x / kWaveSize]);
    if (begin + batch * kWaveSize + lane < end) {
      // The results are scattered 4-byte writes that nothing reads again: marked as streaming
      // they do not take L2 lines from the XCD's part of B (8 % faster at 65,536^2; the same
      // mark on the loads of the lists or of A made the kernel slower).
      store_streaming(out_vals + now.pos, scale * dot);
      if (out_row_idx) store_streaming(out_row_idx + now.pos, now.row);
    }
    now = next;
    next = later;
    scale = next_scale;
  }
}

// Calls f(GS, P, TAIL) with constants for K up to 256: eight lanes a row, so that a request is a line,
// up to four pieces a lane; sixteen lanes beyond, and four where a row has no more than 64 bytes.
template <typename F>
void with_sddmm_shape(int64_t K, F f) {
  const int64_t chunks = (K + 3) / 4;
#define SCORCH_SDDMM_SHAPE(GS, P)                                                                 \
  do {                                                                                            \
    if (K == 4 * GS * P)                                                                          \
      f(std::integral_constant<int, GS>{}, std::integral_constant<int, P>{}, std::false_type{});  \
    else                                                                                          \
      f(std::integral_constant<int, GS>{}, std::integral_constant<int, P>{}, std::true_type{});   \
  } while (0)
  if (K < 4) f(std::integral_constant<int, 4>{}, std::integral_constant<int, 0>{}, std::false_type{});
  else if (chunks <= 4) SCORCH_SDDMM_SHAPE(4, 1);
  else if (chunks <= 8) SCORCH_SDDMM_SHAPE(8, 1);
  else if (chunks <= 16) SCORCH_SDDMM_SHAPE(8, 2);
  else if (chunks <= 24) SCORCH_SDDMM_SHAPE(8, 3);
  else if (chunks <= 32) SCORCH_SDDMM_SHAPE(8, 4);
  else if (chunks <= 48) SCORCH_SDDMM_SHAPE(16, 3);
  else SCORCH_SDDMM_SHAPE(16, 4);
#undef SCORCH_SDDMM_SHAPE
}

constexpr int64_t kSddmmWavefronts = 4096;  // four to a SIMD

template <bool COO>
int launch_sddmm(int M, int K, int64_t nnz, const int *rows, const int *col_idx,
                 const float *mask_vals, const float *A, const float *B, float *out_vals,
                 int *out_row_idx, hipStream_t stream, int batch = 1, int64_t batch_stride_a = 0,
                 int64_t batch_stride_b = 0) {
  mark_launch(stream);
  if (K <= 256) {
    // shorter pieces where 256 entries to a wavefront would leave SIMDs without work
    int per_wave = kEntriesPerWave;
    while (per_wave > kWaveSize && nnz * batch < (int64_t)per_wave * kSddmmWavefronts) per_wave /= 2;
    const int64_t waves = (nnz + per_wave - 1) / per_wave;
    const dim3 grid((unsigned)round_up_8((waves + kWavesPerBlock - 1) / kWavesPerBlock), (unsigned)batch);
    with_sddmm_shape(K, [&](auto gs, auto pieces, auto tail) {
      sddmm_kernel<gs(), pieces(), tail(), COO><<<grid, kBlockThreads, 0, stream>>>(
          M, K, nnz, per_wave, rows, col_idx, mask_vals, A, B, out_vals, out_row_idx, batch_stride_a, batch_stride_b);
    });
  } else {
    const int64_t waves = (nnz + kEntriesPerWave - 1) / kEntriesPerWave;
    const dim3 grid((unsigned)round_up_8((waves + kWavesPerBlock - 1) / kWavesPerBlock), (unsigned)batch);
    auto kernel = K % 4 == 0 && aligned_to(A, 16) && aligned_to(B, 16) ? &sddmm_deep_kernel<4, COO> : &sddmm_deep_kernel<1, COO>;
    kernel<<<grid, kBlockThreads, 0, stream>>>(M, K, nnz, rows, col_idx, mask_vals, A, B, out_vals, out_row_idx,
                                               batch_stride_a, batch_stride_b);
  }
  SCORCH_HIP_CHECK(hipGetLastError());
  mark_launch(stream);
  return SCORCH_HIP_OK;
}

template <bool COO>
int sddmm_entry(const char *fn, int64_t M, int64_t n_cols, int64_t K, int64_t nnz,
                const int32_t *rows, const int32_t *col_idx, const float *mask_vals,
                const float *A, const float *B, float *out_vals, int32_t *out_row_idx,
                void *stream, int64_t batch = 1) {
  if (batch < 0 || batch > 65535)
    return fail(SCORCH_HIP_EUNSUPPORTED, "%s: batch=%lld is outside [0, 65535]", fn, (long long)batch);
  if (batch == 0) return SCORCH_HIP_OK;
  if (M < 0 || n_cols < 0 || K < 0 || nnz < 0)
    return fail(SCORCH_HIP_EINVAL, "%s: negative size (M=%lld n_cols=%lld K=%lld nnz=%lld)", fn,
                (long long)M, (long long)n_cols, (long long)K, (long long)nnz);
  if (M >= INT32_MAX || n_cols > INT32_MAX || K > INT32_MAX || nnz > INT32_MAX)
    return fail(SCORCH_HIP_EUNSUPPORTED, "%s: sizes must fit int32 indices", fn);
  SCORCH_REQUIRE(COO || rows != nullptr, "%s: row_ptr is NULL", fn);
  if (nnz == 0) return SCORCH_HIP_OK;
  SCORCH_REQUIRE(M > 0 && n_cols > 0, "%s: nnz=%lld in an empty mask", fn, (long long)nnz);
  SCORCH_REQUIRE(rows && col_idx && out_vals, "%s: NULL index/value array", fn);
  SCORCH_REQUIRE(K == 0 || (A && B), "%s: NULL dense operand", fn);
  SCORCH_REQUIRE(aligned_to(rows, 4) && aligned_to(col_idx, 4) && aligned_to(mask_vals, 4) &&
                     aligned_to(out_vals, 4) && aligned_to(A, 4) && aligned_to(B, 4) &&
                     aligned_to(out_row_idx, 4),
                 "%s: arrays must be 4-byte aligned", fn);
  return launch_sddmm<COO>((int)M, (int)K, nnz, rows, col_idx, mask_vals, A, B, out_vals,
                           out_row_idx, static_cast<hipStream_t>(stream), (int)batch, M * K, n_cols * K);
}

inline size_t align_up_256(size_t v) { return (v + 255) / 256 * 256; }

// Layout of the per-XCD entry lists inside the caller's buffer.
struct SddmmLists {
  int *list_ptr;   // [9]
  int *entry_pos, *entry_row, *entry_col;  // [nnz] each
  int *totals;        // [kBuckets] and
  int *offsets;       // [kBuckets][stride of sddmm_piece_stride]: used while the lists are built
};

inline int64_t sddmm_pieces(int64_t nnz) { return (nnz + kEntriesPerWave - 1) / kEntriesPerWave; }

inline int64_t sddmm_piece_stride(int64_t nnz) { return (sddmm_pieces(nnz) + kScanPieces - 1) / kScanPieces * kScanPieces; }

inline SddmmLists sddmm_lists(void *buffer, int64_t nnz) {
  char *base = static_cast<char *>(buffer);
  const size_t array = align_up_256((size_t)nnz * sizeof(int32_t));
  SddmmLists l;
  l.list_ptr = reinterpret_cast<int *>(base) + 16;
  l.entry_pos = reinterpret_cast<int *>(base + 256);
  l.entry_row = reinterpret_cast<int *>(base + 256 + array);
  l.entry_col = reinterpret_cast<int *>(base + 256 + 2 * array);
  l.totals = reinterpret_cast<int *>(base) + 32;
  l.offsets = reinterpret_cast<int *>(base + 256 + 3 * array);
  return l;
}

// listed_vals[e] = vals[entry_pos[e]]: the mask's values in the order of the lists.
__global__ __launch_bounds__(kBlockThreads) void sddmm_list_values_kernel(int64_t nnz, const int *__restrict__ entry_pos,
                                                                           const float *__restrict__ vals,
                                                                           float *__restrict__ listed_vals) {
  const int64_t stride = (int64_t)gridDim.x * kBlockThreads;
  for (int64_t e = (int64_t)blockIdx.x * kBlockThreads + threadIdx.x; e < nnz; e += stride)
    listed_vals[e] = vals[entry_pos[e]];
}

__global__ void sddmm_lists_clear_kernel(int *list_ptr) {
  if (threadIdx.x <= kBuckets) list_ptr[threadIdx.x] = 0;
}

}  // namespace scorch

extern "C" {

int scorch_hip_sddmm_coo_f32(int64_t M, int64_t n_cols, int64_t K, int64_t nnz,
                             const int32_t *row_idx, const int32_t *col_idx,
                             const float *mask_vals, const float *A, const float *B,
                             float *out_vals, void *stream) {
  return scorch::sddmm_entry<true>("scorch_hip_sddmm_coo_f32", M, n_cols, K, nnz, row_idx, col_idx,
                                   mask_vals, A, B, out_vals, nullptr, stream);
}

int scorch_hip_sddmm_csr_f32(int64_t M, int64_t n_cols, int64_t K, int64_t nnz,
                             const int32_t *row_ptr, const int32_t *col_idx,
                             const float *mask_vals, const float *A, const float *B,
                             float *out_vals, int32_t *out_row_idx, void *stream) {
  return scorch::sddmm_entry<false>("scorch_hip_sddmm_csr_f32", M, n_cols, K, nnz, row_ptr,
                                    col_idx, mask_vals, A, B, out_vals, out_row_idx, stream);
}

int scorch_hip_sddmm_csr_batched_f32(int64_t batch, int64_t M, int64_t n_cols, int64_t K, int64_t nnz,
                                     const int32_t *row_ptr, const int32_t *col_idx, const float *mask_vals,
                                     const float *A, const float *B, float *out_vals, int32_t *out_row_idx,
                                     void *stream) {
  return scorch::sddmm_entry<false>("scorch_hip_sddmm_csr_batched_f32", M, n_cols, K, nnz, row_ptr, col_idx,
                                    mask_vals, A, B, out_vals, out_row_idx, stream, batch);
}

// B beyond one L2 (4 MiB) and within the eight together, and its rows used often enough.  Where B is 4 MiB the plain kernel
// is as fast (20,000 columns, 600 K entries, K = 50: 17.8 us, by lists 18.0), at 4.9 MiB it no longer is (4 M entries,
// K = 64: 72.7 against 65.1; 6.1 MiB, 10 M entries, K = 16: 99 against 73).
int scorch_hip_sddmm_csr_lists_recommended(int64_t n_cols, int64_t K, int64_t nnz) {
  constexpr int64_t kLeastB = (int64_t)9 << 19, kMostB = (int64_t)20 << 20;  // bytes
  if (K <= 0 || K > 256 || n_cols <= 0 || n_cols > kMostB) return 0;
  const int64_t bytes = n_cols * K * (int64_t)sizeof(float);
  return bytes >= kLeastB && bytes <= kMostB && nnz >= 4 * n_cols;
}

size_t scorch_hip_sddmm_csr_lists_bytes(int64_t nnz) {
  if (nnz < 0) return 0;
  // the 9 list starts (256 bytes), entry numbers, rows and columns, and the per-piece offsets the
  // build works with
  return 256 + 3 * scorch::align_up_256((size_t)nnz * sizeof(int32_t)) +
         scorch::align_up_256((size_t)scorch::sddmm_piece_stride(nnz) * scorch::kBuckets * sizeof(int32_t));
}

int scorch_hip_sddmm_csr_lists(int64_t M, int64_t n_cols, int64_t nnz, const int32_t *row_ptr,
                               const int32_t *col_idx, void *lists, size_t lists_bytes, void *stream) {
  const char *fn = "scorch_hip_sddmm_csr_lists";
  if (M < 0 || n_cols < 0 || nnz < 0)
    return scorch::fail(SCORCH_HIP_EINVAL, "%s: negative size (M=%lld n_cols=%lld nnz=%lld)", fn, (long long)M,
                        (long long)n_cols, (long long)nnz);
  if (M >= INT32_MAX || n_cols > INT32_MAX || nnz > INT32_MAX)
    return scorch::fail(SCORCH_HIP_EUNSUPPORTED, "%s: sizes must fit int32 indices", fn);
  SCORCH_REQUIRE(row_ptr != nullptr && lists != nullptr, "%s: row_ptr or lists is NULL", fn);
  SCORCH_REQUIRE(nnz == 0 || col_idx != nullptr, "%s: col_idx is NULL", fn);
  SCORCH_REQUIRE(scorch::aligned_to(row_ptr, 4) && scorch::aligned_to(col_idx, 4) && scorch::aligned_to(lists, 256),
                 "%s: index arrays must be 4-byte and lists 256-byte aligned", fn);
  if (lists_bytes < scorch_hip_sddmm_csr_lists_bytes(nnz))
    return scorch::fail(SCORCH_HIP_EWORKSPACE, "%s: %zu bytes needed for the lists, %zu given", fn,
                        scorch_hip_sddmm_csr_lists_bytes(nnz), lists_bytes);
  hipStream_t s = static_cast<hipStream_t>(stream);
  scorch::SddmmLists l = scorch::sddmm_lists(lists, nnz);
  if (nnz == 0 || n_cols == 0) {
    scorch::sddmm_lists_clear_kernel<<<1, 64, 0, s>>>(l.list_ptr);
    SCORCH_HIP_CHECK(hipGetLastError());
    return SCORCH_HIP_OK;
  }
  const int cols_per_bucket = (int)((n_cols + scorch::kBuckets - 1) / scorch::kBuckets);
  const int64_t waves = scorch::sddmm_pieces(nnz);
  const dim3 grid((unsigned)((waves + scorch::kWavesPerBlock - 1) / scorch::kWavesPerBlock));
  const int64_t stride = scorch::sddmm_piece_stride(nnz);
  scorch::sddmm_bucket_count_kernel<<<grid, scorch::kBlockThreads, 0, s>>>(nnz, cols_per_bucket, col_idx, stride,
                                                                          l.offsets);
  SCORCH_HIP_CHECK(hipGetLastError());
  scorch::sddmm_bucket_scan_kernel<<<scorch::kBuckets, scorch::kScanThreads, 0, s>>>(waves, stride, l.offsets, l.totals);
  SCORCH_HIP_CHECK(hipGetLastError());
  scorch::sddmm_bucket_fill_kernel<<<grid, scorch::kBlockThreads, 0, s>>>(
      (int)M, nnz, cols_per_bucket, row_ptr, col_idx, l.offsets, stride, l.totals, l.list_ptr, l.entry_pos, l.entry_row,
      l.entry_col);
  SCORCH_HIP_CHECK(hipGetLastError());
  return SCORCH_HIP_OK;
}

int scorch_hip_sddmm_csr_list_values_f32(int64_t nnz, const void *lists, size_t lists_bytes, const float *vals,
                                         float *listed_vals, void *stream) {
  const char *fn = "scorch_hip_sddmm_csr_list_values_f32";
  if (nnz < 0) return scorch::fail(SCORCH_HIP_EINVAL, "%s: negative size", fn);
  if (nnz > INT32_MAX) return scorch::fail(SCORCH_HIP_EUNSUPPORTED, "%s: sizes must fit int32 indices", fn);
  if (nnz == 0) return SCORCH_HIP_OK;
  SCORCH_REQUIRE(lists && vals && listed_vals, "%s: NULL array", fn);
  SCORCH_REQUIRE(scorch::aligned_to(lists, 256) && scorch::aligned_to(vals, 4) && scorch::aligned_to(listed_vals, 4),
                 "%s: lists must be 256-byte aligned, the value arrays 4-byte", fn);
  if (lists_bytes < scorch_hip_sddmm_csr_lists_bytes(nnz))
    return scorch::fail(SCORCH_HIP_EWORKSPACE, "%s: the lists of %lld entries take %zu bytes, %zu given", fn,
                        (long long)nnz, scorch_hip_sddmm_csr_lists_bytes(nnz), lists_bytes);
  const scorch::SddmmLists l = scorch::sddmm_lists(const_cast<void *>(lists), nnz);
  int64_t blocks = (nnz + scorch::kBlockThreads * 4 - 1) / (scorch::kBlockThreads * 4);
  if (blocks > 8192) blocks = 8192;  // the kernel strides
  scorch::sddmm_list_values_kernel<<<dim3((unsigned)blocks), scorch::kBlockThreads, 0,
                                     static_cast<hipStream_t>(stream)>>>(nnz, l.entry_pos, vals, listed_vals);
  SCORCH_HIP_CHECK(hipGetLastError());
  return SCORCH_HIP_OK;
}

int scorch_hip_sddmm_csr_listed_f32(int64_t batch, int64_t M, int64_t n_cols, int64_t K, int64_t nnz,
                                    const void *lists, size_t lists_bytes, const float *mask_vals,
                                    const float *listed_vals, const float *A, const float *B, float *out_vals,
                                    int32_t *out_row_idx, void *stream) {
  const char *fn = "scorch_hip_sddmm_csr_listed_f32";
  if (batch < 0 || batch > 65535)
    return scorch::fail(SCORCH_HIP_EUNSUPPORTED, "%s: batch=%lld is outside [0, 65535]", fn, (long long)batch);
  if (M < 0 || n_cols < 0 || K < 0 || nnz < 0)
    return scorch::fail(SCORCH_HIP_EINVAL, "%s: negative size (M=%lld n_cols=%lld K=%lld nnz=%lld)", fn,
                        (long long)M, (long long)n_cols, (long long)K, (long long)nnz);
  if (M >= INT32_MAX || n_cols > INT32_MAX || K > INT32_MAX || nnz > INT32_MAX)
    return scorch::fail(SCORCH_HIP_EUNSUPPORTED, "%s: sizes must fit int32 indices", fn);
  if (batch == 0 || nnz == 0) return SCORCH_HIP_OK;
  SCORCH_REQUIRE(lists && out_vals, "%s: NULL lists or value array", fn);
  SCORCH_REQUIRE(K == 0 || (A && B), "%s: NULL dense operand", fn);
  SCORCH_REQUIRE(scorch::aligned_to(lists, 256) && scorch::aligned_to(mask_vals, 4) && scorch::aligned_to(listed_vals, 4) &&
                     scorch::aligned_to(out_vals, 4) &&
                     scorch::aligned_to(A, 4) && scorch::aligned_to(B, 4) && scorch::aligned_to(out_row_idx, 4),
                 "%s: lists must be 256-byte aligned, the other arrays 4-byte", fn);
  if (lists_bytes < scorch_hip_sddmm_csr_lists_bytes(nnz))
    return scorch::fail(SCORCH_HIP_EWORKSPACE, "%s: lists of %zu bytes expected, %zu given", fn,
                        scorch_hip_sddmm_csr_lists_bytes(nnz), lists_bytes);
  if (K > 256)
    return scorch::fail(SCORCH_HIP_EUNSUPPORTED, "%s: K=%lld beyond 256 is served by scorch_hip_sddmm_csr_f32 only", fn,
                        (long long)K);
  const scorch::SddmmLists l = scorch::sddmm_lists(const_cast<void *>(lists), nnz);
  hipStream_t s = static_cast<hipStream_t>(stream);
  // a resident grid: every XCD's workgroups walk that XCD's list
  const int64_t waves = (nnz / scorch::kBuckets + scorch::kEntriesPerWave - 1) / scorch::kEntriesPerWave + 1;
  int64_t wgs = (waves + scorch::kWavesPerBlock - 1) / scorch::kWavesPerBlock;
  if (wgs > scorch::kListedWorkgroupsPerXcd) wgs = scorch::kListedWorkgroupsPerXcd;
  const dim3 grid((unsigned)(wgs * 8), (unsigned)batch);
  scorch::mark_launch(s);
  scorch::with_sddmm_shape(K, [&](auto gs, auto pieces, auto tail) {
    scorch::sddmm_listed_kernel<gs(), pieces(), tail()><<<grid, scorch::kBlockThreads, 0, s>>>(
        (int)K, l.list_ptr, l.entry_pos, l.entry_row, l.entry_col, mask_vals, listed_vals, A, B, out_vals, out_row_idx,
        nnz, M * K, n_cols * K);
  });
  SCORCH_HIP_CHECK(hipGetLastError());
  scorch::mark_launch(s);
  return SCORCH_HIP_OK;
}

}  // extern "C"

SCORCH_DEFINE_PRELOAD(sddmm)
