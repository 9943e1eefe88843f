// SpMM with the dense operand in LDS: C = act(A * B + bias), fp32, for a matrix A of few columns and
// many entries -- a sparse weight matrix -- whose rows are about equally long.
//
// The other kernels gather rows of B out of the L2s, which hand out 15 TB/s: nnz * N * 4 bytes, 215 MB
// for 1,024 rows of 205 entries at N = 256.  Here a workgroup keeps a panel of B -- all K rows, P
// columns, K * P * 4 bytes of a CU's 160 KB -- and takes a share of A's rows past it; an entry costs
// its 8 bytes of A from the L2 and P * 4 bytes from LDS.  A panel of B is P columns, so a B that is
// handed over as its transpose (the usual W @ x.T) is read where it lies, P rows of x at a time.
//
// A row is a wavefront's, P / 4 lanes to an entry with 16 bytes each.  The next entries, or the next row's
// first, are on their way while those at hand are used: with four or eight lanes to an entry they
// come one to a lane and go through a strip of LDS of the wavefront's own, from which the lanes that
// share one read it (a load for every share fetches 32 bytes at a time: 88 -> 63 us for 8,192 rows of
// 50, N = 1,024); with one or two lanes to an entry every lane loads what it uses, four or eight
// entries at a time.  At the end of a row the partial sums are added up by exchanging halves: a
// lane keeps two of its four columns, then one, so that the last steps move one value.
//
// The panel's LDS reads are at random rows, so the entries that one access serves fall on the
// same banks now and then (1,024 x 4,096, 205 k entries, N = 256: 58 bytes a clock and CU at P = 8, 42 % of the
// cycles conflicts; at P = 32 17 %); wider panels lose less to that and read A
// less often, and they take more LDS per row of B.  The LDS is busy for half of a launch: the rest is
// the panel's way into it, the entries' loads and the end of every row.  The host picks P and the number of row shares
// from K, N and nnz.
#include <atomic>

#include "spmm.hpp"

namespace scorch {

constexpr int kPanelThreads = 1024;
constexpr int kPanelLds = 160 * 1024;

constexpr int kPanelWaves = kPanelThreads / kWaveSize;

template <int P, int R>
__global__ __launch_bounds__(kPanelThreads) void spmm_panels_kernel(
    int M, int K, int N, const int *__restrict__ row_ptr, const int *__restrict__ col_idx,
    const float *__restrict__ vals, const float *__restrict__ B, int transposed, const float *__restrict__ bias,
    int relu, float *__restrict__ C, int n_panels, int shares, int rows_per_share) {
  constexpr int LPE = P / 4;              // lanes to an entry
  constexpr int SLOTS = kWaveSize / LPE;  // entries a wavefront takes at once
  constexpr bool STAGED = LPE >= 4;
  constexpr int APART = STAGED ? kWaveSize : SLOTS;  // a lane's R entries
  constexpr int BATCH = R * APART;
  constexpr int STEPS = BATCH / SLOTS;
  extern __shared__ float4 s_panel[];     // [K + 1][LPE], row K is zero; then the wavefronts' strips
  int2 *strip = reinterpret_cast<int2 *>(s_panel + (size_t)(K + 1) * LPE) + (threadIdx.x / kWaveSize) * 2 * BATCH;

  const int id = (int)xcd_contiguous(blockIdx.x, gridDim.x);
  const int panel = id / shares, share = id % shares;
  if (panel >= n_panels) return;
  const int n0 = panel * P;
  const int row_end = min(M, (share + 1) * rows_per_share);
  const int lane = wave_lane(), slot = lane / LPE, part = lane % LPE;

  // The wavefront's rows are first, first + 16, ...; lane i holds the i-th's pointers, 64 rows at a time.
  int row = uniform(share * rows_per_share + (int)threadIdx.x / kWaveSize);
  int held = 0, held_begin = 0, held_end = 0;
  auto hold = [&](int from) {
    const int r = from + lane * kPanelWaves;
    held_begin = r < row_end ? row_ptr[r] : 0;
    held_end = r < row_end ? row_ptr[r + 1] : 0;
  };
  int c[R];
  float a[R];
  auto load_entries = [&](int first, int end) {
#pragma unroll
    for (int e = 0; e < R; ++e) {
      const int p = first + (STAGED ? lane : slot) + e * APART;
      const bool ok = p < end;
      c[e] = ok ? col_idx[p] : K;
      a[e] = ok ? vals[p] : 0.0f;
    }
  };
  hold(row);
  int begin = __builtin_amdgcn_readlane(held_begin, 0), end = __builtin_amdgcn_readlane(held_end, 0);
  load_entries(begin, end);

  if (transposed) {  // B[k][n] lies at n * K + k
    constexpr int AHEAD = 32 / P;  // 32 loads in flight
    const int columns = min(P, N - n0);
    for (int k0 = threadIdx.x; k0 < K; k0 += AHEAD * kPanelThreads) {
      float v[AHEAD][P];
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) {
        const int k = min(k0 + i * kPanelThreads, K - 1);
#pragma unroll
        for (int j = 0; j < P; ++j) v[i][j] = j < columns ? B[(size_t)(n0 + j) * (size_t)K + k] : 0.0f;
      }
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) {
        const int k = min(k0 + i * kPanelThreads, K - 1);
#pragma unroll
        for (int l = 0; l < LPE; ++l)
          s_panel[k * LPE + l] = make_float4(v[i][4 * l], v[i][4 * l + 1], v[i][4 * l + 2], v[i][4 * l + 3]);
      }
    }
  } else {
    for (int i = threadIdx.x; i < K * LPE; i += kPanelThreads) {
      const int k = i / LPE, col = n0 + i % LPE * 4;
      const float *from = B + (size_t)k * (size_t)N + col;
      float4 x = make_float4(0, 0, 0, 0);
      if (col + 4 <= N) {
        const Vec<float, 4> v = load_vec<float, 4>(from);
        x = make_float4(v.v[0], v.v[1], v.v[2], v.v[3]);
      } else {
        if (col < N) x.x = from[0];
        if (col + 1 < N) x.y = from[1];
        if (col + 2 < N) x.z = from[2];
      }
      s_panel[i] = x;
    }
  }
  if (threadIdx.x < LPE) s_panel[K * LPE + threadIdx.x] = make_float4(0, 0, 0, 0);
  __syncthreads();

  // (k: the first entry of the batch in c and a; begin, end: its row's)
  int k = begin, buffer = 0;
  float acc[4] = {0, 0, 0, 0};
  while (row < row_end) {
    int cc[R];
    float aa[R];
#pragma unroll
    for (int e = 0; e < R; ++e) {
      if constexpr (STAGED) strip[buffer * BATCH + e * kWaveSize + lane] = make_int2(c[e], __builtin_bit_cast(int, a[e]));
      cc[e] = c[e], aa[e] = a[e];
    }
    k += BATCH;
    const bool row_done = k >= end;
    const int this_row = row;
    if (row_done) {
      row += kPanelWaves;
      if (++held == kWaveSize && row < row_end) {
        hold(row);
        held = 0;
      }
      begin = __builtin_amdgcn_readlane(held_begin, held & (kWaveSize - 1));
      end = __builtin_amdgcn_readlane(held_end, held & (kWaveSize - 1));
      k = begin;
    }
    if (row < row_end) load_entries(k, end);
    if constexpr (STAGED) wave_lds_sync();
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
      int col;
      float v;
      if constexpr (STAGED) {
        const int2 entry = strip[buffer * BATCH + u * SLOTS + slot];
        col = entry.x, v = __builtin_bit_cast(float, entry.y);
      } else {
        col = cc[u], v = aa[u];
      }
      const float4 b = s_panel[col * LPE + part];
      acc[0] += v * b.x;
      acc[1] += v * b.y;
      acc[2] += v * b.z;
      acc[3] += v * b.w;
    }
    buffer ^= 1;
    if (!row_done) continue;
    // slots whose lowest bit is set keep columns 2 and 3 of their four; those with the next bit set the odd one of two
    const bool upper = slot & 1, odd = slot & 2;
    float two[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
      two[j] = (upper ? acc[2 + j] : acc[j]) + __shfl_xor(upper ? acc[j] : acc[2 + j], LPE);
    float sum = (odd ? two[1] : two[0]) + __shfl_xor(odd ? two[0] : two[1], 2 * LPE);
#pragma unroll
    for (int off = 4 * LPE; off < kWaveSize; off <<= 1) sum += __shfl_xor(sum, off);
    const int col = n0 + part * 4 + (upper ? 2 : 0) + (odd ? 1 : 0);
    if (slot < 4 && col < N) {
      if (bias) sum += bias[col];
      if (relu) sum = sum > 0.0f ? sum : 0.0f;
      C[(size_t)this_row * (size_t)N + col] = sum;
    }
    acc[0] = acc[1] = acc[2] = acc[3] = 0.0f;
  }
}

struct PanelShape {
  int width;     // 0: nothing fits
  int in_flight; // entries to a lane
  int shares;    // of A's rows
  double us;     // estimated
};

inline int64_t panel_lds(int64_t K, int width, int in_flight) {
  return (K + 1) * width * 4 + (width >= 16 ? kPanelWaves * 2 * kWaveSize * in_flight * 8 : 0);
}

// Panel width and row shares with the least estimated time: rounds of workgroups (one to a CU, or two of
// half its LDS), each a panel's load at 24 bytes a clock and its share of the entries, in clocks each what
// LDS takes for their pieces of B, and of the rows.
inline PanelShape panel_shape(int64_t M, int64_t K, int64_t N, int64_t nnz) {
  PanelShape best = {0, 0, 0, 0};
  if (M <= 0 || N <= 0 || K > kPanelLds / 16) return best;
  const int64_t mean = (nnz + M - 1) / M;
  for (int width : {32, 16, 8, 4}) {
    const int in_flight = width >= 16 ? 1 : width == 8 ? (mean > 192 ? 8 : 4) : mean > 256 ? 8 : mean > 128 ? 4 : 2;
    const int64_t lds = panel_lds(K, width, in_flight);
    if (lds > kPanelLds) continue;
    const int64_t batch = width >= 16 ? kWaveSize : kWaveSize / (width / 4) * in_flight;
    const double per_entry = width == 32 ? 1.55 : width == 16 ? 1.1 : width == 8 ? 0.57 : 0.30;
    const double work = (double)M * ((double)((mean + batch - 1) / batch * batch) * per_entry + 50);
    const int64_t per_cu = lds <= kPanelLds / 2 ? 2 : 1, slots = 256 * per_cu, panels = (N + width - 1) / width;
    for (int64_t shares = 1; shares <= 512 && (shares == 1 || shares * kPanelWaves <= M); ++shares) {
      const double rounds = (double)((panels * shares + slots - 1) / slots * per_cu);
      const double us = 2.5 + rounds * ((double)lds / 24 + work / (double)shares) / 2400;
      if (best.width == 0 || us < best.us) best = {width, in_flight, (int)shares, us};
      if (panels * shares >= 4 * slots) break;
    }
  }
  return best;
}

template <int P, int R>
int launch_panels(int64_t M, int64_t K, int64_t N, const int *row_ptr, const int *col_idx, const float *vals, const float *B,
                  int transposed, const float *bias, int relu, float *C, int shares, hipStream_t s) {
  const int64_t panels = (N + P - 1) / P;
  const int64_t grid = round_up_8(panels * shares);
  if (grid > INT32_MAX) return fail(SCORCH_HIP_EUNSUPPORTED, "SpMM (panels): %lld workgroups exceed the launch limit", (long long)grid);
  static std::atomic<uint64_t> allowed{0};  // (per kernel) a bit per device: the attribute is a device's own
  int device = 0;
  SCORCH_HIP_CHECK(hipGetDevice(&device));
  const uint64_t bit = 1ull << (device & 63);
  if (device > 63 || !(allowed.load(std::memory_order_acquire) & bit)) {
    SCORCH_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&spmm_panels_kernel<P, R>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, kPanelLds));
    allowed.fetch_or(bit, std::memory_order_release);
  }
  mark_launch(s);
  spmm_panels_kernel<P, R><<<dim3((unsigned)grid), kPanelThreads, (size_t)panel_lds(K, P, R), s>>>(
      (int)M, (int)K, (int)N, row_ptr, col_idx, vals, B, transposed, bias, relu, C, (int)panels, shares,
      (int)((M + shares - 1) / shares));
  SCORCH_HIP_CHECK(hipGetLastError());
  mark_launch(s);
  return SCORCH_HIP_OK;
}

}  // namespace scorch

extern "C" {

int scorch_hip_spmm_csr_rows_panels_recommended(int64_t M, int64_t K, int64_t N, int64_t nnz, int64_t longest_row, int transposed) {
  using namespace scorch;
  if (M <= 0 || K <= 0 || N <= 0 || nnz <= 0) return 0;
  // a row is one wavefront's: rows of about the same length, and long enough to occupy one
  const int64_t mean = nnz / M;
  if (mean < 16 || longest_row > 2 * mean + 64) return 0;
  const PanelShape shape = panel_shape(M, K, N, nnz);
  if (shape.width == 0) return 0;
  return shape.us < spmm_rows_us(M, K, N, nnz) + (transposed ? dense_turn_us(K, N) : 0);
}

int scorch_hip_spmm_csr_rows_panels_f32(int64_t M, int64_t K, int64_t N, int64_t nnz, const int32_t *row_ptr,
                                   const int32_t *col_idx, const float *vals, const float *B, int transposed,
                                   const float *bias, int act, float *C, void *stream) {
  using namespace scorch;
  const char *fn = "scorch_hip_spmm_csr_rows_panels_f32";
  if (int rc = check_csr_args(fn, M, K, nnz, row_ptr, col_idx, vals)) return rc;
  SCORCH_REQUIRE(N >= 0, "%s: negative N=%lld", fn, (long long)N);
  if (N > INT32_MAX - kWaveSize * 4)
    return fail(SCORCH_HIP_EUNSUPPORTED, "%s: N=%lld is too large", fn, (long long)N);
  SCORCH_REQUIRE(act == SCORCH_HIP_ACT_NONE || act == SCORCH_HIP_ACT_RELU, "%s: unknown activation %d", fn, act);
  SCORCH_REQUIRE(act == SCORCH_HIP_ACT_NONE || bias != nullptr, "%s: an activation needs a bias", fn);
  if (M == 0 || N == 0) return SCORCH_HIP_OK;  // nothing to write
  SCORCH_REQUIRE(C != nullptr, "%s: C is NULL", fn);
  SCORCH_REQUIRE(K == 0 || B != nullptr, "%s: B is NULL", fn);
  SCORCH_REQUIRE(aligned_to(B, 4) && aligned_to(C, 4) && aligned_to(vals, 4) && aligned_to(bias, 4),
                 "%s: value arrays must be aligned to their element size", fn);
  const PanelShape shape = panel_shape(M, K, N, nnz);
  if (shape.width == 0) return fail(SCORCH_HIP_EUNSUPPORTED, "%s: K=%lld rows of B do not fit a CU's LDS", fn, (long long)K);
  const int relu = act == SCORCH_HIP_ACT_RELU;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define SCORCH_PANELS(P, R)                           \
  if (shape.width == P && shape.in_flight == R)       \
    return launch_panels<P, R>(M, K, N, row_ptr, col_idx, vals, B, transposed, bias, relu, C, shape.shares, s)
  SCORCH_PANELS(4, 2);
  SCORCH_PANELS(4, 4);
  SCORCH_PANELS(4, 8);
  SCORCH_PANELS(8, 4);
  SCORCH_PANELS(8, 8);
  SCORCH_PANELS(16, 1);
  SCORCH_PANELS(32, 1);
#undef SCORCH_PANELS
  return fail(SCORCH_HIP_ERUNTIME, "%s: no kernel for panels of %d columns", fn, shape.width);
}

}  // extern "C"

SCORCH_DEFINE_PRELOAD(spmm_panels)
