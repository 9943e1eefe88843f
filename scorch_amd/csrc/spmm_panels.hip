// SpMM with the dense operand in LDS: C = act(A * B + bias), fp32, for a matrix A of few columns and
// many entries -- a sparse weight matrix -- whose rows are about equally long.
//
// The other kernels gather rows of B out of the L2s, which hand out 15 TB/s: nnz * N * 4 bytes, 215 MB
// for 1,024 rows of 205 entries at N = 256.  Here a workgroup keeps a panel of B -- all K rows, P
// columns, K * P * 4 bytes of a CU's 160 KB -- and takes a share of A's rows past it; an entry costs
// its 8 bytes of A from the L2 and P * 4 bytes from LDS.  A panel of B is P columns, so a B that is
// handed over as its transpose (the usual W @ x.T) is read where it lies, P rows of x at a time.
//
// A row is a wavefront's, P / 4 lanes to an entry with 16 bytes each.  Its entries come one to a lane, one, two, four or
// eight batches of 64 at a time, by buffer loads whose range is the batch (what lies beyond it costs no bounds check and
// no traffic), and the lanes that share an entry get it by a move inside a quad that the address calculation carries.
// The next batch, or the next row's first, is on its way while the one at hand is used.  (Through a strip of LDS for four
// and eight lanes to an entry, and with a checked load for every share for one and two: 16.5 us for 13.2 with 1,024 x 4,096,
// 205 k entries, N = 256, P = 8; 15.0 for 12.3 with 4,096 x 1,024, P = 32; 70 for 56 with 8,192 x 1,024, N = 1,024, P = 32;
// 101 for 75 with 1,024 x 8,192, P = 4.)  At the end of a row the partial sums are added up by exchanging halves and then
// rows of 16 lanes between registers: a lane keeps two of its four columns, then one; the last steps are rotations.
//
// The panel's LDS reads are at random rows, so the entries that one access serves fall on the same banks now and then;
// wider panels lose less to that and read A less often, and they take more LDS per row of B.  A launch of 12 us is 2 us of
// panel on its way into LDS, 3 to 4 of LDS reads without conflicts, twice that with them, and the end of every row.
// The host picks P and the number of row shares from K, N and nnz.
#include <atomic>

#include "spmm.hpp"

namespace scorch {

constexpr int kPanelThreads = 1024;
constexpr int kPanelLds = 160 * 1024;

constexpr int kPanelWaves = kPanelThreads / kWaveSize;

// x of the lane of each lane's group of LPE that holds the group's entry u mod LPE (u a constant once the caller's
// loop is unrolled), by moves inside a quad, which the instruction that uses the value carries.  With eight lanes to an
// entry, `low` holds the first four lanes' values in both quads of the group and `high` the last four's.
template <int LPE>
struct Shared {
  int low, high;
  Shared() = default;
  __device__ __forceinline__ explicit Shared(int x) : low(x), high(x) {
    if constexpr (LPE == 8) {
      low = __builtin_amdgcn_update_dpp(x, x, 0x114, 0xf, 0xa, false);   // row_shr:4 into the odd quads
      high = __builtin_amdgcn_update_dpp(x, x, 0x104, 0xf, 0x5, false);  // row_shl:4 into the even ones
    }
  }
  __device__ __forceinline__ int of(int u) const {
    if constexpr (LPE == 1) return low;
    if constexpr (LPE == 2)
      return u % 2 ? __builtin_amdgcn_update_dpp(0, low, 0xf5, 0xf, 0xf, true) : __builtin_amdgcn_update_dpp(0, low, 0xa0, 0xf, 0xf, true);
    const int x = LPE == 8 && u % 8 >= 4 ? high : low;
    switch (u % 4) {
      case 0: return __builtin_amdgcn_update_dpp(0, x, 0x00, 0xf, 0xf, true);
      case 1: return __builtin_amdgcn_update_dpp(0, x, 0x55, 0xf, 0xf, true);
      case 2: return __builtin_amdgcn_update_dpp(0, x, 0xaa, 0xf, 0xf, true);
      default: return __builtin_amdgcn_update_dpp(0, x, 0xff, 0xf, 0xf, true);
    }
  }
};

template <int P, int R>
__global__ __launch_bounds__(kPanelThreads) void spmm_panels_kernel(
    int M, int K, int N, const int *__restrict__ row_ptr, const int *__restrict__ col_idx,
    const float *__restrict__ vals, const float *__restrict__ B, int transposed, const float *__restrict__ bias,
    int relu, float *__restrict__ C, int batch, int n_panels, int shares, int rows_per_share, int64_t nnz) {
  constexpr int LPE = P / 4;              // lanes to an entry
  constexpr int BATCH = R * kWaveSize;    // entries at hand: R to a lane
  extern __shared__ float4 s_panel[];     // [K + 1][LPE], row K is zero

  const int id = (int)xcd_contiguous(blockIdx.x, gridDim.x);
  const int share = id % shares, panel = id / shares % n_panels;
  const int product = id / shares / n_panels;  // of a batch over one pattern
  if (product >= batch) return;
  vals += (size_t)product * (size_t)nnz;
  B += (size_t)product * (size_t)K * (size_t)N;
  C += (size_t)product * (size_t)M * (size_t)N;
  const int n0 = panel * P;
  const int row_end = min(M, (share + 1) * rows_per_share);
  const int lane = wave_lane(), part = lane % LPE;

  // The wavefront's rows are first, first + 16, ...; lane i holds the i-th's pointers, 64 rows at a time.
  int row = uniform(share * rows_per_share + (int)threadIdx.x / kWaveSize);
  int held = 0, held_begin = 0, held_end = 0;
  auto hold = [&](int from) {
    const int r = from + lane * kPanelWaves;
    held_begin = r < row_end ? row_ptr[r] : 0;
    held_end = r < row_end ? row_ptr[r + 1] : 0;
  };
  struct Entries {
    int c[R];
    float a[R];
  } even, odd;
  auto load_entries = [&](Entries &to, int first, int end) __attribute__((always_inline)) {  // (loads beyond the row's end give zeros)
    first = uniform(first);
    const int bytes = uniform(max(min(end - first, BATCH), 0) * 4);
    const __amdgpu_buffer_rsrc_t columns = __builtin_amdgcn_make_buffer_rsrc((void *)(col_idx + first), 0, bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t values = __builtin_amdgcn_make_buffer_rsrc((void *)(vals + first), 0, bytes, 0x00020000);
#pragma unroll
    for (int e = 0; e < R; ++e) {
      to.c[e] = __builtin_amdgcn_raw_buffer_load_b32(columns, (e * kWaveSize + lane) * 4, 0, 0);
      to.a[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(values, (e * kWaveSize + lane) * 4, 0, 0));
    }
  };
  hold(row);
  int begin = __builtin_amdgcn_readlane(held_begin, 0), end = __builtin_amdgcn_readlane(held_end, 0);
  load_entries(even, begin, end);

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
  } else if (N >= 4) {
    constexpr int AHEAD = 8, ROWS = kPanelThreads / LPE;
    const int l = threadIdx.x % LPE, col = n0 + 4 * l;
    const int from = min(col, N - 4), beyond = col - from;  // the last columns are loaded with those in front of them
    for (int k0 = threadIdx.x / LPE; k0 < K; k0 += AHEAD * ROWS) {
      Vec<float, 4> x[AHEAD];
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) x[j] = load_vec<float, 4>(B + (size_t)min(k0 + j * ROWS, K - 1) * (size_t)N + from);
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) {
        float4 y = make_float4(x[j].v[0], x[j].v[1], x[j].v[2], x[j].v[3]);
        if (beyond & 1) y = make_float4(y.y, y.z, y.w, 0);
        if (beyond & 2) y = make_float4(y.z, y.w, 0, 0);
        if (beyond >= 4) y = make_float4(0, 0, 0, 0);
        s_panel[min(k0 + j * ROWS, K - 1) * LPE + l] = y;
      }
    }
  } else {
    for (int k = threadIdx.x; k < K; k += kPanelThreads) {
      const float *row_of_B = B + (size_t)k * (size_t)N;
      s_panel[k * LPE] = make_float4(row_of_B[0], N > 1 ? row_of_B[1] : 0.0f, N > 2 ? row_of_B[2] : 0.0f, 0);
#pragma unroll
      for (int l = 1; l < LPE; ++l) s_panel[k * LPE + l] = make_float4(0, 0, 0, 0);
    }
  }
  if (threadIdx.x < LPE) s_panel[K * LPE + threadIdx.x] = make_float4(0, 0, 0, 0);
  __syncthreads();

  // A batch at hand, of the row's entries from k on, while the next one is requested: the two change places from step to step (copied
  // from one to the other they were 16 of a step's 105 vector instructions with four batches to a lane).
  int k = begin;
  float acc[4] = {0, 0, 0, 0};
  auto step = [&](const Entries &at_hand, Entries &next) __attribute__((always_inline)) {
    Shared<LPE> from[R], with[R];  // the byte an entry's row of the panel begins at, and its value
#pragma unroll
    for (int e = 0; e < R; ++e) {
      from[e] = Shared<LPE>((e * kWaveSize + lane < end - k ? at_hand.c[e] : K) * (P * 4));
      with[e] = Shared<LPE>(__builtin_bit_cast(int, at_hand.a[e]));
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
    if (row < row_end) load_entries(next, k, end);
    constexpr int STEPS = R * LPE, AT_ONCE = STEPS < 4 ? STEPS : 4;  // LDS reads in flight
#pragma unroll
    for (int s0 = 0; s0 < STEPS; s0 += AT_ONCE) {
      float4 b[AT_ONCE];
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i) {
        const int u = s0 + i;
        b[i] = *reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(s_panel) + from[u / LPE].of(u % LPE) + part * 16);
      }
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i) {
        const int u = s0 + i;
        const float value = __builtin_bit_cast(float, with[u / LPE].of(u % LPE));
        acc[0] += value * b[i].x;
        acc[1] += value * b[i].y;
        acc[2] += value * b[i].z;
        acc[3] += value * b[i].w;
      }
    }
    if (!row_done) return;
    // The upper half of the wavefront keeps columns 2 and 3 of a lane's four, then odd rows of 16 lanes the odd one of two.
    // (a's upper half changes places with b's lower one, then a's odd rows with b's even ones)
    auto exchanged = [](float a, float b, auto swap) {
      const auto r = swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b));
      const unsigned x = r[0], y = r[1];
      return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
    };
    auto halves = [](unsigned a, unsigned b) { return __builtin_amdgcn_permlane32_swap(a, b, false, false); };
    auto rows = [](unsigned a, unsigned b) { return __builtin_amdgcn_permlane16_swap(a, b, false, false); };
    float sum = exchanged(exchanged(acc[0], acc[2], halves), exchanged(acc[1], acc[3], halves), rows);
    sum += row_rotated<8>(sum);
    if constexpr (LPE <= 4) sum += row_rotated<4>(sum);
    if constexpr (LPE <= 2) sum += row_rotated<2>(sum);
    if constexpr (LPE <= 1) sum += row_rotated<1>(sum);
    const int col = n0 + part * 4 + lane / 32 * 2 + lane / 16 % 2;
    if (lane % 16 < LPE && col < N) {
      if (bias) sum += bias[col];
      if (relu) sum = sum > 0.0f ? sum : 0.0f;
      C[(size_t)this_row * (size_t)N + col] = sum;
    }
    acc[0] = acc[1] = acc[2] = acc[3] = 0.0f;
  };
  while (row < row_end) {
    step(even, odd);
    if (row < row_end) step(odd, even);
  }
}

struct PanelShape {
  int width;     // 0: nothing fits
  int in_flight; // entries to a lane
  int shares;    // of A's rows
  double us;     // estimated
};

inline int64_t panel_lds(int64_t K, int width) { return (K + 1) * width * 4; }

// Panel width and row shares with the least estimated time: what the busiest CU has to do, a panel's load at 24 bytes a clock
// and its share of the entries for each of its workgroups, in clocks each what LDS takes for their pieces of B, and of the
// rows.  (Measured against the estimate, us: 1,024 x 4,096, 200 to a row, N = 256, P = 8 13.2 for 13.9; 7,989 x 3,994, 194,
// N = 379, P = 8 113 for 115; 1,024 x 8,192, 400, N = 1,024, P = 4 75 for 81; 4,096 x 1,024, 49, N = 256, P = 32 12.3 for 11.5;
// 465 x 1,863, 90, N = 167, P = 8 6.4 for 5.9.  The row kernel in its place: 17.0, 167, -, 17.0, 8.5; and at the line between the
// two, 663 x 226, 48, N = 716 6.9 for 8.1, 1,448 x 517, 64, N = 244 6.4 for 7.9, 2,301 x 702, 64, N = 122 6.2 for 7.2.)
inline PanelShape panel_shape_of_width(int64_t M, int64_t K, int64_t N, int64_t nnz, int width, int64_t batch) {
  const int64_t mean = (nnz + M - 1) / M;
  const int in_flight = width >= 16 ? 1 : width == 8 ? (mean > 192 ? 4 : 2) : mean > 256 ? 8 : mean > 128 ? 4 : 2;
  PanelShape best = {0, in_flight, 0, 0};
  const int64_t lds = panel_lds(K, width);
  if (lds > kPanelLds) return best;
  const int64_t in_batch = kWaveSize * in_flight, panels = (N + width - 1) / width * batch;
  const double per_entry = width == 32 ? 1.2 : width == 16 ? 0.8 : width == 8 ? 0.47 : 0.25;
  const double work = (double)M * ((double)((mean + in_batch - 1) / in_batch * in_batch) * per_entry + 50);
  for (int64_t shares = 1; shares <= 512 && (shares == 1 || shares * kPanelWaves <= M); ++shares) {
    const double rounds = (double)((panels * shares + 255) / 256);
    const double us = 2.5 + rounds * ((double)lds / 24 + work / (double)shares) / 2400;
    if (best.width == 0 || us < best.us) best = {width, in_flight, (int)shares, us};
    if (panels * shares >= 2048) break;
  }
  return best;
}

inline PanelShape panel_shape(int64_t M, int64_t K, int64_t N, int64_t nnz) {
  PanelShape best = {0, 0, 0, 0};
  if (M <= 0 || N <= 0 || K > kPanelLds / 16) return best;
  for (int width : {32, 16, 8, 4}) {
    const PanelShape shape = panel_shape_of_width(M, K, N, nnz, width, 1);
    if (shape.width != 0 && (best.width == 0 || shape.us < best.us)) best = shape;
  }
  return best;
}

template <int P, int R>
int launch_panels(int64_t batch, int64_t M, int64_t K, int64_t N, int64_t nnz, const int *row_ptr, const int *col_idx,
                  const float *vals, const float *B, int transposed, const float *bias, int relu, float *C, int shares, hipStream_t s) {
  const int64_t panels = (N + P - 1) / P;
  const int64_t grid = round_up_8(batch * panels * shares);
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
  spmm_panels_kernel<P, R><<<dim3((unsigned)grid), kPanelThreads, (size_t)panel_lds(K, P), s>>>(
      (int)M, (int)K, (int)N, row_ptr, col_idx, vals, B, transposed, bias, relu, C, (int)batch, (int)panels,
      shares, (int)((M + shares - 1) / shares), nnz);
  SCORCH_HIP_CHECK(hipGetLastError());
  mark_launch(s);
  return SCORCH_HIP_OK;
}

// `batch` products over one pattern, vals[h], B[h] and C[h] one behind the other: the panel width that a single one gets, so that
// each has the bits it would have by itself, and row shares for all of them.
int panels_entry(const char *fn, int64_t batch, int64_t M, int64_t K, int64_t N, int64_t nnz, const int32_t *row_ptr,
                 const int32_t *col_idx, const float *vals, const float *B, int transposed, const float *bias, int act, float *C,
                 void *stream) {
  if (int rc = check_csr_args(fn, M, K, nnz, row_ptr, col_idx, vals)) return rc;
  SCORCH_REQUIRE(N >= 0, "%s: negative N=%lld", fn, (long long)N);
  SCORCH_REQUIRE(batch >= 0, "%s: negative batch=%lld", fn, (long long)batch);
  if (N > INT32_MAX - kWaveSize * 4)
    return fail(SCORCH_HIP_EUNSUPPORTED, "%s: N=%lld is too large", fn, (long long)N);
  SCORCH_REQUIRE(act == SCORCH_HIP_ACT_NONE || act == SCORCH_HIP_ACT_RELU, "%s: unknown activation %d", fn, act);
  SCORCH_REQUIRE(act == SCORCH_HIP_ACT_NONE || bias != nullptr, "%s: an activation needs a bias", fn);
  if (batch == 0 || M == 0 || N == 0) return SCORCH_HIP_OK;  // nothing to write
  SCORCH_REQUIRE(C != nullptr, "%s: C is NULL", fn);
  SCORCH_REQUIRE(K == 0 || B != nullptr, "%s: B is NULL", fn);
  SCORCH_REQUIRE(aligned_to(B, 4) && aligned_to(C, 4) && aligned_to(vals, 4) && aligned_to(bias, 4),
                 "%s: value arrays must be aligned to their element size", fn);
  PanelShape shape = panel_shape(M, K, N, nnz);
  if (shape.width == 0) return fail(SCORCH_HIP_EUNSUPPORTED, "%s: K=%lld rows of B do not fit a CU's LDS", fn, (long long)K);
  if (batch > INT32_MAX / N)
    return fail(SCORCH_HIP_EUNSUPPORTED, "%s: a batch of %lld exceeds the launch limit", fn, (long long)batch);
  if (batch > 1) shape = panel_shape_of_width(M, K, N, nnz, shape.width, batch);
  const int relu = act == SCORCH_HIP_ACT_RELU;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define SCORCH_PANELS(P, R)                                                                                            \
  if (shape.width == P && shape.in_flight == R)                                                                        \
    return launch_panels<P, R>(batch, M, K, N, nnz, row_ptr, col_idx, vals, B, transposed, bias, relu, C, shape.shares, s)
  SCORCH_PANELS(4, 2);
  SCORCH_PANELS(4, 4);
  SCORCH_PANELS(4, 8);
  SCORCH_PANELS(8, 2);
  SCORCH_PANELS(8, 4);
  SCORCH_PANELS(16, 1);
  SCORCH_PANELS(32, 1);
#undef SCORCH_PANELS
  return fail(SCORCH_HIP_ERUNTIME, "%s: no kernel for panels of %d columns", fn, shape.width);
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
  return scorch::panels_entry("scorch_hip_spmm_csr_rows_panels_f32", 1, M, K, N, nnz, row_ptr, col_idx, vals, B, transposed, bias,
                              act, C, stream);
}

int scorch_hip_spmm_csr_rows_panels_batched_f32(int64_t batch, int64_t M, int64_t K, int64_t N, int64_t nnz,
                                                const int32_t *row_ptr, const int32_t *col_idx, const float *vals,
                                                const float *B, float *C, void *stream) {
  return scorch::panels_entry("scorch_hip_spmm_csr_rows_panels_batched_f32", batch, M, K, N, nnz, row_ptr, col_idx, vals, B, 0,
                              nullptr, SCORCH_HIP_ACT_NONE, C, stream);
}

}  // extern "C"

SCORCH_DEFINE_PRELOAD(spmm_panels)
