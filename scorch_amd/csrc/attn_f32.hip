// Fused block-sparse attention in fp32 for gfx950: O = softmax(scale * Q K^T restricted to
// a mask of 64 x 64 blocks, optionally with per-block bit masks) V, fp32 operands, fp32
// probabilities, fp32 accumulation.
//
// This is the three-step pipeline SDDMM -> row softmax -> SpMM that the reference runs per head
// in fp32 (bench/bench_sparse_transformer.py:354-372) in one kernel and at the reference's own
// precision: the scores never reach memory.  The structure is that of the bf16 kernel in
// attn.hip (one workgroup = one head x one block row or one stretch of one, a wavefront = 16
// queries, S^T = K Q^T and O^T += V^T P^T so that an MFMA result is the next MFMA's operand
// without any exchange between lanes); what differs is the matrix instruction,
// v_mfma_f32_16x16x4_f32, which contracts four values per lane group at a sixteenth of the bf16
// rate, so the kernel is bound by the matrix cores and everything around them is kept simple:
// tiles go through registers into LDS rows padded by 16 bytes (no bank conflicts for either
// operand), one tile in LDS and the next in registers, the accumulators are rescaled whenever a
// query's running maximum rises.
//
// Lane (g, n) = (lane / 16, lane % 16).  An MFMA takes A[i = n][k = g] and B[k = g][j = n] and
// adds to C[4g .. 4g+3][n].  Which four values of the contraction index a group of four MFMAs
// takes is free as long as both operands agree: step c of slab j uses d = 16 j + 4 g + c, so a
// lane's operands for four steps are 16 contiguous bytes of a row of K (one ds_read_b128) and of
// its query's row of Q (kept in registers).
//
// Sequences of any length: S need not be a multiple of 64 when the caller hands over which columns
// of every block are referred to (block_cols; a column beyond S never is).  Rows of K and V that no
// query of a block attends to are then not read -- zeros stand in, so they may hold anything -- and
// the last block row's queries beyond S compute on row S - 1 and are not stored.
//
// Blocks that are live in part are what a sliding window is made of: of the 64 queries x 64 keys
// of its edge blocks, a wavefront's 16 queries attend to some of the four 16-key tiles only, and a
// global token's block column holds one live key.  Tiles without a live position for the
// wavefront are skipped in both products and in the exponentials (window of 64 and a global token:
// 10.5 of 17 tiles remain).
//
// A NaN or infinity in a row of V belongs to the queries that attend to that key, and in such a block
// not to the others, whose probability for it is 0 (0 x NaN is NaN): the three steps never multiply
// the two.  What goes into LDS is therefore looked at (one fma for two elements); where a partly live
// block has something non-finite in V, those elements become zeros in LDS and leave a flag (NaN,
// infinity, -infinity) at the result elements they belong to, which are given it at the end.  (The
// look costs 1 % -- S = 3,001, 8 heads, D = 64, window of 64 and a global token: 27.0 -> 27.3 us.)
#include "attn_parts.hpp"
#include "common.hpp"

namespace scorch {
namespace attn32 {

constexpr int kBlock = 64;  // mask block edge: queries per workgroup, keys per step
typedef float floatx4 __attribute__((ext_vector_type(4)));

// Combine a value over the four lanes that share a query (lanes n, n + 16, n + 32, n + 48).
template <typename Op>
__device__ __forceinline__ float combine_query_lanes(float x, Op op) {
  const unsigned bits = __builtin_bit_cast(unsigned, x);
  auto r = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
  x = op(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
  const unsigned bits2 = __builtin_bit_cast(unsigned, x);
  auto q = __builtin_amdgcn_permlane32_swap(bits2, bits2, false, false);
  return op(__builtin_bit_cast(float, (unsigned)q[0]), __builtin_bit_cast(float, (unsigned)q[1]));
}

template <int D>
struct Tile {
  // A row of a tile takes D + 4 floats in LDS.  Readers of K (lane n reads 16 bytes of row
  // 16 t + n) then start 4 n banks apart, eight lanes cover the 32 banks; readers of V (lane
  // (g, n) reads one float of row 16 t + 4 g + r at column 16 dt + n) fall on bank
  // n + 16 g mod 32, two lanes per bank, which is what 64 lanes on 32 banks cost anyway.
  static constexpr int kStride = D + 4;
  static constexpr int kFloats = kBlock * kStride;
  static constexpr int kChunksPerRow = D / 4;  // 16-byte chunks
  static constexpr int kChunksPerThread = kBlock * kChunksPerRow / kBlockThreads;
};

constexpr float kDead = -3.0e38f;  // score of an entry the mask leaves out; also "no maximum yet"

// MASKED: blocks may be live in part (block_mask_index); without it every listed block is whole and
// every operand exists, and the code for the rest is left out of the kernel (registers).
template <int D, bool MASKED>
__global__ __launch_bounds__(kBlockThreads)
__attribute__((amdgpu_waves_per_eu(D == 128 ? 2 : 4))) void attn_f32_kernel(
    int S, int n_blocks, int n_heads, const int *__restrict__ block_row_ptr,
    const int *__restrict__ block_col_idx, const int *__restrict__ block_mask_index,
    const unsigned long long *__restrict__ block_masks, const unsigned long long *__restrict__ block_cols,
    const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V, float scale_log2e,
    float *__restrict__ O, int n_items, const int4 *__restrict__ items, int n_slots, float *__restrict__ partials) {
  using T = Tile<D>;
  constexpr int kStride = T::kStride;
  constexpr int kSlabs = D / 16;  // contraction slabs of the first product (four MFMA steps each)
  constexpr int kFeat = D / 16;   // 16-feature tiles of the second product
  constexpr int kCpt = T::kChunksPerThread;
  __shared__ __attribute__((aligned(16))) float s_k[T::kFloats];
  __shared__ __attribute__((aligned(16))) float s_v[T::kFloats];
  constexpr int kFlagWords = kBlock * D / 32;
  __shared__ int s_wild;  // MASKED: the last partly live block whose V holds something non-finite
  __shared__ unsigned s_flags[MASKED ? 3 : 1][MASKED ? kFlagWords : 1];  // bit d of query q's words: result (q, d)

  const int tid = threadIdx.x;
  const int lane = tid & (kWaveSize - 1);
  const int w = uniform(tid / kWaveSize);
  const int g = lane >> 4;
  const int n = lane & 15;
  int head, rank;
  {
    // all workgroups of a head on one XCD when the head count allows it (workgroup ids go round
    // the 8 XCDs): a head's K and V are then fetched into one L2 only
    const int id = blockIdx.x;
    if (n_heads % 8 == 0) {
      const int xcd = id & 7, slot = id >> 3;
      head = xcd + 8 * (slot / n_items);
      rank = slot % n_items;
    } else {
      head = id / n_items;
      rank = id % n_items;
    }
  }
  // work item: a block row, or with `items` a stretch of one (x: block row, y and z: the stretch
  // within block_col_idx, w: where its partial result goes, -1 = it writes O itself)
  int qb, kb_begin, kb_end, part_slot = -1;
  if (items) {
    const int4 item = items[rank];
    qb = uniform(item.x);
    kb_begin = uniform(item.y);
    kb_end = uniform(item.z);
    part_slot = uniform(item.w);
  } else {
    qb = n_blocks - 1 - rank;
    kb_begin = block_row_ptr[qb];
    kb_end = block_row_ptr[qb + 1];
  }
  const size_t head_off = (size_t)head * (size_t)S * D;
  const float *Kh = K + head_off, *Vh = V + head_off;
  const int query_at = qb * kBlock + w * 16 + n;
  const int query = MASKED && query_at >= S ? S - 1 : query_at;

  // The query's row, scaled once: scores then come out of the matrix cores in base-2 exponent
  // units (a negative or zero scale needs nothing special).
  floatx4 q_op[kSlabs];
#pragma unroll
  for (int j = 0; j < kSlabs; ++j) {
    q_op[j] = *reinterpret_cast<const floatx4 *>(Q + head_off + (size_t)query * D + 16 * j + 4 * g);
#pragma unroll
    for (int c = 0; c < 4; ++c) q_op[j][c] *= scale_log2e;
  }

  floatx4 o_acc[kFeat];
#pragma unroll
  for (int dt = 0; dt < kFeat; ++dt) o_acc[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m_run = kDead;
  float l_run = 0.0f;  // this lane's share of the row sum (its 16 keys of every block)

  // Tile traffic: thread `tid` moves chunks tid, tid + 256, ... (16 bytes each) of a 64 x D tile.
  floatx4 k_next[kCpt], v_next[kCpt];
  auto fetch = [&](floatx4 (&next)[kCpt], const float *from, int it) {
    const float *tile = from + (size_t)uniform(block_col_idx[it]) * kBlock * D;
    const unsigned long long cols = MASKED && block_cols ? block_cols[it] : ~0ull;
#pragma unroll
    for (int u = 0; u < kCpt; ++u) {
      const int chunk = tid + u * kBlockThreads;
      if (!MASKED || ((cols >> (chunk / T::kChunksPerRow)) & 1ull))
        next[u] = *reinterpret_cast<const floatx4 *>(tile + (size_t)chunk * 4);
      else
        next[u] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto fetch_k = [&](int it) { fetch(k_next, Kh, it); };
  auto fetch_v = [&](int it) { fetch(v_next, Vh, it); };
  auto store_tile = [&](int it, bool partly) {
#pragma unroll
    for (int u = 0; u < kCpt; ++u) {
      const int chunk = tid + u * kBlockThreads;
      const int at = (chunk / T::kChunksPerRow) * kStride + (chunk % T::kChunksPerRow) * 4;
      *reinterpret_cast<floatx4 *>(&s_k[at]) = k_next[u];
      *reinterpret_cast<floatx4 *>(&s_v[at]) = v_next[u];
    }
    if (MASKED && partly) {
      // infinite or NaN if some element is (a product may overflow too: the block is then looked through in vain)
      float sum = 0.0f, more = 0.0f;
#pragma unroll
      for (int u = 0; u < kCpt; ++u) {
        sum = fmaf(v_next[u][0], v_next[u][1], sum);
        more = fmaf(v_next[u][2], v_next[u][3], more);
      }
      if (!(fabsf(sum + more) < __builtin_inff())) s_wild = it;
    }
  };
  const int my_query_in_block = w * 16 + n;

  // a block that is only partly live: bit j of word i of its mask says whether query i of the block
  // row attends to key j of the block.  The words of the next block are requested a block ahead.
  auto mask_of = [&](int it) { return MASKED ? uniform(block_mask_index[it]) : -1; };
  auto live_word = [&](int mask_at) {
    return mask_at >= 0 ? block_masks[(size_t)mask_at * kBlock + my_query_in_block] : 0ull;
  };
  // the lane's own sixteen bits of its query's word: bit 4 t + r is key 16 t + 4 g + r
  auto own_bits = [&](unsigned long long word) {
    unsigned bits = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) bits |= ((unsigned)(word >> (16 * t + 4 * g)) & 0xfu) << (4 * t);
    return bits;
  };
  int mask_at = kb_begin < kb_end ? mask_of(kb_begin) : -1;
  // (s_wild needs no first value: a number it holds by chance has a block looked through in vain, by everybody)
  if (kb_begin < kb_end) {
    fetch_k(kb_begin);
    fetch_v(kb_begin);
    store_tile(kb_begin, mask_at >= 0);
  }
  __syncthreads();
  unsigned live = own_bits(live_word(mask_at));

  bool flagged = false;  // (the same for the whole workgroup, as what it depends on is)
  for (int it = kb_begin; it < kb_end; ++it) {
    const bool more = it + 1 < kb_end;
    if (more) fetch_k(it + 1);  // in flight while this block is computed (V follows after the scores:
                                // the two sets of staging registers are then not live at once with
                                // the K operands)
    const int next_mask_at = more ? mask_of(it + 1) : -1;
    const unsigned long long next_live = live_word(next_mask_at);
    const int wild_at = MASKED ? s_wild : -1;  // (looked at after the first product, when it has long arrived)

    // One block.  WHOLE: every tile has live positions and (unless `partly`) all of them are; otherwise
    // only the 16-key tiles in `tiles` are computed (bits 0 .. 3, the same for the whole wavefront).
    auto block = [&](auto whole, bool partly, unsigned tiles) {
      constexpr bool kWhole = decltype(whole)::value;
      auto on = [&](int t) { return kWhole || ((tiles >> t) & 1u); };
      // S^T = K Q^T: tile t holds keys 16 t + 4 g + r (r = 0 .. 3) against query n
      floatx4 st[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) st[t] = floatx4{0.f, 0.f, 0.f, 0.f};
      if constexpr (kWhole) {
#pragma unroll
        for (int j = 0; j < kSlabs; ++j) {
          floatx4 k_op[4];
#pragma unroll
          for (int t = 0; t < 4; ++t)
            k_op[t] = *reinterpret_cast<const floatx4 *>(&s_k[(16 * t + n) * kStride + 16 * j + 4 * g]);
#pragma unroll
          for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int t = 0; t < 4; ++t)
              st[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k_op[t][c], q_op[j][c], st[t], 0, 0, 0);
        }
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (on(t)) {
#pragma unroll
            for (int j = 0; j < kSlabs; ++j) {
              const floatx4 k_op = *reinterpret_cast<const floatx4 *>(&s_k[(16 * t + n) * kStride + 16 * j + 4 * g]);
#pragma unroll
              for (int c = 0; c < 4; ++c)
                st[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k_op[c], q_op[j][c], st[t], 0, 0, 0);
            }
          }
      }

      if (more) fetch_v(it + 1);

      if (partly) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (!((live >> (4 * t + r)) & 1u)) st[t][r] = kDead;
      }

      // online softmax, base 2
      float mx = kDead;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, st[t][r]);
      mx = combine_query_lanes(mx, [](float a, float b) { return fmaxf(a, b); });
      if (__any(mx > m_run)) {  // some query's maximum rises: after a row's first key blocks, seldom
        const float m_new = fmaxf(m_run, mx);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);  // (no maximum yet: the sums are 0)
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < kFeat; ++dt)
#pragma unroll
          for (int r = 0; r < 4; ++r) o_acc[dt][r] *= alpha;
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (on(t)) {
#pragma unroll
          for (int r = 0; r < 4; ++r) st[t][r] = __builtin_amdgcn_exp2f(st[t][r] - m_run);
          if (partly) {
            // an entry the mask leaves out: exp2(kDead - m_run) is 0 already unless the query has had no
            // live key so far (m_run = kDead), so it is set
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (!((live >> (4 * t + r)) & 1u)) st[t][r] = 0.0f;
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) l_run += st[t][r];
        }

      if constexpr (!kWhole)
        if (partly && uniform(wild_at) == it) {  // the whole workgroup comes here, before its second product, or nobody does
          int own = threadIdx.x;
          asm volatile("" : "+v"(own));  // (addresses made from it stay in here: the loop has no registers to spare)
          if (!flagged) {
            for (int i = own; i < 3 * kFlagWords; i += kBlockThreads) s_flags[i / kFlagWords][i % kFlagWords] = 0u;
            __syncthreads();
            flagged = true;
          }
          const unsigned long long *words = block_masks + (size_t)mask_at * kBlock;
#pragma unroll 1
          for (int i = own; i < kBlock * D; i += kBlockThreads) {
            const int key = i / D, d = i % D;
            float &v = s_v[key * kStride + d];
            if (fabsf(v) < __builtin_inff()) continue;
            unsigned *flags = s_flags[v > 0.0f ? 1 : v < 0.0f ? 2 : 0] + d / 32;
#pragma unroll 1
            for (int q = 0; q < kBlock; ++q)
              if ((words[q] >> key) & 1ull) atomicOr(flags + q * (D / 32), 1u << (d % 32));
            v = 0.0f;
          }
          __syncthreads();
        }

      // O^T += V^T P^T: step (t, r) contracts keys 16 t + 4 g + r, whose probabilities lane (g, n)
      // holds for query n; the V^T operand is V[that key][16 dt + n]
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (on(t)) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float *v_row = &s_v[(16 * t + 4 * g + r) * kStride + n];
#pragma unroll
            for (int dt = 0; dt < kFeat; ++dt)
              o_acc[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(v_row[16 * dt], st[t][r], o_acc[dt], 0, 0, 0);
          }
        }
    };
    if constexpr (!MASKED) {
      block(std::true_type{}, false, 0xfu);
    } else {
      unsigned tiles = 0xfu;
      if (mask_at >= 0) {
        tiles = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) tiles |= __any((live >> (4 * t)) & 0xfu) ? 1u << t : 0u;
      }
      block(std::false_type{}, mask_at >= 0, (unsigned)uniform((int)tiles));
    }
    mask_at = next_mask_at;
    live = own_bits(next_live);

    __syncthreads();  // every wavefront is done with this tile
    if (more) store_tile(it + 1, mask_at >= 0);
    __syncthreads();
  }

  if (MASKED && flagged) {
#pragma unroll
    for (int dt = 0; dt < kFeat; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int word = my_query_in_block * (D / 32) + dt / 2, bit = 16 * (dt % 2) + 4 * g + r;
        const bool nan = (s_flags[0][word] >> bit) & 1u, up = (s_flags[MASKED ? 1 : 0][word] >> bit) & 1u,
                   down = (s_flags[MASKED ? 2 : 0][word] >> bit) & 1u;
        if (nan || (up && down)) o_acc[dt][r] = __builtin_nanf("");
        else if (up) o_acc[dt][r] += __builtin_inff();
        else if (down) o_acc[dt][r] -= __builtin_inff();
      }
  }
  const float l = combine_query_lanes(l_run, [](float a, float b) { return a + b; });
  if (part_slot >= 0) {
    // a stretch of a block row: unnormalised sums, their reference maximum and the row sum
    float *part = partials + (((size_t)head * n_slots + part_slot) * kBlock + (w * 16 + n)) * (D + 4);
#pragma unroll
    for (int dt = 0; dt < kFeat; ++dt) *reinterpret_cast<floatx4 *>(part + 16 * dt + 4 * g) = o_acc[dt];
    if (g == 0) {
      part[D] = m_run;
      part[D + 1] = l;
    }
    return;
  }
  if (MASKED && query_at >= S) return;
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;  // queries without a live key give zeros
  float *out = O + head_off + (size_t)query * D;
#pragma unroll
  for (int dt = 0; dt < kFeat; ++dt) {
    floatx4 o = o_acc[dt];
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] *= inv;
    *reinterpret_cast<floatx4 *>(out + 16 * dt + 4 * g) = o;
  }
}

// ---- masks whose blocks are live in part: sixteen queries to a team of wavefronts ---------------------------------------
// A sliding window leaves a third of the 16-key tiles of its blocks dead, and different ones to every sixteen queries: the
// kernel above skips them, but its four wavefronts meet at two barriers per key block and wait for whichever has most
// tiles; and a launch of a few hundred workgroups leaves most of the chip's SIMDs with one wavefront's chain.  Here
// sixteen queries have a list of the tiles that are live for them, which up to four wavefronts take in turn: no tile
// of K or V goes through LDS, no barrier until the end, when they put their sums together.  K and V are read
// four times as often, out of the L2s (8 KB for a tile's 32 matrix instructions, 1,024 clocks: 32 bytes a
// clock and CU), the next tile's while one is computed.
//
// Features are numbered for the second product so that a lane's four V operands are one 16-byte piece of a row: tile
// dt = VW h + v holds features 16 VW h + VW i + v, i = 0 .. 15.
//
// SPLIT wavefronts take the tiles of sixteen queries in turn; a workgroup of four has 4 / SPLIT times sixteen.
//
// Bound: a wavefront's chain of reads (work item, block, mask words, K: about 4 us of launches of 6 to 20), then a SIMD's matrix
// and vector instructions, which hardly overlap: 1,024 and about 400 clocks a tile.  See team_wavefronts for what it takes.
template <int D, int SPLIT>
struct TeamTables {
  static constexpr int kQueries = 16, kTeams = kWavesPerBlock / SPLIT;  // queries to a team of SPLIT wavefronts; teams
  static constexpr int kBlocksAtOnce = 16;                              // 64 tiles: one to a lane
  static constexpr int kOthers = SPLIT > 1 ? SPLIT - 1 : 1;
  using Words = unsigned long long[kTeams][kBlocksAtOnce][kQueries];
  using Col = int[kBlocksAtOnce];
  using Sums = float[SPLIT > 1 ? kTeams : 1][kOthers][SPLIT > 1 ? kQueries : 1][D + 4];
  using Flags = unsigned[SPLIT > 1 ? kTeams : 1][kOthers][3][kWaveSize];
  Words words;
  Col col;
  alignas(16) Sums sums;
  Flags flags;
};

// Of a head's work item number `item`, the queries of the `quarter`-th of SPLIT workgroups.
template <int D, int SPLIT>
__device__ __forceinline__ void team_rows(
    typename TeamTables<D, SPLIT>::Words &s_words, typename TeamTables<D, SPLIT>::Col &s_col,
    typename TeamTables<D, SPLIT>::Sums &s_sums, typename TeamTables<D, SPLIT>::Flags &s_flags, int head, int item_at, int quarter, int S, int n_blocks, const int *__restrict__ block_row_ptr,
    const int *__restrict__ block_col_idx, const int *__restrict__ block_mask_index,
    const unsigned long long *__restrict__ block_masks,
    const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V, float scale_log2e,
    float *__restrict__ O, const int4 *__restrict__ items, int n_slots, float *__restrict__ partials) {
  using Tables = TeamTables<D, SPLIT>;
  constexpr int kQueries = Tables::kQueries, kTeams = Tables::kTeams, kBlocksAtOnce = Tables::kBlocksAtOnce, kOthers = Tables::kOthers;
  constexpr int kSlabs = D / 16, kFeat = D / 16;
  constexpr int VW = D == 32 ? 2 : 4, NH = kFeat / VW;

  const int tid = threadIdx.x, lane = tid & (kWaveSize - 1), w = uniform(tid / kWaveSize);
  const int team = w / SPLIT, part = w % SPLIT;
  const int g = lane >> 4, n = lane & 15;
  const int sub = quarter * kTeams + team;  // sixteen queries of the block row
  int qb, kb_begin, kb_end, part_slot = -1;
  if (items) {
    const int4 item = items[item_at];
    qb = uniform(item.x);
    kb_begin = uniform(item.y);
    kb_end = uniform(item.z);
    part_slot = uniform(item.w);
  } else {
    qb = n_blocks - 1 - item_at;
    kb_begin = block_row_ptr[qb];
    kb_end = block_row_ptr[qb + 1];
  }
  const int first_query = qb * kBlock + sub * kQueries;
  const size_t head_off = (size_t)head * (size_t)S * D;
  const float *Kh = K + head_off, *Vh = V + head_off;
  const int query = first_query + n < S ? first_query + n : S - 1;

  floatx4 q_op[kSlabs];
#pragma unroll
  for (int j = 0; j < kSlabs; ++j) q_op[j] = *reinterpret_cast<const floatx4 *>(Q + head_off + (size_t)query * D + 16 * j + 4 * g);

  floatx4 o_acc[kFeat];
#pragma unroll
  for (int dt = 0; dt < kFeat; ++dt) o_acc[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m_run = kDead, l_run = 0.0f;
  unsigned nan_at = 0, up_at = 0, down_at = 0;  // results (bit 4 dt + r) that a NaN or infinity in V belongs to
  bool flagged = false;

  floatx4 k_op[kSlabs];
  float v_op[4][NH][VW];
  unsigned long long live_tiles = 0;  // of the blocks at hand; a team's wavefronts take them in turn
  int number = 0;
  unsigned my_keys = 0;               // of tile `lane`: keys that some query of the sixteen attends to
  auto next_tile = [&]() {            // -1: no more
    while (live_tiles) {
      const int at = __ffsll(live_tiles) - 1;
      live_tiles &= live_tiles - 1;
      if (number++ % SPLIT == part) return at;
    }
    return -1;
  };
  // Rows of K and V that none of the sixteen attends to are not read -- there may be none, or anything -- and zeros
  // stand in: their requests go beyond the buffer (host: S * D * 4 < 2^31), which the hardware answers with
  // zeros and no traffic, and without a branch.  `at`: 4 * block + tile.
  constexpr int kNowhere = (int)0x80000000;
  const __amdgpu_buffer_rsrc_t k_rows = __builtin_amdgcn_make_buffer_rsrc((void *)Kh, 0, S * D * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t v_rows = __builtin_amdgcn_make_buffer_rsrc((void *)Vh, 0, S * D * 4, 0x00020000);
  const int k_lane = (n * D + 4 * g) * 4, v_lane = (4 * g * D + VW * n) * 4;
  auto first_key_of = [&](int at) { return uniform(s_col[at >> 2]) * kBlock + 16 * (at & 3); };
  auto keys_of = [&](int at) { return (unsigned)__builtin_amdgcn_readlane((int)my_keys, at); };
  auto fetch_k = [&](int at) __attribute__((always_inline)) {
    const int from = (keys_of(at) >> n) & 1u ? first_key_of(at) * (D * 4) + k_lane : kNowhere;
#pragma unroll
    for (int j = 0; j < kSlabs; ++j)
      k_op[j] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(k_rows, from + 64 * j, 0, 0));
  };
  auto fetch_v = [&](int at) __attribute__((always_inline)) {
    const int from = first_key_of(at) * (D * 4) + v_lane;
    const unsigned keys = keys_of(at) >> (4 * g);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = (keys >> r) & 1u ? from + r * (D * 4) : kNowhere;
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        Vec<float, VW> x;
        if constexpr (VW == 4)
          x = __builtin_bit_cast(Vec<float, VW>, __builtin_amdgcn_raw_buffer_load_b128(v_rows, row + 64 * VW * h, 0, 0));
        else
          x = __builtin_bit_cast(Vec<float, VW>, __builtin_amdgcn_raw_buffer_load_b64(v_rows, row + 64 * VW * h, 0, 0));
#pragma unroll
        for (int v = 0; v < VW; ++v) v_op[r][h][v] = x.v[v];
      }
    }
  };
  // One tile, whose rows of K have been requested; `next`: the one whose rows are, as soon as these have been used.
  auto compute = [&](int at, int next) __attribute__((always_inline)) {
    fetch_v(at);
    const int block = at >> 2, t = at & 3;
    const unsigned half = reinterpret_cast<const unsigned *>(&s_words[team][block][n])[t >> 1];  // keys 32 (t / 2) ..
    const unsigned live = half >> (16 * (t & 1) + 4 * g);
    floatx4 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < kSlabs; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) st = __builtin_amdgcn_mfma_f32_16x16x4f32(k_op[j][c], q_op[j][c], st, 0, 0, 0);
    if (next >= 0) fetch_k(next);
    const bool partly = !__all((live & 0xfu) == 0xfu);
    if (partly) {
#pragma unroll
      for (int r = 0; r < 4; ++r) st[r] = (live >> r) & 1u ? st[r] : kDead;
    }
    const float mx = fmaxf(fmaxf(st[0], st[1]), fmaxf(st[2], st[3]));
    if (__any(mx > m_run)) {
      const float m_new = fmaxf(m_run, combine_query_lanes(mx, [](float a, float b) { return fmaxf(a, b); }));
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < kFeat; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) o_acc[dt][r] *= alpha;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) st[r] = __builtin_amdgcn_exp2f(st[r] - m_run);
    if (partly) {  // (a query without a live key so far has kDead for its maximum: its dead keys are set to 0)
#pragma unroll
      for (int r = 0; r < 4; ++r) st[r] = (live >> r) & 1u ? st[r] : 0.0f;
    }
    l_run += (st[0] + st[1]) + (st[2] + st[3]);
    if (partly) {  // a NaN or infinity in V belongs to the queries that attend to its key (see the file's head)
      float sum = 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
          for (int v = 0; v < VW; v += 2) sum = fmaf(v_op[r][h][v], v_op[r][h][v + 1], sum);
      if (__any(!(fabsf(sum) < __builtin_inff()))) {
        flagged = true;
        const unsigned row = (unsigned)(s_words[team][block][n] >> (16 * t)) & 0xffffu;
#pragma unroll 1
        for (int key = 0; key < 16; ++key) {
          if (!((row >> key) & 1u)) continue;
          const float *from = Vh + (size_t)(first_key_of(at) + key) * D;
#pragma unroll 1
          for (int i = 0; i < 4 * kFeat; ++i) {
            const int dt = i / 4, r = i % 4;
            const float x = from[16 * VW * (dt / VW) + VW * (4 * g + r) + dt % VW];
            if (fabsf(x) < __builtin_inff()) continue;
            const unsigned bit = 1u << i;
            up_at |= x > 0.0f ? bit : 0u;
            down_at |= x < 0.0f ? bit : 0u;
            nan_at |= x > 0.0f || x < 0.0f ? 0u : bit;
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int v = 0; v < VW; ++v) v_op[r][h][v] = fabsf(v_op[r][h][v]) < __builtin_inff() ? v_op[r][h][v] : 0.0f;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int v = 0; v < VW; ++v)
          o_acc[h * VW + v] = __builtin_amdgcn_mfma_f32_16x16x4f32(v_op[r][h][v], st[r], o_acc[h * VW + v], 0, 0, 0);
  };

  for (int base = kb_begin; base < kb_end; base += kBlocksAtOnce) {  // uniform over the workgroup
    if (base > kb_begin) __syncthreads();  // everyone is done with the words before
    {
      const int i = tid / kQueries, it = base + i;
      unsigned long long word[kTeams];
#pragma unroll
      for (int p = 0; p < kTeams; ++p) word[p] = 0;
      if (it < kb_end) {
        const int mask_at = block_mask_index ? block_mask_index[it] : -1;
        if (tid % kQueries == 0) s_col[i] = block_col_idx[it];
        const unsigned long long *words = block_masks + (size_t)mask_at * kBlock + quarter * kTeams * kQueries + tid % kQueries;
#pragma unroll
        for (int p = 0; p < kTeams; ++p) word[p] = mask_at >= 0 ? words[p * kQueries] : ~0ull;
      }
#pragma unroll
      for (int p = 0; p < kTeams; ++p) s_words[p][i][tid % kQueries] = word[p];
    }
    __syncthreads();
    unsigned long long any = 0;
#pragma unroll
    for (int i = 0; i < kQueries; ++i) any |= s_words[team][lane >> 2][i];
    my_keys = (unsigned)(any >> (16 * (lane & 3))) & 0xffffu;
    live_tiles = __ballot(my_keys != 0);
    if (base == kb_begin)
#pragma unroll
      for (int j = 0; j < kSlabs; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) q_op[j][c] *= scale_log2e;
    int at = next_tile();
    if (at >= 0) fetch_k(at);
    while (at >= 0) {
      const int next = next_tile();
      compute(at, next);
      at = next;
    }
  }

  float l = combine_query_lanes(l_run, [](float a, float b) { return a + b; });
  if constexpr (SPLIT > 1) {
    if (part > 0) {
      float *mine = s_sums[team][part - 1][n];
#pragma unroll
      for (int dt = 0; dt < kFeat; ++dt) *reinterpret_cast<floatx4 *>(mine + 16 * dt + 4 * g) = o_acc[dt];
      if (g == 0) {
        mine[D] = m_run;
        mine[D + 1] = l;
      }
      s_flags[team][part - 1][0][lane] = nan_at;
      s_flags[team][part - 1][1][lane] = up_at;
      s_flags[team][part - 1][2][lane] = down_at;
    }
    flagged = __syncthreads_or(flagged);
    if (part > 0) return;
    float m_all = m_run;
#pragma unroll
    for (int p = 0; p < kOthers; ++p) m_all = fmaxf(m_all, s_sums[team][p][n][D]);
    const float own = __builtin_amdgcn_exp2f(m_run - m_all);
    m_run = m_all;
    l *= own;
#pragma unroll
    for (int dt = 0; dt < kFeat; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) o_acc[dt][r] *= own;
#pragma unroll
    for (int p = 0; p < kOthers; ++p) {
      const float *theirs = s_sums[team][p][n];
      const float weight = __builtin_amdgcn_exp2f(theirs[D] - m_all);
      l += weight * theirs[D + 1];
#pragma unroll
      for (int dt = 0; dt < kFeat; ++dt) {
        const floatx4 o = *reinterpret_cast<const floatx4 *>(theirs + 16 * dt + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r) o_acc[dt][r] += weight * o[r];
      }
    }
    if (flagged) {
#pragma unroll
      for (int p = 0; p < kOthers; ++p) {
        nan_at |= s_flags[team][p][0][lane];
        up_at |= s_flags[team][p][1][lane];
        down_at |= s_flags[team][p][2][lane];
      }
    }
  }
  if (flagged) {
#pragma unroll
    for (int dt = 0; dt < kFeat; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const unsigned bit = 1u << (4 * dt + r);
        if ((nan_at & bit) || ((up_at & bit) && (down_at & bit))) o_acc[dt][r] = __builtin_nanf("");
        else if (up_at & bit) o_acc[dt][r] += __builtin_inff();
        else if (down_at & bit) o_acc[dt][r] -= __builtin_inff();
      }
  }
  float inv = 1.0f;
  float *out;
  if (part_slot >= 0) {
    out = partials + (((size_t)head * n_slots + part_slot) * kBlock + (sub * kQueries + n)) * (D + 4);
    if (g == 0) {
      out[D] = m_run;
      out[D + 1] = l;
    }
  } else {
    if (first_query + n >= S) return;
    inv = l > 0.0f ? 1.0f / l : 0.0f;  // queries without a live key give zeros
    out = O + head_off + (size_t)query * D;
  }
#pragma unroll
  for (int h = 0; h < NH; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      Vec<float, VW> o;
#pragma unroll
      for (int v = 0; v < VW; ++v) o.v[v] = o_acc[h * VW + v][r] * inv;
      *reinterpret_cast<Vec<float, VW> *>(out + 16 * VW * h + VW * (4 * g + r)) = o;
    }
}

// WIDE: the first n_wide items are four workgroups' each, whatever SPLIT: where a few of the items are stretches of a shared-out row, that
// is a row with a query that attends to everything, and the sixteen queries with it have all of the stretch's tiles, the others
// next to none.  A wavefront for the sixteen was what launches waited for.  Window of 64 and a global token, us before and now:
// (3,001 tokens, 8 heads, D = 64) 24.9, 22.4; (4,500, 12, 64) 59.1, 38.4; (8,192, 16, 64) 87.4, 75.8; (2,198, 4, 128) 30.5, 24.3;
// (2,048, 12, 128) 45.0, 38.9; (6,075, 16, 32) 47.1, 41.5.  (In the same kernel without any: 52.3 -> 53.2 for a window of 256, so it is one of its own.)
template <int D, int SPLIT, bool WIDE>
__global__ __launch_bounds__(kBlockThreads)
__attribute__((amdgpu_waves_per_eu(D == 128 ? 2 : 4))) void attn_f32_tiles_kernel(
    int S, int n_blocks, int n_heads, const int *__restrict__ block_row_ptr,
    const int *__restrict__ block_col_idx, const int *__restrict__ block_mask_index,
    const unsigned long long *__restrict__ block_masks,
    const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V, float scale_log2e,
    float *__restrict__ O, int n_items, int n_wide, const int4 *__restrict__ items, int n_slots, float *__restrict__ partials) {
  // First, of every head, a quarter of the wide items and all of the others, and at the end of the launch the wide ones' other quarters,
  // of which most have nothing to do.  (The four of an item one after the other: an XCD's workgroups go to its four shader
  // engines in turn, and one engine got all the long ones; a head's at the end of the head: workgroups with nothing to do
  // took the places of others.)
  const int first = WIDE ? n_wide + (n_items - n_wide) * SPLIT : n_items * SPLIT;
  int id = blockIdx.x, ranks = first, quarter = 0;
  if (WIDE && id >= n_heads * first) {
    id -= n_heads * first;
    ranks = 3 * n_wide;
    quarter = 1;
  }
  int head, rank;
  if (n_heads % 8 == 0) {  // a head's workgroups on one XCD, as above
    const int xcd = id & 7, slot = id >> 3;
    head = xcd + 8 * (slot / ranks);
    rank = slot % ranks;
  } else {
    head = id / ranks;
    rank = id % ranks;
  }
  if constexpr (WIDE) {
    __shared__ union {
      TeamTables<D, SPLIT> usual;
      TeamTables<D, 4> wide;
    } lds;
    if (quarter > 0 || rank < n_wide) {
      quarter += rank / n_wide;
      team_rows<D, 4>(lds.wide.words, lds.wide.col, lds.wide.sums, lds.wide.flags, head, rank % n_wide, quarter, S, n_blocks, block_row_ptr,
                      block_col_idx, block_mask_index, block_masks, Q, K, V, scale_log2e, O, items, n_slots, partials);
      return;
    }
    rank -= n_wide;
    team_rows<D, SPLIT>(lds.usual.words, lds.usual.col, lds.usual.sums, lds.usual.flags, head, n_wide + rank / SPLIT, rank % SPLIT, S,
                        n_blocks, block_row_ptr, block_col_idx, block_mask_index, block_masks, Q, K, V, scale_log2e, O, items, n_slots,
                        partials);
  } else {
    using Tables = TeamTables<D, SPLIT>;
    __shared__ typename Tables::Words words;
    __shared__ typename Tables::Col col;
    __shared__ alignas(16) typename Tables::Sums sums;
    __shared__ typename Tables::Flags flags;
    team_rows<D, SPLIT>(words, col, sums, flags, head, rank / SPLIT, rank % SPLIT, S, n_blocks, block_row_ptr, block_col_idx,
                        block_mask_index, block_masks, Q, K, V, scale_log2e, O, items, n_slots, partials);
  }
}

// Combines the stretches of a block row that was shared out: with m* the largest of the
// stretches' reference maxima, O = sum_p 2^(m_p - m*) O_p / sum_p 2^(m_p - m*) l_p.
// One workgroup per (split row, head); thread t takes query t / 4 and a quarter of the features.
template <int D>
__global__ __launch_bounds__(kBlockThreads) void attn_f32_merge_kernel(int S, int n_slots,
                                                                       const int4 *__restrict__ split_rows,
                                                                       const float *__restrict__ partials,
                                                                       float *__restrict__ O) {
  const int4 row = split_rows[blockIdx.x];  // x: block row, y: first slot, z: number of stretches
  const int head = blockIdx.y;
  constexpr int kLanes = D / 4, kQueries = kBlockThreads / kLanes;  // threads per query, queries per workgroup
  const int q = blockIdx.z * kQueries + threadIdx.x / kLanes, feature = threadIdx.x % kLanes * 4;
  const float *base = partials + (((size_t)head * n_slots + row.y) * kBlock + q) * (D + 4);
  floatx4 acc;
  float l;
  combine_parts<D, kBlock *(D + 4)>(base, row.z, feature, acc, l);
  if (row.x * kBlock + q >= S) return;
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
  for (int r = 0; r < 4; ++r) acc[r] *= inv;
  *reinterpret_cast<floatx4 *>(O + ((size_t)head * S + (size_t)row.x * kBlock + q) * D + feature) = acc;
}

// Wavefronts to sixteen queries in attn_f32_tiles_kernel for masks whose blocks are live in part, 0: the other kernel.
// As many as leave every workgroup a place at once (four to a CU, two for D = 128); what is longer than that goes best with one,
// and with D = 32, whose tiles are half as long as the reads in front of them, by the other kernel unless a few long rows are
// shared out (causal, 2,048 tokens, 16 heads, D = 32: 61 us for 68; window and a global token, 6,075 tokens: 47 for 41).  Windows of 64 and a
// global token, (tokens, heads, D, workgroups of a block row): the other kernel, 1, 2 and 4 wavefronts, us, all without WIDE:
//   (300, 4, 64, 20) 10.8, 11.1, 8.2, 6.6     (2,048, 4, 64, 176) 19.0, 18.5, 15.3, 13.4   (960, 16, 64, 288) 23.6, 22.8, 19.5, 19.5
//   (3,001, 8, 64, 464) 24.6, 23.7, 23.1, 26.5   (2,048, 16, 64, 704) 31.8, 30.3, 30.4, 33.8   (8,192, 16, 64, 2,288) 92.6, 90.2, 92.1, 111
//   (1,472, 8, 32, 224) 13.4, 14.0, 11.9, 11.0   (2,944, 12, 32, 684) 20.0, 22.3, 20.8, 24.0   (6,141, 16, 32, 1,904) 43.6, 44.4, 44.5, 51.0
//   (7,744, 1, 128, 151) 30.8, 30.1, 23.8, 22.4   (2,048, 12, 128, 468) 45.0, 43.2, 45.9, 54.2   (4,992, 16, 128, 1,392) 130, 109, 113, 133
// (Whole blocks: 13.5 for 15.9 at (1,024, 8, 64, 128), but 13.8 for 11.6 at (4,096, 1, 64, 254); they stay with the other kernel.)
inline int team_wavefronts(int D, unsigned workgroups, bool few_stretches) {
  const unsigned places = D == 128 ? 160 : 320;
  if (workgroups <= places) return 4;
  if (workgroups <= 2 * places - 64) return 2;
  return (D == 32 && !few_stretches) || workgroups > INT32_MAX / 16 ? 0 : 1;
}

template <int D>
static int launch(dim3 grid, hipStream_t s, int S, int n_blocks, int H, const int32_t *block_row_ptr,
                  const int32_t *block_col_idx, const int32_t *block_mask_index,
                  const unsigned long long *block_masks, const unsigned long long *block_cols, const float *q,
                  const float *k, const float *v, float scale_log2e, float *o, int n_items, const int4 *items, int n_slots, float *partials,
                  int n_split_rows, const int4 *split_rows) {
  mark_launch(s);
  const bool few_stretches = items && n_slots > 0 && 3 * (int64_t)n_slots <= n_items;  // (of a few long rows: see the tiles' kernel)
  if (const int split = block_mask_index ? team_wavefronts(D, grid.x, few_stretches) : 0; split && (int64_t)S * D * 4 < INT32_MAX) {
    const bool wide = split < 4 && few_stretches;
    const int n_wide = wide ? n_slots : 0;
    auto kernel = split == 4   ? &attn_f32_tiles_kernel<D, 4, false>
                  : split == 2 ? (wide ? &attn_f32_tiles_kernel<D, 2, true> : &attn_f32_tiles_kernel<D, 2, false>)
                               : (wide ? &attn_f32_tiles_kernel<D, 1, true> : &attn_f32_tiles_kernel<D, 1, false>);
    kernel<<<dim3((unsigned)H * (unsigned)(4 * n_wide + (n_items - n_wide) * split)), kBlockThreads, 0, s>>>(
        S, n_blocks, H, block_row_ptr, block_col_idx, block_mask_index, block_masks, q, k, v, scale_log2e, o, n_items, n_wide, items,
        n_slots, partials);
  } else {
    auto kernel = block_mask_index ? &attn_f32_kernel<D, true> : &attn_f32_kernel<D, false>;
    kernel<<<grid, kBlockThreads, 0, s>>>(S, n_blocks, H, block_row_ptr, block_col_idx, block_mask_index, block_masks,
                                          block_cols, q, k, v, scale_log2e, o, n_items, items, n_slots, partials);
  }
  SCORCH_HIP_CHECK(hipGetLastError());
  mark_launch(s);
  if (n_split_rows > 0) {
    const dim3 merge_grid((unsigned)n_split_rows, (unsigned)H, (unsigned)(kBlock * D / 4 / kBlockThreads));
    attn_f32_merge_kernel<D><<<merge_grid, kBlockThreads, 0, s>>>(S, n_slots, split_rows, partials, o);
    SCORCH_HIP_CHECK(hipGetLastError());
    mark_launch(s);
  }
  return SCORCH_HIP_OK;
}

}  // namespace attn32
}  // namespace scorch

extern "C" size_t scorch_hip_attn_blocksparse_f32_workspace_bytes(int64_t H, int64_t n_slots, int64_t D) {
  if (H <= 0 || n_slots <= 0 || D <= 0) return 0;
  return (size_t)H * (size_t)n_slots * scorch::attn32::kBlock * (size_t)(D + 4) * sizeof(float);
}

extern "C" int scorch_hip_attn_blocksparse_f32(
    int64_t H, int64_t S, int64_t D, int64_t block, int64_t n_active_blocks, const int32_t *block_row_ptr,
    const int32_t *block_col_idx, const int32_t *block_mask_index, int64_t n_masks, const uint64_t *block_masks,
    int64_t n_items, const int32_t *items, int64_t n_split_rows, const int32_t *split_rows, int64_t n_slots,
    const float *Q, const float *K, const float *V, float scale, float *O, void *workspace, size_t workspace_bytes,
    void *stream) {
  return scorch_hip_attn_blocksparse_f32_cols(H, S, D, block, n_active_blocks, block_row_ptr, block_col_idx,
                                              block_mask_index, n_masks, block_masks, nullptr, n_items, items,
                                              n_split_rows, split_rows, n_slots, Q, K, V, scale, O, workspace,
                                              workspace_bytes, stream);
}

extern "C" int scorch_hip_attn_blocksparse_f32_cols(
    int64_t H, int64_t S, int64_t D, int64_t block, int64_t n_active_blocks, const int32_t *block_row_ptr,
    const int32_t *block_col_idx, const int32_t *block_mask_index, int64_t n_masks, const uint64_t *block_masks,
    const uint64_t *block_cols, int64_t n_items, const int32_t *items, int64_t n_split_rows, const int32_t *split_rows, int64_t n_slots,
    const float *Q, const float *K, const float *V, float scale, float *O, void *workspace, size_t workspace_bytes,
    void *stream) {
  using namespace scorch;
  const char *fn = "scorch_hip_attn_blocksparse_f32";
  if (H < 0 || S < 0 || D < 0 || block <= 0 || n_active_blocks < 0 || n_masks < 0 || n_items < 0 ||
      n_split_rows < 0 || n_slots < 0)
    return fail(SCORCH_HIP_EINVAL, "%s: negative size (H=%lld S=%lld D=%lld block=%lld)", fn, (long long)H,
                (long long)S, (long long)D, (long long)block);
  if ((D != 32 && D != 64 && D != 128) || block != attn32::kBlock)
    return fail(SCORCH_HIP_EUNSUPPORTED, "%s: only head dimensions 32, 64 and 128 and %d x %d mask blocks are "
                "built (got D=%lld block=%lld)", fn, attn32::kBlock, attn32::kBlock, (long long)D, (long long)block);
  if (S % attn32::kBlock != 0 && (!block_cols || !block_mask_index))
    return fail(SCORCH_HIP_EINVAL, "%s: S=%lld is not a multiple of the block size (and no block_cols)", fn, (long long)S);
  if (H * (S / attn32::kBlock + 1) > INT32_MAX || S * D > INT32_MAX || n_items * H > INT32_MAX || n_slots > INT32_MAX)
    return fail(SCORCH_HIP_EUNSUPPORTED, "%s: H=%lld, S=%lld or the item count too large", fn, (long long)H,
                (long long)S);
  if (H == 0 || S == 0) return SCORCH_HIP_OK;
  SCORCH_REQUIRE(n_items > 0 || block_row_ptr != nullptr, "%s: block_row_ptr is NULL", fn);
  SCORCH_REQUIRE(n_active_blocks == 0 || block_col_idx != nullptr, "%s: block_col_idx is NULL", fn);
  SCORCH_REQUIRE(Q && K && V && O, "%s: NULL Q/K/V/O", fn);
  SCORCH_REQUIRE(aligned_to(Q, 16) && aligned_to(K, 16) && aligned_to(V, 16) && aligned_to(O, 16),
                 "%s: Q, K, V and O must be 16-byte aligned", fn);
  if (block_mask_index) {
    SCORCH_REQUIRE(n_masks == 0 || block_masks != nullptr, "%s: block_masks is NULL", fn);
    SCORCH_REQUIRE(aligned_to(block_masks, 8), "%s: block_masks must be 8-byte aligned", fn);
  }
  SCORCH_REQUIRE(aligned_to(block_cols, 8), "%s: block_cols must be 8-byte aligned", fn);
  const int n_blocks = (int)((S + attn32::kBlock - 1) / attn32::kBlock);
  int work = n_blocks;
  const int4 *item_list = nullptr, *rows = nullptr;
  float *partials = nullptr;
  if (n_items > 0) {
    SCORCH_REQUIRE(items != nullptr && aligned_to(items, 16), "%s: items must be 16-byte aligned", fn);
    SCORCH_REQUIRE(n_split_rows == 0 || (split_rows != nullptr && aligned_to(split_rows, 16)),
                   "%s: split_rows must be 16-byte aligned", fn);
    const size_t need = scorch_hip_attn_blocksparse_f32_workspace_bytes(H, n_slots, D);
    if (need > 0 && (!workspace || workspace_bytes < need || !aligned_to(workspace, 256)))
      return fail(SCORCH_HIP_EWORKSPACE, "%s: a 256-byte aligned workspace of %zu bytes is needed, %zu given", fn,
                  need, workspace ? workspace_bytes : (size_t)0);
    work = (int)n_items;
    item_list = reinterpret_cast<const int4 *>(items);
    rows = reinterpret_cast<const int4 *>(split_rows);
    partials = static_cast<float *>(workspace);
  } else if (n_split_rows > 0 || n_slots > 0) {
    return fail(SCORCH_HIP_EINVAL, "%s: split rows without items", fn);
  }
  const dim3 grid((unsigned)((int64_t)work * H));
  const float scale_log2e = scale * 1.4426950408889634f;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned long long *masks = reinterpret_cast<const unsigned long long *>(block_masks);
#define SCORCH_ATTN32(DIM)                                                                                     \
  return attn32::launch<DIM>(grid, s, (int)S, n_blocks, (int)H, block_row_ptr, block_col_idx, block_mask_index, \
                             masks, reinterpret_cast<const unsigned long long *>(block_cols), Q, K, V, scale_log2e, O, work, item_list, (int)n_slots, partials,          \
                             (int)n_split_rows, rows)
  if (D == 32) SCORCH_ATTN32(32);
  if (D == 64) SCORCH_ATTN32(64);
  SCORCH_ATTN32(128);
#undef SCORCH_ATTN32
}

SCORCH_DEFINE_PRELOAD(attn_f32)
