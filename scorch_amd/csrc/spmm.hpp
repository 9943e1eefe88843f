// Pieces shared by the SpMM kernels of libscorch_hip.so: the merge-path work
// split (spmm.hip), the row-split kernel for short rows (spmm_rows.hip) and the
// kernel for a dense operand stored by column tiles (spmm_tiled.hip).
#pragma once

#include "common.hpp"

namespace scorch {

constexpr int kItemsPerWave = 256;  // most merge items (row ends + nonzeros) per wavefront
constexpr int kMinItemsPerWave = 32;
constexpr int kGather = 8;          // B-row loads in flight per wavefront

enum Epilogue { kEpiNone = 0, kEpiBias = 1, kEpiBiasRelu = 2 };

// Workgroup id -> (column tile, block of wavefront spans).  Workgroups are dealt
// to the 8 XCDs round robin by their linear id, and every XCD has its own L2.
// With a multiple of 8 column tiles, tile t is given to XCD t % 8 and each XCD
// works through its tiles one after the other: the B rows a tile gathers
// (K rows of 64 * VEC elements) are then fetched into one L2 only and stay
// there while the tile is processed.
struct TileMap {
  int tile;
  int64_t block;
};

__device__ __forceinline__ TileMap map_workgroup(int64_t id, int n_tiles, int64_t blocks_per_tile) {
  TileMap m;
  if (n_tiles > 1 && (n_tiles & 7) == 0) {
    const int xcd = (int)(id & 7);
    const int64_t slot = id >> 3;
    m.tile = xcd + 8 * (int)(slot / blocks_per_tile);
    m.block = slot % blocks_per_tile;
  } else {
    m.tile = (int)(id / blocks_per_tile);
    const int64_t rem = id % blocks_per_tile;
    // rem & 7 is the XCD when blocks_per_tile is a multiple of 8 (the SpMM launchers
    // see to that): every XCD gets one contiguous eighth of the chunks, so that B
    // rows shared by neighbouring rows of A are found in its L2
    m.block = (blocks_per_tile & 7) == 0 ? xcd_contiguous(rem, blocks_per_tile) : rem;
  }
  return m;
}

template <typename T, int EPI>
__device__ __forceinline__ T apply_epilogue(typename Acc<T>::type acc, T bias) {
  T r = (T)acc;
  if (EPI != kEpiNone) r = r + bias;
  if (EPI == kEpiBiasRelu) r = r > (T)0 ? r : (T)0;
  return r;
}

// Chunk boundaries.  Chunk c nominally covers the merged positions [c * items,
// (c + 1) * items).  A boundary that falls inside a row moves forward to just
// after the row's end marker when that is at most `snap` items away: the row
// is then summed by one chunk and leaves no carry.  Most rows are short, so
// most boundaries snap, and carries remain for rows that really span chunks.
// The result depends on the nominal position only, so the two chunks on either
// side of a boundary agree on it.  x: rows finished before the boundary, y:
// nonzeros before it.
constexpr int kSnapItems = 64;

struct Boundary {
  int x, y;
};

__device__ __forceinline__ Boundary chunk_boundary(int64_t d, int M, int64_t total_items,
                                                   const int *__restrict__ row_ptr, int snap) {
  Boundary b;
  if (d >= total_items) {
    b.x = M;
    b.y = (int)(total_items - M);
    return b;
  }
  auto row_end_key = [&](int i) { return (int64_t)row_ptr[i + 1] + i; };
  b.x = wave_count_below(M, d, row_end_key);
  b.y = uniform((int)(d - b.x));
  if (b.x < M) {
    const int begin = uniform(row_ptr[b.x]), end = uniform(row_ptr[b.x + 1]);
    const int64_t after_marker = (int64_t)end + b.x + 1;
    if (begin < b.y && after_marker - d <= snap) {  // the row is under way and nearly done
      b.x += 1;
      b.y = end;
    }
  }
  return b;
}

// A boundary computed beforehand (spmm_bounds_kernel): record c of `bounds`.
__device__ __forceinline__ Boundary load_boundary(const Boundary *__restrict__ bounds, int64_t c) {
  const int2 raw = *reinterpret_cast<const int2 *>(bounds + c);
  Boundary b;
  b.x = uniform(raw.x);
  b.y = uniform(raw.y);
  return b;
}

// Several products over one sparsity pattern in one launch (grid.y = problem; one per
// attention head): how far apart, in elements, the problems' value arrays, dense operands,
// results and carry rows lie.  All zero for a single product.
struct SpmmBatch {
  int64_t vals, b, c, carry;
};

// Shape of the work split.  A chunk holds nominally up to 256 merge items, one
// chunk per wavefront; small problems use smaller chunks, so that they are
// spread over more, shorter wavefronts.  (A wavefront that walked two or more
// consecutive chunks with one carry for all of them was measured: the same
// time on a graph with uniform neighbours, slower -- 0.81 against 0.69 ms on the
// 4,096-neighbour graph -- where neighbouring rows share columns, because an XCD
// then has a wider stretch of rows in flight than its L2 covers.)
struct SpmmSplit {
  int items_per_chunk;
  int snap;        // see chunk_boundary
  int64_t spans;   // chunks = wavefronts with work = carry records
};

// ---- rows cut by chunk boundaries, folded without a second launch -----------------------------
// The chunks that share a row leave their parts (carry_val, and the chunk that ends the row its
// part in C) and take a ticket from the row's counter; the one that takes the last adds the parts up
// in the order spmm_fixup_kernel keeps: the same bits, one launch less (3 to 8 us of a product that
// takes 7 to 20; 24 of 1,340 on the million-node graph).
//   Counters are zero before a launch and after it: whoever takes a counter's last ticket clears it.  They live in memory of their own, one
// buffer per stream, since launches that overlap must not share them.
//   Parts and counters cross between XCDs, whose L2s are not coherent with each other: parts are
// written and read with agent-scope accesses, which go past the L2, and a wavefront waits until
// its own have been acknowledged before it takes its ticket.  (A release fence instead would make
// the L2 write all of its dirty lines back, at every row.)
struct RowSpan {
  int first, last;  // chunks; the last one ends the row
};
// Row `row`'s chunks: nominal positions of its first entry and its end marker, the latter's chunk
// corrected for a boundary inside the row that has moved past the marker (chunk_boundary).
__device__ __forceinline__ RowSpan row_span(int row, int begin, int end, int items, int snap) {
  const int64_t p0 = (int64_t)begin + row, marker = (int64_t)end + row;  // below 2^32
  RowSpan s;
  s.first = (int)((unsigned)p0 / (unsigned)items);
  s.last = (int)((unsigned)marker / (unsigned)items);
  const int64_t d = (int64_t)s.last * items;
  if (d > p0 && marker + 1 - d <= snap) --s.last;
  return s;
}

// Whether this wavefront is the last of the row's to get here.  Its own parts are in memory when
// its ticket is taken.
__device__ __forceinline__ bool last_ticket(int *counter, int parts) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  int taken = 0;
  if (wave_lane() == 0)
    taken = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  taken = uniform(taken);
  if (taken != parts - 1) return false;
  if (wave_lane() == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

template <typename T, int VEC>
__device__ __forceinline__ void store_part(T *p, const Vec<T, VEC> &x) {
#pragma unroll
  for (int v = 0; v < VEC; ++v) __hip_atomic_store(p + v, x.v[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T, int VEC>
__device__ __forceinline__ Vec<T, VEC> load_part(const T *p) {
  Vec<T, VEC> x;
#pragma unroll
  for (int v = 0; v < VEC; ++v) x.v[v] = __hip_atomic_load(p + v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return x;
}

// The sum of the parts of chunks from, from + step, ... (count of them) in their order.  One lane, VEC columns.
template <typename T, int VEC>
__device__ __forceinline__ Vec<T, VEC> sum_parts(const T *__restrict__ carry_val, int N, int col0, int from, int step, int count) {
  using A = typename Acc<T>::type;
  A sum[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) sum[v] = (A)0;
  constexpr int kBatch = 8;  // in flight
  auto part_at = [&](int i) { return load_part<T, VEC>(carry_val + (size_t)(from + i * step) * (size_t)N + col0); };
  int i = 0;
  for (; i + kBatch <= count; i += kBatch) {
    Vec<T, VEC> part[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) part[u] = part_at(i + u);
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
#pragma unroll
      for (int v = 0; v < VEC; ++v) sum[v] += (A)part[u].v[v];
  }
  for (; i < count; ++i) {
    const Vec<T, VEC> part = part_at(i);
#pragma unroll
    for (int v = 0; v < VEC; ++v) sum[v] += (A)part.v[v];
  }
  Vec<T, VEC> o;
#pragma unroll
  for (int v = 0; v < VEC; ++v) o.v[v] = (T)sum[v];
  return o;
}

// A chunk's part of row `row` (entries [begin, end)) is in memory: take its ticket and, as the last, fold
// the row into C.  carry: the part is chunk's carry; else what the row's last chunk has stored in C.
// A row of more than kFoldGroup carries is folded in two levels -- groups of kFoldGroup consecutive carries,
// then the groups' sums, kept where each group's first carry was -- so that a 50,000-entry row neither
// queues up hundreds of chunks at one counter nor ends in one wavefront adding hundreds of parts (with
// one level 100,000 nodes at N = 16 took 49 us, with a second launch 28).
// counters: two per chunk, the groups' and the rows', each at the first chunk of its own.
constexpr int kFoldGroup = 16;
template <typename T, int VEC, int EPI>
__device__ __forceinline__ void finish_part(int row, int begin, int end, int64_t chunk, bool carry, int items, int snap,
                                            int64_t n_chunks, int *__restrict__ counters, int N, int col0, bool folds,
                                            T *__restrict__ carry_val, T *__restrict__ C, const T (&bias_v)[VEC]) {
  using A = typename Acc<T>::type;
  const RowSpan span = row_span(row, begin, end, items, snap);
  const int n = span.last - span.first;
  int *const rows = counters + n_chunks;
  int parts = n, step = 1;
  if (n > kFoldGroup) {
    parts = (n + kFoldGroup - 1) / kFoldGroup;
    step = kFoldGroup;
    if (carry) {
      const int first = span.first + ((int)chunk - span.first) / kFoldGroup * kFoldGroup;
      const int count = span.last - first < kFoldGroup ? span.last - first : kFoldGroup;
      if (!last_ticket(counters + first, count)) return;
      if (folds) {
        const Vec<T, VEC> sum = sum_parts<T, VEC>(carry_val, N, col0, first, 1, count);
        store_part<T, VEC>(carry_val + (size_t)first * (size_t)N + col0, sum);
      }
    }
  }
  if (!last_ticket(rows + span.first, parts + 1) || !folds) return;
  T *dst = C + (size_t)row * (size_t)N + col0;
  Vec<T, VEC> o = load_part<T, VEC>(dst);
  const Vec<T, VEC> sum = sum_parts<T, VEC>(carry_val, N, col0, span.first, step, parts);
#pragma unroll
  for (int v = 0; v < VEC; ++v) o.v[v] = apply_epilogue<T, EPI>((A)sum.v[v] + (A)o.v[v], bias_v[v]);
  store_vec<T, VEC>(dst, o);
}

// Narrow tiles pay off when N is small: a row of B is at most 256 bytes, so
// full-width tiles would leave lanes idle or fall back to 4-byte loads.  Returns the tile width in
// bytes, or 0 for wide tiles.  (Tiling a wide B by columns so that K narrow rows
// stay in one XCD's L2 was measured and lost: the workgroups resident on an XCD
// span several tiles at once and evict each other's slices.)
inline int narrow_tile_bytes(int64_t N, size_t elem) {
  const int64_t row_bytes = N * (int64_t)elem;
  return row_bytes <= 256 ? (int)row_bytes : 0;
}

inline SpmmSplit spmm_split(int64_t M, int64_t nnz, int64_t N, size_t elem) {
  const int64_t total = M + nnz;
  SpmmSplit sp;
  // every column tile (up to 1 KiB of a row) walks all chunks again
  const int64_t tiles = (N * (int64_t)elem + 1023) / 1024;
  const int64_t per_wave = total * (tiles > 0 ? tiles : 1) / 8192;  // 256 CUs x 32 wavefronts
  sp.items_per_chunk = kMinItemsPerWave;
  while (sp.items_per_chunk < kItemsPerWave && sp.items_per_chunk * 2 <= per_wave)
    sp.items_per_chunk *= 2;
  sp.snap = sp.items_per_chunk < kSnapItems ? sp.items_per_chunk : kSnapItems;
  sp.spans = (total + sp.items_per_chunk - 1) / sp.items_per_chunk;
  return sp;
}

// Chunks of spmm_grouped_kernel, one to a workgroup: few enough to be resident at once, six workgroups to a
// CU (20,000 nodes, 820 K items, N = 32: 2,000 chunks, which take two rounds, 15.0 us, 1,500 13.3), of 128
// items at least (2,708 nodes, N = 16: 6.3 us, of 256 7.1) and 1,024 at most.
constexpr int kGroupedItems = 1024, kGroupedItemsMin = 128;
inline SpmmSplit grouped_split(int64_t M, int64_t nnz) {
  const int64_t total = M + nnz, resident = 1536;
  int64_t items = ((total + resident - 1) / resident + 31) / 32 * 32;
  items = items < kGroupedItemsMin ? kGroupedItemsMin : items > kGroupedItems ? kGroupedItems : items;
  return {(int)items, kSnapItems, (total + items - 1) / items};
}
// Where narrow rows are split that way.  Large products are bound by their traffic, of which the kernel with
// a lane group per row makes less (see there); up to here the chain of reads counts (100,000 nodes of 3 + 1,
// N = 16: 17.5 -> 13.2 us, of 12 + 1, N = 64: 54.9 -> 51.7; 300,000 of 6 + 1, 2.1 M items: N = 31 75.4 against 77.7).
constexpr int64_t kGroupedMost = 2 << 20;  // merge items
inline bool grouped_chunks(int64_t M, int64_t nnz, int64_t N, size_t elem) {
  return narrow_tile_bytes(N, elem) && M + nnz <= kGroupedMost;
}
// The split whose boundaries a plan keeps for products with N columns.
inline SpmmSplit planned_split(int64_t M, int64_t nnz, int64_t N, size_t elem) {
  return grouped_chunks(M, nnz, N, elem) ? grouped_split(M, nnz) : spmm_split(M, nnz, N, elem);
}
inline size_t spmm_bounds_bytes(int64_t M, int64_t nnz, int64_t N, size_t elem) {
  return (size_t)(planned_split(M, nnz, N, elem).spans + 1) * sizeof(Boundary);
}

// Carry records the workspace must hold: the most any kernel variant produces
// for this shape (one record per chunk of the wide-tile split).
inline int64_t spmm_num_chunks(int64_t M, int64_t nnz, int64_t N, size_t elem) {
  const SpmmSplit sp = spmm_split(M, nnz, N, elem);
  return (M + nnz + sp.items_per_chunk - 1) / sp.items_per_chunk;
}

// The tiled kernel's split (spmm_tiled.hip): one chunk for every wavefront of a resident grid, if the
// chunks are small enough for that; a chunk is then staged once for all tiles.  512 chunks are four
// wavefronts to each of an XCD's 128 SIMDs, 768 six (what its registers allow); other numbers leave
// some CUs with one workgroup more than others, and the XCD waits for them in every tile (528 chunks 0.190 ms, 512
// 0.158 on the decoder shape).  Few items make short chunks: 512 rows of 32, N = 4,096, 64 -> 28 us, 4,096 rows of 64
// of 16,384, N = 512, 172 -> 31.  (spans 0: the shape does not split this way.)
constexpr int kTiledItemsMax = 384;
inline SpmmSplit tiled_split(int64_t M, int64_t nnz, int64_t N, size_t elem) {
  for (const int64_t wavefronts : {512, 768}) {
    int64_t items = (M + nnz + wavefronts - 1) / wavefronts;
    if (items > kTiledItemsMax || N * (int64_t)elem < 2048 || wavefronts * N * (int64_t)elem > ((int64_t)64 << 20)) continue;
    if (items < 16) items = 16;
    return {(int)items, kSnapItems, (M + nnz + items - 1) / items};
  }
  return {0, 0, 0};
}

inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Workspace layout: carry_row int32[num_chunks] padded to 256 bytes, then
// carry_val T[num_chunks * N] padded likewise.
inline size_t spmm_workspace_bytes(int64_t M, int64_t nnz, int64_t N, size_t elem) {
  const size_t usual = (size_t)spmm_num_chunks(M, nnz, N, elem), tiled = (size_t)tiled_split(M, nnz, N, elem).spans;
  const size_t chunks = usual > tiled ? usual : tiled;
  return align_up(chunks * sizeof(int), 256) + align_up(chunks * (size_t)N * elem, 256);
}

// A batch of products over one pattern: one carry_row array, then carry_val for every problem.
inline size_t spmm_batched_workspace_bytes(int64_t batch, int64_t M, int64_t nnz, int64_t N, size_t elem) {
  const size_t chunks = (size_t)spmm_num_chunks(M, nnz, N, elem);
  return align_up(chunks * sizeof(int), 256) + align_up((size_t)batch * chunks * (size_t)N * elem, 256);
}

// Elements per lane.  Rows of B and C need no alignment beyond their elements' (load_vec), and N
// need not be a multiple of the vector: the last lane of a row takes its last VEC columns, some of
// which its neighbour computes as well, to the same bits.  (An odd N with one element per lane
// took longer: a product with N = 37 on 50,021 nodes 43 -> 37 us, N = 15 on 100,000 27 -> 19.)  A full wavefront per row: the widest
// vector (at most 16 bytes) that keeps all 64 lanes busy (64 * VEC <= N), else the narrowest that
// covers N with one column tile.
inline int pick_vec(int64_t N, size_t elem) {
  const int kMaxVec = (int)(16 / elem);
  for (int vec = kMaxVec; vec > 1; vec /= 2)
    if ((int64_t)kWaveSize * vec <= N) return vec;
  for (int vec = 2; vec <= kMaxVec; vec *= 2)
    if (vec <= N && (int64_t)kWaveSize * vec >= N && (int64_t)kWaveSize * (vec / 2) < N) return vec;
  return 1;
}

// A lane group per row: the widest vector not wider than the row, and the lanes (a power of two,
// two at least) that cover it.
template <typename T>
int narrow_vec(int64_t N) {
  int vec = (int)(16 / sizeof(T));
  while (vec > 1 && vec > N) vec /= 2;
  return vec;
}

// Vectors in a column tile, one lane each.  A vector moved back from the row's end (lane_column) shares
// columns with the one before it.  Lanes of one wavefront may: they do everything in step.  Two tiles
// may not: the wavefronts that fold a row (finish_part) read its sums where they stand, and one would
// read what the other has written.  So a last tile of a single such vector is given another by tiles of
// fewer lanes (N = 257: 63 + 2 vectors instead of 64 + 1; as many tiles, the same loads of B).
inline int tile_lanes(int64_t N, int vec) {
  const int64_t vectors = (N + vec - 1) / vec;
  int lanes = kWaveSize;
  if (N % vec != 0)
    while (vectors > lanes && vectors % lanes == 1) --lanes;
  return lanes;
}

// First column of a lane: its place in the row, moved back where the vector would pass the end.
// (>= N: the lane has nothing to do.)
template <int VEC>
__device__ __forceinline__ int lane_column(int col, int N) {
  return col < N && col + VEC > N ? N - VEC : col;
}

// End of the run of equal carry rows that starts at `start` (a member): a 64-way
// search by the whole wavefront.  The members of a run are consecutive, so
// "same row" holds up to the end and nowhere after.
__device__ __forceinline__ int64_t carry_run_end(const int *__restrict__ carry_row, int64_t start,
                                                 int64_t num_chunks, int row) {
  const int lane = wave_lane();
  int64_t last = start, stop = num_chunks;  // a known member; the first position known to lie beyond
  while (stop - last > 1) {
    const int64_t step = (stop - last + kWaveSize) / (kWaveSize + 1);
    const int64_t probe = last + (int64_t)(lane + 1) * step;
    const bool same = probe < stop && carry_row[probe] == row;
    const int members = __popcll(__ballot(same));  // lanes 0 .. members - 1
    const int64_t reached = last + (int64_t)members * step;
    if (members < kWaveSize && reached + step < stop) stop = reached + step;  // lane `members` saw the end
    last = reached;
  }
  return last + 1;
}

// Folds the carries into C.  A wavefront looks at kFixupChunks consecutive
// chunks' carry rows (one lane each, one load); those that head a run of equal
// rows are then taken one after the other by the whole wavefront, lanes on
// columns: the run is summed in chunk order and added to the row of C, with
// the epilogue.  Few chunks leave a carry (see chunk_boundary), so most
// wavefronts only look: fewer, wider-looking wavefronts cost less to start,
// while a matrix of long rows, where every chunk leaves a carry, still has
// its heads spread over many wavefronts.
constexpr int kFixupChunks = 8;
template <typename T, int VEC, int EPI>
__global__ __launch_bounds__(kBlockThreads) void spmm_fixup_kernel(
    int N, int64_t num_chunks, const int *__restrict__ carry_row, const T *__restrict__ carry_val,
    T *__restrict__ C, const T *__restrict__ bias, SpmmBatch batch) {
  using A = typename Acc<T>::type;
  using VecT = Vec<T, VEC>;
  carry_val += blockIdx.y * batch.carry;
  C += blockIdx.y * batch.c;
  const int lane = wave_lane();
  const int64_t wave = (int64_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWaveSize;
  const int64_t c = wave * kFixupChunks + lane;
  int row = -1, after = -1;
  if (lane < kFixupChunks && c < num_chunks) {
    row = carry_row[c];
    after = c + 1 < num_chunks ? carry_row[c + 1] : -1;
    if (row >= 0 && c > 0 && carry_row[c - 1] == row) row = -1;  // not the head of its run
  }
  unsigned long long pending = __ballot(row >= 0);
  while (pending) {  // uniform over the wavefront
    const int owner = __ffsll(pending) - 1;
    pending &= pending - 1;
    const int r = __shfl(row, owner);
    const int64_t start = c - lane + owner;
    // a run of one, the usual case, needs no search
    const int64_t end = __shfl(after, owner) != r ? start + 1 : carry_run_end(carry_row, start, num_chunks, r);
    for (int col0 = lane * VEC; col0 < N; col0 += kWaveSize * VEC) {
      VecT *dst = reinterpret_cast<VecT *>(C + (size_t)r * (size_t)N + col0);
      VecT o = *dst;  // issued before the carries so that both are in flight together
      // groups of kFoldGroup carries, then the groups' sums: the order of finish_part
      A sum[VEC];
#pragma unroll
      for (int v = 0; v < VEC; ++v) sum[v] = (A)0;
      int64_t e = start;
      constexpr int kBatch = 2 * kFoldGroup;  // loads in flight: a long row spans hundreds of chunks
      for (; e + kBatch <= end; e += kBatch) {
        VecT part[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
          part[u] = *reinterpret_cast<const VecT *>(carry_val + (size_t)(e + u) * (size_t)N + col0);
#pragma unroll
        for (int h = 0; h < kBatch; h += kFoldGroup) {
          A group[VEC];
#pragma unroll
          for (int v = 0; v < VEC; ++v) group[v] = (A)0;
#pragma unroll
          for (int u = 0; u < kFoldGroup; ++u)
#pragma unroll
            for (int v = 0; v < VEC; ++v) group[v] += (A)part[h + u].v[v];
#pragma unroll
          for (int v = 0; v < VEC; ++v) sum[v] += (A)(T)group[v];
        }
      }
      while (e < end) {
        A group[VEC];
#pragma unroll
        for (int v = 0; v < VEC; ++v) group[v] = (A)0;
        const int64_t stop = e + kFoldGroup < end ? e + kFoldGroup : end;
        for (; e < stop; ++e) {
          const VecT part = *reinterpret_cast<const VecT *>(carry_val + (size_t)e * (size_t)N + col0);
#pragma unroll
          for (int v = 0; v < VEC; ++v) group[v] += (A)part.v[v];
        }
#pragma unroll
        for (int v = 0; v < VEC; ++v) sum[v] += (A)(T)group[v];
      }
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const T b = EPI != kEpiNone ? bias[col0 + v] : (T)0;
        o.v[v] = apply_epilogue<T, EPI>(sum[v] + (A)o.v[v], b);
      }
      *dst = o;
    }
  }
}

// ---- which kernel: estimates in microseconds --------------------------------------------------------
// Fitted to 70 shapes between 256 x 1,024 and 8,192 x 8,192, 8 to 800 entries a row, N = 32 to 4,096, on
// which they are within a third; kernels that differ by less than that are close to each other anyway.
//
// The row-split kernel: what the L2s hand out, 21 TB/s while the K rows of a column tile (1 KiB) fit one
// of them, 9.5 when most gathers miss.
inline double spmm_rows_us(int64_t M, int64_t K, int64_t N, int64_t nnz) {
  const double slice = (double)K * (double)(N * 4 < 1024 ? N * 4 : 1024) / (1 << 20);
  return 2.5 + (double)nnz * (double)N * 4 / (slice <= 4 ? 21e6 : slice <= 8 ? 15e6 : 9.5e6) + (double)M * (double)N * 4 / 4e6;
}
// Turning a transposed operand first, and reading it from memory rather than the L2s after that.
inline double dense_turn_us(int64_t K, int64_t N) {
  const double us = 4.5 + (double)K * (double)N * 4 / 0.7e6;
  return us < 12 ? us : 12;
}
// The tiled kernel: an XCD's tiles one after the other.
inline double spmm_tiled_us(int64_t K, int64_t N, int64_t nnz) {
  const int64_t rounds = ((N * 4 + 127) / 128 + 7) / 8;
  return 2.5 + (double)rounds * (1.0 + (double)nnz * 128 / (K <= 4096 ? 4.2e6 : 3.3e6));
}

}  // namespace scorch
