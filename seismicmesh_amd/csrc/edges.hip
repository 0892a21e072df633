// Sorted unique edges and the per-vertex edge lists the force scatter uses.
//
// Replaces SeismicMesh/geometry/cpp/fast_geometry.cpp:49-77 (unique_edges:
// (min,max) per pair, std::sort, std::unique) as called by
// generation/mesh_generator.py:680-688 (_get_edges).
//
// Method: the sort key of an edge is (min, max) with min a vertex id, so the
// lexicographic sort is a counting sort on min (one bucket per vertex: a
// histogram, an exclusive scan and a scatter) followed by a sort of each
// bucket's max ids.  Cells near each other in the list share most of their
// edges, so a block first drops the duplicates among its own cells in LDS
// and only what is left is counted and scattered.  Buckets then hold a
// vertex's higher neighbours and few duplicates: up to 16 ids are sorted in
// one thread's registers, up to 64 by one wave, one id per lane; long
// buckets (arbitrary user input) by a whole workgroup in LDS or, beyond
// that, in global memory.  The remaining duplicates are dropped inside each
// sorted bucket; a second scan turns the per-bucket unique counts into
// output offsets.  For a 2D triangulation with neighbour links each shared
// edge is produced once in the first place (by the lower-numbered of its two
// cells) and neither the LDS pass nor the second scan is needed.  The output
// is exactly the reference's sorted unique edge list.
#include "common.h"
#include "edges.h"

namespace smk {

namespace {

// Cells of 2D triangulations with neighbour links: adj[3 c + k] is the cell
// across the edge opposite local vertex k, or < 0.  An edge shared by two
// kept cells is produced once, by the lower-numbered one, so every bucket is
// free of duplicates and its offsets are the output offsets.
struct LinkSrc {
  static constexpr int per = 3;
  const int32_t *cells;
  const uint8_t *keep;  // optional cell mask
  const int32_t *adj;
  int64_t n;
  __device__ inline bool get(int64_t i, int j, int32_t &a, int32_t &b) const {
    if (keep && !keep[i]) return false;
    // local edge j joins vertices j and (j + 1) % 3: opposite vertex (j + 2) % 3
    const int32_t o = adj[3 * i + (j + 2) % 3];
    if (o >= 0 && o < i && (!keep || keep[o])) return false;
    const int32_t u = cells[3 * i + j], v = cells[3 * i + (j + 1) % 3];
    a = u < v ? u : v;
    b = u < v ? v : u;
    return true;
  }
};

// Few pairs for the number of vertices: counted and scattered as they are.
struct PairSrc {
  static constexpr int per = 1;
  const int32_t *pairs;
  int64_t n;
  __device__ inline bool get(int64_t i, int, int32_t &a, int32_t &b) const {
    const int32_t u = pairs[2 * i], v = pairs[2 * i + 1];
    a = u < v ? u : v;
    b = u < v ? v : u;
    return true;
  }
};

// Items without links: pairs (NV = 2), triangles (3) or tetrahedra (4).  A
// block of kItemThreads threads takes kPer items a thread.
struct ItemSrc {
  const int32_t *ids;   // NV per item
  const uint8_t *keep;  // optional mask
  int64_t n;
};
constexpr int kItemThreads = 512;
constexpr int kTable = 4096;  // LDS hash slots (vertices, pairs), 12 bits
template <int NV>
struct ItemShape {
  static constexpr int pairs = NV == 2 ? 1 : (NV == 3 ? 3 : 6);
  static constexpr int per = NV == 4 ? 1 : 2;
  static constexpr int items = kItemThreads * per;
  static constexpr int cap = items * pairs;  // pairs of one block
  static_assert(cap <= kTable * 3 / 4 && items * NV <= kTable * 3 / 4, "tables stay 3/4 full");
};

__device__ inline uint32_t hash12(uint32_t x) { return (x * 2654435761u) >> 20; }

// slot of v in an open-addressed LDS table (-1: empty), inserted if new.
// Sixteen consecutive vertices start at consecutive slots, so that the
// lanes that walk the table touch whole lines of the per-vertex arrays.
__device__ inline int vertex_slot(int32_t *vk, int32_t v) {
  uint32_t h = (hash12((uint32_t)v >> 4) & ~15u) | ((uint32_t)v & 15);
  for (;;) {
    int32_t o = vk[h];
    if (o == v) return (int)h;
    if (o == -1) o = atomicCAS(&vk[h], -1, v);
    if (o == -1 || o == v) return (int)h;
    h = (h + 1) & (kTable - 1);
  }
}

// The distinct pairs among a block's items: vertices become their slot in an
// LDS table (12 bits), a pair the 24-bit key of its two slots in a second
// one.  The distinct pairs are appended to the block's segment of `list`
// (cap pairs, see item_count for its length) and counted by first endpoint,
// one global atomic per distinct endpoint of the block.
// Bound by the atomics: 2.8 M lattice tetrahedra have 17 M pairs, 5 M after
// this pass; counting and scattering runs of sorted ids straight from the
// cells took 110 + 153 us, this pass and k_item_scatter 67 + 50 us.
template <int NV>
__global__ __launch_bounds__(kItemThreads) void k_item_count(ItemSrc src, int32_t *cnt,
                                                            int2 *list) {
  using S = ItemShape<NV>;
  __shared__ int32_t vk[kTable], vc[kTable];
  __shared__ uint32_t pk[kTable];
  __shared__ int32_t npairs;
  const int tid = threadIdx.x;
  const int64_t blk = xcd_block();
  for (int k = tid; k < kTable; k += kItemThreads) {
    vk[k] = -1;
    vc[k] = 0;
    pk[k] = ~0u;
  }
  if (tid == 0) npairs = 0;
  __syncthreads();
#pragma unroll
  for (int it = 0; it < S::per; ++it) {
    const int64_t i = blk * S::items + it * kItemThreads + tid;
    if (i >= src.n || (src.keep && !src.keep[i])) continue;
    int32_t v[NV];
    int sl[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = src.ids[NV * i + k];
#pragma unroll
    for (int k = 0; k < NV; ++k) sl[k] = vertex_slot(vk, v[k]);
#pragma unroll
    for (int x = 0; x < NV; ++x)
#pragma unroll
      for (int y = x + 1; y < NV; ++y) {
        const uint32_t key =
            v[x] < v[y] ? (uint32_t)(sl[x] << 12 | sl[y]) : (uint32_t)(sl[y] << 12 | sl[x]);
        uint32_t h = hash12(key);
        for (;;) {
          uint32_t o = pk[h];
          if (o == key) break;
          if (o == ~0u) o = atomicCAS(&pk[h], ~0u, key);
          if (o == ~0u || o == key) break;
          h = (h + 1) & (kTable - 1);
        }
      }
  }
  __syncthreads();
  int2 *seg = list + blk * S::cap;
  const int lane = tid % 64;
  for (int k = tid; k < kTable; k += kItemThreads) {
    const uint32_t key = pk[k];
    const uint64_t m = __ballot(key != ~0u);
    int32_t base = 0;
    if (lane == 0 && m) base = atomicAdd(&npairs, (int32_t)__popcll(m));
    base = __shfl(base, 0);
    if (key != ~0u) {
      atomicAdd(&vc[key >> 12], 1);
      seg[base + (int32_t)__popcll(m & ((1ull << lane) - 1))] =
          make_int2(vk[key >> 12], vk[key & (kTable - 1)]);
    }
  }
  __syncthreads();
  for (int k = tid; k < kTable; k += kItemThreads)
    if (vc[k]) atomicAdd(&cnt[vk[k]], vc[k]);
  // the last segment is cut off at the last item
  const int64_t left = src.n - blk * S::items;
  const int32_t cap = (int32_t)(left < S::items ? left : S::items) * S::pairs;
  if (tid == 0 && npairs < cap) seg[cap - 1] = make_int2(~npairs, 0);
}

// The listed pairs into their buckets: the block ranks its pairs by first
// endpoint in LDS and reserves each bucket's slots with one global atomic.
template <int NV>
__global__ __launch_bounds__(kItemThreads) void k_item_scatter(int64_t n, const int2 *list,
                                                              const int32_t *rowptr, int32_t *cur,
                                                              int32_t *col) {
  using S = ItemShape<NV>;
  constexpr int R = S::cap / kItemThreads;
  __shared__ int32_t vk[kTable], vc[kTable];
  const int tid = threadIdx.x;
  const int64_t blk = xcd_block();
  if (blk * S::items >= n) return;
  for (int k = tid; k < kTable; k += kItemThreads) {
    vk[k] = -1;
    vc[k] = 0;
  }
  const int2 *seg = list + blk * S::cap;
  const int64_t left = n - blk * S::items;
  const int32_t cap = (int32_t)(left < S::items ? left : S::items) * S::pairs;
  // a segment that is not full ends with the complement of its length
  const int32_t last = seg[cap - 1].x;
  const int32_t m = last < 0 ? ~last : cap;
  __syncthreads();
  int32_t b[R], sl[R], rank[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int32_t e = k * kItemThreads + tid;
    if (e >= m) continue;
    const int2 pr = seg[e];
    b[k] = pr.y;
    sl[k] = vertex_slot(vk, pr.x);
    rank[k] = atomicAdd(&vc[sl[k]], 1);
  }
  __syncthreads();
  for (int k = tid; k < kTable; k += kItemThreads)
    if (vc[k]) vc[k] = rowptr[vk[k]] + atomicAdd(&cur[vk[k]], vc[k]);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < R; ++k)
    if (k * kItemThreads + tid < m) col[vc[sl[k]] + rank[k]] = b[k];
}

// cnt2 (optional): the same edges counted by their second endpoint
template <class Src>
__global__ void k_count(Src src, int32_t *cnt, int32_t *cnt2) {
  int64_t i = (int64_t)xcd_block() * blockDim.x + threadIdx.x;
  if (i >= src.n) return;
  for (int j = 0; j < Src::per; ++j) {
    int32_t a, b;
    if (src.get(i, j, a, b)) {
      atomicAdd(&cnt[a], 1);
      if (cnt2) atomicAdd(&cnt2[b], 1);
    }
  }
}

template <class Src>
__global__ void k_scatter(Src src, const int32_t *rowptr, int32_t *cur, int32_t *col) {
  int64_t i = (int64_t)xcd_block() * blockDim.x + threadIdx.x;
  if (i >= src.n) return;
  for (int j = 0; j < Src::per; ++j) {
    int32_t a, b;
    if (src.get(i, j, a, b)) {
      int32_t pos = rowptr[a] + atomicAdd(&cur[a], 1);
      col[pos] = b;
    }
  }
}

constexpr int kRegSort = 16;    // buckets up to this size: per-thread sort
constexpr int kWaveSort = 64;   // up to this size: one wave, one id per lane
constexpr int kLdsSort = 4096;  // up to this size: one workgroup, LDS bitonic

// Sorts 16 register values with a bitonic network: every index is a
// compile-time constant after unrolling, so the values never leave VGPRs.
__device__ inline void sort16(int32_t (&v)[16]) {
#pragma unroll
  for (int size = 2; size <= 16; size <<= 1) {
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int j = k ^ stride;
        if (j > k) {
          const bool up = (k & size) == 0;
          int32_t a = v[k], b = v[j];
          int32_t lo = a < b ? a : b, hi = a < b ? b : a;
          v[k] = up ? lo : hi;
          v[j] = up ? hi : lo;
        }
      }
    }
  }
}

constexpr int kRows = 256;    // buckets of one workgroup (and its threads)
constexpr int kFewRows = 32;  // the same where buckets are few and long
constexpr int kStage = 4096;  // ids staged in LDS for them
// kFewRows buckets a workgroup up to this many buckets of 8 ids and more (1024
// workgroups, what the chip holds at once)
constexpr int64_t kDenseRows = 32768;
// lists of pairs up to this long, and fewer than 8 to a vertex, are counted as
// they are
constexpr int64_t kPlainPairs = 16384;

// Sorts one id per lane (INT32_MAX past the bucket's end wl) with a bitonic
// network, partners exchanged by lane shuffles, and writes the distinct ids
// to b; returns their number.
__device__ inline int32_t sort_wave(int32_t *b, int32_t wl) {
  const int lane = threadIdx.x % 64;
  int32_t v = lane < wl ? b[lane] : INT32_MAX;
#pragma unroll
  for (int size = 2; size <= 64; size <<= 1) {
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      const int32_t o = __shfl_xor(v, stride);
      const bool up = (lane & size) == 0;
      const bool low = (lane & stride) == 0;
      // the lower lane of a pair keeps the smaller value in an ascending
      // block, the larger in a descending one
      v = (low == up) ? (v < o ? v : o) : (v < o ? o : v);
    }
  }
  const int32_t prev = __shfl_up(v, 1);
  const bool first = lane < wl && (lane == 0 || v != prev);
  const uint64_t m = __ballot(first);
  if (first) b[(int32_t)__popcll(m & ((1ull << lane) - 1))] = v;
  return (int32_t)__popcll(m);
}

// Sorts R consecutive buckets and leaves each one's distinct ids, ascending,
// at its start.  The buckets are one contiguous piece of col, moved through
// LDS in whole lines (in global memory if it is longer than kStage or, with
// STAGE false, for short lists and buckets of about one id, where the threads'
// own reads are whole lines: 3 M of them 29 us through LDS, 25 without); a
// thread sorts its own bucket if short, a wave the ones of up to kWaveSort
// ids one after the other; longer ones are listed (one atomic per wave that
// has any) for the workgroup pass.  Listing the middle ones too and sorting
// them in a pass of their own took 95 + 139 us on 512 k lattice vertices; now
// 17 us.  R = kFewRows spreads the middle ones over all waves of a workgroup:
// 1.7 k buckets of 20 to 60 ids, 64 of them to a wave 57 us, 8 to a wave 12.
template <int R, bool STAGE>
__global__ __launch_bounds__(kRows) void k_row_sort(int64_t nrows, const int32_t *rowptr,
                                                    int32_t *col, int32_t *ucnt,
                                                    int32_t *long_rows, int32_t *nlong) {
  __shared__ int32_t sh[STAGE ? kStage : 1];
  __shared__ int32_t piece[R < kRows ? R + 1 : 1];
  const int tid = threadIdx.x, lane = tid % 64;
  const int64_t r0 = (int64_t)xcd_block() * R, r = r0 + tid;
  if (r == 0) ucnt[nrows] = 0;  // the scan's last input (its total slot)
  if (r0 >= nrows) return;
  const int64_t r1 = r0 + R < nrows ? r0 + R : nrows;
  const int32_t c0 = STAGE ? rowptr[r0] : 0, n = STAGE ? rowptr[r1] - c0 : 0;
  const bool staged = STAGE && n <= kStage;
  if (R < kRows) {
    if (tid <= R) piece[tid] = rowptr[r < nrows ? r : nrows] - c0;
    __syncthreads();
  }
  int32_t *buf = col + c0;
  if (staged) {
    for (int32_t k = tid; k < n; k += kRows) sh[k] = buf[k];
    __syncthreads();
    buf = sh;
  }
  const bool row = tid < R && r < nrows;
  const int32_t s = row ? rowptr[r] - c0 : 0, len = row ? rowptr[r + 1] - c0 - s : 0;
  const uint64_t lm = __ballot(len > kWaveSort);
  if (lm) {
    const int lead = __builtin_ctzll(lm);
    int32_t base = 0;
    if (lane == lead) base = atomicAdd(nlong, (int32_t)__popcll(lm));
    base = __shfl(base, lead);
    if (len > kWaveSort) {
      long_rows[base + (int32_t)__popcll(lm & ((1ull << lane) - 1))] = (int32_t)r;
      ucnt[r] = 0;  // filled by the workgroup pass
    }
  }
  if (row && len <= kRegSort) {
    int32_t v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = k < len ? buf[s + k] : INT32_MAX;
    sort16(v);
    int32_t u = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (k < len && (k == 0 || v[k] != v[k - 1])) buf[s + u++] = v[k];
    ucnt[r] = u;
  }
  if (R < kRows) {
    for (int w = tid / 64; w < R; w += kRows / 64) {
      const int32_t ws = piece[w], wl = piece[w + 1] - ws;
      if (wl <= kRegSort || wl > kWaveSort) continue;
      const int32_t u = sort_wave(buf + ws, wl);
      if (lane == 0) ucnt[r0 + w] = u;
    }
  } else {
    for (uint64_t mid = __ballot(len > kRegSort && len <= kWaveSort); mid; mid &= mid - 1) {
      const int w = __builtin_ctzll(mid);
      const int32_t ws = __shfl(s, w), wl = __shfl(len, w);
      const int32_t u = sort_wave(buf + ws, wl);
      if (lane == w) ucnt[r] = u;
    }
  }
  if (!staged) return;
  __syncthreads();
  for (int32_t k = tid; k < n; k += kRows) col[c0 + k] = sh[k];
}

// Long buckets, one workgroup each: a bitonic sort in LDS (padded with
// INT32_MAX) for buckets up to kLdsSort ids (pass `big` = false, many
// workgroups), or in the global staging area for longer ones (pass `big` =
// true, launched with a single workgroup so the staging area is private).
__device__ inline void long_sort_rows(unsigned b, unsigned nb, const int32_t *long_rows,
                                      const int32_t *nlong, const int32_t *rowptr, int32_t *col,
                                      int32_t *ucnt, int32_t *stage, int big, int32_t *sh,
                                      int32_t *red) {
  const int nl = *nlong;
  for (int li = (int)b; li < nl; li += (int)nb) {
    const int32_t r = long_rows[li];
    const int32_t s = rowptr[r], e = rowptr[r + 1];
    const int32_t len = e - s;
    int32_t p2 = 1;
    while (p2 < len) p2 <<= 1;
    const bool lds = p2 <= kLdsSort;
    if (lds == (big != 0)) continue;
    int32_t *buf = lds ? sh : stage;
    for (int32_t k = threadIdx.x; k < p2; k += blockDim.x) buf[k] = k < len ? col[s + k] : INT32_MAX;
    __threadfence_block();
    __syncthreads();
    for (int32_t size = 2; size <= p2; size <<= 1) {
      for (int32_t stride = size >> 1; stride > 0; stride >>= 1) {
        for (int32_t k = threadIdx.x; k < p2; k += blockDim.x) {
          int32_t j = k ^ stride;
          if (j > k) {
            bool up = (k & size) == 0;
            int32_t x = buf[k], y = buf[j];
            if ((x > y) == up) {
              buf[k] = y;
              buf[j] = x;
            }
          }
        }
        __threadfence_block();
        __syncthreads();
      }
    }
    // the distinct ids to the bucket's start, each thread a piece of them
    const int32_t piece = (len + (int32_t)blockDim.x - 1) / (int32_t)blockDim.x;
    const int32_t k0 = piece * (int32_t)threadIdx.x;
    const int32_t k1 = k0 + piece < len ? k0 + piece : len;
    int32_t u = 0;
    for (int32_t k = k0; k < k1; ++k) u += (k == 0 || buf[k] != buf[k - 1]);
    red[threadIdx.x] = u;
    __syncthreads();
    if (threadIdx.x == 0) {
      int32_t t = 0;
      for (int k = 0; k < (int)blockDim.x; ++k) {
        const int32_t c = red[k];
        red[k] = t;
        t += c;
      }
      ucnt[r] = t;
    }
    __syncthreads();
    u = red[threadIdx.x];
    for (int32_t k = k0; k < k1; ++k)
      if (k == 0 || buf[k] != buf[k - 1]) col[s + u++] = buf[k];
    __syncthreads();
  }
}

// workgroups for the LDS-sized long buckets: a graded 3D mesh has
// thousands of rows over 64 ids (vertices where the size changes), and
// 64 workgroups working through them one bitonic sort at a time took
// 150-400 us per launch on the EAGE-shaped workload; idle ones exit at once
constexpr unsigned kLongBlocks = 1024;

// The long buckets, in one launch of 256-thread workgroups: the first
// kLongBlocks take the LDS-sized ones, the last one the buckets sorted in
// the global staging area (one workgroup, so the staging area is private to
// it).
__global__ void k_long_sorts(const int32_t *long_rows, const int32_t *nlong,
                             const int32_t *rowptr, int32_t *col, int32_t *ucnt, int32_t *stage) {
  __shared__ int32_t sh[kLdsSort];
  __shared__ int32_t red[256];
  const unsigned b = blockIdx.x;
  if (b < kLongBlocks)
    long_sort_rows(b, kLongBlocks, long_rows, nlong, rowptr, col, ucnt, stage, 0, sh, red);
  else
    long_sort_rows(0, 1, long_rows, nlong, rowptr, col, ucnt, stage, 1, sh, red);
}

// The edges of kRows consecutive buckets, one contiguous piece of the
// output, a thread per edge so that both the ids' reads and the edges'
// writes are whole lines; an edge finds its bucket by bisecting the
// buckets' offsets in LDS.  (A wave per bucket took 70 us for 3.5 M edges,
// now 12 us.)  len (optional): only that many of a bucket's slots are written.
__global__ __launch_bounds__(kRows) void k_emit(int64_t nrows, const int32_t *rowptr,
                                                const int32_t *col, const int32_t *eptr,
                                                const int32_t *len, int32_t *edges,
                                                SecondLists second) {
  __shared__ int32_t off[kRows + 1], start[kRows];
  const int tid = threadIdx.x;
  const int64_t r0 = (int64_t)xcd_block() * kRows;
  if (r0 >= nrows) return;
  const int nr = (int)(nrows - r0 < kRows ? nrows - r0 : kRows);
  if (tid < nr) {
    off[tid] = eptr[r0 + tid];
    start[tid] = rowptr[r0 + tid];
  }
  if (tid == 0) off[nr] = eptr[r0 + nr];
  __syncthreads();
  for (int32_t o = off[0] + tid; o < off[nr]; o += kRows) {
    int lo = 0, hi = nr;  // off[lo] <= o < off[hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) / 2;
      if (off[mid] <= o) lo = mid;
      else hi = mid;
    }
    if (len && o - off[lo] >= len[r0 + lo]) continue;
    const int32_t b = col[start[lo] + (o - off[lo])];
    edges[2 * (int64_t)o] = (int32_t)(r0 + lo);
    edges[2 * (int64_t)o + 1] = b;
    if (second.list) second.list[second.ptr[b] + atomicAdd(&second.cur[b], 1)] = o;
  }
}

__global__ void k_count_to_i64(const int32_t *c, int64_t *out) { *out = (int64_t)*c; }

template <int NV>
int item_pass(const ItemSrc &src, bool count, int32_t *rowptr, int32_t *cur, int2 *list,
              int32_t *col, hipStream_t s) {
  const dim3 grid(blocks_for(src.n, ItemShape<NV>::items));
  if (count)
    hipLaunchKernelGGL((k_item_count<NV>), grid, dim3(kItemThreads), 0, s, src, rowptr, list);
  else
    hipLaunchKernelGGL((k_item_scatter<NV>), grid, dim3(kItemThreads), 0, s, src.n,
                       (const int2 *)list, (const int32_t *)rowptr, cur, col);
  SM_LAUNCH_CHECK();
  return SM_OK;
}

inline size_t al(size_t b) { return (b + 255) & ~(size_t)255; }

}  // namespace

size_t unique_edges_workspace(int64_t npairs, int64_t nvert) {
  size_t b = 0;
  b += al((nvert + 1) * 4);  // cnt -> rowptr
  b += al((nvert + 1) * 4);  // cur
  b += al(npairs * 4);       // col
  b += al((nvert + 1) * 4);  // ucnt -> eptr
  b += al((nvert + 1) * 4);  // long rows
  b += al((nvert + 1) * 4);  // unused; the size a caller asks for stays what it was
  b += al(8 * 4);            // counters
  b += al((size_t)npairs * 2 * 4 + 4096 * 4);  // blocks' pairs; staging for very long buckets
  b += 2 * scan_workspace(nvert + 1);
  return b;
}

int32_t *unique_edges_offsets(void *ws, int64_t npairs, int64_t nvert, bool adj) {
  // workspace order: rowptr, cur, col, eptr (see unique_edges_run); with
  // neighbour links the bucket offsets are the output offsets
  char *w = reinterpret_cast<char *>(ws);
  if (adj) return reinterpret_cast<int32_t *>(w);
  w += al((nvert + 1) * 4);
  w += al((nvert + 1) * 4);
  w += al(npairs * 4);
  return reinterpret_cast<int32_t *>(w);
}

int unique_edges_run(const int32_t *pairs, const int32_t *cells, const uint8_t *keep,
                     const int32_t *adj, const SecondLists *second, int dim, int64_t n,
                     int64_t npairs, int64_t nvert, int32_t *edges, int32_t *count32,
                     int64_t *count64, void *ws, size_t ws_bytes, hipStream_t s) {
  SM_CHECK(!adj || (cells && dim == 2), SM_ERR_ARG, "unique edges: adjacency needs 2D cells");
  SM_CHECK(!second || (adj && second->ptr && second->cur && second->list), SM_ERR_ARG,
           "unique edges: second-endpoint lists need neighbour links");
  const SecondLists sl = second ? *second : SecondLists{nullptr, nullptr, nullptr};
  SM_CHECK(ws_bytes >= unique_edges_workspace(npairs, nvert), SM_ERR_CAPACITY,
           "unique edges: workspace %zu < %zu bytes", ws_bytes,
           unique_edges_workspace(npairs, nvert));
  char *w = reinterpret_cast<char *>(ws);
  int32_t *rowptr = reinterpret_cast<int32_t *>(w); w += al((nvert + 1) * 4);
  int32_t *cur = reinterpret_cast<int32_t *>(w); w += al((nvert + 1) * 4);
  int32_t *col = reinterpret_cast<int32_t *>(w); w += al(npairs * 4);
  int32_t *eptr = reinterpret_cast<int32_t *>(w); w += al((nvert + 1) * 4);
  int32_t *longr = reinterpret_cast<int32_t *>(w); w += al((nvert + 1) * 4);
  w += al((nvert + 1) * 4);
  int32_t *ctr = reinterpret_cast<int32_t *>(w); w += al(8 * 4);
  int32_t *stage = reinterpret_cast<int32_t *>(w);
  w += al((size_t)npairs * 2 * 4 + 4096 * 4);
  void *sws = w;

  int rc;
  {
    FillList fl{{rowptr, cur, ctr, sl.ptr, sl.cur}, {nvert + 1, nvert + 1, 8, nvert + 1, nvert + 1}};
    if ((rc = fill_list(fl, second ? 5 : 3, 0, s))) return rc;
  }
  const int B = 256;
  int32_t *total = count32 ? count32 : ctr + 3;
  const LinkSrc link{cells, keep, adj, n};
  const ItemSrc item{cells ? cells : pairs, keep, n};
  // Pairs of which there is no more than one to a vertex share little that a
  // block could drop or count together, and small lists do not pay for the
  // tables.  (The 3 M edges of a path: 163 us through the tables, 122 as they
  // are; in a random order 393 and 356; 16 k random pairs of 5 k vertices 50
  // and 32-37.  With 1.5 pairs to a vertex, sorted, 93 and 114; in a random
  // order 205 and 192.  4.3 k pairs of 216 vertices 32 and 40.)
  const bool plain = !cells && (n <= nvert || (n <= kPlainPairs && n < 8 * nvert));
  const PairSrc pair{pairs, n};
  const auto items = [&](bool count) {
    int2 *list = reinterpret_cast<int2 *>(stage);
    if (plain && count) {
      hipLaunchKernelGGL(k_count<PairSrc>, dim3(blocks_for(n, B)), dim3(B), 0, s, pair, rowptr,
                         (int32_t *)nullptr);
      SM_LAUNCH_CHECK();
      return (int)SM_OK;
    }
    if (plain) {
      hipLaunchKernelGGL(k_scatter<PairSrc>, dim3(blocks_for(n, B)), dim3(B), 0, s, pair,
                         (const int32_t *)rowptr, cur, col);
      SM_LAUNCH_CHECK();
      return (int)SM_OK;
    }
    if (!cells) return item_pass<2>(item, count, rowptr, cur, list, col, s);
    if (dim == 2) return item_pass<3>(item, count, rowptr, cur, list, col, s);
    return item_pass<4>(item, count, rowptr, cur, list, col, s);
  };
  if (n > 0 && adj) {
    hipLaunchKernelGGL(k_count<LinkSrc>, dim3(blocks_for(n, B)), dim3(B), 0, s, link, rowptr, sl.ptr);
    SM_LAUNCH_CHECK();
  } else if (n > 0 && (rc = items(true))) {
    return rc;
  }
  // with adjacency the buckets hold no duplicates: their offsets and total
  // are the output's
  if (second)
    rc = scan_exclusive2(rowptr, rowptr, total, sl.ptr, sl.ptr, nullptr, nvert + 1, sws, s);
  else
    rc = scan_exclusive(rowptr, rowptr, nvert + 1, adj ? total : ctr + 1, sws, s);
  if (rc) return rc;
  if (n > 0 && adj) {
    hipLaunchKernelGGL(k_scatter<LinkSrc>, dim3(blocks_for(n, B)), dim3(B), 0, s, link,
                       (const int32_t *)rowptr, cur, col);
    SM_LAUNCH_CHECK();
  } else if (n > 0 && (rc = items(false))) {
    return rc;
  }
  if (nvert > 0) {
    if (!adj && nvert <= kDenseRows && npairs >= 8 * nvert)
      hipLaunchKernelGGL((k_row_sort<kFewRows, true>), dim3(blocks_for(nvert, kFewRows)),
                         dim3(kRows), 0, s, nvert, (const int32_t *)rowptr, col, eptr, longr,
                         ctr + 2);
    else if (plain)
      hipLaunchKernelGGL((k_row_sort<kRows, false>), dim3(blocks_for(nvert, kRows)), dim3(kRows), 0,
                         s, nvert, (const int32_t *)rowptr, col, eptr, longr, ctr + 2);
    else
      hipLaunchKernelGGL((k_row_sort<kRows, true>), dim3(blocks_for(nvert, kRows)), dim3(kRows), 0, s,
                         nvert, (const int32_t *)rowptr, col, eptr, longr, ctr + 2);
    SM_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_long_sorts, dim3(kLongBlocks + 1), dim3(256), 0, s, longr, ctr + 2,
                       rowptr, col, eptr, stage);
    SM_LAUNCH_CHECK();
  }
  if (!adj) {
    if (nvert == 0 && (rc = fill<int32_t>(eptr, 1, 0, s))) return rc;
    if ((rc = scan_exclusive(eptr, eptr, nvert + 1, total, sws, s))) return rc;
  }
  if (nvert > 0) {
    hipLaunchKernelGGL(k_emit, dim3(blocks_for(nvert, kRows)), dim3(kRows), 0, s, nvert, rowptr,
                       col, adj ? (const int32_t *)rowptr : (const int32_t *)eptr,
                       adj ? (const int32_t *)eptr : nullptr, edges, sl);
    SM_LAUNCH_CHECK();
  }
  if (count64) {
    hipLaunchKernelGGL(k_count_to_i64, dim3(1), dim3(1), 0, s, total, count64);
    SM_LAUNCH_CHECK();
  }
  return SM_OK;
}

}  // namespace smk

extern "C" size_t sm_unique_edges_workspace(int64_t npairs, int64_t nvert) {
  return smk::unique_edges_workspace(npairs, nvert);
}

extern "C" int sm_unique_edges(const int32_t *pairs, int64_t npairs, int64_t nvert,
                               int32_t *edges, int64_t *count, void *ws, size_t ws_bytes,
                               void *stream) {
  SM_CHECK(npairs >= 0 && nvert >= 0, SM_ERR_ARG, "unique_edges: negative size");
  SM_CHECK(npairs == 0 || (pairs && edges), SM_ERR_ARG, "unique_edges: null pointer");
  SM_CHECK(count && ws, SM_ERR_ARG, "unique_edges: null count/workspace");
  return smk::unique_edges_run(pairs, nullptr, nullptr, nullptr, nullptr, 2, npairs, npairs, nvert,
                               edges, nullptr, count, ws, ws_bytes, smk::stream_of(stream));
}

extern "C" size_t sm_cell_edges_workspace(int64_t ncells, int dim, int64_t nvert) {
  return smk::unique_edges_workspace(ncells * (dim == 2 ? 3 : 6), nvert);
}

extern "C" int sm_cell_edges(const int32_t *cells, int64_t ncells, int dim, int64_t nvert,
                             int32_t *edges, int64_t *count, void *ws, size_t ws_bytes,
                             void *stream) {
  SM_CHECK(dim == 2 || dim == 3, SM_ERR_ARG, "cell_edges: dim must be 2 or 3");
  SM_CHECK(ncells >= 0 && nvert >= 0, SM_ERR_ARG, "cell_edges: negative size");
  SM_CHECK(ncells == 0 || (cells && edges), SM_ERR_ARG, "cell_edges: null pointer");
  SM_CHECK(count && ws, SM_ERR_ARG, "cell_edges: null count/workspace");
  int64_t np = ncells * (dim == 2 ? 3 : 6);
  return smk::unique_edges_run(nullptr, cells, nullptr, nullptr, nullptr, dim, ncells, np, nvert,
                               edges, nullptr, count, ws, ws_bytes, smk::stream_of(stream));
}
