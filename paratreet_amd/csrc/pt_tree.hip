// Octree build over sorted Morton keys, all levels at once.
//
// Reference: Subtree::buildTree / recursiveBuild / getType (src/Subtree.h:
// 262-349), OctTree::findChildsLastParticle (src/Modularization.C:60-65) and
// the key helpers of src/Utility.h:9-130.  The reference recurses depth-first;
// here the whole tree follows from local comparisons of the sorted keys.  With
// c(a, b) the number of leading octal digits keys a and b share, the cell of
// depth d that holds particle i
//   - starts at i when c(i - 1, i) < d, and then holds more than B particles
//     exactly when c(i, i + B) >= d, so the internal nodes starting at i are
//     the depths (c(i - 1, i), c(i, i + B)];
//   - is a leaf starting at i at depth c(i, i + B) + 1 when an internal node
//     starts at i, and otherwise at depth c(i - 1, i) + 1 when the deepest
//     cell i shares with i - 1 is internal.
// Four launches, whatever the depth: per-wave counts of internal nodes by
// depth and of leaves (tree_count_kernel), one exclusive scan of the counts in
// (depth, wave) order (tree_scan_kernel: level order, and particle order
// inside a level), each internal node's id and each leaf's bucket
// (tree_assign_kernel), and the 8 children records of every internal node
// (tree_children_kernel).  The 8 children of a node get consecutive ids, so a
// node stores only its first child.  Node identity across implementations is
// the key.
//
// Why not a launch per level: every level's cost was its ~20 dependent key
// loads and its launch, 11 launches (104 us) at 1M particles, and the leaf
// marks, their scan and the bucket ids were six more.  The whole evaluation
// went from 3144 to 3031 us at 1M (FP32C), from 928 to 856 at 100k and from
// 382 to 337 at 1k (FP64).
#include "pt_common.h"
#include "pt_kernels.h"

namespace {

constexpr int kTreeRows = PT_TREE_ROWS;        // count rows: depths, leaves, faults
constexpr int kLeafRow = PT_MAX_DEPTH;         // depths 0..20 hold the internal nodes
constexpr int kFaultRow = PT_MAX_DEPTH + 1;
constexpr int kTreeWaves = 4;

// How the keys were sorted: mask keeps the ordered bits, digits is the number
// of whole octal digits among them, and internal nodes have depth <= deepest
// (the last key level is never split; with fewer ordered digits a cell that
// would have to be split below them counts as a fault and the host sorts the
// full keys).
struct KeyOrder {
  uint64_t mask;
  int32_t digits;
  int32_t deepest;
};

__host__ __device__ inline KeyOrder key_order(int bits) {
  KeyOrder o;
  o.mask = bits >= 64 ? ~0ull : ~0ull << (64 - bits);
  o.digits = (bits - 1) / 3;
  o.deepest = o.digits - 1;
  return o;
}

// Leading octal digits a and b share (bit 63 is the placeholder of every key).
__device__ __forceinline__ int shared_digits(uint64_t a, uint64_t b, const KeyOrder& o) {
  const uint64_t x = (a ^ b) & o.mask;
  const int c = x ? (__clzll((long long)x) - 1) / 3 : o.digits;
  return c < o.digits ? c : o.digits;
}

// What starts at particle i, 16 bits: the shared digits with i - 1 plus one,
// the deepest internal node starting at i plus one (no more than the former
// when there is none), and whether a leaf starts at i.
__device__ __forceinline__ uint32_t pack_meta(int lo, int hi, bool leaf) {
  return (uint32_t)(lo + 1) | ((uint32_t)(hi + 1) << 5) | (leaf ? 1u << 10 : 0u);
}

// One wave per wtile consecutive particles.  counts[row * pitch + wave].
__global__ void __launch_bounds__(kTreeWaves * PT_WAVE)
tree_count_kernel(const uint64_t* __restrict__ keys, int64_t n, int bucket, KeyOrder o,
                  int64_t wtile, int32_t nw, int32_t pitch, uint16_t* __restrict__ meta,
                  uint32_t* __restrict__ counts) {
  const int lane = threadIdx.x & (PT_WAVE - 1);
  const int64_t w = (int64_t)blockIdx.x * kTreeWaves + threadIdx.x / PT_WAVE;
  if (w >= nw) return;
  const int64_t end = (w + 1) * wtile < n ? (w + 1) * wtile : n;
  uint32_t cnt = 0;  // lane r: row r
  for (int64_t base = w * wtile; base < end; base += PT_WAVE) {
    const int64_t i = base + lane;
    int lo = 0, hi = -1;
    bool leaf = false, fault = false;
    if (i < end) {
      const uint64_t k = keys[i];
      lo = i > 0 ? shared_digits(keys[i - 1], k, o) : -1;
      const int win = i + bucket < n ? shared_digits(k, keys[i + bucket], o) : -1;
      fault = o.digits < PT_MAX_DEPTH && win > o.deepest;
      hi = win < o.deepest ? win : o.deepest;
      if (hi > lo) {
        leaf = true;
      } else if (lo < 0) {
        leaf = true;  // the root is a leaf
      } else if (lo <= o.deepest) {
        // is the cell of depth lo around i internal?  Its start is at most
        // bucket particles back, unless it then holds more than that already
        const uint64_t top = k >> (63 - 3 * lo);
        int64_t a = i - bucket;
        if (a >= 0 && (keys[a] >> (63 - 3 * lo)) == top) {
          leaf = true;
        } else {
          // first particle of the cell, in (a, i]
          int64_t l = a < 0 ? 0 : a + 1, h = i;
          while (l < h) {
            const int64_t mid = l + ((h - l) >> 1);
            if ((keys[mid] >> (63 - 3 * lo)) >= top) h = mid;
            else l = mid + 1;
          }
          leaf = l + bucket < n && (keys[l + bucket] >> (63 - 3 * lo)) == top;
        }
      }
      meta[i] = (uint16_t)pack_meta(lo, hi, leaf);
    }
    const uint32_t nl = (uint32_t)__popcll(__ballot(leaf));
    const uint32_t nf = (uint32_t)__popcll(__ballot(fault));
    cnt += lane == kLeafRow ? nl : 0u;
    cnt += lane == kFaultRow ? nf : 0u;
    if (__ballot(hi > lo) != 0ull) {
      for (int d = 0; d <= o.deepest; d++) {
        const uint32_t c = (uint32_t)__popcll(__ballot(lo < d && d <= hi));
        cnt += lane == d ? c : 0u;
      }
    }
  }
  if (lane < kTreeRows) counts[(int64_t)lane * pitch + w] = cnt;
}

// Exclusive scan of each row of the count table, a work-group per row (at most
// kScanThreads * kScanItems entries, all loaded at once), and the row totals
// behind the table.  One work-group over the whole table, 11 rounds of loads
// and barriers for 1M particles' 90k entries, took 86 us.
constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr int64_t kTreeMaxWaves = kScanThreads * kScanItems;

__global__ void __launch_bounds__(kScanThreads)
tree_scan_kernel(uint32_t* __restrict__ counts, int32_t nw, int32_t pitch) {
  __shared__ uint32_t wsum[kScanThreads / PT_WAVE];
  const int lane = threadIdx.x & (PT_WAVE - 1), wave = threadIdx.x / PT_WAVE;
  uint4* row = reinterpret_cast<uint4*>(counts + (int64_t)blockIdx.x * pitch);
  const int i0 = threadIdx.x * kScanItems;
  uint4 q[kScanItems / 4];
  uint32_t v[kScanItems], run = 0;
#pragma unroll
  for (int j = 0; j < kScanItems / 4; j++)
    q[j] = i0 + 4 * j < nw ? row[threadIdx.x * (kScanItems / 4) + j] : uint4{0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < kScanItems; j++) {
    const uint32_t a = (j & 3) == 0 ? q[j / 4].x : (j & 3) == 1 ? q[j / 4].y
                       : (j & 3) == 2 ? q[j / 4].z : q[j / 4].w;
    v[j] = run;
    run += i0 + j < nw ? a : 0u;
  }
  const uint32_t incl = (uint32_t)pt_wave_incl_scan((int)run);
  if (lane == PT_WAVE - 1) wsum[wave] = incl;
  __syncthreads();
  uint32_t before = incl - run;
  for (int k = 0; k < wave; k++) before += wsum[k];
#pragma unroll
  for (int j = 0; j < kScanItems / 4; j++)
    if (i0 + 4 * j < nw)
      row[threadIdx.x * (kScanItems / 4) + j] =
          uint4{before + v[4 * j], before + v[4 * j + 1], before + v[4 * j + 2],
                before + v[4 * j + 3]};
  if (threadIdx.x == kScanThreads - 1)
    counts[(int64_t)kTreeRows * pitch + blockIdx.x] = before + run;
}

// The running count of a row at the start of the wave's tile, one row per
// lane, moves on as the wave goes through its particles; the latest internal
// node of depth d at or before particle i is then the parent of what starts
// at i with depth d + 1.  The first wave also writes what the host reads back
// (pt_launch_build's status); nothing is built when the tree does not fit or
// the sort did not order enough bits.
__global__ void __launch_bounds__(kTreeWaves * PT_WAVE)
tree_assign_kernel(const uint64_t* __restrict__ keys, int64_t n, int bucket, KeyOrder o,
                   int64_t wtile, int32_t nw, int32_t pitch, int64_t level_cap,
                   const uint16_t* __restrict__ meta, const uint32_t* __restrict__ counts,
                   int64_t* __restrict__ status, PtTree t, int32_t* __restrict__ level_nodes, int2* __restrict__ internal,
                   uint32_t* __restrict__ bucket_of, int32_t* __restrict__ bucket_node) {
  const int lane = threadIdx.x & (PT_WAVE - 1);
  const int64_t w = (int64_t)blockIdx.x * kTreeWaves + threadIdx.x / PT_WAVE;
  if (w >= nw) return;
  const int64_t end = (w + 1) * wtile < n ? (w + 1) * wtile : n;
  const uint32_t tot = lane < kTreeRows ? counts[(int64_t)kTreeRows * pitch + lane] : 0u;
  // internal nodes in (depth, particle) order: a depth's count starts behind
  // the shallower ones
  const uint32_t row0 = (uint32_t)pt_wave_incl_scan((int)tot) - tot;
  const uint32_t internals = (uint32_t)__builtin_amdgcn_readlane((int)row0, kLeafRow);
  const uint32_t leaves = (uint32_t)__builtin_amdgcn_readlane((int)tot, kLeafRow);
  const uint32_t faults = (uint32_t)__builtin_amdgcn_readlane((int)tot, kFaultRow);
  const bool fits = (int64_t)internals <= level_cap, ok = fits && faults == 0;
  if (w == 0) {
    if (lane == 0) {
      status[0] = ok ? 1 + 8 * (int64_t)internals : 0;
      status[1] = ok ? (int64_t)leaves : 0;
      status[2] = fits ? 0 : (int64_t)internals;
      status[PT_TREE_STATUS - 1] = faults;
    }
    if (lane <= PT_MAX_DEPTH + 1) status[3 + lane] = lane < kLeafRow ? (int64_t)tot : 0;
  }
  if (!ok) return;
  uint32_t at = lane < kTreeRows ? counts[(int64_t)lane * pitch + w] : 0u;
  at += lane < kLeafRow ? row0 : 0u;
  const unsigned long long upto = ~0ull >> (PT_WAVE - 1 - lane);
  if (w == 0 && lane == 0) {
    const bool inner = n > bucket;
    t.key[0] = 1;
    t.begin[0] = 0;
    t.count[0] = (int32_t)n;
    t.depth[0] = 0;
    t.type[0] = inner ? PT_NODE_INTERNAL : PT_NODE_LEAF;
    t.parent[0] = -1;
    if (!inner) t.first_child[0] = -1;
  }
  for (int64_t base = w * wtile; base < end; base += PT_WAVE) {
    const int64_t i = base + lane;
    const bool valid = i < end;
    const uint32_t mt = valid ? meta[i] : pack_meta(0, -1, false);
    const int lo = (int)(mt & 31u) - 1, hi = (int)((mt >> 5) & 31u) - 1;
    const bool leaf = (mt >> 10) & 1u;
    const uint64_t k = valid ? keys[i] : 0ull;
    const int ldepth = hi > lo ? hi + 1 : lo + 1;  // of the leaf that starts here
    int64_t up = -1;       // latest internal node of depth d - 1
    int64_t lparent = -1;  // the leaf's parent
    for (int d = 0; d <= o.deepest; d++) {
      const bool start = lo < d && d <= hi;
      const unsigned long long m = __ballot(start);
      const uint32_t before = (uint32_t)__builtin_amdgcn_readlane((int)at, d);
      const int64_t idx = (int64_t)before + __popcll(m & upto) - 1;
      if (start) {
        level_nodes[idx] = d == 0 ? 0 : (int32_t)(1 + 8 * up + (int)((k >> (63 - 3 * d)) & 7u));
        internal[idx] = make_int2((int)i, d);
      }
      up = idx;
      if (d == ldepth - 1) lparent = idx;
      at += lane == d ? (uint32_t)__popcll(m) : 0u;
    }
    const unsigned long long lm = __ballot(leaf);
    const uint32_t lbefore = (uint32_t)__builtin_amdgcn_readlane((int)at, kLeafRow);
    const uint32_t b = lbefore + (uint32_t)__popcll(lm & upto) - 1u;
    if (valid) bucket_of[i] = b;
    if (leaf)
      bucket_node[b] = ldepth == 0 ? 0
                                   : (int32_t)(1 + 8 * lparent +
                                               (int)((k >> (63 - 3 * ldepth)) & 7u));
    at += lane == kLeafRow ? (uint32_t)__popcll(lm) : 0u;
  }
}

// The 8 children of every internal node, a lane each: lane c > 0 searches the
// start of child c, lane 0 the node's end, and each lane takes its end from
// the next lane's start.  Most nodes hold a few buckets, so the first probe,
// 32 buckets on, leaves ~10 of the ~20 dependent loads of a search over
// everything behind the node.
__global__ void __launch_bounds__(256)
tree_children_kernel(const uint64_t* __restrict__ keys, int64_t n, int bucket, KeyOrder o,
                     const int64_t* __restrict__ status, PtTree t,
                     const int32_t* __restrict__ level_nodes, const int2* __restrict__ internal) {
  const int64_t total = status[0] > 0 ? status[0] - 1 : 0;  // 8 per internal node
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t g = blockIdx.x * 256ll + threadIdx.x; g < total; g += stride) {
    const int64_t idx = g >> 3;
    const int c = (int)(g & 7);
    const int2 in = internal[idx];
    const int64_t b = in.x;
    const int d = in.y;
    const int32_t p = level_nodes[idx];
    const uint64_t key = keys[b] >> (63 - 3 * d);
    const uint64_t child = (key << 3) | (uint64_t)c;
    // the first particle whose key, cut to the depth, is not below `want`
    const int shift = c == 0 ? 63 - 3 * d : 60 - 3 * d;
    const uint64_t want = c == 0 ? key + 1 : child;
    int64_t l = b, h = n;
    const int64_t probe = b + 32 * (int64_t)bucket;
    if (probe < n) {
      if ((keys[probe] >> shift) >= want) h = probe;
      else l = probe + 1;
    }
    while (l < h) {
      const int64_t mid = l + ((h - l) >> 1);
      if ((keys[mid] >> shift) >= want) h = mid;
      else l = mid + 1;
    }
    const int lane = __lane_id();
    const int next = __shfl((int)l, (lane & ~7) | ((c + 1) & 7), PT_WAVE);
    const int32_t start = c == 0 ? (int32_t)b : (int32_t)l;
    const int32_t count = next - start;
    const int ty = count == 0 ? PT_NODE_EMPTY
                              : (count > bucket && d + 1 <= o.deepest ? PT_NODE_INTERNAL
                                                                      : PT_NODE_LEAF);
    const int64_t id = 1 + g;
    t.key[id] = child;
    t.begin[id] = start;
    t.count[id] = count;
    t.depth[id] = d + 1;
    t.type[id] = ty;
    t.parent[id] = p;
    // an internal child's first child is written by its own lanes
    if (ty != PT_NODE_INTERNAL) t.first_child[id] = -1;
    if (c == 0) t.first_child[p] = (int32_t)id;
  }
}

// After a sort of the keys' top bits only (ties kept in input order), puts
// every leaf's particles in full (key, input index) order: the sort the rest
// of the path expects.  Exact when every split of the build used only sorted
// bits, i.e. each leaf holds whole groups of equal sorted bits.  One thread
// per bucket (non-empty leaf; status[1] of them): up to 16 particles are
// sorted in registers by an odd-even transposition network, up to kFixupMax
// by insertion in place.
__device__ __forceinline__ bool pair_less(uint64_t ka, uint32_t va, uint64_t kb, uint32_t vb) {
  return ka < kb || (ka == kb && va < vb);
}

__global__ void __launch_bounds__(256)
leaf_fixup_kernel(const PtTree t, const int32_t* __restrict__ bucket_node,
                  const int64_t* __restrict__ status, uint64_t* __restrict__ keys,
                  uint32_t* __restrict__ perm) {
  const int64_t i = blockIdx.x * 256ll + threadIdx.x;
  if (i >= status[1]) return;
  const int32_t leaf = bucket_node[i];
  const int64_t b = t.begin[leaf];
  const int32_t n = t.count[leaf];
  if (n < 2 || n > kFixupMax) return;
  if (n <= 16) {
    uint64_t k[16];
    uint32_t v[16];
#pragma unroll
    for (int j = 0; j < 16; j++) {
      k[j] = j < n ? keys[b + j] : ~0ull;
      v[j] = j < n ? perm[b + j] : ~0u;
    }
#pragma unroll
    for (int r = 0; r < 16; r++) {
#pragma unroll
      for (int j = r & 1; j + 1 < 16; j += 2) {
        if (pair_less(k[j + 1], v[j + 1], k[j], v[j])) {
          const uint64_t tk = k[j];
          k[j] = k[j + 1];
          k[j + 1] = tk;
          const uint32_t tv = v[j];
          v[j] = v[j + 1];
          v[j + 1] = tv;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 16; j++) {
      if (j < n) {
        keys[b + j] = k[j];
        perm[b + j] = v[j];
      }
    }
    return;
  }
  for (int j = 1; j < n; j++) {
    const uint64_t kj = keys[b + j];
    const uint32_t vj = perm[b + j];
    int q = j - 1;
    while (q >= 0 && pair_less(kj, vj, keys[b + q], perm[b + q])) {
      keys[b + q + 1] = keys[b + q];
      perm[b + q + 1] = perm[b + q];
      q--;
    }
    keys[b + q + 1] = kj;
    perm[b + q + 1] = vj;
  }
}

inline unsigned grid_for(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

int pt_launch_leaf_fixup(const PtTree& t, int64_t max_buckets, const int32_t* bucket_node,
                         const int64_t* status, uint64_t* keys, uint32_t* perm, hipStream_t s) {
  if (max_buckets <= 0) return 0;
  leaf_fixup_kernel<<<grid_for(max_buckets), 256, 0, s>>>(t, bucket_node, status, keys, perm);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Waves over n particles, whole 64-particle chunks each: 256 particles, more
// when that would pass kTreeMaxWaves.
static int64_t wave_tile(int64_t n) {
  const int64_t t = (n + kTreeMaxWaves - 1) / kTreeMaxWaves;
  return ((t < 256 ? 256 : t) + PT_WAVE - 1) / PT_WAVE * PT_WAVE;
}

int64_t pt_tree_scratch_bytes(int64_t n) {
  return (PT_TREE_ROWS * (kTreeMaxWaves < n ? kTreeMaxWaves : n + 4) + PT_TREE_ROWS) * 4 + 256;
}

int pt_launch_build(const uint64_t* keys, int64_t n, int bucket, int bits, const PtTree& t,
                    int64_t level_cap, int32_t* level_nodes, int2* internal, uint16_t* meta,
                    uint32_t* bucket_of, int32_t* bucket_node, void* scratch, int64_t* status,
                    hipStream_t s) {
  if (n <= 0 || bits < 4 || bits > 64) return -1;
  const KeyOrder o = key_order(bits);
  uint32_t* counts = (uint32_t*)scratch;
  const int64_t wtile = wave_tile(n);
  const int32_t nw = (int32_t)((n + wtile - 1) / wtile);
  const int32_t pitch = (nw + 3) / 4 * 4;
  const unsigned grid = (unsigned)((nw + kTreeWaves - 1) / kTreeWaves);
  tree_count_kernel<<<grid, kTreeWaves * PT_WAVE, 0, s>>>(keys, n, bucket, o, wtile, nw, pitch,
                                                          meta, counts);
  tree_scan_kernel<<<kTreeRows, kScanThreads, 0, s>>>(counts, nw, pitch);
  tree_assign_kernel<<<grid, kTreeWaves * PT_WAVE, 0, s>>>(
      keys, n, bucket, o, wtile, nw, pitch, level_cap, meta, counts, status, t, level_nodes,
      internal, bucket_of, bucket_node);
  const unsigned most = grid_for(8 * level_cap);
  tree_children_kernel<<<most < 4096u ? most : 4096u, 256, 0, s>>>(keys, n, bucket, o, status, t,
                                                                   level_nodes, internal);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}
