// Node moments: leaf CentroidData and the upward pass, in FP64.
//
// Reference: CentroidData(const Particle*, n, depth) and operator+=
// (examples/CentroidData.h:41-73), MultipoleMoments::operator+= for particles
// and for expansions, quadrupole branch (examples/MultipoleMoments.h:204-353),
// calculateRadiusFarthestCorner / calculateRadiusBox (:458-482), and the merge
// order of Subtree::populateTree (src/Subtree.h:351-384).
//
// populateTree pushes every non-empty leaf (DFS order), then every empty leaf
// (DFS order) into a FIFO and enqueues a parent when its 8th child has been
// merged into it.  The merges are order-dependent at rounding level, so each
// parent here merges its children in the order that FIFO pops them:
// non-empty leaves by child index, then empty leaves by child index, then
// internal children ordered by the pair (h, b) computed below.  A frontier
// node (no internal child) has h = 0 and b = its last-popped leaf child's pop
// rank; any other node takes (h + 1, b) of its last-popped internal child.  Pop
// order among internal nodes is lexicographic in (h, b): every leaf is popped
// before every internal node, and an internal node is enqueued right after its
// last child is popped.  Leaf pop ranks are encoded monotonically as the
// left-aligned key (DFS order of disjoint nodes) with bit 63 marking empties.
//
// The file is compiled with -ffp-contract=off: every multiply and add rounds
// separately, as in the reference source, so the results are bit-exact with a
// CPU evaluation of the same operations.
#include "pt_common.h"
#include "pt_kernels.h"

namespace {

// Quad layout of both passes: four neighbouring lanes hold one node, lane
// l < 3 the l-th coordinate (cm_l, the second moments q_ll and q_{l,l+1 mod 3},
// the box's l-th faces) and lane 3 the softening (and the node's mass and
// radius when they are stored).  A merge is then one divide instead of four,
// the other lanes' differences come by a quad permutation, and records are
// read and written in 32-byte rows.  The operations on each field, and their
// order, are those of the reference's expressions.
constexpr int kNext = 0xC9;  // lane 0 <- 1, 1 <- 2, 2 <- 0, 3 <- 3

struct QuadNode {
  double v;         // cm_l, or the softening
  double qd, qo;    // q_ll, q_{l,l+1 mod 3} (lane 3: not used)
  double lo, hi;    // box faces
  double mass;      // in every lane
};

__device__ __forceinline__ QuadNode quad_default() {
  return QuadNode{0.0, 0.0, 0.0, INFINITY, -INFINITY, 0.0};
}

// q += m d d^T for this lane's two components, each product taken in the order
// m * d_first * d_second of the reference (xy, yz: own first; xz: x first).
__device__ __forceinline__ void quad_outer(double m, double d, bool swap, double& dd,
                                           double& od) {
  const double e = pt_quad_f64<kNext>(d);
  dd = m * d * d;
  od = m * (swap ? e : d) * (swap ? d : e);
}

// MultipoleMoments::operator+=(Particle) (examples/MultipoleMoments.h:275-353):
// a particle of mass pm whose coordinate (lane 3: softening) is pv.
__device__ __forceinline__ void quad_add_particle(QuadNode& d, double pm, double pv, bool swap) {
  const double m1 = d.mass;
  d.mass += pm;
  const double old = d.v;
  const bool none = d.mass == 0.0;
  d.v = none ? 0.5 * (old + pv) : (m1 * old + pm * pv) / d.mass;
  double dd, od;
  quad_outer(m1, old - d.v, swap, dd, od);
  d.qd = none ? d.qd : d.qd + dd;
  d.qo = none ? d.qo : d.qo + od;
  quad_outer(pm, pv - d.v, swap, dd, od);
  d.qd = none ? d.qd : d.qd + dd;
  d.qo = none ? d.qo : d.qo + od;
}

// CentroidData::operator+= (examples/CentroidData.h:61-73) with
// MultipoleMoments::operator+= (examples/MultipoleMoments.h:204-271), without
// its last step, the radius: no merge reads the radius it sets (a merge into
// a massless node copies the child's and the next radius overwrites it), so
// one radius after the merges gives the value of the last one bit for bit.
__device__ __forceinline__ void quad_merge(QuadNode& d, const QuadNode& c, bool swap) {
  if (c.lo < d.lo) d.lo = c.lo;
  if (c.hi > d.hi) d.hi = c.hi;
  const double m1 = d.mass;
  d.mass += c.mass;
  const double old = d.v;
  const double sum = (m1 * old + c.mass * c.v) / d.mass;
  double dd, od, cd, co;
  quad_outer(m1, old - sum, swap, dd, od);
  quad_outer(c.mass, c.v - sum, swap, cd, co);
  if (d.mass == 0.0) {
    d.v = 0.5 * (old + c.v);
  } else if (m1 == 0.0) {
    d.v = c.v;
    d.qd = c.qd;
    d.qo = c.qo;
    d.mass = c.mass;
  } else if (c.mass != 0.0) {
    d.v = sum;
    d.qd = (d.qd + dd) + (c.qd + cd);
    d.qo = (d.qo + od) + (c.qo + co);
  }
}

// x^2 + y^2 + z^2 over the quad's first three lanes, in every lane.
__device__ __forceinline__ double quad_len2(double e) {
  const double s = e * e;
  return pt_quad_f64<0x00>(s) + pt_quad_f64<0x55>(s) + pt_quad_f64<0xAA>(s);
}

// The smallest float >= v (v >= 0, finite).
__device__ __forceinline__ float round_up_f32(double v) {
  float f = (float)v;
  if ((double)f < v) f = __int_as_float(__float_as_int(f) + 1);
  return f;
}

// Stores node i's CentroidData and its walk and interaction records from the
// quad's final values.  Leaves also get their reach and softening bounds
// (leaf_soft: the largest particle softening, any value in other lanes than
// 3) and, when non-empty, their bucket record (bucket index
// bucket_of[begin]).
__device__ __forceinline__ void quad_store(const PtTree& t, int64_t i, int l, const QuadNode& d,
                                           double radius, double leaf_soft,
                                           double* __restrict__ nd, const PtPackOut& o) {
  const double qxx = pt_quad_f64<0x00>(d.qd), qyy = pt_quad_f64<0x55>(d.qd),
               qzz = pt_quad_f64<0xAA>(d.qd);
  double* r = nd + i * PT_ND_STRIDE;
  r[l] = d.v;
  r[4 + l] = l < 3 ? d.qd : d.mass;
  r[8 + l] = l < 3 ? d.qo : radius;
  r[12 + l] = l < 3 ? d.lo : 0.0;
  r[16 + l] = l < 3 ? d.hi : 0.0;
  const int32_t count = t.count[i], type = t.type[i], begin = t.begin[i];
  const double d1 = d.v - d.lo, d2 = d.hi - d.v;
  const double reach2 = quad_len2(d1 > d2 ? d1 : d2);
  // TreeNode: {cx, cy, cz, radius} then {count, first_child} {type, begin}
  // {leaf_reach, leaf_soft} {node_soft, pad}, one 8-byte piece per lane
  double* a = reinterpret_cast<double*>(o.tnode + i);
  a[l] = l < 3 ? d.v : radius;
  int2 w;
  if (l == 0) w = make_int2(count, t.first_child[i]);
  if (l == 1) w = make_int2(type, begin);
  const bool leaf = type == PT_NODE_LEAF;
  const float ls = __int_as_float(
      pt_quad_i32<0xFF>(__float_as_int(leaf ? round_up_f32(leaf_soft) : 0.f)));
  if (l == 2)
    w = make_int2(__float_as_int(leaf ? round_up_f32(sqrt(reach2)) : 0.f), __float_as_int(ls));
  if (l == 3)
    w = make_int2(__float_as_int(type == PT_NODE_INTERNAL ? round_up_f32(d.v) : 0.f), 0);
  reinterpret_cast<int2*>(o.tnode + i)[4 + l] = w;
  double* g = reinterpret_cast<double*>(o.gn + i);
  g[l] = d.v;
  g[4 + l] = l < 3 ? d.qd : d.mass;
  g[8 + l] = l < 3 ? d.qo : 0.5 * (qxx + qyy + qzz);
  // GravNode32: centre and softening, then {qxx qxy} {qyy qyz} {qzz qxz} {mass soft}
  reinterpret_cast<double*>(o.gn32 + i)[l] = d.v;
  reinterpret_cast<float2*>(o.gn32 + i)[4 + l] =
      make_float2((float)(l < 3 ? d.qd : d.mass), (float)(l < 3 ? d.qo : d.v));
  if (leaf && count > 0) {
    double* b = reinterpret_cast<double*>(o.bk + o.bucket_of[begin]);
    b[l] = l < 3 ? d.lo : 0.0;
    b[4 + l] = l < 3 ? d.hi : 0.0;
    b[8 + l] = d.v;
    if (l < 2)
      reinterpret_cast<int2*>(b + 12)[l] = l == 0 ? make_int2((int)i, begin) : make_int2(count, 0);
  }
}

static_assert(sizeof(TreeNode) == 64 && sizeof(GravNode) == 96 && sizeof(GravNode32) == 64 &&
                  sizeof(Bucket) == 128,
              "record layouts written by quad_store");

// A quad per node: a leaf runs the sequential particle recurrence of the
// CentroidData leaf constructor (examples/CentroidData.h:41-59) in sorted
// particle order; an empty leaf stores the default CentroidData; internal
// nodes are left to the upward pass.  Bound by the recurrence's chain of
// dependent divides, one per particle; its inputs are loaded kPre particles
// ahead.
__global__ void __launch_bounds__(256)
leaf_kernel(const PtTree t, int64_t nn, const double* __restrict__ x,
            const double* __restrict__ y, const double* __restrict__ z,
            const double* __restrict__ m, const double* __restrict__ e, double* __restrict__ nd,
            const PtPackOut o) {
  const int64_t id = blockIdx.x * 64ll + (threadIdx.x >> 2);
  const int l = threadIdx.x & 3;
  if (id >= nn) return;
  const int ty = t.type[id];
  if (ty == PT_NODE_INTERNAL) return;
  const bool swap = l == 2;
  QuadNode d = quad_default();
  double radius = 0.0, smax = 0.0;
  if (ty == PT_NODE_LEAF) {
    const int64_t b = t.begin[id];
    const int32_t n = t.count[id];
    const double* __restrict__ mine = l == 0 ? x : l == 1 ? y : l == 2 ? z : e;
    constexpr int kPre = 8;
    for (int32_t k0 = 0; k0 < n; k0 += kPre) {
      double pv[kPre], pm[kPre];
#pragma unroll
      for (int k = 0; k < kPre; k++) {
        if (k0 + k < n) {
          pv[k] = mine[b + k0 + k];
          pm[k] = m[b + k0 + k];
        }
      }
#pragma unroll
      for (int k = 0; k < kPre; k++) {
        if (k0 + k < n) {
          quad_add_particle(d, pm[k], pv[k], swap);
          if (pv[k] < d.lo) d.lo = pv[k];
          if (pv[k] > d.hi) d.hi = pv[k];
          smax = pv[k] > smax ? pv[k] : smax;
        }
      }
    }
    // calculateRadiusBox (examples/MultipoleMoments.h:473-482)
    radius = n > 1 ? 0.5 * sqrt(quad_len2(d.hi - d.lo)) : 1.0;
  }
  quad_store(t, id, l, d, radius, smax, nd, o);
}

__device__ __forceinline__ uint64_t left_align(uint64_t k) {
  const int depth = (63 - __clzll(k)) / 3;
  return k << (PT_KEY_BITS - (3 * depth + 1));
}

__device__ __forceinline__ unsigned quad_or(unsigned v) {
  v |= (unsigned)pt_quad_i32<0xB1>((int)v);
  return v | (unsigned)pt_quad_i32<0x4E>((int)v);
}

// The larger of (h, b) and the CTRL-permuted lane's, lexicographically.
template <int CTRL>
__device__ __forceinline__ void quad_max_hb(int32_t& h, uint64_t& b) {
  const int32_t oh = pt_quad_i32<CTRL>(h);
  const uint64_t ob = pt_quad_u64<CTRL>(b);
  if (oh > h || (oh == h && ob > b)) {
    h = oh;
    b = ob;
  }
}

// Children of child index O's lane among a lane's two: the internal ones that
// come before (h, b) are counted into rank[].
template <int O>
__device__ __forceinline__ void quad_rank(const int32_t (&h)[2], const uint64_t (&b)[2],
                                          int (&rank)[2]) {
  constexpr int bc = (O >> 1) * 0x55;
  const int32_t oh = pt_quad_i32<bc>(h[O & 1]);
  const uint64_t ob = pt_quad_u64<bc>(b[O & 1]);
#pragma unroll
  for (int j = 0; j < 2; j++)
    rank[j] += oh >= 0 && (oh < h[j] || (oh == h[j] && ob < b[j])) ? 1 : 0;
}

// One internal node per quad, its children final.  Lane l finds the pop
// positions of children 2 l and 2 l + 1; then every lane loads its column of
// the 8 children's records in pop order, all in flight at once, and merges
// them in that order.
__device__ __forceinline__ void upward_node(const PtTree& t, int32_t p, int l,
                                            double* __restrict__ nd, int32_t* __restrict__ ord_h,
                                            uint64_t* __restrict__ ord_b, const PtPackOut& o) {
  const int64_t fc = t.first_child[p];
  int ctype[2];
  int32_t h[2];
  uint64_t b[2], ckey[2];
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int64_t ch = fc + 2 * l + j;
    ctype[j] = t.type[ch];
    ckey[j] = t.key[ch];
    h[j] = ord_h[ch];
    b[j] = ord_b[ch];
  }
  unsigned leafm = 0, emptym = 0;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const bool inner = ctype[j] == PT_NODE_INTERNAL;
    h[j] = inner ? h[j] : -1;
    b[j] = inner ? b[j] : 0;
    leafm |= (ctype[j] == PT_NODE_LEAF ? 1u : 0u) << (2 * l + j);
    emptym |= (ctype[j] == PT_NODE_EMPTY ? 1u : 0u) << (2 * l + j);
  }
  leafm = quad_or(leafm);
  emptym = quad_or(emptym);
  const int n_leaf = __popc(leafm), n_first = n_leaf + __popc(emptym);
  int rank[2] = {0, 0};
  if (__ballot(n_first < 8) != 0ull) {
    quad_rank<0>(h, b, rank);
    quad_rank<1>(h, b, rank);
    quad_rank<2>(h, b, rank);
    quad_rank<3>(h, b, rank);
    quad_rank<4>(h, b, rank);
    quad_rank<5>(h, b, rank);
    quad_rank<6>(h, b, rank);
    quad_rank<7>(h, b, rank);
  }
  unsigned order = 0;
  int32_t hmax = -1;
  uint64_t bmax = 0, bleaf = 0;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int c = 2 * l + j;
    const unsigned below = (1u << c) - 1u;
    const int pos = ctype[j] == PT_NODE_LEAF    ? __popc(leafm & below)
                    : ctype[j] == PT_NODE_EMPTY ? n_leaf + __popc(emptym & below)
                                                : n_first + rank[j];
    order |= (unsigned)c << (4 * pos);
    if (h[j] > hmax || (h[j] == hmax && b[j] > bmax)) {
      hmax = h[j];
      bmax = b[j];
    }
    uint64_t r = left_align(ckey[j]) >> 1;
    if (ctype[j] == PT_NODE_EMPTY) r |= 1ull << 63;
    bleaf = r > bleaf ? r : bleaf;
  }
  order = quad_or(order);
  if (n_first < 8) {
    quad_max_hb<0xB1>(hmax, bmax);
    quad_max_hb<0x4E>(hmax, bmax);
    hmax++;
  } else {
    // frontier node: h = 0, b = rank of the last-popped leaf child
    hmax = 0;
    bmax = bleaf;
    quad_max_hb<0xB1>(hmax, bmax);
    quad_max_hb<0x4E>(hmax, bmax);
  }
  if (l == 0) {
    ord_h[p] = hmax;
    ord_b[p] = bmax;
  }
  double row[8][5];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const double* r = nd + (fc + ((order >> (4 * j)) & 15u)) * PT_ND_STRIDE + l;
#pragma unroll
    for (int k = 0; k < 5; k++) row[j][k] = r[4 * k];
  }
  const bool swap = l == 2;
  QuadNode d = quad_default();
#pragma unroll
  for (int j = 0; j < 8; j++) {
    QuadNode c{row[j][0], row[j][1], row[j][2], row[j][3], row[j][4],
               pt_quad_f64<0xFF>(row[j][1])};
    quad_merge(d, c, swap);
  }
  // calculateRadiusFarthestCorner (examples/MultipoleMoments.h:458-469); an
  // internal node holds more than one particle
  const double d1 = d.v - d.lo, d2 = d.hi - d.v;
  const double radius = sqrt(quad_len2(d1 > d2 ? d1 : d2));
  quad_store(t, p, l, d, radius, 0.0, nd, o);
}

// A quad per internal node of one level (deepest level first).  Latency bound:
// two dependent loads, then eight merges of one divide each, 7.5 us a level at
// 1M particles.  One thread per node took 18 us on a level of any size (168
// scattered 8-byte loads per thread, then 8 x 4 divides); with the leaves' 52
// -> 41 us and the small levels' run 64 -> 23 us (1k particles) the evaluation
// went from 3031 to 2950 us at 1M and from 337 to 271 at 1k.
constexpr int kUpThreads = 64;

__global__ void __launch_bounds__(kUpThreads)
upward_kernel(const PtTree t, const int32_t* __restrict__ level_nodes, int32_t nl,
              double* __restrict__ nd, int32_t* __restrict__ ord_h, uint64_t* __restrict__ ord_b,
              const PtPackOut o) {
  const int64_t li = (int64_t)blockIdx.x * (kUpThreads / 4) + (threadIdx.x >> 2);
  if (li >= nl) return;
  upward_node(t, level_nodes[li], threadIdx.x & 3, nd, ord_h, ord_b, o);
}

// A run of consecutive small levels in one work-group, deepest first, with a
// work-group barrier between levels (a level reads what the one below wrote;
// all waves of the group share the CU's caches).
constexpr int kRunThreads = 1024;

__global__ void __launch_bounds__(kRunThreads)
upward_run_kernel(const PtTree t, const int32_t* __restrict__ level_nodes, PtLevelRun run,
                  double* __restrict__ nd, int32_t* __restrict__ ord_h,
                  uint64_t* __restrict__ ord_b, const PtPackOut o) {
  for (int k = 0; k < run.nlev; k++) {
    const int32_t off = run.off[k], cnt = run.cnt[k];
    for (int32_t li = threadIdx.x >> 2; li < cnt; li += blockDim.x / 4)
      upward_node(t, level_nodes[off + li], threadIdx.x & 3, nd, ord_h, ord_b, o);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// HEXADECAPOLE moments (the -DHEXADECAPOLE build, examples/Makefile:5).
//
// The reference keeps reduced (trace-free) moments to fourth order per node
// (FMOMR, examples/moments.h), built per particle and shifted to parents
// (examples/MultipoleMoments.h:244-252,317-330).  As written its leaf update
// runs only while the node radius is positive, and the leaf constructor sets
// the radius after adding the particles (examples/CentroidData.h:41-59), so
// every FMOMR stays zero.  These kernels compute what the code intends: the
// raw third and fourth moments R(a,b,c) = sum m dx^a dy^b dz^c about each
// node's centre of mass (leaves sum their particles in sorted order; a parent
// sums its children's moments moved to its centre of mass by the binomial
// expansion, children in index order), then the trace-free parts together
// with the second moments q of the quadrupole pass.  Same operations, in the
// same order, as the oracle's restatement.
// ---------------------------------------------------------------------------

// index of component (a, b, .) among those of order l (a descending, then b)
__device__ __forceinline__ int hx_index(int l, int a, int b) {
  return (l - a) * (l - a + 1) / 2 + (l - a - b);
}

__device__ __forceinline__ double hx_binom(int n, int k) {
  // rows 0-4 of Pascal's triangle
  constexpr double t[5][5] = {{1, 0, 0, 0, 0}, {1, 1, 0, 0, 0}, {1, 2, 1, 0, 0},
                              {1, 3, 3, 1, 0}, {1, 4, 6, 4, 1}};
  return t[n][k];
}

__device__ __forceinline__ void hx_pow(double v, double p[5]) {
  p[0] = 1.0;
  p[1] = v;
  p[2] = p[1] * v;
  p[3] = p[2] * v;
  p[4] = p[3] * v;
}

// One thread per bucket: raw moments about the leaf's centre of mass.
__global__ void __launch_bounds__(256)
hexa_leaf_kernel(const PtTree t, const int32_t* __restrict__ bucket_node, int64_t nb,
                 const double* __restrict__ x, const double* __restrict__ y,
                 const double* __restrict__ z, const double* __restrict__ m,
                 const double* __restrict__ nd, int64_t nn, double* __restrict__ raw) {
  const int64_t bi = blockIdx.x * 256ll + threadIdx.x;
  if (bi >= nb) return;
  const int64_t id = bucket_node[bi];
  const double cx = nd[id * PT_ND_STRIDE + PT_ND_CM + 0], cy = nd[id * PT_ND_STRIDE + PT_ND_CM + 1],
               cz = nd[id * PT_ND_STRIDE + PT_ND_CM + 2];
  double r[PT_HEXA_RAW];
#pragma unroll
  for (int k = 0; k < PT_HEXA_RAW; k++) r[k] = 0.0;
  const int64_t b = t.begin[id], n = t.count[id];
  for (int64_t i = b; i < b + n; i++) {
    double px[5], py[5], pz[5];
    hx_pow(x[i] - cx, px);
    hx_pow(y[i] - cy, py);
    hx_pow(z[i] - cz, pz);
    const double mi = m[i];
#pragma unroll
    for (int l = 3; l <= 4; l++)
#pragma unroll
      for (int a = l; a >= 0; a--)
#pragma unroll
        for (int bb = l - a; bb >= 0; bb--) {
          const int c = l - a - bb;
          r[(l == 3 ? 0 : 10) + hx_index(l, a, bb)] += ((mi * px[a]) * py[bb]) * pz[c];
        }
  }
#pragma unroll
  for (int k = 0; k < PT_HEXA_RAW; k++) raw[k * nn + id] = r[k];
}

// raw moment of exponents (i, j, k) of a child: mass, second moments q
// (xx xy xz yy yz zz), third/fourth from its raw record
__device__ __forceinline__ double hx_child(const double* __restrict__ nd,
                                           const double* __restrict__ raw, int64_t nn,
                                           int64_t ch, double mass, int i, int j, int k) {
  const int l = i + j + k;
  if (l == 0) return mass;
  if (l == 2) return nd[ch * PT_ND_STRIDE + PT_ND_Q(hx_index(2, i, j))];
  if (l == 3) return raw[hx_index(3, i, j) * nn + ch];
  return raw[(10 + hx_index(4, i, j)) * nn + ch];
}

// One thread per internal node of one level (deepest level first, after the
// quadrupole pass has fixed every centre of mass).
__global__ void __launch_bounds__(256)
hexa_up_kernel(const PtTree t, const int32_t* __restrict__ level_nodes, int32_t nl,
               const double* __restrict__ nd, int64_t nn, double* __restrict__ raw) {
  const int64_t li = blockIdx.x * 256ll + threadIdx.x;
  if (li >= nl) return;
  const int64_t p = level_nodes[li];
  double r[PT_HEXA_RAW];
#pragma unroll
  for (int k = 0; k < PT_HEXA_RAW; k++) r[k] = 0.0;
  const double pmass = nd[p * PT_ND_STRIDE + PT_ND_MASS];
  if (pmass != 0.0) {
    const double pc[3] = {nd[p * PT_ND_STRIDE + PT_ND_CM + 0], nd[p * PT_ND_STRIDE + PT_ND_CM + 1],
                          nd[p * PT_ND_STRIDE + PT_ND_CM + 2]};
    const int32_t fc = t.first_child[p];
    for (int c = 0; c < 8; c++) {
      const int64_t ch = fc + c;
      const double cm = nd[ch * PT_ND_STRIDE + PT_ND_MASS];
      if (cm == 0.0) continue;
      double px[5], py[5], pz[5];
      hx_pow(nd[ch * PT_ND_STRIDE + PT_ND_CM + 0] - pc[0], px);
      hx_pow(nd[ch * PT_ND_STRIDE + PT_ND_CM + 1] - pc[1], py);
      hx_pow(nd[ch * PT_ND_STRIDE + PT_ND_CM + 2] - pc[2], pz);
#pragma unroll
      for (int l = 3; l <= 4; l++)
#pragma unroll
        for (int a = l; a >= 0; a--)
#pragma unroll
          for (int b = l - a; b >= 0; b--) {
            const int cc = l - a - b;
            double sum = 0.0;
#pragma unroll
            for (int i = 0; i <= a; i++)
#pragma unroll
              for (int j = 0; j <= b; j++)
#pragma unroll
                for (int k = 0; k <= cc; k++) {
                  if (i + j + k == 1) continue;
                  const double coef = hx_binom(a, i) * hx_binom(b, j) * hx_binom(cc, k);
                  sum += (((coef * px[a - i]) * py[b - j]) * pz[cc - k]) *
                         hx_child(nd, raw, nn, ch, cm, i, j, k);
                }
            r[(l == 3 ? 0 : 10) + hx_index(l, a, b)] += sum;
          }
    }
  }
#pragma unroll
  for (int k = 0; k < PT_HEXA_RAW; k++) raw[k * nn + p] = r[k];
}

// Trace-free moments and the HEXADECAPOLE records of every node.
__global__ void __launch_bounds__(256)
hexa_pack_kernel(const PtTree t, const double* __restrict__ nd, const double* __restrict__ raw,
                 int64_t nn, HexNode* __restrict__ hn, HexOpen* __restrict__ ho) {
  const int64_t i = blockIdx.x * 256ll + threadIdx.x;
  if (i >= nn) return;
  const int ty = t.type[i];
  double r[PT_HEXA_RAW];
#pragma unroll
  for (int k = 0; k < PT_HEXA_RAW; k++) r[k] = ty == PT_NODE_EMPTY ? 0.0 : raw[k * nn + i];
  double q[6];
#pragma unroll
  for (int k = 0; k < 6; k++) q[k] = nd[i * PT_ND_STRIDE + PT_ND_Q(k)];
#define R3(a, b) r[hx_index(3, a, b)]
#define R4(a, b) r[10 + hx_index(4, a, b)]
  const double tr = q[0] + q[3] + q[5];
  const double vx = R3(3, 0) + R3(1, 2) + R3(1, 0);
  const double vy = R3(2, 1) + R3(0, 3) + R3(0, 1);
  const double vz = R3(2, 0) + R3(0, 2) + R3(0, 0);
  const double txx = R4(4, 0) + R4(2, 2) + R4(2, 0);
  const double tyy = R4(2, 2) + R4(0, 4) + R4(0, 2);
  const double tzz = R4(2, 0) + R4(0, 2) + R4(0, 0);
  const double txy = R4(3, 1) + R4(1, 3) + R4(1, 1);
  const double txz = R4(3, 0) + R4(1, 2) + R4(1, 0);
  const double tyz = R4(2, 1) + R4(0, 3) + R4(0, 1);
  const double ss = txx + tyy + tzz;
  HexNode h;
  h.cx = nd[i * PT_ND_STRIDE + PT_ND_CM + 0];
  h.cy = nd[i * PT_ND_STRIDE + PT_ND_CM + 1];
  h.cz = nd[i * PT_ND_STRIDE + PT_ND_CM + 2];
  h.mass = nd[i * PT_ND_STRIDE + PT_ND_MASS];
  h.soft = nd[i * PT_ND_STRIDE + PT_ND_SOFT];
  h.h[0] = q[0] - tr * (1.0 / 3.0);
  h.h[1] = q[3] - tr * (1.0 / 3.0);
  h.h[2] = q[1];
  h.h[3] = q[2];
  h.h[4] = q[4];
  h.h[5] = R3(3, 0) - vx * (3.0 / 5.0);
  h.h[6] = R3(1, 2) - vx * (1.0 / 5.0);
  h.h[7] = R3(2, 1) - vy * (1.0 / 5.0);
  h.h[8] = R3(0, 3) - vy * (3.0 / 5.0);
  h.h[9] = R3(2, 0) - vz * (1.0 / 5.0);
  h.h[10] = R3(0, 2) - vz * (1.0 / 5.0);
  h.h[11] = R3(1, 1);
  h.h[12] = (R4(4, 0) - txx * (6.0 / 7.0)) + ss * (3.0 / 35.0);
  h.h[13] = R4(1, 3) - txy * (3.0 / 7.0);
  h.h[14] = R4(3, 1) - txy * (3.0 / 7.0);
  h.h[15] = (R4(0, 4) - tyy * (6.0 / 7.0)) + ss * (3.0 / 35.0);
  h.h[16] = R4(3, 0) - txz * (3.0 / 7.0);
  h.h[17] = R4(0, 3) - tyz * (3.0 / 7.0);
  h.h[18] = (R4(2, 2) - (txx + tyy) * (1.0 / 7.0)) + ss * (1.0 / 35.0);
  h.h[19] = R4(2, 1) - tyz * (1.0 / 7.0);
  h.h[20] = R4(1, 2) - txz * (1.0 / 7.0);
#undef R3
#undef R4
#pragma unroll
  for (int k = 0; k < 6; k++) h.pad[k] = 0.0;
  hn[i] = h;
  HexOpen o;
  o.lox = nd[i * PT_ND_STRIDE + PT_ND_LO + 0];
  o.loy = nd[i * PT_ND_STRIDE + PT_ND_LO + 1];
  o.loz = nd[i * PT_ND_STRIDE + PT_ND_LO + 2];
  o.hix = nd[i * PT_ND_STRIDE + PT_ND_HI + 0];
  o.hiy = nd[i * PT_ND_STRIDE + PT_ND_HI + 1];
  o.hiz = nd[i * PT_ND_STRIDE + PT_ND_HI + 2];
  o.soft = h.soft;
  o.pad = 0.0;
  ho[i] = o;
}

inline unsigned grid_for(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

int pt_launch_leaf_moments(const PtTree& t, int64_t nn, const double* x, const double* y,
                           const double* z, const double* m, const double* e, double* nd,
                           const PtPackOut& o, hipStream_t s) {
  if (nn <= 0) return 0;
  leaf_kernel<<<(unsigned)((nn + 63) / 64), 256, 0, s>>>(t, nn, x, y, z, m, e, nd, o);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_upward_run(const PtTree& t, const int32_t* level_nodes, const PtLevelRun& run,
                         double* nd, int32_t* ord_h, uint64_t* ord_b, const PtPackOut& o,
                         hipStream_t s) {
  if (run.nlev <= 0) return 0;
  int32_t most = 0;
  for (int k = 0; k < run.nlev; k++) most = run.cnt[k] > most ? run.cnt[k] : most;
  const int threads = most >= kRunThreads / 4 ? kRunThreads : (most * 4 + 63) / 64 * 64;
  upward_run_kernel<<<1, threads, 0, s>>>(t, level_nodes, run, nd, ord_h, ord_b, o);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_upward_level(const PtTree& t, const int32_t* level_nodes, int32_t nl, double* nd,
                           int32_t* ord_h, uint64_t* ord_b, const PtPackOut& o, hipStream_t s) {
  if (nl <= 0) return 0;
  constexpr int per = kUpThreads / 4;
  upward_kernel<<<(unsigned)((nl + per - 1) / per), kUpThreads, 0, s>>>(t, level_nodes, nl, nd,
                                                                        ord_h, ord_b, o);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}


int pt_launch_hexa_leaf(const PtTree& t, const int32_t* bucket_node, int64_t nb, const double* x,
                        const double* y, const double* z, const double* m, const double* nd,
                        int64_t nn, double* raw, hipStream_t s) {
  if (nb <= 0) return 0;
  hexa_leaf_kernel<<<grid_for(nb), 256, 0, s>>>(t, bucket_node, nb, x, y, z, m, nd, nn, raw);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_hexa_level(const PtTree& t, const int32_t* level_nodes, int32_t nl,
                         const double* nd, int64_t nn, double* raw, hipStream_t s) {
  if (nl <= 0) return 0;
  hexa_up_kernel<<<grid_for(nl), 256, 0, s>>>(t, level_nodes, nl, nd, nn, raw);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_hexa_pack(const PtTree& t, const double* nd, const double* raw, int64_t nn,
                        HexNode* hn, HexOpen* ho, hipStream_t s) {
  if (nn <= 0) return 0;
  hexa_pack_kernel<<<grid_for(nn), 256, 0, s>>>(t, nd, raw, nn, hn, ho);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}
