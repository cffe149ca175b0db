// Adjoint (vector-Jacobian products) of the gravity interactions, FP64 and
// FP32 (shifted coordinates, FP64 sums).
//
// For a cotangent w_i on every particle's acceleration these kernels compute
//   g_j  = sum_i (da_i/dx_j)^T w_i      (positions)
//   gm_j = sum_i (da_i/dm_j)^T w_i      (masses)
// for the tree force of GravityVisitor::node / leaf
// (examples/GravityVisitor.h:37-160,184-224) on the interactions the forward
// pass evaluates (the lists of pt_launch_group_traverse: per group of
// consecutive buckets, the union of the buckets' lists with member masks), and
// for the FP64 direct sum.
//
// leaf() pair (target t, source j, d = x_j + off - x_t):  a_t += m_j b(|d|) d:
//   da_t/dd = m_j K,  K = b I + (b'/|d|) d d^T  (symmetric), so the target
//   gets -m_j K w_t, the source +m_j K w_t and the source mass b d.w_t.
// node() pair (target t, node s, r = x_t - cm_s - off), quadrupole form
//   a = -qir3 r + c q,  q = Q r,  qir = r.q / 2,  qir3 = b M + d qir - c tr:
//   (da/dr)^T w = -qir3 w - k1 r (r.w) - d q (r.w) + c Q w + (c'/|r|) r (q.w),
//   k1 = (M b' + qir d' - tr c') / |r|;
//   the target gets it, the node centre gets minus it, the node mass
//   -b (r.w), each stored quadrupole component d(a.w)/dQ, and the node
//   softening d(a.w)/dtwoh (softened branch only).
// addGravity (the openSoftening branch): a = M dd/|dd|^3, dd = cm + off - x_t,
//   T = M (I/|dd|^3 - 3 dd dd^T/|dd|^5); the target gets -T w, the centre
//   +T w, the mass dd.w/|dd|^3.
// Node cotangents then flow to member particles through the closed forms of
// the moments (MultipoleMoments::operator+=, examples/MultipoleMoments.h:
// 204-270, is the parallel-axis merge of M = sum m, cm = sum m x / M,
// Q = sum m u u^T with u = x - cm, soft = sum m e / M):
//   dcm/dx_j = m_j/M I,  dQ_kl/dx_j = m_j (e_k u_l + u_k e_l),
//   dM/dm_j = 1, dcm/dm_j = u_j/M, dQ/dm_j = u_j u_j^T, dsoft/dm_j = (e_j - soft)/M.
// Opening decisions (open, openSoftening) are piecewise constant and held
// fixed.
#include "pt_common.h"
#include "pt_kernels.h"
#include "pt_walk.h"

#include <algorithm>

namespace {

constexpr int kANT = PT_GROUP_TARGETS;  // targets per pass over a group's lists
constexpr int kNodeAdj = 11;  // node cotangent: cm(3), M, Q(6: xx xy xz yy yz zz), soft
constexpr int kNodeRow = 12;  // its record in memory
// Nodes of the top levels (ids < kHotNodes in level order) are in the lists
// of most buckets; their cotangents are accumulated into kHotParts private
// copies (chosen by work-group) and summed afterwards, so concurrent atomic
// adds to one address come from 1/kHotParts of the work-groups.
constexpr int64_t kHotNodes = 16384;
constexpr int kHotParts = 32;

// GravityVisitor::SPLINE force factor b and db/dr (examples/GravityVisitor.h:
// 82-120); r is |d|, dir = 1 / r, twoh the summed softening.
__device__ __forceinline__ void spline_b_db(double r, double dir, double twoh, double& b,
                                            double& db) {
  if (r < twoh) {
    const double dih = 2.0 / twoh;
    const double u = r * dih;
    if (u < 1.0) {
      b = dih * dih * dih * (4.0 / 3.0 - 6.0 / 5.0 * u * u + 1.0 / 2.0 * u * u * u);
      db = dih * dih * dih * dih * (-12.0 / 5.0 * u + 3.0 / 2.0 * u * u);
    } else {
      b = -1.0 / 15.0 * dir * dir * dir +
          dih * dih * dih * (8.0 / 3.0 - 3.0 * u + 6.0 / 5.0 * u * u - 1.0 / 6.0 * u * u * u);
      db = 1.0 / 5.0 * dir * dir * dir * dir +
           dih * dih * dih * dih * (-3.0 + 12.0 / 5.0 * u - 1.0 / 2.0 * u * u);
    }
  } else {
    const double a = dir;
    b = a * a * a;
    db = -3.0 * b * a;
  }
}

// GravityVisitor::SPLINEQ b, c, d (examples/GravityVisitor.h:37-78, the
// expressions as written there), their r-derivatives (br, cr, dr_) and their
// twoh-derivatives at fixed r (bt, ct, dt_).
struct SplineQ {
  double b, c, d, br, cr, dr_, bt, ct, dt_;
};

__device__ __forceinline__ SplineQ splineq_grad(double r, double dir, double r2, double twoh) {
  double b, c, d, br, cr, dr_, bt, ct, dt_;
  if (r2 < twoh * twoh) {
    const double dih = 2.0 / twoh;
    const double u = dih * r;
    const double dih2 = dih * dih, dih3 = dih2 * dih, dih4 = dih3 * dih, dih5 = dih4 * dih,
                 dih6 = dih5 * dih;
    double bD, cD, dD;  // derivatives with respect to dih at fixed r
    if (u < 1.0) {
      b = dih3 * 4.0 / 3.0 - 6.0 / 5.0 * u * u + 1.0 / 2.0 * u * u * u;
      c = dih5 * 12.0 / 5.0 - 3.0 / 2.0 * u;
      d = 3.0 / 2.0 * dih6 * dir;
      br = dih * (-12.0 / 5.0 * u + 3.0 / 2.0 * u * u);
      cr = -3.0 / 2.0 * dih;
      dr_ = -3.0 / 2.0 * dih6 * dir * dir;
      bD = 4.0 * dih2 + r * (-12.0 / 5.0 * u + 3.0 / 2.0 * u * u);
      cD = 12.0 * dih4 - 3.0 / 2.0 * r;
      dD = 9.0 * dih5 * dir;
    } else {
      const double dir2 = dir * dir, dir3 = dir2 * dir;
      b = -1.0 / 15.0 * dir3 + dih3 * 8.0 / 3.0 - 3.0 * u + 6.0 / 5.0 * u * u -
            1.0 / 6.0 * u * u * u;
      c = -1.0 / 5.0 * dir3 * dir2 + 3.0 * dih4 * dir - dih5 * 12.0 / 5.0 + 1.0 / 2.0 * u;
      d = -dir3 * dir3 * dir + 3.0 * dih4 * dir3 - 1.0 / 2.0 * dih6 * dir;
      br = 1.0 / 5.0 * dir2 * dir2 + dih * (-3.0 + 12.0 / 5.0 * u - 1.0 / 2.0 * u * u);
      cr = dir3 * dir3 - 3.0 * dih4 * dir2 + 1.0 / 2.0 * dih;
      dr_ = 7.0 * dir3 * dir3 * dir2 - 9.0 * dih4 * dir2 * dir2 + 1.0 / 2.0 * dih6 * dir2;
      bD = 8.0 * dih2 + r * (-3.0 + 12.0 / 5.0 * u - 1.0 / 2.0 * u * u);
      cD = 12.0 * dih3 * dir - 12.0 * dih4 + 1.0 / 2.0 * r;
      dD = 12.0 * dih3 * dir3 - 3.0 * dih5 * dir;
    }
    const double dd_dt = -0.5 * dih2;  // d(dih)/d(twoh)
    bt = bD * dd_dt;
    ct = cD * dd_dt;
    dt_ = dD * dd_dt;
  } else {
    const double a = dir;
    b = a * a * a;
    c = 3.0 * b * a * a;
    d = 5.0 * c * a * a;
    br = -3.0 * b * a;
    cr = -5.0 * c * a;
    dr_ = -7.0 * d * a;
    bt = ct = dt_ = 0.0;
  }
  // built once from scalars: field stores in the branches can be merged into
  // one store through a pointer select, which keeps the struct in scratch memory
  return SplineQ{b, c, d, br, cr, dr_, bt, ct, dt_};
}

struct TgtA {
  double x, y, z, e, wx, wy, wz;
  int32_t bt, pad;  // bt: the target's bucket within its group
};

// Squared distance from the box [lo, hi] to the point p.
__device__ __forceinline__ double box_dsq(const double lo[3], const double hi[3], double px,
                                          double py, double pz) {
  const double p[3] = {px, py, pz};
  double d = 0.0;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const double t = p[k] < lo[k] ? lo[k] - p[k] : (p[k] > hi[k] ? p[k] - hi[k] : 0.0);
    d += t * t;
  }
  return d;
}

// The far classification of a pass: a closed node whose centre lies farther
// from the box around the group's buckets than twice its softening plus the
// largest bucket softening fails both openSoftening tests for every member
// (each member's box and centre lie inside that box), and one farther than
// its softening plus the largest target softening is beyond the softened
// range of every pair; a source particle likewise beyond its softening plus
// the largest target softening, and a leaf when its centre is farther than
// its reach plus those softenings.  Margins of 2e-4 on the reaches and 1e-4
// on the squares also cover the FP32 form's shifted coordinates.
// Per wave, in LDS: lo[3], hi[3] of the box around the group's buckets, the
// largest bucket softening, the largest target softening of the pass.
constexpr int kPassFar = 8;

__device__ __forceinline__ bool node_far_pass(const double* __restrict__ f, double cx, double cy,
                                              double cz, double soft) {
  const double dsq = box_dsq(f, f + 3, cx, cy, cz);
  const double mono = 2.0 * (soft + f[6]);
  const double reach = (soft + f[7]) * 1.0002;
  const double m = mono > reach ? mono : reach;
  return dsq > 1.0001 * m * m;
}

__device__ __forceinline__ bool leaf_far_pass(const double* __restrict__ f, double cx, double cy,
                                              double cz, double lreach, double lsoft) {
  const double dsq = box_dsq(f, f + 3, cx, cy, cz);
  const double reach = (lreach + lsoft + f[7]) * 1.0002;
  return dsq > 1.0001 * reach * reach;
}

// The target gradients of a pass, in LDS: kAccCols partial sums per target and
// component, one per lane of each half wave; lane l adds to column l % 32 of
// row 3 t + component.  The odd stride spreads the rows over the banks for the
// final sums.  In registers (96 per lane, and the loop over the targets
// unrolled for their sake) they left one wave per SIMD, whose dependent FP64
// chains kept 45% of the issue slots.
constexpr int kAccCols = 32;
constexpr int kAccStride = kAccCols + 1;

__device__ __forceinline__ void lds_add(double* p, double v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// acc: the calling lane's column of row 0.
__device__ __forceinline__ void tgt_add(double* __restrict__ acc, int t, double x, double y,
                                        double z) {
  double* a = acc + t * (3 * kAccStride);
  lds_add(a, x);
  lds_add(a + kAccStride, y);
  lds_add(a + 2 * kAccStride, z);
}

// The column sums of the pass's ng targets, added to their records (from g).
__device__ __forceinline__ void tgt_flush(const double* __restrict__ s_acc, int ng,
                                          double* __restrict__ g) {
  const int row = threadIdx.x;
  if (row < 3 * ng) {
    const double* a = s_acc + row * kAccStride;
    double v = 0.0;
    for (int k = 0; k < kAccCols; k++) v += a[k];
    atomicAdd(g + 4 * (row / 3) + row % 3, v);
  }
}

// Source cotangents of a wave leave it through LDS, so that consecutive lanes
// add to consecutive fields of a record: the memory takes an atomic
// instruction one request per line, and with a field per instruction every
// lane's request was its own (256k clustered particles, FP64: 4930 -> 3800 us
// of adjoint, 2370 without any).
// F: fields per lane; s_val holds PT_WAVE * F values, the lane's own in
// s_val[lane * F ...], s_dst its record or null.
template <int F, class T>
__device__ __forceinline__ void record_add(const T* __restrict__ s_val, double* const* s_dst) {
  const int lane = threadIdx.x;
#pragma unroll
  for (int i = 0; i < F; i++) {
    const int q = i * PT_WAVE + lane;
    double* const d = s_dst[q / F];
    const T v = s_val[q];
    if (d && v != T(0)) atomicAdd(d + q % F, (double)v);
  }
}

// One node() list entry against the pass's targets (FP64): the target
// gradients into acc, the node cotangent into lam; mono: the members for which
// openSoftening sends the node to addGravity.  FAR (wave-uniform): every pair
// is a node() pair beyond its softening, b = 1/r^3, c = 3/r^5, d = 15/r^7 with
// derivatives -c r, -d r, -7 d / r and none in the softening.
template <bool FAR>
__device__ __forceinline__ void node_entry_pairs(const GravNode& s, unsigned mask, unsigned mono,
                                                 const TgtA* __restrict__ st, int ng, double ox,
                                                 double oy, double oz, double* __restrict__ acc,
                                                 double (&lam)[kNodeAdj]) {
  const double cx = s.cx + ox, cy = s.cy + oy, cz = s.cz + oz;
  double trace = 0.0;  // the part common to d(a.w)/dQ's diagonal
#pragma unroll 1
  for (int t = 0; t < ng; t++) {
    const TgtA tt = st[t];
    if ((mask >> tt.bt) & 1u) {
      if (!FAR && ((mono >> tt.bt) & 1u)) {
        const double dx = cx - tt.x, dy = cy - tt.y, dz = cz - tt.z;
        const double r2 = dx * dx + dy * dy + dz * dz;
        if (r2 != 0) {
          const double ir = pt_rsqrt64(r2);
          const double ir3 = ir * ir * ir;
          const double dw = dx * tt.wx + dy * tt.wy + dz * tt.wz;
          const double f = -3.0 * s.mass * ir3 * ir * ir * dw;
          const double Tx = s.mass * ir3 * tt.wx + f * dx;
          const double Ty = s.mass * ir3 * tt.wy + f * dy;
          const double Tz = s.mass * ir3 * tt.wz + f * dz;
          tgt_add(acc, t, -Tx, -Ty, -Tz);
          lam[0] += Tx;
          lam[1] += Ty;
          lam[2] += Tz;
          lam[3] += dw * ir3;
        }
      } else {
        const double rx = (tt.x - s.cx) - ox, ry = (tt.y - s.cy) - oy, rz = (tt.z - s.cz) - oz;
        const double r2 = fma(rx, rx, fma(ry, ry, rz * rz));
        const double ir = pt_rsqrt64(r2);
        const double qx = fma(s.qxx, rx, fma(s.qxy, ry, s.qxz * rz));
        const double qy = fma(s.qxy, rx, fma(s.qyy, ry, s.qyz * rz));
        const double qz = fma(s.qxz, rx, fma(s.qyz, ry, s.qzz * rz));
        const double qir = 0.5 * fma(qx, rx, fma(qy, ry, qz * rz));
        const double rw = fma(rx, tt.wx, fma(ry, tt.wy, rz * tt.wz));
        const double qw = fma(qx, tt.wx, fma(qy, tt.wy, qz * tt.wz));
        double b, c, d, k1, k2;
        if (FAR) {
          const double a2 = ir * ir;
          b = ir * a2;
          c = 3.0 * b * a2;
          d = 5.0 * c * a2;
          k1 = fma(-c, s.mass, d * fma(-7.0 * a2, qir, s.tr));
          k2 = -d;
        } else {
          const SplineQ q = splineq_grad(r2 * ir, ir, r2, s.soft + tt.e);
          b = q.b;
          c = q.c;
          d = q.d;
          k1 = fma(s.mass, q.br, fma(qir, q.dr_, -s.tr * q.cr)) * ir;
          k2 = q.cr * ir;
          lam[10] += fma(-fma(q.bt, s.mass, fma(q.dt_, qir, -q.ct * s.tr)), rw, q.ct * qw);
        }
        const double qir3 = fma(b, s.mass, fma(d, qir, -c * s.tr));
        // J = -qir3 w + (k2 (q.w) - k1 (r.w)) r - d (r.w) q + c Q w; with
        // p = c w - d (r.w) r / 2 its last two terms are Q p - d (r.w) q / 2
        const double s1 = fma(k2, qw, -k1 * rw);
        const double hd = -0.5 * (d * rw);
        const double px = fma(hd, rx, c * tt.wx), py = fma(hd, ry, c * tt.wy),
                     pz = fma(hd, rz, c * tt.wz);
        const double Qpx = fma(s.qxx, px, fma(s.qxy, py, s.qxz * pz));
        const double Qpy = fma(s.qxy, px, fma(s.qyy, py, s.qyz * pz));
        const double Qpz = fma(s.qxz, px, fma(s.qyz, py, s.qzz * pz));
        const double Jx = fma(-qir3, tt.wx, fma(s1, rx, fma(hd, qx, Qpx)));
        const double Jy = fma(-qir3, tt.wy, fma(s1, ry, fma(hd, qy, Qpy)));
        const double Jz = fma(-qir3, tt.wz, fma(s1, rz, fma(hd, qz, Qpz)));
        tgt_add(acc, t, Jx, Jy, Jz);
        lam[0] -= Jx;
        lam[1] -= Jy;
        lam[2] -= Jz;
        lam[3] = fma(-b, rw, lam[3]);
        // d(a.w)/dQ per stored component: r_k p_l + r_l p_k, on the diagonal
        // r_k p_k + c (r.w) / 2
        lam[4] = fma(rx, px, lam[4]);
        lam[5] = fma(ry, px, fma(rx, py, lam[5]));
        lam[6] = fma(rz, px, fma(rx, pz, lam[6]));
        lam[7] = fma(ry, py, lam[7]);
        lam[8] = fma(rz, py, fma(ry, pz, lam[8]));
        lam[9] = fma(rz, pz, lam[9]);
        trace = fma(c, rw, trace);
      }
    }
  }
  lam[4] = fma(0.5, trace, lam[4]);
  lam[7] = fma(0.5, trace, lam[7]);
  lam[9] = fma(0.5, trace, lam[9]);
}

// One source particle against the pass's targets (FP64).  FAR (wave-uniform):
// every pair is beyond its softening, so not the target itself.  The source's
// position gradient is summed before its mass factor.
template <bool FAR>
__device__ __forceinline__ void particle_pairs(double jx, double jy, double jz, double jm,
                                               double je, unsigned jmask,
                                               const TgtA* __restrict__ st, int ng,
                                               double* __restrict__ acc, double& sgx, double& sgy,
                                               double& sgz, double& sgm) {
  double kx = 0.0, ky = 0.0, kz = 0.0;
#pragma unroll 2
  for (int t = 0; t < ng; t++) {
    const TgtA tt = st[t];
    if ((jmask >> tt.bt) & 1u) {
      const double dx = jx - tt.x, dy = jy - tt.y, dz = jz - tt.z;
      const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
      if (FAR || r2 != 0) {
        const double ir = pt_rsqrt64(r2);
        const double dw = fma(dx, tt.wx, fma(dy, tt.wy, dz * tt.wz));
        double bb, f;  // f = b'(r) (d.w) / r
        if (FAR) {
          const double a2 = ir * ir;
          bb = ir * a2;
          f = -3.0 * (bb * a2) * dw;
        } else {
          double db;
          spline_b_db(r2 * ir, ir, je + tt.e, bb, db);
          f = db * ir * dw;
        }
        const double Kx = fma(bb, tt.wx, f * dx);
        const double Ky = fma(bb, tt.wy, f * dy);
        const double Kz = fma(bb, tt.wz, f * dz);
        tgt_add(acc, t, -jm * Kx, -jm * Ky, -jm * Kz);
        kx += Kx;
        ky += Ky;
        kz += Kz;
        sgm = fma(bb, dw, sgm);
      }
    }
  }
  sgx += jm * kx;
  sgy += jm * ky;
  sgz += jm * kz;
}

// One wave per bucket group (consecutive buckets, at most PT_GROUP_TARGETS
// particles unless one bucket is larger; neighbouring buckets share most of
// their sources, so a group's union list is far shorter than the sum of its
// buckets' lists).  Node sources: one list entry per lane, looping over the
// group's targets (PT_GROUP_TARGETS per pass) from LDS and evaluating the
// pairs whose target bucket is in the entry's member mask; the node cotangent
// is summed over the targets of a pass before one atomic add per field.  Leaf
// sources: flattened to one source particle per lane (the leaf's mask
// carried along); the source's gradient is summed over the targets of a pass
// before its atomic adds.  Target gradients are summed in LDS (tgt_add).  One
// wave per work-group, in an order that keeps every XCD supplied
// (pt_part_item); the waves of a grid column share a group's lists, every
// gridDim.y-th chunk each.
__global__ void __launch_bounds__(PT_WAVE)
adjoint_group_kernel(const Bucket* __restrict__ bk, const int32_t* __restrict__ gfirst,
                     const int32_t* __restrict__ gnb, const uint32_t* __restrict__ ngroups,
                     const TreeNode* __restrict__ nodes,
                    const GravNode* __restrict__ gn, const double* __restrict__ px,
                    const double* __restrict__ py, const double* __restrict__ pz,
                    const double* __restrict__ pm, const double* __restrict__ pe,
                    const int64_t* __restrict__ pp_off, const int32_t* __restrict__ pp,
                    const uint8_t* __restrict__ ppm, const int64_t* __restrict__ pc_off,
                    const int32_t* __restrict__ pc, const uint8_t* __restrict__ pcm,
                    double ox, double oy, double oz, const double* __restrict__ wx,
                    const double* __restrict__ wy, const double* __restrict__ wz,
                    double* __restrict__ gs, double* __restrict__ lam_node,
                    double* __restrict__ hot, int64_t nhot) {
  __shared__ TgtA s_t[kANT];
  __shared__ Bucket s_bk[PT_GROUP_BUCKETS];
  __shared__ int32_t s_beg[PT_WAVE];
  __shared__ double s_far[kPassFar];
  __shared__ double s_acc[kANT * 3 * kAccStride];
  __shared__ double s_val[PT_WAVE * kNodeAdj];
  __shared__ double* s_dst[PT_WAVE];
  const int lane = threadIdx.x;
  const int64_t gi = pt_part_item((int32_t)ngroups[0]);
  if (gi < 0) return;
  const int nbk = gnb[gi];
  const int64_t b0 = gfirst[gi];
  if (lane < nbk) s_bk[lane] = bk[b0 + lane];
  __builtin_amdgcn_wave_barrier();
  // the group's targets are consecutive: its buckets' ranges in order
  const int64_t first = s_bk[0].begin;
  const int nt = (int)((int64_t)s_bk[nbk - 1].begin + s_bk[nbk - 1].count - first);
  const int64_t pc0 = pc_off[gi], pc1 = pc_off[gi + 1];
  const int64_t pp0 = pp_off[gi], pp1 = pp_off[gi + 1];
  if (lane < 7) {
    // the group's box and largest bucket softening
    double v = lane < 3 ? INFINITY : (lane < 6 ? -INFINITY : 0.0);
    for (int k = 0; k < nbk; k++) {
      const Bucket& bb = s_bk[k];
      const double c[7] = {bb.lox, bb.loy, bb.loz, bb.hix, bb.hiy, bb.hiz, bb.soft};
      v = lane < 3 ? fmin(v, c[lane]) : fmax(v, c[lane]);
    }
    s_far[lane] = v;
  }
  for (int g0 = 0; g0 < nt; g0 += kANT) {
    const int ng = (nt - g0) < kANT ? (nt - g0) : kANT;
    // member buckets with a target in this pass
    unsigned pass = 0;
    for (int k = 0; k < nbk; k++) {
      const int64_t lo = s_bk[k].begin, hi = lo + s_bk[k].count;
      if (hi > first + g0 && lo < first + g0 + ng) pass |= 1u << k;
    }
    __builtin_amdgcn_wave_barrier();
    if (lane < ng) {
      const int64_t i = first + g0 + lane;
      int bt = 0;
      for (int k = 1; k < nbk; k++)
        if (i >= s_bk[k].begin) bt = k;
      s_t[lane] = TgtA{px[i], py[i], pz[i], pe[i], wx[i], wy[i], wz[i], bt, 0};
    }
    for (int k = lane; k < 3 * ng * kAccStride; k += PT_WAVE) s_acc[k] = 0.0;
    __syncthreads();
    double* const acc = s_acc + lane % kAccCols;
    if (lane == 0) {
      double emax = 0.0;
      for (int t = 0; t < ng; t++) emax = s_t[t].e > emax ? s_t[t].e : emax;
      s_far[7] = emax;
    }
    __syncthreads();

    // ---- node() sources: in chunks in which every entry is far no member's
    // openSoftening can hold, so its tests are skipped
    for (int64_t e0 = pc0 + blockIdx.y * PT_WAVE; e0 < pc1; e0 += gridDim.y * PT_WAVE) {
      const int64_t e = e0 + lane;
      const unsigned mask = e < pc1 ? (unsigned)pcm[e] & pass : 0u;
      double* dst = nullptr;
      if (mask != 0u) {
        const int32_t sid = pc[e];
        const GravNode s = gn[sid];
        const bool far = node_far_pass(s_far, s.cx + ox, s.cy + oy, s.cz + oz, s.soft);
        // over the lanes holding an entry (the others are inactive here)
        const bool all_far = __ballot(!far) == 0ull;
        double lam[kNodeAdj];
#pragma unroll
        for (int k = 0; k < kNodeAdj; k++) lam[k] = 0.0;
        // members for which openSoftening sends it to addGravity (none when
        // every entry of the chunk is far)
        unsigned mono = 0;
        if (!all_far) {
          for (unsigned mm = mask; mm != 0u; mm &= mm - 1u) {
            const int k = __builtin_ctz(mm);
            if (pt_open_softening(s.cx + ox, s.cy + oy, s.cz + oz, s.soft, s_bk[k]))
              mono |= 1u << k;
          }
        }
        if (all_far)
          node_entry_pairs<true>(s, mask, 0u, s_t, ng, ox, oy, oz, acc, lam);
        else
          node_entry_pairs<false>(s, mask, mono, s_t, ng, ox, oy, oz, acc, lam);
        dst = sid < nhot ? hot + ((int64_t)(blockIdx.x % kHotParts) * nhot + sid) * kNodeRow
                         : lam_node + (int64_t)sid * kNodeRow;
#pragma unroll
        for (int k = 0; k < kNodeAdj; k++) s_val[lane * kNodeAdj + k] = lam[k];
      }
      s_dst[lane] = dst;
      __syncthreads();
      record_add<kNodeAdj>(s_val, s_dst);
      __syncthreads();
    }

    // ---- leaf() sources, flattened to particles, the leaves that may hold a
    // softened pair first: windows past them take the branch-free form
    for (int64_t l0 = pp0 + blockIdx.y * PT_WAVE; l0 < pp1; l0 += gridDim.y * PT_WAVE) {
      const int64_t l = l0 + lane;
      int32_t cnt = 0, beg = 0;
      bool isnear = false;
      const unsigned msk = l < pp1 ? (unsigned)ppm[l] & pass : 0u;
      if (msk != 0u) {
        const TreeNode nd = nodes[pp[l]];
        cnt = nd.count;
        beg = nd.begin;
        isnear = !leaf_far_pass(s_far, nd.cx + ox, nd.cy + oy, nd.cz + oz, nd.leaf_reach,
                                nd.leaf_soft);
      }
      const int cn = isnear ? cnt : 0, cf = isnear ? 0 : cnt;
      const int incl_n = pt_wave_incl_scan(cn);
      const int incl_f = pt_wave_incl_scan(cf);
      const int near_total = __builtin_amdgcn_readlane(incl_n, PT_WAVE - 1);
      const int total = near_total + __builtin_amdgcn_readlane(incl_f, PT_WAVE - 1);
      // each entry's first slot, near entries first
      const int exc = isnear ? incl_n - cn : near_total + incl_f - cf;
      int carry = 0;
      for (int s0 = 0; s0 < total; s0 += PT_WAVE) {
        const bool wfar = s0 >= near_total;
        // a slot's entry: the lane of the last entry start at or below it in
        // this window (marks by start slot, a ballot of the marks), or the
        // previous window's last entry
        int32_t* mark = s_beg;
        mark[lane] = -1;
        __builtin_amdgcn_wave_barrier();
        if (cnt > 0 && exc >= s0 && exc < s0 + PT_WAVE) mark[exc - s0] = lane;
        __builtin_amdgcn_wave_barrier();
        const unsigned long long starts = __ballot(mark[lane] >= 0);
        const unsigned long long upto = starts & (~0ull >> (PT_WAVE - 1 - lane));
        const int leaf = upto ? mark[PT_WAVE - 1 - __clzll(upto)] : carry;
        carry = __builtin_amdgcn_readlane(leaf, PT_WAVE - 1);
        const int lbeg = __shfl(beg, leaf, PT_WAVE);
        const int lexc = __shfl(exc, leaf, PT_WAVE);
        const unsigned jmask = (unsigned)__shfl((int)msk, leaf, PT_WAVE);
        const int slot = s0 + lane;
        double* dst = nullptr;
        if (slot < total) {
          const int64_t j = (int64_t)lbeg + (slot - lexc);
          const double jx = px[j] + ox, jy = py[j] + oy, jz = pz[j] + oz;
          const double jm = pm[j], je = pe[j];
          double sgx = 0.0, sgy = 0.0, sgz = 0.0, sgm = 0.0;
          if (wfar)
            particle_pairs<true>(jx, jy, jz, jm, je, jmask, s_t, ng, acc, sgx, sgy, sgz, sgm);
          else
            particle_pairs<false>(jx, jy, jz, jm, je, jmask, s_t, ng, acc, sgx, sgy, sgz, sgm);
          s_val[lane * 4] = sgx;
          s_val[lane * 4 + 1] = sgy;
          s_val[lane * 4 + 2] = sgz;
          s_val[lane * 4 + 3] = sgm;
          dst = gs + 4 * j;
        }
        s_dst[lane] = dst;
        __syncthreads();
        record_add<4>(s_val, s_dst);
        __syncthreads();
      }
      __builtin_amdgcn_wave_barrier();
    }

    __syncthreads();
    tgt_flush(s_acc, ng, gs + 4 * (first + g0));
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// FP32 form: the same pair expressions in FP32 on coordinates shifted to the
// centre of the group's box (in FP64, then rounded), with the hardware reciprocal
// and reciprocal square root; every sum that spans pairs (target gradients,
// node and source-particle cotangents) is carried in FP64.
// ---------------------------------------------------------------------------

__device__ __forceinline__ float rcp32(float x) { return __builtin_amdgcn_rcpf(x); }

// spline_b_db in FP32; ir = 1 / r.
__device__ __forceinline__ void spline_b_db32(float r, float ir, float twoh, float& b, float& db) {
  if (r < twoh) {
    const float dih = 2.0f * rcp32(twoh);
    const float u = r * dih;
    const float dih3 = dih * dih * dih;
    if (u < 1.0f) {
      b = dih3 * (4.0f / 3.0f - 6.0f / 5.0f * u * u + 1.0f / 2.0f * u * u * u);
      db = dih3 * dih * (-12.0f / 5.0f * u + 3.0f / 2.0f * u * u);
    } else {
      b = -1.0f / 15.0f * ir * ir * ir +
          dih3 * (8.0f / 3.0f - 3.0f * u + 6.0f / 5.0f * u * u - 1.0f / 6.0f * u * u * u);
      db = 1.0f / 5.0f * ir * ir * ir * ir +
           dih3 * dih * (-3.0f + 12.0f / 5.0f * u - 1.0f / 2.0f * u * u);
    }
  } else {
    b = ir * ir * ir;
    db = -3.0f * b * ir;
  }
}

struct SplineQ32 {
  float b, c, d, br, cr, dr_, bt, ct, dt_;
};

// splineq_grad in FP32; ir = 1 / r.
__device__ __forceinline__ SplineQ32 splineq_grad32(float r, float ir, float r2, float twoh) {
  float b, c, d, br, cr, dr_, bt, ct, dt_;
  const float dir = ir;
  if (r2 < twoh * twoh) {
    const float dih = 2.0f * rcp32(twoh);
    const float u = dih * r;
    const float dih2 = dih * dih, dih3 = dih2 * dih, dih4 = dih3 * dih, dih5 = dih4 * dih,
                dih6 = dih5 * dih;
    float bD, cD, dD;
    if (u < 1.0f) {
      b = dih3 * 4.0f / 3.0f - 6.0f / 5.0f * u * u + 1.0f / 2.0f * u * u * u;
      c = dih5 * 12.0f / 5.0f - 3.0f / 2.0f * u;
      d = 3.0f / 2.0f * dih6 * dir;
      br = dih * (-12.0f / 5.0f * u + 3.0f / 2.0f * u * u);
      cr = -3.0f / 2.0f * dih;
      dr_ = -3.0f / 2.0f * dih6 * dir * dir;
      bD = 4.0f * dih2 + r * (-12.0f / 5.0f * u + 3.0f / 2.0f * u * u);
      cD = 12.0f * dih4 - 3.0f / 2.0f * r;
      dD = 9.0f * dih5 * dir;
    } else {
      const float dir2 = dir * dir, dir3 = dir2 * dir;
      b = -1.0f / 15.0f * dir3 + dih3 * 8.0f / 3.0f - 3.0f * u + 6.0f / 5.0f * u * u -
            1.0f / 6.0f * u * u * u;
      c = -1.0f / 5.0f * dir3 * dir2 + 3.0f * dih4 * dir - dih5 * 12.0f / 5.0f + 1.0f / 2.0f * u;
      d = -dir3 * dir3 * dir + 3.0f * dih4 * dir3 - 1.0f / 2.0f * dih6 * dir;
      br = 1.0f / 5.0f * dir2 * dir2 + dih * (-3.0f + 12.0f / 5.0f * u - 1.0f / 2.0f * u * u);
      cr = dir3 * dir3 - 3.0f * dih4 * dir2 + 1.0f / 2.0f * dih;
      dr_ = 7.0f * dir3 * dir3 * dir2 - 9.0f * dih4 * dir2 * dir2 + 1.0f / 2.0f * dih6 * dir2;
      bD = 8.0f * dih2 + r * (-3.0f + 12.0f / 5.0f * u - 1.0f / 2.0f * u * u);
      cD = 12.0f * dih3 * dir - 12.0f * dih4 + 1.0f / 2.0f * r;
      dD = 12.0f * dih3 * dir3 - 3.0f * dih5 * dir;
    }
    const float dd_dt = -0.5f * dih2;
    bt = bD * dd_dt;
    ct = cD * dd_dt;
    dt_ = dD * dd_dt;
  } else {
    const float a = dir;
    b = a * a * a;
    c = 3.0f * b * a * a;
    d = 5.0f * c * a * a;
    br = -3.0f * b * a;
    cr = -5.0f * c * a;
    dr_ = -7.0f * d * a;
    bt = ct = dt_ = 0.0f;
  }
  // built once from scalars: field stores in the branches can be merged into
  // one store through a pointer select, which keeps the struct in scratch memory
  return SplineQ32{b, c, d, br, cr, dr_, bt, ct, dt_};
}

struct TgtA32 {
  float x, y, z, e, wx, wy, wz;
  int32_t bt;
};

// node_entry_pairs in FP32; cx, cy, cz: the node's centre in the group's frame.
template <bool FAR>
__device__ __forceinline__ void node_entry_pairs32(const GravNode32& s, float cx, float cy,
                                                   float cz, unsigned mask, unsigned mono,
                                                   const TgtA32* __restrict__ st, int ng,
                                                   double* __restrict__ acc,
                                                   float (&lam)[kNodeAdj]) {
  const float tr = 0.5f * (s.qxx + s.qyy + s.qzz);
  float trace = 0.0f;
#pragma unroll 1
  for (int t = 0; t < ng; t++) {
    const TgtA32 tt = st[t];
    if ((mask >> tt.bt) & 1u) {
      if (!FAR && ((mono >> tt.bt) & 1u)) {
        const float dx = cx - tt.x, dy = cy - tt.y, dz = cz - tt.z;
        const float r2 = dx * dx + dy * dy + dz * dz;
        if (r2 != 0.0f) {
          const float ir = __builtin_amdgcn_rsqf(r2);
          const float ir3 = ir * ir * ir;
          const float dw = dx * tt.wx + dy * tt.wy + dz * tt.wz;
          const float f = -3.0f * s.mass * ir3 * ir * ir * dw;
          const float Tx = s.mass * ir3 * tt.wx + f * dx;
          const float Ty = s.mass * ir3 * tt.wy + f * dy;
          const float Tz = s.mass * ir3 * tt.wz + f * dz;
          tgt_add(acc, t, -(double)Tx, -(double)Ty, -(double)Tz);
          lam[0] += Tx;
          lam[1] += Ty;
          lam[2] += Tz;
          lam[3] += dw * ir3;
        }
      } else {
        const float rx = tt.x - cx, ry = tt.y - cy, rz = tt.z - cz;
        const float r2 = fmaf(rx, rx, fmaf(ry, ry, rz * rz));
        const float ir = __builtin_amdgcn_rsqf(r2);
        const float qx = fmaf(s.qxx, rx, fmaf(s.qxy, ry, s.qxz * rz));
        const float qy = fmaf(s.qxy, rx, fmaf(s.qyy, ry, s.qyz * rz));
        const float qz = fmaf(s.qxz, rx, fmaf(s.qyz, ry, s.qzz * rz));
        const float qir = 0.5f * fmaf(qx, rx, fmaf(qy, ry, qz * rz));
        const float rw = fmaf(rx, tt.wx, fmaf(ry, tt.wy, rz * tt.wz));
        const float qw = fmaf(qx, tt.wx, fmaf(qy, tt.wy, qz * tt.wz));
        float b, c, d, k1, k2;
        if (FAR) {
          const float a2 = ir * ir;
          b = ir * a2;
          c = 3.0f * b * a2;
          d = 5.0f * c * a2;
          k1 = fmaf(-c, s.mass, d * fmaf(-7.0f * a2, qir, tr));
          k2 = -d;
        } else {
          const SplineQ32 q = splineq_grad32(r2 * ir, ir, r2, s.soft + tt.e);
          b = q.b;
          c = q.c;
          d = q.d;
          k1 = fmaf(s.mass, q.br, fmaf(qir, q.dr_, -tr * q.cr)) * ir;
          k2 = q.cr * ir;
          lam[10] += fmaf(-fmaf(q.bt, s.mass, fmaf(q.dt_, qir, -q.ct * tr)), rw, q.ct * qw);
        }
        const float qir3 = fmaf(b, s.mass, fmaf(d, qir, -c * tr));
        const float s1 = fmaf(k2, qw, -k1 * rw);
        const float hd = -0.5f * (d * rw);
        const float px = fmaf(hd, rx, c * tt.wx), py = fmaf(hd, ry, c * tt.wy),
                    pz = fmaf(hd, rz, c * tt.wz);
        const float Qpx = fmaf(s.qxx, px, fmaf(s.qxy, py, s.qxz * pz));
        const float Qpy = fmaf(s.qxy, px, fmaf(s.qyy, py, s.qyz * pz));
        const float Qpz = fmaf(s.qxz, px, fmaf(s.qyz, py, s.qzz * pz));
        const float Jx = fmaf(-qir3, tt.wx, fmaf(s1, rx, fmaf(hd, qx, Qpx)));
        const float Jy = fmaf(-qir3, tt.wy, fmaf(s1, ry, fmaf(hd, qy, Qpy)));
        const float Jz = fmaf(-qir3, tt.wz, fmaf(s1, rz, fmaf(hd, qz, Qpz)));
        tgt_add(acc, t, (double)Jx, (double)Jy, (double)Jz);
        lam[0] -= Jx;
        lam[1] -= Jy;
        lam[2] -= Jz;
        lam[3] = fmaf(-b, rw, lam[3]);
        lam[4] = fmaf(rx, px, lam[4]);
        lam[5] = fmaf(ry, px, fmaf(rx, py, lam[5]));
        lam[6] = fmaf(rz, px, fmaf(rx, pz, lam[6]));
        lam[7] = fmaf(ry, py, lam[7]);
        lam[8] = fmaf(rz, py, fmaf(ry, pz, lam[8]));
        lam[9] = fmaf(rz, pz, lam[9]);
        trace = fmaf(c, rw, trace);
      }
    }
  }
  lam[4] = fmaf(0.5f, trace, lam[4]);
  lam[7] = fmaf(0.5f, trace, lam[7]);
  lam[9] = fmaf(0.5f, trace, lam[9]);
}

// particle_pairs in FP32, the target gradients summed in FP64.
template <bool FAR>
__device__ __forceinline__ void particle_pairs32(float jx, float jy, float jz, float jm, float je,
                                                 unsigned jmask, const TgtA32* __restrict__ st,
                                                 int ng, double* __restrict__ acc, float& sgx,
                                                 float& sgy, float& sgz, float& sgm) {
#pragma unroll 2
  for (int t = 0; t < ng; t++) {
    const TgtA32 tt = st[t];
    if ((jmask >> tt.bt) & 1u) {
      const float dx = jx - tt.x, dy = jy - tt.y, dz = jz - tt.z;
      const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
      if (FAR || r2 != 0.0f) {
        const float ir = __builtin_amdgcn_rsqf(r2);
        float bb, db;
        if (FAR) {
          bb = ir * ir * ir;
          db = -3.0f * bb * ir;
        } else {
          spline_b_db32(r2 * ir, ir, je + tt.e, bb, db);
        }
        const float dw = fmaf(dx, tt.wx, fmaf(dy, tt.wy, dz * tt.wz));
        const float f = db * ir * dw;
        const float Kx = jm * fmaf(bb, tt.wx, f * dx);
        const float Ky = jm * fmaf(bb, tt.wy, f * dy);
        const float Kz = jm * fmaf(bb, tt.wz, f * dz);
        tgt_add(acc, t, -(double)Kx, -(double)Ky, -(double)Kz);
        sgx += Kx;
        sgy += Ky;
        sgz += Kz;
        sgm = fmaf(bb, dw, sgm);
      }
    }
  }
}

// adjoint_group_kernel in the FP32 form (same work mapping; node moments from
// the FP32 copies, node centres and softening decisions from the FP64 fields
// of the same records).
__global__ void __launch_bounds__(PT_WAVE)
adjoint_group32_kernel(const Bucket* __restrict__ bk, const int32_t* __restrict__ gfirst,
                       const int32_t* __restrict__ gnb, const uint32_t* __restrict__ ngroups,
                      const TreeNode* __restrict__ nodes, const GravNode32* __restrict__ gn32,
                      const double* __restrict__ px,
                      const double* __restrict__ py, const double* __restrict__ pz,
                      const double* __restrict__ pm, const double* __restrict__ pe,
                      const int64_t* __restrict__ pp_off, const int32_t* __restrict__ pp,
                      const uint8_t* __restrict__ ppm, const int64_t* __restrict__ pc_off,
                      const int32_t* __restrict__ pc, const uint8_t* __restrict__ pcm,
                      double ox, double oy, double oz, const double* __restrict__ wx,
                      const double* __restrict__ wy, const double* __restrict__ wz,
                      double* __restrict__ gs, double* __restrict__ lam_node,
                      double* __restrict__ hot, int64_t nhot) {
  __shared__ TgtA32 s_t[kANT];
  __shared__ Bucket s_bk[PT_GROUP_BUCKETS];
  __shared__ int32_t s_beg[PT_WAVE];
  __shared__ double s_far[kPassFar];
  __shared__ double s_acc[kANT * 3 * kAccStride];
  __shared__ float s_val[PT_WAVE * kNodeAdj];
  __shared__ double* s_dst[PT_WAVE];
  const int lane = threadIdx.x;
  const int64_t gi = pt_part_item((int32_t)ngroups[0]);
  if (gi < 0) return;
  const int nbk = gnb[gi];
  const int64_t b0 = gfirst[gi];
  if (lane < nbk) s_bk[lane] = bk[b0 + lane];
  __builtin_amdgcn_wave_barrier();
  // the group's targets are consecutive: its buckets' ranges in order
  const int64_t first = s_bk[0].begin;
  const int nt = (int)((int64_t)s_bk[nbk - 1].begin + s_bk[nbk - 1].count - first);
  // FP32 frame: the centre of the box around the group's bucket boxes
  double lx = s_bk[0].lox, ly = s_bk[0].loy, lz = s_bk[0].loz;
  double hx = s_bk[0].hix, hy = s_bk[0].hiy, hz = s_bk[0].hiz;
  for (int k = 1; k < nbk; k++) {
    lx = fmin(lx, s_bk[k].lox);
    ly = fmin(ly, s_bk[k].loy);
    lz = fmin(lz, s_bk[k].loz);
    hx = fmax(hx, s_bk[k].hix);
    hy = fmax(hy, s_bk[k].hiy);
    hz = fmax(hz, s_bk[k].hiz);
  }
  const double ccx = (lx + hx) * 0.5, ccy = (ly + hy) * 0.5, ccz = (lz + hz) * 0.5;
  if (lane < 7) {
    // the group's box and largest bucket softening
    double v = lane < 3 ? INFINITY : (lane < 6 ? -INFINITY : 0.0);
    for (int k = 0; k < nbk; k++) {
      const Bucket& bb = s_bk[k];
      const double c[7] = {bb.lox, bb.loy, bb.loz, bb.hix, bb.hiy, bb.hiz, bb.soft};
      v = lane < 3 ? fmin(v, c[lane]) : fmax(v, c[lane]);
    }
    s_far[lane] = v;
  }
  const int64_t pc0 = pc_off[gi], pc1 = pc_off[gi + 1];
  const int64_t pp0 = pp_off[gi], pp1 = pp_off[gi + 1];
  for (int g0 = 0; g0 < nt; g0 += kANT) {
    const int ng = (nt - g0) < kANT ? (nt - g0) : kANT;
    // member buckets with a target in this pass
    unsigned pass = 0;
    for (int k = 0; k < nbk; k++) {
      const int64_t lo = s_bk[k].begin, hi = lo + s_bk[k].count;
      if (hi > first + g0 && lo < first + g0 + ng) pass |= 1u << k;
    }
    __builtin_amdgcn_wave_barrier();
    if (lane < ng) {
      const int64_t i = first + g0 + lane;
      int bt = 0;
      for (int k = 1; k < nbk; k++)
        if (i >= s_bk[k].begin) bt = k;
      s_t[lane] = TgtA32{(float)(px[i] - ccx), (float)(py[i] - ccy), (float)(pz[i] - ccz),
                               (float)pe[i], (float)wx[i], (float)wy[i], (float)wz[i], bt};
    }
    for (int k = lane; k < 3 * ng * kAccStride; k += PT_WAVE) s_acc[k] = 0.0;
    __syncthreads();
    double* const acc = s_acc + lane % kAccCols;
    if (lane == 0) {
      double emax = 0.0;
      for (int t = 0; t < ng; t++) emax = fmax(emax, (double)s_t[t].e);
      s_far[7] = emax;
    }
    __syncthreads();

    // ---- node() sources
    for (int64_t e0 = pc0 + blockIdx.y * PT_WAVE; e0 < pc1; e0 += gridDim.y * PT_WAVE) {
      const int64_t e = e0 + lane;
      const unsigned mask = e < pc1 ? (unsigned)pcm[e] & pass : 0u;
      double* dst = nullptr;
      if (mask != 0u) {
        const int32_t sid = pc[e];
        const GravNode32 s = gn32[sid];
        const double cxd = s.cx + ox, cyd = s.cy + oy, czd = s.cz + oz;
        // over the lanes holding an entry (the others are inactive here)
        const bool all_far = __ballot(!node_far_pass(s_far, cxd, cyd, czd, s.soft64)) == 0ull;
        // members for which openSoftening sends it to addGravity (none when
        // every entry of the chunk is far)
        unsigned mono = 0;
        if (!all_far) {
          for (unsigned mm = mask; mm != 0u; mm &= mm - 1u) {
            const int k = __builtin_ctz(mm);
            if (pt_open_softening(cxd, cyd, czd, s.soft64, s_bk[k])) mono |= 1u << k;
          }
        }
        const float cx = (float)(cxd - ccx), cy = (float)(cyd - ccy), cz = (float)(czd - ccz);
        float lam[kNodeAdj];
#pragma unroll
        for (int k = 0; k < kNodeAdj; k++) lam[k] = 0.0f;
        if (all_far)
          node_entry_pairs32<true>(s, cx, cy, cz, mask, 0u, s_t, ng, acc, lam);
        else
          node_entry_pairs32<false>(s, cx, cy, cz, mask, mono, s_t, ng, acc, lam);
        dst = sid < nhot ? hot + ((int64_t)(blockIdx.x % kHotParts) * nhot + sid) * kNodeRow
                         : lam_node + (int64_t)sid * kNodeRow;
#pragma unroll
        for (int k = 0; k < kNodeAdj; k++) s_val[lane * kNodeAdj + k] = lam[k];
      }
      s_dst[lane] = dst;
      __syncthreads();
      record_add<kNodeAdj>(s_val, s_dst);
      __syncthreads();
    }

    // ---- leaf() sources, flattened to particles, the leaves that may hold a
    // softened pair first: windows past them take the branch-free form
    for (int64_t l0 = pp0 + blockIdx.y * PT_WAVE; l0 < pp1; l0 += gridDim.y * PT_WAVE) {
      const int64_t l = l0 + lane;
      int32_t cnt = 0, beg = 0;
      bool isnear = false;
      const unsigned msk = l < pp1 ? (unsigned)ppm[l] & pass : 0u;
      if (msk != 0u) {
        const TreeNode nd = nodes[pp[l]];
        cnt = nd.count;
        beg = nd.begin;
        isnear = !leaf_far_pass(s_far, nd.cx + ox, nd.cy + oy, nd.cz + oz, nd.leaf_reach,
                                nd.leaf_soft);
      }
      const int cn = isnear ? cnt : 0, cf = isnear ? 0 : cnt;
      const int incl_n = pt_wave_incl_scan(cn);
      const int incl_f = pt_wave_incl_scan(cf);
      const int near_total = __builtin_amdgcn_readlane(incl_n, PT_WAVE - 1);
      const int total = near_total + __builtin_amdgcn_readlane(incl_f, PT_WAVE - 1);
      // each entry's first slot, near entries first
      const int exc = isnear ? incl_n - cn : near_total + incl_f - cf;
      int carry = 0;
      for (int s0 = 0; s0 < total; s0 += PT_WAVE) {
        const bool wfar = s0 >= near_total;
        // a slot's entry: the lane of the last entry start at or below it in
        // this window (marks by start slot, a ballot of the marks), or the
        // previous window's last entry
        int32_t* mark = s_beg;
        mark[lane] = -1;
        __builtin_amdgcn_wave_barrier();
        if (cnt > 0 && exc >= s0 && exc < s0 + PT_WAVE) mark[exc - s0] = lane;
        __builtin_amdgcn_wave_barrier();
        const unsigned long long starts = __ballot(mark[lane] >= 0);
        const unsigned long long upto = starts & (~0ull >> (PT_WAVE - 1 - lane));
        const int leaf = upto ? mark[PT_WAVE - 1 - __clzll(upto)] : carry;
        carry = __builtin_amdgcn_readlane(leaf, PT_WAVE - 1);
        const int lbeg = __shfl(beg, leaf, PT_WAVE);
        const int lexc = __shfl(exc, leaf, PT_WAVE);
        const unsigned jmask = (unsigned)__shfl((int)msk, leaf, PT_WAVE);
        const int slot = s0 + lane;
        double* dst = nullptr;
        if (slot < total) {
          const int64_t j = (int64_t)lbeg + (slot - lexc);
          const float jx = (float)((px[j] + ox) - ccx), jy = (float)((py[j] + oy) - ccy),
                      jz = (float)((pz[j] + oz) - ccz);
          const float jm = (float)pm[j], je = (float)pe[j];
          float sgx = 0.0f, sgy = 0.0f, sgz = 0.0f, sgm = 0.0f;
          if (wfar)
            particle_pairs32<true>(jx, jy, jz, jm, je, jmask, s_t, ng, acc, sgx, sgy, sgz, sgm);
          else
            particle_pairs32<false>(jx, jy, jz, jm, je, jmask, s_t, ng, acc, sgx, sgy, sgz, sgm);
          s_val[lane * 4] = sgx;
          s_val[lane * 4 + 1] = sgy;
          s_val[lane * 4 + 2] = sgz;
          s_val[lane * 4 + 3] = sgm;
          dst = gs + 4 * j;
        }
        s_dst[lane] = dst;
        __syncthreads();
        record_add<4>(s_val, s_dst);
        __syncthreads();
      }
      __builtin_amdgcn_wave_barrier();
    }

    __syncthreads();
    tgt_flush(s_acc, ng, gs + 4 * (first + g0));
    __syncthreads();
  }
}

// Pushes node cotangents to every particle through the closed-form moments of
// its leaf and each ancestor (parent links up to the root).
__global__ void __launch_bounds__(256)
adjoint_down_kernel(int64_t n, const uint32_t* __restrict__ bucket_of,
                    const int32_t* __restrict__ bucket_node,
                    const int32_t* __restrict__ parent, const GravNode* __restrict__ gn,
                    const double* __restrict__ lam_node, const double* __restrict__ gs,
                    const uint32_t* __restrict__ perm, const double* __restrict__ px, const double* __restrict__ py,
                    const double* __restrict__ pz, const double* __restrict__ pm,
                    const double* __restrict__ pe, double* __restrict__ gx,
                    double* __restrict__ gy, double* __restrict__ gz,
                    double* __restrict__ gmass) {
  const int64_t j = blockIdx.x * 256ll + threadIdx.x;
  if (j >= n) return;
  int32_t s = bucket_node[bucket_of[j]];
  const double x = px[j], y = py[j], z = pz[j], m = pm[j], e = pe[j];
  double ax = 0.0, ay = 0.0, az = 0.0, am = 0.0;
  while (s >= 0) {
    const GravNode g = gn[s];
    if (g.mass != 0.0) {
      double l[kNodeAdj];
#pragma unroll
      for (int k = 0; k < kNodeAdj; k++) l[k] = lam_node[(int64_t)s * kNodeRow + k];
      const double ux = x - g.cx, uy = y - g.cy, uz = z - g.cz;
      const double im = 1.0 / g.mass;
      ax += m * (im * l[0] + 2.0 * l[4] * ux + l[5] * uy + l[6] * uz);
      ay += m * (im * l[1] + l[5] * ux + 2.0 * l[7] * uy + l[8] * uz);
      az += m * (im * l[2] + l[6] * ux + l[8] * uy + 2.0 * l[9] * uz);
      am += l[3] + (l[0] * ux + l[1] * uy + l[2] * uz) * im + l[4] * ux * ux + l[5] * ux * uy +
            l[6] * ux * uz + l[7] * uy * uy + l[8] * uy * uz + l[9] * uz * uz +
            l[10] * (e - g.soft) * im;
    }
    s = parent[s];
  }
  const uint32_t i = perm[j];
  gx[i] += gs[4 * j] + ax;
  gy[i] += gs[4 * j + 1] + ay;
  gz[i] += gs[4 * j + 2] + az;
  gmass[i] += gs[4 * j + 3] + am;
}

// FP64 direct sum of the leaf() kernel over every pair, one block per target.
__global__ void __launch_bounds__(256)
direct_all_kernel(int64_t n, const double* __restrict__ x, const double* __restrict__ y,
                  const double* __restrict__ z, const double* __restrict__ m,
                  const double* __restrict__ e, double* __restrict__ ax, double* __restrict__ ay,
                  double* __restrict__ az, double* __restrict__ pot) {
  __shared__ double red[3][256 / PT_WAVE];
  const int64_t i = blockIdx.x;
  const double tx = x[i], ty = y[i], tz = z[i], te = e[i];
  double sx = 0.0, sy = 0.0, sz = 0.0;
  for (int64_t j = threadIdx.x; j < n; j += 256) {
    const double dx = x[j] - tx, dy = y[j] - ty, dz = z[j] - tz;
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (r2 != 0) {
      double b, db;
      const double r = sqrt(r2);
      spline_b_db(r, 1.0 / r, e[j] + te, b, db);
      const double f = b * m[j];
      sx += dx * f;
      sy += dy * f;
      sz += dz * f;
    }
  }
  sx = pt_wave_sum(sx);
  sy = pt_wave_sum(sy);
  sz = pt_wave_sum(sz);
  const int wave = threadIdx.x / PT_WAVE;
  if ((threadIdx.x & (PT_WAVE - 1)) == 0) {
    red[0][wave] = sx;
    red[1][wave] = sy;
    red[2][wave] = sz;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double r[3] = {0, 0, 0};
    for (int w = 0; w < 256 / PT_WAVE; w++)
      for (int k = 0; k < 3; k++) r[k] += red[k][w];
    ax[i] = r[0];
    ay[i] = r[1];
    az[i] = r[2];
    pot[i] = 0.0;
  }
}

// Exact VJP of the direct sum, one block per particle i:
//   g_i += sum_j K_ij (m_i w_j - m_j w_i),  gm_i += sum_j b_ij (x_i - x_j).w_j.
__global__ void __launch_bounds__(256)
direct_adjoint_kernel(int64_t n, const double* __restrict__ x, const double* __restrict__ y,
                      const double* __restrict__ z, const double* __restrict__ m,
                      const double* __restrict__ e, const double* __restrict__ wx,
                      const double* __restrict__ wy, const double* __restrict__ wz,
                      double* __restrict__ gx, double* __restrict__ gy, double* __restrict__ gz,
                      double* __restrict__ gmass) {
  __shared__ double red[4][256 / PT_WAVE];
  const int64_t i = blockIdx.x;
  const double tx = x[i], ty = y[i], tz = z[i], te = e[i], tm = m[i];
  const double twx = wx[i], twy = wy[i], twz = wz[i];
  double sx = 0.0, sy = 0.0, sz = 0.0, sm = 0.0;
  for (int64_t j = threadIdx.x; j < n; j += 256) {
    const double dx = x[j] - tx, dy = y[j] - ty, dz = z[j] - tz;
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (r2 != 0) {
      const double r = sqrt(r2);
      double b, db;
      spline_b_db(r, 1.0 / r, e[j] + te, b, db);
      const double vx = tm * wx[j] - m[j] * twx;
      const double vy = tm * wy[j] - m[j] * twy;
      const double vz = tm * wz[j] - m[j] * twz;
      const double dv = dx * vx + dy * vy + dz * vz;
      const double f = db / r * dv;
      sx += b * vx + f * dx;
      sy += b * vy + f * dy;
      sz += b * vz + f * dz;
      sm -= b * (dx * wx[j] + dy * wy[j] + dz * wz[j]);
    }
  }
  sx = pt_wave_sum(sx);
  sy = pt_wave_sum(sy);
  sz = pt_wave_sum(sz);
  sm = pt_wave_sum(sm);
  const int wave = threadIdx.x / PT_WAVE;
  if ((threadIdx.x & (PT_WAVE - 1)) == 0) {
    red[0][wave] = sx;
    red[1][wave] = sy;
    red[2][wave] = sz;
    red[3][wave] = sm;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double r[4] = {0, 0, 0, 0};
    for (int w = 0; w < 256 / PT_WAVE; w++)
      for (int k = 0; k < 4; k++) r[k] += red[k][w];
    gx[i] += r[0];
    gy[i] += r[1];
    gz[i] += r[2];
    gmass[i] += r[3];
  }
}

// Reverse of one kick-drift step (v' = v + dt a(x), x' = x + dt v'):
//   w = dt^2 lx' + dt lv'  (cotangent of a(x)),  lv = lv' + dt lx'.
// lx itself becomes lx' + (da/dx)^T w once the VJP has been added.
__global__ void __launch_bounds__(256)
adjoint_w_kernel(int64_t n, double dt, const double* __restrict__ lx,
                 const double* __restrict__ ly, const double* __restrict__ lz,
                 double* __restrict__ lvx, double* __restrict__ lvy, double* __restrict__ lvz,
                 double* __restrict__ wx, double* __restrict__ wy, double* __restrict__ wz) {
  const int64_t i = blockIdx.x * 256ll + threadIdx.x;
  if (i >= n) return;
  const double dt2 = dt * dt;
  wx[i] = dt2 * lx[i] + dt * lvx[i];
  wy[i] = dt2 * ly[i] + dt * lvy[i];
  wz[i] = dt2 * lz[i] + dt * lvz[i];
  lvx[i] += dt * lx[i];
  lvy[i] += dt * ly[i];
  lvz[i] += dt * lz[i];
}

__global__ void __launch_bounds__(256)
gather3_kernel(const uint32_t* __restrict__ perm, int64_t n, const double* __restrict__ a,
               const double* __restrict__ b, const double* __restrict__ c,
               double* __restrict__ as, double* __restrict__ bs, double* __restrict__ cs) {
  const int64_t i = blockIdx.x * 256ll + threadIdx.x;
  if (i >= n) return;
  const uint32_t j = perm[i];
  as[i] = a[j];
  bs[i] = b[j];
  cs[i] = c[j];
}

// out[perm[i]] += in[i] for four arrays (sorted -> caller order).
// n x 3 interleaved <-> three arrays.
__global__ void __launch_bounds__(256)
split3_kernel(int64_t n, const double* __restrict__ v, double* __restrict__ a,
              double* __restrict__ b, double* __restrict__ c) {
  const int64_t i = blockIdx.x * 256ll + threadIdx.x;
  if (i >= n) return;
  a[i] = v[3 * i];
  b[i] = v[3 * i + 1];
  c[i] = v[3 * i + 2];
}

__global__ void __launch_bounds__(256)
join3_kernel(int64_t n, const double* __restrict__ a, const double* __restrict__ b,
             const double* __restrict__ c, double* __restrict__ v) {
  const int64_t i = blockIdx.x * 256ll + threadIdx.x;
  if (i >= n) return;
  v[3 * i] = a[i];
  v[3 * i + 1] = b[i];
  v[3 * i + 2] = c[i];
}

// lam_node = the sum of the private copies, for the hot nodes (len values).
__global__ void __launch_bounds__(256)
hot_reduce_kernel(const double* __restrict__ hot, int64_t len, double* __restrict__ lam_node) {
  const int64_t q = blockIdx.x * 256ll + threadIdx.x;
  if (q >= len) return;
  double v = 0.0;
  for (int p = 0; p < kHotParts; p++) v += hot[p * len + q];
  lam_node[q] = v;
}

inline unsigned grid_for(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

int64_t pt_adjoint_node_scratch(int64_t nn) {
  return (int64_t)kNodeRow * (nn + kHotParts * std::min<int64_t>(nn, kHotNodes));
}

int pt_launch_adjoint_groups(int precision, const Bucket* bk, const int32_t* gfirst,
                             const int32_t* gnb, const uint32_t* ngroups, int64_t ns,
                             const TreeNode* nodes, const GravNode* gn,
                             const GravNode32* gn32, const double* x,
                             const double* y, const double* z, const double* m, const double* e,
                             const int64_t* pp_off, const int32_t* pp, const uint8_t* ppm,
                             const int64_t* pc_off, const int32_t* pc, const uint8_t* pcm,
                             const double off[3], const double* wx, const double* wy,
                             const double* wz, double* gs, double* lam_node, int64_t nn,
                             hipStream_t s) {
  if (ns <= 0) return 0;
  // lam_node holds pt_adjoint_node_scratch(nn) doubles, all zero on entry:
  // the node cotangents, then the private copies of the hot ones
  const int64_t nhot = std::min<int64_t>(nn, kHotNodes);
  double* hot = lam_node + (int64_t)kNodeRow * nn;
  // few groups share their lists among several waves, up to 64k work-groups in
  // all: 64k particles (8k slots), FP32, 1418 us at 1 wave, 1190 at 4, 1155 at
  // 8; 256k (53k slots), FP64, 3720 at 1, 3780 at 2, 4380 at 8
  const int64_t share = std::min<int64_t>(8, std::max<int64_t>(1, 65536 / ns));
  const dim3 grid((unsigned)pt_part_blocks(ns), (unsigned)share);
  if (precision != 0)  // the compensated-FP32 precision
    adjoint_group32_kernel<<<grid, PT_WAVE, 0, s>>>(
        bk, gfirst, gnb, ngroups, nodes, gn32, x, y, z, m, e, pp_off, pp, ppm, pc_off, pc, pcm,
        off[0], off[1], off[2], wx, wy, wz, gs, lam_node, hot, nhot);
  else
    adjoint_group_kernel<<<grid, PT_WAVE, 0, s>>>(
        bk, gfirst, gnb, ngroups, nodes, gn, x, y, z, m, e, pp_off, pp, ppm, pc_off, pc, pcm,
        off[0], off[1], off[2], wx, wy, wz, gs, lam_node, hot, nhot);
  hot_reduce_kernel<<<grid_for(nhot * kNodeRow), 256, 0, s>>>(hot, nhot * kNodeRow, lam_node);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_adjoint_down(int64_t n, const uint32_t* bucket_of, const int32_t* bucket_node,
                           const int32_t* parent, const GravNode* gn,
                           const double* lam_node, const double* gs, const uint32_t* perm,
                           const double* x, const double* y, const double* z, const double* m,
                           const double* e, double* gx, double* gy, double* gz, double* gm,
                           hipStream_t s) {
  if (n <= 0) return 0;
  adjoint_down_kernel<<<grid_for(n), 256, 0, s>>>(n, bucket_of, bucket_node, parent, gn,
                                                  lam_node, gs, perm, x, y, z, m, e, gx, gy, gz,
                                                  gm);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_direct_all(int64_t n, const double* x, const double* y, const double* z,
                         const double* m, const double* e, double* ax, double* ay, double* az,
                         double* pot, hipStream_t s) {
  if (n <= 0) return 0;
  direct_all_kernel<<<(unsigned)n, 256, 0, s>>>(n, x, y, z, m, e, ax, ay, az, pot);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_direct_adjoint(int64_t n, const double* x, const double* y, const double* z,
                             const double* m, const double* e, const double* wx,
                             const double* wy, const double* wz, double* gx, double* gy,
                             double* gz, double* gm, hipStream_t s) {
  if (n <= 0) return 0;
  direct_adjoint_kernel<<<(unsigned)n, 256, 0, s>>>(n, x, y, z, m, e, wx, wy, wz, gx, gy, gz, gm);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_adjoint_w(int64_t n, double dt, const double* lx, const double* ly,
                        const double* lz, double* lvx, double* lvy, double* lvz, double* wx,
                        double* wy, double* wz, hipStream_t s) {
  if (n <= 0) return 0;
  adjoint_w_kernel<<<grid_for(n), 256, 0, s>>>(n, dt, lx, ly, lz, lvx, lvy, lvz, wx, wy, wz);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_gather3(const uint32_t* perm, int64_t n, const double* a, const double* b,
                      const double* c, double* as, double* bs, double* cs, hipStream_t s) {
  if (n <= 0) return 0;
  gather3_kernel<<<grid_for(n), 256, 0, s>>>(perm, n, a, b, c, as, bs, cs);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_split3(int64_t n, const double* v, double* a, double* b, double* c, hipStream_t s) {
  if (n <= 0) return 0;
  split3_kernel<<<grid_for(n), 256, 0, s>>>(n, v, a, b, c);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_join3(int64_t n, const double* a, const double* b, const double* c, double* v,
                    hipStream_t s) {
  if (n <= 0) return 0;
  join3_kernel<<<grid_for(n), 256, 0, s>>>(n, a, b, c, v);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}
