// evp1d_pair_adj.hpp - the gradient's reverse sweep in the pair form: two
// subcycles of a tile per workgroup.
//
// The reverse of a subcycle reads its neighbours as the forward does: the
// stress adjoint of a T point takes g (the adjoint of the str sums) and the
// velocities of the points cc, ee, ne, se, and the stepu adjoint of a U point
// the contributions of the T points q, nw(q), sse(q), sw(q).  So the reverse
// of [stress, stepu] pairs runs on the forward's tiles and tables (PairPlan),
// with g in place of the velocities that change and the stress adjoints'
// four velocity contributions in place of str1..8.
#pragma once

#include <hip/hip_runtime.h>

#include "evp1d_adjoint.hpp"
#include "evp1d_pair.hpp"

// One launch, entered after the stepu adjoint of subcycle k: the stress
// adjoint of k, the stepu adjoint of k - 1 (level 1), the stress adjoint of
// k - 1 and the stepu adjoint of k - 2 (level 2).  Every value is what
// k_stress_adj and k_stepu_adj compute, in the same order of additions.  The
// adjoint stresses, ub and g are read by neighbouring tiles, so each has two
// buffers; the accumulators belong to one tile each.
//
// What bounds it: bytes first, then the latency of the phases.  At 1280x1520
// (31x19, 512 threads) a launch moves 890 MB at 4.7 TB/s (190 us for two
// subcycles; streaming reaches 5.5 TB/s), where k_stepu_adj and k_stress_adj
// move 1612 MB in 260 us: the adjoint stresses, ub, g and the accumulators go
// through memory once per two subcycles, the velocity contributions never.
// The launch bounds of k_pair (128 VGPRs, two 512-thread workgroups per CU)
// hold because stress_adjoint is fenced (122 spilled registers without, 223
// us with 11, 193 with 8); the tables of a 31x19 tile are at most 81 136 of
// the 81 920 bytes of LDS that two workgroups per CU leave each.  Keeping the
// U points' level-1 sums for level 2 in registers saves a pass over the three
// accumulators (225 -> 205 us); the strength sum the same way beats reading
// and writing its accumulator at both levels (190 against 200 us).
struct PairAdjBufs {
  const double2 *sg_in, *ub_in, *g_in;   // [6][ls] pairs; by slot; by slot (zero off the stepu range)
  double2 *sg_out, *ub_out, *g_out;
  // velocities of the states k - 1, k - 2 and k - 3, by slot - u_begin
  const double2 *xa, *xb, *xc;
  const double2 *velc;                   // by slot: the velocities that never change
  int nu;
  double *gstr, *gcw, *gfx, *gfy;
  evp1d::AdjScalars as;
};

template <int B, bool NT>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(4))) void k_pair_adj(PairView f, PairAdjBufs bf,
                                                                                      int capv) {
  extern __shared__ double2 lds[];
  const int cap = f.cap;
  double2 *gt = lds + 4 * cap, *vt = gt + capv, *ubt = vt + capv;
  const evp1d::PairTile pt = f.tiles[tile_of(blockIdx.x, gridDim.x, f.xcd != 0)];
  const evp1d::TileDesc &t = pt.t;
  const int nA = t.a1 - t.a0, nB = t.b1 - t.b0, nO = nA + nB, nS = nO + t.nh, nT = nS + pt.nx, nE = nT + pt.nq;
  const int nUo = nB + (t.c1 - t.c0), nU = nUo + pt.ne;
  const double2 *pc = f.pc;
  const long lp = f.lp;
  const int me = threadIdx.x;
  auto uslot = [&](int k) { return k < nB ? t.b0 + k : k < nUo ? t.c0 + (k - nB) : f.elist[pt.e0 + (k - nUo)]; };
  auto vel = [&](int j) {
    const unsigned u = (unsigned)(j - f.u_begin);
    return *(u < (unsigned)bf.nu ? bf.xa + u : bf.velc + j);
  };
  auto put = [&](int k, const double *vb) {   // read back as cc, ee, se, ne of a U point's T neighbours
    lds[k] = make_double2(vb[0], vb[1]);
    lds[cap + k] = make_double2(vb[2], vb[3]);
    lds[2 * cap + k] = make_double2(vb[4], vb[5]);
    lds[3 * cap + k] = make_double2(vb[6], vb[7]);
  };
  double sb[12];       // adjoint stresses of entry `me` (me < nS)
  double gs = 0.0;     // d/d strength of entry `me`, level 1
  auto level1 = [&](int k) {
    if (k < nT) {
      const int4 n = f.tnbr[pt.n0 + k];
      const int g = n.x;
      double s[12];
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        const double2 v = in2<NT>(bf.sg_in + (c * f.ls + g));
        s[2 * c] = v.x;
        s[2 * c + 1] = v.y;
      }
      const double2 m0 = pc[g], m1 = pc[lp + g], m2 = pc[2 * lp + g];
      const double2 cc = vel(g), ve = vel(n.y), vn = vel(n.z), vs = vel(n.w);
      const double2 g0 = bf.g_in[g], ge = bf.g_in[n.y], gn = bf.g_in[n.z], gx = bf.g_in[n.w];
      const double str_b[8] = {g0.x, ge.x, gx.x, gn.x, g0.y, gx.y, ge.y, gn.y};
      double vb[8];
      const double b = evp1d::stress_adjoint(bf.as, cc.x, cc.y, ve.x, ve.y, vs.x, vs.y, vn.x, vn.y, m0.x, m0.y,
                                             f.strength[g], m1.x, m1.y, m2.x, m2.y, s, str_b, vb);
      if (k == me) {
        gs = b;
#pragma unroll
        for (int c = 0; c < 12; ++c) sb[c] = s[c];
      }
      put(k, vb);
    } else {
      const double zero[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      put(k, zero);
    }
  };
  for (int k = me + B; k < nE; k += B) level1(k);
  if (me < nE) level1(me);
  // memory inputs of one stepu adjoint
  struct UIn {
    uint2 w;
    double2 c[5];
    double2 v;
  };
  auto uload = [&](int k, int q, const double2 *x) {
    UIn u;
    u.w = f.uloc[pt.u0 + k];
    u.c[0] = pc[3 * lp + q];
    u.c[1] = pc[4 * lp + q];
    u.c[2] = pc[5 * lp + q];
    u.c[3] = pc[7 * lp + q];
    u.c[4] = pc[8 * lp + q];
    u.v = x[q - f.u_begin];
    return u;
  };
  // ub: the stored part of the velocity adjoint; vn: the update's result
  auto stepu = [&](const UIn &u, double2 ub, double2 vn, evp1d::StepuAdj &o) {
    const double2 a = lds[u.w.x & 0xffffu];
    const double2 b = lds[cap + (u.w.x >> 16)];
    const double2 c = lds[2 * cap + (u.w.y & 0xffffu)];
    const double2 e = lds[3 * cap + (u.w.y >> 16)];
    ub.x += a.x; ub.y += a.y;
    ub.x += b.x; ub.y += b.y;
    ub.x += e.x; ub.y += e.y;
    ub.x += c.x; ub.y += c.y;
    evp1d::stepu_adjoint(bf.as.s, u.v.x, u.v.y, u.c[0].x, u.c[0].y, u.c[1].x, u.c[1].y, u.c[2].x, u.c[2].y, u.c[3].x,
                         u.c[3].y, u.c[4].x, u.c[4].y, vn.x, vn.y, ub.x, ub.y, o);
  };
  struct Acc {
    double fx, fy, cw;
  };
  auto accs = [&](int q) { return Acc{in1<NT>(bf.gfx + q), in1<NT>(bf.gfy + q), in1<NT>(bf.gcw + q)}; };
  auto store = [&](int q, const Acc &a) {
    out1<NT>(bf.gfx + q, a.fx);
    out1<NT>(bf.gfy + q, a.fy);
    out1<NT>(bf.gcw + q, a.cw);
  };
  auto plus = [](Acc a, const evp1d::StepuAdj &o) { return Acc{a.fx + o.fx_b, a.fy + o.fy_b, a.cw + o.cw_b}; };
  auto level1u = [&](int k, const UIn &u, double2 ub, double2 vn, evp1d::StepuAdj &o) {
    stepu(u, ub, vn, o);
    gt[k] = make_double2(o.gx, o.gy);
    vt[k] = u.v;
    if (k < nUo) ubt[k] = make_double2(o.uold_b, o.vold_b);
  };
  int q1 = 0;
  UIn u1;
  double2 b1, n1;
  Acc a1{0.0, 0.0, 0.0};
  if (me < nU) {
    q1 = uslot(me);
    u1 = uload(me, q1, bf.xb);
    b1 = bf.ub_in[q1];
    n1 = bf.xa[q1 - f.u_begin];
    if (me < nUo) a1 = accs(q1);
  }
  __syncthreads();
  if (me < nU) {
    evp1d::StepuAdj o;
    level1u(me, u1, b1, n1, o);
    a1 = plus(a1, o);
  }
  for (int k = me + B; k < nU; k += B) {
    const int q = uslot(k);
    Acc a{0.0, 0.0, 0.0};
    if (k < nUo) a = accs(q);
    evp1d::StepuAdj o;
    level1u(k, uload(k, q, bf.xb), bf.ub_in[q], bf.xa[q - f.u_begin], o);
    if (k < nUo) store(q, plus(a, o));
  }
  // level 2, stress adjoint of entry me (velocities that are no U1 entry
  // never change, and g is zero there)
  constexpr unsigned kFix = evp1d::PairPlan::kFixBase;
  int g2 = 0;
  uint2 w2 = make_uint2(0u, 0u);
  double2 c2[4], m0, m1, m2;
  double st = 0.0;
  if (me < nS) {
    const int4 n = f.tnbr[pt.n0 + me];
    g2 = n.x;
    w2 = f.vloc[pt.v0 + me];
    const unsigned e[4] = {w2.x & 0xffffu, w2.x >> 16, w2.y & 0xffffu, w2.y >> 16};
    const int ns[4] = {g2, n.y, n.z, n.w};
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (e[c] >= kFix) c2[c] = bf.velc[ns[c]];
    m0 = pc[g2];
    m1 = pc[lp + g2];
    m2 = pc[2 * lp + g2];
    st = f.strength[g2];
    if (me < nO) gs = in1<NT>(bf.gstr + g2) + gs;
  }
  __syncthreads();
  if (me < nS) {
    const unsigned e[4] = {w2.x & 0xffffu, w2.x >> 16, w2.y & 0xffffu, w2.y >> 16};
    double2 v[4], g[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) g[c] = e[c] >= kFix ? make_double2(0.0, 0.0) : gt[e[c]];
    const double str_b[8] = {g[0].x, g[1].x, g[3].x, g[2].x, g[0].y, g[3].y, g[1].y, g[2].y};
    evp1d::stress_adjoint_sums(m0.x, m0.y, m1.x, m1.y, m2.x, m2.y, str_b, sb);
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = e[c] >= kFix ? c2[c] : vt[e[c]];
    double vb[8];
    const double b =
        evp1d::stress_adjoint_corners(bf.as, v[0].x, v[0].y, v[1].x, v[1].y, v[3].x, v[3].y, v[2].x, v[2].y, m0.x,
                                      m0.y, st, m1.x, m1.y, m2.x, m2.y, sb, vb);
    if (me < nO) {
#pragma unroll
      for (int c = 0; c < 6; ++c) out2<NT>(bf.sg_out + (c * f.ls + g2), make_double2(sb[2 * c], sb[2 * c + 1]));
      out1<NT>(bf.gstr + g2, gs + b);
    }
    put(me, vb);
  }
  // level 2, stepu adjoint of the owned U points
  auto level2u = [&](int k, int q, const UIn &u, const Acc &a) {
    evp1d::StepuAdj o;
    stepu(u, ubt[k], vt[k], o);
    out2<NT>(bf.ub_out + q, make_double2(o.uold_b, o.vold_b));
    out2<NT>(bf.g_out + q, make_double2(o.gx, o.gy));
    store(q, plus(a, o));
  };
  int q2 = 0;
  UIn u2;
  if (me < nUo) {
    q2 = uslot(me);
    u2 = uload(me, q2, bf.xc);
  }
  __syncthreads();
  if (me < nUo) level2u(me, q2, u2, a1);
  for (int k = me + B; k < nUo; k += B) {
    const int q = uslot(k);
    level2u(k, q, uload(k, q, bf.xc), accs(q));
  }
}

// LDS of a reverse launch: the contributions' table, then g, velocity and
// velocity adjoint of the velocity entries
inline size_t pair_adj_lds(int cap, int capv) { return (size_t)(4 * cap + 3 * capv) * sizeof(double2); }
