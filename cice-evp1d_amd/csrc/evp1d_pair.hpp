// evp1d_pair.hpp - the pair form: two subcycles of a tile per workgroup.
//
// Included by the 1D list's and the 2D block path's device files, which
// instantiate the kernel for their own constants and outputs.
#pragma once

#include <hip/hip_runtime.h>

#include "evp1d_cache.hpp"
#include "evp1d_point.hpp"
#include "evp1d_tiles.hpp"
#include "evp1d_xcd.hpp"

// Level 1 runs stress on the tile's T1 entries (owned, halo, T1-only) from the
// input state (PairBufs), then stepu on its U1 entries into an LDS
// velocity table; level 2 runs stress on the owned and halo entries from
// those velocities and the level-1 stresses, then stepu on the owned U
// points, and writes the state two subcycles on to vel_out / sig_out (two
// buffers each).  Every point computes exactly what the one-subcycle kernels
// compute, so results are bit-identical; neighbour tiles evaluate the border
// rings again instead of exchanging them, which halves the loads and stores
// of the state and the constant fields per subcycle.  Level-2 stress entry k
// is thread k (the plan guarantees at most B of them), so its level-1
// stresses stay in that thread's registers.  The constant fields come
// from a copy packed in pairs at the start of the run, the
// stresses live during the run in pairs too: one
// 16-byte load per pair, since the kernel's time follows its load
// instructions.  Each level-1 stress entry's slot and ee, ne, se neighbour
// slots come from one per-tile int4 (PairPlan::tnbr), so a halo or T1-only
// entry reaches its velocities after two dependent loads, not three.
//
// The kernel serves both the 1D list (V0 = false) and the 2D block path
// (V0 = true), which differ in the metric terms they are given and in the
// arrays that the last launch of a run writes:
//   V0 = false: stress constants (dxT, dyT), (hte, htn), (htem1, htnm1) and
//     strength; str1..8, strintx, strinty and Cb by slot
//   V0 = true: stress constants (dxt, dyt), (strength, dmin), (cxp, cyp),
//     (cxm, cym), (dxhy, dyhx); str1..8, strintx, strinty, taubx and tauby by
//     the slot's cell of the block arrays
template <bool V0>
constexpr int kPairT = V0 ? 5 : 3;   // stress pairs; stepu's seven follow
constexpr int kPairU = 7;
struct PairView {
  const evp1d::PairTile *tiles;
  const int32_t *hlist, *xlist, *elist;
  const uint2 *uloc;        // per U1 entry: own | nw << 16, sse | sw << 16 (str table entries)
  const uint2 *vloc;        // per T2 entry: cc | ee << 16, ne | se << 16 (velocity table entries)
  const double2 *cstr;      // [4][nk]: s15, s27, s36, s48 of the constant entries
  const int *cnz;           // nonzero when some constant entry has a bit set (else all are +0.0)
  long nk;
  int cap;                  // entries of the str table (the velocity table follows it)
  int xcd;                  // XCD-aware tile order
  const double2 *pc;        // [kPairT + kPairU][lp]: the constant fields in pairs
  long lp;
  const double *strength;   // V0 = false: by slot
  long ls;                  // stresses: [6][ls] pairs (p1 p2, p3 p4, m1 m2, m3 m4, 12_1 12_2, 12_3 12_4)
  const int4 *tnbr;         // per level-1 stress entry (PairTile::n0 + k): slot, ee, ne, se (PairPlan::tnbr, tsrc)
  const int32_t *fix;       // fixed copy-list sources of level-2 ghost reads (PairPlan::fix)
  // gradient trajectory (k_pair<.., TRAJ>): the velocities of the stepu
  // slots after the launch's first subcycle (tr_mid) and after its second
  // (tr_end, null when the handle's own buffer is the only copy wanted),
  // indexed by slot - u_begin
  double2 *tr_mid, *tr_end;
  int u_begin;
  // written by the last launch of a run; cb is taubx for V0
  double2 *s15, *s27, *s36, *s48;
  double *strintx, *strinty, *cb, *tauby;
  const int32_t *cell;      // V0: slot -> cell of those arrays
  evp1d::Scalars s;
};

// the buffers that alternate between launches: input velocities and
// stresses, output velocities and stresses
struct PairBufs {
  const double2 *vel;
  double2 *vel_out;
  const double2 *sg_in;
  double2 *sg_out;
};

// At most 128 VGPRs (4 waves per SIMD): workgroups of 256, 512 or 1024
// threads then fill 16 waves per CU.  TRAJ: the gradient's forward sweep,
// which also stores both subcycles' stepu-slot velocities (f.tr_mid,
// f.tr_end); the values computed are the same.
//
// Each barrier waits for LDS only, so global loads issued before it stay in
// flight across it: every thread loads the memory inputs of its first entry
// of the next phase (level-1 stepu, level-2 stress, level-2 stepu) before
// the barrier that ends the current phase, and that phase starts on values
// already in registers instead of one memory round trip after the barrier.
//
// NT: the cache hints (evp1d_cache.hpp).  The streams a launch reads or
// writes once (stresses in and out, the T points' constant fields,
// velocities and trajectory written) become non-temporal loads and stores,
// so that the cache can keep what every launch reads again (the U points'
// constant fields, velocities, tables).
template <int B, bool V0, bool TRAJ, bool FIX, bool NT>
__device__ __forceinline__ void pair_tile(const PairView &f, PairBufs bf, int last, int tix) {
  extern __shared__ double2 lds[];
  const int cap = f.cap;
  double2 *vt = lds + 4 * cap;
  const evp1d::PairTile pt = f.tiles[tix];
  const evp1d::TileDesc &t = pt.t;
  const int nA = t.a1 - t.a0, nB = t.b1 - t.b0, nO = nA + nB, nS = nO + t.nh, nT = nS + pt.nx, nE = nT + pt.nq;
  const int nUo = nB + (t.c1 - t.c0), nU = nUo + pt.ne;
  const bool cz = *f.cnz == 0;
  auto tslot = [&](int k) {
    return k < nA ? t.a0 + k : k < nO ? t.b0 + (k - nA) : k < nS ? f.hlist[t.h0 + (k - nO)] : f.xlist[pt.x0 + (k - nS)];
  };
  auto uslot = [&](int k) { return k < nB ? t.b0 + k : k < nUo ? t.c0 + (k - nB) : f.elist[pt.e0 + (k - nUo)]; };
  auto put = [&](int k, const evp1d::StressOut &o) {
    lds[k] = make_double2(o.str[0], o.str[4]);
    lds[cap + k] = make_double2(o.str[1], o.str[6]);
    lds[2 * cap + k] = make_double2(o.str[2], o.str[5]);
    lds[3 * cap + k] = make_double2(o.str[3], o.str[7]);
  };
  const double2 *pc = f.pc;
  const long lp = f.lp;
  // memory inputs of one stepu evaluation: its str table entries and the
  // seven packed constant pairs of slot q
  struct UIn {
    uint2 w;
    double2 c[kPairU];
  };
  auto uload = [&](int k, int q) {
    UIn u;
    u.w = f.uloc[pt.u0 + k];
#pragma unroll
    for (int c = 0; c < kPairU; ++c) u.c[c] = pc[(kPairT<V0> + c) * lp + q];
    return u;
  };
  auto stepu = [&](const UIn &u, double2 v, evp1d::StepuOut &o) {
    const double2 a = lds[u.w.x & 0xffffu];
    const double2 b = lds[cap + (u.w.x >> 16)];
    const double2 c = lds[2 * cap + (u.w.y & 0xffffu)];
    const double2 e = lds[3 * cap + (u.w.y >> 16)];
    const double2 *k = u.c;
    evp1d::stepu_point(f.s, v.x, v.y, k[0].x, k[0].y, k[1].x, k[1].y, k[2].x, k[2].y, k[3].x, k[3].y, k[4].x,
                       k[4].y, k[5].x, k[6].x, k[6].y, k[5].y, a.x, b.x, c.x, e.x, a.y, c.y, b.y, e.y, o);
  };
  const int me = threadIdx.x;
  double sg[12];   // level-1 stresses of entry `me` when me < nS
  // entry `me`'s metric pairs and strength, loaded at level 1 and used again
  // at level 2 (the same slot)
  double2 m2[kPairT<V0>];
  double st2 = 0.0;
  auto stress = [&](double2 cc, double2 ve, double2 vn, double2 vs, const double2 *m, double st, const double *sig,
                    evp1d::StressOut &o) {
    if constexpr (V0)
      evp1d::stress_core(f.s, cc.x, cc.y, ve.x, ve.y, vs.x, vs.y, vn.x, vn.y, m[0].x, m[0].y, m[1].x, m[2].x, m[2].y,
                         m[3].x, m[3].y, m[1].y, m[4].x, m[4].y, sig, o);
    else
      evp1d::stress_point(f.s, cc.x, cc.y, ve.x, ve.y, vs.x, vs.y, vn.x, vn.y, m[0].x, m[0].y, st, m[1].x, m[1].y,
                          m[2].x, m[2].y, sig, o);
  };
  // level 1, stress (or constants) of entry k
  auto level1 = [&](int k) {
    if (k < nT) {
      // slot (FIX: the slot of its velocity) and ee, ne, se of the entry
      const int4 n = f.tnbr[pt.n0 + k];
      const int g = k < nO || FIX ? tslot(k) : n.x;
      double sig[12];
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        const double2 v = in2<NT>(bf.sg_in + (c * f.ls + g));
        sig[2 * c] = v.x;
        sig[2 * c + 1] = v.y;
      }
      // (V0's loop here and the scalars at the head of PairView give another
      // schedule: 61.3 in place of 60.8 us per subcycle at 1280x1520)
      double2 m[kPairT<V0>];
      if constexpr (V0) {
#pragma unroll
        for (int c = 0; c < kPairT<V0>; ++c) m[c] = in2<NT>(pc + (c * lp + g));
      } else {
        m[0] = in2<NT>(pc + g);
        m[1] = in2<NT>(pc + (lp + g));
        m[2] = in2<NT>(pc + (2 * lp + g));
      }
      const double st = V0 ? 0.0 : in1<NT>(f.strength + g);
      evp1d::StressOut o;
      const double2 cc = bf.vel[FIX ? n.x : g], ve = bf.vel[n.y], vn = bf.vel[n.z], vs = bf.vel[n.w];
      stress(cc, ve, vn, vs, m, st, sig, o);
      if (k == me) {
#pragma unroll
        for (int c = 0; c < kPairT<V0>; ++c) m2[c] = m[c];
        st2 = st;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          sg[c] = o.sp[c];
          sg[4 + c] = o.sm[c];
          sg[8 + c] = o.s12[c];
        }
      }
      put(k, o);
    } else {
      double2 p15, p27, p36, p48;
      if (cz) {
        p15 = p27 = p36 = p48 = make_double2(0.0, 0.0);
      } else {
        const long j = pt.q0 + (k - nT);
        p15 = f.cstr[j];
        p27 = f.cstr[f.nk + j];
        p36 = f.cstr[2 * f.nk + j];
        p48 = f.cstr[3 * f.nk + j];
      }
      lds[k] = p15;
      lds[cap + k] = p27;
      lds[2 * cap + k] = p36;
      lds[3 * cap + k] = p48;
    }
  };
  // entries me + B, me + 2B, ... first and entry me (kept for level 2) last,
  // so no other evaluation overlaps the lifetime of its stresses
  for (int k = me + B; k < nE; k += B) level1(k);
  if (me < nE) level1(me);
  // level 1, stepu, entry me: inputs loaded before the barrier
  int q1 = 0;
  UIn u1;
  double2 v1;
  if (me < nU) {
    q1 = uslot(me);
    u1 = uload(me, q1);
    v1 = bf.vel[q1];
  }
  __syncthreads();
  // level 1, stepu: every U1 entry into the velocity table
  if (me < nU) {
    evp1d::StepuOut o;
    stepu(u1, v1, o);
    vt[me] = make_double2(o.uvel, o.vvel);
    if (TRAJ && me < nUo) out2<NT>(f.tr_mid + (q1 - f.u_begin), vt[me]);
  }
  for (int k = me + B; k < nU; k += B) {
    const int q = uslot(k);
    const UIn u = uload(k, q);
    evp1d::StepuOut o;
    stepu(u, bf.vel[q], o);
    vt[k] = make_double2(o.uvel, o.vvel);
    if (TRAJ && k < nUo) out2<NT>(f.tr_mid + (q - f.u_begin), vt[k]);
  }
  // level 2, stress of entry me: memory inputs loaded before the barrier
  // (velocities that are no U1 entry never change, kNoEntry: from memory;
  // a ghost on the copy list whose source is no U1 entry: kFixBase + j, the
  // source's unchanging velocity or zero)
  constexpr unsigned kNo = evp1d::PairPlan::kNoEntry, kFix = evp1d::PairPlan::kFixBase;
  int g2 = 0;
  uint2 w2 = make_uint2(0u, 0u);
  double2 c2[4];
  if (me < nS) {
    const int4 n = f.tnbr[pt.n0 + me];
    g2 = me < nO || FIX ? tslot(me) : n.x;
    w2 = f.vloc[pt.v0 + me];
    c2[0] = bf.vel[g2];
    if (!FIX) {   // no copy list: every entry is a table entry or kNoEntry
      if ((w2.x >> 16) == kNo || (w2.y & 0xffffu) == kNo || (w2.y >> 16) == kNo) {
        c2[1] = bf.vel[n.y];
        c2[2] = bf.vel[n.z];
        c2[3] = bf.vel[n.w];
      }
    } else {
      const unsigned e[4] = {w2.x & 0xffffu, w2.x >> 16, w2.y & 0xffffu, w2.y >> 16};
      const int ns[4] = {g2, n.y, n.z, n.w};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (e[c] == kNo) {
          c2[c] = bf.vel[ns[c]];
        } else if (e[c] >= kFix) {
          const int s = f.fix[pt.f0 + (int)(e[c] - kFix)];
          c2[c] = s < 0 ? make_double2(0.0, 0.0) : bf.vel[s];
        }
      }
    }
  }
  __syncthreads();
  // level 2, stress: owned and halo entries, one per thread
  if (me < nS) {
    const unsigned e0 = w2.x & 0xffffu, e1 = w2.x >> 16, e2 = w2.y & 0xffffu, e3 = w2.y >> 16;
    const double2 cc = e0 >= kFix ? c2[0] : vt[e0];
    const double2 ve = e1 >= kFix ? c2[1] : vt[e1];
    const double2 vn = e2 >= kFix ? c2[2] : vt[e2];
    const double2 vs = e3 >= kFix ? c2[3] : vt[e3];
    evp1d::StressOut o;
    stress(cc, ve, vn, vs, m2, st2, sg, o);
    const int g = g2;
    if (me < nO) {
      out2<NT>(bf.sg_out + g, make_double2(o.sp[0], o.sp[1]));
      out2<NT>(bf.sg_out + (f.ls + g), make_double2(o.sp[2], o.sp[3]));
      out2<NT>(bf.sg_out + (2 * f.ls + g), make_double2(o.sm[0], o.sm[1]));
      out2<NT>(bf.sg_out + (3 * f.ls + g), make_double2(o.sm[2], o.sm[3]));
      out2<NT>(bf.sg_out + (4 * f.ls + g), make_double2(o.s12[0], o.s12[1]));
      out2<NT>(bf.sg_out + (5 * f.ls + g), make_double2(o.s12[2], o.s12[3]));
      if (last) {
        const int c = V0 ? f.cell[g] : g;
        out2<NT>(f.s15 + c, make_double2(o.str[0], o.str[4]));
        out2<NT>(f.s27 + c, make_double2(o.str[1], o.str[6]));
        out2<NT>(f.s36 + c, make_double2(o.str[2], o.str[5]));
        out2<NT>(f.s48 + c, make_double2(o.str[3], o.str[7]));
      }
    }
    put(me, o);
  }
  // level 2, stepu of entry me: inputs loaded before the barrier
  int q2 = 0;
  UIn u2;
  if (me < nUo) {
    q2 = uslot(me);
    u2 = uload(me, q2);
  }
  __syncthreads();
  // level 2, stepu: the owned U points
  auto level2u = [&](int k, int q, const UIn &u) {
    evp1d::StepuOut o;
    stepu(u, vt[k], o);
    out2<NT>(bf.vel_out + q, make_double2(o.uvel, o.vvel));
    if (TRAJ && f.tr_end) out2<NT>(f.tr_end + (q - f.u_begin), make_double2(o.uvel, o.vvel));
    if (last) {
      const int c = V0 ? f.cell[q] : q;
      out1<NT>(f.strintx + c, o.strintx);
      out1<NT>(f.strinty + c, o.strinty);
      out1<NT>(f.cb + c, V0 ? -(o.uvel * o.Cb) : o.Cb);
      if (V0) out1<NT>(f.tauby + c, -(o.vvel * o.Cb));
    }
  };
  if (me < nUo) level2u(me, q2, u2);
  for (int k = me + B; k < nUo; k += B) {
    const int q = uslot(k);
    level2u(k, q, uload(k, q));
  }
}

template <int B, bool V0, bool TRAJ = false, bool FIX = false, bool NT = false>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(4))) void k_pair(PairView f, PairBufs bf, int last) {
  pair_tile<B, V0, TRAJ, FIX, NT>(f, bf, last, tile_of(blockIdx.x, gridDim.x, f.xcd != 0));
}

// block sizes (one level-2 stress per thread) and LDS limit of the pair form
constexpr int kNumPairBlocks = 3;
constexpr int kPairBlocks[kNumPairBlocks] = {256, 512, 1024};
constexpr int kPairMaxLds = 160 * 1024;
// LDS of a pair launch: str table and velocity table
inline size_t pair_lds(int cap, int capv) { return (size_t)(4 * cap + capv) * sizeof(double2); }
inline int pair_block_index(int b) {
  for (int i = 0; i < kNumPairBlocks; ++i)
    if (kPairBlocks[i] == b) return i;
  return -1;
}
