// rk_step.hip -- the per-step kernels of the velocity-Verlet DEM step on
// CDNA4 (gfx950), FP64 throughout, no floating-point atomics.
//
//   k_predict   Rockable::velocityVerletStep predictor (Rockable.cpp:1979-2055)
//               + ServoFunction (DrivingSystem.cpp:242-268) and
//               velocityControlledDrive (Rockable.cpp:1856-1900)
//   k_geom      update_interactions (Rockable.cpp:2968-2974 ->
//               Interaction.cpp:147-326) fused with build_activeInteractions
//               (3005-3029): contact geometry of every listed entry; the
//               active ones go to a compact list
//   k_law       ForceLaw::computeInteraction (3035-3046, ForceLaw_*.cpp) on
//               the active list; writes each active entry's terms for body i
//               and body j (incrementResultants, 2752-2789) into the two
//               resultant slots of the entry
//   k_gather    initialise_particle_forces_and_moments (2869-2929) +
//               compute_resultants (3267-3272) as a per-body ordered sum over
//               the body's slots, which hold its incident entries in the
//               serial order of the reference, + compute_accelerations_from_
//               resultants (3419-3552) + the closing kick (2120-2155)
//   k_gather_heavy  the same for bodies with many slots, one workgroup each
//   k_guard_check  the end of a guarded step: the displacement check, and the
//               freeze after a bond was marked
//   k_breakage  breakage_of_interfaces (3350-3413), once the host knows of a
//               marked bond (every step without the guard)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <mutex>

#include "rk_device.hpp"
#include "rk_model.hpp"

namespace rk {

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ v3 kpos(const BodyKin& b) { return V(b.px, b.py, b.pz); }
__device__ __forceinline__ v3 kvel(const BodyKin& b) { return V(b.vx, b.vy, b.vz); }
__device__ __forceinline__ v3 kvrot(const BodyKin& b) { return V(b.wx, b.wy, b.wz); }
__device__ __forceinline__ qt kq(const BodyKin& b) {
  qt q;
  q.w = b.qw;
  q.x = b.qx;
  q.y = b.qy;
  q.z = b.qz;
  return q;
}
__device__ __forceinline__ v3 ld3(const double* p) { return V(p[0], p[1], p[2]); }
__device__ __forceinline__ void st3(double* p, v3 v) {
  p[0] = v.x;
  p[1] = v.y;
  p[2] = v.z;
}

// A rebuild found due by the device guard suspends the step kernels until
// the host has rebuilt the list (every thread reads the same flag).
__device__ __forceinline__ bool frozen(const Dev& d) {
  return d.guard_on && *(volatile const int*)&d.guard->frozen;
}

// Particle::GlobVertex (Particle.cpp:55-57): pos + Q * (homothety * vertex)
__device__ __forceinline__ v3 glob_vertex(const DevShapes& sh, const BodyKin& b, int v) {
  const double* p = sh.vtx + 3 * (sh.voff[b.shape] + v);
  v3 hv = vsc(b.h, V(p[0], p[1], p[2]));
  return vadd(kpos(b), qrot(kq(b), hv));
}

// v(Qj) - v(Qi) (Interaction.cpp:162)
__device__ __forceinline__ v3 rel_vel(v3 pos, const BodyKin& Pi, const BodyKin& Pj) {
  v3 a = vsub(kvel(Pj), vcross(vsub(pos, kpos(Pj)), kvrot(Pj)));
  v3 b = vsub(kvel(Pi), vcross(vsub(pos, kpos(Pi)), kvrot(Pi)));
  return vsub(a, b);
}

__device__ __forceinline__ double prm(const DevParams& p, int id, int g1, int g2) {
  if (g1 < 0 || g2 < 0 || g1 >= p.G || g2 >= p.G) return 0.0;
  return p.tab[(id * p.G + g1) * p.G + g2];
}

// The contact parameters of a pair of groups.
struct ContactPar {
  double kn, kt, mu, kr, mur, en2;
};
__device__ __forceinline__ int group_pair(const DevParams& p, int g1, int g2) {
  return (g1 < 0 || g2 < 0 || g1 >= p.G || g2 >= p.G) ? -1 : g1 * p.G + g2;
}
template <int LAW>
__device__ __forceinline__ ContactPar contact_par(const DevParams& p, int gpair) {
  ContactPar c;
  const int n = p.G * p.G;
  const double* t = p.tab + (gpair < 0 ? 0 : gpair);
  c.kn = t[P_KN * n];
  c.kt = t[P_KT * n];
  c.mu = t[P_MU * n];
  c.kr = t[P_KR * n];
  c.mur = t[P_MUR * n];
  c.en2 = LAW == LAW_AVALANCHE ? t[P_EN2 * n] : 0.0;
  if (gpair < 0) c.kn = c.kt = c.mu = c.kr = c.mur = c.en2 = 0.0;
  return c;
}

struct Kin {
  v3 n, pos, vel;
  double dn, prev_dn;
  bool deact;
};

// The global vertices of a body, computed once per step by k_glob.
__device__ __forceinline__ v3 gvtx(const double* g, int v) { return V(g[3 * v], g[3 * v + 1], g[3 * v + 2]); }

// even-odd crossing test of P against a face (Interaction.cpp:236-253), one
// of its edges: toggles odd
__device__ __forceinline__ void cross_edge(v3 A, v3 B, v3 v1, v3 v2, double ori1, double ori2, int& odd) {
  double pa1 = vdot(A, v1), pb1 = vdot(B, v1);
  double pa2 = vdot(A, v2), pb2 = vdot(B, v2);
  if ((pa2 < ori2 && pb2 >= ori2) || (pb2 < ori2 && pa2 >= ori2)) {
    if (pa1 + (ori2 - pa2) / (pb2 - pa2) * (pb1 - pa1) < ori1) odd = 1 - odd;
  }
}

// Per entry, the global-vertex indices (and face range) its contact geometry
// reads, resolved once per list change rather than through the bodies'
// shapes at every step (which costs a chain of dependent loads):
//   VV (vi, vj, -, -); VE (vi, j's edge ends); EE (i's edge ends, j's edge
//   ends); VF (vi, start of j's face in sh.fidx, its vertex count, bvoff[j]).
// edesc_s: the same with the indices of the shapes' vertex table (and j's
// first vertex there for bvoff[j]).
__device__ __forceinline__ void reset_list(const Dev& d) {
  for (int k = 0; k < 8; k++) d.ls->cnt[0][k] = d.ls->cnt[1][k] = 0;
  d.ls->gen = 0;
  d.ls->want[0] = d.ls->want[1] = 1;
  d.ls->again = 1;
}
__global__ void __launch_bounds__(kBlock) k_entry_desc(Dev d) {
  if (blockIdx.x == 0) {
    // a new list: the evaluation list starts anew, and the motion bounds'
    // frame takes the mean velocity of up to 2048 free bodies spread over all
    // (any frame is valid; a mean that is not finite is none)
    __shared__ double red[3][kBlock];
    const int t = threadIdx.x, nfree = d.nb - d.nDriven, n = min(nfree, 2048);
    v3 u = V(0.0, 0.0, 0.0);
    for (int k = t; k < n; k += kBlock) u = vadd(u, kvel(d.kin[d.nDriven + (int)((long)k * nfree / n)]));
    red[0][t] = u.x;
    red[1][t] = u.y;
    red[2][t] = u.z;
    for (int h = kBlock / 2; h > 0; h >>= 1) {
      __syncthreads();
      if (t < h)
        for (int k = 0; k < 3; k++) red[k][t] += red[k][t + h];
    }
    if (t == 0) {
      reset_list(d);
      for (int k = 0; k < 3; k++) {
        const double m = n > 0 ? red[k][0] / n : 0.0;
        d.drift[k] = fabs(m) < 1e6 ? m : 0.0;
      }
    }
  }
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < d.ne; e += gridDim.x * blockDim.x) {
    const int i = d.ei[e], j = d.ej[e];
    const uint32_t sub = d.esub[e];
    const int type = (int)(sub >> 30), isub = (int)((sub >> 15) & 0x7fffu), jsub = (int)(sub & 0x7fffu);
    const int bi = d.bvoff[i], bj = d.bvoff[j];
    const int shi = d.kin[i].shape, shj = d.kin[j].shape;
    const int dvi = d.sh.voff[shi] - bi, dvj = d.sh.voff[shj] - bj;
    int4 q = make_int4(bi + isub, 0, 0, 0), r;
    if (type == VV) {
      q.y = bj + jsub;
    } else if (type == VE) {
      const int* ed = d.sh.edge + 2 * (d.sh.eoff[shj] + jsub);
      q.y = bj + ed[0];
      q.z = bj + ed[1];
    } else if (type == VF) {
      const int gface = d.sh.foff[shj] + jsub;
      q.y = d.sh.fstart[gface];
      q.z = d.sh.fstart[gface + 1] - q.y;
      q.w = bj;
    } else {
      const int* edi = d.sh.edge + 2 * (d.sh.eoff[shi] + isub);
      const int* edj = d.sh.edge + 2 * (d.sh.eoff[shj] + jsub);
      q = make_int4(bi + edi[0], bi + edi[1], bj + edj[0], bj + edj[1]);
    }
    r = type == EE   ? make_int4(q.x + dvi, q.y + dvi, q.z + dvj, q.w + dvj)
        : type == VF ? make_int4(q.x + dvi, q.y, q.z, q.w + dvj)
                     : make_int4(q.x + dvi, q.y + dvj, q.z + dvj, 0);
    d.edesc[e] = q;
    d.edesc_s[e] = r;
  }
}

// Interaction::UpdateDispatcher (Interaction.cpp:147-326) without the
// relative velocity (the law computes it), on the positions p of the
// entry's vertices: VV i, j; VE i, j's edge; EE i's edge, j's edge; VF i, the
// face's first three and last vertices.  nbv: the face's vertex count; a
// face of more than four (or fewer than three) takes the others from
// face(k).
template <class Face>
__device__ __forceinline__ void update_kinematics(int type, int nbv, const v3 p[5], double Ri, double Rj, Kin& k,
                                                  Face face) {
  if (type == VV) {
    v3 posi = p[0];
    v3 posj = p[1];
    k.n = vsub(posi, posj);
    k.dn = vnormalize(&k.n) - (Ri + Rj);
    k.pos = vsub(posi, vsc(Ri + 0.5 * k.dn, k.n));
  } else if (type == VE) {
    v3 posj1 = p[1];
    v3 posj2 = p[2];
    v3 posi = p[0];
    v3 E = vsub(posj2, posj1);
    v3 v = vsub(posi, posj1);
    double r = vdot(v, E) / vdot(E, E);
    if (r <= 0.0 || r >= 1.0) {
      k.deact = true;
      return;
    }
    k.n = vsub(posi, vadd(posj1, vsc(r, E)));
    k.dn = vnormalize(&k.n) - (Ri + Rj);
    k.pos = vsub(posi, vsc(Ri + 0.5 * k.dn, k.n));
  } else if (type == VF) {
    v3 A = p[1];
    v3 B = p[2];
    v3 C = p[4];
    v3 posi = p[0];
    v3 v = vsub(posi, A);
    v3 v1 = vsub(B, A);
    vnormalize(&v1);
    v3 v2 = vsub(C, A);
    k.n = vcross(v1, v2);
    vnormalize(&k.n);
    double dist = vdot(v, k.n);
    if (dist < 0.0) {
      k.n = vneg(k.n);
      dist = -dist;
    }
    v3 P = vsub(posi, vsc(dist, k.n));
    v2 = vcross(k.n, v1);
    int odd = 0;
    const double ori1 = vdot(P, v1), ori2 = vdot(P, v2);
    if (nbv == 3 || nbv == 4) {
      cross_edge(A, B, v1, v2, ori1, ori2, odd);
      cross_edge(B, p[3], v1, v2, ori1, ori2, odd);
      if (nbv == 4) cross_edge(p[3], C, v1, v2, ori1, ori2, odd);
      cross_edge(C, A, v1, v2, ori1, ori2, odd);
    } else {
      v3 a = A;
      for (int iva = 0; iva < nbv; iva++) {
        const v3 b = face(iva + 1 == nbv ? 0 : iva + 1);
        cross_edge(a, b, v1, v2, ori1, ori2, odd);
        a = b;
      }
    }
    if (odd != 0) {
      k.dn = dist - (Ri + Rj);
      k.pos = vsub(posi, vsc(Ri + 0.5 * k.dn, k.n));
    } else {
      k.deact = true;  // n keeps the new face normal, pos and vel stay stale
    }
  } else {
    v3 posi1 = p[0];
    v3 posi2 = p[1];
    v3 posj1 = p[2];
    v3 posj2 = p[3];
    v3 Ei = vsub(posi2, posi1);
    v3 Ej = vsub(posj2, posj1);
    v3 v = vsub(posi1, posj1);
    double c = vdot(Ei, Ei), dd = vdot(Ej, Ej), e = vdot(Ei, Ej);
    double f = (c * dd) - (e * e);
    if (fabs(f) > 1.0e-12) {
      f = 1.0 / f;
      double a = vdot(Ei, v), b = vdot(Ej, v);
      double s = (e * b - a * dd) * f;
      double t = (c * b - e * a) * f;
      if (s <= 0.0 || s >= 1.0 || t <= 0.0 || t >= 1.0) {
        k.deact = true;
        return;
      }
      k.n = vsub(vadd(posi1, vsc(s, Ei)), vadd(posj1, vsc(t, Ej)));
      k.dn = vnormalize(&k.n) - (Ri + Rj);
      k.pos = vsub(vadd(posi1, vsc(s, Ei)), vsc(Ri + 0.5 * k.dn, k.n));
    } else {
      k.deact = true;
    }
  }
}

// The same on an entry's resolved global vertices q (k_entry_desc), as the
// steps that evaluate every entry read them.
__device__ __forceinline__ void update_kinematics_gv(const Dev& d, int type, int4 q, double Ri, double Rj, Kin& k) {
  v3 p[5];
  int nbv = 0, fs = 0, bj = 0;
  p[0] = gvtx(d.gv, q.x);
  if (type == VF) {
    fs = q.y;
    nbv = q.z;
    bj = q.w;
    const int* fv = d.sh.fidx + fs;
    p[1] = gvtx(d.gv, bj + fv[0]);
    p[2] = gvtx(d.gv, bj + fv[1]);
    p[3] = gvtx(d.gv, bj + fv[nbv > 2 ? 2 : 0]);
    p[4] = gvtx(d.gv, bj + fv[nbv - 1]);
  } else {
    p[1] = gvtx(d.gv, q.y);
    p[2] = type == VV ? p[1] : gvtx(d.gv, q.z);
    p[3] = type == EE ? gvtx(d.gv, q.w) : p[2];
    p[4] = p[3];
  }
  update_kinematics(type, nbv, p, Ri, Rj, k, [&](int a) { return gvtx(d.gv, bj + d.sh.fidx[fs + a]); });
}

struct Hist {
  double fn;
  v3 ft, mom;
};

// ForceLaw_Default::computeInteraction (ForceLaw_Default.cpp:57-131), FT_CORR off
__device__ void law_default(const ContactPar& cp, const StepParams& sp, const Kin& k, double damp, const BodyKin& Pi,
                            const BodyKin& Pj, Hist& h) {
  if (k.dn > 0.0) {
    h.fn = 0.0;
    h.ft = V(0, 0, 0);
    h.mom = V(0, 0, 0);
    return;
  }
  const double kn = cp.kn, kt = cp.kt, mu = cp.mu, kr = cp.kr, mur = cp.mur;
  double vn = vdot(k.vel, k.n);
  double fne = -kn * k.dn;
  double fnv = damp * vn;
  h.fn = fne + fnv;
  if (h.fn < 0.0) h.fn = 0.0;
  v3 vt = vsub(k.vel, vsc(vn, k.n));
  h.ft = vadd(h.ft, vsc(kt, vsc(sp.dt, vt)));
  double threshold = fabs(mu * fne);
  double ft_square = vdot(h.ft, h.ft);
  if (ft_square > 0.0 && ft_square >= threshold * threshold) h.ft = vsc(threshold / sqrt(ft_square), h.ft);
  if (kr > 0.0) {
    h.mom = vadd(h.mom, vsc(sp.dt, vsc(kr, vsub(kvrot(Pj), kvrot(Pi)))));
    double threshold_mom = fabs(mur * h.fn);
    double mom_square = vdot(h.mom, h.mom);
    if (mom_square > 0.0 && mom_square >= threshold_mom * threshold_mom)
      h.mom = vsc(threshold_mom / sqrt(mom_square), h.mom);
  }
}

// ForceLaw_Avalanche::computeInteraction (ForceLaw_Avalanche.cpp:57-136)
__device__ void law_avalanche(const Dev& d, const ContactPar& cp, const StepParams& sp, const Kin& k, int i,
                              const BodyKin& Pi, const BodyKin& Pj, Hist& h) {
  if (k.dn > 0.0) {
    h.fn = 0.0;
    h.ft = V(0, 0, 0);
    h.mom = V(0, 0, 0);
    return;
  }
  const double kn = cp.kn, en2 = cp.en2, kt = cp.kt, mu = cp.mu, kr = cp.kr, mur = cp.mur;
  double prev_dn = k.prev_dn;
  if (prev_dn > 0.0) prev_dn = 0.0;
  double delta_Dn = k.dn - prev_dn;
  if (delta_Dn > 0.0)
    h.fn = -kn * en2 * k.dn;
  else if (delta_Dn < 0.0)
    h.fn += -kn * delta_Dn;
  if (h.fn < 0.0) h.fn = 0.0;
  v3 vt = vsub(k.vel, vsc(vdot(k.vel, k.n), k.n));
  h.ft = vadd(h.ft, vsc(kt, vsc(sp.dt, vt)));
  double threshold_ft = fabs(mu * h.fn);
  double ft_square = vdot(h.ft, h.ft);
  if (ft_square > 0.0 && ft_square > threshold_ft * threshold_ft)
    h.ft = vsc(threshold_ft / sqrt(ft_square), h.ft);
  h.mom = vadd(h.mom, vsc(sp.dt, vsc(kr, vsub(kvrot(Pj), kvrot(Pi)))));
  const BodyKin& P = (i < d.nDriven) ? Pj : Pi;
  v3 branch = vsub(k.pos, kpos(P));
  double r = vdot(branch, kvrot(P)) / vdot(kvrot(P), kvrot(P));
  branch = vsub(branch, vsc(r, kvrot(P)));
  double threshold_mom = fabs(mur * sqrt(vnorm2(branch)) * h.fn);
  double mom_square = vdot(h.mom, h.mom);
  if (mom_square > 0.0 && mom_square > threshold_mom * threshold_mom)
    h.mom = vsc(threshold_mom / sqrt(mom_square), h.mom);
}

// ForceLaw_StickedLinks::computeInteraction (ForceLaw_StickedLinks.cpp:75-215)
// bp: the bond's interface parameters (read for stick >= 0)
__device__ void law_sticked(const Dev& d, const ContactPar& cp, const double bp[8], const StepParams& sp, const Kin& k,
                            double damp, int stick, int i, int j, const BodyKin& Pi, const BodyKin& Pj, Hist& h,
                            bool paramsInInterfaces) {
  if (stick >= 0) {
    double kn = 0.0, kt = 0.0, kr = 0.0, fn0 = 1.0, ft0 = 1.0, mom0 = 1.0, power = 1.0;
    double dn0 = bp[7];
    const int g1 = Pi.group, g2 = Pj.group;
    if (paramsInInterfaces) {
      kn = bp[0];
      kt = bp[1];
      kr = bp[2];
      fn0 = bp[3];
      ft0 = bp[4];
      mom0 = bp[5];
      power = bp[6];
    } else if (d.cluster[i] == d.cluster[j]) {
      kn = prm(d.par, P_KN_IN, g1, g2);
      kt = prm(d.par, P_KT_IN, g1, g2);
      kr = prm(d.par, P_KR_IN, g1, g2);
      fn0 = prm(d.par, P_FN0_IN, g1, g2);
      ft0 = prm(d.par, P_FT0_IN, g1, g2);
      mom0 = prm(d.par, P_MOM0_IN, g1, g2);
      power = prm(d.par, P_POW_IN, g1, g2);
      dn0 = 0.0;
    } else {
      kn = prm(d.par, P_KN_OUT, g1, g2);
      kt = prm(d.par, P_KT_OUT, g1, g2);
      kr = prm(d.par, P_KR_OUT, g1, g2);
      fn0 = prm(d.par, P_FN0_OUT, g1, g2);
      ft0 = prm(d.par, P_FT0_OUT, g1, g2);
      mom0 = prm(d.par, P_MOM0_OUT, g1, g2);
      power = prm(d.par, P_POW_OUT, g1, g2);
    }
    double vn = vdot(k.vel, k.n);
    double fne = -kn * (k.dn - dn0);
    double fnv = damp * vn;
    h.fn = fne + fnv;
    v3 vt = vsub(k.vel, vsc(vn, k.n));
    h.ft = vadd(h.ft, vsc(kt, vsc(sp.dt, vt)));
    v3 ftv = vsc(damp, vt);
    h.ft = vadd(h.ft, ftv);
    h.mom = vadd(h.mom, vsc(sp.dt, vsc(kr, vsub(kvrot(Pj), kvrot(Pi)))));
    // power 2 (every generated deck, the interfaces' default): x * x, which
    // is what glibc's pow(x, 2.0) returns for every x (exhaustive sampling
    // in tests/test_pow_square.py), so the break decision is the host's bit
    // for bit; another power goes through the device pow (within an ulp of
    // glibc's, the decision differing only for a yield within an ulp of 0)
    const double rt = sqrt(vnorm2(h.ft)) / ft0, rm = sqrt(vnorm2(h.mom)) / mom0;
    const double pt = power == 2.0 ? rt * rt : pow(rt, power);
    const double pm = power == 2.0 ? rm * rm : pow(rm, power);
    double yield = pt + pm - h.fn / fn0 - 1.0;
    if (yield > 0.0) {  // idempotent stores, consumed at the end of the step
      d.ifc.brk[stick] = 1;
      d.flags[0] = 1;
    }
  } else {
    if (k.dn > 0.0) {
      h.fn = 0.0;
      h.ft = V(0, 0, 0);
      h.mom = V(0, 0, 0);
      return;
    }
    const double kn = cp.kn, kt = cp.kt, mu = cp.mu, kr = cp.kr, mur = cp.mur;
    double vn = vdot(k.vel, k.n);
    double fne = -kn * k.dn;
    double fnv = damp * vn;
    h.fn = fne + fnv;
    if (h.fn < 0.0) h.fn = 0.0;
    v3 vt = vsub(k.vel, vsc(vn, k.n));
    h.ft = vadd(h.ft, vsc(kt, vsc(sp.dt, vt)));
    double threshold = fabs(mu * h.fn);
    double ft_square = vdot(h.ft, h.ft);
    if (ft_square > 0.0 && ft_square >= threshold * threshold) h.ft = vsc(threshold / sqrt(ft_square), h.ft);
    h.mom = vadd(h.mom, vsc(sp.dt, vsc(kr, vsub(kvrot(Pj), kvrot(Pi)))));
    double threshold_mom = fabs(mur * h.fn);
    double mom_square = vdot(h.mom, h.mom);
    if (mom_square > 0.0 && mom_square >= threshold_mom * threshold_mom)
      h.mom = vsc(threshold_mom / sqrt(mom_square), h.mom);
  }
}

// The geometry pass of one listed entry e (Interaction::UpdateDispatcher,
// Rockable.cpp:2934-2977): its gap, and for an active entry its kinematics in
// a (returns true); an inactive entry gets its gap and activity byte here,
// and with skipping its far-entry key.
// kinematics(k): the contact kinematics; old: the entry's activity byte and
// ci, cj its bodies' motion bounds, which only an inactive entry needs.
template <bool GEOM_ALL, class Kinematics, class Old, class Bounds>
__device__ __forceinline__ bool geom_entry(const Dev& d, int e, bool skipping, int i, int j, int stick, const BodyKin& Pi,
                                           const BodyKin& Pj, ActiveKin& a, Kinematics kinematics, Old old_act,
                                           Bounds bounds) {
  bool act = false;
  Kin k;
  k.deact = false;
  k.prev_dn = 0.0;  // the previous dn is read by the law, for active entries only
  if (stick >= 0) {  // a bond may run on stale geometry after a deactivation
    const EGeom& g = d.egeo[e];
    k.n = V(g.nx, g.ny, g.nz);
    k.pos = V(g.px, g.py, g.pz);
  }
  kinematics(k);
  if (k.deact) k.dn = 0.0;  // Interaction::deactivate (Interaction.cpp:123-128)
  act = (k.dn < 0.0) || (stick >= 0);
  if (act) {
    a.nx = k.n.x;
    a.ny = k.n.y;
    a.nz = k.n.z;
    a.px = k.pos.x;
    a.py = k.pos.y;
    a.pz = k.pos.z;
    a.dn = k.dn;
    a.prev_dn = 0.0;  // (unused: the law reads the previous dn itself)
    a.e = e;
    a.deact = k.deact ? 1 : 0;
    a.i = i;
    a.j = j;
  } else {
    // activity byte: bit 0 active, bit 1 history maybe non-zero; the
    // history and the slot flags are written only when they change
    const uint8_t old = old_act();
    uint8_t now = old & 2;
    if (k.deact) {
      if (old & 2) {
        EState o;
        o.fn = 0.0;
        o.ftx = o.fty = o.ftz = 0.0;
        o.momx = o.momy = o.momz = 0.0;
        d.est[e] = o;
        now = 0;
      }
      d.edn[e] = 0.0;
      if (skipping) d.ekey[e] = -INFINITY;
    } else {
      d.edn[e] = k.dn;  // stale fn/ft/mom are kept (Rockable.cpp:3022)
      if (skipping && now == 0) {
        // the key of a zero-history entry (a body without a finite bound
        // never lets its entries be skipped)
        double ci, cj;
        bounds(ci, cj);
        d.ekey[e] = (ci < INFINITY && cj < INFINITY) ? k.dn + ci + cj : -INFINITY;
      }
      if (GEOM_ALL) {
        const v3 vel = rel_vel(k.pos, Pi, Pj);
        EGeom g;
        g.nx = k.n.x;
        g.ny = k.n.y;
        g.nz = k.n.z;
        g.px = k.pos.x;
        g.py = k.pos.y;
        g.pz = k.pos.z;
        g.vx = vel.x;
        g.vy = vel.y;
        g.vz = vel.z;
        d.egeo[e] = g;
      }
    }
    if (now != old) {
      d.eact[e] = now;
      if (old & 1) {
        const int2 slots = reinterpret_cast<const int2*>(d.spos)[e];
        d.sact[slots.x] = 0;
        d.sact[slots.y] = 0;
      }
    }
  }
  return act;
}

// The force phase: geometry, then law, as two kernels or fused in one.
//  geometry  every listed entry: contact geometry from the body poses
//            (Interaction::UpdateDispatcher without the relative velocity).
//            An inactive entry gets its new dn (or the zeroed history of a
//            deactivation) and cleared activity flags; an active one (dn < 0
//            or bonded) keeps its geometry for the law.
//  law       every active entry: relative velocity, the force law, the
//            history and the two resultant slots.
// Two kernels: k_geom writes the active entries of geometry block b to
// akin[b * BS, b * BS + acount[b]) (ballot + block prefix, no atomics) and
// k_law gives a wavefront to each block's list.  Fused: k_interact keeps
// them in LDS.
//
// The geometry pass of one block of BS entries (block index blk): returns
// whether this thread's entry is active, with its kinematics in a.  Every
// thread of the block calls it (it synchronises the block).
template <bool GEOM_ALL, int BS, bool SORT = true>
__device__ __forceinline__ bool geom_pass(const Dev& d, int blk, int (*wtype)[5], short* perm, ActiveKin& a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // SORT: the block's entries are taken in the order of their contact type
  // (a counting sort in LDS; entries past the end last), so that a wavefront
  // runs one branch of update_kinematics instead of all four; without it
  // each thread takes its own entry, one dependent load and two barriers
  // sooner, its wavefront running the branches of the types it holds.
  // The far-entry skip (only when no geometry of inactive entries is
  // written): an inactive entry with zero history whose gap is proven
  // positive is left as it is; it sorts past the end.
  const bool skipping = !GEOM_ALL && d.skip_far;
  if (SORT) {
    const int e0 = blk * BS + (int)threadIdx.x;
    int ty = e0 < d.ne ? (int)(d.esub[e0] >> 30) : 4;
    if (skipping && e0 < d.ne && d.eact[e0] == 0 &&
        d.ekey[e0] - d.cbound[d.ei[e0]] - d.cbound[d.ej[e0]] > kSkipMargin)
      ty = 4;
    unsigned long long mine = 0ull;
#pragma unroll
    for (int t = 0; t < 5; t++) {
      const unsigned long long m = __ballot(ty == t);
      if (ty == t) mine = m;
      if (lane == 0) wtype[wave][t] = __popcll(m);
    }
    __syncthreads();
    int rank = 0;
    for (int t = 0; t < 5; t++)
      for (int w = 0; w < BS / 64; w++) rank += (t < ty || (t == ty && w < wave)) ? wtype[w][t] : 0;
    rank += __popcll(mine & ((1ull << lane) - 1ull));
    perm[rank] = (short)threadIdx.x;
    __syncthreads();
  }
  const int e = blk * BS + (SORT ? (int)perm[threadIdx.x] : (int)threadIdx.x);
  bool act = false;
  bool skip = false;
  if (skipping && e < d.ne && d.eact[e] == 0)
    skip = d.ekey[e] - d.cbound[d.ei[e]] - d.cbound[d.ej[e]] > kSkipMargin;
  if (d.skip_count) {  // counts for the measurement of the skip (off in production)
    const unsigned long long ms = __ballot(skip), mz = __ballot(e < d.ne && d.eact[e] == 0),
                             ml = __ballot(e < d.ne);
    if (lane == 0) {
      atomicAdd(d.skip_count, (unsigned long long)__popcll(ms));
      atomicAdd(d.skip_count + 1, (unsigned long long)__popcll(mz));
      atomicAdd(d.skip_count + 2, (unsigned long long)__popcll(ml));
    }
  }
  if (e < d.ne && !skip) {
    const int i = d.ei[e], j = d.ej[e];
    const int stick = d.ifc.n > 0 ? d.estick[e] : -1;  // bonds exist only with interfaces
    const BodyKin &Pi = d.kin[i], &Pj = d.kin[j];
    act = geom_entry<GEOM_ALL>(
        d, e, skipping, i, j, stick, Pi, Pj, a,
        [&](Kin& k) { update_kinematics_gv(d, (int)(d.esub[e] >> 30), d.edesc[e], Pi.R, Pj.R, k); },
        [&] { return d.eact[e]; },
        [&](double& ci, double& cj) {
          ci = d.cbound[i];
          cj = d.cbound[j];
        });
  }
  return act;
}

// Rank of this thread's active entry among the block's (ballot + LDS
// prefix, no atomics) and the block's count of active entries.
template <int BS>
__device__ __forceinline__ int active_rank(bool act, int* wcount, int* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long m = __ballot(act);
  if (lane == 0) wcount[wave] = __popcll(m);
  __syncthreads();
  int base = 0, tot = 0;
  for (int w = 0; w < BS / 64; w++) {
    base += w < wave ? wcount[w] : 0;
    tot += wcount[w];
  }
  *total = tot;
  return base + __popcll(m & ((1ull << lane) - 1ull));
}

template <bool GEOM_ALL, int BS>
__global__ void __launch_bounds__(BS) k_geom(Dev d) {
  __shared__ int wcount[BS / 64];
  __shared__ int wtype[BS / 64][5];
  __shared__ short perm[BS];
  if (frozen(d)) return;
  for (TileLoop L = xcd_tiles((d.ne + BS - 1) / BS); L.t < L.end; L.t += L.step) {
    const int blk = L.t;
    ActiveKin a;
    const bool act = geom_pass<GEOM_ALL, BS>(d, blk, wtype, perm, a);
    int total = 0;
    const int r = active_rank<BS>(act, wcount, &total);
    if (act) d.akin[(size_t)blk * BS + r] = a;
    if (threadIdx.x == 0) d.acount[blk] = total;
    __syncthreads();
  }
}

// The force law of one active entry (kinematics in a): history, both
// resultant slots, activity flags.
// What the law reads of an active entry's own state.
struct EntryState {
  EState s;
  double damp, dn;
  int2 slots;
  int stick;
  uint8_t act;
  ContactPar cp;
  double bp[8];
};
// PRE: the entry's own state is in x (else it is read where it is needed).
template <int LAW, bool PRE>
__device__ __forceinline__ void law_item(const Dev& d, const StepParams& sp, int write_geom_all, int pii,
                                         const ActiveKin& a, const BodyKin& Pi, const BodyKin& Pj,
                                         const EntryState& x) {
  const int e = a.e;
  const int i = a.i, j = a.j;
  const int stick = PRE ? x.stick : d.estick[e];
  Kin k;
  k.n = V(a.nx, a.ny, a.nz);
  k.pos = V(a.px, a.py, a.pz);
  k.dn = a.dn;
  // the previous step's dn (the Avalanche law's only; a deactivation zeroes it)
  k.prev_dn = (LAW == LAW_AVALANCHE && !a.deact) ? (PRE ? x.dn : d.edn[e]) : 0.0;
  k.deact = a.deact != 0;
  Hist h;
  if (k.deact) {  // a bond keeps its stale velocity; the history restarts
    const EGeom& g = d.egeo[e];
    k.vel = V(g.vx, g.vy, g.vz);
    h.fn = 0.0;
    h.ft = V(0, 0, 0);
    h.mom = V(0, 0, 0);
  } else {
    k.vel = rel_vel(k.pos, Pi, Pj);
    const EState s = PRE ? x.s : d.est[e];
    h.fn = s.fn;
    h.ft = V(s.ftx, s.fty, s.ftz);
    h.mom = V(s.momx, s.momy, s.momz);
  }
  const double damp = LAW == LAW_AVALANCHE ? 0.0 : PRE ? x.damp : d.edamp[e];  // (the Avalanche law has none)
  const ContactPar cp = PRE ? x.cp : contact_par<LAW>(d.par, group_pair(d.par, Pi.group, Pj.group));
  if (LAW == LAW_AVALANCHE)
    law_avalanche(d, cp, sp, k, i, Pi, Pj, h);
  else if (LAW == LAW_STICKED)
    law_sticked(d, cp, PRE ? x.bp : d.ifc.par + 8 * (size_t)(stick >= 0 ? stick : 0), sp, k, damp, stick, i, j, Pi, Pj, h,
                pii != 0);
  else
    law_default(cp, sp, k, damp, Pi, Pj, h);
  EState o;
  o.fn = h.fn;
  o.ftx = h.ft.x;
  o.fty = h.ft.y;
  o.ftz = h.ft.z;
  o.momx = h.mom.x;
  o.momy = h.mom.y;
  o.momz = h.mom.z;
  d.est[e] = o;
  d.edn[e] = k.dn;
  // incrementResultants (Rockable.cpp:2756-2764), both sides
  v3 f = vadd(vsc(h.fn, k.n), h.ft);
  v3 Ci = vsub(k.pos, kpos(Pi));
  v3 Cj = vsub(k.pos, vadd(kpos(Pj), V(0.0, 0.0, 0.0)));
  v3 mi = vadd(vcross(Ci, f), h.mom);
  v3 mj = vsub(vcross(Cj, vneg(f)), h.mom);
  // the two resultant slots: body i adds (f, mi), body j adds (-f, mj);
  // x + (-y) is x - y exactly, so the serial sums are unchanged
  const int2 slots = PRE ? x.slots : reinterpret_cast<const int2*>(d.spos)[e];
  double* ci = d.sval + 6 * (size_t)slots.x;
  double* cj = d.sval + 6 * (size_t)slots.y;
  st3(ci, f);
  st3(ci + 3, mi);
  st3(cj, vneg(f));
  st3(cj + 3, mj);
  // Geometry is persistent for bonds (a deactivated bond keeps its stale n,
  // pos, vel); for other entries it is written when an output is due.
  if (stick >= 0 || (write_geom_all && !k.deact)) {
    EGeom g;
    g.nx = k.n.x;
    g.ny = k.n.y;
    g.nz = k.n.z;
    g.px = k.pos.x;
    g.py = k.pos.y;
    g.pz = k.pos.z;
    g.vx = k.vel.x;
    g.vy = k.vel.y;
    g.vz = k.vel.z;
    d.egeo[e] = g;
  }
  const uint8_t old = PRE ? x.act : d.eact[e];
  if (old != 3) {
    d.eact[e] = 3;
    if (!(old & 1)) {
      d.sact[slots.x] = 1;
      d.sact[slots.y] = 1;
    }
  }
}

// The law of an active entry apart from its geometry pass.
template <int LAW>
__device__ __forceinline__ void law_entry(const Dev& d, const StepParams& sp, int write_geom_all, int pii,
                                          const ActiveKin& a) {
  const BodyKin Pi = d.kin[a.i];
  const BodyKin Pj = d.kin[a.j];
  law_item<LAW, false>(d, sp, write_geom_all, pii, a, Pi, Pj, EntryState{});
}

// Each wavefront takes W (at most kLawGroup) consecutive geometry blocks
// and spreads their active entries over its lanes, so that lanes are not left
// idle by blocks with few active entries.
constexpr int kLawGroup = 8;

template <int LAW>
__global__ void __launch_bounds__(kBlock, LAW == LAW_STICKED ? 2 : 4) k_law(Dev d, StepParams sp, int write_geom_all, int pii, int ngeom, int W) {
  if (frozen(d)) return;
  const int waves = (ngeom + W - 1) / W;
  for (TileLoop L = xcd_tiles((waves + kBlock / 64 - 1) / (kBlock / 64)); L.t < L.end; L.t += L.step) {
  const int g0 = (int)((L.t * (unsigned)blockDim.x + threadIdx.x) >> 6) * W;  // first geometry block
  if (g0 >= ngeom) continue;
  const int lane = threadIdx.x & 63;
  // inclusive prefix sums of the active counts of the W blocks (lanes < W)
  int incl = (lane < W && g0 + lane < ngeom) ? d.acount[g0 + lane] : 0;
  for (int o = 1; o < kLawGroup; o <<= 1) {
    const int t = __shfl_up(incl, o, 64);
    if (lane >= o) incl += t;
  }
  int pre[kLawGroup];
#pragma unroll
  for (int m = 0; m < kLawGroup; m++) pre[m] = __shfl(incl, m, 64);
  const int total = pre[kLawGroup - 1];
  for (int t = lane; t < total; t += 64) {
    int gb = 0, before = 0;
#pragma unroll
    for (int m = 0; m < kLawGroup; m++)
      if (pre[m] <= t) {
        gb = m + 1;
        before = pre[m];
      }
    const ActiveKin a = d.akin[(size_t)(g0 + gb) * d.geom_block + (t - before)];
    law_entry<LAW>(d, sp, write_geom_all, pii, a);
  }
  }
}

// Geometry and force law fused: the block's active entries go to LDS instead
// of the global active list, and the block's first threads apply the law to
// them after the geometry pass (no second launch, no round trip of the
// active kinematics through memory).
template <int LAW, bool GEOM_ALL, bool SORT>
__global__ void __launch_bounds__(kBlock, LAW == LAW_STICKED ? 2 : 4) k_interact(Dev d, StepParams sp, int write_geom_all, int pii) {
  __shared__ int wcount[kBlock / 64];
  __shared__ int wtype[kBlock / 64][5];
  __shared__ short perm[kBlock];
  __shared__ ActiveKin sa[kBlock];
  if (frozen(d)) return;
  for (TileLoop L = xcd_tiles((d.ne + kBlock - 1) / kBlock); L.t < L.end; L.t += L.step) {
    ActiveKin a;
    const bool act = geom_pass<GEOM_ALL, kBlock, SORT>(d, L.t, wtype, perm, a);
    int total = 0;
    const int r = active_rank<kBlock>(act, wcount, &total);
    if (act) sa[r] = a;
    __syncthreads();
    if ((int)threadIdx.x < total) law_entry<LAW>(d, sp, write_geom_all, pii, sa[threadIdx.x]);
    __syncthreads();
  }
}

// Geometry and force law of one entry of the evaluation list.  Everything it
// may read is read at once, before the geometry: its own state (an entry on
// the list is more often active than not), the bodies, the vertices in their
// shapes' frames, the law's parameters, the motion bounds; the reads then
// share one latency.  The vertices are moved by the bodies' poses here
// (glob_vertex's expression): a listed entry reads few of them, and computing
// them saves the round trip of every vertex through memory (264 bytes per
// hull and step).
template <int LAW>
__device__ __forceinline__ void eval_item(const Dev& d, const StepParams& sp, int pii, const ListItem& it) {
  const int e = it.e, i = it.i, j = it.j, type = it.kind & 3;
  EntryState x;
  x.s = d.est[e];
  x.dn = LAW == LAW_AVALANCHE ? d.edn[e] : 0.0;
  x.act = d.eact[e];
  x.stick = d.ifc.n > 0 ? d.estick[e] : -1;  // bonds exist only with interfaces; one may have broken since
  x.slots = it.slots;
  x.damp = it.damp;
  x.cp = contact_par<LAW>(d.par, it.gpair);
  if (LAW == LAW_STICKED && it.stick >= 0) {
    const double* bp = d.ifc.par + 8 * (size_t)it.stick;
#pragma unroll
    for (int q = 0; q < 8; q++) x.bp[q] = bp[q];
  }
  const BodyKin &Pi = d.kin[i], &Pj = d.kin[j];
  const double cbi = d.cbound[i], cbj = d.cbound[j];
  v3 r[5];
#pragma unroll
  for (int q = 0; q < 4; q++) r[q] = gvtx(d.sh.vtx, it.v[q]);
  r[4] = gvtx(d.sh.vtx, it.v4);
  const v3 ci = kpos(Pi), cj = kpos(Pj);
  const qt Qi = kq(Pi), Qj = kq(Pj);
  const double Hi = Pi.h, Hj = Pj.h, Ri = Pi.R, Rj = Pj.R;
  auto of_j = [&](v3 u) { return vadd(cj, qrot(Qj, vsc(Hj, u))); };
  ActiveKin a;
  if (geom_entry<false>(
          d, e, true, i, j, x.stick, Pi, Pj, a,
          [&](Kin& k) {
            v3 p[5];
            p[0] = vadd(ci, qrot(Qi, vsc(Hi, r[0])));
            // the second vertex is i's for two edges, else j's
            const bool ee = type == EE;
            p[1] = vadd(ee ? ci : cj, qrot(ee ? Qi : Qj, vsc(ee ? Hi : Hj, r[1])));
            if (type != VV) p[2] = of_j(r[2]);
            if (type == EE || type == VF) p[3] = of_j(r[3]);
            if (type == VF) p[4] = of_j(r[4]);
            update_kinematics(type, it.kind >> 2, p, Ri, Rj, k, [&](int n) {
              const int4 q = d.edesc_s[e];
              return of_j(gvtx(d.sh.vtx, q.w + d.sh.fidx[q.y + n]));
            });
          },
          [&] { return x.act; },
          [&](double& bi, double& bj) {
            bi = cbi;
            bj = cbj;
          }))
    law_item<LAW, true>(d, sp, 0, pii, a, Pi, Pj, x);
}

constexpr int kListTile = 1024;
// One tile's test (entries e0, e0 + 256, ... per thread): the entries that
// may need evaluation while the new list holds go to part, at places taken
// from count; their range there is returned.
__device__ __forceinline__ int2 list_tile(const Dev& d, int e0, ListItem* part, int* count) {
  constexpr int M = kListTile / kBlock;
  __shared__ int wcnt[M][kBlock / 64];
  __shared__ int at;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  unsigned keep = 0u;  // bit r: entry e0 + 256 r
#pragma unroll
  for (int r = 0; r < M; r++) {
    // the activity byte, key and pair together (one round trip), then the bounds
    const int e = e0 + r * kBlock;
    if (e < d.ne) {
      const uint8_t ea = d.eact[e];
      const double key = d.ekey[e];
      const int bi = d.ei[e], bj = d.ej[e];
      keep |= (ea == 0 && key - d.ahead[bi] - d.ahead[bj] > kSkipMargin) ? 0u : 1u << r;
    }
  }
  // rank the entries, in entry order: every wavefront's counts for the M
  // rows first, one barrier, then each thread its own places
  unsigned long long mask[M];
#pragma unroll
  for (int r = 0; r < M; r++) {
    mask[r] = __ballot(keep >> r & 1u);
    if (lane == 0) wcnt[r][wave] = __popcll(mask[r]);
  }
  __syncthreads();
  int n = 0;
#pragma unroll
  for (int r = 0; r < M; r++)
#pragma unroll
    for (int w = 0; w < kBlock / 64; w++) n += wcnt[r][w];
  if (t == 0) at = atomicAdd(count, n);
  __syncthreads();
  int k = at;
  const int first = k;
#pragma unroll
  for (int r = 0; r < M; r++) {
    int before = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; w++) {
      const int c = wcnt[r][w];
      before += w < wave ? c : 0;
      tot += c;
    }
    if (keep >> r & 1u) {
      const int e = e0 + r * kBlock;
      ListItem it;
      it.e = e;
      it.i = d.ei[e];
      it.j = d.ej[e];
      const int type = (int)(d.esub[e] >> 30);
      const int4 q = d.edesc_s[e];
      it.kind = type;
      it.v[0] = it.v[1] = it.v[2] = it.v[3] = it.v4 = q.x;
      if (type == VF) {
        const int* fv = d.sh.fidx + q.y;
        it.kind |= q.z << 2;
        it.v[1] = q.w + fv[0];
        it.v[2] = q.w + fv[1];
        it.v[3] = q.w + fv[q.z > 2 ? 2 : 0];
        it.v4 = q.w + fv[q.z - 1];
      } else {
        it.v[1] = q.y;
        if (type != VV) it.v[2] = q.z;
        if (type == EE) it.v[3] = q.w;
      }
      it.gpair = group_pair(d.par, d.kin[it.i].group, d.kin[it.j].group);
      it.stick = d.ifc.n > 0 ? d.estick[e] : -1;
      it.pad = 0;
      it.slots = reinterpret_cast<const int2*>(d.spos)[e];
      it.damp = d.edamp[e];
      part[k + before + __popcll(mask[r] & ((1ull << lane) - 1ull))] = it;
    }
    k += tot;
  }
  __syncthreads();  // the items are read by other threads; wcnt and at are free again
  return make_int2(first, k);
}

// The measurement of the skip (count_skips): entries whose gap the current
// bounds prove positive, inactive entries with zero history, entries.
__global__ void __launch_bounds__(kBlock) k_count_skips(Dev d) {
  if (frozen(d)) return;
  unsigned long long cnt[3] = {0ull, 0ull, 0ull};
  for (int e0 = blockIdx.x * blockDim.x; e0 < d.ne; e0 += gridDim.x * blockDim.x) {
    const int e = e0 + (int)threadIdx.x;
    const bool in = e < d.ne, zero = in && d.eact[e] == 0;
    const bool far = zero && d.ekey[e] - d.cbound[d.ei[e]] - d.cbound[d.ej[e]] > kSkipMargin;
    cnt[0] += __popcll(__ballot(far));
    cnt[1] += __popcll(__ballot(zero));
    cnt[2] += __popcll(__ballot(in));
  }
  if ((threadIdx.x & 63) == 0)
    for (int k = 0; k < 3; k++) atomicAdd(d.skip_count + k, cnt[k]);
}

// The force phase on the evaluation list (Dev::elist).  Most steps take the
// list as it stands: a lane per listed entry, geometry then law, nothing
// read of the others (four in five in a settled packing).  A step whose
// predictor found the list outdated takes the entries in tiles of 1024: each
// is tested against the motion bounds (coalesced reads of the activity byte,
// the key and the pair; the bounds are per body and stay in L2), those that
// may need evaluation while the bodies stay within their allowances are
// appended to the tile's XCD part of the new list (one atomic per tile), and
// evaluated.  The entries are independent (each writes its own state and its
// own two resultant slots), so neither the list's order nor an entry on it
// without need changes a result.
// What bounds it is the chain of an entry's dependent loads (the list's
// words, the item, its state with its bodies and vertices) and, from some
// 10^5 items, the entry states gathered one in five.  Testing every entry at
// every step, 1024 to a workgroup, ran a workgroup's evaluations in up to
// four rounds of a longer chain, however few workgroups a small packing has:
// 15.4 us for 517 spheres, 34.6 us for the 50 005-body pour (205 000 of its
// 1.12 M entries listed), 38.5 us for the 90 006-body slope, 24.4 and 34.2 us
// for 1 201 and 13 001 bonded cubes; on the list 14.0, 30.1, 36.8, 12.5 and
// 27.5 us, of which a new list every 17 steps or so is 2 to 4 us, and the
// predictor writes no vertices (22.4 -> 17.4 us at 50 005 bodies).
// XCD parts: the workgroups on XCD x (block mod 8) take that XCD's tiles and
// its part of the list, so that its L2 holds the bodies they read.
template <int LAW>
__global__ void __launch_bounds__(kBlock, LAW == LAW_STICKED ? 2 : 3) k_interact_list(Dev d, StepParams sp, int pii, int par) {
  const int t = threadIdx.x;
  const int x = (int)blockIdx.x & 7, kx = (int)blockIdx.x >> 3, nx = ((int)gridDim.x - x + 7) >> 3;
  // every control word in one round of loads
  const bool stop = frozen(d);
  const ListState* ls = d.ls;
  const int want = *(volatile const int*)&ls->want[par], gen = ls->gen, n0 = ls->cnt[0][x], n1 = ls->cnt[1][x];
  if (stop) return;
  if (blockIdx.x == 0 && t == 0) d.ls->want[1 - par] = 0;  // the next predictor sets it, nothing reads it now
  // XCD x's tiles, as xcd_block shares them out
  const int ntile = (d.ne + kListTile - 1) / kListTile, q8 = ntile >> 3, r8 = ntile & 7;
  const int tile0 = x < r8 ? x * (q8 + 1) : r8 * (q8 + 1) + (x - r8) * q8;
  const int tile1 = tile0 + q8 + (x < r8 ? 1 : 0);
  ListItem* part = d.elist + (size_t)tile0 * kListTile;
  // one round over the whole part, the workgroup's lanes taking every
  // (nx 256)-th place; or a round per tile over the tile's own items
  for (int tile = tile0 + kx; want ? tile < tile1 : tile == tile0 + kx; tile += nx) {
    int2 r = make_int2(kx * kBlock, gen & 1 ? n1 : n0);
    if (want) r = list_tile(d, tile * kListTile + t, part, &d.ls->cnt[(gen + 1) & 1][x]);
    const int stride = want ? kBlock : nx * kBlock;
    for (int k = r.x + t; k < r.y; k += stride) eval_item<LAW>(d, sp, pii, part[k]);
  }
}

// The gaps of the entries the last step skipped, from the current poses:
// what that step would have computed for them (Interaction::UpdateDispatcher,
// deactivate() giving 0).  The test is the skip's own with the bounds of the
// last step, so it also takes entries that step evaluated with a positive
// gap (recomputed to the same bits) and never an entry not evaluated since
// its key was cleared (a new list's entries keep the gap the merge gave).
__global__ void __launch_bounds__(kBlock) k_refresh_gaps(Dev d) {
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < d.ne; e += gridDim.x * blockDim.x) {
    if (d.eact[e] != 0 || !(d.ekey[e] - d.cbound[d.ei[e]] - d.cbound[d.ej[e]] > kSkipMargin)) continue;
    Kin k;
    k.deact = false;
    k.prev_dn = 0.0;
    update_kinematics_gv(d, (int)(d.esub[e] >> 30), d.edesc[e], d.kin[d.ei[e]].R, d.kin[d.ej[e]].R, k);
    d.edn[e] = k.deact ? 0.0 : k.dn;
  }
}

__global__ void __launch_bounds__(kBlock) k_reset_keys(Dev d) {
  if (blockIdx.x == 0 && threadIdx.x == 0) reset_list(d);
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < d.ne; e += gridDim.x * blockDim.x) d.ekey[e] = -INFINITY;
}

__device__ __forceinline__ v3 euler_domega(v3 I, v3 w, v3 M) {
  return V((M.x - (I.z - I.y) * w.y * w.z) / I.x, (M.y - (I.x - I.z) * w.z * w.x) / I.y,
           (M.z - (I.y - I.x) * w.x * w.y) / I.z);
}

// The body force of a free body as (F, M), returned by value: reference
// outputs merged across the branches compile to a stack copy (scratch).
struct FM {
  v3 F, M;
};
__device__ __forceinline__ FM body_force(const Dev& d, int b, const BodyKin& P) {
  FM r;
  r.F = V(0.0, 0.0, 0.0);
  r.M = V(0.0, 0.0, 0.0);
  if (d.bf == BF_ATTRACTING) {  // BodyForce_AttractingPoint.cpp:51-59
    v3 dir = vsub(V(d.bf_point[0], d.bf_point[1], d.bf_point[2]), kpos(P));
    double l2 = vnorm2(dir);
    if (l2 > 0.0) {
      double inv = 1.0 / sqrt(l2);
      dir = V(dir.x * inv, dir.y * inv, dir.z * inv);
      r.F = vsc(d.mass[b] * d.bf_acc, dir);
    }
  } else if (d.bf == BF_PREFDIR) {  // BodyForce_PreferredDirection.cpp:54-75
    v3 axis = V(d.bf_axis[0], d.bf_axis[1], d.bf_axis[2]);
    v3 axisB = qrot(kq(P), V(d.bf_axisBody[0], d.bf_axisBody[1], d.bf_axisBody[2]));
    vnormalize(&axisB);
    v3 u = vcross(axis, axisB);
    vnormalize(&u);
    double cosa = vdot(axisB, axis);
    double angle = acos(cosa);
    double sgn = -1.0;
    if (cosa < 0.0) {
      sgn = 1.0;
      angle = M_PI - angle;
    }
    r.M = vsc(angle, vsc(d.bf_Kr * sgn, u));
  } else if (d.bf == BF_VISCOUS) {  // BodyForce_ViscousFluid.cpp:51-62
    v3 velSqr = V(P.vx * P.vx, P.vy * P.vy, P.vz * P.vz);
    r.F = vsc(0.5 * 0.47 * d.bf_fluidDensity * d.bf_surface[b], velSqr);
  }
  return r;
}

// initialise_particle_forces_and_moments (Rockable.cpp:2869-2929): body force
// for free bodies, imposed force and moment values for driven ones.
// BF false: the deck has no body force (the kernel then holds none of its code).
template <bool BF = true>
__device__ __forceinline__ void init_resultants(const Dev& d, int b, const BodyKin& P, bool driven, v3& F, v3& M,
                                                int& c0, int& c1) {
  F = V(0.0, 0.0, 0.0);
  M = V(0.0, 0.0, 0.0);
  c0 = c1 = 0;
  if (BF && !driven && d.bf != BF_NONE) {
    const FM bf = body_force(d, b, P);
    F = vadd(F, bf.F);
    M = vadd(M, bf.M);
  }
  if (driven && d.nctrl > 0) {
    c0 = d.ctrl_off[b];
    c1 = d.ctrl_off[b + 1];
    // selects rather than a switch: a switch over components compiles to
    // an indexed store into a stack copy of (F, M), i.e. scratch memory
    for (int q = c0; q < c1; q++) {
      const DevControl& C = d.ctrl[d.ctrl_idx[q]];
      const int ty = C.type;
      const double v = C.value;
      F.x = ty == C_X_FOR ? v : F.x;
      F.y = ty == C_Y_FOR ? v : F.y;
      F.z = ty == C_Z_FOR ? v : F.z;
      M.x = ty == C_XROT_MOM ? v : ty == C_XYZROT_MOM ? C.vx : M.x;
      M.y = ty == C_YROT_MOM ? v : ty == C_XYZROT_MOM ? C.vy : M.y;
      M.z = ty == C_ZROT_MOM ? v : ty == C_XYZROT_MOM ? C.vz : M.z;
    }
  }
}

__device__ __forceinline__ double pick(const v3& F, const v3& M, int c) {
  return c == 0 ? F.x : c == 1 ? F.y : c == 2 ? F.z : c == 3 ? M.x : c == 4 ? M.y : M.z;
}

// compute_accelerations_from_resultants (Rockable.cpp:3419-3552) into acc and
// arot, and with kick the closing half kick (2120-2155) of P's velocities.
// m, I: the body's mass and principal inertia (loaded by the caller, early)
__device__ __forceinline__ void accelerate(const Dev& d, const StepParams& sp, int kick, BodyKin& P, bool driven, v3 F,
                                           v3 M, int c0, int c1, double m, v3 I, v3& acc, v3& arot) {
  const qt Q = kq(P);
  if (driven) {
    acc = V(0.0, 0.0, 0.0);
    arot = V(0.0, 0.0, 0.0);
    for (int qq = c0; qq < c1; qq++) {
      const DevControl& C = d.ctrl[d.ctrl_idx[qq]];
      const int ty = C.type;
      acc.x = ty == C_X_FOR ? F.x / m : acc.x;
      acc.y = ty == C_Y_FOR ? F.y / m : acc.y;
      acc.z = ty == C_Z_FOR ? F.z / m : acc.z;
      // selects rather than branches on the component (branches compile to
      // an indexed store into a stack copy of arot, i.e. scratch memory)
      const bool all = ty == C_XYZROT_MOM;
      const bool rx = all || ty == C_XROT_MOM, ry = all || ty == C_YROT_MOM, rz = all || ty == C_ZROT_MOM;
      if (rx || ry || rz) {
        const qt Qinv = qconj(Q);
        const v3 w = V(rx ? P.wx : 0.0, ry ? P.wy : 0.0, rz ? P.wz : 0.0);
        const v3 omega = qrot(Qinv, w);
        const v3 Mb = qrot(Qinv, M);
        const v3 dw = qrot(Q, euler_domega(I, omega, Mb));
        arot.x = rx ? dw.x : arot.x;
        arot.y = ry ? dw.y : arot.y;
        arot.z = rz ? dw.z : arot.z;
      }
    }
  } else {
    acc = vadd(vdiv(F, m), V(sp.gx, sp.gy, sp.gz));
    qt Qinv = qconj(Q);
    v3 omega = qrot(Qinv, kvrot(P));
    v3 Mb = qrot(Qinv, M);
    arot = qrot(Q, euler_domega(I, omega, Mb));
  }
  if (!kick) return;
  if (driven) {
    for (int qq = c0; qq < c1; qq++) {
      const DevControl& C = d.ctrl[d.ctrl_idx[qq]];
      const int ty = C.type;
      const v3 w = vadd(kvrot(P), vsc(sp.dt_2, arot));
      P.vx = ty == C_X_FOR ? P.vx + sp.dt_2 * acc.x : P.vx;
      P.vy = ty == C_Y_FOR ? P.vy + sp.dt_2 * acc.y : P.vy;
      P.vz = ty == C_Z_FOR ? P.vz + sp.dt_2 * acc.z : P.vz;
      P.wx = ty == C_XROT_MOM || ty == C_XYZROT_MOM ? w.x : P.wx;
      P.wy = ty == C_YROT_MOM || ty == C_XYZROT_MOM ? w.y : P.wy;
      P.wz = ty == C_ZROT_MOM || ty == C_XYZROT_MOM ? w.z : P.wz;
    }
  } else {
    v3 v = vadd(kvel(P), vsc(sp.dt_2, acc));
    v3 w = vadd(kvrot(P), vsc(sp.dt_2, arot));
    P.vx = v.x;
    P.vy = v.y;
    P.vz = v.z;
    P.wx = w.x;
    P.wy = w.y;
    P.wz = w.z;
  }
}
__device__ __forceinline__ void store_resultants(const Dev& d, int b, v3 F, v3 M, v3 acc, v3 arot) {
  st3(d.force + 3 * (size_t)b, F);
  st3(d.moment + 3 * (size_t)b, M);
  st3(d.acc + 3 * (size_t)b, acc);
  st3(d.arot + 3 * (size_t)b, arot);
}

// A body finished by itself: resultants, accelerations, kicked velocities.
__device__ __forceinline__ void finish_body(const Dev& d, const StepParams& sp, int kick, int b, BodyKin& P,
                                            bool driven, v3 F, v3 M, int c0, int c1, double m, v3 I) {
  v3 acc, arot;
  accelerate(d, sp, kick, P, driven, F, M, c0, c1, m, I, acc, arot);
  store_resultants(d, b, F, M, acc, arot);
  if (!kick) return;
  BodyKin* out = d.kin + b;
  out->vx = P.vx;
  out->vy = P.vy;
  out->vz = P.vz;
  out->wx = P.wx;
  out->wy = P.wy;
  out->wz = P.wz;
}

// dynamicCheckUpdateNL (Rockable.cpp:1571-1596), accumulation for one body
// at the end of its step: deltaPos += vel dt, deltaQ += Q.dot(vrot) dt, then
// the running max of |deltaPos|^2 and min of deltaQ.w as order keys (NaNs are
// ignored as the serial comparisons ignore them).  rst: the accumulations
// restart (a rebuild at the previous step).
__device__ __forceinline__ unsigned long long wkey(double w) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(w);
  return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
struct GuardAcc {
  unsigned long long kp, kw;  // max key of |deltaPos|^2, min key of deltaQ.w
};
__device__ __forceinline__ void guard_body(const Dev& d, const StepParams& sp, int b, const BodyKin& P, bool rst,
                                           GuardAcc& a) {
  v3 dp = rst ? V(0.0, 0.0, 0.0) : ld3(d.gdpos + 3 * (size_t)b);
  dp = vadd(dp, vsc(sp.dt, kvel(P)));
  st3(d.gdpos + 3 * (size_t)b, dp);
  const double tmp1 = vnorm2(dp);
  if (tmp1 == tmp1) {
    const unsigned long long k1 = (unsigned long long)__double_as_longlong(tmp1);
    a.kp = k1 > a.kp ? k1 : a.kp;
  }
  const qt dq = qdot(kq(P), kvrot(P));
  double* g = d.gdq + 4 * (size_t)b;
  qt q;
  if (rst) {
    q.w = 1.0;
    q.x = q.y = q.z = 0.0;
  } else {
    q.w = g[0];
    q.x = g[1];
    q.y = g[2];
    q.z = g[3];
  }
  q.w += dq.w * sp.dt;
  q.x += dq.x * sp.dt;
  q.y += dq.y * sp.dt;
  q.z += dq.z * sp.dt;
  g[0] = q.w;
  g[1] = q.x;
  g[2] = q.y;
  g[3] = q.z;
  double w = q.w;
  if (w > 1.0) w = 1.0;
  if (w < -1.0) w = -1.0;
  if (w == w) {
    const unsigned long long k2 = wkey(w);
    a.kw = k2 < a.kw ? k2 : a.kw;
  }
}
__device__ __forceinline__ bool guard_reset(const Dev& d) { return *(volatile const int*)&d.guard->reset != 0; }

// predict_free: the new pose and velocities of free body b (Rockable.cpp:
// 2036-2055) in P; store_predicted writes them back
__device__ __forceinline__ void predict_free_with(const StepParams& sp, BodyKin& P, v3 a, v3 ar) {
  v3 pos = vadd(kpos(P), vadd(vsc(sp.dt, kvel(P)), vsc(sp.dt2_2, a)));
  v3 vel = vadd(kvel(P), vsc(sp.dt_2, a));
  qt Q = kq(P);
  const v3 w = kvrot(P);
  Q = qadd_scaled(Q, qdot(Q, w), sp.dt);
  Q = qadd_scaled(Q, qddot(Q, w, ar), sp.dt2_2);
  qnormalize(&Q);
  v3 w2 = vadd(w, vsc(sp.dt_2, ar));
  P.px = pos.x;
  P.py = pos.y;
  P.pz = pos.z;
  P.qw = Q.w;
  P.qx = Q.x;
  P.qy = Q.y;
  P.qz = Q.z;
  P.vx = vel.x;
  P.vy = vel.y;
  P.vz = vel.z;
  P.wx = w2.x;
  P.wy = w2.y;
  P.wz = w2.z;
}
__device__ __forceinline__ void predict_free(const Dev& d, const StepParams& sp, int b, BodyKin& P) {
  predict_free_with(sp, P, ld3(d.acc + 3 * (size_t)b), ld3(d.arot + 3 * (size_t)b));
}
// The far-entry skip's motion bound of one predicted body: no vertex of it
// moved by more than |dx| + 2 |dQ| rmax in this step (for unit quaternions
// |Q' v Q'* - Q v Q*| <= 2 |Q' - Q| |v|), plus a rounding allowance.
// It also sets the allowance ahead of it (24 steps of this motion, at least
// ahead_min) and asks for a new evaluation list when the bound passes limit,
// what the list in use was written for (a NaN does too).  Not where the next
// step takes no list (par -1): the bound stays past the limit and the
// predictor of the first step that takes one asks.
constexpr double kAheadSteps = 24.0;
__device__ __forceinline__ void set_bound(const Dev& d, int b, double bound, double step, double limit, int par) {
  d.cbound[b] = bound;
  d.ahead[b] = bound + fmax(kAheadSteps * step, d.ahead_min);
  if (par >= 0 && !(bound <= limit)) d.ls->want[par] = 1;
}
__device__ __forceinline__ void add_motion_bound_with(const Dev& d, const StepParams& sp, int b, const BodyKin& old,
                                                      const BodyKin& P, double cb, double rmax, double limit,
                                                      v3 drift, int par) {
  if (!d.skip_far) return;
  const double dx = P.px - old.px - sp.dt * drift.x, dy = P.py - old.py - sp.dt * drift.y,
               dz = P.pz - old.pz - sp.dt * drift.z;
  const double qw = P.qw - old.qw, qx = P.qx - old.qx, qy = P.qy - old.qy, qz = P.qz - old.qz;
  const double step = sqrt(dx * dx + dy * dy + dz * dz) + 2.0 * sqrt(qw * qw + qx * qx + qy * qy + qz * qz) * rmax;
  const double mag = fabs(P.px) + fabs(P.py) + fabs(P.pz);
  set_bound(d, b, cb + (step + 1e-15 * (1.0 + mag)), step, limit, par);
}
// The bound of driven body b, from cb: without a control it stays where it is,
// which in the moving frame is a motion of |D|.  One thread of a launch
// writes a body's limit, bound and allowance, so that the limit is the
// allowance the list was written for.
__device__ __forceinline__ void driven_bound(const Dev& d, const StepParams& sp, int b, double cb, double limit, v3 drift,
                                             int par) {
  if (!(cb < INFINITY)) return;
  const double ux = sp.dt * drift.x, uy = sp.dt * drift.y, uz = sp.dt * drift.z;
  const double step = sqrt(ux * ux + uy * uy + uz * uz);
  set_bound(d, b, cb + (step + 1e-15), step, limit, par);
}
// all of them, spread over a predictor's threads (thread `first` of `stride`)
__device__ __forceinline__ void driven_bounds(const Dev& d, const StepParams& sp, int first, int stride, int par) {
  if (!d.skip_far) return;
  for (int b = first; b < d.nDriven; b += stride)
    driven_bound(d, sp, b, d.cbound[b], d.climit[b], ld3(d.drift), par);
}
__device__ __forceinline__ void add_motion_bound(const Dev& d, const StepParams& sp, int b, const BodyKin& old,
                                                 const BodyKin& P, int par) {
  if (!d.skip_far) return;
  add_motion_bound_with(d, sp, b, old, P, d.cbound[b], d.rmax[b], d.climit[b], ld3(d.drift), par);
}

typedef double d2 __attribute__((ext_vector_type(2)));  // one 16-byte access

// A body record (BodyKin, 16 doubles) in LDS at r.
__device__ __forceinline__ BodyKin rec_load(const double* r) {
  BodyKin P;
  P.px = r[0];
  P.py = r[1];
  P.pz = r[2];
  P.qw = r[3];
  P.qx = r[4];
  P.qy = r[5];
  P.qz = r[6];
  P.vx = r[7];
  P.vy = r[8];
  P.vz = r[9];
  P.wx = r[10];
  P.wy = r[11];
  P.wz = r[12];
  P.R = r[13];
  P.h = r[14];
  P.shape = __double2loint(r[15]);
  P.group = __double2hiint(r[15]);
  return P;
}
__device__ __forceinline__ void rec_store_motion(double* r, const BodyKin& P) {
  r[0] = P.px;
  r[1] = P.py;
  r[2] = P.pz;
  r[3] = P.qw;
  r[4] = P.qx;
  r[5] = P.qy;
  r[6] = P.qz;
  r[7] = P.vx;
  r[8] = P.vy;
  r[9] = P.vz;
  r[10] = P.wx;
  r[11] = P.wy;
  r[12] = P.wz;
}
constexpr int kRec = 17;  // LDS doubles per record (16, and one so that the per-body reads spread over the banks)
static_assert(sizeof(BodyKin) == 16 * sizeof(double), "a body record is 16 doubles");

// Bit k of the result: byte k of x (each 0 or 1).
__device__ __forceinline__ unsigned byte_bits(unsigned x) { return ((x & 0x01010101u) * 0x10204080u) >> 28; }

// compute_resultants (Rockable.cpp:3267-3272) as a per-body sum in slot
// order, with initialise_particle_forces_and_moments, the accelerations and
// the closing kick.  A workgroup takes NB free bodies, whose slots are
// consecutive, or one driven body:
//   1. the T threads read all the slots' activity bytes (16 each, up to
//      16 T slots at a time) and rank the active ones into an LDS list;
//   2. they read the active slots' terms (48 bytes each), 2 T slots at a
//      time, into LDS;
//   3. lanes of each body, one to three components of (F, M) each, add its terms in
//      slot order, so every component is the reference's bit for bit;
//   4. one thread per body finishes it.  The records (128 bytes) are read at
//      the start and written back whole, in contiguous doubles, through LDS.
// What bounds it is the chain of dependent loads (slot range, activity,
// terms): here three, whatever the bodies' slot counts.  Before, 16 lanes
// took one body, read its activity 64 bytes and its terms 8 slots at a time,
// so a wall with 200 slots or a bonded cube with 18 active ones waited for
// many loads in turn, and 4 of a wavefront's lanes finished its bodies:
// 15.7 us for 706 bodies, 22.6 us for 50 005, 40.3 us for 90 006 with the
// displacement check, 13.7 us for 13 001 bonded cubes; at first 6.6, 14.8, 23.4
// and 10.3 us, before the predictor joined (below).
// With fuse the step after this one follows at once, and the free bodies take
// its predictor (and their listed vertices) here, while their records and
// accelerations are at hand: one launch and one pass over the records less,
// and the resultants and accelerations, which only the predictor or a read-out
// uses, are not stored.  Apart, the two kernels took 14.8 + 11.3 us for
// 50 005 bodies, fused 22.4 us; 6.6 + 7.5 and 8.7 us for 706 bodies, where a
// launch counts most.
// Driven bodies come first, one workgroup each (a wall's many slots fill it),
// or with MANY driven_per of them (below); then, a wavefront each, the 64-slot chunks of the heavy bodies, whose
// partial sums (from -0.0, the identity of addition) k_heavy_finish takes.
// Bodies with more than heavy_min slots are left to the heavy kernels.  With
// guard, the displacement check accumulates each finished body and every
// workgroup stores its maxima in gpart[2 blockIdx.x].  One tile per workgroup
// whatever the persistent option: in a loop over tiles the compiler keeps the
// loop's invariants in 196 registers (102 without).

// The sum of one component (lanes gl < 6) over the slots [k0, k1) of one
// chunk of at most 64 slots by one wavefront, from -0.0, in slot order
// (inactive slots as -0.0: x + (-0.0) == x for every x).
__device__ __forceinline__ double sum_chunk(const Dev& d, int k0, int k1, int lane, double* lds) {
  const int k = k0 + lane;
  d2 v[3];
#pragma unroll
  for (int q = 0; q < 3; q++) v[q] = d2{-0.0, -0.0};
  if (k < k1 && d.sact[k]) {
    const d2* t = reinterpret_cast<const d2*>(d.sval + 6 * (size_t)k);
#pragma unroll
    for (int q = 0; q < 3; q++) v[q] = t[q];
  }
  d2* out = reinterpret_cast<d2*>(lds + 6 * lane);
#pragma unroll
  for (int q = 0; q < 3; q++) out[q] = v[q];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  double s = -0.0;
  if (lane < 6) {
#pragma unroll 16
    for (int q = 0; q < 64; q++) s += lds[6 * q + lane];
  }
  return s;
}

// Driven bodies per workgroup: one up to 2 047 of them, whose workgroups are
// resident at once with many others'; beyond (a bed of glued grains) as
// many as leave 1 024 to 2 047 workgroups, at most 32.  A step of 40 005 spheres,
// 10 005 of them driven, took 70.6 us with a workgroup each and the driven
// bodies' bounds moved by one workgroup, 27.0 us so; 171 and 51 us for 160 005
// spheres, 40 005 of them driven.
constexpr int kDrivenMany = 2048;
__host__ __device__ __forceinline__ int driven_per(int nDriven) {
  const int n = nDriven / 1024;
  return n < 1 ? 1 : n > 32 ? 32 : n;
}

// T threads; BF: the deck has a body force; MANY: kDrivenMany driven bodies or more
template <int T, int NB, bool BF, bool MANY>
__global__ void __launch_bounds__(T, 4) k_gather(Dev d, StepParams sp, GatherArgs A) {
  constexpr int kLanes = T / NB;  // lanes per body in the sums (8, 4 or 2)
  constexpr int kComp = kLanes >= 6 ? 1 : kLanes >= 3 ? 2 : 3;  // components per lane
  constexpr int kCap = 2 * T;   // slots' terms in LDS
  constexpr int kWin = 16 * T;  // slots scanned at a time
  __shared__ double rec[NB * kRec];
  __shared__ __align__(16) double vals[kCap * 6];
  __shared__ unsigned short list[kWin];
  __shared__ int pre[T + 1];
  __shared__ unsigned short act[T];
  __shared__ int wsum[T / 64];
  __shared__ double fm[NB][6];
  __shared__ unsigned long long heavy;  // MANY: bit k: body b0 + k is left to the heavy kernels
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int kick = A.kick, guard = A.guard;
  // (gather_blocks sizes the grid by the same rule)
  const int nchunk = A.fuse ? 0 : (d.nhch + T / 64 - 1) / (T / 64);
  const int tile = xcd_block((int)blockIdx.x, (int)gridDim.x);
  const int per = MANY ? driven_per(d.nDriven) : 1, ndt = MANY ? (d.nDriven + per - 1) / per : d.nDriven;
  const bool driven = tile < ndt, chunks = !driven && tile < ndt + nchunk;
  const int b0 = driven ? tile * per : d.nDriven + (tile - ndt - nchunk) * NB;
  const int nbk = chunks ? 0 : driven ? min(per, d.nDriven - b0) : min(NB, d.nb - b0);
  // one round of loads: the control words, the slot ranges, the records and
  // what finishing a body needs (in turn they took two latencies more: 7.5 us
  // for 517 spheres, 17.2 us for 50 005 hulls; so 6.6 and 16.5 us)
  int stop = 0, due = 0, again = 0;
  if (d.guard_on) {
    const volatile DevGuard* G = d.guard;
    const int fr = G->frozen, nu = G->nu, re = G->reset, fl = *(volatile const int*)d.flags;
    stop = fr;
    due = nu | fl;
    again = re;
  }
  const int want = *(volatile const int*)&d.ls->want[A.par];
  constexpr int kLoads = (8 * NB + T - 1) / T;
  static_assert(NB <= 64, "the first wavefront's threads have a body each");
  d2* kd = reinterpret_cast<d2*>(d.kin + b0);
  d2 x[kLoads];
#pragma unroll
  for (int r = 0; r < kLoads; r++)
    if (t + r * T < 8 * nbk) x[r] = kd[t + r * T];
  const int k0 = chunks ? 0 : d.soff[b0], kend = chunks ? 0 : d.soff[b0 + nbk];
  const int b = b0 + t;
  double mb = 1.0, cb = 0.0, rmx = 0.0, lim = 0.0, ah = 0.0;
  v3 Ib = V(1.0, 1.0, 1.0), drift = V(0.0, 0.0, 0.0);
  bool run = false;
  if (t < nbk) {
    mb = d.mass[b];
    Ib = ld3(d.inertia + 3 * (size_t)b);
    run = d.soff[b + 1] - d.soff[b] <= d.heavy_min;
    if (d.skip_far) {
      cb = d.cbound[b];
      rmx = d.rmax[b];
      lim = d.climit[b];
      ah = d.ahead[b];
      drift = ld3(d.drift);
    }
  }
  // the summing lanes' bodies and slot ranges
  const int lb = t / kLanes, lc = t % kLanes;
  const bool sums = lb < nbk && lc * kComp < 6;
  const int sb0 = sums ? d.soff[b0 + lb] : 0, sb1 = sums ? d.soff[b0 + lb + 1] : 0;
  if (stop) return;
  const bool rst = guard && again;
  // (the check that follows this step freezes the later ones on the same words)
  const bool predict = A.fuse && !due;
  // this step's force phase wrote a new evaluation list, for the allowances
  const bool relisted = A.listed && want != 0;
  const int npar = A.listed ? 1 - A.par : -1;  // (a run's steps all take the list, or none but its last does)
  if (relisted) lim = ah;
  if (relisted && blockIdx.x == 0 && t == 0) {
    const int g = d.ls->gen + 1;
    for (int k = 0; k < 8; k++) d.ls->cnt[(g + 1) & 1][k] = 0;
    d.ls->gen = g;
    if (d.ls->again) {
      d.ls->again = 0;
      d.ls->want[1 - A.par] = 1;
    }
  }
  GuardAcc ga;
  ga.kp = 0ull;
  ga.kw = ~0ull;
  if (chunks) {
    const int c = (tile - ndt) * (T / 64) + wv;
    if (c < d.nhch) {
      const int2 r = d.hch[c];
      const double s = sum_chunk(d, r.x, r.y, lane, vals + 64 * 6 * wv);
      if (lane < 6) d.hpart[6 * (size_t)c + lane] = s;
    }
  }
  // every body's limit, also a heavy one's; here the driven ones' bounds too
  // (a body's limit, bound and allowance are written by this thread alone)
  if (d.skip_far && t < nbk) {
    if (relisted) d.climit[b] = lim;
    if (driven && predict) driven_bound(d, sp, b, cb, lim, drift, npar);
  }
  if (chunks || (driven && nbk == 1 && kend - k0 > d.heavy_min)) {  // no body to finish
    if (guard && t == 0) {
      if (A.fuse && !chunks) guard_body(d, sp, b0, d.kin[b0], rst, ga);  // (else k_heavy_finish does)
      d.gpart[2 * (size_t)blockIdx.x] = ga.kp;
      d.gpart[2 * (size_t)blockIdx.x + 1] = ga.kw;
    }
    return;
  }
#pragma unroll
  for (int r = 0; r < kLoads; r++)
    if (t + r * T < 8 * nbk) {
      const int k = t + r * T;
      double* to = rec + (k >> 3) * kRec + 2 * (k & 7);
      to[0] = x[r].x;
      to[1] = x[r].y;
    }
  if (MANY) {
    const unsigned long long h = __ballot(t < nbk && !run);
    if (t == 0) heavy = h;
  }
  __syncthreads();
  int c0 = 0, c1 = 0;
  if (t < nbk) {
    v3 F, M;
    init_resultants<BF>(d, b, rec_load(rec + t * kRec), driven, F, M, c0, c1);
    fm[t][0] = F.x;
    fm[t][1] = F.y;
    fm[t][2] = F.z;
    fm[t][3] = M.x;
    fm[t][4] = M.y;
    fm[t][5] = M.z;
  }
  double s[kComp];
  bool first = true;
  // MANY leaves a heavy body's slots (a wall's among glued grains) out: [ka, kb)
  // are those up to the next one
  unsigned long long skip = MANY ? heavy : 0ull;
  int ka = k0, kb = MANY && skip ? d.soff[b0 + __ffsll(skip) - 1] : kend;
  for (int w0 = ka & ~15;; w0 += kWin) {
    while (MANY && skip && w0 >= kb) {
      ka = d.soff[b0 + __ffsll(skip)];
      skip &= skip - 1ull;
      kb = skip ? d.soff[b0 + __ffsll(skip) - 1] : kend;
      w0 = ka & ~15;
    }
    if (w0 >= kb) break;
    const int pos = w0 + 16 * t;
    unsigned m = 0u;
    if (pos < kb) {
      const uint4 x = *reinterpret_cast<const uint4*>(d.sact + pos);
      m = byte_bits(x.x) | byte_bits(x.y) << 4 | byte_bits(x.z) << 8 | byte_bits(x.w) << 12;
      if (pos < ka) m &= 0xffffu << (ka - pos);
      if (pos + 16 > kb) m &= 0xffffu >> (pos + 16 - kb);
    }
    int incl = __popc(m);
    const int mine = incl;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
    }
    if (lane == 63) wsum[wv] = incl;
    __syncthreads();
    int base = 0, total = 0;
#pragma unroll
    for (int w = 0; w < T / 64; w++) {
      base += w < wv ? wsum[w] : 0;
      total += wsum[w];
    }
    int r = base + incl - mine;
    pre[t] = r;
    act[t] = (unsigned short)m;
    if (t == 0) pre[T] = total;
    for (unsigned rest = m; rest; rest &= rest - 1u) list[r++] = (unsigned short)(16 * t + __ffs((int)rest) - 1);
    __syncthreads();
    // ranks of a body's slots within the window's list
    auto rank = [&](int k) -> int {
      const int q = min(max(k - w0, 0), kWin);
      if (q == kWin) return pre[T];
      return pre[q >> 4] + __popc((unsigned)act[q >> 4] & ((1u << (q & 15)) - 1u));
    };
    int lo = 0, hi = 0;
    if (sums) {
      if (first)
#pragma unroll
        for (int c = 0; c < kComp; c++) s[c] = fm[lb][lc * kComp + c];
      lo = rank(sb0);
      hi = rank(sb1);
    }
    first = false;
    for (int p0 = 0; p0 < total; p0 += kCap) {
      const int n = min(kCap, total - p0);
      d2 v[2][3];
#pragma unroll
      for (int h = 0; h < 2; h++)
        if (t + h * T < n) {
          const d2* x =
              reinterpret_cast<const d2*>(d.sval + 6 * (size_t)(w0 + (int)list[p0 + t + h * T]));
#pragma unroll
          for (int q = 0; q < 3; q++) v[h][q] = x[q];
        }
#pragma unroll
      for (int h = 0; h < 2; h++)
        if (t + h * T < n) {
          d2* x = reinterpret_cast<d2*>(vals + 6 * (t + h * T));
#pragma unroll
          for (int q = 0; q < 3; q++) x[q] = v[h][q];
        }
      __syncthreads();
      if (sums) {
        const int e = min(hi - p0, n);
        const double* x = vals + lc * kComp;
#pragma unroll 4
        for (int q = max(lo - p0, 0); q < e; q++)
#pragma unroll
          for (int c = 0; c < kComp; c++) s[c] += x[6 * q + c];
      }
      __syncthreads();
    }
  }
  if (sums && !first)
#pragma unroll
    for (int c = 0; c < kComp; c++) fm[lb][lc * kComp + c] = s[c];
  __syncthreads();
  if (run) {
    BodyKin P = rec_load(rec + t * kRec);  // (again: not held in registers over the sums)
    const v3 F = V(fm[t][0], fm[t][1], fm[t][2]), M = V(fm[t][3], fm[t][4], fm[t][5]);
    v3 acc, arot;
    accelerate(d, sp, kick, P, driven, F, M, c0, c1, mb, Ib, acc, arot);
    if (guard) guard_body(d, sp, b, P, rst, ga);
    if (predict && !driven) {
      const BodyKin old = P;
      predict_free_with(sp, P, acc, arot);
      add_motion_bound_with(d, sp, b, old, P, cb, rmx, lim, drift, npar);
    } else {
      store_resultants(d, b, F, M, acc, arot);
    }
    if (kick) rec_store_motion(rec + t * kRec, P);
  } else if (MANY && t < nbk && guard && A.fuse) {  // (in other steps k_heavy_finish does it)
    guard_body(d, sp, b, rec_load(rec + t * kRec), rst, ga);
  }
  __syncthreads();
  if (kick)
    for (int k = t; k < 8 * nbk; k += T) {
      const double* r = rec + (k >> 3) * kRec + 2 * (k & 7);
      kd[k] = d2{r[0], r[1]};
    }
  if (predict && !driven && A.glob != GLOB_NONE)
    for (int k = d.bvoff[b0] + t; k < d.bvoff[b0 + nbk]; k += T) {
      const int bb = d.bvbody[k];
      if (d.soff[bb + 1] == d.soff[bb]) continue;
      const BodyKin P = rec_load(rec + (bb - b0) * kRec);
      st3(d.gv + 3 * (size_t)k, glob_vertex(d.sh, P, k - d.bvoff[bb]));
    }
  if (!guard) return;
  // only the threads t < NB (the first wavefront) finish bodies
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long op = __shfl_xor(ga.kp, off, 64), ow = __shfl_xor(ga.kw, off, 64);
    ga.kp = op > ga.kp ? op : ga.kp;
    ga.kw = ow < ga.kw ? ow : ga.kw;
  }
  if (t == 0) {
    d.gpart[2 * (size_t)blockIdx.x] = ga.kp;
    d.gpart[2 * (size_t)blockIdx.x + 1] = ga.kw;
  }
}

// A passive heavy body (its force and moment feed nothing back into the
// motion; exact_sums off): the initial force and moment plus its chunks'
// partial sums, reduced by one workgroup of four wavefronts in a fixed order
// (thread t adds chunks t, t + 256, ... in turn, a butterfly over each
// wavefront's lanes, then (w0 + w1) + (w2 + w3)).  Deterministic; it
// differs from the serial sum only by rounding.
__device__ __forceinline__ void guard_heavy(const Dev& d, const StepParams& sp, int b, const BodyKin& P) {
  GuardAcc a;
  a.kp = 0ull;
  a.kw = ~0ull;
  guard_body(d, sp, b, P, guard_reset(d), a);
  if (a.kp) atomicMax(&d.guard->maxpos2, a.kp);
  if (a.kw != ~0ull) atomicMin(&d.guard->minw, a.kw);
}

static_assert(kBlock == 256, "k_heavy_finish combines four wavefronts");
__global__ void __launch_bounds__(kBlock) k_heavy_finish(Dev d, StepParams sp, int kick, int guard) {
  __shared__ double red[kBlock / 64][6];
  if (frozen(d)) return;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  for (TileLoop T = xcd_tiles(d.nheavy); T.t < T.end; T.t += T.step) {
    const int h = T.t;
    const int b = d.heavy[h];
    if (!d.passive[b] || d.exact_sums) continue;  // the same for the whole workgroup
    double a[6] = {-0.0, -0.0, -0.0, -0.0, -0.0, -0.0};
    for (int c = d.hch_off[h] + t; c < d.hch_off[h + 1]; c += kBlock) {
      const double* p = d.hpart + 6 * (size_t)c;
#pragma unroll
      for (int q = 0; q < 6; q++) a[q] += p[q];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
      for (int q = 0; q < 6; q++) a[q] += __shfl_xor(a[q], off, 64);
    if (lane == 0)
#pragma unroll
      for (int q = 0; q < 6; q++) red[wv][q] = a[q];
    __syncthreads();
    if (t == 0) {
#pragma unroll
      for (int q = 0; q < 6; q++) a[q] = (red[0][q] + red[1][q]) + (red[2][q] + red[3][q]);
      BodyKin P = d.kin[b];
      const bool driven = b < d.nDriven;
      v3 F, M;
      int c0, c1;
      init_resultants(d, b, P, driven, F, M, c0, c1);
      finish_body(d, sp, kick, b, P, driven, vadd(F, V(a[0], a[1], a[2])), vadd(M, V(a[3], a[4], a[5])), c0, c1,
                  d.mass[b], ld3(d.inertia + 3 * (size_t)b));
      if (guard) guard_heavy(d, sp, b, P);
    }
    __syncthreads();
  }
}

// compute_resultants for a heavy body that is not passive (or any heavy
// body with exact_sums): the serial sum, one workgroup per body.  Waves 1-3
// stage chunks of kHeavyChunk slots into LDS (inactive slots as -0.0, the
// identity of addition: x + (-0.0) == x for every x), double-buffered, while
// lanes 0-5 of wave 0 add them in order, one lane per component.
constexpr int kHeavyChunk = 512;

__global__ void __launch_bounds__(kBlock) k_gather_heavy(Dev d, StepParams sp, int kick, int guard) {
  __shared__ double lds[2 * kHeavyChunk * 6];
  if (frozen(d)) return;
  const int b = d.heavy[blockIdx.x];
  const int t = threadIdx.x;
  const int k0 = d.soff[b], k1 = d.soff[b + 1];
  if (d.passive[b] && !d.exact_sums) return;  // summed by chunks
  BodyKin P = d.kin[b];
  const bool driven = b < d.nDriven;
  v3 F, M;
  int c0, c1;
  init_resultants(d, b, P, driven, F, M, c0, c1);
  const uint8_t* act = d.sact;
  const double* val = d.sval;
  const int len = k1 - k0;
  const int nchunks = (len + kHeavyChunk - 1) / kHeavyChunk;
  const int wave = t >> 6, lane = t & 63;
  double s = pick(F, M, lane < 6 ? lane : 0);
  auto stage = [&](int c) {
    double* buf = lds + (c & 1) * kHeavyChunk * 6;
    const int kb = k0 + c * kHeavyChunk;
    const int n = min(kHeavyChunk, k1 - kb);
    for (int idx = t - 64; idx < n; idx += kBlock - 64) {
      const int k = kb + idx;
      const bool on = act[k] != 0;
      const double* v = val + 6 * (size_t)k;
#pragma unroll
      for (int q = 0; q < 6; q++) buf[6 * idx + q] = on ? v[q] : -0.0;
    }
  };
  if (wave > 0 && nchunks > 0) stage(0);
  __syncthreads();
  for (int c = 0; c < nchunks; c++) {
    if (wave > 0) {
      if (c + 1 < nchunks) stage(c + 1);
    } else if (lane < 6) {
      const double* buf = lds + (c & 1) * kHeavyChunk * 6 + lane;
      const int n = min(kHeavyChunk, k1 - (k0 + c * kHeavyChunk));
      for (int idx = 0; idx < n; idx++) s += buf[6 * idx];
    }
    __syncthreads();
  }
  if (wave == 0) {
    const double fx = __shfl(s, 0), fy = __shfl(s, 1), fz = __shfl(s, 2);
    const double mx = __shfl(s, 3), my = __shfl(s, 4), mz = __shfl(s, 5);
    if (lane == 0) {
      finish_body(d, sp, kick, b, P, driven, V(fx, fy, fz), V(mx, my, mz), c0, c1, d.mass[b],
                  ld3(d.inertia + 3 * (size_t)b));
      if (guard) guard_heavy(d, sp, b, P);
    }
  }
}

// locate entry (owner, other, sub) in the owner's sorted run
__device__ int find_entry(const Dev& d, int owner, int other, uint32_t sub) {
  int lo = d.istart[owner], hi = d.istart[owner + 1];
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    bool less = (d.ej[mid] < other) || (d.ej[mid] == other && d.esub[mid] < sub);
    if (less)
      lo = mid + 1;
    else
      hi = mid;
  }
  if (lo < d.istart[owner + 1] && d.ej[lo] == other && d.esub[lo] == sub) return lo;
  return -1;
}

// breakage_of_interfaces (Rockable.cpp:3350-3413), a thread per interface.  In
// the guarded loop one launch per step that breaks a bond.  (By the one
// workgroup of k_guard_check, 1 024 marks at a time, such a step of 226 000
// interfaces took 2.95 ms with its rebuild, instead of 2.83.)
__global__ void k_breakage(Dev d) {
  if (frozen(d)) return;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= d.ifc.n || !d.ifc.brk[k]) return;
  d.ifc.brk[k] = 0;
  if (!d.ifc.alive[k]) return;
  const uint64_t key = d.ifc.key[k];
  const int bi = (int)(key >> 32), bj = (int)(key & 0xffffffffu);
  const int g1 = d.kin[bi].group, g2 = d.kin[bj].group;
  for (int q = d.ifc.bond_off[k]; q < d.ifc.bond_off[k + 1]; q++) {
    const int* bk = d.ifc.bond_key + 3 * q;
    const int e = find_entry(d, bi, bj, pack_sub(bk[0], bk[1], bk[2]));
    if (e < 0) continue;
    d.estick[e] = -1;
    EState s = d.est[e];
    if (d.edn[e] >= 0.0) {
      s.fn = 0.0;
      s.ftx = s.fty = s.ftz = 0.0;
    } else {
      v3 T = V(s.ftx, s.fty, s.ftz);
      double FT = vnormalize(&T);
      double mu = prm(d.par, P_MU, g1, g2);
      double thr = fabs(mu * s.fn);
      if (FT > thr) {
        v3 ft = vsc(thr, T);
        s.ftx = ft.x;
        s.fty = ft.y;
        s.ftz = ft.z;
      }
    }
    d.est[e] = s;
  }
  d.ifc.alive[k] = 0;
  // for the host's accounting (it sorts them: interface order); an interface
  // breaks once, so the list holds at most n
  d.ifc.broken[atomicAdd(d.ifc.nbroken, 1)] = k;
  d.flags[0] = 1;  // needUpdate
}

// the end of a step of the integrate() loop (Rockable.cpp:2690-2740): a
// needUpdate left by the previous check makes the rebuild due now (the step
// kernels then wait for the host); then the check itself, on the maxima of
// the gather's workgroups (nparts pairs in gpart; max and min do not depend
// on the order).  The step index lives on the device, so that a captured
// sequence of steps replays as is.
constexpr int kCheckBlock = 1024;
// A bond that the law marked (flags) freezes the steps after this one; the host
// then breaks the interfaces (k_breakage) before it rebuilds.  A launch of that
// at every step took 4 us for nothing.
__global__ void __launch_bounds__(kCheckBlock) k_guard_check(Dev d, int nparts) {
  __shared__ unsigned long long red[2][kCheckBlock / 64];
  if (frozen(d)) return;
  unsigned long long kp = 0ull, kw = ~0ull;
  for (int k = threadIdx.x; k < nparts; k += kCheckBlock) {
    const unsigned long long p = d.gpart[2 * (size_t)k], w = d.gpart[2 * (size_t)k + 1];
    kp = p > kp ? p : kp;
    kw = w < kw ? w : kw;
  }
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long op = __shfl_xor(kp, off, 64), ow = __shfl_xor(kw, off, 64);
    kp = op > kp ? op : kp;
    kw = ow < kw ? ow : kw;
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = kp;
    red[1][threadIdx.x >> 6] = kw;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int k = 1; k < kCheckBlock / 64; k++) {
    kp = red[0][k] > kp ? red[0][k] : kp;
    kw = red[1][k] < kw ? red[1][k] : kw;
  }
  DevGuard* G = d.guard;
  const long long step = G->step;
  G->step = step + 1;
  if (d.note) *(volatile long long*)&d.note->done = step + 1;
  const int rebuild_now = G->nu;
  G->nu = 0;
  if (d.disp_check) {
    if (kp > G->maxpos2) G->maxpos2 = kp;
    if (kw < G->minw) G->minw = kw;
    G->reset = 0;
    const double mp = sqrt(__longlong_as_double((long long)G->maxpos2));
    const bool rot = G->minw != ~0ull && G->minw <= wkey(d.wstar);
    if (mp >= d.disp || rot) {
      G->nu = 1;
      G->reset = 1;
      G->maxpos2 = 0ull;
      G->minw = ~0ull;
    }
  }
  // a rebuild is due after this step: the check of the step before asked
  // for it, or an interface breaks in this step (breakage_of_interfaces sets
  // needUpdate, Rockable.cpp:3410, and the loop rebuilds at once, 2693)
  if (rebuild_now || *(volatile const int*)d.flags != 0) {
    G->frozen = 1;
    G->frozen_step = step;
    if (d.note) *(volatile int32_t*)&d.note->frozen = 1;
  }
}

// The 16 statistics the rebuild-interval network reads (per-body speed, spin,
// acceleration and accumulated displacement, and the guard's running
// maxima), scaled by the guard's thresholds.  Pass 1: per-block partials;
// pass 2: one workgroup reduces them in a fixed order (no atomics).
constexpr int kFeatPart = 9;
__global__ void __launch_bounds__(kBlock) k_guard_feat_part(Dev d, StepParams sp, double disp, double* part) {
  __shared__ double red[kFeatPart][kBlock];
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  const int t = threadIdx.x;
  double v[kFeatPart] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (b < d.nb) {
    const BodyKin& P = d.kin[b];
    const double vn = sqrt(vnorm2(kvel(P))), wn = sqrt(vnorm2(kvrot(P))), an = sqrt(vnorm2(ld3(d.acc + 3 * (size_t)b)));
    const double dx = d.gdpos ? sqrt(vnorm2(ld3(d.gdpos + 3 * (size_t)b))) : 0.0;
    v[0] = vn;                                     // max |v|
    v[1] = vn;                                     // sum |v|
    v[2] = vn * vn;                                // sum |v|^2
    v[3] = wn;                                     // max |w|
    v[4] = wn;                                     // sum |w|
    v[5] = an;                                     // max |a|
    v[6] = an;                                     // sum |a|
    v[7] = dx;                                     // sum |dx|
    v[8] = (vn * sp.dt > 0.01 * disp) ? 1.0 : 0.0;  // moving bodies
  }
  for (int k = 0; k < kFeatPart; k++) red[k][t] = (v[k] == v[k]) ? v[k] : 0.0;
  __syncthreads();
  for (int h = kBlock / 2; h > 0; h >>= 1) {
    if (t < h)
      for (int k = 0; k < kFeatPart; k++) {
        const bool mx = (k == 0 || k == 3 || k == 5);
        red[k][t] = mx ? fmax(red[k][t], red[k][t + h]) : red[k][t] + red[k][t + h];
      }
    __syncthreads();
  }
  if (t < kFeatPart) part[(size_t)blockIdx.x * kFeatPart + t] = red[t][0];
}

__global__ void __launch_bounds__(kBlock) k_guard_feat_final(Dev d, StepParams sp, const double* part, int nparts,
                                                             double disp, double angle, long long since,
                                                             long long last, float* feat) {
  // thread t takes the partials t, t + 256, ... in turn, then a fixed tree
  // over the threads (the same order whatever the scheduling)
  __shared__ double red[kFeatPart][kBlock];
  const int t = threadIdx.x;
  double a[kFeatPart] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int q = t; q < nparts; q += kBlock)
#pragma unroll
    for (int k = 0; k < kFeatPart; k++) {
      const double x = part[(size_t)q * kFeatPart + k];
      const bool mx = (k == 0 || k == 3 || k == 5);
      a[k] = mx ? fmax(a[k], x) : a[k] + x;
    }
#pragma unroll
  for (int k = 0; k < kFeatPart; k++) red[k][t] = a[k];
  for (int h = kBlock / 2; h > 0; h >>= 1) {
    __syncthreads();
    if (t < h)
#pragma unroll
      for (int k = 0; k < kFeatPart; k++) {
        const bool mx = (k == 0 || k == 3 || k == 5);
        red[k][t] = mx ? fmax(red[k][t], red[k][t + h]) : red[k][t] + red[k][t + h];
      }
  }
  if (t != 0) return;
#pragma unroll
  for (int k = 0; k < kFeatPart; k++) a[k] = red[k][0];
  const double nb = d.nb > 0 ? (double)d.nb : 1.0;
  const double ds = disp > 0.0 ? disp : 1.0, an = angle > 0.0 ? angle : 1.0, dt = sp.dt;
  double dxmax = 0.0, rot = 0.0;
  if (d.guard) {
    dxmax = sqrt(__longlong_as_double((long long)d.guard->maxpos2));
    if (d.guard->minw != ~0ull && d.wstar < 1.0 && d.wstar >= -1.0) {
      const unsigned long long k = d.guard->minw;
      const unsigned long long u = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
      const double w = __longlong_as_double((long long)u);
      rot = (1.0 - w) / (1.0 - d.wstar);
    }
  }
  double f[16];
  f[0] = dxmax / ds;
  f[1] = rot;
  f[2] = a[0] * dt / ds;
  f[3] = a[1] / nb * dt / ds;
  f[4] = sqrt(a[2] / nb) * dt / ds;
  f[5] = a[3] * dt / an;
  f[6] = a[4] / nb * dt / an;
  f[7] = a[5] * dt * dt / ds;
  f[8] = a[6] / nb * dt * dt / ds;
  f[9] = log1p(fmax(0.0, (1.0 - f[0]) / fmax(f[2], 1e-12))) / 10.0;
  f[10] = log1p((double)since) / 10.0;
  f[11] = log1p((double)last) / 10.0;
  f[12] = a[8] / nb;
  f[13] = a[7] / nb / ds;
  f[14] = fmin(f[2] * (double)since, 10.0);
  f[15] = 1.0;
  for (int k = 0; k < 16; k++) {
    double x = f[k] == f[k] ? f[k] : 0.0;
    x = x > 10.0 ? 10.0 : (x < -10.0 ? -10.0 : x);
    feat[k] = (float)x;
  }
}

// Particle::GlobVertex (Particle.cpp:55-57): one thread per vertex of the
// first nv vertices (every body's, or the driven bodies', which come first),
// of every body (all) or of the bodies with slots in the current list (the
// only ones the force phase reads; the list builder reads all).
__global__ void __launch_bounds__(kBlock) k_glob(Dev d, int all, int nv) {
  if (frozen(d)) return;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nv; k += gridDim.x * blockDim.x) {
    const int b = d.bvbody[k];
    if (!all && d.soff[b + 1] == d.soff[b]) continue;
    const BodyKin& P = d.kin[b];
    st3(d.gv + 3 * (size_t)k, glob_vertex(d.sh, P, k - d.bvoff[b]));
  }
}

// ServoFunction (DrivingSystem.cpp:251-494), then the controlled bodies in
// list order (Rockable.cpp:1856-1900, 1988-2033), all by one thread.  The
// tritri servos read the walls' inner faces here; the shakers' and the
// ramp's values (functions of t only) come from the host in sp.servo_v.
// The servo of the driving system (DrivingSystem.cpp:242-496): the control
// values it imposes, from the walls' positions before any control moves them.
__device__ void drive_servo(const Dev& d, const StepParams& sp) {
  const int ic = d.servo_icontr;
  if (d.servo >= 1 && d.servo <= 4 && ic + 5 < d.nctrl) {
    const int* id = d.servo_ids;
    const double Xmin = d.kin[id[0]].px + d.kin[id[0]].R;
    const double Xmax = d.kin[id[1]].px - d.kin[id[1]].R;
    const double Ymin = d.kin[id[2]].py + d.kin[id[2]].R;
    const double Ymax = d.kin[id[3]].py - d.kin[id[3]].R;
    const double Zmin = d.kin[id[4]].pz + d.kin[id[4]].R;
    const double Zmax = d.kin[id[5]].pz - d.kin[id[5]].R;
    const double dX = fabs(Xmax - Xmin), dY = fabs(Ymax - Ymin), dZ = fabs(Zmax - Zmin);
    const double surfX = dY * dZ, surfY = dX * dZ, surfZ = dY * dX;
    const double p = d.servo_pressure;
    DevControl* C = d.ctrl + ic;
    if (d.servo == 1) {  // isostatic (251-268)
      C[1].value = -p * surfX;
      C[3].value = -p * surfY;
      C[5].value = -p * surfZ;
    } else if (d.servo == 2) {  // biaxial (280-298)
      C[1].value = -p * surfX;
      C[5].value = -p * surfZ;
    } else if (d.servo == 3) {  // custom (328-353): force-driven walls only
      const double* v = d.servo_val;
      if (C[0].type == C_X_FOR) C[0].value = v[0] * surfX;
      if (C[1].type == C_X_FOR) C[1].value = -v[1] * surfX;
      if (C[2].type == C_Y_FOR) C[2].value = v[2] * surfY;
      if (C[3].type == C_Y_FOR) C[3].value = -v[3] * surfY;
      if (C[4].type == C_Z_FOR) C[4].value = v[4] * surfZ;
      if (C[5].type == C_Z_FOR) C[5].value = -v[5] * surfZ;
    } else {  // Lode angle (369-392)
      const double dSig = d.lode_rate * sp.t;
      C[1].value = -(p + dSig) * surfX;
      C[3].value = -(p + d.lode_a * dSig) * surfY;
      C[5].value = -(p + d.lode_b * dSig) * surfZ;
    }
  } else if (d.servo >= 5 && d.servo <= 7 && ic + 2 < d.nctrl) {  // shakers
    d.ctrl[ic].value = sp.servo_v[0];
    d.ctrl[ic + 1].value = sp.servo_v[1];
    d.ctrl[ic + 2].value = sp.servo_v[2];
  } else if (d.servo == 8 && ic < d.nctrl) {  // ramp
    d.ctrl[ic].value = sp.servo_v[0];
  }
}

// The controls of the predictor (Rockable.cpp:1979-2035): first the
// velocity controls of every control in list order, then the force and
// moment ones.  A control reads and writes only its own body, so the two
// passes restricted to one body give that body's state whatever the other
// bodies' controls do.
__device__ __forceinline__ void control_vel(const Dev& d, const StepParams& sp, const DevControl& C) {
  BodyKin* p = d.kin + C.i;
  switch (C.type) {
    case C_X_VEL:
      p->vx = C.value;
      p->px += sp.dt * C.value;
      break;
    case C_Y_VEL:
      p->vy = C.value;
      p->py += sp.dt * C.value;
      break;
    case C_Z_VEL:
      p->vz = C.value;
      p->pz += sp.dt * C.value;
      break;
    case C_XROT_VEL:
    case C_YROT_VEL:
    case C_ZROT_VEL:
    case C_XYZROT_VEL: {
      v3 w;
      if (C.type == C_XROT_VEL)
        w = V(C.value, 0.0, 0.0);
      else if (C.type == C_YROT_VEL)
        w = V(0.0, C.value, 0.0);
      else if (C.type == C_ZROT_VEL)
        w = V(0.0, 0.0, C.value);
      else
        w = V(C.vx, C.vy, C.vz);
      qt Q = kq(*p);
      Q = qadd_scaled(Q, qdot(Q, w), sp.dt);
      qnormalize(&Q);
      p->qw = Q.w;
      p->qx = Q.x;
      p->qy = Q.y;
      p->qz = Q.z;
    } break;
    default: break;
  }
}
__device__ __forceinline__ void control_force(const Dev& d, const StepParams& sp, const DevControl& C) {
  BodyKin* p = d.kin + C.i;
  const double* a = d.acc + 3 * (size_t)C.i;
  const double* ar = d.arot + 3 * (size_t)C.i;
  switch (C.type) {
    case C_X_FOR:
      p->px += sp.dt * p->vx + sp.dt2_2 * a[0];
      p->vx += sp.dt_2 * a[0];
      break;
    case C_Y_FOR:
      p->py += sp.dt * p->vy + sp.dt2_2 * a[1];
      p->vy += sp.dt_2 * a[1];
      break;
    case C_Z_FOR:
      p->pz += sp.dt * p->vz + sp.dt2_2 * a[2];
      p->vz += sp.dt_2 * a[2];
      break;
    case C_XROT_MOM:
    case C_YROT_MOM:
    case C_ZROT_MOM:
    case C_XYZROT_MOM: {
      v3 w;
      if (C.type == C_XROT_MOM)
        w = V(p->wx * 1.0, p->wx * 0.0, p->wx * 0.0);
      else if (C.type == C_YROT_MOM)
        w = V(p->wy * 0.0, p->wy * 1.0, p->wy * 0.0);
      else if (C.type == C_ZROT_MOM)
        w = V(p->wz * 0.0, p->wz * 0.0, p->wz * 1.0);
      else
        w = V(p->wx, p->wy, p->wz);
      qt Q = kq(*p);
      Q = qadd_scaled(Q, qdot(Q, w), sp.dt);
      qnormalize(&Q);
      p->qw = Q.w;
      p->qx = Q.x;
      p->qy = Q.y;
      p->qz = Q.z;
      if (C.type == C_XROT_MOM)
        p->wx += sp.dt_2 * ar[0];
      else if (C.type == C_YROT_MOM)
        p->wy += sp.dt_2 * ar[1];
      else if (C.type == C_ZROT_MOM)
        p->wz += sp.dt_2 * ar[2];
      else {
        v3 nw = vadd(V(p->wx, p->wy, p->wz), vsc(sp.dt_2, V(ar[0], ar[1], ar[2])));
        p->wx = nw.x;
        p->wy = nw.y;
        p->wz = nw.z;
      }
    } break;
    default: break;
  }
}

// All controls by one thread in list order (the servo first).
__device__ void drive_controls(const Dev& d, const StepParams& sp) {
  drive_servo(d, sp);
  for (int c = 0; c < d.nctrl; c++) control_vel(d, sp, d.ctrl[c]);
  for (int c = 0; c < d.nctrl; c++) control_force(d, sp, d.ctrl[c]);
}

// The controls by the threads of one workgroup (every thread calls it): the
// servo by thread 0, then each driven body's controls in list order by one
// thread (ctrl_parallel: every control acts on a driven body), else all of
// them by thread 0.
__device__ void drive_controls_block(const Dev& d, const StepParams& sp) {
  if (d.nctrl <= 0) return;
  if (!d.ctrl_parallel) {
    if (threadIdx.x == 0) drive_controls(d, sp);
    return;
  }
  if (threadIdx.x == 0) drive_servo(d, sp);
  __syncthreads();  // the servo's values are read by the other threads
  for (int b = threadIdx.x; b < d.nDriven; b += blockDim.x) {
    const int q0 = d.ctrl_off[b], q1 = d.ctrl_off[b + 1];
    for (int q = q0; q < q1; q++) control_vel(d, sp, d.ctrl[d.ctrl_idx[q]]);
    for (int q = q0; q < q1; q++) control_force(d, sp, d.ctrl[d.ctrl_idx[q]]);
  }
}

__device__ __forceinline__ void store_predicted(const Dev& d, int b, const BodyKin& P) {
  BodyKin* out = d.kin + b;
  out->px = P.px;
  out->py = P.py;
  out->pz = P.pz;
  out->qw = P.qw;
  out->qx = P.qx;
  out->qy = P.qy;
  out->qz = P.qz;
  out->vx = P.vx;
  out->vy = P.vy;
  out->vz = P.vz;
  out->wx = P.wx;
  out->wy = P.wy;
  out->wz = P.wz;
}

// The driven bodies of the next step, where the resultant kernel took the
// free bodies' predictor: their controls, and their listed vertices (with
// driven_glob; else k_glob follows).
__global__ void __launch_bounds__(kBlock) k_drive(Dev d, StepParams sp, int driven_glob) {
  if (frozen(d)) return;
  drive_controls_block(d, sp);
  if (!driven_glob) return;
  __syncthreads();
  for (int k = threadIdx.x; k < d.nvdriven; k += blockDim.x) {
    const int b = d.bvbody[k];
    if (d.soff[b + 1] == d.soff[b]) continue;
    const BodyKin& P = d.kin[b];
    st3(d.gv + 3 * (size_t)k, glob_vertex(d.sh, P, k - d.bvoff[b]));
  }
}

// glob: also the global vertices of the free bodies with listed slots, from
// the new pose (the driven bodies' follow in k_glob)
__global__ void __launch_bounds__(kBlock) k_predict(Dev d, StepParams sp, int glob, int par) {
  if (frozen(d)) return;
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x == 0) drive_controls_block(d, sp);
  driven_bounds(d, sp, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x, par);
  // free bodies (Rockable.cpp:2036-2055), a grid-stride loop
  for (int b = gid; b < d.nb; b += gridDim.x * blockDim.x) {
    if (b < d.nDriven) continue;
    BodyKin P = d.kin[b];
    const BodyKin old = P;
    predict_free(d, sp, b, P);
    store_predicted(d, b, P);
    add_motion_bound(d, sp, b, old, P, par);
    if (glob && d.soff[b + 1] != d.soff[b]) {
      const int v0 = d.bvoff[b], nv = d.bvoff[b + 1] - v0;
      for (int v = 0; v < nv; v++) st3(d.gv + 3 * (size_t)(v0 + v), glob_vertex(d.sh, P, v));
    }
  }
}

// The predictor by workgroups of 64 free bodies.  The tile's 64 body records
// (128 bytes each) are read and written whole by the 256 threads in
// contiguous doubles through LDS (17 doubles per record there, so that the
// per-body reads spread over the banks); one thread per body computes its
// new state in between and keeps the pose in LDS; then the 256 threads share
// those bodies' vertices (global vertices of the listed ones).  Rewriting a
// record's unchanged fields (R, h, shape, group) stores the bits it read.
// The driven bodies' motion bounds are kept by the wavefronts that wait for the
// first one (ahead of the bodies they took 1.4 us of a step of 300 hulls).
// The driven bodies are moved by thread 0 of workgroup 0 (controls); with
// driven_glob, workgroup 0 then writes their listed global vertices (else
// k_glob does after this kernel).
__global__ void __launch_bounds__(kBlock) k_predict_blk(Dev d, StepParams sp, int driven_glob, int par) {
  __shared__ double rec[64 * kRec];
  __shared__ double pose[64][8];    // px py pz qw qx qy qz h
  __shared__ int shp[64];           // shape, or -1 if the body is not listed
  if (frozen(d)) return;
  const int t = threadIdx.x;
  if (blockIdx.x == 0) {
    drive_controls_block(d, sp);
    if (driven_glob) {
      __syncthreads();  // the driven poses, written by thread 0, are visible to the workgroup
      for (int k = t; k < d.nvdriven; k += blockDim.x) {
        const int b = d.bvbody[k];
        if (d.soff[b + 1] == d.soff[b]) continue;
        const BodyKin& P = d.kin[b];
        st3(d.gv + 3 * (size_t)k, glob_vertex(d.sh, P, k - d.bvoff[b]));
      }
    }
  }
  const int nfree = d.nb - d.nDriven;
  for (int tile = blockIdx.x; tile * 64 < nfree; tile += gridDim.x) {
    const int b0 = d.nDriven + tile * 64;
    const int bend = min(b0 + 64, d.nb);
    const int nd = 16 * (bend - b0);
    double* kd = reinterpret_cast<double*>(d.kin + b0);
    for (int k = t; k < nd; k += blockDim.x) rec[(k >> 4) * kRec + (k & 15)] = kd[k];
    // the body's other inputs loaded with the records, so that their
    // latencies overlap
    v3 acc = V(0.0, 0.0, 0.0), arot = acc;
    double cb = 0.0, rmx = 0.0, lim = 0.0;
    v3 drift = acc;
    bool listed = false;
    if (t < 64 && b0 + t < bend) {
      const int b = b0 + t;
      acc = ld3(d.acc + 3 * (size_t)b);
      arot = ld3(d.arot + 3 * (size_t)b);
      if (d.skip_far) {
        cb = d.cbound[b];
        rmx = d.rmax[b];
        lim = d.climit[b];
        drift = ld3(d.drift);
      }
      listed = d.soff[b + 1] != d.soff[b];
    }
    // a driven body's for a thread of the other wavefronts
    const int db = (int)blockIdx.x * (kBlock - 64) + t - 64;
    const bool drv = t >= 64 && tile == (int)blockIdx.x && db < d.nDriven && d.skip_far;
    if (drv) {
      cb = d.cbound[db];
      lim = d.climit[db];
      drift = ld3(d.drift);
    }
    __syncthreads();
    if (t < 64) {
      const int b = b0 + t;
      shp[t] = -1;
      if (b < bend) {
        double* r = rec + t * kRec;
        BodyKin P = rec_load(r);
        const BodyKin old = P;
        predict_free_with(sp, P, acc, arot);
        rec_store_motion(r, P);
        add_motion_bound_with(d, sp, b, old, P, cb, rmx, lim, drift, par);
        if (listed) {
          pose[t][0] = P.px;
          pose[t][1] = P.py;
          pose[t][2] = P.pz;
          pose[t][3] = P.qw;
          pose[t][4] = P.qx;
          pose[t][5] = P.qy;
          pose[t][6] = P.qz;
          pose[t][7] = P.h;
          shp[t] = P.shape;
        }
      }
    } else if (drv) {
      driven_bound(d, sp, db, cb, lim, drift, par);
      const int stride = (int)gridDim.x * (kBlock - 64);
      driven_bounds(d, sp, db + stride, stride, par);
    }
    __syncthreads();
    for (int k = t; k < nd; k += blockDim.x) kd[k] = rec[(k >> 4) * kRec + (k & 15)];
    for (int k = d.bvoff[b0] + t; k < d.bvoff[bend]; k += blockDim.x) {
      const int b = d.bvbody[k], lb = b - b0;
      if (shp[lb] < 0) continue;
      BodyKin P;
      P.px = pose[lb][0];
      P.py = pose[lb][1];
      P.pz = pose[lb][2];
      P.qw = pose[lb][3];
      P.qx = pose[lb][4];
      P.qy = pose[lb][5];
      P.qz = pose[lb][6];
      P.h = pose[lb][7];
      P.shape = shp[lb];
      st3(d.gv + 3 * (size_t)k, glob_vertex(d.sh, P, k - d.bvoff[b]));
    }
    __syncthreads();
  }
}

// The predictor with one thread per vertex of the free bodies, each
// wavefront holding whole bodies (wavefront w: vertices [wvstart[w],
// wvstart[w + 1])): every lane computes its body's new state, the lane of
// vertex 0 stores it and every lane of a listed body its global vertex.  The
// lanes of a body read its old state in the same load instruction, before
// any of them stores, so the body is read whole before it is overwritten.
// The driven bodies (controls by thread 0) and their vertices are left to
// k_glob after it.
__global__ void __launch_bounds__(kBlock) k_predict_vtx(Dev d, StepParams sp, int par) {
  if (frozen(d)) return;
  if (blockIdx.x == 0) drive_controls_block(d, sp);
  driven_bounds(d, sp, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x, par);
  const int lane = threadIdx.x & 63;
  for (int wv = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6); wv < d.nwv;
       wv += (int)((gridDim.x * blockDim.x) >> 6)) {
    const int k = d.wvstart[wv] + lane;
    if (k >= d.wvstart[wv + 1]) continue;
    const int b = d.bvbody[k];
    const int v = k - d.bvoff[b];
    const bool listed = d.soff[b + 1] != d.soff[b];
    if (v != 0 && !listed) continue;
    BodyKin P = d.kin[b];
    const BodyKin old = P;
    predict_free(d, sp, b, P);
    if (v == 0) {
      store_predicted(d, b, P);
      add_motion_bound(d, sp, b, old, P, par);
    }
    if (listed) st3(d.gv + 3 * (size_t)k, glob_vertex(d.sh, P, v));
  }
}

// The bodies' state as the arrays the caller reads: pos, Q, vel and vrot (13
// doubles a body), with all also acc, arot, force and moment (25).  One thread
// per double written, in order: out may lie in host memory, which is written
// in whole lines then.
__global__ void __launch_bounds__(kBlock) k_pack_bodies(Dev d, double* out, int all) {
  const long nb = d.nb, n = (all ? 25l : 13l) * nb;
  const double* kin = reinterpret_cast<const double*>(d.kin);
  for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long)gridDim.x * blockDim.x) {
    double x;
    if (k < 3 * nb) {
      x = kin[16 * (k / 3) + k % 3];
    } else if (k < 7 * nb) {
      const long q = k - 3 * nb;
      x = kin[16 * (q / 4) + 3 + q % 4];
    } else if (k < 13 * nb) {
      const long q = k - 7 * nb, at = q < 3 * nb ? 7 : 10, r = q < 3 * nb ? q : q - 3 * nb;
      x = kin[16 * (r / 3) + at + r % 3];
    } else {
      const long q = k - 13 * nb;
      x = q < 3 * nb ? d.acc[q] : q < 6 * nb ? d.arot[q - 3 * nb] : q < 9 * nb ? d.force[q - 6 * nb] : d.moment[q - 9 * nb];
    }
    out[k] = x;
  }
}

// The active entries' records for a read-out, in entry order: counts per
// block of 1024 entries, their scan by one workgroup, the records.  The host
// copies only those (176 bytes each) instead of every listed entry's arrays
// (206 bytes, one in ten active in a settled packing).
constexpr int kActiveTile = 1024;
__global__ void __launch_bounds__(kBlock) k_active_count(Dev d, int32_t* block) {
  __shared__ int w[kBlock / 64];
  int n = 0;
  for (int r = 0; r < kActiveTile / kBlock; r++) {
    const int e = blockIdx.x * kActiveTile + r * kBlock + (int)threadIdx.x;
    n += __popcll(__ballot(e < d.ne && (d.eact[e] & 1)));
  }
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = n;
  __syncthreads();
  if (threadIdx.x == 0) block[blockIdx.x] = w[0] + w[1] + w[2] + w[3];
}
// exclusive, in place; the total after the last block's
__global__ void __launch_bounds__(kBlock) k_active_scan(int n, int32_t* block) {
  __shared__ int sc[kBlock];
  const int t = threadIdx.x;
  int carry = 0;
  for (int b0 = 0; b0 < n; b0 += kBlock) {
    const int v = b0 + t < n ? block[b0 + t] : 0;
    sc[t] = v;
    for (int o = 1; o < kBlock; o <<= 1) {
      __syncthreads();
      const int x = t >= o ? sc[t - o] : 0;
      __syncthreads();
      sc[t] += x;
    }
    __syncthreads();
    if (b0 + t < n) block[b0 + t] = carry + sc[t] - v;
    carry += sc[kBlock - 1];
    __syncthreads();
  }
  if (t == 0) block[n] = carry;
}
__global__ void __launch_bounds__(kBlock) k_active_records(Dev d, const int32_t* block, rk_interaction* out, int cap) {
  __shared__ int w[kActiveTile / kBlock][kBlock / 64];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  unsigned long long mask[kActiveTile / kBlock];
#pragma unroll
  for (int r = 0; r < kActiveTile / kBlock; r++) {
    const int e = blockIdx.x * kActiveTile + r * kBlock + t;
    mask[r] = __ballot(e < d.ne && (d.eact[e] & 1));
    if (lane == 0) w[r][wv] = __popcll(mask[r]);
  }
  __syncthreads();
  int base = block[blockIdx.x];
#pragma unroll
  for (int r = 0; r < kActiveTile / kBlock; r++) {
    int before = 0, tot = 0;
    for (int q = 0; q < kBlock / 64; q++) {
      before += q < wv ? w[r][q] : 0;
      tot += w[r][q];
    }
    const int e = blockIdx.x * kActiveTile + r * kBlock + t;
    const int k = base + before + __popcll(mask[r] & ((1ull << lane) - 1ull));
    base += tot;
    if (!(mask[r] >> lane & 1ull) || k >= cap) continue;
    rk_interaction o;
    const uint32_t sub = d.esub[e];
    const EState s = d.est[e];
    const EGeom g = d.egeo[e];
    o.i = d.ei[e];
    o.j = d.ej[e];
    o.type = (int32_t)(sub >> 30);
    o.isub = (int32_t)((sub >> 15) & 0x7fffu);
    o.jsub = (int32_t)(sub & 0x7fffu);
    o.stick = d.estick[e];
    o.n[0] = g.nx;
    o.n[1] = g.ny;
    o.n[2] = g.nz;
    o.dn = d.edn[e];
    o.pos[0] = g.px;
    o.pos[1] = g.py;
    o.pos[2] = g.pz;
    o.vel[0] = g.vx;
    o.vel[1] = g.vy;
    o.vel[2] = g.vz;
    o.fn = s.fn;
    o.ft[0] = s.ftx;
    o.ft[1] = s.fty;
    o.ft[2] = s.ftz;
    o.mom[0] = s.momx;
    o.mom[1] = s.momy;
    o.mom[2] = s.momz;
    o.damp = d.edamp[e];
    out[k] = o;
  }
}

}  // namespace

int body_block(const Dev& d) { return d.body_block == 64 || d.body_block == 128 ? d.body_block : 256; }

// workgroups for T tiles (persistent kernels loop over their tiles)
dim3 grid_for(const Dev& d, long T) { return dim3(persistent_grid((int)std::max(1L, T), d.persist)); }

void launch_glob(const Dev& d, int all, int nv, hipStream_t s) {
  if (nv <= 0) return;
  const int bs = body_block(d);
  hipLaunchKernelGGL(k_glob, grid_for(d, (nv + bs - 1) / bs), dim3(bs), 0, s, d, all || !d.soff ? 1 : 0, nv);
}

void launch_glob(const Dev& d, int all, hipStream_t s) { launch_glob(d, all, d.nvtot, s); }

void launch_refresh_gaps(const Dev& d, hipStream_t s) {
  if (d.ne <= 0 || !d.skip_far) return;
  hipLaunchKernelGGL(k_refresh_gaps, dim3(std::min((d.ne + kBlock - 1) / kBlock, 65536)), dim3(kBlock), 0, s, d);
}

void launch_reset_keys(const Dev& d, hipStream_t s) {
  if (d.ne <= 0 || !d.ekey) return;
  hipLaunchKernelGGL(k_reset_keys, dim3(std::min((d.ne + kBlock - 1) / kBlock, 65536)), dim3(kBlock), 0, s, d);
}

void launch_entry_desc(const Dev& d, hipStream_t s) {
  if (d.ne <= 0 || !d.edesc) return;
  hipLaunchKernelGGL(k_entry_desc, dim3((d.ne + kBlock - 1) / kBlock), dim3(kBlock), 0, s, d);
}

void launch_predict(const Dev& d, const StepParams& sp, int glob, int par, hipStream_t s) {
  const int n = d.nb > 0 ? d.nb : 1, bs = body_block(d);
  if (glob == GLOB_NONE) {
    hipLaunchKernelGGL(k_predict, grid_for(d, (n + bs - 1) / bs), dim3(bs), 0, s, d, sp, 0, par);
    return;
  }
  par = -1;  // the step takes no list
  const bool listed = glob == GLOB_LISTED && d.soff;  // else every body's vertices
  if (listed && d.fuse_glob == 3 && d.nb > d.nDriven) {
    // workgroups of 64 free bodies, their vertices from the poses in LDS; a
    // few driven bodies' vertices by workgroup 0 after the controls
    const int tiles = (d.nb - d.nDriven + 63) / 64;
    const int driven_glob = d.nvdriven <= 1024 ? 1 : 0;
    hipLaunchKernelGGL(k_predict_blk, grid_for(d, tiles), dim3(kBlock), 0, s, d, sp, driven_glob, par);
    if (!driven_glob) launch_glob(d, 0, d.nvdriven, s);
    return;
  }
  if (listed && d.fuse_glob == 2 && d.nwv > 0) {
    // one thread per vertex of the free bodies, wavefronts of whole bodies
    const int wpb = kBlock / 64;
    hipLaunchKernelGGL(k_predict_vtx, grid_for(d, (d.nwv + wpb - 1) / wpb), dim3(kBlock), 0, s, d, sp, par);
    launch_glob(d, 0, d.nvdriven, s);
    return;
  }
  const int fused = listed && d.fuse_glob != 0;  // the free bodies' in k_predict
  hipLaunchKernelGGL(k_predict, grid_for(d, (n + bs - 1) / bs), dim3(bs), 0, s, d, sp, fused, par);
  launch_glob(d, listed ? 0 : 1, fused ? d.nvdriven : d.nvtot, s);
}

void launch_pack_bodies(const Dev& d, double* out, int all, hipStream_t s) {
  const long n = ((all ? 25l : 13l) * d.nb + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(k_pack_bodies, dim3((int)std::min(n, 65536L)), dim3(kBlock), 0, s, d, out, all);
}

int active_blocks(const Dev& d) { return (d.ne + kActiveTile - 1) / kActiveTile; }

void launch_active_count(const Dev& d, int32_t* block, hipStream_t s) {
  const int n = active_blocks(d);
  if (n > 0) hipLaunchKernelGGL(k_active_count, dim3(n), dim3(kBlock), 0, s, d, block);
  hipLaunchKernelGGL(k_active_scan, dim3(1), dim3(kBlock), 0, s, n, block);
}

void launch_active_records(const Dev& d, const int32_t* block, rk_interaction* out, int cap, hipStream_t s) {
  const int n = active_blocks(d);
  if (n > 0 && cap > 0) hipLaunchKernelGGL(k_active_records, dim3(n), dim3(kBlock), 0, s, d, block, out, cap);
}

void launch_drive(const Dev& d, const StepParams& sp, int glob, hipStream_t s) {
  if (d.nctrl <= 0) return;  // no body moves by a control: poses and vertices stay
  const int driven_glob = glob != GLOB_NONE && d.nvdriven <= 1024 ? 1 : 0;
  hipLaunchKernelGGL(k_drive, dim3(1), dim3(kBlock), 0, s, d, sp, driven_glob);
  if (glob != GLOB_NONE && !driven_glob) launch_glob(d, 0, d.nvdriven, s);
}

template <int BS>
void launch_geom(const Dev& d, int write_geom_all, hipStream_t s) {
  const dim3 g = grid_for(d, (d.ne + BS - 1) / BS), bl(BS);
  if (write_geom_all)
    hipLaunchKernelGGL((k_geom<true, BS>), g, bl, 0, s, d);
  else
    hipLaunchKernelGGL((k_geom<false, BS>), g, bl, 0, s, d);
}

template <bool GEOM_ALL, bool SORT>
void launch_fused_sorted(const Dev& d, const StepParams& sp, int write_geom_all, hipStream_t s) {
  const dim3 g = grid_for(d, (d.ne + kBlock - 1) / kBlock), bl(kBlock);
  if (sp.law == LAW_AVALANCHE)
    hipLaunchKernelGGL((k_interact<LAW_AVALANCHE, GEOM_ALL, SORT>), g, bl, 0, s, d, sp, write_geom_all, 0);
  else if (sp.law == LAW_STICKED)
    hipLaunchKernelGGL((k_interact<LAW_STICKED, GEOM_ALL, SORT>), g, bl, 0, s, d, sp, write_geom_all,
                       d.paramsInInterfaces);
  else
    hipLaunchKernelGGL((k_interact<LAW_DEFAULT, GEOM_ALL, SORT>), g, bl, 0, s, d, sp, write_geom_all, 0);
}

bool uses_list(const Dev& d, int write_geom_all) {
  return !write_geom_all && d.fuse_law && d.skip_far && d.skip_seg >= 512 && (d.elist || d.ne <= 0);
}

// The grid of the list kernel: a lane for each second entry (a list holds a
// tenth to a third of them, bonds more), up to 2048 workgroups, twice what
// the chip holds of it; a multiple of 8, so that every XCD part has its
// workgroups.  Up to 256 workgroups a lane for every entry of a part's tiles,
// so that a small list, whose few tiles fill some parts only, is done in one
// round however much of it is listed: at a lane for two entries the 3 660 of
// a plate pressed on 900 spheres took 17.4 us, so 9.5 (12.7 by the per-step
// test of every entry), the 1 650 of 517 spheres 8.3 and 6.7 us.
void launch_list(const Dev& d, const StepParams& sp, int par, hipStream_t s) {
  const long tiles = ((long)d.ne + kListTile - 1) / kListTile;
  const long round = std::min(256L, (tiles + 7) / 8 * (8 * kListTile / kBlock));
  const long want = std::max(round, ((long)d.ne + 2 * kBlock - 1) / (2 * kBlock));
  const int g = (int)std::min(2048L, (want + 7) & ~7L);
  const dim3 grid(std::max(8, persistent_grid(g, d.persist))), bl(kBlock);
  if (d.skip_count) hipLaunchKernelGGL(k_count_skips, dim3(std::min((d.ne + kBlock - 1) / kBlock, 2048)), bl, 0, s, d);
  if (sp.law == LAW_AVALANCHE)
    hipLaunchKernelGGL((k_interact_list<LAW_AVALANCHE>), grid, bl, 0, s, d, sp, 0, par);
  else if (sp.law == LAW_STICKED)
    hipLaunchKernelGGL((k_interact_list<LAW_STICKED>), grid, bl, 0, s, d, sp, d.paramsInInterfaces, par);
  else
    hipLaunchKernelGGL((k_interact_list<LAW_DEFAULT>), grid, bl, 0, s, d, sp, 0, par);
}

template <bool GEOM_ALL>
void launch_fused(const Dev& d, const StepParams& sp, int write_geom_all, hipStream_t s) {
  if (d.type_sort)
    launch_fused_sorted<GEOM_ALL, true>(d, sp, write_geom_all, s);
  else
    launch_fused_sorted<GEOM_ALL, false>(d, sp, write_geom_all, s);
}

void launch_interact(const Dev& d, const StepParams& sp, int write_geom_all, int par, hipStream_t s) {
  if (d.ne <= 0) return;
  if (uses_list(d, write_geom_all)) {
    launch_list(d, sp, par, s);
    return;
  }
  if (d.fuse_law) {
    if (write_geom_all)
      launch_fused<true>(d, sp, write_geom_all, s);
    else
      launch_fused<false>(d, sp, write_geom_all, s);
    return;
  }
  switch (d.geom_block) {
    case 64: launch_geom<64>(d, write_geom_all, s); break;
    case 128: launch_geom<128>(d, write_geom_all, s); break;
    case 512: launch_geom<512>(d, write_geom_all, s); break;
    default: launch_geom<256>(d, write_geom_all, s); break;
  }
  const dim3 bl(kBlock);
  // W geometry blocks per wavefront
  const int gbs = (d.geom_block == 64 || d.geom_block == 128 || d.geom_block == 512) ? d.geom_block : 256;
  const int ngeom = (d.ne + gbs - 1) / gbs;
  const int W = std::min(std::max(d.law_group, 1), kLawGroup);
  const int waves = (ngeom + W - 1) / W;
  const dim3 gl = grid_for(d, (waves + kBlock / 64 - 1) / (kBlock / 64));
  if (sp.law == LAW_AVALANCHE)
    hipLaunchKernelGGL(k_law<LAW_AVALANCHE>, gl, bl, 0, s, d, sp, write_geom_all, 0, ngeom, W);
  else if (sp.law == LAW_STICKED)
    hipLaunchKernelGGL(k_law<LAW_STICKED>, gl, bl, 0, s, d, sp, write_geom_all, d.paramsInInterfaces, ngeom, W);
  else
    hipLaunchKernelGGL(k_law<LAW_DEFAULT>, gl, bl, 0, s, d, sp, write_geom_all, 0, ngeom, W);
}

// k_gather's free bodies per workgroup: 32, so that a small packing spreads
// over more workgroups and a bonded body's many terms fit one LDS pass; 64
// from 131 072 bodies, where workgroups abound and the lanes that finish
// the bodies count.  64 against 32, 128 threads: 33.5 and 44.0 us for 288 005
// spheres, 35.8 and 39.9 us for 160 005 hulls, 89.2 and 91.7 us for 200 001
// bonded cubes.
constexpr int kGatherLarge = 1 << 17;
bool gather_many(const Dev& d) { return d.nDriven >= kDrivenMany; }
int gather_bodies(const Dev& d) { return !gather_many(d) && d.nb - d.nDriven >= kGatherLarge ? 64 : 32; }

// and its threads: 256 where all workgroups are resident at once anyway (up to
// 1024 of them) or bodies have many slots, whose terms then take fewer passes;
// 128 where workgroups queue, since only one wavefront finishes the bodies and
// the others' places are worth more to a second workgroup.  256 against 128:
// 12.9 and 16.2 us for 13 001 bonded cubes (63 slots each), 9.7 and 10.5 us
// for 706 hulls, but 28.7 and 22.7 us for the 90 006-body slope (45 slots),
// 12.3 and 9.2 us for 47 000 spheres.  At 63 slots the many groups of 100 001
// cubes take 51.9 and 55.1 us, those of 40 001 26.9 and 24.5: the line on
// slots lies between what was measured, not at a crossing.
int gather_threads(const Dev& d) {
  if (gather_bodies(d) == 64 || gather_many(d)) return 128;
  const bool few = (d.nb - d.nDriven + 31) / 32 <= 1024, many_slots = 2.0 * d.ne > 56.0 * d.nb;
  return few || many_slots ? 256 : 128;
}

// k_gather's workgroups: the driven bodies, the heavy chunks one to a
// wavefront, the free bodies
int gather_blocks(const Dev& d, int fuse) {
  const int nb = gather_bodies(d), wv = gather_threads(d) / 64;
  const int per = gather_many(d) ? driven_per(d.nDriven) : 1;
  return (d.nDriven + per - 1) / per + (fuse ? 0 : (d.nhch + wv - 1) / wv) + (d.nb - d.nDriven + nb - 1) / nb;
}

int gather_blocks_max(int nb, int nhch) { return nb + (nhch + 1) / 2 + 8; }

void launch_gather(const Dev& d, const StepParams& sp, GatherArgs A, hipStream_t s) {
  if (d.nb <= 0) return;
  A.guard = A.guard && A.kick;
  const int kick = A.kick, guard = A.guard;
  const dim3 blocks(gather_blocks(d, A.fuse));
  const bool bf = d.bf != BF_NONE, large = gather_bodies(d) == 64, wide = gather_threads(d) == 256;
  if (gather_many(d) && bf)
    hipLaunchKernelGGL((k_gather<128, 32, true, true>), blocks, dim3(128), 0, s, d, sp, A);
  else if (gather_many(d))
    hipLaunchKernelGGL((k_gather<128, 32, false, true>), blocks, dim3(128), 0, s, d, sp, A);
  else if (large && bf)
    hipLaunchKernelGGL((k_gather<128, 64, true, false>), blocks, dim3(128), 0, s, d, sp, A);
  else if (large)
    hipLaunchKernelGGL((k_gather<128, 64, false, false>), blocks, dim3(128), 0, s, d, sp, A);
  else if (wide && bf)
    hipLaunchKernelGGL((k_gather<256, 32, true, false>), blocks, dim3(256), 0, s, d, sp, A);
  else if (wide)
    hipLaunchKernelGGL((k_gather<256, 32, false, false>), blocks, dim3(256), 0, s, d, sp, A);
  else if (bf)
    hipLaunchKernelGGL((k_gather<128, 32, true, false>), blocks, dim3(128), 0, s, d, sp, A);
  else
    hipLaunchKernelGGL((k_gather<128, 32, false, false>), blocks, dim3(128), 0, s, d, sp, A);
  if (d.nheavy > 0 && !A.fuse) {
    hipLaunchKernelGGL(k_heavy_finish, grid_for(d, d.nheavy), dim3(kBlock), 0, s, d, sp, kick, guard);
    if (d.nheavy_exact > 0)
      hipLaunchKernelGGL(k_gather_heavy, dim3(d.nheavy), dim3(kBlock), 0, s, d, sp, kick, guard);
  }
}

// --- statistics of the packing (DataExtractor-style quantities) -----------
// Partial sums per workgroup (a fixed tree in LDS), then one workgroup
// reduces the partials in a fixed order: the results do not depend on
// scheduling.
constexpr int kStatBody = 4;   // KE translation, KE rotation, max |v|, free bodies
constexpr int kStatEntry = 5;  // active, contacts (dn < 0), active pairs, sum dn, min dn

__device__ __forceinline__ void stat_block_reduce(double (*red)[kBlock], int nval, const int* is_max, int t) {
  __syncthreads();
  for (int h = kBlock / 2; h > 0; h >>= 1) {
    if (t < h)
      for (int k = 0; k < nval; k++)
        red[k][t] = is_max[k] == 1   ? fmax(red[k][t], red[k][t + h])
                    : is_max[k] == 2 ? fmin(red[k][t], red[k][t + h])
                                     : red[k][t] + red[k][t + h];
    __syncthreads();
  }
}

__global__ void __launch_bounds__(kBlock) k_stat_bodies(Dev d, double* part) {
  __shared__ double red[kStatBody][kBlock];
  const int t = threadIdx.x;
  const int b = blockIdx.x * kBlock + t;
  double v[kStatBody] = {0.0, 0.0, 0.0, 0.0};
  if (b < d.nb && b >= d.nDriven) {
    const BodyKin P = d.kin[b];
    const double m = d.mass[b];
    const v3 I = ld3(d.inertia + 3 * (size_t)b);
    const v3 vel = kvel(P);
    const v3 wb = qrot(qconj(kq(P)), kvrot(P));
    const double v2 = vdot(vel, vel);
    v[0] = 0.5 * m * v2;
    v[1] = 0.5 * (I.x * wb.x * wb.x + I.y * wb.y * wb.y + I.z * wb.z * wb.z);
    v[2] = sqrt(v2);
    v[3] = 1.0;
  }
  for (int k = 0; k < kStatBody; k++) red[k][t] = v[k];
  const int ops[kStatBody] = {0, 0, 1, 0};
  stat_block_reduce(red, kStatBody, ops, t);
  if (t < kStatBody) part[(size_t)blockIdx.x * kStatBody + t] = red[t][0];
}

__global__ void __launch_bounds__(kBlock) k_stat_entries(Dev d, double* part) {
  __shared__ double red[kStatEntry][kBlock];
  const int t = threadIdx.x;
  const int e = blockIdx.x * kBlock + t;
  double v[kStatEntry] = {0.0, 0.0, 0.0, 0.0, INFINITY};
  if (e < d.ne && (d.eact[e] & 1)) {
    const double dn = d.edn[e];
    v[0] = 1.0;
    if (dn < 0.0) {
      v[1] = 1.0;
      v[3] = dn;
      v[4] = dn;
    }
    // the first active entry of its body pair (entries are sorted by pair)
    bool head = true;
    const int i = d.ei[e], j = d.ej[e];
    for (int k = e - 1; k >= 0 && d.ei[k] == i && d.ej[k] == j; k--)
      if (d.eact[k] & 1) {
        head = false;
        break;
      }
    v[2] = head ? 1.0 : 0.0;
  }
  for (int k = 0; k < kStatEntry; k++) red[k][t] = v[k];
  const int ops[kStatEntry] = {0, 0, 0, 0, 2};
  stat_block_reduce(red, kStatEntry, ops, t);
  if (t < kStatEntry) part[(size_t)blockIdx.x * kStatEntry + t] = red[t][0];
}

// out[0..3] body statistics, out[4..8] entry statistics
__global__ void __launch_bounds__(kBlock) k_stat_final(const double* pb, int nbp, const double* pe, int nep,
                                                       double* out) {
  // thread t takes the partials t, t + 256, ... in turn, then a fixed tree
  // over the threads (the same order whatever the scheduling)
  constexpr int NS = kStatBody + kStatEntry;
  __shared__ double red[NS][kBlock];
  const int t = threadIdx.x;
  double s[NS] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, INFINITY};
  for (int q = t; q < nbp; q += kBlock) {
    s[0] += pb[kStatBody * q];
    s[1] += pb[kStatBody * q + 1];
    s[2] = fmax(s[2], pb[kStatBody * q + 2]);
    s[3] += pb[kStatBody * q + 3];
  }
  for (int q = t; q < nep; q += kBlock) {
    for (int k = 0; k < 4; k++) s[kStatBody + k] += pe[kStatEntry * q + k];
    s[kStatBody + 4] = fmin(s[kStatBody + 4], pe[kStatEntry * q + 4]);
  }
#pragma unroll
  for (int k = 0; k < NS; k++) red[k][t] = s[k];
  for (int h = kBlock / 2; h > 0; h >>= 1) {
    __syncthreads();
    if (t < h)
#pragma unroll
      for (int k = 0; k < NS; k++) {
        const double a = red[k][t], b = red[k][t + h];
        red[k][t] = k == 2 ? fmax(a, b) : k == NS - 1 ? fmin(a, b) : a + b;
      }
  }
  __syncthreads();
  if (t < NS) out[t] = red[t][0];
}

int stat_parts(const Dev& d) {
  return std::max(1, (d.nb + kBlock - 1) / kBlock) * kStatBody + std::max(1, (d.ne + kBlock - 1) / kBlock) * kStatEntry;
}

void launch_stats(const Dev& d, double* part, double* out, hipStream_t s) {
  const int nbp = std::max(1, (d.nb + kBlock - 1) / kBlock), nep = std::max(1, (d.ne + kBlock - 1) / kBlock);
  double* pe = part + (size_t)nbp * kStatBody;
  hipLaunchKernelGGL(k_stat_bodies, dim3(nbp), dim3(kBlock), 0, s, d, part);
  hipLaunchKernelGGL(k_stat_entries, dim3(nep), dim3(kBlock), 0, s, d, pe);
  hipLaunchKernelGGL(k_stat_final, dim3(1), dim3(kBlock), 0, s, part, nbp, pe, nep, out);
}

// Scratch of rk_get_stats_noalloc: partial sums and outputs of the
// statistics kernels in a fixed array of each device (8 MiB, held until the
// process ends), so that the call allocates nothing.  Host code never uses
// the array's name as an address: stat_scratch() looks the device address up
// once per device (hipGetSymbolAddress, with that device current) and the
// kernels receive that address.  Every call on one device shares the array;
// calls that overlap on one device race.
static __device__ __align__(256) double scratch[kStatScratchDoubles];

int stat_scratch(double** ptr, char* err, size_t errlen) {
  static std::mutex mu;
  static double* addr[64] = {};
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    snprintf(err, errlen, "stat_scratch: no current device");
    return -1;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      snprintf(err, errlen, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
      return -1;
    }
    addr[dev] = static_cast<double*>(p);
  }
  *ptr = addr[dev];
  return 0;
}

__global__ void k_guard_set_step(Dev d, long long step) {
  if (threadIdx.x == 0) d.guard->step = step;
}

void launch_guard(const Dev& d, int fuse, hipStream_t s) {
  const int nparts = (d.disp_check && d.nb > 0) ? gather_blocks(d, fuse) : 0;
  hipLaunchKernelGGL(k_guard_check, dim3(1), dim3(kCheckBlock), 0, s, d, nparts);
}

void launch_guard_set_step(const Dev& d, long long step, hipStream_t s) {
  hipLaunchKernelGGL(k_guard_set_step, dim3(1), dim3(64), 0, s, d, step);
}

void launch_guard_features(const Dev& d, const StepParams& sp, double disp, double angle, long long since,
                           long long last, double* part, float* feat, hipStream_t s) {
  const int np = std::max(1, (d.nb + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_guard_feat_part, dim3(np), dim3(kBlock), 0, s, d, sp, disp, part);
  hipLaunchKernelGGL(k_guard_feat_final, dim3(1), dim3(kBlock), 0, s, d, sp, part, np, disp, angle, since, last, feat);
}

void launch_breakage(const Dev& d, const StepParams& sp, hipStream_t s) {
  (void)sp;
  if (d.ifc.n <= 0) return;
  hipLaunchKernelGGL(k_breakage, dim3((d.ifc.n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, d);
}

}  // namespace rk
