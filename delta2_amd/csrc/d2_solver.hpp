// d2_solver.hpp -- sequential impulses of one cluster (host/device code).
//
// strategy::SequentialImpulses::solve (strategies/contact_force/
// sequential_impulses.cpp:104-638) over a cluster's filtered contacts, in
// the reference's Gauss-Seidel order (so the result is its result): setup of
// the local contacts (:109-163), impulses from
// gravity (:171-180, contact_force_strategy.cpp:10-13), warm start
// (sequential_impulses_warm_start.cpp:12-29) and its impulses (:185-213),
// the first prediction (:215-227), the normal pass (:231-375, at most 1000
// sweeps), the friction pass (:392-571, at most 100 sweeps), the new future
// states (:624-626) and the warm-store update (warm_start.cpp:31-54).
// Not computed, because nothing observable depends on them: the friction
// pass's drift terms (:432-438, :455-503; they feed only an offset impulse
// the reference never applies), unused d1 values and contact_draws.
//
// The arithmetic is in per-contact and per-particle functions (sv_*).  Two
// walks call them: solve_cluster below, one thread contact by contact (the
// device's k_sv_solve_small, a lane per cluster, and the host's check against
// the oracle), and the device's k_sv_solve, a block per cluster, which runs
// contacts that share no dynamic particle side by side.
//
// What does not change during a solve is formed once.  The torques of offset
// impulses stay zero, so a particle's predicted rotation is the same in every
// prediction (sequential_impulses.cpp:46-70 turns the future state by its own
// L): it is turned once, and a contact's local points are rotated once; a
// prediction then is v = v_f + imp / m, x = x_f + (off / m) t, L = L_f + rot.
//
// The includer defines D2_HD and includes d2_geom.hpp.  Evaluation orders
// match the oracle's restatement (dot left to right, M*v row by row, Hamilton
// products).
#pragma once

namespace d2 {

// The warm store: open addressing over 64-bit keys (lower body id << 32 |
// upper body id), EMPTY = ~0; values are the stored impulses.  Keys are
// never removed, so a lookup that meets an empty slot has missed.
constexpr unsigned long long WARM_EMPTY = ~0ull;
struct WarmTable {
  unsigned long long* keys;
  double* vals;
  unsigned long long mask;   // capacity - 1 (a power of two)
  unsigned long long* used;  // number of keys
};
D2_HD unsigned long long warm_key(int a, int b) {
  const unsigned lo = (unsigned)(a < b ? a : b), hi = (unsigned)(a < b ? b : a);
  return ((unsigned long long)lo << 32) | hi;
}
D2_HD unsigned long long warm_hash(unsigned long long k) {
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  return k;
}
D2_HD bool warm_find(const WarmTable& W, unsigned long long key, double& v) {
  for (unsigned long long h = warm_hash(key) & W.mask;; h = (h + 1) & W.mask) {
    const unsigned long long k = W.keys[h];
    if (k == key) {
      v = W.vals[h];
      return true;
    }
    if (k == WARM_EMPTY) return false;
  }
}
// Insert or overwrite (the caller keeps the load factor below one half).
D2_HD void warm_put(const WarmTable& W, unsigned long long key, double v) {
  for (unsigned long long h = warm_hash(key) & W.mask;; h = (h + 1) & W.mask) {
    unsigned long long k = W.keys[h];
    if (k == WARM_EMPTY) {
#if defined(__HIP_DEVICE_COMPILE__)
      k = atomicCAS(W.keys + h, WARM_EMPTY, key);
      if (k == WARM_EMPTY) atomicAdd(W.used, 1ull);
#else
      W.keys[h] = key;
      ++*W.used;
#endif
      if (k == WARM_EMPTY || k == key) {
        W.vals[h] = v;
        return;
      }
    } else if (k == key) {
      W.vals[h] = v;
      return;
    }
  }
}

struct SolverState {
  quat q;
  v3<double> x, v, L;
};
D2_HD SolverState sv_load(const double* r) {
  return SolverState{quat{r[0], r[1], r[2], r[3]}, {r[4], r[5], r[6]}, {r[7], r[8], r[9]}, {r[10], r[11], r[12]}};
}
D2_HD v3<double> sv_neg(v3<double> a) { return {-a.x, -a.y, -a.z}; }
// v^T M v with the row vector v^T M formed first (rn.transpose() * M * rn).
D2_HD double sv_quad(v3<double> v, const double* M) {
  const v3<double> u{(v.x * M[0] + v.y * M[3]) + v.z * M[6], (v.x * M[1] + v.y * M[4]) + v.z * M[7],
                     (v.x * M[2] + v.y * M[5]) + v.z * M[8]};
  return dot(u, v);
}
// model/forces.h:101-108: (-force) x (point - centre of mass), arm = point - centre
D2_HD v3<double> sv_torque(v3<double> f, v3<double> arm) { return cross(sv_neg(f), arm); }
D2_HD v3<double> sv_normalized(v3<double> a) {
  const double z = dot(a, a);
  return z > 0.0 ? dvs(a, sqrt(z)) : a;
}
// The rotated part of transform(p, pose(q, x)); the point is sv_turn + x (a
// rigid pose's w is 1, so the homogeneous divide changes nothing).
D2_HD v3<double> sv_turn(quat q, v3<double> p) {
  double r[9];
  qrot(q, r);
  return {(r[0] * p.x + r[1] * p.y) + r[2] * p.z, (r[3] * p.x + r[4] * p.y) + r[5] * p.z,
          (r[6] * p.x + r[7] * p.y) + r[8] * p.z};
}
// sequential_impulses.cpp:46-70 (the future state's own L drives the turn)
D2_HD SolverState sv_update(const SolverState& f, double t, v3<double> imp, v3<double> off, v3<double> rimp,
                                   v3<double> roff, double mass, const double* ii) {
  SolverState u;
  u.v = add(f.v, dvs(imp, mass));
  u.x = add(f.x, scl(dvs(off, mass), t));
  u.L = add(f.L, rimp);
  double Iw[9];
  world_inv_inertia(f.q, ii, Iw);
  const v3<double> om = mul33v(Iw, add(f.L, sclL(t, roff)));
  const v3<double> d = scl(sclL(0.5, om), t);
  quat e{1.0, 0.0, 0.0, 0.0};
  if (!(vlen(d) == 0.0)) {
    const double n = vlen(d);
    const v3<double> s = scl(dvs(d, n), (double)sin(n));
    e = quat{(double)cos(n), s.x, s.y, s.z};
  }
  u.q = qmul(e, f.q);
  return u;
}
D2_HD double sv_max(double a, double b) { return (a < b) ? b : a; }  // std::max
D2_HD double sv_min(double a, double b) { return (b < a) ? b : a; }  // std::min

// One cluster.  Inputs per hit h (the cluster's filtered contacts in gathered
// order): A, B (3 each), eps_a + eps_b and the two bodies' local indices;
// per local particle k: its body id.  `ord` receives the hits' sorted order
// (the caller sorts by proportion |A - B| / (eps_a + eps_b) with the std::sort
// replay and passes the permutation).  Scratch per hit and per particle is
// the caller's.  Returns false (nothing written) where the reference returns
// false; on success the particles' future states are written to their body
// records and out_h[11 * h] gets (normal, impulse, impulse offset, friction
// impulse, tangential velocity) for hit h (in gathered order).
struct ClusterSolve {
  // inputs
  int nh, np;
  const double* hA;    // [nh][3]
  const double* hB;    // [nh][3]
  const double* heps;  // [nh] eps_a + eps_b
  const int* hl;       // [nh][2] local particle indices of a and b
  const int* hpc;      // [nh] contacts of the hit's body pair in the cluster
  const int* ord;      // [nh] sorted order (hit ids)
  const int* pbody;    // [np] body ids
  double* bodies;      // body records (40 doubles)
  const double* mass;  // per body
  const double* fric;  // per body
  double t;
  v3<double> g;
  WarmTable warm;
  double* hs;  // scratch per hit (sorted position): [nh][CH], then [nh][CC]
  double* ps;  // scratch per particle: [np][SP]
  double* out_h;  // [nh][11]
};
// Scratch per contact: what every sweep touches (CH doubles: normal, the two
// rotated local points, outer distance, slop, effective mass, impulse, offset
// impulse, the last change of impulse, and the friction's torques of the even
// and the odd sweeps, a's then b's) and the rest (CC: local points, arms at
// the start, friction impulse, tangential velocity).  Strides of the records
// are odd, so records side by side start in different LDS banks.
constexpr int CH_N = 0, CH_WA = 3, CH_WB = 6, CH_OUTER = 9, CH_SLOP = 10, CH_MEFF = 11, CH_IMP = 12, CH_OFF = 13,
              CH_U = 14, CH_LR = 17, CH = 29;
constexpr int CC_LA = 0, CC_LB = 3, CC_RA = 6, CC_RB = 9, CC_LF = 12, CC_VT = 15, CC = 18;
constexpr int SH = CH + CC;
// Scratch per particle: predicted state, accumulated impulses, the future
// state the solve started from, mass, body-frame inverse inertia, the
// impulse at the start of the sweep, predicted rotation.
constexpr int SP_X = 0, SP_V = 3, SP_L = 6, SP_IMP = 9, SP_ROT = 12, SP_OFF = 15, SP_FX = 18, SP_FV = 21, SP_FL = 24,
              SP_MASS = 27, SP_IB = 28, SP_LAST = 37, SP_Q = 40, SP = 45;

D2_HD v3<double> ld3(const double* p) { return {p[0], p[1], p[2]}; }
D2_HD void st3(double* p, v3<double> v) { p[0] = v.x, p[1] = v.y, p[2] = v.z; }

// A local contact (:109-163) of hit h into c (CH) and k (CC); false where the
// reference gives the cluster up.
D2_HD bool sv_contact_setup(const ClusterSolve& S, int h, double* c, double* k) {
  const int ba = S.pbody[S.hl[2 * h]], bb = S.pbody[S.hl[2 * h + 1]];
  const double* ra = S.bodies + 40 * (size_t)ba;
  const double* rb = S.bodies + 40 * (size_t)bb;
  const v3<double> A = ld3(S.hA + 3 * h), B = ld3(S.hB + 3 * h);
  const double start = vlen(sub(A, B));
  if (start < 1e-6 && S.t > 1e-4) return false;
  const SolverState fa = sv_load(ra + 14), fb = sv_load(rb + 14);
  double m[16], mi[16];
  pose(fa.q, fa.x, m);
  inv44(m, mi);
  st3(k + CC_LA, xform(mi, A));
  pose(fb.q, fb.x, m);
  inv44(m, mi);
  st3(k + CC_LB, xform(mi, B));
  const v3<double> gn = dvs(sub(B, A), 2.0);
  st3(c + CH_N, sv_normalized(gn));
  const v3<double> r_A = sub(A, fa.x), r_B = sub(B, fb.x);
  st3(k + CC_RA, r_A), st3(k + CC_RB, r_B);
  const v3<double> rn_A = cross(r_A, gn), rn_B = cross(r_B, gn);
  double k_normal = 0.0;
  if (ra[38] == 0.0) k_normal += 1.0 / S.mass[ba] + sv_quad(rn_A, ra + 28);
  if (rb[38] == 0.0) k_normal += 1.0 / S.mass[bb] + sv_quad(rn_B, rb + 28);
  c[CH_MEFF] = k_normal < 1e-6 ? 0.0 : 1.0 / k_normal;
  c[CH_OFF] = 0.0;
  const double outer = S.heps[h] * 0.25;
  const double lower_slop = sv_max(outer * 0.2, outer - start);
  c[CH_OUTER] = outer, c[CH_SLOP] = lerp(lower_slop, outer * 0.2, 0.3);
  for (int j = 0; j < 3; ++j) k[CC_LF + j] = 0.0;
  // warm start (warm_start.cpp:12-29) and its impulses at the states the
  // solve starts from (:185-213): the change of impulse and both torques
  double w;
  c[CH_IMP] = warm_find(S.warm, warm_key(ba, bb), w) ? w * 0.75 : 0.0;
  const v3<double> u = scl(sv_neg(ld3(c + CH_N)), c[CH_IMP]);
  st3(c + CH_U, u);
  st3(c + CH_LR, sv_torque(u, sub(add(sv_turn(fa.q, ld3(k + CC_LA)), fa.x), fa.x)));
  st3(c + CH_LR + 3, sv_torque(sv_neg(u), sub(add(sv_turn(fb.q, ld3(k + CC_LB)), fb.x), fb.x)));
  return true;
}
// A particle at its future state, with the impulse from gravity (:171-180).
D2_HD void sv_particle_setup(const ClusterSolve& S, int b, double* p) {
  const double* r = S.bodies + 40 * (size_t)b;
  for (int j = 0; j < 3; ++j) {
    p[SP_X + j] = p[SP_FX + j] = r[18 + j];
    p[SP_V + j] = p[SP_FV + j] = r[21 + j];
    p[SP_L + j] = p[SP_FL + j] = r[24 + j];
    p[SP_ROT + j] = 0.0, p[SP_OFF + j] = 0.0;
  }
  for (int j = 0; j < 4; ++j) p[SP_Q + j] = r[14 + j];
  for (int j = 0; j < 9; ++j) p[SP_IB + j] = r[28 + j];
  p[SP_MASS] = S.mass[b];
  st3(p + SP_IMP, scl(sclL(S.mass[b], S.g), S.t));
}
// A particle's accumulated impulses, for walks over its own contacts.
struct SvAcc {
  v3<double> imp, rot, off;
};
D2_HD SvAcc sv_acc(const double* p) { return SvAcc{ld3(p + SP_IMP), ld3(p + SP_ROT), ld3(p + SP_OFF)}; }
D2_HD void sv_acc_store(const SvAcc& a, double* p) {
  st3(p + SP_IMP, a.imp), st3(p + SP_ROT, a.rot), st3(p + SP_OFF, a.off);
}
// One contact's warm-start impulse on its particle of side 0 (a) or 1 (b).
D2_HD void sv_warm_apply(SvAcc& a, const double* c, int side) {
  const v3<double> u = ld3(c + CH_U);
  a.imp = side ? sub(a.imp, u) : add(a.imp, u);
  a.rot = add(a.rot, ld3(c + CH_LR + 3 * side));
}
// sequential_impulses.cpp:46-70 with the rotation already turned.
D2_HD void sv_integrate(double* p, double t) {
  const double m = p[SP_MASS];
  st3(p + SP_V, add(ld3(p + SP_FV), dvs(ld3(p + SP_IMP), m)));
  st3(p + SP_X, add(ld3(p + SP_FX), scl(dvs(ld3(p + SP_OFF), m), t)));
  st3(p + SP_L, add(ld3(p + SP_FL), ld3(p + SP_ROT)));
}
// The first prediction of a dynamic particle (:215-227): its rotation and state.
D2_HD void sv_predict(double* p, double t) {
  const v3<double> z{0.0, 0.0, 0.0};
  const SolverState f{quat{p[SP_Q], p[SP_Q + 1], p[SP_Q + 2], p[SP_Q + 3]}, ld3(p + SP_FX), ld3(p + SP_FV),
                      ld3(p + SP_FL)};
  const quat q = sv_update(f, t, z, z, z, z, p[SP_MASS], p + SP_IB).q;
  p[SP_Q] = q.w, p[SP_Q + 1] = q.x, p[SP_Q + 2] = q.y, p[SP_Q + 3] = q.z;
  sv_integrate(p, t);
}
// A contact's local points rotated as its particles are from here on, and
// the friction's torques before its first sweep (zero).
D2_HD void sv_contact_turn(double* c, const double* k, const double* pa, const double* pb) {
  st3(c + CH_WA, sv_turn(quat{pa[SP_Q], pa[SP_Q + 1], pa[SP_Q + 2], pa[SP_Q + 3]}, ld3(k + CC_LA)));
  st3(c + CH_WB, sv_turn(quat{pb[SP_Q], pb[SP_Q + 1], pb[SP_Q + 2], pb[SP_Q + 3]}, ld3(k + CC_LB)));
  for (int j = 0; j < 6; ++j) c[CH_LR + 6 + j] = 0.0;
}
// One side of a contact in the normal pass (:231-375): the point's arm, its
// position and its velocity along the normal.
struct SvSide {
  v3<double> arm;
  double dn, vn;
};
D2_HD SvSide sv_side(const double* p, v3<double> w, v3<double> n) {
  const v3<double> x = ld3(p + SP_X), p1 = add(w, x);
  SvSide s;
  s.arm = sub(p1, x);
  s.dn = dot(p1, n);
  s.vn = dot(add(ld3(p + SP_V), cross(mul33v(p + SP_IB, ld3(p + SP_L)), s.arm)), n);
  return s;
}
// The contact's impulses after one visit: d1 the gap, v1 the closing speed.
D2_HD void sv_contact_step(double* c, double d1, double v1, double t, double& du, double& doff) {
  const double damp = 0.1, outer = c[CH_OUTER], m = c[CH_MEFF];
  const double last = c[CH_IMP], last_off = c[CH_OFF];
  const double dimp = d1 < outer ? (v1 * m) * damp : -last;
  const double imp = sv_max(last + dimp, 0.0);
  const double pen = outer - d1;
  const double dof = d1 < outer ? ((damp * m) * sv_max(0.0, pen - c[CH_SLOP])) / t : -last_off;
  const double off = sv_max(last_off + dof, 0.0);
  c[CH_IMP] = imp, c[CH_OFF] = off;
  du = imp - last, doff = off - last_off;
}
// The visit's impulse f, its torque and its offset impulse fo on a particle.
D2_HD void sv_apply(double* p, v3<double> f, v3<double> fo, v3<double> arm) {
  st3(p + SP_IMP, add(ld3(p + SP_IMP), f));
  st3(p + SP_ROT, add(ld3(p + SP_ROT), sv_torque(f, arm)));
  st3(p + SP_OFF, add(ld3(p + SP_OFF), fo));
}
// One contact of a friction sweep (:392-571): both passes' values from the
// particles' states, which a sweep's impulses do not change before its end.
// par: the sweep's parity.  Returns whether the impulse still moves.
D2_HD bool sv_friction(const ClusterSolve& S, int h, double* c, double* k, const double* pa, const double* pb, int par) {
  const int ba = S.pbody[S.hl[2 * h]], bb = S.pbody[S.hl[2 * h + 1]];
  const bool sa = S.bodies[40 * (size_t)ba + 38] != 0.0, sb = S.bodies[40 * (size_t)bb + 38] != 0.0;
  const v3<double> n = ld3(c + CH_N), z{0.0, 0.0, 0.0};
  const v3<double> xa = ld3(pa + SP_X), xb = ld3(pb + SP_X);
  const v3<double> armA = sub(add(ld3(c + CH_WA), xa), xa), armB = sub(add(ld3(c + CH_WB), xb), xb);
  const v3<double> v1A = sa ? z : add(ld3(pa + SP_V), cross(mul33v(pa + SP_IB, ld3(pa + SP_L)), armA));
  const v3<double> v1B = sb ? z : add(ld3(pb + SP_V), cross(mul33v(pb + SP_IB, ld3(pb + SP_L)), armB));
  const v3<double> v1AB = sub(v1A, v1B);
  const v3<double> vt = sub(v1AB, sclL(dot(v1AB, n), n));
  st3(k + CC_VT, vt);
  const double mu = sv_min(S.fric[ba], S.fric[bb]);
  const double max_force = (c[CH_IMP] * mu) * 10;
  const v3<double> tan = sv_normalized(vt);
  const v3<double> rtA = cross(ld3(k + CC_RA), tan), rtB = cross(ld3(k + CC_RB), tan);
  double kt = 0.0;
  if (!sa) kt += 1.0 / pa[SP_MASS] + sv_quad(rtA, pa + SP_IB);
  if (!sb) kt += 1.0 / pb[SP_MASS] + sv_quad(rtB, pb + SP_IB);
  const double mt = kt < 1e-6 ? 0.0 : 1.0 / kt;
  const v3<double> delta = scl(scl(sv_neg(vt), mt), 0.9);
  v3<double> fit = add(ld3(k + CC_LF), delta);
  const double len = vlen(fit);
  const double cl = (len < 0.0) ? 0.0 : (max_force < len) ? max_force : len;  // std::clamp(len, 0, max)
  fit = scl(sv_normalized(fit), cl);
  const v3<double> u = dvs(sub(fit, ld3(k + CC_LF)), (double)S.hpc[h]);
  st3(k + CC_LF, fit);
  st3(c + CH_U, u);
  st3(c + CH_LR + 6 * par, sv_torque(fit, armA));
  st3(c + CH_LR + 6 * par + 3, sv_torque(sv_neg(fit), armB));
  return vlen(u) > 1e-4;
}
// A contact's friction impulse and torque (the last sweep's taken out) on its
// particle; the offset friction totals stay zero, (0 - 0) / count.
D2_HD void sv_friction_apply(SvAcc& a, const double* c, int side, int par) {
  const v3<double> u = ld3(c + CH_U), z{0.0, 0.0, 0.0};
  a.imp = side ? sub(a.imp, u) : add(a.imp, u);
  a.rot = add(sub(a.rot, ld3(c + CH_LR + 6 * (par ^ 1) + 3 * side)), ld3(c + CH_LR + 6 * par + 3 * side));
  a.off = side ? sub(a.off, z) : add(a.off, z);
}
D2_HD bool sv_moved(const double* p) { return vlen(sub(ld3(p + SP_IMP), ld3(p + SP_LAST))) > 1e-6; }
// The new future state (:624-626) of a dynamic particle.
D2_HD void sv_store_future(const double* p, double* r) {
  for (int j = 0; j < 4; ++j) r[14 + j] = p[SP_Q + j];
  for (int j = 0; j < 3; ++j) r[18 + j] = p[SP_X + j], r[21 + j] = p[SP_V + j], r[24 + j] = p[SP_L + j];
}
D2_HD void sv_store_out(const double* c, const double* k, double* o) {
  for (int j = 0; j < 3; ++j) o[j] = c[CH_N + j], o[5 + j] = k[CC_LF + j], o[8 + j] = k[CC_VT + j];
  o[3] = c[CH_IMP], o[4] = c[CH_OFF];
}

// The sequential walk: contact by contact, in sorted order.
D2_HD bool solve_cluster(const ClusterSolve& S) {
  const int nh = S.nh, np = S.np;
  const double t = S.t;
  auto hot = [&](int c) { return S.hs + (size_t)CH * c; };
  auto cold = [&](int c) { return S.hs + (size_t)CH * nh + (size_t)CC * c; };
  auto part = [&](int c, int side) { return S.ps + (size_t)SP * S.hl[2 * S.ord[c] + side]; };
  auto is_static = [&](int k) { return S.bodies[40 * (size_t)S.pbody[k] + 38] != 0.0; };
  for (int c = 0; c < nh; ++c)
    if (!sv_contact_setup(S, S.ord[c], hot(c), cold(c))) return false;
  for (int k = 0; k < np; ++k) sv_particle_setup(S, S.pbody[k], S.ps + (size_t)SP * k);
  for (int c = 0; c < nh; ++c)
    for (int side = 0; side < 2; ++side) {
      SvAcc a = sv_acc(part(c, side));
      sv_warm_apply(a, hot(c), side);
      sv_acc_store(a, part(c, side));
    }
  for (int k = 0; k < np; ++k)
    if (!is_static(k)) sv_predict(S.ps + (size_t)SP * k, t);
  for (int c = 0; c < nh; ++c) sv_contact_turn(hot(c), cold(c), part(c, 0), part(c, 1));
  if (nh > 0) {
    bool converged = false;  // normal pass (:231-375)
    for (int it = 0; !converged && it < 1000; ++it) {
      for (int k = 0; k < np; ++k) st3(S.ps + (size_t)SP * k + SP_LAST, ld3(S.ps + (size_t)SP * k + SP_IMP));
      for (int c = 0; c < nh; ++c) {
        double *pa = part(c, 0), *pb = part(c, 1), *s = hot(c);
        const v3<double> n = ld3(s + CH_N);
        const SvSide A = sv_side(pa, ld3(s + CH_WA), n), B = sv_side(pb, ld3(s + CH_WB), n);
        double du, doff;
        sv_contact_step(s, B.dn - A.dn, A.vn - B.vn, t, du, doff);
        const v3<double> u = scl(sv_neg(n), du), uo = scl(sv_neg(n), doff);
        sv_apply(pa, u, uo, A.arm);
        sv_apply(pb, sv_neg(u), sv_neg(uo), B.arm);
        for (int side = 0; side < 2; ++side)
          if (!is_static(S.hl[2 * S.ord[c] + side])) sv_integrate(part(c, side), t);
      }
      converged = true;
      for (int k = 0; k < np && converged; ++k)
        if (sv_moved(S.ps + (size_t)SP * k)) converged = false;
    }
    converged = false;  // friction pass (:392-571)
    for (int it = 0; !converged && it < 100; ++it) {
      converged = true;
      for (int c = 0; c < nh; ++c)
        if (sv_friction(S, S.ord[c], hot(c), cold(c), part(c, 0), part(c, 1), it & 1)) converged = false;
      for (int c = 0; c < nh; ++c)
        for (int side = 0; side < 2; ++side) {
          SvAcc a = sv_acc(part(c, side));
          sv_friction_apply(a, hot(c), side, it & 1);
          sv_acc_store(a, part(c, side));
        }
      for (int k = 0; k < np; ++k)
        if (!is_static(k)) sv_integrate(S.ps + (size_t)SP * k, t);
    }
  }
  for (int k = 0; k < np; ++k)  // a static body's future state stays as it was
    if (!is_static(k)) sv_store_future(S.ps + (size_t)SP * k, S.bodies + 40 * (size_t)S.pbody[k]);
  // warm store: each body pair keeps its last contact's impulse
  for (int c = 0; c < nh; ++c) {
    const int h = S.ord[c];
    warm_put(S.warm, warm_key(S.pbody[S.hl[2 * h]], S.pbody[S.hl[2 * h + 1]]), hot(c)[CH_IMP]);
  }
  for (int c = 0; c < nh; ++c) sv_store_out(hot(c), cold(c), S.out_h + 11 * (size_t)S.ord[c]);
  return true;
}

}  // namespace d2
