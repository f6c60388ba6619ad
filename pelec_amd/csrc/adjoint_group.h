// Discrete adjoint of the BDF reactor (adjoint.h: the operations, their transposes, tape and
// checkpoint layout) with one cell per group of lanes: component k of the Nordsieck array, of its
// adjoint and of every cotangent on lane k, matrices inverted with one row per lane (whole_cell.h).
#pragma once
#include "adjoint.h"
#include "whole_cell.h"

namespace pelec {

// The kinetics are compiled once and called: the integrator, its polish and the backward sweep evaluate
// them at a dozen places.
template <class Mech>
__device__ __noinline__ double adj_rhs(double t, double yl, int l, double rhoe0, double rhoesrc,
                                       double srcl, double tm, double* sh, double* xt,
                                       const double* rmul) {
  return GroupKin<Mech>::template rhs<true>(t, yl, l, rhoe0, rhoesrc, srcl, tm, lds_ptr(sh),
                                            lds_ptr(xt), rmul);
}
template <class Mech>
__device__ __noinline__ JacOut adj_jac(double t, double yl, int l, double rhoe0, double rhoesrc,
                                       double srcl, double tm, double* sh, double* xt,
                                       double* ws, const double* rmul) {
  return GroupKin<Mech>::template jac<true>(t, yl, l, rhoe0, rhoesrc, srcl, tm, lds_ptr(sh),
                                            lds_ptr(xt), ws, rmul);
}

template <class Mech>
struct AdjGroup {
  using K = GroupKin<Mech>;
  static constexpr int G = K::G, N = K::N, n = K::n, RS = GTape<n>::RS;
  using Grp = Group<G>;

  // problem
  int l;
  double rhoe0, rhoesrc, srcl, tm, at, tstop;
  BdfParams prm;
  const double* rmul;  // rate multipliers by position
  BdfScalars& S;       // one per group, in LDS
  double *sh, *xt;     // LDS block, tables of the wave
  double *ws, *wx;     // Jacobian workspaces: the saved Jacobian; polish and backward sweep
  // state
  double z[BDF_QMAX + 1], ac, ew, Mi[n];
  int kap;
  // tape
  double* base = nullptr;
  int cap = 0, count = 0;
  bool overflow = false;
  double* last_correct = nullptr;
  // adjoint
  double lam[BDF_QMAX + 1], gp[K::RR], ge, gy0;

  __device__ AdjGroup(BdfScalars& s) : S(s) {}
  __device__ lds_double* lds() const { return lds_ptr(sh); }

  // ---- tape (GTape's records): the header by the group's first lane, the vector one lane each
  __device__ double* next(int op) {
    if (!base) return nullptr;
    if (count >= cap) {
      overflow = true;
      return nullptr;
    }
    double* r = base + (int64_t)count * RS;
    ++count;
    if (l == 0) r[0] = op;
    return r;
  }
  struct Vec : RegV<n, G> {
    AdjGroup* c;
    __device__ void put(double* r, int i, double x) const {
      if (c->l == 0) r[i] = x;
    }
    __device__ void coeffs(double* r, const double* lc) const {
      for (int j = 0; j <= BDF_QMAX; ++j) put(r, 5 + j, lc[j]);
    }
    __device__ void rec_rescale(int q, double eta) const {
      if (double* r = c->next(OP_RESCALE)) {
        put(r, 1, q);
        put(r, 4, eta);
      }
      Grp::sync();
    }
    __device__ void rec_pascal(int q, double sign) const {
      if (double* r = c->next(OP_PASCAL)) {
        put(r, 1, q);
        put(r, 4, sign);
      }
      Grp::sync();
    }
    __device__ void rec_order_up(int q, int L, int ia, double A1, const double* lc) const {
      if (double* r = c->next(OP_ORDER_UP)) {
        put(r, 1, q);
        put(r, 2, L);
        put(r, 3, ia);
        put(r, 4, A1);
        coeffs(r, lc);
      }
      Grp::sync();
    }
    __device__ void rec_order_down(int q, const double* lc) const {
      if (double* r = c->next(OP_ORDER_DOWN)) {
        put(r, 1, q);
        coeffs(r, lc);
      }
      Grp::sync();
    }
    __device__ void rec_correct(const BdfScalars& S, bool save, int qmax) const {
      c->last_correct = nullptr;
      if (double* r = c->next(OP_CORRECT)) {
        c->last_correct = r;
        put(r, 1, S.q);
        put(r, 2, save ? 1 : 0);
        put(r, 3, qmax);
        put(r, 4, S.gamma);
        coeffs(r, S.l);
        put(r, 11, 1.0 / S.l[1]);
        put(r, 12, S.tn);
        if (c->l < n) r[16 + c->l] = c->z[0] + c->ac;
      }
      Grp::sync();
    }
    __device__ void rec_mark_save() const {
      if (c->last_correct) put(c->last_correct, 2, 1);
      Grp::sync();
    }
    __device__ void rec_state(int op, double h, double t) const {
      if (double* r = c->next(op)) {
        put(r, 4, h);
        put(r, 12, t);
        if (c->l < n) r[16 + c->l] = c->z[0];
      }
      Grp::sync();
    }
  };
  __device__ Vec vec() { return Vec{{{}, z, ac, ew, at}, this}; }

  // ---- forward integration (BdfCell with POLISH)
  __device__ double f(double t, double yl) {
    S.nfe++;
    return adj_rhs<Mech>(t, yl, l, rhoe0, rhoesrc, srcl, tm, sh, xt, rmul);
  }
  // row l of I - g J (or of its transpose) from a Jacobian workspace
  __device__ void matrix(double (&a)[n], const double* w, double g, bool transposed) const {
    const int lo = after(l, g);
    const double* p = transposed ? w + (lo < n ? lo : 0) * G : w + lo;
#pragma unroll
    for (int c = 0; c < n; ++c) a[c] = K::load_l2(p + (transposed ? c : c * G));
#pragma unroll
    for (int c = 0; c < n; ++c) a[c] = fma(-g, a[c], c == lo ? 1.0 : 0.0);
    Grp::sync();
  }
  __device__ int lsetup() {
    if (jac_decide(S)) adj_jac<Mech>(S.tn, z[0], l, rhoe0, rhoesrc, srcl, tm, sh, xt, ws, rmul);
    matrix(Mi, ws, S.gamma, false);
    return K::invert(Mi, l, kap, lds());
  }
  // acor = gamma f(tn, zn0 + acor) - zn1 / l1 solved to convergence (exact Jacobian each iteration)
  __device__ void polish() {
    const double rl1 = 1.0 / S.l[1];
    for (int it = 0; it < 8; ++it) {
      const double y = z[0] + ac;
      double b = S.gamma * f(S.tn, y) - rl1 * z[1] - ac;
      adj_jac<Mech>(S.tn, y, l, rhoe0, rhoesrc, srcl, tm, sh, xt, wx, rmul);
      double a[n];
      int k;
      matrix(a, wx, S.gamma, false);
      if (K::invert(a, l, k, lds()) != 0) break;
      b = K::solve(a, k, b, l, lds());
      ac += b;
      if (!K::any(!(fabs(b) <= 1e-14 * fabs(z[0] + ac) + 1e-300))) break;
    }
    const double w = ac * ew;
    S.acnrm = sqrt(Grp::sum(w * w) / n);
  }
  __device__ int nls(bool setup) {
    for (;;) {
      LaneVal ft;
      ft.x = f(S.tn, z[0]);
      if (setup) {
        const int ier = lsetup();
        after_setup(S);
        setup = false;
        if (ier != 0) return 3;
      }
      ac = 0.0;
      S.m = 0;
      int r;
      for (;;) {
        r = newton_correct<n>(S, vec(), ft,
                              [&](LaneVal& b) { b.x = K::solve(Mi, kap, b.x, l, lds()); });
        if (r != 1) break;
        ft.x = f(S.tn, z[0] + ac);
      }
      if (r == 0) {
        polish();
        return 0;
      }
      if (r == 3) return 3;
      setup = true;  // stale Jacobian: rebuild and retry
      S.convfail = 2;
    }
  }
  __device__ int step() {
    step_prologue<n>(S, vec(), prm.qmax);
    for (;;) {
      const bool cs = begin_attempt<n>(S, vec(), tstop);
      if (nls(cs) != 0) {
        const int s = conv_fail<n>(S, vec());
        if (s >= 0) return s;
        continue;
      }
      const double dsm = S.acnrm * S.tq[2];
      if (dsm <= 1.0) {
        finish_step<n>(S, vec(), dsm, prm.qmax);
        return CELL_OK;
      }
      const int s = error_test_fail<n>(S, vec(), dsm, prm.qmax);
      if (s >= 0) return s;
      if (s == -2) {
        vec().rec_state(OP_RESTART, S.h, S.tn);
        z[1] = S.h * f(S.tn, z[0]);
      }
    }
  }
  __device__ void start(double y0, double tout) {
    scalars_reset(S, prm.qmax);
    tstop = tout;
    z[0] = y0;
#pragma unroll
    for (int j = 1; j <= BDF_QMAX; ++j) z[j] = 0.0;
    ac = 0.0;
    set_ewt<n>(vec(), prm);
    z[1] = f(S.tn, z[0]);
    S.h = hin<n>(S, vec(), tout,
                 [&](double t, const LaneVal& y, LaneVal& out) { out.x = f(t, y.x); });
    if ((S.tn + S.h - tout) * S.h > 0.0) S.h = (tout - S.tn) * (1.0 - 4.0 * cv::UROUND);
    S.hscale = S.h;
    S.hprime = S.h;
    z[1] *= S.h;
    vec().rec_state(OP_INIT, S.h, 0.0);
  }
  __device__ int advance() {
    if (S.nst >= prm.max_steps) return CELL_MAXSTEPS;
    set_ewt<n>(vec(), prm);
    const int s = step();
    if (s != CELL_OK) return s;
    return reached_tstop(S, tstop) ? CELL_OK : -1;
  }

  // ---- checkpoints: z, the integrator scalars, the saved Jacobian
  __device__ void save(double* p) const {
    if (l < n) {
#pragma unroll
      for (int j = 0; j <= BDF_QMAX; ++j) p[j * n + l] = z[j];
    }
    double* q = p + (BDF_QMAX + 1) * n;
    const uint64_t* w = reinterpret_cast<const uint64_t*>(&S);
    for (int k = l; k < BDF_SCALAR_WORDS; k += G) __builtin_memcpy(q + k, w + k, 8);
    q += BDF_SCALAR_WORDS;
    if (l < n)
      for (int c = 0; c < n; ++c) q[c * n + l] = K::load_l2(ws + c * G + l);
    Grp::sync();
  }
  __device__ void load(const double* p) {
    if (l < n) {
#pragma unroll
      for (int j = 0; j <= BDF_QMAX; ++j) z[j] = p[j * n + l];
    }
    const double* q = p + (BDF_QMAX + 1) * n;
    uint64_t* w = reinterpret_cast<uint64_t*>(&S);
    for (int k = l; k < BDF_SCALAR_WORDS; k += G) __builtin_memcpy(w + k, q + k, 8);
    q += BDF_SCALAR_WORDS;
    if (l < n)
      for (int c = 0; c < n; ++c) ws[c * G + l] = q[c * n + l];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    Grp::sync();
    // the Newton matrix in use at the checkpoint: I - gammap J, inverted again (deterministic)
    matrix(Mi, ws, S.gammap, false);
    (void)K::invert(Mi, l, kap, lds());
  }

  // ---- backward sweep
  // out += s J^T v; gp += s (df/dp)^T v; ge += s fe . v, J and o evaluated by the last adj_jac into
  // wx (its q_j still in LDS)
  __device__ void vjp(const JacOut& o, double v, double s, double& out) {
    lds_double* sm = lds();
    lds_double* vv = sm + K::O_V;
    lds_double* wv = sm + K::O_PS;
    vv[l] = v;
    const double vT = Grp::bcast(v, N) / o.D;
    wv[l] = l < N ? Mech::G_WT[l] * (v - o.ek * vT) : 0.0;
    ge += s * Grp::sum(o.fe * v);
    Grp::sync();
    const double* p = wx + (l < n ? l : 0) * G;
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < n; ++k) acc = fma(K::load_l2(p + k), vv[k], acc);
    out += l < n ? s * acc : 0.0;
#pragma unroll
    for (int r = 0; r < K::RR; ++r) {
      const int j = Mech::G_RORD[G * r + l];
      if (j >= 0) {
        double nw = 0.0;
#pragma unroll
        for (int u = 0; u < 6; ++u) {
          const int k = Mech::T_NSPC[j][u];
          if (k >= 0) nw += Mech::T_NNU[j][u] * wv[k];
        }
        gp[r] += s * sm[K::O_Q + G * r + l] * nw;
      }
    }
    Grp::sync();
  }
  __device__ JacOut jac_x(double t, double y) {
    return adj_jac<Mech>(t, y, l, rhoe0, rhoesrc, srcl, tm, sh, xt, wx, rmul);
  }
  __device__ static void add_at(double (&a)[BDF_QMAX + 1], int i, double x, bool set) {
#pragma unroll
    for (int j = 0; j <= BDF_QMAX; ++j) a[j] = j == i ? (set ? x : a[j] + x) : a[j];
  }
  // adjoint of one tape record (records are walked last to first)
  __device__ void back(const double* r) {
    const int op = (int)r[0], q = (int)r[1];
    double lc[BDF_QMAX + 1];
#pragma unroll
    for (int j = 0; j <= BDF_QMAX; ++j) lc[j] = r[5 + j];
    const double y = l < n ? r[16 + l] : 0.0;
    if (op == OP_RESCALE) {
      double fac = 1.0;
#pragma unroll
      for (int j = 1; j <= BDF_QMAX; ++j) {
        fac *= r[4];
        lam[j] = j <= q ? lam[j] * fac : lam[j];
      }
    } else if (op == OP_PASCAL) {
      const double sg = r[4];
#pragma unroll
      for (int k = BDF_QMAX; k >= 1; --k)
#pragma unroll
        for (int j = k; j <= BDF_QMAX; ++j) lam[j] = (k <= q && j <= q) ? lam[j] + sg * lam[j - 1] : lam[j];
    } else if (op == OP_ORDER_UP) {
      const int L = (int)r[2], ia = (int)r[3];
      double lL = sel(lam, L);
#pragma unroll
      for (int j = 2; j <= BDF_QMAX; ++j) lL = j <= q ? lL + lc[j] * lam[j] : lL;
      lL *= r[4];
      if (ia != L) add_at(lam, L, 0.0, true);
      add_at(lam, ia, lL, ia == L);
    } else if (op == OP_ORDER_DOWN) {
      double s = 0.0;
#pragma unroll
      for (int j = 2; j < BDF_QMAX; ++j) s = j < q ? s + lc[j] * lam[j] : s;
      add_at(lam, q, -s, false);
    } else if (op == OP_CORRECT) {
      const bool save = r[2] != 0.0;
      const int qmax = (int)r[3];
      const double gamma = r[4], rl1 = r[11], t = r[12];
      double nu = 0.0;
#pragma unroll
      for (int j = 0; j <= BDF_QMAX; ++j) nu = j <= q ? nu + lc[j] * lam[j] : nu;
      if (save) {
        nu += sel(lam, qmax);
        add_at(lam, qmax, 0.0, true);
      }
      const JacOut o = jac_x(t, y);
      {
        double a[n];
        int k;
        matrix(a, wx, gamma, true);  // rows of M^T
        (void)K::invert(a, l, k, lds());
        nu = K::solve(a, k, nu, l, lds());
      }
      vjp(o, nu, gamma, lam[0]);
      lam[1] -= rl1 * nu;
    } else if (op == OP_RESTART) {
      const double l1 = lam[1];
      lam[1] = 0.0;
      const JacOut o = jac_x(r[12], y);
      vjp(o, l1, r[4], lam[0]);
    } else if (op == OP_INIT) {
      gy0 = lam[0];
      const JacOut o = jac_x(0.0, y);
      vjp(o, lam[1], r[4], gy0);
    }
    Grp::sync();
  }
};

}  // namespace pelec
