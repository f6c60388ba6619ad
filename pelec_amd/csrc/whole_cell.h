// Whole integration of a cell by one group of lanes, the state in registers.
//
// A group of G lanes (G = 16, 32 or 64 for n <= 16, 32, 64; Mech::G_W) takes a cell of the call from
// an atomic queue, integrates it over dt and takes the next: lane k holds component k of the
// Nordsieck array, the accumulated correction and the error weights, and row k of the inverse
// Newton matrix. Nothing but the cell's inputs and outputs (and its Jacobian, once per evaluation)
// crosses HBM, one launch serves a call of any size, and a cell never waits for another.
// The step logic is bdf_core.h; the kinetics come from the generated lane-group tables (Mech::G_*).
#pragma once
#include <hip/hip_runtime.h>

#include "batched.h"
#include "bdf_core.h"
#include "group_model.h"

namespace pelec {

typedef double dv2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) dv2 lds_dv2;
typedef __attribute__((address_space(3))) char lds_char;
typedef unsigned uv4 __attribute__((ext_vector_type(4)));

// Register accessor of the step logic: component l of the cell on lane l. Every lane runs every
// component loop once, with its own registers whatever the index, so the lanes of a group never
// part in the step logic; lanes without a component hold zeros.
template <int n, int G>
struct RegV : NoTape {
  static constexpr bool kMemory = false;
  static constexpr bool kRegister = true;
  static constexpr int kStep = n;
  double (&z)[BDF_QMAX + 1];
  double &a, &e;
  double at;  // absolute tolerance of the lane's component
  __device__ static constexpr int c0() { return 0; }
  __device__ static double sum(double x) { return Group<G>::sum(x); }
  __device__ static double max(double x) { return Group<G>::max(x); }
  template <int m>
  using Arr = LaneVal;
  __device__ double& Z(int j, int) const { return z[j]; }
  __device__ double& A(int) const { return a; }
  __device__ double& E(int) const { return e; }
  // columns at a run-time index: selects, so the history stays in registers
  __device__ double ZR(int j, int) const { return sel(z, j); }
  __device__ void ZW(int j, int, double x) const {
#pragma unroll
    for (int k = 0; k <= BDF_QMAX; ++k) z[k] = k == j ? x : z[k];
  }
};

// exp and log of the kinetics by table (P. T. P. Tang, ACM TOMS 15 (1989) 144 and 16 (1990) 378): a
// third of the instructions of the library's, which are the larger part of a right-hand side
// (GRI-Mech 3.0, 16,384 cells: 23.6 -> 22.0 ms; H2/air 32^3: 2.10 -> 1.97 ms). The
// tables are XT_WORDS doubles of LDS per wave: 2^(j/32), and c_j = 2 / (1 + (j + 1/2)/32) with -log c_j / 2.
constexpr int XT_WORDS = 96;
__device__ inline void fill_tables(lds_double* xt) {
  const int j = threadIdx.x & 31;
  if ((threadIdx.x & 63) < 32) {
    const double c = 1.0 / (1.0 + (j + 0.5) / 32.0);
    xt[j] = exp2(j / 32.0);
    xt[32 + j] = 2.0 * c;
    xt[64 + j] = -log(c);
  }
  Group<64>::sync();
}
// e^x = 2^k 2^(j/32) e^r, |r| <= ln 2 / 64, e^r by its series to r^6 (r^7/5040 < 2^-58); below -746: 0.
__device__ inline double fexp(double x, const lds_double* xt) {
  x = x < -746.0 ? -746.0 : x;
  const double kd = __builtin_rint(x * 46.16624130844683);  // 32 / ln 2
  const int k = (int)kd;
  const double t = xt[k & 31];
  // ln 2 / 32 in two parts, the first with 27 zero bits: k times it is exact
  double r = fma(-kd, 0x1.62e42f8p-6, x);
  r = fma(-kd, 4.06140840434059e-10, r);
  double q = fma(r, 1.0 / 720.0, 1.0 / 120.0);
  q = fma(r, q, 1.0 / 24.0);
  q = fma(r, q, 1.0 / 6.0);
  q = fma(r, q, 0.5);
  q = fma(r * r, q, r);
  return ldexp(fma(t, q, t), k >> 5);
}
// log x of a positive, normal x: e ln 2 - log c_j + log(1 + r), |r| <= 1/64, by its series to r^8
// (r^9/9 < 2^-57); within an ulp of the result or of 1, whichever is larger.
__device__ inline double flog(double x, const lds_double* xt) {
  const double m = __builtin_amdgcn_frexp_mant(x);  // [1/2, 1)
  const int e = __builtin_amdgcn_frexp_exp(x) - 1;
  const int j = (__double2hiint(m) >> 15) & 31;
  const double r = fma(m, xt[32 + j], -1.0);
  const double l = xt[64 + j];
  double q = fma(r, -1.0 / 8.0, 1.0 / 7.0);
  q = fma(r, q, -1.0 / 6.0);
  q = fma(r, q, 1.0 / 5.0);
  q = fma(r, q, -1.0 / 4.0);
  q = fma(r, q, 1.0 / 3.0);
  q = fma(r, q, -0.5);
  q = fma(r * r, q, r);
  return fma((double)e, 0.69314718055994530942, l) + q;
}

// The kinetics are inlined wherever they are used: as soon as two kernels of a library call them the
// compiler makes them functions, and a call in k_cell's loop costs 100 to 140 B of scratch per lane
// (drm19, 65,536 cells: 15.1 ms against 13.5).
#define PELEC_INLINE __device__ __forceinline__

// What jac() leaves beside the matrix: the lane's e_k, rho c_v, and df/d(rho e0) of its component.
struct JacOut {
  double ek, D, fe;
};

// Kinetics, Jacobian and Newton matrix of one cell on a group of lanes.
template <class Mech>
struct GroupKin {
  static constexpr int G = Mech::G_W;
  static constexpr int N = Mech::NSP;
  static constexpr int n = N + 1;
  static constexpr int RR = Mech::G_RR;
  static constexpr int P = RR * G;
  static constexpr int NS = Mech::T_NSETS;
  using Grp = Group<G>;
  static constexpr int even(int x) { return (x + 1) & ~1; }
  // LDS block of a cell (doubles, every part 16-byte aligned)
  static constexpr int O_RP = 0;                    // {C_k, exp(-g_k/RT)}, entry N: {1, 1}
  static constexpr int O_PP = O_RP + 2 * (N + 1);   // {C_k, exp(g_k/RT)}
  static constexpr int O_M = O_PP + 2 * (N + 1);    // third-body concentration per set
  static constexpr int O_Q = O_M + even(NS);        // q by position; entry P: 0
  static constexpr int O_PS = O_Q + P + 2;          // partial production rates
  static constexpr int RHS_WORDS = O_PS + G;
  // between right-hand sides their block serves the linear algebra
  static constexpr int O_V = O_RP;                  // vector exchange (G <= 4(N+1))
  static constexpr int O_PR = O_RP;                 // pivot row of the factorisation (n + 1 <= 4(N+1))
  // Jacobian part
  static constexpr int O_HR = RHS_WORDS;            // h_k/RT, entry N: 0
  static constexpr int O_JV = O_HR + even(N + 1);   // the Jacobian's terms (G_NJ, and a 0)
  static constexpr int WORDS = O_JV + even(Mech::G_NJ + 1);
  // the cell's Jacobian workspace: element (k, c) at [c * G + k], G_JC columns (the n of the
  // Jacobian, and the sums over dq/dM of each efficiency set and over dq/dT)
  static constexpr int JAC_SIZE = Mech::G_JC * G;

  // Jacobian elements are written by whichever lane sums them and read by their row's lane: from the L2.
  PELEC_INLINE static double load_l2(const double* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // any lane of the caller's group
  PELEC_INLINE static bool any(bool p) {
    const unsigned long long b = __ballot(p);
    if constexpr (G == 64) return b != 0ull;
    const unsigned long long m = ((1ull << (G & 63)) - 1ull) << (threadIdx.x & 63 & ~(G - 1));
    return (b & m) != 0ull;
  }
  PELEC_INLINE static void load_e(double (&c)[6], bool lo, int l) {
    const dv2* p = reinterpret_cast<const dv2*>(&Mech::G_E[lo ? 0 : 1][0][l][0]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const dv2 v = p[i * G];
      c[2 * i] = v.x;
      c[2 * i + 1] = v.y;
    }
  }
  PELEC_INLINE static void e_cv(const double (&c)[6], double T, double& e, double& cv) {
    e = fma(T, fma(T, fma(T, fma(T, fma(T, c[5], c[4]), c[3]), c[2]), c[1]), c[0]);
    cv = fma(T, fma(T, fma(T, fma(T, 5.0 * c[5], 4.0 * c[4]), 3.0 * c[3]), 2.0 * c[2]), c[1]);
  }

  // T(e, Y): Newton on sum_k Y_k e_k(T), species k on lane k, from the guess T; |dT| <= 1e-12 T.
  // The iteration also ends after |dT| <= 1e-7 T: it converges quadratically, so the next
  // correction would be below (cv'/2cv) dT^2 ~ 1e-14 T -- unless a species' fit changed branch.
  // On return ec holds the lane's coefficients at T and ek, cvk are evaluated at T.
  PELEC_INLINE static double T_from_e(double e, double Yl, int l, double T, double tm,
                                    double (&ec)[6], double& ek, double& cvk) {
    bool lo = T < tm;
    load_e(ec, lo, l);
    for (int it = 0; it < 20; ++it) {
      e_cv(ec, T, ek, cvk);
      const double fv = Grp::sum(Yl * ek) - e;
      const double dv = Grp::sum(Yl * cvk);
      const double dT = -fv * recip(dv);
      T += dT;
      const bool lo2 = T < tm;
      const bool flip = any(lo2 != lo);
      if (flip) {
        lo = lo2;
        load_e(ec, lo, l);
      }
      if (fabs(dT) <= (flip ? 1e-12 : 1e-7) * T) break;
    }
    e_cv(ec, T, ek, cvk);
    return T;
  }

  // Arrhenius record of the reaction at position p, loaded ahead of its use.
  struct Record {
    dv2 ab;
    double ear;
    uint64_t pk;
  };
  PELEC_INLINE static Record record(int p) {
    return Record{reinterpret_cast<const dv2*>(&Mech::G_RA[0][0])[p], Mech::G_RE[p],
                  Mech::G_RP[p]};
  }

  // Reaction at position p (lane l of a round). JAC: also its derivatives into rb (8 x G).
  template <bool JAC, bool MUL>
  PELEC_INLINE static void reaction(const Record& rc_, int p, int l, double T, double lnT,
                                  double invT, lds_double* sh, const lds_double* xt,
                                  const double* rmul) {
    const dv2 ab = rc_.ab;
    const double ear = rc_.ear;
    const uint64_t pk = rc_.pk;
    const double karr = ab.x * fexp(ab.y * lnT - ear * invT, xt);
    double kf = karr, dkdM = 0.0, dlnk = 0.0;
    if (JAC) dlnk = (ab.y + ear * invT) * invT;
    const int kind = (int)(pk >> 56) & 3;
    if (kind) {
      const double Mj = sh[O_M + ((int)(pk >> 48) & 255)];
      kf = karr * Mj;
      dkdM = karr;
      if (Mech::G_NFO > 0 && kind == 2) {
        const double l0 = Mech::G_LOW[0][p], l1 = Mech::G_LOW[1][p], l2 = Mech::G_LOW[2][p];
        const double k0r = fexp(l0 + l1 * lnT - l2 * invT, xt);
        const double Pr = fmax(k0r * Mj, 1e-300);
        const double iPr1 = recip(1.0 + Pr);
        double F = 1.0, g = 0.0, dlnF_T = 0.0;
        if (Mech::G_TROEK[p]) {
          constexpr double LOG10E = 0.43429448190325182765;
          double lFc, iFc = 0.0, dFc = 0.0;
          if constexpr (Mech::G_TCONST) {
            lFc = Mech::G_TROE[0][p];
          } else {
            const double t0 = Mech::G_TROE[0][p], t2 = Mech::G_TROE[2][p], t4 = Mech::G_TROE[4][p];
            const double e3 = fexp(Mech::G_TROE[1][p] * T, xt);
            const double e1 = fexp(Mech::G_TROE[3][p] * T, xt);
            const double e2 = Mech::G_TROE[5][p] != 0.0 ? fexp(-t4 * invT, xt) : 0.0;
            const double Fc = fmax(t0 * e3 + t2 * e1 + e2, 1e-300);
            lFc = flog(Fc, xt) * LOG10E;
            if (JAC) {
              iFc = 1.0 / Fc;
              dFc = Mech::G_TROE[6][p] * e3 + Mech::G_TROE[7][p] * e1 + t4 * invT * invT * e2;
            }
          }
          const double cc = -0.4 - 0.67 * lFc, nn = 0.75 - 1.27 * lFc;
          const double xx = flog(Pr, xt) * LOG10E + cc;
          const double DD = recip(nn - 0.14 * xx);
          const double f1 = xx * DD;
          const double iden = recip(1.0 + f1 * f1);
          F = fexp(Mech::T_LN10 * lFc * iden, xt);
          if (JAC) {
            g = -lFc * 2.0 * f1 * nn * DD * DD * iden * iden;
            const double df1 = (-0.67 * nn + 1.27 * xx) * DD * DD;
            const double dlF = iden - lFc * 2.0 * f1 * df1 * iden * iden;
            dlnF_T = dlF * dFc * iFc;
          }
        }
        kf = karr * Pr * iPr1 * F;
        if (JAC) {
          const double dlnPr = (l1 + l2 * invT) * invT;
          dkdM = karr * k0r * F * (iPr1 * iPr1 + g * iPr1);
          dlnk = dlnk + dlnPr * iPr1 + g * dlnPr + dlnF_T;
        }
      }
    }
    if constexpr (MUL) {
      const double rm = rmul[p];
      kf *= rm;
      dkdM *= rm;
    }
    const int lo = (int)pk, hi = (int)(pk >> 32);
    const int r0 = lo & 255, r1 = (lo >> 8) & 255, r2 = (lo >> 16) & 255;
    const int p0 = (lo >> 24) & 255, p1 = hi & 255, p2 = (hi >> 8) & 255;
    const lds_dv2* rp = (const lds_dv2*)(sh + O_RP);
    const lds_dv2* pp = (const lds_dv2*)(sh + O_PP);
    const dv2 a0 = rp[r0], a1 = rp[r1], a2 = rp[r2];
    const dv2 b0 = pp[p0], b1 = pp[p1], b2 = pp[p2];
    const double rc = Mech::T_REFC * invT, irc = Mech::T_IREFC * T;
    const int dnu = ((hi >> 27) & 7) - 2;
    const double f1 = dnu > 0 ? irc : rc;
    double fac = dnu == 0 ? 1.0 : f1;
    if (dnu == 2 || dnu == -2) fac *= f1;
    const bool rev = (hi >> 26) & 1;
    // 1/Kc = prod fexp(g_p/RT) prod fexp(-g_r/RT) (P_atm/RT)^-dnu
    const double iKc = rev ? (b0.y * b1.y * b2.y) * (a0.y * a1.y * a2.y) * fac : 0.0;
    const double r01 = a0.x * a1.x, p01 = b0.x * b1.x;
    const double Pb = p01 * b2.x;
    const double net = r01 * a2.x - iKc * Pb;
    sh[O_Q + p] = kf * net;
    if constexpr (JAC) {
      lds_double* jv = sh + O_JV;
      const lds_double* hr = sh + O_HR;
      const double dlnKc =
          ((hr[p0] + hr[p1] + hr[p2]) - (hr[r0] + hr[r1] + hr[r2]) - double(dnu)) * invT;
      const double kb = -kf * iKc;
      const double d[6] = {kf * a1.x * a2.x, kf * a0.x * a2.x, kf * r01,
                           kb * b1.x * b2.x, kb * b0.x * b2.x, kb * p01};
      const int sl[6] = {r0, r1, r2, p0, p1, p2};
      int o = Mech::G_JD[p];
#pragma unroll
      for (int u = 0; u < 6; ++u)
        if (sl[u] != N) jv[o++] = d[u];
      jv[Mech::G_DT + p] = rev ? kf * (dlnk * net + iKc * Pb * dlnKc) : kf * dlnk * net;
      if (kind) jv[Mech::G_DM + p] = dkdM * net;
    }
  }

  // Species thermo of lane l into LDS and the third-body sums: what the reactions read.
  PELEC_INLINE static void load_g(double (&c)[8], bool lo, int l) {
    const dv2* p = reinterpret_cast<const dv2*>(&Mech::G_G[lo ? 0 : 1][0][l][0]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const dv2 v = p[i * G];
      c[2 * i] = v.x;
      c[2 * i + 1] = v.y;
    }
  }
  // Concentrations into LDS and the third-body sums, which need no temperature.
  PELEC_INLINE static void third_bodies(double Cl, int l, lds_double* sh) {
    if (l <= N) sh[O_RP + 2 * l] = l < N ? Cl : 1.0;
    if (l == 0) sh[O_Q + P] = 0.0;
    if constexpr (NS > 0) {
      double md[Mech::G_MN];
      int mi[Mech::G_MN];
#pragma unroll
      for (int e = 0; e < Mech::G_MN; ++e) {  // (0 on lanes without a set)
        md[e] = Mech::G_MD[e][l];
        mi[e] = Mech::G_MI[e][l];
      }
      double M = Grp::sum(Cl);
      Grp::sync();
#pragma unroll
      for (int e = 0; e < Mech::G_MN; ++e) M += md[e] * sh[O_RP + 2 * mi[e]];
      if (l < NS) sh[O_M + l] = M;
    }
  }
  // c: the g/RT coefficients of branch lo0, loaded before T was known
  template <bool JAC>
  PELEC_INLINE static void prelude(double T, double lnT, double invT, double Cl, int l, double tm,
                                   double (&c)[8], bool lo0, lds_double* sh, const lds_double* xt) {
    const bool lo = T < tm;
    if (any(lo != lo0)) load_g(c, lo, l);
    const double gRT = fma(T, fma(T, fma(T, fma(T, c[4], c[3]), c[2]), c[1]), c[0]) - c[5] * lnT +
                       c[6] * invT;
    const double E = fexp(gRT, xt);
    const double iE = recip(E);  // lanes >= N: coefficients 0, so E = iE = 1
    if (l <= N) {
      sh[O_RP + 2 * l + 1] = iE;
      ((lds_dv2*)(sh + O_PP))[l] = dv2{l < N ? Cl : 1.0, E};
      if (JAC) {
        const dv2* p = reinterpret_cast<const dv2*>(&Mech::G_H[lo ? 0 : 1][0][l][0]);
        const dv2 h0 = p[0], h1 = p[G], h2 = p[2 * G];
        sh[O_HR + l] = fma(T, fma(T, fma(T, fma(T, h2.x, h1.y), h1.x), h0.y), h0.x) + h2.y * invT;
      }
    }
    Grp::sync();
  }

  // production rate of species l from the q in LDS: a chunk of entries per lane, then the chunks
  // of each species
  struct Gather {
    uv4 e[Mech::G_L8];
    int cp;
  };
  PELEC_INLINE static Gather load_gather(int l) {
    Gather g;
#pragma unroll
    for (int i = 0; i < Mech::G_L8; ++i)
      g.e[i] = *reinterpret_cast<const uv4*>(&Mech::G_GE[i][l][0]);
    g.cp = Mech::G_CP[l];
    return g;
  }
  PELEC_INLINE static double gather(const Gather& g, int l, lds_double* sh) {
    double acc = 0.0;
    const lds_char* q = (const lds_char*)(sh + O_Q);
#pragma unroll
    for (int i = 0; i < Mech::G_L8; ++i)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const unsigned w = g.e[i][u];
        const double q0 = *(const lds_double*)(q + (w & 0xfff));
        const double q1 = *(const lds_double*)(q + ((w >> 16) & 0xfff));
        acc = fma((double)((int)(w << 16) >> 28), q0, acc);
        acc = fma((double)((int)w >> 28), q1, acc);
      }
    sh[O_PS + l] = acc;
    Grp::sync();
    const int b = g.cp & 255, m = g.cp >> 8;
    double wd = 0.0;
#pragma unroll
    for (int u = 0; u < Mech::G_CMAX; ++u)
      if (u < m) wd += sh[O_PS + b + u];
    return wd;
  }

  // log of a temperature (NaN where it is not one)
  PELEC_INLINE static double log_T(double T, const lds_double* xt) {
    return T > 0.0 ? flog(T, xt) : __builtin_nan("");
  }

  // f(t, y) for the lane's component (0 on lanes >= n).
  template <bool MUL = false>
  PELEC_INLINE static double rhs(double t, double yl, int l, double rhoe0, double rhoesrc,
                               double srcl, double tm, lds_double* sh, const lds_double* xt,
                               const double* rmul = nullptr) {
    l = after(l, yl);
    const bool sp = l < N;
    const double ys = sp ? yl : 0.0;
    // the tables of the first phases are loaded ahead of the temperature
    Record nx = record(l);
    const double iwt = Mech::G_IWT[l];
    const double Tg = Grp::bcast(yl, N);
    const bool lo0 = Tg < tm;
    double gc[8];
    load_g(gc, lo0, l);
    const double Cl = ys * iwt;
    third_bodies(Cl, l, sh);
    const double irho = recip(Grp::sum(ys));
    double ec[6], ek, cvk;
    const double T = T_from_e((rhoe0 + t * rhoesrc) * irho, ys * irho, l, Tg, tm, ec, ek, cvk);
    const double lnT = log_T(T, xt), invT = recip(T);
    prelude<false>(T, lnT, invT, Cl, l, tm, gc, lo0, sh, xt);
    const Gather ge = load_gather(after(l, T));
    const double Wk = Mech::G_WT[after(l, T)];
    const double D = Grp::sum(ys * cvk);
#pragma unroll 1
    for (int r = 0; r < RR; ++r) {
      const Record rc = nx;
      const int p = G * r + l;
      nx = record(p + (r + 1 < RR ? G : 0));
      reaction<false, MUL>(rc, p, l, T, lnT, invT, sh, xt, rmul);
    }
    Grp::sync();
    const double wd = gather(ge, l, sh);
    const double fk = sp ? Wk * wd + srcl : 0.0;
    const double num = rhoesrc - Grp::sum(ek * fk);
    Grp::sync();
    return l == N ? num * recip(D) : fk;
  }

  // Exact Jacobian of rhs() into ws (JAC_SIZE doubles; columns 0..n-1). The reactions leave their
  // derivatives in LDS, each lane sums the elements that the schedule deals it (terms in fours, an
  // element's sum stored when its last term is added), then the rows' lanes finish them. Adding each
  // reaction's terms to the rows instead would take n x n doubles of LDS per cell (23 KB at n = 54: one wave
  // per SIMD) or an L2 atomic per term (107 k to 312 k cycles a Jacobian, n = 22 to 54; 34 k to 65 k
  // this way).
  template <bool MUL = false>
  PELEC_INLINE static JacOut jac(double t, double yl, int l, double rhoe0, double rhoesrc, double srcl,
                             double tm, lds_double* sh, const lds_double* xt, double* ws,
                             const double* rmul = nullptr) {
    l = after(l, yl);
    const bool sp = l < N;
    double* wl = ws + l;
#pragma unroll 4
    for (int c = 0; c < Mech::G_JC; ++c) wl[c * G] = 0.0;
    const double ys = sp ? yl : 0.0;
    const double Tg = Grp::bcast(yl, N);
    const bool lo0 = Tg < tm;
    double gc[8];
    load_g(gc, lo0, l);
    const double Cl = ys * Mech::G_IWT[l];
    third_bodies(Cl, l, sh);
    const double irho = 1.0 / Grp::sum(ys);
    double ec[6], ek, cvk;
    const double T = T_from_e((rhoe0 + t * rhoesrc) * irho, ys * irho, l, Tg, tm, ec, ek, cvk);
    const double lnT = log_T(T, xt), invT = recip(T);
    prelude<true>(T, lnT, invT, Cl, l, tm, gc, lo0, sh, xt);
    if (l == 0) sh[O_JV + Mech::G_NJ] = 0.0;
#pragma unroll 1
    for (int r = 0; r < RR; ++r) {
      const int p = after(G * r + l, lnT);
      reaction<true, MUL>(record(p), p, l, T, lnT, invT, sh, xt, rmul);
    }
    const Gather ge = load_gather(after(l, T));
    // the zeros are in memory before other lanes store over them; the terms are in LDS
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    Grp::sync();
    const double wd = gather(ge, l, sh);
    double acc = 0.0;
    uv4 nx = *reinterpret_cast<const uv4*>(&Mech::G_JE[0][l][0]);
#pragma unroll 1
    for (int i = 0; i < Mech::G_JT4; ++i) {
      const uv4 e = nx;
      nx = *reinterpret_cast<const uv4*>(&Mech::G_JE[i + 1 < Mech::G_JT4 ? i + 1 : i][l][0]);
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = sh[O_JV + (e[u] & 0xfff)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        acc = fma((double)((int)(e[u] << 16) >> 28), v[u], acc);
        if (e[u] & 0x10000u) {
          ws[e[u] >> 17] = acc;
          acc = 0.0;
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    // energy row and the T-elimination (CellModel::jac)
    double tb[NS > 0 ? NS : 1], tbs = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      tb[s] = load_l2(wl + (n + s) * G);
      tbs += tb[s];
    }
    const double dwdT = load_l2(wl + (n + NS) * G);
    const double Wk = Mech::G_WT[l];
    const double fk = sp ? Wk * wd + srcl : 0.0;
    const double Bk = Wk * dwdT;
    const double dcvk = fma(T, fma(T, fma(T, 20.0 * ec[5], 12.0 * ec[4]), 6.0 * ec[3]), 2.0 * ec[2]);
    const double D = Grp::sum(ys * cvk);
    const double dDdT = Grp::sum(ys * dcvk);
    const double num = rhoesrc - Grp::sum(ek * fk);
    const double dNdT = -Grp::sum(cvk * fk + ek * Bk);
    const double iD = 1.0 / D;
    const double fT = num * iD;
    const double dfTdT = (dNdT - fT * dDdT) * iD;
    const double b = Bk * iD;
    // columns in batches: a batch's loads are in flight together
    constexpr int CBJ = 6;
#pragma unroll 1
    for (int m0 = 0; m0 < N; m0 += CBJ) {
      double av[CBJ];
#pragma unroll
      for (int u = 0; u < CBJ; ++u) av[u] = load_l2(wl + (m0 + u < N ? m0 + u : N) * G);
#pragma unroll
      for (int u = 0; u < CBJ; ++u) {
        const int m = m0 + u;
        if (m >= N) break;
        double a = av[u] + tbs;
#pragma unroll
        for (int s = 0; s < NS; ++s) a += tb[s] * Mech::T_EFFD[s][m];
        a *= Wk * Mech::IW[m];  // 0 on lanes without a species
        // T row, column m: dNdx_m = -sum_k e_k A_km
        const double dNdx = -Grp::sum(ek * a);
        const double em = Grp::bcast(ek, m), cm = Grp::bcast(cvk, m);
        const double tr = (dNdx - fT * cm) * iD - dfTdT * em * iD;
        wl[m * G] = l == N ? tr : a - b * em;
      }
    }
    Grp::sync();
    return JacOut{ek, D, l == N ? dfTdT * iD : b};
  }

  // a b + c into a register of its own: the row shift of invert() would otherwise cost a move per
  // column (the compiler prefers the two-address form).
  PELEC_INLINE static double fma3(double a, double b, double c) {
    double r;
    __asm__("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
  }
  PELEC_INLINE static double fma3_uniform(double a, double b, double c) {  // b in scalar registers
    double r;
    __asm__("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    return r;
  }

  // The group's pivot for a column: the largest of the rows' high words of |a| with the lane in the
  // low six bits (used rows: the lane alone), so the pivot is within 2^-14 of the largest entry.
  PELEC_INLINE static unsigned pivot_key(double a, bool used, int l) {
    const unsigned hi = (unsigned)__double2hiint(a) & 0x7fffffc0u;
    unsigned x = (used ? 0u : hi) | (unsigned)l;
    if constexpr (G > 32) {
      const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
      x = max(r[0], r[1]);
    }
    if constexpr (G > 16) {
      const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
      x = max(r[0], r[1]);
    }
    x = max(x, (unsigned)row_ror<8>((int)x));
    x = max(x, (unsigned)row_ror<4>((int)x));
    x = max(x, (unsigned)row_ror<2>((int)x));
    return max(x, (unsigned)row_ror<1>((int)x));
  }

  // a <- row of the inverse of the matrix whose row l is in a (lanes < n), by Gauss-Jordan
  // elimination with partial pivoting, rows staying on their lanes: with lane p the pivot of
  // column kap(p), lane p ends with row kap(p) of the inverse, its columns in pivot order (column c
  // belongs to the right-hand side component of the lane that was column c's pivot). The pivot search
  // is one 32-bit maximum (pivot_key). Pivot rows are broadcast as they stand -- by v_readlane where a
  // wave holds one cell (VALU time, no LDS round trip and no share of the CU's LDS bandwidth), through
  // LDS where it holds several (a read per cell and a select per column) -- and scaled once at the end: the
  // other rows' multipliers carry 1 / pivot. Measured: GRI-Mech 3.0 (n = 54), 16,384 cells, 25.4 ms
  // through LDS, 23.0 ms by v_readlane; four cells per wave (n = 10) 7.7 k cycles an inversion
  // through LDS, 11.5 k by v_readlane. Returns 0, or k + 1 when column k has no usable pivot.
  PELEC_INLINE static int invert(double (&a)[n], int l, int& kap, lds_double* sh) {
    l = after(l, a[0]);
    [[maybe_unused]] lds_dv2* pr = (lds_dv2*)(sh + O_PR);
    bool used = l >= n;
    kap = 0;
    int ier = 0;
    double scale = 0.0;
    unsigned best = pivot_key(a[0], used, l);
    // every step eliminates the column in a[0] and stores the row shifted down by one, so the loop
    // is rolled (unrolled it is n times the code, more than the instruction cache at n = 54) and
    // after n steps every column is back in its place
#pragma unroll 1
    for (int k = 0; k < n; ++k) {
      if (best < 64u && ier == 0) ier = k + 1;
      const bool piv = !used && l == (int)(best & 63u);
      double pv;
      int pl = 0;
      if constexpr (G == 64) {
        pl = __builtin_amdgcn_readfirstlane((int)(best & 63u));
        pv = lane_read(a[0], pl);
      } else {
        pv = __shfl(a[0], (int)(best & 63u), G);
      }
      if constexpr (G < 64) {
        if (piv) {
#pragma unroll
          for (int c = 0; c < n; c += 2)
            pr[c / 2] = dv2{c + 1 < n ? a[c + 1 < n ? c + 1 : 0] : 1.0,
                            c + 2 < n ? a[c + 2 < n ? c + 2 : 0] : 1.0};
        }
        Grp::sync();
      }
      const double inv = recip(pv);
      const double nf = piv ? 0.0 : -a[0] * inv;
      const double last = piv ? 1.0 : 0.0;
      if (piv) {
        scale = inv;
        used = true;
        kap = k;
      }
      if constexpr (G == 64) {
        // one cell per wave: the pivot row by v_readlane, four columns ahead of their use (a scalar
        // register read back at once stalls); the row's last entry is 1
#pragma unroll
        for (int c = 0; c < n - 1; c += 4) {
          double p[4];
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (c + u < n - 1) p[u] = lane_read(a[c + u + 1], pl);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (c + u < n - 1) a[c + u] = fma3_uniform(nf, p[u], a[c + u + 1]);
          if (c == 0) best = pivot_key(a[0], used, l);  // the next search, beside the update
        }
        a[n - 1] = nf + last;
      } else {
#pragma unroll
        for (int c = 0; c < n; c += 2) {
          const dv2 p = pr[c / 2];
          a[c] = fma3(nf, p.x, c + 1 < n ? a[c + 1 < n ? c + 1 : 0] : last);
          if (c + 1 < n)
            a[c + 1 < n ? c + 1 : 0] = fma3(nf, p.y, c + 2 < n ? a[c + 2 < n ? c + 2 : 0] : last);
          if (c == 0) best = pivot_key(a[0], used, l);
          if (c % 16 == 14) __asm__ __volatile__("" ::: "memory");  // at most 16 columns in flight
        }
        Grp::sync();
      }
    }
#pragma unroll
    for (int c = 0; c < n; ++c) a[c] *= scale;
    return ier;
  }

  // x_l of M x = b from invert()'s rows; b_l on lane l (0 on lanes >= n).
  PELEC_INLINE static double solve(const double (&a)[n], int kap, double b, int l, lds_double* sh) {
    lds_double* v = sh + O_V;
    if (l < n) v[kap] = b;
    Grp::sync();
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
    for (int c = 0; c < n; c += 2) {
      const dv2 p = ((const lds_dv2*)v)[c / 2];
      if (c & 2) {
        s2 = fma(a[c], p.x, s2);
        if (c + 1 < n) s3 = fma(a[c + 1 < n ? c + 1 : c], p.y, s3);
      } else {
        s0 = fma(a[c], p.x, s0);
        if (c + 1 < n) s1 = fma(a[c + 1 < n ? c + 1 : c], p.y, s1);
      }
    }
    const double x = (s0 + s1) + (s2 + s3);
    Grp::sync();
    if (l < n) v[kap] = x;
    Grp::sync();
    const double xl = l < n ? v[l] : 0.0;
    Grp::sync();
    return xl;
  }
};

// The integrator state of a cell that is neither a lane's component nor in registers: one copy
// per group in LDS.
struct CellState {
  BdfScalars S;
  double hg, hub, hlb;  // cvHin's iteration
  int count, pad;
  int64_t g;  // the cell
  double rhoe0, rhoesrc;
};

}  // namespace pelec
