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
typedef int iv4 __attribute__((ext_vector_type(4)));

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
  static constexpr int O_V = O_PS + G;              // vector exchange
  static constexpr int RHS_WORDS = O_V + G;
  static constexpr int O_PR = O_RP;                 // pivot row and pivot of the factorisation (n + 3 <= 4(N+1))
  // Jacobian part
  static constexpr int O_HR = RHS_WORDS;            // h_k/RT, entry N: 0
  static constexpr int O_RB = O_HR + even(N + 1);   // per-round reaction derivatives, 8 x G
  static constexpr int WORDS = O_RB + 8 * G;
  typedef __attribute__((address_space(1))) double glb_double;

  // The cell's Jacobian lives in device memory, element (l, c) at Jg[c * CS + l * RS] (columns of G
  // in the workspace of a group, rows of n for a caller's array): every element is read and written
  // by one lane only, the adds of jac() are performed at the L2 (in program order per address), and
  // reads go there too.
  __device__ static double load_l2(const double* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // any lane of the caller's group
  __device__ static bool any(bool p) {
    const unsigned long long b = __ballot(p);
    if constexpr (G == 64) return b != 0ull;
    const unsigned long long m = ((1ull << (G & 63)) - 1ull) << (threadIdx.x & 63 & ~(G - 1));
    return (b & m) != 0ull;
  }
  __device__ static void load_e(double (&c)[6], bool lo, int l) {
    const dv2* p = reinterpret_cast<const dv2*>(&Mech::G_E[lo ? 0 : 1][0][l][0]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const dv2 v = p[i * G];
      c[2 * i] = v.x;
      c[2 * i + 1] = v.y;
    }
  }
  __device__ static void e_cv(const double (&c)[6], double T, double& e, double& cv) {
    e = fma(T, fma(T, fma(T, fma(T, fma(T, c[5], c[4]), c[3]), c[2]), c[1]), c[0]);
    cv = fma(T, fma(T, fma(T, fma(T, 5.0 * c[5], 4.0 * c[4]), 3.0 * c[3]), 2.0 * c[2]), c[1]);
  }

  // T(e, Y): Newton on sum_k Y_k e_k(T), species k on lane k, from the guess T; |dT| <= 1e-12 T.
  // The iteration also ends after |dT| <= 1e-7 T: it converges quadratically, so the next
  // correction would be below (cv'/2cv) dT^2 ~ 1e-14 T -- unless a species' fit changed branch.
  // On return ec holds the lane's coefficients at T and ek, cvk are evaluated at T.
  __device__ static double T_from_e(double e, double Yl, int l, double T, double tm,
                                    double (&ec)[6], double& ek, double& cvk) {
    bool lo = T < tm;
    load_e(ec, lo, l);
    for (int it = 0; it < 20; ++it) {
      e_cv(ec, T, ek, cvk);
      const double fv = Grp::sum(Yl * ek) - e;
      const double dv = Grp::sum(Yl * cvk);
      const double dT = -fv / dv;
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

  // Reaction at position p (lane l of a round). JAC: also its derivatives into rb (8 x G).
  template <bool JAC, bool MUL>
  __device__ static void reaction(int p, int l, double T, double lnT, double invT, lds_double* sh,
                                  const double* rmul) {
    const dv2 ab = reinterpret_cast<const dv2*>(&Mech::G_RA[0][0])[p];
    const double ear = Mech::G_RE[p];
    const uint64_t pk = Mech::G_RP[p];
    const double karr = ab.x * exp(ab.y * lnT - ear * invT);
    double kf = karr, dkdM = 0.0, dlnk = 0.0;
    if (JAC) dlnk = (ab.y + ear * invT) * invT;
    const int kind = (int)(pk >> 56) & 3;
    if (kind) {
      const double Mj = sh[O_M + ((int)(pk >> 48) & 255)];
      kf = karr * Mj;
      dkdM = karr;
      if (Mech::G_NFO > 0 && kind == 2) {
        const double l0 = Mech::G_LOW[0][p], l1 = Mech::G_LOW[1][p], l2 = Mech::G_LOW[2][p];
        const double k0r = exp(l0 + l1 * lnT - l2 * invT);
        const double Pr = fmax(k0r * Mj, 1e-300);
        const double iPr1 = 1.0 / (1.0 + Pr);
        double F = 1.0, g = 0.0, dlnF_T = 0.0;
        if (Mech::G_TROEK[p]) {
          const double t0 = Mech::G_TROE[0][p], t2 = Mech::G_TROE[2][p], t4 = Mech::G_TROE[4][p];
          const double e3 = exp(Mech::G_TROE[1][p] * T), e1 = exp(Mech::G_TROE[3][p] * T);
          const double e2 = Mech::G_TROE[5][p] != 0.0 ? exp(-t4 * invT) : 0.0;
          const double Fc = t0 * e3 + t2 * e1 + e2;
          const double lFc = log10(Fc);
          const double cc = -0.4 - 0.67 * lFc, nn = 0.75 - 1.27 * lFc;
          const double xx = log10(Pr) + cc;
          const double DD = 1.0 / (nn - 0.14 * xx);
          const double f1 = xx * DD;
          const double iden = 1.0 / (1.0 + f1 * f1);
          F = exp(Mech::T_LN10 * lFc * iden);
          if (JAC) {
            g = -lFc * 2.0 * f1 * nn * DD * DD * iden * iden;
            const double df1 = (-0.67 * nn + 1.27 * xx) * DD * DD;
            const double dlF = iden - lFc * 2.0 * f1 * df1 * iden * iden;
            const double dFc = Mech::G_TROE[6][p] * e3 + Mech::G_TROE[7][p] * e1 +
                               t4 * invT * invT * e2;
            dlnF_T = dlF * dFc / Fc;
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
    // 1/Kc = prod exp(g_p/RT) prod exp(-g_r/RT) (P_atm/RT)^-dnu
    const double iKc = rev ? (b0.y * b1.y * b2.y) * (a0.y * a1.y * a2.y) * fac : 0.0;
    const double r01 = a0.x * a1.x, p01 = b0.x * b1.x;
    const double Pb = p01 * b2.x;
    const double net = r01 * a2.x - iKc * Pb;
    sh[O_Q + p] = kf * net;
    if constexpr (JAC) {
      lds_double* rb = sh + O_RB + l;
      const lds_double* hr = sh + O_HR;
      const double dlnKc =
          ((hr[p0] + hr[p1] + hr[p2]) - (hr[r0] + hr[r1] + hr[r2]) - double(dnu)) * invT;
      rb[0] = kf * a1.x * a2.x;
      rb[G] = kf * a0.x * a2.x;
      rb[2 * G] = kf * r01;
      const double kb = -kf * iKc;
      rb[3 * G] = kb * b1.x * b2.x;
      rb[4 * G] = kb * b0.x * b2.x;
      rb[5 * G] = kb * p01;
      rb[6 * G] = rev ? kf * (dlnk * net + iKc * Pb * dlnKc) : kf * dlnk * net;
      rb[7 * G] = kind ? dkdM * net : 0.0;
    }
  }

  // Species thermo of lane l into LDS and the third-body sums: what the reactions read.
  template <bool JAC>
  __device__ static void prelude(double T, double lnT, double invT, double Cl, int l, double tm,
                                 lds_double* sh) {
    const bool lo = T < tm;
    double c[8];
    {
      const dv2* p = reinterpret_cast<const dv2*>(&Mech::G_G[lo ? 0 : 1][0][l][0]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const dv2 v = p[i * G];
        c[2 * i] = v.x;
        c[2 * i + 1] = v.y;
      }
    }
    const double gRT = fma(T, fma(T, fma(T, fma(T, c[4], c[3]), c[2]), c[1]), c[0]) - c[5] * lnT +
                       c[6] * invT;
    const double E = exp(gRT);
    const double iE = 1.0 / E;  // lanes >= N: coefficients 0, so E = iE = 1
    if (l <= N) {
      const double C = l < N ? Cl : 1.0;
      ((lds_dv2*)(sh + O_RP))[l] = dv2{C, iE};
      ((lds_dv2*)(sh + O_PP))[l] = dv2{C, E};
      if (JAC) {
        const dv2* p = reinterpret_cast<const dv2*>(&Mech::G_H[lo ? 0 : 1][0][l][0]);
        const dv2 h0 = p[0], h1 = p[G], h2 = p[2 * G];
        sh[O_HR + l] = fma(T, fma(T, fma(T, fma(T, h2.x, h1.y), h1.x), h0.y), h0.x) + h2.y * invT;
      }
    }
    if (l == 0) sh[O_Q + P] = 0.0;
    if constexpr (NS > 0) {
      const double ctot = Grp::sum(Cl);
      Grp::sync();
      if (l < NS) {
        double M = ctot;
#pragma unroll
        for (int e = 0; e < Mech::G_MN; ++e)
          M += Mech::G_MD[e][l] * sh[O_RP + 2 * Mech::G_MI[e][l]];
        sh[O_M + l] = M;
      }
    }
    Grp::sync();
  }

  // production rate of species l from the q in LDS: a chunk of entries per lane, then the chunks
  // of each species
  __device__ static double gather(int l, lds_double* sh) {
    double acc = 0.0;
    const lds_char* q = (const lds_char*)(sh + O_Q);
#pragma unroll
    for (int i = 0; i < Mech::G_L4; ++i) {
      const iv4 e = *reinterpret_cast<const iv4*>(&Mech::G_GE[i][l][0]);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        acc = fma((double)(e[u] >> 24), *(const lds_double*)(q + (e[u] & 0xffff)), acc);
    }
    sh[O_PS + l] = acc;
    Grp::sync();
    const int cp = Mech::G_CP[l], b = cp & 255, m = cp >> 8;
    double wd = 0.0;
#pragma unroll
    for (int u = 0; u < Mech::G_CMAX; ++u)
      if (u < m) wd += sh[O_PS + b + u];
    return wd;
  }

  // f(t, y) for the lane's component (0 on lanes >= n).
  template <bool MUL = false>
  __device__ static double rhs(double t, double yl, int l, double rhoe0, double rhoesrc,
                               double srcl, double tm, lds_double* sh,
                               const double* rmul = nullptr) {
    l = after(l, yl);
    const bool sp = l < N;
    const double ys = sp ? yl : 0.0;
    const double irho = 1.0 / Grp::sum(ys);
    double ec[6], ek, cvk;
    const double T = T_from_e((rhoe0 + t * rhoesrc) * irho, ys * irho, l, Grp::bcast(yl, N), tm,
                              ec, ek, cvk);
    const double lnT = log(T), invT = 1.0 / T;
    prelude<false>(T, lnT, invT, ys * Mech::G_IWT[l], l, tm, sh);
#pragma unroll 1
    for (int r = 0; r < RR; ++r) reaction<false, MUL>(after(G * r + l, lnT), l, T, lnT, invT, sh, rmul);
    Grp::sync();
    const double wd = gather(l, sh);
    const double fk = sp ? Mech::G_WT[l] * wd + srcl : 0.0;
    const double num = rhoesrc - Grp::sum(ek * fk);
    const double D = Grp::sum(ys * cvk);
    Grp::sync();
    return l == N ? num / D : fk;
  }

  // Exact Jacobian of rhs() into Jg (row l on lane l). The rows are summed in device memory rather
  // than LDS: n x n doubles of LDS per cell (23 KB at n = 54) would leave one wave per SIMD.
  template <bool MUL = false, int CS = G, int RS = 1>
  __device__ static void jac(double t, double yl, int l, double rhoe0, double rhoesrc, double srcl,
                             double tm, lds_double* sh, double* Jg, const double* rmul = nullptr) {
    l = after(l, yl);
    const bool sp = l < N;
    double* Jr = Jg + l * RS;
    if (l < n)
#pragma unroll 4
      for (int m = 0; m < n; ++m) Jr[m * CS] = 0.0;  // column N stays 0
    const double ys = sp ? yl : 0.0;
    const double irho = 1.0 / Grp::sum(ys);
    double ec[6], ek, cvk;
    const double T = T_from_e((rhoe0 + t * rhoesrc) * irho, ys * irho, l, Grp::bcast(yl, N), tm,
                              ec, ek, cvk);
    const double lnT = log(T), invT = 1.0 / T;
    prelude<true>(T, lnT, invT, ys * Mech::G_IWT[l], l, tm, sh);
    double dwdT = 0.0, tb[NS > 0 ? NS : 1];
#pragma unroll
    for (int s = 0; s < NS; ++s) tb[s] = 0.0;
#pragma unroll 1
    for (int r = 0; r < RR; ++r) {
      Grp::sync();  // the previous round's derivatives have been read
      reaction<true, MUL>(after(G * r + l, lnT), l, T, lnT, invT, sh, rmul);
      Grp::sync();
      const int e1 = Mech::G_JO[r + 1];
#pragma unroll 1
      for (int i = Mech::G_JO[r]; i < e1; ++i) {
        const int je = Mech::G_JE[i][l];
        if (je) {
          const int q = je & 255;
          const double nu = (double)((je << 16) >> 24);
          const uint64_t pk = Mech::G_RP[G * r + q];
          const lds_double* rb = sh + O_RB + q;
          dwdT += nu * rb[6 * G];
#pragma unroll
          for (int u = 0; u < 6; ++u) {
            const int m = (int)(pk >> (8 * u)) & 255;
            if (m < N)
              __builtin_amdgcn_global_atomic_fadd_f64((glb_double*)(Jr + m * CS), nu * rb[u * G]);
          }
          if (NS > 0 && G * r < Mech::G_NTB) {
            const int kind = (int)(pk >> 56) & 3, ef = (int)(pk >> 48) & 255;
            const double c = kind ? nu * rb[7 * G] : 0.0;
#pragma unroll
            for (int s = 0; s < NS; ++s) tb[s] += s == ef ? c : 0.0;
          }
        }
      }
    }
    const double wd = gather(l, sh);
    // energy row and the T-elimination (CellModel::jac)
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
    double tbs = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) tbs += tb[s];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // the adds are done
#pragma unroll 2
    for (int m = 0; m < N; ++m) {
      double a = sp ? load_l2(Jr + m * CS) + tbs : 0.0;
#pragma unroll
      for (int s = 0; s < NS; ++s) a += tb[s] * Mech::T_EFFD[s][m];
      a *= Wk * Mech::IW[m];
      // T row, column m: dNdx_m = -sum_k e_k A_km
      const double dNdx = -Grp::sum(ek * a);
      const double em = Grp::bcast(ek, m), cm = Grp::bcast(cvk, m);
      if (l < n) Jr[m * CS] = sp ? a - b * em : (dNdx - fT * cm) * iD - dfTdT * em * iD;
    }
    Grp::sync();
  }

  // a <- row of the inverse of the matrix whose row l is in a (lanes < n), by Gauss-Jordan
  // elimination with partial pivoting, rows staying on their lanes: with lane p the pivot of
  // column kap(p), lane p ends with row kap(p) of the inverse, its columns in pivot order (column c
  // belongs to the right-hand side component of the lane that was column c's pivot). The pivot search
  // is a maximum over |a| with the lane in the low six mantissa bits (a choice among values equal to
  // 2^-46). Pivot rows are broadcast through LDS as they stand and scaled once at the end: the other
  // rows' multipliers carry 1 / pivot. Returns 0, or k + 1 when column k has no usable pivot.
  __device__ static int invert(double (&a)[n], int l, int& kap, lds_double* sh) {
    l = after(l, a[0]);
    lds_dv2* pr = (lds_dv2*)(sh + O_PR);
    bool used = l >= n;
    kap = 0;
    int ier = 0;
    double scale = 0.0;
    // every step eliminates the column in a[0] and stores the row shifted down by one, so the loop
    // is rolled (unrolled it is n times the code, more than the instruction cache at n = 54) and
    // after n steps every column is back in its place
#pragma unroll 1
    for (int k = 0; k < n; ++k) {
      const double v = used ? 0.0 : fabs(a[0]);
      const long long key = (__double_as_longlong(v) & ~63ll) | l;
      const double best = Grp::max(__longlong_as_double(key));
      if (!(best >= 2.3e-308) && ier == 0) ier = k + 1;
      const bool piv = !used && l == (int)(__double_as_longlong(best) & 63);
      if (piv) {
        pr[(n + 1) / 2] = dv2{a[0], 0.0};
#pragma unroll
        for (int c = 0; c < n; c += 2)
          pr[c / 2] = dv2{c + 1 < n ? a[c + 1 < n ? c + 1 : 0] : 1.0,
                          c + 2 < n ? a[c + 2 < n ? c + 2 : 0] : 1.0};
      }
      Grp::sync();
      const double inv = 1.0 / pr[(n + 1) / 2].x;
      const double f = piv ? 0.0 : a[0] * inv;
      const double last = piv ? 1.0 : 0.0;
      if (piv) {
        scale = inv;
        used = true;
        kap = k;
      }
#pragma unroll
      for (int c = 0; c < n; c += 2) {
        const dv2 p = pr[c / 2];
        a[c] = fma(-f, p.x, c + 1 < n ? a[c + 1 < n ? c + 1 : 0] : last);
        if (c + 1 < n) a[c + 1 < n ? c + 1 : 0] = fma(-f, p.y, c + 2 < n ? a[c + 2 < n ? c + 2 : 0] : last);
        if (c % 16 == 14) __asm__ __volatile__("" ::: "memory");  // at most 16 columns in flight
      }
      Grp::sync();
    }
#pragma unroll
    for (int c = 0; c < n; ++c) a[c] *= scale;
    return ier;
  }

  // x_l of M x = b from invert()'s rows; b_l on lane l (0 on lanes >= n).
  __device__ static double solve(const double (&a)[n], int kap, double b, int l, lds_double* sh) {
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
};

}  // namespace pelec
