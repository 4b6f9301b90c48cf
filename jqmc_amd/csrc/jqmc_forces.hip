// gfx950 kernels of the position derivatives of the local energy and of ln|Psi| per walker, and of the
// space-warp force terms (jqmc_mcmc.py:744-852, swct.py:63-150).  The reference takes them by JAX
// reverse-mode differentiation of compute_local_energy and evaluate_ln_wavefunction; here the same
// derivatives come from a hand-written adjoint, flattened over electrons and quadrature points like the
// local energy itself (AO values recomputed in every pass, never stored):
//
//   k_el_prep, k_el_hrows   q_e and h_e = C^T q_e, the lists of electrons with projected ECP terms
//   k_fr_kinetic  lanes = 64 electrons: Jastrow gradient gJ_e, D1_e, T_e, d ln|Psi| / dR_n
//   k_fr_points   lanes = quadrature points: the ratios rho_k, then a second AO sweep for the adjoints of the
//                 points and nuclei and the ECP parts of the adjoints of the J3 field (gbar_e) and AO row (w_e)
//   k_fr_adjoint  lanes = 64 electrons: the kinetic parts of gbar_e and w_e
//   k_fr_qbar     qbar_e = C w_e on the matrix cores
//   k_init_jsums, k_init_jfield_mfma   the J3 value adjoint J^T sum_{f<e} gbar_f + J sum_{f>e} gbar_f: the
//                 operator of the J3 field itself, so the same matrix-core product
//   k_fr_pairing  per walker: Gbar^-1, Gbar = -G^-T Gbar^-1 G^-T and the orbital-value adjoints phibar_e;
//                 k_el_hrows adds C^T phibar_e to the J3 value adjoint
//   k_fr_orbital  lanes = 64 electrons: AO gradient / Hessian / gradient of the Laplacian contracted with the
//                 AO-space adjoints into dE/dr_e and, with the opposite sign, into the nuclei
//   k_fr_out      per walker: the J1 / J2, Coulomb and local-ECP pair terms, the sums over electrons, ion-ion
//                 forces and the space-warp products
//
// The kinetic energy is written T = -1/2 sum_e [L_e + 2 D1_e . gJ_e + lJ_e + |gJ_e|^2] with
// D1_e = grad a(r_e) . h_e and L_e = lap a(r_e) . h_e, so its adjoints are local to each electron's row or
// column of G plus the dependence of q_e on G^-1 and on the other spin's orbitals.  Sums per nucleus are kept
// per electron (and wave) and added in a fixed order.  Plain FP64 systems only.
//
// 2048 benzene walkers (30 electrons, 228 AOs, 12 nuclei, six points per electron): 20.8 ms as one kernel with
// one wave per walker (two waves per SIMD, J3 times every gbar row element by element, three exponentials per
// AO and pass), 2.39 ms so: points 0.83, J3 product 0.34, adjoint 0.25, orbital 0.23, kinetic 0.22, out 0.20.
#pragma once

#include "jqmc_derivs.hip"
#include "jqmc_elp.hip"

namespace jqmc {

// f', f'', f''' of the one-body term of one electron-nucleus pair (jastrow_factor.py:672-711).
__device__ __forceinline__ void j1_f123(int type, double a, double c, double A, double r, double& f1, double& f2,
                                        double& f3) {
  if (type == 1) {
    const double e = exp_nonpos(-a * c * r);
    f1 = -A * c / 2.0 * e;
    f2 = A * a * c * c / 2.0 * e;
    f3 = -A * a * a * c * c * c / 2.0 * e;
  } else {
    const double den = 1.0 + a * c * r;
    f1 = -A / (2.0 * den * den);
    f2 = A * a * c / (den * den * den);
    f3 = -3.0 * A * a * a * c * c / (den * den * den * den);
  }
}

// f', f'', f''' of the two-body pair function (jastrow_factor.py:1207-1230).
__device__ __forceinline__ void j2_f123(int type, double a, double r, double& f1, double& f2, double& f3) {
  if (type == 2) {
    const double den = 1.0 + a * r;
    f1 = 0.5 / (den * den);
    f2 = -a / (den * den * den);
    f3 = 3.0 * a * a / (den * den * den * den);
  } else {
    const double e = exp_nonpos(-a * r);
    f1 = 0.5 * e;
    f2 = -a / 2.0 * e;
    f3 = a * a / 2.0 * e;
  }
}

// d/du [ dJ . grad f(|u|) + lc lap f(|u|) ] = (f'' (u^.dJ) - f'/r (u^.dJ) + lc (f''' + 2f''/r - 2f'/r^2)) u^
// + f'/r dJ, into out (added).
__device__ __forceinline__ void radial_adjoint(double ux, double uy, double uz, double f1, double f2, double f3,
                                               const double* dJ, double lc, double* out) {
  const double r = fmax(sqrt(ux * ux + uy * uy + uz * uz), 1.0e-12);
  const double hx = ux / r, hy = uy / r, hz = uz / r;
  const double ud = hx * dJ[0] + hy * dJ[1] + hz * dJ[2];
  const double c = f2 * ud - f1 / r * ud + lc * (f3 + 2.0 * f2 / r - 2.0 * f1 / (r * r));
  out[0] += c * hx + f1 / r * dJ[0];
  out[1] += c * hy + f1 / r * dJ[1];
  out[2] += c * hz + f1 / r * dJ[2];
}

// dP_n/dx of the tabulated Legendre polynomials P_0..P_6.
__device__ __forceinline__ double legendre_d(int n, double x) {
  switch (n) {
    case 0: return 0.0;
    case 1: return 1.0;
    case 2: return 3.0 * x;
    case 3: return 0.5 * (15.0 * x * x - 3.0);
    case 4: return 0.125 * (140.0 * x * x * x - 60.0 * x);
    case 5: return 0.125 * (315.0 * x * x * x * x - 210.0 * x * x + 15.0);
    case 6: return (1386.0 * x * x * x * x * x - 1260.0 * x * x * x + 210.0 * x) / 16.0;
    default: return __builtin_nan("");
  }
}

// ---------------------------------------------------------------- buffers

// One call's arrays over M = W n_el flattened electrons i = w n_el + e; sums per nucleus are [n][c][i].
struct FrJob {
  const Sys* sys;
  WalkT<double> wk;
  int64_t W;
  const double* RT;              // quadrature rotations (NULL: identity)
  const double *Q, *H;           // q rows (M, n_orb) and h rows (M, n_ao)
  const double *jold, *vpot;     // k_el_prep: J1 + J2 at the electrons, bare potential
  const int *elist, *necp;
  double *te, *jc;               // (M) kinetic energies, a(r_e) . g_e
  double* el;                    // (FR_EL, M): gJ, dJ = -(D1 + gJ), D1, S_e (non-local ECP energy), 1 where listed
  double *wv, *gbar;             // (M, n_ao) adjoints of the AO rows and of the J3 fields
  const double* a0;              // (M, n_ao) AO-value adjoints (without - S_e g_e)
  double *qbar, *phib, *t;       // (M, n_orb)
  int phib_add;                  // phib holds the J3 part of the AO-value adjoints already
  double *RA, *RL;               // dE/dR_n and d ln|Psi|/dR_n (opposite sign) by electron
  double* part;                  // FR_WAVES x the same size: partial sums of the waves; then (W, n_nuc, 12)
  double* re;                    // (3, M) dE/dr_e
  double* pt;                    // (W, n_el, nv, 4) points of the listed electrons and s_k
};
constexpr int FR_EL = 11, FR_WAVES = 4;

// Pointers of a call over W walkers carved from base (NULL: the number of doubles only).
struct FrBuf {
  double *q, *h, *wv, *gbar, *x, *qbar, *phib, *t, *te, *jc, *el, *jold, *vpot, *RA, *RL, *part, *re, *pt;
  int *elist, *necp;
  int64_t doubles;
  FrBuf(const Sys& s, int64_t W, double* base) {
    double* p = base;
    auto take = [&](int64_t n) {
      double* r = p;
      p += n;
      return r;
    };
    const int64_t M = W * s.n_el, na = s.n_ao, no = s.n_orb, nn = 3 * (int64_t)s.n_nuc;
    q = take(M * no);
    h = s.orb_is_mo ? take(M * na) : q;
    wv = take(M * na);
    gbar = s.j3_on ? take(M * na) : nullptr;
    x = s.j3_on ? take(M * na) : nullptr;
    qbar = s.orb_is_mo ? take(M * no) : wv;
    phib = take(M * no);
    t = take(M * no);
    te = take(M);
    jc = take(M);
    el = take(FR_EL * M);
    jold = take(M);
    vpot = take(W);
    RA = take(nn * M);
    RL = take(nn * M);
    part = take(FR_WAVES * nn * M);
    re = take(3 * M);
    pt = take(s.ecp_on ? 4 * M * s.nv : 0);
    elist = reinterpret_cast<int*>(take((M + 1) / 2));
    necp = reinterpret_cast<int*>(take((W + 1) / 2));
    doubles = p - base;
  }
};

// Walkers that a call of W takes at a time, so that its workspace stays bounded (benzene: 1.3 GB): at most 2^17
// electrons, 2048 blocks of the launches over electrons, in parts of equal size.  32768 walkers of N (7 electrons)
// took 1286 us in parts of 4096 walkers and 800 so, H2 1122 and 471 us (with the waves of k_fr_out below).
constexpr int64_t FR_ELECTRONS = 1 << 17;
inline int64_t fr_chunk(const Sys& s, int64_t W) {
  const int64_t most = FR_ELECTRONS / s.n_el, parts = (W + most - 1) / most;
  return parts > 0 ? (W + parts - 1) / parts : 0;
}

// Size limit of the systems taken, in bytes: one walker's vectors of every pass within 64 KiB, as one wave per
// walker would hold them in LDS.  No launch needs this much (k_fr_pairing 16 n_up^2 bytes, at most 64 KiB with
// n_up <= 64; the others fixed tiles); the limit stands, so that what is refused does not change.
inline int64_t forces_lds_bytes(const Sys& s) {
  const int64_t ne = s.n_el, nv = std::max(s.nv, 1), na = s.n_ao, no = s.n_orb, nu = s.n_up, nn = s.n_nuc;
  return 8 * (6 * ne + nu * nu + 9 + 14 * nv + std::max(s.ecp_max_terms, 1) + no + 8 * na + std::max(no, nu) + 6 * nn +
              10 * ne + (int64_t)s.n_shell * PTS_CHUNK);
}

// ---------------------------------------------------------------- AO derivatives

// Radial factor sum c e^{-Z r^2} of a piece and its derivatives: grad R = R[1] x, grad R[1] = R[2] x, ... (the
// record holds -Z log2 e), NR of them.
template <int NR>
__device__ __forceinline__ void piece_radials(const PieceHead<double>& hd, double r2, double* R) {
  auto sum = [&](auto Nc) {
    constexpr int NP = decltype(Nc)::value;
    double e[NP];
    piece_exps<NP>(hd, r2, e);
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const double z = (2.0 * LN2) * hd.zc[2 * q];
      double v = hd.zc[2 * q + 1] * e[q];
#pragma unroll
      for (int k = 0; k < NR; ++k) {
        R[k] = q == 0 ? v : R[k] + v;
        v *= z;
      }
    }
  };
  const int np = hd.info & 15;
  if (np == 3)
    sum(std::integral_constant<int, 3>{});
  else if (np == 1)
    sum(std::integral_constant<int, 1>{});
  else if (np == 2)
    sum(std::integral_constant<int, 2>{});
  else
    sum(std::integral_constant<int, 4>{});
}
template <int NR>
__device__ __forceinline__ void table_radials(CSys& s, int p, double r2, double* R) {
#pragma unroll
  for (int k = 0; k < NR; ++k) R[k] = 0.0;
  const CPtr<PieceMore<double>> more = cview(s.pm64) + p;
  const int q1 = more->p1;
  for (int q = more->p0; q < q1; ++q) {
    const double Z = cview(s.td.prim_exp)[q];
    double v = cview(s.td.prim_coef)[q] * exp_nonpos(-Z * r2);
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      R[k] += v;
      v *= -2.0 * Z;
    }
  }
}

// x^n and its derivatives up to the third.
__device__ __forceinline__ void pow_d(int n, double x, double* d) {
  const double f = (double)n;
  d[0] = ipow(x, n);
  d[1] = n >= 1 ? f * ipow(x, n - 1) : 0.0;
  d[2] = n >= 2 ? f * (f - 1.0) * ipow(x, n - 2) : 0.0;
  d[3] = n >= 3 ? f * (f - 1.0) * (f - 2.0) * ipow(x, n - 3) : 0.0;
}

// Polynomial of AO a from the term tables: value, gradient, Laplacian and, with kThird, the Hessian
// (xx, yy, zz, xy, xz, yz) and the gradient of the Laplacian.
struct PolyD {
  double P, G[3], lap, H[6], gl[3];
};
template <bool kThird>
__device__ __forceinline__ PolyD table_poly(CSys& s, int a, double dx, double dy, double dz) {
  PolyD r{};
  const CPtr<int> tp = cview(s.ao_tp);
  const CPtr<int> pw = cview(s.term_pow);
  const int t1 = tp[a + 1];
  for (int t = tp[a]; t < t1; ++t) {
    const double c = cview(s.td.term_coef)[t];
    double X[4], Y[4], Z[4];
    pow_d(pw[3 * t], dx, X);
    pow_d(pw[3 * t + 1], dy, Y);
    pow_d(pw[3 * t + 2], dz, Z);
    r.P += c * (X[0] * Y[0] * Z[0]);
    r.G[0] += c * (X[1] * Y[0] * Z[0]);
    r.G[1] += c * (X[0] * Y[1] * Z[0]);
    r.G[2] += c * (X[0] * Y[0] * Z[1]);
    const double hx = c * (X[2] * Y[0] * Z[0]), hy = c * (X[0] * Y[2] * Z[0]), hz = c * (X[0] * Y[0] * Z[2]);
    r.lap += hx + hy + hz;
    if constexpr (kThird) {
      r.H[0] += hx;
      r.H[1] += hy;
      r.H[2] += hz;
      r.H[3] += c * (X[1] * Y[1] * Z[0]);
      r.H[4] += c * (X[1] * Y[0] * Z[1]);
      r.H[5] += c * (X[0] * Y[1] * Z[1]);
      r.gl[0] += c * (X[3] * Y[0] * Z[0] + X[1] * Y[2] * Z[0] + X[1] * Y[0] * Z[2]);
      r.gl[1] += c * (X[2] * Y[1] * Z[0] + X[0] * Y[3] * Z[0] + X[0] * Y[1] * Z[2]);
      r.gl[2] += c * (X[2] * Y[0] * Z[1] + X[0] * Y[2] * Z[1] + X[0] * Y[0] * Z[3]);
    }
  }
  return r;
}

// Monomial i of degree L, its gradient and Laplacian.
template <int L, int I>
__device__ __forceinline__ void mono_vgl(double x, double y, double z, double& P, double* G, double& lap) {
  constexpr int a = Mono<L>::nx(I), b = Mono<L>::ny(I), c = Mono<L>::nz(I);
  auto pw = [](double v, int n) { return n <= 0 ? 1.0 : (n == 1 ? v : (n == 2 ? v * v : v * v * v)); };
  const double X = pw(x, a), Y = pw(y, b), Z = pw(z, c);
  P = X * Y * Z;
  G[0] = a > 0 ? (a * pw(x, a - 1)) * (Y * Z) : 0.0;
  G[1] = b > 0 ? (b * pw(y, b - 1)) * (X * Z) : 0.0;
  G[2] = c > 0 ? (c * pw(z, c - 1)) * (X * Y) : 0.0;
  lap = (a > 1 ? (a * (a - 1)) * (pw(x, a - 2) * (Y * Z)) : 0.0) + (b > 1 ? (b * (b - 1)) * (pw(y, b - 2) * (X * Z)) : 0.0) +
        (c > 1 ? (c * (c - 1)) * (pw(z, c - 2) * (X * Y)) : 0.0);
}

// f(I) for I = 0 .. N - 1 with I a compile-time constant.
template <int N, int I = 0, typename F>
__device__ __forceinline__ void unroll_c(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unroll_c<N, I + 1>(f);
  }
}

// Calls f with the degree of the piece as a constant.
template <typename F>
__device__ __forceinline__ void with_degree(int l, F&& f) {
  if (l == 0)
    f(std::integral_constant<int, 0>{});
  else if (l == 1)
    f(std::integral_constant<int, 1>{});
  else if (l == 2)
    f(std::integral_constant<int, 2>{});
  else
    f(std::integral_constant<int, 3>{});
}

// f'(r) / r of the two-body and one-body terms.
__device__ __forceinline__ double j2_slope(const JasPar& J, double r, double ri) {
  if (J.j2_type == 2) {
    const double i = rcp_nr(fma(J.a2, r, 1.0));
    return 0.5 * i * i * ri;
  }
  return 0.5 * exp2_prod(-J.a2 * LOG2E, r) * ri;
}
__device__ __forceinline__ double j1_slope(const JasPar& J, double c, double A, double r, double ri) {
  const double ac = J.a1 * c;
  if (J.j1_type == 1) return -A * (c / 2.0) * exp2_prod(-ac * LOG2E, r) * ri;
  const double i = rcp_nr(fma(ac, r, 1.0));
  return -0.5 * A * i * i * ri;
}

// ---------------------------------------------------------------- electrons, 64 per block

// Staged tiles of a block of 64 flattened electrons: thread (lane) takes columns c3 .. c3 + 2 of rows
// r4 + 16 r of a chunk.
struct FrTile {
  int c3, r4, n_rows, na;
  __device__ __forceinline__ FrTile(int lane, int rows, int n_ao) : c3(3 * (lane & 3)), r4(lane >> 2), n_rows(rows), na(n_ao) {}
  // rows past the last electron repeat it, columns past the chunk's end hold other AOs (all unused)
  __device__ __forceinline__ int64_t at(int r, int x, int a0) const {
    return (int64_t)(r4 + 16 * r < n_rows ? r4 + 16 * r : n_rows - 1) * na + (a0 + c3 + x < na ? a0 + c3 + x : na - 1);
  }
  __device__ __forceinline__ void load(const double* src, int a0, double* v) const {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int x = 0; x < 3; ++x) v[3 * r + x] = src ? src[at(r, x, a0)] : 0.0;
  }
  __device__ __forceinline__ void to_lds(double* t, const double* v, const double* sc) const {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int x = 0; x < 3; ++x) t[(r4 + 16 * r) * EL_LD + c3 + x] = v[3 * r + x] * sc[x];
  }
  __device__ __forceinline__ void to_mem(double* dst, int a0, int n, const double* t, const double* sc,
                                         const double* add) const {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r4 + 16 * r < n_rows)
#pragma unroll
        for (int x = 0; x < 3; ++x)
          if (c3 + x < n)
            dst[(int64_t)(r4 + 16 * r) * na + a0 + c3 + x] = fma(t[(r4 + 16 * r) * EL_LD + c3 + x], sc[x], add[3 * r + x]);
  }
};

// Adds x to the sums of nucleus n ([n][c][i], p at i); the first time that a wave comes to n they are stored
// (p was cleared), which needs no read: AOs are ordered by nucleus as a rule.
struct NucSums {
  double* p;
  int64_t M;
  uint64_t seen = 0;
  __device__ __forceinline__ NucSums(double* p_, int64_t M_) : p(p_), M(M_) {}
  __device__ __forceinline__ void add(int n, const double* x, bool act) {
    const bool first = n < 64 && !(seen >> n & 1);
    if (n < 64) seen |= 1ull << n;
    if (act)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        double* q = p + (int64_t)(3 * n + c) * M;
        *q = first ? x[c] : *q + x[c];
      }
  }
};

// Lanes = 64 flattened electrons, the chunks of the AO range split over the four waves in order.  Bound by
// the latency of the rows of h and g and of the sums per nucleus (14 % vector issue; 0.84 GB in 219 us for 2048
// benzene walkers).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) k_fr_kinetic(FrJob J) {
  extern __shared__ double smem[];
  CSys& s = csys(J.sys);
  const int wave = wave_id(), lane = lane_id();
  const int nu = s.n_up, nd = s.n_dn, ne = s.n_el, na = s.n_ao, nn = s.n_nuc;
  const int64_t M = J.W * ne, i0 = (int64_t)blockIdx.x * EL_KIN_ROWS;
  const int n_rows = M - i0 < EL_KIN_ROWS ? (int)(M - i0) : EL_KIN_ROWS;
  double* h_s = smem + wave * 2 * EL_KIN_ROWS * EL_LD;
  double* g_s = h_s + EL_KIN_ROWS * EL_LD;
  const bool act = lane < n_rows;
  const int64_t i = i0 + (act ? lane : 0), w = i / ne;
  const int e = (int)(i - w * ne);
  const double* ru = J.wk.r_up + w * 3 * nu;
  const double* rd = J.wk.r_dn + w * 3 * nd - 3 * nu;
  const double* rp = (e < nu ? ru : rd) + 3 * e;
  const double ex = rp[0], ey = rp[1], ez = rp[2];
  double* RL = J.part + wave * 3 * nn * M + i;
  NucSums sums(RL, M);
  if (act) {
    for (int k = 0; k < 3 * nn; ++k) RL[k * M] = 0.0;
    if (wave == 0) {
      for (int k = 0; k < 3 * nn; ++k) J.RA[k * M + i] = 0.0;
      for (int k = 0; k < 3; ++k) J.re[k * M + i] = 0.0;
    }
  }
  const FrTile T(lane, n_rows, na);
  const bool j3 = s.j3_on;
  const double* gsrc = j3 ? J.wk.jfield + i0 * na : nullptr;
  const double* hsrc = J.H + i0 * na;
  const CPtr<int> chk = cview(s.el_chunks);
  const int cb = s.n_chunk * wave / FR_WAVES, ce = s.n_chunk * (wave + 1) / FR_WAVES;
  const CPtr<PieceRec<double>> rec = cview(s.pc64);

  // ---- first sweep: the fields
  double D[3] = {0, 0, 0}, Lh = 0.0, gJ[3] = {0, 0, 0}, lJ = 0.0, jc = 0.0;
  {
    double dD[3] = {0, 0, 0}, dG[3] = {0, 0, 0};
    int nuc = -1;
    auto flush = [&]() {
      if (nuc >= 0) {
        const double x[3] = {dD[0] + dG[0], dD[1] + dG[1], dD[2] + dG[2]};
        sums.add(nuc, x, act);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          D[c] += dD[c];
          gJ[c] += dG[c];
          dD[c] = dG[c] = 0.0;
        }
      }
    };
    double hr[12], gr[12];
    if (cb < ce) {
      T.load(hsrc, chk[4 * cb + 2], hr);
      T.load(gsrc, chk[4 * cb + 2], gr);
    }
    PieceHead<double> hd;
    hd.load(rec + (cb < ce ? chk[4 * cb] : 0));
    const double* hrow = h_s + lane * EL_LD;
    const double* grow = g_s + lane * EL_LD;
    for (int c = cb; c < ce; ++c) {
      double sc[3];
#pragma unroll
      for (int x = 0; x < 3; ++x) sc[x] = s.el_scale[c * EL_CH + T.c3 + x];
      T.to_lds(h_s, hr, sc);
      T.to_lds(g_s, gr, sc);
      lds_order();
      if (c + 1 < ce) {
        T.load(hsrc, chk[4 * c + 6], hr);
        T.load(gsrc, chk[4 * c + 6], gr);
      }
      const int p1 = chk[4 * c + 1], ca = chk[4 * c + 2];
      for (int p = chk[4 * c]; p < p1; ++p) {
        const int o = hd.a0 - ca, info = hd.info, a0 = hd.a0;
        if (const int n = cview(s.ao_nuc)[a0]; n != nuc) {
          flush();
          nuc = n;
        }
        const double dx = ex - hd.c[0], dy = ey - hd.c[1], dz = ez - hd.c[2];
        const double r2u = dx * dx + dy * dy + dz * dz;
        double R[3];
        if (info & PIECE_ANY) {
          table_radials<3>(s, p, r2u, R);
          hd.load(rec + p + 1);
          const int n = info >> 16;
          for (int q = 0; q < n; ++q) {
            const PolyD y = table_poly<false>(s, a0 + q, dx, dy, dz);
            const double h = hrow[o + q], g = grow[o + q], pr = y.P * R[1];
            const double v[3] = {fma(pr, dx, R[0] * y.G[0]), fma(pr, dy, R[0] * y.G[1]), fma(pr, dz, R[0] * y.G[2])};
            const double vl = R[0] * y.lap + 2.0 * R[1] * (dx * y.G[0] + dy * y.G[1] + dz * y.G[2]) +
                              (3.0 * R[1] + r2u * R[2]) * y.P;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              dD[k] = fma(h, v[k], dD[k]);
              dG[k] = fma(g, v[k], dG[k]);
            }
            Lh = fma(h, vl, Lh);
            lJ = fma(g, vl, lJ);
            jc = fma(g, R[0] * y.P, jc);
          }
          continue;
        }
        const double r2 = fmin(r2u, EXP2_XMAX);
        piece_radials<3>(hd, r2, R);
        hd.load(rec + p + 1);
        with_degree((info >> 4) & 15, [&](auto Lc) {
          constexpr int l = decltype(Lc)::value, N = Mono<l>::N;
          const double ll = fma(r2, R[2], (3.0 + 2.0 * l) * R[1]);  // Laplacian factor of degree l
          auto add = [&](const double* f, double* d, double& L_, double& P) {
            double G[3], lap;
            poly_vgl<l>(f, dx, dy, dz, P, G, lap);
            const double mp = R[1] * P;
            d[0] += fma(mp, dx, R[0] * G[0]);
            d[1] += fma(mp, dy, R[0] * G[1]);
            d[2] += fma(mp, dz, R[0] * G[2]);
            L_ = fma(ll, P, L_);
            if constexpr (l >= 2) L_ = fma(R[0], lap, L_);
          };
          double P, f[N];
#pragma unroll
          for (int q = 0; q < N; ++q) f[q] = hrow[o + q];
          add(f, dD, Lh, P);
          if (j3) {
#pragma unroll
            for (int q = 0; q < N; ++q) f[q] = grow[o + q];
            add(f, dG, lJ, P);
            jc = fma(R[0], P, jc);
          }
        });
      }
      lds_order();
    }
    flush();
  }
  const JasPar JP(s);
  if (JP.j1_type) {
    for (int n = wave; n < nn; n += FR_WAVES) {
      const CPtr<double> q = cview(s.nuc_pos) + 3 * n;
      const double u[3] = {ex - q[0], ey - q[1], ez - q[2]};
      const double r = fmax(sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]), 1.0e-12);
      double f1, f2, f3;
      j1_f123(JP.j1_type, JP.a1, cview(s.j1_c)[n], cview(s.j1_A)[n], r, f1, f2, f3);
      const double fr = f1 / r, x[3] = {fr * u[0], fr * u[1], fr * u[2]};
#pragma unroll
      for (int c = 0; c < 3; ++c) gJ[c] += x[c];
      sums.add(n, x, act);
      lJ += f2 + 2.0 * fr;
    }
  }
  if (JP.j2_type) {
    for (int f = wave; f < ne; f += FR_WAVES) {
      const double* q = (f < nu ? ru : rd) + 3 * f;
      const double dx = ex - q[0], dy = ey - q[1], dz = ez - q[2];
      double ri;
      const double r = sqrt_nr(fmax(dx * dx + dy * dy + dz * dz, 1.0e-24), ri);
      double f1, f2, f3;
      j2_f123(JP.j2_type, JP.a2, r, f1, f2, f3);
      const bool on = f != e;
      const double fr = on ? f1 * ri : 0.0;
      gJ[0] += fr * dx;
      gJ[1] += fr * dy;
      gJ[2] += fr * dz;
      lJ += on ? f2 + 2.0 * fr : 0.0;
    }
  }
  // the totals
  double v[9] = {D[0], D[1], D[2], Lh, gJ[0], gJ[1], gJ[2], lJ, jc};
#pragma unroll
  for (int q = 0; q < 9; ++q) h_s[q * WAVE + lane] = v[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    v[q] = smem[q * WAVE + lane];
    for (int x = 1; x < FR_WAVES; ++x) v[q] += smem[x * 2 * EL_KIN_ROWS * EL_LD + q * WAVE + lane];
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    D[c] = v[c];
    gJ[c] = v[4 + c];
  }
  const double dJ[3] = {-(D[0] + gJ[0]), -(D[1] + gJ[1]), -(D[2] + gJ[2])};
  if (act) {
    if (wave == 0) {
      J.te[i] = -0.5 * (v[3] + 2.0 * (D[0] * gJ[0] + D[1] * gJ[1] + D[2] * gJ[2]) + v[7] +
                        (gJ[0] * gJ[0] + gJ[1] * gJ[1] + gJ[2] * gJ[2]));
      J.jc[i] = v[8];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        J.el[c * M + i] = gJ[c];
        J.el[(3 + c) * M + i] = dJ[c];
        J.el[(6 + c) * M + i] = D[c];
      }
      J.el[9 * M + i] = J.el[10 * M + i] = 0.0;
    }
    // the sums of d ln|Psi| / dR, written before the barriers
    for (int k = wave; k < 3 * nn; k += FR_WAVES) {
      double x = 0.0;
#pragma unroll
      for (int q = 0; q < FR_WAVES; ++q) x += J.part[((int64_t)q * 3 * nn + k) * M + i];
      J.RL[k * M + i] = x;
    }
  }
}

// The adjoints of the same electrons' J3 field, gbar_e = dJ . grad a - 1/2 lap a, and AO row,
// w_e = -gJ . grad a - 1/2 lap a, onto the parts that k_fr_points left for the listed electrons (gbar_e
// without - S_e a(r_e)).  Bound by writing and reading these rows.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) k_fr_adjoint(FrJob J) {
  extern __shared__ double smem[];
  CSys& s = csys(J.sys);
  const int wave = wave_id(), lane = lane_id();
  const int nu = s.n_up, nd = s.n_dn, ne = s.n_el, na = s.n_ao;
  const int64_t M = J.W * ne, i0 = (int64_t)blockIdx.x * EL_KIN_ROWS;
  const int n_rows = M - i0 < EL_KIN_ROWS ? (int)(M - i0) : EL_KIN_ROWS;
  double* h_s = smem + wave * 2 * EL_KIN_ROWS * EL_LD;
  double* g_s = h_s + EL_KIN_ROWS * EL_LD;
  const int64_t i = i0 + (lane < n_rows ? lane : 0), w = i / ne;
  const int e = (int)(i - w * ne);
  const double* rp = e < nu ? J.wk.r_up + (w * nu + e) * 3 : J.wk.r_dn + (w * nd + (e - nu)) * 3;
  const double ex = rp[0], ey = rp[1], ez = rp[2];
  const FrTile T(lane, n_rows, na);
  const bool j3 = s.j3_on;
  const CPtr<int> chk = cview(s.el_chunks);
  const int cb = s.n_chunk * wave / FR_WAVES, ce = s.n_chunk * (wave + 1) / FR_WAVES;
  const CPtr<PieceRec<double>> rec = cview(s.pc64);
  double gJ[3], dJ[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    gJ[c] = J.el[c * M + i];
    dJ[c] = J.el[(3 + c) * M + i];
  }
  const double S = J.el[9 * M + i];
  bool listed[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int q = T.r4 + 16 * r;
    listed[r] = q < n_rows && J.el[10 * M + i0 + q] != 0.0;
  }
  double wr[12], br[12];
  auto load = [&](int c) {
    const int a0 = chk[4 * c + 2];
#pragma unroll
    for (int q = 0; q < 12; ++q) {
      const int64_t at = i0 * na + T.at(q / 3, q % 3, a0);
      wr[q] = listed[q / 3] ? J.wv[at] : 0.0;
      br[q] = listed[q / 3] && j3 ? J.gbar[at] : 0.0;
    }
  };
  if (cb < ce) load(cb);
  PieceHead<double> hd;
  hd.load(rec + (cb < ce ? chk[4 * cb] : 0));
  double* wrow = h_s + lane * EL_LD;
  double* brow = g_s + lane * EL_LD;
  for (int c = cb; c < ce; ++c) {
    const int p1 = chk[4 * c + 1], ca = chk[4 * c + 2];
    for (int p = chk[4 * c]; p < p1; ++p) {
      const int o = hd.a0 - ca, info = hd.info, a0 = hd.a0;
      const double dx = ex - hd.c[0], dy = ey - hd.c[1], dz = ez - hd.c[2];
      const double r2u = dx * dx + dy * dy + dz * dz;
      const double gd = gJ[0] * dx + gJ[1] * dy + gJ[2] * dz, dd = dJ[0] * dx + dJ[1] * dy + dJ[2] * dz;
      double R[3];
      auto put = [&](int q, double P, const double* G, double lap) {
        const double pr = P * R[1];
        wrow[o + q] = -fma(pr, gd, R[0] * (gJ[0] * G[0] + gJ[1] * G[1] + gJ[2] * G[2])) - 0.5 * lap;
        brow[o + q] = fma(pr, dd, R[0] * (dJ[0] * G[0] + dJ[1] * G[1] + dJ[2] * G[2])) - 0.5 * lap - S * (R[0] * P);
      };
      if (info & PIECE_ANY) {
        table_radials<3>(s, p, r2u, R);
        hd.load(rec + p + 1);
        const int n = info >> 16;
        for (int q = 0; q < n; ++q) {
          const PolyD y = table_poly<false>(s, a0 + q, dx, dy, dz);
          put(q, y.P, y.G,
              R[0] * y.lap + 2.0 * R[1] * (dx * y.G[0] + dy * y.G[1] + dz * y.G[2]) + (3.0 * R[1] + r2u * R[2]) * y.P);
        }
        continue;
      }
      const double r2 = fmin(r2u, EXP2_XMAX);
      piece_radials<3>(hd, r2, R);
      hd.load(rec + p + 1);
      with_degree((info >> 4) & 15, [&](auto Lc) {
        constexpr int l = decltype(Lc)::value, N = Mono<l>::N;
        const double ll = fma(r2, R[2], (3.0 + 2.0 * l) * R[1]);
        unroll_c<N>([&](auto I) {
          double P, G[3], lap;
          mono_vgl<l, decltype(I)::value>(dx, dy, dz, P, G, lap);
          put(decltype(I)::value, P, G, fma(ll, P, R[0] * lap));
        });
      });
    }
    double sc[3];
#pragma unroll
    for (int x = 0; x < 3; ++x) sc[x] = s.el_scale[c * EL_CH + T.c3 + x];
    lds_order();
    T.to_mem(J.wv + i0 * na, ca, chk[4 * c + 3], h_s, sc, wr);
    if (j3) T.to_mem(J.gbar + i0 * na, ca, chk[4 * c + 3], g_s, sc, br);
    if (c + 1 < ce) load(c + 1);
    lds_order();
  }
}

// ---------------------------------------------------------------- quadrature points

// A wave takes up to ten listed electrons of four walkers, one quadrature point per lane (an electron with
// more than 64 points one part after the other).  Two AO sweeps: ratios, then the adjoints; per chunk of
// twelve AOs the values at the points go through LDS and are summed per electron into w_e and gbar_e, per
// run of AOs on one nucleus the gradients are summed into dE/dR.  Bound by the FP64 vector rate (44 %) and the
// latency of the staged rows: three waves per SIMD with some words spilled outside the sweeps took 829 us for
// 2048 benzene walkers, two waves 1129 us.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) k_fr_points(FrJob J, int n_groups) {
  __shared__ double h_sh[4][EL_SLOTS * EL_LD + 3], g_sh[4][EL_SLOTS * EL_LD + 3];
  __shared__ double v_sh[4][EL_CH * (WAVE + 1)], r_sh[4][3 * (WAVE + 1)], c_sh[4][2 * WAVE], j_sh[4][3][WAVE];
  CSys& s = csys(J.sys);
  const int wave = wave_id(), lane = lane_id();
  const int nu = s.n_up, nd = s.n_dn, ne = s.n_el, na = s.n_ao, nn = s.n_nuc, nv = s.nv;
  const int64_t M = J.W * ne;
  const int npt = nv < WAVE ? nv : WAVE, parts = (nv + WAVE - 1) / WAVE;
  int n_slots = WAVE / npt;
  if (n_slots > EL_SLOTS) n_slots = EL_SLOTS;
  // the first group of every four walkers, then the second, ... (see k_el_points)
  const int64_t id = (int64_t)blockIdx.x * 4 + wave, n_quad = (J.W + 3) / 4, gi = id / n_quad;
  if (gi >= n_groups) return;
  const int64_t w0 = 4 * (id - gi * n_quad);
  const CPtr<int> cnt = cview(J.necp);
  const int c0 = cnt[w0], c1 = w0 + 1 < J.W ? cnt[w0 + 1] : 0, c2 = w0 + 2 < J.W ? cnt[w0 + 2] : 0,
            c3 = w0 + 3 < J.W ? cnt[w0 + 3] : 0;
  const int base = (int)gi * n_slots;
  int total = c0 + c1 + c2 + c3 - base;
  if (total > n_slots) total = n_slots;
  if (total <= 0) return;
  auto slot = [&](int sl, int64_t& w, int& e, int& rank, int& nuc) {
    int x = base + (sl < total ? sl : 0), wl = 0;
    if (x >= c0) {
      x -= c0;
      ++wl;
      if (x >= c1) {
        x -= c1;
        ++wl;
        if (x >= c2) {
          x -= c2;
          ++wl;
        }
      }
    }
    rank = x;
    w = w0 + wl;
    const int y = J.elist[w * ne + x];
    e = y & 255;
    nuc = y >> 8;
  };
  int64_t w;
  int e, rank, nuc;
  const int my = (int)(((float)lane + 0.5f) / (float)npt);
  slot(my, w, e, rank, nuc);
  const int myrow = my < total ? my : 0;
  // staged elements: column lane % 12 of rows lane / 12 and lane / 12 + 5; and this lane's (slot, component)
  const int scol = lane % EL_CH, srow = lane < 60 ? lane / EL_CH : EL_SLOTS;
  int64_t rowof[2], red_i = 0;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    int64_t wr;
    int er, t0, t1;
    slot(srow + 5 * r, wr, er, t0, t1);
    rowof[r] = (wr * ne + er) * na;
  }
  const int red_s = lane / 3, red_c = lane - 3 * red_s;
  const bool red = red_s < total;
  int red_nuc;
  {
    int64_t wr;
    int er, t0;
    slot(red_s, wr, er, t0, red_nuc);
    red_i = wr * ne + er;
  }
  const double* ru = J.wk.r_up + w * 3 * nu;
  const double* rd = J.wk.r_dn + w * 3 * nd - 3 * nu;
  const double* rp = (e < nu ? ru : rd) + 3 * e;
  const double ex = rp[0], ey = rp[1], ez = rp[2];
  double Rm[9] = {1.0, 0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0, 1.0};
  if (J.RT) {
#pragma unroll
    for (int q = 0; q < 9; ++q) Rm[q] = J.RT[9 * w + q];
  }
  const int64_t i = w * ne + e;
  const bool j3 = s.j3_on;
  const CPtr<int> chk = cview(s.el_chunks);
  const CPtr<PieceRec<double>> rec = cview(s.pc64);
  const int n_chunk = s.n_chunk;
  const JasPar JP(s);
  double* h_s = h_sh[wave];
  double* g_s = g_sh[wave];
  double* v_s = v_sh[wave];
  double* r_s = r_sh[wave];
  double* c_s = c_sh[wave];  // (c_k = W_k e^dJ, s_k = W_k rho_k) per point
  const double* hrow = h_s + myrow * EL_LD;
  const double* grow = g_s + myrow * EL_LD;
  double hr[2], gr[2], gsc = 0.0;
  auto load = [&](int c) {
    const int a = chk[4 * c + 2] + scol < na ? chk[4 * c + 2] + scol : na - 1;
    gsc = s.el_scale[c * EL_CH + scol];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      hr[r] = J.H[rowof[r] + a];
      gr[r] = j3 ? J.wk.jfield[rowof[r] + a] : 0.0;
    }
  };
  auto stage = [&]() {
    if (lane < 60) {
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        h_s[(srow + 5 * r) * EL_LD + scol] = hr[r] * gsc;
        g_s[(srow + 5 * r) * EL_LD + scol] = gr[r] * gsc;
      }
    }
  };
  // sum of x over the points of this lane's (slot, component), x given per lane and component
  auto slot_sum = [&](const double* x) {
#pragma unroll
    for (int c = 0; c < 3; ++c) r_s[c * (WAVE + 1) + lane] = x[c];
    lds_order();
    double t = 0.0;
    if (red)
      for (int q = 0; q < npt; ++q) t += r_s[red_c * (WAVE + 1) + red_s * npt + q];
    lds_order();
    return t;
  };

  for (int part = 0; part < parts; ++part) {
    const int k = part * WAVE + lane - my * npt;
    const bool valid = my < total && k < nv;
    const int kk = valid ? k : 0;
    const double m0 = s.mesh_pts[3 * kk], m1 = s.mesh_pts[3 * kk + 1], m2 = s.mesh_pts[3 * kk + 2];
    const double g0 = m0 * Rm[0] + m1 * Rm[3] + m2 * Rm[6], g1 = m0 * Rm[1] + m1 * Rm[4] + m2 * Rm[7],
                 g2 = m0 * Rm[2] + m1 * Rm[5] + m2 * Rm[8];
    const double rx = s.nuc_pos[3 * nuc] - ex, ry = s.nuc_pos[3 * nuc + 1] - ey, rz = s.nuc_pos[3 * nuc + 2] - ez;
    double gni;
    const double rn2 = rx * rx + ry * ry + rz * rz, rn = sqrt(rn2), ri = 1.0 / rn;
    sqrt_nr(g0 * g0 + g1 * g1 + g2 * g2, gni);
    const double px = ex + (rx + rn * g0), py = ey + (ry + rn * g1), pz = ez + (rz + rn * g2);
    const double hx = -rx * ri, hy = -ry * ri, hz = -rz * ri;  // (r_e - R) / |r_e - R|
    // projector weight W_k = sum_t V_t (2 l + 1) P_l(cos) w_k and its gradient with respect to r_e - R (each
    // where it is used: registers)
    auto projector = [&](double& pwt, double* dW) {
      pwt = 0.0;
      const double cth = (hx * g0 + hy * g1 + hz * g2) * gni, wk_ = s.mesh_w[kk];
      double rad = 0.0, ang = 0.0;
      const int nt = s.ecp_nt[nuc];
      for (int t = 0; t < nt; ++t) {
        const int o = nuc * s.ecp_max_terms + t, l = s.ecp_l[o];
        const double V = (ri * ri) * s.ecp_coef[o] * rpow(rn, s.ecp_pow[o]) * exp2_prod(-s.ecp_exp[o] * LOG2E, rn2);
        const double f = (2 * l + 1) * wk_, leg = f * legendre(l, cth);
        pwt += V * leg;
        rad += V * ((s.ecp_pow[o] - 2.0) * ri - 2.0 * s.ecp_exp[o] * rn) * leg;
        ang += V * f * legendre_d(l, cth);
      }
      const double ai = ang * ri;
      dW[0] = rad * hx + ai * (g0 * gni - cth * hx);
      dW[1] = rad * hy + ai * (g1 * gni - cth * hy);
      dW[2] = rad * hz + ai * (g2 * gni - cth * hz);
    };
    // J1 + J2 at the point and its gradient
    double jn = 0.0, JG[3] = {0.0, 0.0, 0.0};
    if (JP.j2_type)
      for (int f = 0; f < ne; ++f) {
        const double* q = (f < nu ? ru : rd) + 3 * f;
        const double dx = px - q[0], dy = py - q[1], dz = pz - q[2];
        double qi;
        const double r = sqrt_nr(fmax(dx * dx + dy * dy + dz * dz, 1.0e-24), qi);
        const double u = j2_value(JP, r), fr = f == e ? 0.0 : j2_slope(JP, r, qi);
        jn += f == e ? 0.0 : u;
        JG[0] += fr * dx;
        JG[1] += fr * dy;
        JG[2] += fr * dz;
      }
    if (JP.j1_type)
      for (int n = 0; n < nn; ++n) {
        const CPtr<double> q = cview(s.nuc_pos) + 3 * n;
        const double dx = px - q[0], dy = py - q[1], dz = pz - q[2];
        double qi;
        const double r = sqrt_nr(fmax(dx * dx + dy * dy + dz * dz, 1.0e-24), qi);
        const double c = cview(s.j1_c)[n], A = cview(s.j1_A)[n], fr = j1_slope(JP, c, A, r, qi);
        jn += j1_value(JP, c, A, r);
        JG[0] += fr * dx;
        JG[1] += fr * dy;
        JG[2] += fr * dz;
      }

#pragma unroll
    for (int c = 0; c < 3; ++c) j_sh[wave][c][lane] = JG[c];

    // ---- first sweep: the ratio
    double det = 0.0, dj = 0.0;
    {
      PieceHead<double> hd;
      hd.load(rec);
      load(0);
      for (int c = 0; c < n_chunk; ++c) {
        stage();
        lds_order();
        if (c + 1 < n_chunk) load(c + 1);
        const int p1 = chk[4 * c + 1], ca = chk[4 * c + 2];
        for (int p = chk[4 * c]; p < p1; ++p) {
          const int o = hd.a0 - ca, info = hd.info, a0 = hd.a0;
          const double dx = px - hd.c[0], dy = py - hd.c[1], dz = pz - hd.c[2];
          const double r2 = dx * dx + dy * dy + dz * dz;
          if (info & PIECE_ANY) {
            double R[1];
            table_radials<1>(s, p, r2, R);
            hd.load(rec + p + 1);
            const int n = info >> 16;
            for (int q = 0; q < n; ++q) {
              const double v = R[0] * poly_at<double>(s, a0 + q, dx, dy, dz);
              det = fma(v, hrow[o + q], det);
              dj = fma(v, grow[o + q], dj);
            }
            continue;
          }
          const double nr = piece_radial(hd, fmin(r2, EXP2_XMAX));
          hd.load(rec + p + 1);
          with_degree((info >> 4) & 15, [&](auto Lc) {
            constexpr int l = decltype(Lc)::value, N = Mono<l>::N;
            double f[N];
#pragma unroll
            for (int q = 0; q < N; ++q) f[q] = hrow[o + q];
            det = fma(nr, poly_dot<l>(f, dx, dy, dz), det);
#pragma unroll
            for (int q = 0; q < N; ++q) f[q] = grow[o + q];
            dj = fma(nr, poly_dot<l>(f, dx, dy, dz), dj);
          });
        }
        lds_order();
      }
    }
    const double Ek = exp(dj + ((jn - J.jold[i]) - (j3 ? J.jc[i] : 0.0)));
    double pwt, dW[3];
    projector(pwt, dW);
    const double rho = det * Ek, cw = valid ? pwt * Ek : 0.0, sk = valid ? pwt * rho : 0.0;
    c_s[2 * lane] = cw;
    c_s[2 * lane + 1] = sk;
    if (valid) {
      double* q = J.pt + (((w * ne + rank) * nv) + k) * 4;
      q[0] = px;
      q[1] = py;
      q[2] = pz;
      q[3] = sk;
    }
    lds_order();
    if (red && red_c == 0) {
      double t = 0.0;
      for (int q = 0; q < npt; ++q) t += c_s[2 * (red_s * npt + q) + 1];
      J.el[9 * M + red_i] += t;
      J.el[10 * M + red_i] = 1.0;
    }

    // ---- second sweep: pb = d E / d point, per nucleus the opposite of its sum, w_e and gbar_e
    double pb[3] = {0.0, 0.0, 0.0}, acc[3] = {0.0, 0.0, 0.0};
    int nuc_run = -1;
    uint64_t seen = part ? ~0ull : 0;  // as in NucSums
    auto to_nucleus = [&](int n, const double* x) {
      const double t = slot_sum(x);
      const bool first = n < 64 && !(seen >> n & 1);
      if (n < 64) seen |= 1ull << n;
      if (red) {
        double* q = J.RA + (int64_t)(3 * n + red_c) * M + red_i;
        *q = first ? -t : *q - t;
      }
    };
    auto flush = [&]() {
      if (nuc_run >= 0) {
        to_nucleus(nuc_run, acc);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          pb[c] += acc[c];
          acc[c] = 0.0;
        }
      }
    };
    PieceHead<double> hd;
    hd.load(rec);
    load(0);
    for (int c = 0; c < n_chunk; ++c) {
      stage();
      lds_order();
      const int p1 = chk[4 * c + 1], ca = chk[4 * c + 2], nc = chk[4 * c + 3];
      const double sc = gsc;
      if (c + 1 < n_chunk) load(c + 1);
      for (int p = chk[4 * c]; p < p1; ++p) {
        const int o = hd.a0 - ca, info = hd.info, a0 = hd.a0;
        if (const int n = cview(s.ao_nuc)[a0]; n != nuc_run) {
          flush();
          nuc_run = n;
        }
        const double dx = px - hd.c[0], dy = py - hd.c[1], dz = pz - hd.c[2];
        const double r2 = dx * dx + dy * dy + dz * dz;
        double R[2];
        if (info & PIECE_ANY) {
          table_radials<2>(s, p, r2, R);
          hd.load(rec + p + 1);
          const int n = info >> 16;
          for (int q = 0; q < n; ++q) {
            const PolyD y = table_poly<false>(s, a0 + q, dx, dy, dz);
            const double f = cw * hrow[o + q] + sk * grow[o + q], fp = f * y.P * R[1], fr = f * R[0];
            acc[0] += fma(fp, dx, fr * y.G[0]);
            acc[1] += fma(fp, dy, fr * y.G[1]);
            acc[2] += fma(fp, dz, fr * y.G[2]);
            v_s[(o + q) * (WAVE + 1) + lane] = R[0] * y.P;
          }
        } else {
          piece_radials<2>(hd, fmin(r2, EXP2_XMAX), R);
          hd.load(rec + p + 1);
          with_degree((info >> 4) & 15, [&](auto Lc) {
            constexpr int l = decltype(Lc)::value, N = Mono<l>::N;
            double f[N], P, G[3], lap;
#pragma unroll
            for (int q = 0; q < N; ++q) f[q] = fma(cw, hrow[o + q], sk * grow[o + q]);
            poly_vgl<l>(f, dx, dy, dz, P, G, lap);
            const double mp = R[1] * P;
            acc[0] += fma(mp, dx, R[0] * G[0]);
            acc[1] += fma(mp, dy, R[0] * G[1]);
            acc[2] += fma(mp, dz, R[0] * G[2]);
            unroll_c<N>([&](auto I) {
              double m, mg[3], ml;
              mono_vgl<l, decltype(I)::value>(dx, dy, dz, m, mg, ml);
              v_s[(o + decltype(I)::value) * (WAVE + 1) + lane] = R[0] * m;
            });
          });
        }
      }
      lds_order();
      // the electron's sums over its points
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int row = srow + 5 * r;
        if (row < total && scol < nc) {
          double tw = 0.0, tg = 0.0;
#pragma unroll 3
          for (int q = 0; q < npt; ++q) {
            const double v = v_s[scol * (WAVE + 1) + row * npt + q];
            tw = fma(c_s[2 * (row * npt + q)], v, tw);
            tg = fma(c_s[2 * (row * npt + q) + 1], v, tg);
          }
          const int64_t at = rowof[r] + ca + scol;
          J.wv[at] = part ? fma(sc, tw, J.wv[at]) : sc * tw;
          if (j3) J.gbar[at] = part ? fma(sc, tg, J.gbar[at]) : sc * tg;
        }
      }
      lds_order();
    }
    flush();
    if (JP.j1_type)
      for (int n = 0; n < nn; ++n) {
        const CPtr<double> q = cview(s.nuc_pos) + 3 * n;
        const double dx = px - q[0], dy = py - q[1], dz = pz - q[2];
        double qi;
        const double r = sqrt_nr(fmax(dx * dx + dy * dy + dz * dz, 1.0e-24), qi);
        const double f = sk * j1_slope(JP, cview(s.j1_c)[n], cview(s.j1_A)[n], r, qi);
        const double x[3] = {f * dx, f * dy, f * dz};
        to_nucleus(n, x);
      }
#pragma unroll
    for (int c = 0; c < 3; ++c) pb[c] = fma(sk, j_sh[wave][c][lane], pb[c]);
    projector(pwt, dW);
    // point r' = R + |r_e - R| g~: d r' / d r_e = g~ (r_e - R)^T / |r_e - R|, the rest moves with R
    const double gp = g0 * pb[0] + g1 * pb[1] + g2 * pb[2], rv = valid ? rho : 0.0;
    const double xe[3] = {fma(hx, gp, rv * dW[0]), fma(hy, gp, rv * dW[1]), fma(hz, gp, rv * dW[2])};
    const double te = slot_sum(xe), tp = slot_sum(pb);
    if (red) {
      J.re[red_c * M + red_i] += te;
      J.RA[(int64_t)(3 * red_nuc + red_c) * M + red_i] += tp - te;
    }
  }
}

// ---------------------------------------------------------------- orbital adjoints

// qbar_e = C w_e of the MO systems on the matrix cores, wave (w, row tile).
__global__ void __launch_bounds__(256) k_fr_qbar(FrJob J) {
  CSys& s = csys(J.sys);
  const int wave = wave_id(), lane = lane_id(), il = lane & 15, ih = lane >> 4;
  const int nu = s.n_up, nd = s.n_dn, ne = s.n_el, no = s.n_orb, na = s.n_ao;
  const int nut = (nu + 15) / 16, nt = nut + (nd + 15) / 16;
  const int64_t id = (int64_t)blockIdx.x * 4 + wave, w = id / nt;
  if (w >= J.W) return;
  const int rt = (int)(id - w * nt);
  const bool up = rt < nut;
  const int e0 = 16 * (up ? rt : rt - nut), n_sp = up ? nu : nd, off = up ? 0 : nu;
  const double* X = J.wv + (w * ne + off) * (int64_t)na;
  double* Y = J.qbar + (w * ne + off) * (int64_t)no;
  const double* C = up ? s.td.mo_up : s.td.mo_dn;
  const int er = e0 + il;
  for (int c0 = 0; c0 < no; c0 += 16) {
    const int c = c0 + il;
    const auto acc = mfma_rows(
        na, ih, [&](int k) { return (k < na && er < n_sp) ? X[(int64_t)er * na + k] : 0.0; },
        [&](int k) { return (k < na && c < no) ? C[(int64_t)c * na + k] : 0.0; });
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = e0 + JfMfma<double>::row(q, ih);
      if (r < n_sp && c < no) Y[(int64_t)r * no + c] = acc[q];
    }
  }
}

// One block per walker, its waves (fr_pairing_waves) on the 16 x 16 tiles of each product in turn; Gbar and one
// intermediate (n_up^2 each) in LDS.
inline int fr_pairing_waves(const Sys& s) { return std::min(FR_WAVES, (s.n_up + 15) / 16 * ((s.n_orb + 15) / 16)); }
__global__ void __launch_bounds__(256) k_fr_pairing(FrJob J) {
  extern __shared__ double smem[];
  CSys& s = csys(J.sys);
  const int wave = wave_id(), lane = lane_id(), il = lane & 15, ih = lane >> 4, nw = blockDim.x / WAVE;
  const int nu = s.n_up, nd = s.n_dn, ne = s.n_el, no = s.n_orb, un = s.n_unp;
  const int64_t w = blockIdx.x;
  const double* Gi = J.wk.Ginv + w * nu * nu;
  const double* P = J.wk.pair + w * ne * no;
  const double* qb = J.qbar + w * ne * (int64_t)no;
  double* t = J.t + w * ne * (int64_t)no;
  double* ph = J.phib + w * ne * (int64_t)no;
  double *A = smem, *B = smem + nu * nu;
  const bool add = J.phib_add;
  // st(r, c, sum_k fa(r, k) fb(k, c)) over an m x n product of depth d
  auto product = [&](int m, int n, int d, auto fa, auto fb, auto st) {
    const int ct = (n + 15) / 16, tiles = (m + 15) / 16 * ct;
    for (int x = wave; x < tiles; x += nw) {
      const int r0 = x / ct * 16, c0 = (x - x / ct * ct) * 16, r = r0 + il, c = c0 + il;
      const auto acc = mfma_rows(
          d, ih, [&](int k) { return (k < d && r < m) ? fa(r, k) : 0.0; },
          [&](int k) { return (k < d && c < n) ? fb(k, c) : 0.0; });
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int rr = r0 + JfMfma<double>::row(q, ih);
        if (rr < m && c < n) st(rr, c, acc[q]);
      }
    }
  };
  // Gbar^-1[j][c]: row j < n_dn: pair_dn_j . qbar_c + pair_up_c . qbar_{n_up + j}; the rows of unpaired
  // orbitals Lambda_u[:, j - n_dn] . qbar_c
  product(
      nu, nu, no, [&](int j, int k) { return j < nd ? P[(int64_t)(nu + j) * no + k] : s.td.lam_u[(int64_t)k * un + (j - nd)]; },
      [&](int k, int c) { return qb[(int64_t)c * no + k]; }, [&](int j, int c, double v) { A[j * nu + c] = v; });
  __syncthreads();
  product(
      nd, nu, no, [&](int j, int k) { return qb[(int64_t)(nu + j) * no + k]; },
      [&](int k, int c) { return P[(int64_t)c * no + k]; }, [&](int j, int c, double v) { A[j * nu + c] += v; });
  // sum over the other spin's electrons f of G^-1[..] qbar_f
  product(
      nu, no, nd, [&](int e, int j) { return Gi[j * nu + e]; },
      [&](int j, int l) { return qb[(int64_t)(nu + j) * no + l]; },
      [&](int e, int l, double v) { t[(int64_t)e * no + l] = v; });
  product(
      nd, no, nu, [&](int j, int c) { return Gi[j * nu + c]; }, [&](int c, int l) { return qb[(int64_t)c * no + l]; },
      [&](int j, int l, double v) { t[(int64_t)(nu + j) * no + l] = v; });
  __syncthreads();
  // Gbar = -G^-T (Gbar^-1 G^-T)
  product(
      nu, nu, nu, [&](int j, int m) { return A[j * nu + m]; }, [&](int m, int c) { return Gi[c * nu + m]; },
      [&](int j, int c, double v) { B[j * nu + c] = v; });
  __syncthreads();
  product(
      nu, nu, nu, [&](int i, int j) { return Gi[j * nu + i]; }, [&](int j, int c) { return B[j * nu + c]; },
      [&](int i, int c, double v) { A[i * nu + c] = -v; });
  __syncthreads();
  // phibar: Gbar against the other spin's pair rows, Lambda_p (up) or Lambda_p^T (dn) against t
  product(
      nu, no, nu, [&](int e, int j) { return A[e * nu + j]; },
      [&](int j, int k) { return j < nd ? P[(int64_t)(nu + j) * no + k] : s.td.lam_u[(int64_t)k * un + (j - nd)]; },
      [&](int e, int k, double v) { ph[(int64_t)e * no + k] = add ? ph[(int64_t)e * no + k] + v : v; });
  product(
      nd, no, nu, [&](int j, int i) { return A[i * nu + j]; }, [&](int i, int k) { return P[(int64_t)i * no + k]; },
      [&](int j, int k, double v) {
        double* q = ph + (int64_t)(nu + j) * no + k;
        *q = add ? *q + v : v;
      });
  __syncthreads();
  product(
      nu, no, no, [&](int e, int l) { return t[(int64_t)e * no + l]; },
      [&](int l, int k) { return s.td.lam_pT[(int64_t)l * no + k]; },
      [&](int e, int k, double v) { ph[(int64_t)e * no + k] += v; });
  product(
      nd, no, no, [&](int j, int l) { return t[(int64_t)(nu + j) * no + l]; },
      [&](int l, int k) { return s.td.lam_p[(int64_t)l * no + k]; },
      [&](int j, int k, double v) { ph[(int64_t)(nu + j) * no + k] += v; });
}

// Coefficients of sum_i f_i (u . grad) P_i over the monomials of degree L - 1, added to out.
template <int L>
__device__ __forceinline__ void poly_along(const double* f, const double* u, double* out) {
  unroll_c<Mono<L>::N>([&](auto I) {
    constexpr int a = Mono<L>::nx(decltype(I)::value), b = Mono<L>::ny(decltype(I)::value),
                  c = Mono<L>::nz(decltype(I)::value);
    const double v = f[decltype(I)::value];
    if constexpr (a > 0) out[mono_index(L - 1, a - 1, b)] = fma(a * u[0], v, out[mono_index(L - 1, a - 1, b)]);
    if constexpr (b > 0) out[mono_index(L - 1, a, b - 1)] = fma(b * u[1], v, out[mono_index(L - 1, a, b - 1)]);
    if constexpr (c > 0) out[mono_index(L - 1, a, b)] = fma(c * u[2], v, out[mono_index(L - 1, a, b)]);
  });
}

// Lanes = 64 flattened electrons, waves = quarters of the AO range.  The energy depends on the AO row of
// electron e as Phi = a0 . a + sum_c (-gJ_c h + dJ_c g) . d_c a - 1/2 (h + g) . lap a with these coefficients
// held fixed; grad Phi is dE/dr_e and, AO by AO, minus the force on its centre.  Per piece the coefficients of
// all its AOs are turned into polynomials first (B, G, A of degree L; the divergence of u B + w G of degree
// L - 1; the Laplacian of E = -(B + G) / 2 of degree L - 2), so that the four radial factors enter once per
// piece.  Bound by the FP64 vector rate and the three coefficient rows.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_fr_orbital(FrJob J) {
  extern __shared__ double smem[];
  CSys& s = csys(J.sys);
  const int wave = wave_id(), lane = lane_id();
  const int nu = s.n_up, nd = s.n_dn, ne = s.n_el, na = s.n_ao, nn = s.n_nuc;
  const int64_t M = J.W * ne, i0 = (int64_t)blockIdx.x * EL_KIN_ROWS;
  const int n_rows = M - i0 < EL_KIN_ROWS ? (int)(M - i0) : EL_KIN_ROWS;
  constexpr int TILE = EL_KIN_ROWS * EL_LD;
  double* h_s = smem + wave * 3 * TILE;
  double* g_s = h_s + TILE;
  double* a_s = g_s + TILE;
  const bool act = lane < n_rows;
  const int64_t i = i0 + (act ? lane : 0), w = i / ne;
  const int e = (int)(i - w * ne);
  const double* rp = e < nu ? J.wk.r_up + (w * nu + e) * 3 : J.wk.r_dn + (w * nd + (e - nu)) * 3;
  const double ex = rp[0], ey = rp[1], ez = rp[2];
  double* RA = J.part + wave * 3 * nn * M + i;
  if (act)
    for (int k = 0; k < 3 * nn; ++k) RA[k * M] = 0.0;
  NucSums sums(RA, M);
  double u[3], v[3];  // -gJ and dJ
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    u[c] = -J.el[c * M + i];
    v[c] = J.el[(3 + c) * M + i];
  }
  const FrTile T(lane, n_rows, na);
  const bool j3 = s.j3_on;
  double Sr[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    Sr[r] = j3 ? J.el[9 * M + i0 + (T.r4 + 16 * r < n_rows ? T.r4 + 16 * r : n_rows - 1)] : 0.0;
  const CPtr<int> chk = cview(s.el_chunks);
  const int cb = s.n_chunk * wave / FR_WAVES, ce = s.n_chunk * (wave + 1) / FR_WAVES;
  const CPtr<PieceRec<double>> rec = cview(s.pc64);
  double hr[12], gr[12], ar[12];
  auto load = [&](int c) {
    const int a0 = chk[4 * c + 2];
    T.load(J.H + i0 * na, a0, hr);
    T.load(j3 ? J.wk.jfield + i0 * na : nullptr, a0, gr);
    T.load(J.a0 + i0 * na, a0, ar);
  };
  if (cb < ce) load(cb);
  PieceHead<double> hd;
  hd.load(rec + (cb < ce ? chk[4 * cb] : 0));
  const double* hrow = h_s + lane * EL_LD;
  const double* grow = g_s + lane * EL_LD;
  const double* arow = a_s + lane * EL_LD;
  double re[3] = {0, 0, 0}, acc[3] = {0, 0, 0};
  int nuc = -1;
  auto flush = [&]() {
    if (nuc >= 0) {
      sums.add(nuc, acc, act);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        re[c] += acc[c];
        acc[c] = 0.0;
      }
    }
  };
  for (int c = cb; c < ce; ++c) {
    double sc[3];
#pragma unroll
    for (int x = 0; x < 3; ++x) sc[x] = s.el_scale[c * EL_CH + T.c3 + x];
#pragma unroll
    for (int q = 0; q < 12; ++q) ar[q] -= Sr[q / 3] * gr[q];
    T.to_lds(h_s, hr, sc);
    T.to_lds(g_s, gr, sc);
    T.to_lds(a_s, ar, sc);
    lds_order();
    if (c + 1 < ce) load(c + 1);
    const int p1 = chk[4 * c + 1], ca = chk[4 * c + 2];
    for (int p = chk[4 * c]; p < p1; ++p) {
      const int o = hd.a0 - ca, info = hd.info, a0 = hd.a0;
      if (const int n = cview(s.ao_nuc)[a0]; n != nuc) {
        flush();
        nuc = n;
      }
      const double dx = ex - hd.c[0], dy = ey - hd.c[1], dz = ez - hd.c[2], d[3] = {dx, dy, dz};
      const double r2u = dx * dx + dy * dy + dz * dz;
      double R[4];
      if (info & PIECE_ANY) {
        table_radials<4>(s, p, r2u, R);
        hd.load(rec + p + 1);
        const int n = info >> 16;
        for (int q = 0; q < n; ++q) {
          const PolyD y = table_poly<true>(s, a0 + q, dx, dy, dz);
          const double hv = hrow[o + q], gv = grow[o + q], av = arow[o + q], a2 = -0.5 * (hv + gv);
          const double a1[3] = {u[0] * hv + v[0] * gv, u[1] * hv + v[1] * gv, u[2] * hv + v[2] * gv};
          const double xa = dx * a1[0] + dy * a1[1] + dz * a1[2], ga = y.G[0] * a1[0] + y.G[1] * a1[1] + y.G[2] * a1[2];
          const double xg = dx * y.G[0] + dy * y.G[1] + dz * y.G[2], l1 = 3.0 * R[1] + r2u * R[2];
          const double Ha[3] = {y.H[0] * a1[0] + y.H[3] * a1[1] + y.H[4] * a1[2],
                                y.H[3] * a1[0] + y.H[1] * a1[1] + y.H[5] * a1[2],
                                y.H[4] * a1[0] + y.H[5] * a1[1] + y.H[2] * a1[2]};
          const double Hx[3] = {y.H[0] * dx + y.H[3] * dy + y.H[4] * dz, y.H[3] * dx + y.H[1] * dy + y.H[5] * dz,
                                y.H[4] * dx + y.H[5] * dy + y.H[2] * dz};
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            const double first = y.G[k] * R[0] + y.P * R[1] * d[k];
            const double second = Ha[k] * R[0] + (y.G[k] * xa + ga * d[k]) * R[1] + y.P * (a1[k] * R[1] + d[k] * xa * R[2]);
            const double third = y.gl[k] * R[0] + y.lap * R[1] * d[k] + 2.0 * ((y.G[k] + Hx[k]) * R[1] + xg * R[2] * d[k]) +
                                 y.G[k] * l1 + y.P * d[k] * (5.0 * R[2] + r2u * R[3]);
            acc[k] += av * first + second + a2 * third;
          }
        }
        continue;
      }
      const double r2 = fmin(r2u, EXP2_XMAX);
      piece_radials<4>(hd, r2, R);
      hd.load(rec + p + 1);
      with_degree((info >> 4) & 15, [&](auto Lc) {
        constexpr int l = decltype(Lc)::value, N = Mono<l>::N;
        double B[N], G[N], A[N], lap;
#pragma unroll
        for (int q = 0; q < N; ++q) {
          B[q] = hrow[o + q];
          G[q] = grow[o + q];
          A[q] = arow[o + q];
        }
        double Bv, Gv, Av, Bg[3], Gg[3], Ag[3];
        poly_vgl<l>(B, dx, dy, dz, Bv, Bg, lap);
        poly_vgl<l>(G, dx, dy, dz, Gv, Gg, lap);
        poly_vgl<l>(A, dx, dy, dz, Av, Ag, lap);
        const double ux = u[0] * dx + u[1] * dy + u[2] * dz, vx = v[0] * dx + v[1] * dy + v[2] * dz;
        const double Ev = -0.5 * (Bv + Gv), Vx = fma(ux, Bv, vx * Gv);
        if constexpr (l >= 1) {
          constexpr int N1 = Mono<l - 1>::N;
          double Dc[N1], Dv, Dg[3];
#pragma unroll
          for (int q = 0; q < N1; ++q) Dc[q] = 0.0;
          poly_along<l>(B, u, Dc);
          poly_along<l>(G, v, Dc);
          poly_vgl<(l >= 1 ? l - 1 : 0)>(Dc, dx, dy, dz, Dv, Dg, lap);
          Av += Dv;
#pragma unroll
          for (int k = 0; k < 3; ++k) Ag[k] += Dg[k];
        }
        if constexpr (l >= 2) {
          constexpr int N2 = Mono<l - 2>::N;
          double Lc2[N2], Lv, Lg[3];
#pragma unroll
          for (int q = 0; q < N2; ++q) Lc2[q] = 0.0;
          unroll_c<N>([&](auto I) {
            constexpr int a = Mono<l>::nx(decltype(I)::value), b = Mono<l>::ny(decltype(I)::value),
                          c_ = Mono<l>::nz(decltype(I)::value);
            const double E = -0.5 * (B[decltype(I)::value] + G[decltype(I)::value]);
            if constexpr (a > 1) Lc2[mono_index(l - 2, a - 2, b)] = fma((double)(a * (a - 1)), E, Lc2[mono_index(l - 2, a - 2, b)]);
            if constexpr (b > 1) Lc2[mono_index(l - 2, a, b - 2)] = fma((double)(b * (b - 1)), E, Lc2[mono_index(l - 2, a, b - 2)]);
            if constexpr (c_ > 1) Lc2[mono_index(l - 2, a, b)] = fma((double)(c_ * (c_ - 1)), E, Lc2[mono_index(l - 2, a, b)]);
          });
          poly_vgl<(l >= 2 ? l - 2 : 0)>(Lc2, dx, dy, dz, Lv, Lg, lap);
          Av += Lv;
#pragma unroll
          for (int k = 0; k < 3; ++k) Ag[k] += Lg[k];
        }
        // Phi = (A + div V + lap E) R + (V . x) R1 + ((2 l + 3) R1 + r^2 R2) E
        const double e1 = fma(r2, R[2], (2.0 * l + 3.0) * R[1]);
        const double cx = R[1] * Av + R[2] * fma(2.0 * l + 5.0, Ev, Vx) + r2 * R[3] * Ev;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          double x = fma(cx, d[k], R[1] * fma(u[k], Bv, v[k] * Gv));
          if constexpr (l >= 1)
            x += R[0] * Ag[k] + R[1] * fma(ux, Bg[k], vx * Gg[k]) - 0.5 * e1 * (Bg[k] + Gg[k]);
          acc[k] += x;
        }
      });
    }
    lds_order();
  }
  flush();
#pragma unroll
  for (int c = 0; c < 3; ++c) h_s[c * WAVE + lane] = re[c];
  __syncthreads();
  if (act) {
    if (wave == 0) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        double x = J.re[c * M + i];
        for (int q = 0; q < FR_WAVES; ++q) x += smem[q * 3 * TILE + c * WAVE + lane];
        J.re[c * M + i] = x;
      }
    }
    for (int k = wave; k < 3 * nn; k += FR_WAVES) {
      double x = J.RA[k * M + i];
#pragma unroll
      for (int q = 0; q < FR_WAVES; ++q) x -= J.part[((int64_t)q * 3 * nn + k) * M + i];
      J.RA[k * M + i] = x;
    }
  }
}

// ---------------------------------------------------------------- the walkers' results

struct FrOut {
  double *e_L, *dE_dr, *dE_dR, *dlnpsi_dr, *dlnpsi_dR, *force_HF, *force_PP;
  int swct;
};

// One block per walker, lanes = electrons; the partners, points and nuclei in four parts shared by the block's waves,
// whose number changes no bit.  Four waves as long as all walkers' fit the chip (three per SIMD), then no more than
// the walker has partners for: 2048 walkers of H2 (2 electrons), whole call, 98 us with four waves and 87 with one
// (k_fr_pairing alike); 64 walkers 69 and 74.
inline int fr_out_waves(const Sys& s, int64_t W) {
  return W * FR_WAVES <= 3 * 1024 ? FR_WAVES : std::min(FR_WAVES, (std::max(s.n_el, s.n_nuc) + 3) / 4);
}
__global__ void __launch_bounds__(256) k_fr_out(FrJob J, FrOut O) {
  __shared__ double p_sh[FR_WAVES][3][WAVE];
  CSys& s = csys(J.sys);
  const int wave = wave_id(), lane = lane_id(), nw = blockDim.x / WAVE;
  const int nu = s.n_up, nd = s.n_dn, ne = s.n_el, nn = s.n_nuc, nv = s.nv;
  const int64_t w = blockIdx.x, M = J.W * ne;
  double* sums = J.part + w * 12 * nn;  // per nucleus: dE/dR, -dln|Psi|/dR, warped parts of both
  for (int k = threadIdx.x; k < 12 * nn; k += blockDim.x) sums[k] = 0.0;
  const CPtr<double> ru = cview(J.wk.r_up) + w * 3 * nu;
  const CPtr<double> rd = cview(J.wk.r_dn) + w * 3 * nd;
  const CPtr<double> el = cview(J.el) + w * ne;
  const CPtr<double> np = cview(s.nuc_pos);
  const int n_ecp = s.ecp_on && nv > 0 ? J.necp[w] : 0;
  const JasPar JP(s);
  double en[2] = {0.0, 0.0};
  __syncthreads();
  for (int e0 = 0; e0 < ne; e0 += WAVE) {
    const int e = e0 + lane < ne ? e0 + lane : e0;
    const bool act = e0 + lane < ne;
    const int64_t i = w * ne + e;
    const double* rp = e < nu ? J.wk.r_up + (w * nu + e) * 3 : J.wk.r_dn + (w * nd + (e - nu)) * 3;
    const double ex = rp[0], ey = rp[1], ez = rp[2];
    double re[3], dJ[3], dl[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      dJ[c] = J.el[(3 + c) * M + i];
      dl[c] = -dJ[c];  // D1 + gJ = d ln|Psi| / d r_e
    }
    const double S = J.el[9 * M + i];
    if (act) {
      en[0] += J.te[i];
      en[1] += S;
    }
    if (e0 > 0) __syncthreads();
    for (int g = wave; g < FR_WAVES; g += nw) {
#pragma unroll
      for (int c = 0; c < 3; ++c) re[c] = g == 0 ? J.re[c * M + i] : 0.0;
      // e-e pairs: e's own terms and those of its partners together (each is odd in r_e - r_f)
      for (int f = g; f < ne; f += FR_WAVES) {
        const CPtr<double> q = f < nu ? ru + 3 * f : rd + 3 * (f - nu);
        const double ux = ex - q[0], uy = ey - q[1], uz = ez - q[2];
        const double d2 = ux * ux + uy * uy + uz * uz;
        if (f == e) continue;
        const double d = sqrt(d2), c0 = -1.0 / (d2 * d);
        re[0] += c0 * ux;
        re[1] += c0 * uy;
        re[2] += c0 * uz;
        if (JP.j2_type) {
          double f1, f2, f3;
          const double r = fmax(d, 1.0e-12);
          j2_f123(JP.j2_type, JP.a2, r, f1, f2, f3);
          const double D[3] = {dJ[0] - el[3 * M + f], dJ[1] - el[4 * M + f], dJ[2] - el[5 * M + f]};
          radial_adjoint(ux, uy, uz, f1, f2, f3, D, -1.0, re);
          const double c = -(S + el[9 * M + f]) * f1 / r;
          re[0] += c * ux;
          re[1] += c * uy;
          re[2] += c * uz;
        }
      }
      // the other electrons' quadrature points move with r_e through J2
      if (JP.j2_type)
        for (int j = g; j < n_ecp; j += FR_WAVES) {
          const int x = cview(J.elist)[w * ne + j] & 255;
          const CPtr<double> q = cview(J.pt) + (w * ne + j) * (int64_t)nv * 4;
          for (int k = 0; k < nv; ++k) {
            const double ux = q[4 * k] - ex, uy = q[4 * k + 1] - ey, uz = q[4 * k + 2] - ez;
            double ri;
            const double r = sqrt_nr(fmax(ux * ux + uy * uy + uz * uz, 1.0e-24), ri);
            const double c = x == e ? 0.0 : q[4 * k + 3] * j2_slope(JP, r, ri);
            re[0] -= c * ux;
            re[1] -= c * uy;
            re[2] -= c * uz;
          }
        }
      // nuclei
      for (int n = g; n < nn; n += FR_WAVES) {
        const double ux = ex - np[3 * n], uy = ey - np[3 * n + 1], uz = ez - np[3 * n + 2];
        const double d2 = ux * ux + uy * uy + uz * uz, d = sqrt(d2);
        double v[3] = {0.0, 0.0, 0.0}, c = s.nuc_charge[n] / (d2 * d);  // -Z / d
        if (s.ecp_on)
          for (int t = 0; t < s.ecpl_nt[n]; ++t) {
            const int o = n * s.ecp_max_local + t;
            const double Vl = (1.0 / d2) * s.ecpl_coef[o] * rpow(d, s.ecpl_pow[o]) * exp_nonpos(-s.ecpl_exp[o] * d2);
            c += Vl * ((s.ecpl_pow[o] - 2.0) / d - 2.0 * s.ecpl_exp[o] * d) / d;
          }
        if (JP.j1_type) {
          double f1, f2, f3;
          const double r = fmax(d, 1.0e-12);
          j1_f123(JP.j1_type, JP.a1, s.j1_c[n], s.j1_A[n], r, f1, f2, f3);
          radial_adjoint(ux, uy, uz, f1, f2, f3, dJ, -0.5, v);
          c -= S * f1 / r;
        }
        const double u[3] = {ux, uy, uz};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          v[k] += c * u[k];
          re[k] += v[k];
          if (act) J.RA[(int64_t)(3 * n + k) * M + i] -= v[k];
        }
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) p_sh[g][c][lane] = re[c];
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      re[c] = p_sh[0][c][lane];
      for (int q = 1; q < FR_WAVES; ++q) re[c] += p_sh[q][c][lane];
    }
    if (act && wave == 0) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if (O.dE_dr) O.dE_dr[3 * i + c] = re[c];
        if (O.dlnpsi_dr) O.dlnpsi_dr[3 * i + c] = dl[c];
      }
    }
    // sums over the electrons; space-warp weights omega_ne = |r_e - R_n|^-4 / sum_m |r_e - R_m|^-4
    // (swct.py:63-150)
    double K = 0.0, dK[3] = {0.0, 0.0, 0.0};
    if (O.swct)
      for (int n = 0; n < nn; ++n) {
        const double ux = ex - np[3 * n], uy = ey - np[3 * n + 1], uz = ez - np[3 * n + 2];
        const double i2 = 1.0 / (ux * ux + uy * uy + uz * uz), k = i2 * i2, c = -4.0 * k * i2;
        K += k;
        dK[0] += c * ux;
        dK[1] += c * uy;
        dK[2] += c * uz;
      }
    const double Ki = O.swct ? 1.0 / K : 0.0;
    for (int n = wave; n < nn; n += nw) {
      double x[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
      if (act) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          x[c] = J.RA[(int64_t)(3 * n + c) * M + i];
          x[3 + c] = J.RL[(int64_t)(3 * n + c) * M + i];
        }
        if (O.swct) {
          const double u[3] = {ex - np[3 * n], ey - np[3 * n + 1], ez - np[3 * n + 2]};
          const double i2 = 1.0 / (u[0] * u[0] + u[1] * u[1] + u[2] * u[2]), k = i2 * i2, om = k * Ki;
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            x[6 + c] = om * re[c];
            x[9 + c] = om * dl[c] + 0.5 * ((-4.0 * k * i2) * u[c] * Ki - om * dK[c] * Ki);
          }
        }
      }
      wave_sum_k<12>(x);
      if (lane == 0)
#pragma unroll
        for (int c = 0; c < 12; ++c) sums[12 * n + c] += x[c];
    }
  }
  wave_sum_k<2>(en);
  if (threadIdx.x == 0 && O.e_L) O.e_L[w] = en[0] + (J.vpot[w] + s.ion_ion) + en[1];
  __syncthreads();
  for (int k = threadIdx.x; k < 3 * nn; k += blockDim.x) {
    const int n = k / 3, c = k - 3 * n;
    double F = sums[12 * n + c];
    for (int m = 0; m < nn; ++m) {  // ion-ion repulsion
      if (m == n) continue;
      const double ux = s.nuc_pos[3 * n] - s.nuc_pos[3 * m], uy = s.nuc_pos[3 * n + 1] - s.nuc_pos[3 * m + 1],
                   uz = s.nuc_pos[3 * n + 2] - s.nuc_pos[3 * m + 2];
      const double d2 = ux * ux + uy * uy + uz * uz;
      F += -s.nuc_charge[n] * s.nuc_charge[m] / (d2 * sqrt(d2)) * (c == 0 ? ux : (c == 1 ? uy : uz));
    }
    const double ln = -sums[12 * n + 3 + c];
    if (O.dE_dR) O.dE_dR[w * 3 * nn + k] = F;
    if (O.dlnpsi_dR) O.dlnpsi_dR[w * 3 * nn + k] = ln;
    if (O.force_HF) O.force_HF[w * 3 * nn + k] = F + sums[12 * n + 6 + c];
    if (O.force_PP) O.force_PP[w * 3 * nn + k] = ln + sums[12 * n + 9 + c];
  }
}

}  // namespace jqmc
