// Local energy and lattice Hamiltonian over flattened items (the E_L and LRDMC path).
//
// compute_local_energy_fast (hamiltonians.py:225-290) and _body_step_core (jqmc_gfmc.py:4807-5045) of
// all walkers as three launches whose wavefronts are full whatever the walker's size:
//
//   k_el_prep     per walker: the nearest nucleus of every electron and the list of those with
//                 projected ECP terms, J1 + J2 at the electrons, bare Coulomb and local ECP; and, on
//                 other blocks, q_e = [M | Lambda_u] G^-1[:, e] (up) or M' G^-1[e, :]^T (dn) of every
//                 electron on the matrix cores
//   k_el_kinetic  T_e (wavefunction.py:1141-1207) and c_e = a(r_e) . g_e, lanes = 64 consecutive
//                 electrons of the flattened (walker, electron) list, the AO range shared by the waves
//                 of the block
//   k_el_points   ratios at the quadrature points of the listed electrons (coulomb_potential.py:1477-1712)
//                 and, for LRDMC, at the six lattice neighbours of every electron (wavefunction.py:
//                 1779-1860); a wave takes as many electrons as 64 lanes hold, one point per lane
//
// The determinant fields h_e = C^T q_e (one row of n_ao per electron) are never stored: each wave forms
// them for its electrons twelve AOs at a time on the matrix cores (v_mfma_f64_16x16x4f64) from q_e and a
// packed copy of C, next to the J3 field rows g_e, in its own LDS tile; the vector units then run the
// AO basis shell after shell at wave-uniform indices against that tile.  What bounds it is the FP64
// vector rate: one exponential per primitive and point (16 instructions) and a few FMAs per AO.  One
// wavefront per walker, which this replaces, ran at 38 % of the issue rate behind its loads of h_e and
// g_e rows (4.5 GB per launch of 16384 benzene walkers) and left 34 of 64 lanes idle in the kinetic part.
// E_L of 16384 benzene walkers 6450 us then, 2500 us so (points 1880, kinetic 430, prep 190); 1500 walkers of the
// 56-electron chain 1901 and 687 us.
#pragma once

#include "jqmc_el.hip"
#include "jqmc_sweep_batched.hip"

namespace jqmc {

using CSys = const __attribute__((address_space(4))) Sys;
__device__ __forceinline__ CSys& csys(const Sys* p) { return *(CSys*)p; }

constexpr double LOG2E = 1.4426950408889634, LN2 = 0.6931471805599453;
constexpr int EL_ROWS = 16;           // rows of a tile of k_el_points (one MFMA tile) ...
constexpr int EL_SLOTS = 10;          // ... and the electrons a wave takes at most (six points each)
constexpr int EL_LD = EL_CH + 1;      // doubles per LDS row of a tile: odd, so that rows spread over the banks
constexpr int EL_KIN_ROWS = 64;       // electrons per block of k_el_kinetic
constexpr int EL_KIN_WAVES = 4;

// ---------------------------------------------------------------- arithmetic

// p[i] = p[i] f[i] + c for i < N as one block of three-address FMAs with c in scalar registers: the N
// chains advance together, and the compiler cannot turn a step into a copy and a two-address FMA.
template <int N>
__device__ __forceinline__ void fma_step(double* p, const double* f, double c) {
  if constexpr (N == 1)
    asm("v_fma_f64 %0, %0, %1, %2" : "+v"(p[0]) : "v"(f[0]), "s"(c));
  else if constexpr (N == 2)
    asm("v_fma_f64 %0, %0, %2, %4\n\tv_fma_f64 %1, %1, %3, %4" : "+v"(p[0]), "+v"(p[1]) : "v"(f[0]), "v"(f[1]), "s"(c));
  else if constexpr (N == 3)
    asm("v_fma_f64 %0, %0, %3, %6\n\tv_fma_f64 %1, %1, %4, %6\n\tv_fma_f64 %2, %2, %5, %6"
        : "+v"(p[0]), "+v"(p[1]), "+v"(p[2])
        : "v"(f[0]), "v"(f[1]), "v"(f[2]), "s"(c));
  else
    asm("v_fma_f64 %0, %0, %4, %8\n\tv_fma_f64 %1, %1, %5, %8\n\tv_fma_f64 %2, %2, %6, %8\n\tv_fma_f64 %3, %3, %7, %8"
        : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3])
        : "v"(f[0]), "v"(f[1]), "v"(f[2]), "v"(f[3]), "s"(c));
}

// The largest argument x given to exp2_prods: beyond it every 2^(z x) of a basis (z x below -1075) is 0.
constexpr double EXP2_XMAX = 1.0e20;

// k = (int)t with the saturation of the hardware conversion (in C++ a t outside the range is undefined).
__device__ __forceinline__ int sat_int(double t) {
  int k;
  asm("v_cvt_i32_f64 %0, %1" : "=v"(k) : "v"(t));
  return k;
}

// e[i] = 2^(z[i] x) for -1e20 <= z[i] <= 0 <= x <= EXP2_XMAX: the integer part k of t = z x, the remainder
// f = z x - k by one fma (|f| <= 1/2, no rounding of the product) and the degree-11 Chebyshev interpolant of
// 2^f (relative error 2e-17 with its rounded coefficients).  Past |t| = 2^53 the remainder is the rounding
// error of the product, at most 2^-53 1e40 here, so that the polynomial stays finite and ldexp gives 0.
template <int N>
__device__ __forceinline__ void exp2_prods(const double* z, double x, double* e) {
  double f[N], p[N];
  int k[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const double t = rint(z[i] * x);
    f[i] = fma(z[i], x, -t);
    k[i] = sat_int(t);
    p[i] = 4.4558179083360645e-10;
  }
  fma_step<N>(p, f, 7.074194297288521e-09);
  fma_step<N>(p, f, 1.0178057087733941e-07);
  fma_step<N>(p, f, 1.3215432535912375e-06);
  fma_step<N>(p, f, 1.5252733841556773e-05);
  fma_step<N>(p, f, 0.00015403530463724353);
  fma_step<N>(p, f, 0.001333355814640647);
  fma_step<N>(p, f, 0.009618129107587256);
  fma_step<N>(p, f, 0.055504108664821625);
  fma_step<N>(p, f, 0.24022650695910158);
  fma_step<N>(p, f, 0.6931471805599453);
#pragma unroll
  for (int i = 0; i < N; ++i) e[i] = ldexp(fma(p[i], f[i], 1.0), k[i]);
}
// The same for any x >= 0.
__device__ __forceinline__ double exp2_prod(double z, double x) {
  double e;
  exp2_prods<1>(&z, fmin(x, EXP2_XMAX), &e);
  return e;
}

// 1 / x for normal x away from the ends of the range: two Newton steps on the hardware reciprocal.
__device__ __forceinline__ double rcp_nr(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(y, fma(-x, y, 1.0), y);
  return fma(y, fma(-x, y, 1.0), y);
}

// sqrt(x) and its reciprocal for x >= 0 (below 1e-280: taken as that): one Goldschmidt step on the hardware
// reciprocal square root, then one residual correction of each.  For distances whose reciprocal is not used, is
// cut off first, or is checked afterwards (bare_terms).
__device__ __forceinline__ double sqrt_nr(double x, double& inv) {
  x = fmax(x, 1.0e-280);
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  g = fma(fma(-g, g, x), h, g);
  const double i = h + h;
  inv = fma(i, fma(-g, i, 1.0), i);
  return g;
}

// The same for every x, the reciprocal of 0 infinite.
__device__ __forceinline__ double sqrt_inv(double x, double& inv) {
  double r = sqrt_nr(x, inv);
  if (!(x >= 1.0e-280 && x <= 1.0e300)) {
    r = sqrt(x);
    inv = 1.0 / r;
  }
  return r;
}

struct JasPar {
  int j1_type, j2_type;
  double a1, a2, h1, h2;  // parameters and 1 / (2 parameter)
  __device__ __forceinline__ explicit JasPar(CSys& s)
      : j1_type(s.j1_type), j2_type(s.j2_type), a1(s.j1_param), a2(s.j2_param), h1(1.0 / (2.0 * s.j1_param)),
        h2(1.0 / (2.0 * s.j2_param)) {}
};

// u(r) of jastrow_factor.py:1207-1230 and of 672-711 for one nucleus (c, A).
__device__ __forceinline__ double j2_value(const JasPar& J, double r) {
  if (J.j2_type == 2) return 0.5 * r * rcp_nr(fma(J.a2, r, 1.0));
  return J.h2 * (1.0 - exp2_prod(-J.a2 * LOG2E, r));
}
__device__ __forceinline__ double j1_value(const JasPar& J, double c, double A, double r) {
  const double ac = J.a1 * c;
  if (J.j1_type == 1) return -A * (J.h1 * (1.0 - exp2_prod(-ac * LOG2E, r)));
  return -A * (0.5 * r * rcp_nr(fma(ac, r, 1.0)));
}

// ---------------------------------------------------------------- one launch, several systems

// One walker set of a launch: blocks [prep0, ...), [kin0, ...), [pts0, ...) of the three kernels are
// its own.  lr: lattice Hamiltonian (val: the candidate list of every walker), else E_L (val: the
// non-local sum of every listed electron).
template <typename T>
struct ElJob {
  const Sys* sys;
  WalkT<T> wk;
  int64_t W;
  const double* RT;   // rotations read by the points (NULL: identity)
  double* RT_new;     // rotations drawn by k_el_prep (NULL: none) ...
  double* RT_copy;    // ... and their copy for the caller
  double *Q, *H;      // q rows (W, N, n_orb); h rows (W, N, n_ao) when they are not formed on the fly
  double *te, *jc, *jold, *vpot, *val, *t_elec;
  int *elist, *necp;  // listed electrons e | nucleus << 8 (W, N) and their number (W)
  double* tau;        // GFMC_t: time left (walkers without any sit out)
  int64_t* nproj;
  int* act;
  double tau0, alat;
  uint64_t seed;
  int64_t step, val_ld;
  int lr, dlt, random_mesh, it, tau_mode, measure;
  int64_t prep0, q_blocks, kin0, pts0, lat_groups;
  int ecp_groups;     // waves per four walkers that the listed electrons need at most
};

constexpr int EL_MAX_JOBS = 8;
template <typename T>
struct ElJobs {
  int n;
  ElJob<T> job[EL_MAX_JOBS];
};

template <typename T>
__device__ __forceinline__ bool el_active(const ElJob<T>& J, int64_t w) {
  return !(J.tau_mode && J.it > 0) || J.tau[w] > 0.0;
}

// ---------------------------------------------------------------- prep

// Sixteen rows of a product on the matrix cores by one wave, operands straight from memory: fa(k) is
// A(row = lane & 15, k), fb(k) is B(k, column = lane & 15); K padded to four with zeros by the callers.
template <typename FA, typename FB>
__device__ __forceinline__ JfMfma<double>::v4 mfma_rows(int K, int ih, FA fa, FB fb) {
  JfMfma<double>::v4 acc = {0, 0, 0, 0};
#pragma unroll 4
  for (int k0 = 0; k0 < K; k0 += 4) acc = JfMfma<double>::mma(fa(k0 + ih), fb(k0 + ih), acc);
  return acc;
}

__device__ __forceinline__ double ecp_local_nr(CSys& s, int n, double d, double dinv) {
  double v = 0.0;
  const double d2 = d * d;
  for (int k = 0; k < s.ecpl_nt[n]; ++k) {
    const int o = n * s.ecp_max_local + k;
    v += (dinv * dinv) * s.ecpl_coef[o] * rpow(d, s.ecpl_pow[o]) * exp2_prod(-s.ecpl_exp[o] * LOG2E, d2);
  }
  return v;
}

// Bare Coulomb and local ECP terms of electron e (each pair of electrons half) by plain divisions: where the fast
// reciprocals left no number of ordinary size, so that the energy of coincident particles is infinite.
__device__ __forceinline__ double bare_terms(CSys& s, bool ions, const double* rr, int e) {
  const double x = rr[3 * e], y = rr[3 * e + 1], z = rr[3 * e + 2];
  double v = 0.0;
  for (int n = 0; n < s.n_nuc; ++n) {
    const double dx = s.nuc_pos[3 * n] - x, dy = s.nuc_pos[3 * n + 1] - y, dz = s.nuc_pos[3 * n + 2] - z;
    const double d = sqrt(dx * dx + dy * dy + dz * dz);
    if (ions) v += -s.nuc_charge[n] / d;
    if (s.ecp_on) v += ecp_local_nr(s, n, d, 1.0 / d);
  }
  for (int f = 0; f < s.n_el; ++f) {
    const double dx = x - rr[3 * f], dy = y - rr[3 * f + 1], dz = z - rr[3 * f + 2];
    if (f != e) v += 0.5 / sqrt(dx * dx + dy * dy + dz * dz);
  }
  return v;
}

// Blocks [0, q_blocks) of a job: wave (w, row tile) forms q of 16 electrons of one spin block of walker
// w.  The others: one wave per walker.
template <typename T>
__global__ void __launch_bounds__(256) k_el_prep(ElJobs<T> M) {
  __shared__ double rr_s[4][3 * 128];  // n_up <= 64, so at most 128 electrons
  const int64_t bid = wide_block();
  int kj = 0;
  while (kj + 1 < M.n && M.job[kj + 1].prep0 <= bid) ++kj;
  const ElJob<T>& J = M.job[kj];
  CSys& s = csys(J.sys);
  const int64_t blk = bid - J.prep0;
  const int wave = wave_id(), lane = lane_id();
  const int nu = s.n_up, nd = s.n_dn, ne = s.n_el, no = s.n_orb;
  if (blk < J.q_blocks) {
    const int nut = (nu + 15) / 16, nt = nut + (nd + 15) / 16;
    const int64_t id = blk * 4 + wave, w = id / nt;
    if (w >= J.W || !el_active(J, w)) return;
    const int rt = (int)(id - w * nt), il = lane & 15, ih = lane >> 4;
    const bool up = rt < nut;
    const int e0 = 16 * (up ? rt : rt - nut), n_sp = up ? nu : nd, off = up ? 0 : nu;
    const double* Gi = J.wk.Ginv + w * nu * nu;
    const double* Pw = J.wk.pair + w * ne * no;
    double* Qw = J.Q + (w * ne + off) * no;
    const int er = e0 + il;
    for (int c0 = 0; c0 < no; c0 += 16) {
      const int c = c0 + il;
      auto fa = [&](int k) { return (k < nu && er < n_sp) ? (up ? Gi[k * nu + er] : Gi[er * nu + k]) : 0.0; };
      auto fb = [&](int k) {
        if (k >= nu || c >= no) return 0.0;
        if (!up) return Pw[(int64_t)k * no + c];
        return k < nd ? Pw[(int64_t)(nu + k) * no + c] : s.td.lam_u[(int64_t)c * s.n_unp + (k - nd)];
      };
      const auto acc = mfma_rows(nu, ih, fa, fb);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = e0 + JfMfma<double>::row(q, ih);
        if (r < n_sp && c < no) Qw[(int64_t)r * no + c] = acc[q];
      }
    }
    return;
  }
  const int64_t w = (blk - J.q_blocks) * 4 + wave;
  if (w >= J.W) return;
  if (J.lr && !J.measure) {
    if (J.tau_mode && w == 0 && lane == 0) J.act[J.it & 1] = 0;  // counted by this round's moves
    if (J.it == 0 && lane == 0) {
      J.tau[w] = J.tau0;
      J.nproj[w] = 0;
    }
  }
  if (!el_active(J, w)) {
    if (lane == 0) J.necp[w] = 0;
    return;
  }
  double* rr = rr_s[wave];
  for (int k = lane; k < 3 * nu; k += WAVE) rr[k] = J.wk.r_up[w * 3 * nu + k];
  for (int k = lane; k < 3 * nd; k += WAVE) rr[3 * nu + k] = J.wk.r_dn[w * 3 * nd + k];
  if (J.RT_new) {
    double R[9] = {1.0, 0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0, 1.0};
    if (J.random_mesh) rotation_RT(J.seed, (uint32_t)w, (uint64_t)J.step, STREAM_LRDMC, R);
    if (lane == 0) {
      for (int k = 0; k < 9; ++k) {
        J.RT_new[9 * w + k] = R[k];
        if (J.RT_copy) J.RT_copy[9 * w + k] = R[k];
      }
    }
  }
  wave_sync();
  const JasPar JP(s);
  const bool nonlocal = s.ecp_on && s.nv > 0;
  const CPtr<double> np = cview(s.nuc_pos);
  const CPtr<double> nc = cview(s.nuc_charge);
  double pot = 0.0;
  int n_ecp = 0;
  for (int e0 = 0; e0 < ne; e0 += WAVE) {
    const int e = e0 + lane;
    bool has = false;
    int best = 0;
    if (e < ne) {
      const double x = rr[3 * e], y = rr[3 * e + 1], z = rr[3 * e + 2];
      const double pot0 = pot;
      double old = 0.0, bd = 1.0e300;
      for (int n = 0; n < s.n_nuc; ++n) {
        const double dx = np[3 * n] - x, dy = np[3 * n + 1] - y, dz = np[3 * n + 2] - z;
        const double d = sqrt(dx * dx + dy * dy + dz * dz);
        if (d < bd) {
          bd = d;
          best = n;
        }
        const double di = rcp_nr(d);
        if (!J.lr) pot += -nc[n] * di;
        if (s.ecp_on) pot += ecp_local_nr(s, n, d, di);
        if (JP.j1_type) old += j1_value(JP, s.j1_c[n], s.j1_A[n], d);
      }
      for (int f = 0; f < ne; ++f) {
        if (f == e) continue;
        const double dx = x - rr[3 * f], dy = y - rr[3 * f + 1], dz = z - rr[3 * f + 2];
        double ri;
        const double r = sqrt_nr(dx * dx + dy * dy + dz * dz, ri);
        pot += 0.5 * ri;
        if (JP.j2_type) old += j2_value(JP, r);
      }
      J.jold[w * ne + e] = old;
      if (!(fabs(pot) <= 1.0e120)) pot = pot0 + bare_terms(s, !J.lr, rr, e);
      if (nonlocal) has = s.ecp_nt[best] > 0;
    }
    const uint64_t mask = __ballot(has);
    if (has) J.elist[w * ne + n_ecp + __popcll(mask & ((1ull << lane) - 1ull))] = e | (best << 8);
    n_ecp += __popcll(mask);
  }
  pot = wave_sum(pot);
  if (lane == 0) {
    J.necp[w] = n_ecp;
    J.vpot[w] = pot;
  }
}

// h rows of systems whose orbital count exceeds the register form (more than 64 MOs): H = Q C on the
// matrix cores, wave (w, row tile); kAdd: onto the rows that H holds.
template <typename T, bool kAdd = false>
__global__ void __launch_bounds__(256) k_el_hrows(ElJob<T> J) {
  CSys& s = csys(J.sys);
  const int wave = wave_id(), lane = lane_id(), il = lane & 15, ih = lane >> 4;
  const int nu = s.n_up, nd = s.n_dn, ne = s.n_el, no = s.n_orb, na = s.n_ao;
  const int nut = (nu + 15) / 16, nt = nut + (nd + 15) / 16;
  const int64_t id = (int64_t)blockIdx.x * 4 + wave, w = id / nt;
  if (w >= J.W || !el_active(J, w)) return;
  const int rt = (int)(id - w * nt);
  const bool up = rt < nut;
  const int e0 = 16 * (up ? rt : rt - nut), n_sp = up ? nu : nd, off = up ? 0 : nu;
  const double* Qw = J.Q + (w * ne + off) * (int64_t)no;
  double* Hw = J.H + (w * ne + off) * (int64_t)na;
  const double* C = up ? s.td.mo_up : s.td.mo_dn;
  const int er = e0 + il;
  for (int c0 = 0; c0 < na; c0 += 16) {
    const int c = c0 + il;
    const auto acc = mfma_rows(
        no, ih, [&](int k) { return (k < no && er < n_sp) ? Qw[(int64_t)er * no + k] : 0.0; },
        [&](int k) { return (k < no && c < na) ? C[(int64_t)k * na + c] : 0.0; });
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = e0 + JfMfma<double>::row(q, ih);
      if (r < n_sp && c < na) Hw[(int64_t)r * na + c] = kAdd ? Hw[(int64_t)r * na + c] + acc[q] : acc[q];
    }
  }
}

// ---------------------------------------------------------------- AO pieces

// Index of the monomial x^nx y^ny z^(L-nx-ny) in the canonical order of degree L.
__host__ __device__ constexpr int mono_index(int L, int nx, int ny) {
  return (L - nx) * (L - nx + 1) / 2 + (L - nx - ny);
}
template <int L>
struct Mono {
  static constexpr int N = (L + 1) * (L + 2) / 2;
  static __host__ __device__ constexpr int nx(int i) {
    int x = L;
    while ((L - x + 1) * (L - x + 2) / 2 <= i) --x;
    return x;
  }
  static __host__ __device__ constexpr int ny(int i) { return L - nx(i) - (i - mono_index(L, nx(i), L - nx(i))); }
  static __host__ __device__ constexpr int nz(int i) { return L - nx(i) - ny(i); }
};

// sum_i h_i P_i(x, y, z) over the canonical monomials of degree L, nested.
template <int L>
__device__ __forceinline__ double poly_dot(const double* h, double x, double y, double z) {
  if constexpr (L == 0) {
    return h[0];
  } else if constexpr (L == 1) {
    return fma(z, h[2], fma(y, h[1], x * h[0]));
  } else if constexpr (L == 2) {
    const double a = fma(z, h[2], fma(y, h[1], x * h[0])), b = fma(z, h[4], y * h[3]);
    return fma(z * z, h[5], fma(y, b, x * a));
  } else {
    const double q = poly_dot<2>(h, x, y, z);  // x times the monomials that hold x
    const double b = fma(z, fma(z, h[8], y * h[7]), y * (y * h[6]));
    return fma(z * z, z * h[9], fma(y, b, x * q));
  }
}

// Value, gradient and Laplacian of sum_i h_i P_i.
template <int L>
__device__ __forceinline__ void poly_vgl(const double* h, double x, double y, double z, double& P, double* G,
                                         double& lap) {
  if constexpr (L == 0) {
    P = h[0];
    G[0] = G[1] = G[2] = 0.0;
    lap = 0.0;
  } else if constexpr (L == 1) {
    P = poly_dot<1>(h, x, y, z);
    G[0] = h[0];
    G[1] = h[1];
    G[2] = h[2];
    lap = 0.0;
  } else if constexpr (L == 2) {
    G[0] = fma(2.0 * x, h[0], fma(y, h[1], z * h[2]));
    G[1] = fma(2.0 * y, h[3], fma(x, h[1], z * h[4]));
    G[2] = fma(2.0 * z, h[5], fma(x, h[2], y * h[4]));
    P = 0.5 * fma(x, G[0], fma(y, G[1], z * G[2]));  // degree-2 homogeneous
    lap = 2.0 * (h[0] + h[3] + h[5]);
  } else {
    const double xx = x * x, xy = x * y, xz = x * z, yy = y * y, yz = y * z, zz = z * z;
    const double m[6] = {xx, xy, xz, yy, yz, zz}, d[3] = {x, y, z};
    G[0] = G[1] = G[2] = lap = 0.0;
#pragma unroll
    for (int i = 0; i < Mono<3>::N; ++i) {
      const int a = Mono<3>::nx(i), b = Mono<3>::ny(i), c = Mono<3>::nz(i);
      if (a > 0) G[0] = fma(a * h[i], m[mono_index(2, a - 1, b)], G[0]);
      if (b > 0) G[1] = fma(b * h[i], m[mono_index(2, a, b - 1)], G[1]);
      if (c > 0) G[2] = fma(c * h[i], m[mono_index(2, a, b)], G[2]);
      if (a > 1) lap = fma(a * (a - 1) * h[i], d[mono_index(1, a - 2, b)], lap);
      if (b > 1) lap = fma(b * (b - 1) * h[i], d[mono_index(1, a, b - 2)], lap);
      if (c > 1) lap = fma(c * (c - 1) * h[i], d[mono_index(1, a, b)], lap);
    }
    P = (1.0 / 3.0) * fma(x, G[0], fma(y, G[1], z * G[2]));
  }
}

// The words of a piece record that every piece needs, in scalar registers: read together (one wait), and
// those of the next piece as soon as the exponentials of the current one are done.
template <typename U>
struct PieceHead {
  double c[3];
  int info, a0;
  U zc[2 * PIECE_P];
  __device__ __forceinline__ void load(CPtr<PieceRec<U>> r) {
#pragma unroll
    for (int q = 0; q < 3; ++q) c[q] = r->c[q];
    info = r->info;
    a0 = r->a0;
#pragma unroll
    for (int q = 0; q < 2 * PIECE_P; ++q) zc[q] = r->zc[q];
  }
};

// Exponentials of the N primitives of a piece at squared distance r2, the chains together.
template <int N>
__device__ __forceinline__ void piece_exps(const PieceHead<double>& h, double r2, double* e) {
  double z[N];
#pragma unroll
  for (int q = 0; q < N; ++q) z[q] = h.zc[2 * q];
  exp2_prods<N>(z, r2, e);
}

// Radial factor of a piece at squared distance r2 (FP32: summed in the order of the primitives).
template <int N>
__device__ __forceinline__ double piece_radial(const PieceHead<double>& h, double r2) {
  double e[N];
  piece_exps<N>(h, r2, e);
  double nr = h.zc[1] * e[0];
#pragma unroll
  for (int q = 1; q < N; ++q) nr = fma(h.zc[2 * q + 1], e[q], nr);
  return nr;
}
template <int N>
__device__ __forceinline__ float piece_radial(const PieceHead<float>& h, float r2) {
  float nr = 0;
#pragma unroll
  for (int q = 0; q < N; ++q) nr += h.zc[2 * q + 1] * exp_nonpos(-h.zc[2 * q] * r2);
  return nr;
}
template <typename U>
__device__ __forceinline__ U piece_radial(const PieceHead<U>& h, U r2) {
  const int np = h.info & 15;
  if (np == 3) return piece_radial<3>(h, r2);
  if (np == 1) return piece_radial<1>(h, r2);
  if (np == 2) return piece_radial<2>(h, r2);
  return piece_radial<4>(h, r2);
}
// The same from the primitive tables.
template <typename U>
__device__ __forceinline__ U table_radial(CSys& s, CPtr<PieceMore<U>> r, U r2) {
  U nr = 0;
  const int p1 = r->p1;
  for (int p = r->p0; p < p1; ++p) nr += cview(tabs_c<U>(s).prim_coef)[p] * exp_nonpos(-cview(tabs_c<U>(s).prim_exp)[p] * r2);
  return nr;
}

// Monomial or term sum of AO a at (dx, dy, dz), tables read at the wave-uniform index a.
template <typename U>
__device__ __forceinline__ U poly_at(CSys& s, int a, U dx, U dy, U dz) {
  const int m = cview(s.ao_meta)[a];
  if (m & AO_UNIT_TERM) return ipow(dx, (m >> 16) & 15) * ipow(dy, (m >> 20) & 15) * ipow(dz, (m >> 24) & 15);
  const CPtr<int> tp = cview(s.ao_tp);
  const CPtr<int> pw = cview(s.term_pow);
  const CPtr<U> tc = cview(tabs_c<U>(s).term_coef);
  U P = 0;
  const int t1 = tp[a + 1];
  for (int t = tp[a]; t < t1; ++t) P += tc[t] * (ipow(dx, pw[3 * t]) * ipow(dy, pw[3 * t + 1]) * ipow(dz, pw[3 * t + 2]));
  return P;
}

// One piece at a point in FP32: every AO value is formed and rounded, then summed in AO order against the
// field rows h (FP64) and g.  (In FP64 the fields carry the AO scales, and the polynomial is summed
// against them before the radial factor.)
template <int L>
__device__ __forceinline__ void piece_point(CPtr<PieceMore<float>> r, float nr, const double* h, const float* g, float dx,
                                            float dy, float dz, double& det, float& dj) {
  auto pw = [](int n, float x) { return n == 0 ? 1.0f : (n == 1 ? x : (n == 2 ? x * x : x * x * x)); };
#pragma unroll
  for (int i = 0; i < Mono<L>::N; ++i) {
    const float P = pw(Mono<L>::nx(i), dx) * pw(Mono<L>::ny(i), dy) * pw(Mono<L>::nz(i), dz);
    const float v = r->sc[i] * (nr * P);
    det += (double)v * h[i];
    dj += v * g[i];
  }
}

// Orders this wave's LDS accesses for the compiler; the hardware takes one wave's LDS instructions in
// order, so loads issued before it stay in flight.
__device__ __forceinline__ void lds_order() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------- points

// KQ: k-steps of four orbitals (Sys::el_ks: 4, 8, 12 or 16, for up to 16 .. 64 orbitals), whose q stay in
// registers; 0: the h rows are read from memory.  KQ = 4 fits four waves per SIMD (16384 benzene walkers 1904 us,
// 2118 with three); more q registers would spill there, so the others take three.
template <typename T, int KQ>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(KQ == 4 ? 4 : 3))) k_el_points(ElJobs<T> M) {
  using MF = JfMfma<double>;
  __shared__ double h_sh[4][2][EL_ROWS * EL_LD + 3];
  __shared__ T g_sh[4][2][EL_ROWS * EL_LD + 3];
  __shared__ double stash[4][2][WAVE];
  int kj = 0;
  while (kj + 1 < M.n && M.job[kj + 1].pts0 <= (int64_t)blockIdx.x) ++kj;
  const ElJob<T>& J = M.job[kj];
  CSys& s = csys(J.sys);
  const int wave = wave_id(), lane = lane_id(), il = lane & 15, ih = lane >> 4;
  const int64_t id = ((int64_t)blockIdx.x - J.pts0) * 4 + wave;
  const int nu = s.n_up, ne = s.n_el, na = s.n_ao, no = s.n_orb;
  const bool lat = id < J.lat_groups;
  const int nv = lat ? 6 : s.nv;
  const int npt = nv < WAVE ? nv : WAVE, parts = (nv + WAVE - 1) / WAVE;
  int n_slots = WAVE / npt;
  if (n_slots > EL_SLOTS) n_slots = EL_SLOTS;

  // ---- the wave's electrons: slot -> (walker, electron, place in the walker's list)
  int64_t w0;
  int base, total, c0 = 0, c1 = 0, c2 = 0;
  if (lat) {
    const int64_t i0 = id * n_slots;
    w0 = i0 / ne;
    base = (int)(i0 - w0 * ne);
    const int64_t left = J.W * ne - i0;
    total = left < n_slots ? (int)left : n_slots;
  } else {
    // the first group of every four walkers, then the second, ...: the groups past the end of the lists come
    // last and do not leave some of the dies with less work than the others
    const int64_t r = id - J.lat_groups, n_quad = (J.W + 3) / 4, gi = r / n_quad;
    if (gi >= J.ecp_groups) return;
    w0 = 4 * (r - gi * n_quad);
    const CPtr<int> cnt = cview(J.necp);
    c0 = cnt[w0];
    c1 = w0 + 1 < J.W ? cnt[w0 + 1] : 0;
    c2 = w0 + 2 < J.W ? cnt[w0 + 2] : 0;
    const int c3 = w0 + 3 < J.W ? cnt[w0 + 3] : 0;
    base = (int)gi * n_slots;
    total = (c0 + c1 + c2 + c3) * parts - base;
    if (total > n_slots) total = n_slots;
  }
  if (total <= 0) return;
  auto slot = [&](int sl, int64_t& w, int& e, int& rank, int& part, int& nuc) {
    int i = base + (sl < total ? sl : 0), wl = 0;
    part = 0;
    nuc = 0;
    if (lat) {
      while (i >= ne) {
        i -= ne;
        ++wl;
      }
      rank = e = i;
    } else {
      if (parts > 1) {
        part = i % parts;
        i = i / parts;
      }
      if (i >= c0) {
        i -= c0;
        ++wl;
        if (i >= c1) {
          i -= c1;
          ++wl;
          if (i >= c2) {
            i -= c2;
            ++wl;
          }
        }
      }
      rank = i;
      const int x = J.elist[(w0 + wl) * ne + i];
      e = x & 255;
      nuc = x >> 8;
    }
    w = w0 + wl;
  };
  int64_t w;
  int e, rank, part, nuc;
  const int my = (int)(((float)lane + 0.5f) / (float)npt);  // lane / npt
  slot(my, w, e, rank, part, nuc);
  const int k = part * WAVE + lane - my * npt;
  bool valid = my < total && k < nv;
  if (lat && J.tau_mode) {
    valid = valid && el_active(J, w);
    if (!__any(valid)) return;
  }
  // staged elements: column lane % 12 of the rows lane / 12 + 5 r of the tile, r < n_st (rows without a slot
  // repeat slot 0), as offsets from the first walker's rows; and the matrix operand's row
  constexpr int ST = (EL_SLOTS + 4) / 5;
  const int n_st = (total + 4) / 5, scol = lane % EL_CH, srow = lane < 60 ? lane / EL_CH : 0;
  unsigned rowof[ST];
  int64_t arow = 0;
  bool aup = true, aok = false;
#pragma unroll
  for (int r = 0; r < ST; ++r) {
    rowof[r] = 0;
    if (r < n_st) {
      int64_t wr;
      int er, t0, t1, t2;
      slot(srow + 5 * r, wr, er, t0, t1, t2);
      rowof[r] = (unsigned)(((int)(wr - w0) * ne + er) * na);
    }
  }
  if constexpr (KQ > 0) {
    int er, t0, t1, t2;
    int64_t wr;
    slot(il, wr, er, t0, t1, t2);
    arow = (wr * ne + er) * no;
    aup = er < nu;
    aok = il < total;
  }

  // ---- the point
  const double* rp = e < nu ? J.wk.r_up + (w * nu + e) * 3 : J.wk.r_dn + (w * s.n_dn + (e - nu)) * 3;
  const double ex = rp[0], ey = rp[1], ez = rp[2];
  double R[9] = {1.0, 0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0, 1.0};
  if (J.RT) {
#pragma unroll
    for (int q = 0; q < 9; ++q) R[q] = J.RT[9 * w + q];
  }
  double px, py, pz, pwt = 0.0;
  if (lat) {
    const int kk = valid ? k : 0, axis = kk >> 1;
    const double sa = (kk & 1) ? -J.alat : J.alat;
    px = ex + sa * (axis == 0 ? R[0] : (axis == 1 ? R[3] : R[6]));
    py = ey + sa * (axis == 0 ? R[1] : (axis == 1 ? R[4] : R[7]));
    pz = ez + sa * (axis == 0 ? R[2] : (axis == 1 ? R[5] : R[8]));
  } else {
    const int kk = valid ? k : 0;
    const double m0 = s.mesh_pts[3 * kk], m1 = s.mesh_pts[3 * kk + 1], m2 = s.mesh_pts[3 * kk + 2];
    const double gx = m0 * R[0] + m1 * R[3] + m2 * R[6], gy = m0 * R[1] + m1 * R[4] + m2 * R[7],
                 gz = m0 * R[2] + m1 * R[5] + m2 * R[8];
    const double rx = s.nuc_pos[3 * nuc] - ex, ry = s.nuc_pos[3 * nuc + 1] - ey, rz = s.nuc_pos[3 * nuc + 2] - ez;
    double ri, gi;
    const double rn2 = rx * rx + ry * ry + rz * rz, rn = sqrt_inv(rn2, ri);
    sqrt_nr(gx * gx + gy * gy + gz * gz, gi);
    px = ex + (rx + rn * gx);
    py = ey + (ry + rn * gy);
    pz = ez + (rz + rn * gz);
    const double cth = -((rx * gx + ry * gy + rz * gz) * (ri * gi));
    const int nt = s.ecp_nt[nuc];
    const double wk_ = s.mesh_w[kk];
    for (int t = 0; t < nt; ++t) {
      const int o = nuc * s.ecp_max_terms + t, l = s.ecp_l[o];
      const double V = (ri * ri) * s.ecp_coef[o] * rpow(rn, s.ecp_pow[o]) * exp2_prod(-s.ecp_exp[o] * LOG2E, rn2);
      // the common projectors s and p without the table's select chain
      const double leg = s.ecp_lmax <= 2 ? (l == 0 ? 1.0 : cth) : legendre(l, cth);
      pwt += V * ((2 * l + 1) * leg * wk_);
    }
  }

  // ---- J1 + J2 at the point
  const JasPar JP(s);
  double jn = 0.0;
  if (JP.j2_type) {
    const double* ru = J.wk.r_up + w * 3 * nu;
    const double* rd = J.wk.r_dn + w * 3 * s.n_dn - 3 * nu;
#pragma unroll 2
    for (int f = 0; f < ne; ++f) {
      const double* q = (f < nu ? ru : rd) + 3 * f;
      const double dx = px - q[0], dy = py - q[1], dz = pz - q[2];
      double ri;
      const double u = j2_value(JP, sqrt_nr(dx * dx + dy * dy + dz * dz, ri));
      jn += f == e ? 0.0 : u;
    }
  }
  if (JP.j1_type) {
    for (int n = 0; n < s.n_nuc; ++n) {
      const CPtr<double> q = cview(s.nuc_pos) + 3 * n;
      const double dx = px - q[0], dy = py - q[1], dz = pz - q[2];
      double ri;
      jn += j1_value(JP, cview(s.j1_c)[n], cview(s.j1_A)[n], sqrt_nr(dx * dx + dy * dy + dz * dz, ri));
    }
  }

  // ---- the AO basis, one chunk of at most EL_CH AOs after the other: the tile of the next chunk is on
  // its way (J3 rows and packed C in registers, its h rows on the matrix cores) during the current one
  const bool j3 = s.j3_on;
  const T* gsrc = j3 ? J.wk.jfield + w0 * ne * na : nullptr;
  const double* hsrc = KQ == 0 ? J.H + w0 * ne * na : nullptr;
  // kept in LDS meanwhile (registers): the Jastrow terms besides a . g and the projector weight
  stash[wave][0][lane] = (jn - J.jold[w * ne + e]) - (j3 ? J.jc[w * ne + e] : 0.0);
  stash[wave][1][lane] = pwt;
  // where the point's element goes (LRDMC)
  const int64_t out = w * J.val_ld + (lat ? 6 * e : 6 * ne + rank * nv) + k;
  const CPtr<int> chk = cview(s.el_chunks);  // (first piece, end piece, first AO, number of AOs)
  const int n_chunk = s.n_chunk;
  constexpr int KR = KQ > 0 ? KQ : 1;
  double qa[KR], bu[KR], gsc = 1.0;
  const bool two = !s.mo_same;
  if constexpr (KQ > 0) {
#pragma unroll
    for (int q = 0; q < KQ; ++q) qa[q] = (aok && 4 * q + ih < no) ? J.Q[arow + 4 * q + ih] : 0.0;
  }
  T gr[ST];
  double hr[ST];
#pragma unroll
  for (int r = 0; r < ST; ++r) {
    gr[r] = 0;
    hr[r] = 0.0;
  }
  // the rows of chunk c on their way; columns past the chunk's end hold other AOs of the row (unused)
  auto load = [&](int c) {
    const int a0 = chk[4 * c + 2];
    const unsigned a = a0 + scol < na ? a0 + scol : na - 1;
    double sc = 1.0;
    if constexpr (std::is_same<T, double>::value) sc = s.el_scale[(unsigned)(c * EL_CH + scol)];
#pragma unroll
    for (int r = 0; r < ST; ++r)
      if (r < n_st) {
        if (j3) gr[r] = gsrc[rowof[r] + a];
        if constexpr (KQ == 0) hr[r] = hsrc[rowof[r] + a];
      }
    if constexpr (KQ > 0) {
      const double* cp = s.el_cup + (int64_t)c * KQ * WAVE;
#pragma unroll
      for (int q = 0; q < KQ; ++q)
        bu[q] = cp[(unsigned)(q * WAVE + lane)];
    }
    if constexpr (std::is_same<T, double>::value) gsc = sc;
  };
  auto rows = [&](int c) {
    MF::v4 acc = {0, 0, 0, 0};
    if constexpr (KQ > 0) {
#pragma unroll
      for (int q = 0; q < KQ; ++q) acc = MF::mma((!two || aup) ? qa[q] : 0.0, bu[q], acc);
      if (two) {
        const double* cp = s.el_cdn + (int64_t)c * KQ * WAVE;
#pragma unroll
        for (int q = 0; q < KQ; ++q) acc = MF::mma(aup ? 0.0 : qa[q], cp[(unsigned)(q * WAVE + lane)], acc);
      }
    }
    return acc;
  };
  auto store_g = [&](int b) {
    if (lane < 60) {
#pragma unroll
      for (int r = 0; r < ST; ++r)
        if (r < n_st) {
          const int o = (srow + 5 * r) * EL_LD + scol;
          if constexpr (std::is_same<T, double>::value) {
            g_sh[wave][b][o] = gr[r] * gsc;
            if constexpr (KQ == 0) h_sh[wave][b][o] = hr[r] * gsc;
          } else {
            g_sh[wave][b][o] = gr[r];
            if constexpr (KQ == 0) h_sh[wave][b][o] = hr[r];
          }
        }
    }
  };
  auto store_h = [&](int b, const MF::v4& acc) {
    if constexpr (KQ > 0) {
      if (il < EL_CH)
#pragma unroll
        for (int q = 0; q < 4; ++q) h_sh[wave][b][MF::row(q, ih) * EL_LD + il] = acc[q];
    }
  };
  PieceHead<T> hd;
  hd.load(cview(pieces<T>(s)));
  load(0);
  store_g(0);
  store_h(0, rows(0));
  if (n_chunk > 1) load(1);
  lds_order();
  double det = 0.0;
  T dj = 0;
  const int myrow = my < total ? my : 0;
  for (int c = 0; c < n_chunk; ++c) {
    MF::v4 nxt = {0, 0, 0, 0};
    if (c + 1 < n_chunk) {
      nxt = rows(c + 1);
      store_g((c + 1) & 1);
      if (c + 2 < n_chunk) load(c + 2);
    }
    lds_order();
    const double* hrow = h_sh[wave][c & 1] + myrow * EL_LD;
    const T* grow = g_sh[wave][c & 1] + myrow * EL_LD;
    const int p1 = chk[4 * c + 1], ca = chk[4 * c + 2];
    const CPtr<PieceRec<T>> rec = cview(pieces<T>(s));
    for (int p = chk[4 * c]; p < p1; ++p) {
      const int o = hd.a0 - ca, info = hd.info;
      const T dx = (T)(px - hd.c[0]), dy = (T)(py - hd.c[1]), dz = (T)(pz - hd.c[2]);
      T r2 = dx * dx + dy * dy + dz * dz;
      if (info & PIECE_ANY) {
        const T nr = table_radial<T>(s, cview(pieces_more<T>(s)) + p, r2);
        const int n = info >> 16, a0 = hd.a0;
        hd.load(rec + p + 1);
        for (int i = 0; i < n; ++i) {
          T v = nr * poly_at<T>(s, a0 + i, dx, dy, dz);
          if constexpr (!std::is_same<T, double>::value) v = cview(s.tf.ao_scale)[a0 + i] * v;
          det += (double)v * hrow[o + i];
          dj += v * grow[o + i];
        }
        continue;
      }
      if constexpr (std::is_same<T, double>::value) r2 = fmin(r2, EXP2_XMAX);
      // the field words of an s or p shell before the exponentials (an s shell reads two words too many)
      const double h[3] = {hrow[o], hrow[o + 1], hrow[o + 2]};
      const T g[3] = {grow[o], grow[o + 1], grow[o + 2]};
      const T nr = piece_radial(hd, r2);
      hd.load(rec + p + 1);  // the table ends with a blank record
      const int l = (info >> 4) & 15;
      auto dot = [&](auto Lc) {
        constexpr int l = decltype(Lc)::value, N = Mono<l>::N;
        if constexpr (std::is_same<T, double>::value) {
          // h, then g (in an f shell one after the other: twenty words would cost a wave per SIMD)
          double f[N];
#pragma unroll
          for (int i = 0; i < N; ++i) f[i] = i < 3 ? h[i] : hrow[o + i];
          det = fma(nr, poly_dot<l>(f, dx, dy, dz), det);
          if constexpr (l == 3) lds_order();
#pragma unroll
          for (int i = 0; i < N; ++i) f[i] = i < 3 ? g[i] : grow[o + i];
          dj = fma(nr, poly_dot<l>(f, dx, dy, dz), dj);
        } else {
          double hh[N];
          T gg[N];
#pragma unroll
          for (int i = 0; i < N; ++i) {
            hh[i] = i < 3 ? h[i] : hrow[o + i];
            gg[i] = i < 3 ? g[i] : grow[o + i];
          }
          piece_point<l>(cview(pieces_more<T>(s)) + p, nr, hh, gg, dx, dy, dz, det, dj);
        }
      };
      if (l == 0)
        dot(std::integral_constant<int, 0>{});
      else if (l == 1)
        dot(std::integral_constant<int, 1>{});
      else if (l == 2)
        dot(std::integral_constant<int, 2>{});
      else
        dot(std::integral_constant<int, 3>{});
    }
    lds_order();
    if (c + 1 < n_chunk) store_h((c + 1) & 1, nxt);
    lds_order();
  }
  const double jr = exp((double)dj + stash[wave][0][lane]);
  pwt = stash[wave][1][lane];
  if (J.lr) {
    if (!valid) return;
    if (lat) {
      J.val[out] = -1.0 / (2.0 * (J.alat * J.alat)) * (det * jr);
    } else {
      // t-move: V = w_P Psi(r')/Psi(r); DLA t-move: V = w_P det ratio and the Jastrow ratio multiplies
      // the fixed-node part only (jqmc_gfmc.py:4956-5021); a positive element is kept as it is
      const double V = J.dlt ? pwt * det : pwt * (det * jr);
      J.val[out] = (J.dlt && V < 0.0) ? V * jr : V;
    }
    return;
  }
  // the electron's sum over its points, in order, through LDS
  double* red = h_sh[wave][0];
  red[lane] = valid ? pwt * (det * jr) : 0.0;
  lds_order();
  if (lane < total) {
    double v = 0.0;
    const int n = npt;
    for (int q = 0; q < n; ++q) v += red[lane * npt + q];
    int64_t ws;
    int es, rs, ps, ns;
    slot(lane, ws, es, rs, ps, ns);
    J.val[ws * J.val_ld + (int64_t)rs * parts + ps] = v;
  }
}

// ---------------------------------------------------------------- kinetic

// LDS of a block: the q rows (KQ > 4) and per wave the tiles of h and g.
template <typename T>
__host__ __device__ inline int64_t el_kin_lds(int no, int kq, int nw) {
  return (kq > 4 ? (int64_t)EL_KIN_ROWS * (no | 1) * 8 : 0) + (int64_t)nw * EL_KIN_ROWS * EL_LD * (8 + (int64_t)sizeof(T));
}

// T_e = -1/2 [L_e + 2 D_e . gJ_e + lJ_e + |gJ_e|^2], D_e / L_e the gradient / Laplacian of a . h_e and
// gJ_e / lJ_e those of the Jastrow.  The waves of a block take chunks wid, wid + nw, ... of the AO range
// and every nw-th J1 / J2 partner of the same 64 electrons; wave 0 adds the partial sums in wave order.
// Per piece the polynomials of all its AOs are summed against the field rows first, so that the radial
// moments enter once per piece.
template <typename T, int KQ>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_el_kinetic(ElJobs<T> M) {
  using MF = JfMfma<double>;
  extern __shared__ double smem[];
  int kj = 0;
  while (kj + 1 < M.n && M.job[kj + 1].kin0 <= (int64_t)blockIdx.x) ++kj;
  const ElJob<T>& J = M.job[kj];
  CSys& s = csys(J.sys);
  const int wave = wave_id(), lane = lane_id(), il = lane & 15, ih = lane >> 4, nw = blockDim.x / WAVE;
  const int nu = s.n_up, nd = s.n_dn, ne = s.n_el, na = s.n_ao, no = s.n_orb;
  const int64_t i0 = ((int64_t)blockIdx.x - J.kin0) * EL_KIN_ROWS, tot = J.W * ne;
  const int n_rows = tot - i0 < EL_KIN_ROWS ? (int)(tot - i0) : EL_KIN_ROWS;
  const int64_t w0 = i0 / ne;
  const int eb = (int)(i0 - w0 * ne);
  const int n_w = (eb + n_rows - 1) / ne + 1;  // walkers of the block
  if (J.tau_mode && J.it > 0) {  // uniform across the block
    bool any = false;
    for (int q = 0; q < n_w; ++q) any = any || J.tau[w0 + q] > 0.0;
    if (!any) return;
  }
  double* q_s = smem;
  const int qld = no | 1;
  double* h_s = q_s + (KQ > 4 ? EL_KIN_ROWS * qld : 0) + (int64_t)wave * EL_KIN_ROWS * EL_LD;
  T* g_s = reinterpret_cast<T*>(q_s + (KQ > 4 ? EL_KIN_ROWS * qld : 0) + (int64_t)nw * EL_KIN_ROWS * EL_LD) +
           (int64_t)wave * EL_KIN_ROWS * EL_LD;
  if constexpr (KQ > 4) {
    for (int q = threadIdx.x; q < n_rows * no; q += blockDim.x) {
      const int r = q / no;
      q_s[r * qld + (q - r * no)] = J.Q[i0 * no + q];
    }
    __syncthreads();
  }
  const bool act = lane < n_rows;
  const int le = act ? eb + lane : eb, wl = le / ne, e = le - wl * ne;
  const double* ru = J.wk.r_up + (w0 + wl) * 3 * nu;
  const double* rd = J.wk.r_dn + (w0 + wl) * 3 * nd - 3 * nu;
  const double* rp = (e < nu ? ru : rd) + 3 * e;
  const double ex = rp[0], ey = rp[1], ez = rp[2];

  constexpr int KR = KQ == 4 ? 4 : 1;
  const int n_chunk = s.n_chunk;
  const bool two = !s.mo_same;
  const T* gsrc = s.j3_on ? J.wk.jfield + i0 * na : nullptr;
  const double* hsrc = KQ == 0 ? J.H + i0 * na : nullptr;
  const CPtr<int> chk = cview(s.el_chunks);
  double qa[4][KR], bu[KR];
  bool aup[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int r = 16 * t + il;
    aup[t] = (eb + r) % ne < nu;
    if constexpr (KQ == 4) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        qa[t][q] = (r < n_rows && 4 * q + ih < no) ? J.Q[(i0 + r) * no + 4 * q + ih] : 0.0;
    }
  }
  T gr[12];
  double hr[KQ == 0 ? 12 : 1];
  const int c3 = 3 * (lane & 3), r4 = lane >> 2;  // staged columns c3 .. c3 + 2 of rows r4 + 16 r
  auto load = [&](int c) {
    const int a0 = chk[4 * c + 2];
    // rows past the last electron repeat it, columns past the chunk's end hold other AOs (all unused)
    unsigned ac[3];
#pragma unroll
    for (int x = 0; x < 3; ++x) ac[x] = a0 + c3 + x < na ? a0 + c3 + x : na - 1;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const unsigned o = (unsigned)(r4 + 16 * r < n_rows ? r4 + 16 * r : n_rows - 1) * na;
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        gr[3 * r + x] = gsrc ? gsrc[o + ac[x]] : (T)0;
        if constexpr (KQ == 0) hr[3 * r + x] = hsrc[o + ac[x]];
      }
    }
    if constexpr (KQ == 4) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        bu[q] = s.el_kup[(int64_t)c * KQ * WAVE + (unsigned)(q * WAVE + lane)];
    }
  };
  auto store = [&](int c) {
    double sc[3];
#pragma unroll
    for (int x = 0; x < 3; ++x) sc[x] = s.el_scale[c * EL_CH + c3 + x];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        const int o = (r4 + 16 * r) * EL_LD + c3 + x;
        g_s[o] = gr[3 * r + x];
        if constexpr (KQ == 0) h_s[o] = hr[3 * r + x] * sc[x];
      }
    if constexpr (KQ > 0) {
      MF::v4 acc[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t] = MF::v4{0, 0, 0, 0};
      if constexpr (KQ == 4) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double b2 = two ? s.el_kdn[(int64_t)c * KQ * WAVE + (unsigned)(q * WAVE + lane)] : 0.0;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            acc[t] = MF::mma((!two || aup[t]) ? qa[t][q] : 0.0, bu[q], acc[t]);
            if (two) acc[t] = MF::mma(aup[t] ? 0.0 : qa[t][q], b2, acc[t]);
          }
        }
      } else {
#pragma unroll 4
        for (int q = 0; q < KQ; ++q) {
          const double b = s.el_kup[(int64_t)c * KQ * WAVE + (unsigned)(q * WAVE + lane)];
          const double b2 = two ? s.el_kdn[(int64_t)c * KQ * WAVE + (unsigned)(q * WAVE + lane)] : 0.0;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int r = 16 * t + il;
            const double a = (r < n_rows && 4 * q + ih < no) ? q_s[r * qld + 4 * q + ih] : 0.0;
            acc[t] = MF::mma((!two || aup[t]) ? a : 0.0, b, acc[t]);
            if (two) acc[t] = MF::mma(aup[t] ? 0.0 : a, b2, acc[t]);
          }
        }
      }
      if (il < EL_CH)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q) h_s[(16 * t + MF::row(q, ih)) * EL_LD + il] = acc[t][q];
    }
  };

  double D[3] = {0, 0, 0}, Lh = 0.0, gJ[3] = {0, 0, 0}, lJ = 0.0, jc = 0.0;
  PieceHead<double> hd;
  hd.load(cview(s.pc64) + (wave < n_chunk ? chk[4 * wave] : 0));
  if (wave < n_chunk) load(wave);
  const double* hrow = h_s + lane * EL_LD;
  const T* grow = g_s + lane * EL_LD;
  for (int c = wave; c < n_chunk; c += nw) {
    store(c);
    lds_order();
    if (c + nw < n_chunk) load(c + nw);
    const int p1 = chk[4 * c + 1], ca = chk[4 * c + 2];
    const CPtr<PieceRec<double>> rec = cview(s.pc64);
    const int p_next = c + nw < n_chunk ? chk[4 * (c + nw)] : 0;
    for (int p = chk[4 * c]; p < p1; ++p) {
      const int o = hd.a0 - ca, info = hd.info;
      const double dx = ex - hd.c[0], dy = ey - hd.c[1], dz = ez - hd.c[2];
      const double r2u = dx * dx + dy * dy + dz * dz;
      if (info & PIECE_ANY) {
        const int a0 = hd.a0, n = info >> 16;
        double nr = 0.0, znr = 0.0, z2nr = 0.0;
        const CPtr<PieceMore<double>> more = cview(s.pm64) + p;
        const int q1 = more->p1;
        for (int q = more->p0; q < q1; ++q) {
          const double Z = cview(s.td.prim_exp)[q], v = cview(s.td.prim_coef)[q] * exp_nonpos(-Z * r2u);
          nr += v;
          znr += Z * v;
          z2nr += Z * Z * v;
        }
        hd.load(rec + (p + 1 < p1 ? p + 1 : p_next));
        const double m2 = -2.0 * znr, l0 = 4.0 * r2u * z2nr - 6.0 * znr;
        for (int i = 0; i < n; ++i) {
          const int a = a0 + i;
          const CPtr<int> tp = cview(s.ao_tp);
          const CPtr<int> pw = cview(s.term_pow);
          const CPtr<double> tc = cview(s.td.term_coef);
          double P = 0.0, G[3] = {0, 0, 0}, lap = 0.0;
          const int t1 = tp[a + 1];
          for (int t = tp[a]; t < t1; ++t) {
            const double c_ = tc[t];
            const int nx = pw[3 * t], ny = pw[3 * t + 1], nz = pw[3 * t + 2];
            const double fx = ipow(dx, nx), fy = ipow(dy, ny), fz = ipow(dz, nz);
            const double qx = nx > 0 ? nx * ipow(dx, nx - 1) : 0.0, qy = ny > 0 ? ny * ipow(dy, ny - 1) : 0.0,
                         qz = nz > 0 ? nz * ipow(dz, nz - 1) : 0.0;
            const double qqx = nx > 1 ? nx * (nx - 1.0) * ipow(dx, nx - 2) : 0.0,
                         qqy = ny > 1 ? ny * (ny - 1.0) * ipow(dy, ny - 2) : 0.0,
                         qqz = nz > 1 ? nz * (nz - 1.0) * ipow(dz, nz - 2) : 0.0;
            P += c_ * (fx * fy * fz);
            G[0] += c_ * (qx * fy * fz);
            G[1] += c_ * (fx * qy * fz);
            G[2] += c_ * (fx * fy * qz);
            lap += c_ * (qqx * fy * fz + fx * qqy * fz + fx * fy * qqz);
          }
          const double rdg = dx * G[0] + dy * G[1] + dz * G[2];
          const double v0 = fma(m2 * P, dx, nr * G[0]), v1 = fma(m2 * P, dy, nr * G[1]), v2 = fma(m2 * P, dz, nr * G[2]),
                       vl = nr * lap + 2.0 * m2 * rdg + l0 * P;
          const double h = hrow[o + i];
          D[0] = fma(h, v0, D[0]);
          D[1] = fma(h, v1, D[1]);
          D[2] = fma(h, v2, D[2]);
          Lh = fma(h, vl, Lh);
          if (gsrc) {
            const double g = (double)grow[o + i] * cview(s.td.ao_scale)[a];
            gJ[0] = fma(g, v0, gJ[0]);
            gJ[1] = fma(g, v1, gJ[1]);
            gJ[2] = fma(g, v2, gJ[2]);
            lJ = fma(g, vl, lJ);
            jc = fma(g, nr * P, jc);
          }
        }
        continue;
      }
      const double r2 = fmin(r2u, EXP2_XMAX);
      // radial moments sum c e, sum Z c e, sum Z^2 c e (the record holds -Z log2 e)
      double nr = 0.0, znr = 0.0, z2nr = 0.0;
      auto moments = [&](auto Nc) {
        constexpr int NP = decltype(Nc)::value;
        double ee[NP];
        piece_exps<NP>(hd, r2, ee);
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          const double z = hd.zc[2 * q], v = hd.zc[2 * q + 1] * ee[q], zv = z * v;
          nr += v;
          znr += zv;
          z2nr = fma(z, zv, z2nr);
        }
      };
      const int np = info & 15, l = (info >> 4) & 15;
      if (np == 3)
        moments(std::integral_constant<int, 3>{});
      else if (np == 1)
        moments(std::integral_constant<int, 1>{});
      else if (np == 2)
        moments(std::integral_constant<int, 2>{});
      else
        moments(std::integral_constant<int, 4>{});
      hd.load(rec + (p + 1 < p1 ? p + 1 : p_next));
      const double m2 = (2.0 * LN2) * znr;
      auto piece = [&](auto Lc) {
        constexpr int l = decltype(Lc)::value, N = Mono<l>::N;
        // Laplacian factor of a homogeneous polynomial of degree l: 4 r^2 Z2 - (6 + 4 l) Z1
        const double ll = fma(4.0 * LN2 * LN2 * r2, z2nr, ((6.0 + 4.0 * l) * LN2) * znr);
        auto add = [&](const double* f, double* g, double& L, double& P) {
          double G[3], lap;
          poly_vgl<l>(f, dx, dy, dz, P, G, lap);
          const double mp = m2 * P;
          if constexpr (l == 0) {
            g[0] = fma(mp, dx, g[0]);
            g[1] = fma(mp, dy, g[1]);
            g[2] = fma(mp, dz, g[2]);
          } else {
            g[0] += fma(mp, dx, nr * G[0]);
            g[1] += fma(mp, dy, nr * G[1]);
            g[2] += fma(mp, dz, nr * G[2]);
          }
          L = fma(ll, P, L);
          if constexpr (l >= 2) L = fma(nr, lap, L);
        };
        double P, f[N];
#pragma unroll
        for (int i = 0; i < N; ++i) f[i] = hrow[o + i];
        add(f, D, Lh, P);
        if (gsrc) {
          const CPtr<PieceMore<double>> more = cview(s.pm64) + p;
#pragma unroll
          for (int i = 0; i < N; ++i) f[i] = (double)grow[o + i] * more->sc[i];
          add(f, gJ, lJ, P);
          jc = fma(nr, P, jc);
        }
      };
      if (l == 0)
        piece(std::integral_constant<int, 0>{});
      else if (l == 1)
        piece(std::integral_constant<int, 1>{});
      else if (l == 2)
        piece(std::integral_constant<int, 2>{});
      else
        piece(std::integral_constant<int, 3>{});
    }
    lds_order();
  }
  const JasPar JP(s);
  if (JP.j1_type) {
    for (int n = wave; n < s.n_nuc; n += nw) {
      const CPtr<double> q = cview(s.nuc_pos) + 3 * n;
      const double dx = ex - q[0], dy = ey - q[1], dz = ez - q[2];
      double ri;
      const double r = sqrt_nr(fmax(dx * dx + dy * dy + dz * dz, 1.0e-24), ri);
      const double c = cview(s.j1_c)[n], A = cview(s.j1_A)[n], ac = JP.a1 * c;
      double f1, f2;
      if (JP.j1_type == 1) {
        const double x = exp2_prod(-ac * LOG2E, r);
        f1 = -A * (c / 2.0) * x;
        f2 = A * (ac * c / 2.0) * x;
      } else {
        const double i = rcp_nr(fma(ac, r, 1.0));
        f1 = -0.5 * A * i * i;
        f2 = A * ac * i * i * i;
      }
      const double fr = f1 * ri;
      gJ[0] += fr * dx;
      gJ[1] += fr * dy;
      gJ[2] += fr * dz;
      lJ += f2 + 2.0 * fr;
    }
  }
  if (JP.j2_type) {
    for (int f = wave; f < ne; f += nw) {
      const double* q = (f < nu ? ru : rd) + 3 * f;
      const double dx = ex - q[0], dy = ey - q[1], dz = ez - q[2];
      double ri;
      const double r = sqrt_nr(fmax(dx * dx + dy * dy + dz * dz, 1.0e-24), ri);
      double f1, f2;
      if (JP.j2_type == 2) {
        const double i = rcp_nr(fma(JP.a2, r, 1.0));
        f1 = 0.5 * i * i;
        f2 = -JP.a2 * i * i * i;
      } else {
        const double x = exp2_prod(-JP.a2 * LOG2E, r);
        f1 = 0.5 * x;
        f2 = -(JP.a2 / 2.0) * x;
      }
      const bool on = f != e;
      const double fr = on ? f1 * ri : 0.0;
      gJ[0] += fr * dx;
      gJ[1] += fr * dy;
      gJ[2] += fr * dz;
      lJ += on ? f2 + 2.0 * fr : 0.0;
    }
  }
  // partial sums of waves 1 .. nw - 1 through LDS (the tiles are free now)
  double v[9] = {D[0], D[1], D[2], Lh, gJ[0], gJ[1], gJ[2], lJ, jc};
  if (nw > 1) {
    double* red = h_s;
#pragma unroll
    for (int q = 0; q < 9; ++q) red[q * WAVE + lane] = v[q];
    __syncthreads();
    if (wave == 0)
      for (int x = 1; x < nw; ++x)
#pragma unroll
        for (int q = 0; q < 9; ++q) v[q] += red[(int64_t)x * EL_KIN_ROWS * EL_LD + q * WAVE + lane];
  }
  if (wave == 0 && act) {
    const double T_ = -0.5 * (v[3] + 2.0 * (v[0] * v[4] + v[1] * v[5] + v[2] * v[6]) + v[7] +
                              (v[4] * v[4] + v[5] * v[5] + v[6] * v[6]));
    J.te[i0 + lane] = T_;
    J.jc[i0 + lane] = v[8];
    if (J.t_elec) J.t_elec[i0 + lane] = T_;
  }
}

// ---------------------------------------------------------------- the walkers' energies

// One wave per walker: e_L from the parts, and the far-off walkers of the mixed form's FP64 guard.
template <typename T>
__global__ void __launch_bounds__(256) k_el_final(ElJob<T> J, double* e_L, double* kin_out, double* v_out, int parts,
                                                  ElGuard guard) {
  CSys& s = csys(J.sys);
  const int lane = lane_id(), ne = s.n_el;
  const int64_t w = (int64_t)blockIdx.x * 4 + wave_id();
  if (w >= J.W) return;
  double v[2] = {0.0, 0.0};
  for (int e = lane; e < ne; e += WAVE) v[0] += J.te[w * ne + e];
  const int n = J.necp[w] * parts;
  for (int k = lane; k < n; k += WAVE) v[1] += J.val[w * J.val_ld + k];
  wave_sum_k<2>(v);
  if (lane == 0) {
    const double pot = (J.vpot[w] + s.ion_ion) + v[1], e = v[0] + pot;
    e_L[w] = e;
    if (kin_out) kin_out[w] = v[0];
    if (v_out) v_out[w] = pot;
    if (guard.list && !(fabs(e - guard.e_ref) <= guard.width)) guard.list[atomicAdd(guard.n, 1)] = (int)w;
  }
}

}  // namespace jqmc
