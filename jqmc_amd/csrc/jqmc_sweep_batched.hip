// Move-synchronous Metropolis sweep: the n_moves proposals of a sweep are taken one move at a
// time across all walkers, so that the per-walker dependency chain of a move runs in a launch
// with one wavefront per walker (throughput, not latency, bound), and the J3 field products of
// every walker that accepted (t1 = J3 dA, t2 = J3^T dA) become one tiled GEMM per move with the
// field updates fused into its epilogue.  Per sweep:
//
//   k_sweep_begin     R_AS of the current (G, G^-1) per walker; spin-block field offsets zeroed
//   n_moves times:
//     k_sweep_propose one wavefront per walker: draws, proposal, AO values, Jastrow / determinant
//                     ratios, AS factor, acceptance; on accept the walker state (position, AO /
//                     orbital / pair rows, G, G^-1) is updated in place and dA is left in the
//                     workspace with the moved electron's index
//     k_sweep_jfield_mfma  [T1 | T2] = [J3 | J3^T] x dA of the walkers that accepted on the matrix
//                     cores, a wave per 16 of them and 16 or 32 AOs, then the J3 field increments of
//                     jastrow_factor.py:4121-4135 on those
//   k_sweep_flush     spin-block offsets added to every field row; R_AS stored
//
// The draws, proposal and acceptance are those of k_vmc_sweep (jqmc_mcmc.py:4316-4531) on the
// same Philox counters, so both kernels take the same decisions.
#pragma once

#include "jqmc_kernels.hip"
#include "jqmc_sr.hip"

namespace jqmc {

// Per-walker workspace of the move-synchronous sweep.
template <typename T>
struct SweepWs {
  T* dA;       // (W, n_ao) AO change of the last proposal
  T* Oup;      // (W, n_ao) field offset of every up electron
  T* Odn;      // (W, n_ao) field offset of every dn electron
  double* Ro;  // (W) AS factor of the current state
  int* mv;     // (W) electron moved by the last move, -1 when rejected
  __host__ __device__ static int64_t bytes(const Sys& s, int64_t W) {
    const int64_t na = s.n_ao;
    int64_t b = 3 * W * na * (int64_t)sizeof(T);
    b = (b + 7) & ~(int64_t)7;
    return b + W * (int64_t)sizeof(double) + W * (int64_t)sizeof(int);
  }
  SweepWs() = default;
  __host__ __device__ SweepWs(void* base, const Sys& s, int64_t W) {
    const int64_t na = s.n_ao;
    char* p = static_cast<char*>(base);
    dA = reinterpret_cast<T*>(p);
    Oup = dA + W * na;
    Odn = Oup + W * na;
    int64_t off = (3 * W * na * (int64_t)sizeof(T) + 7) & ~(int64_t)7;
    Ro = reinterpret_cast<double*>(p + off);
    mv = reinterpret_cast<int*>(p + off + W * (int64_t)sizeof(double));
  }
};

// dst[i] = src[i] (+ src2[i]) for i < n by one wavefront: each lane issues its U loads before any
// of its LDS stores, so the loads of a row are in flight together (LDS is reached through generic
// pointers here, which the compiler may not reorder around).
template <typename T, int U = 4>
__device__ __forceinline__ void stage_row(T* dst, const T* __restrict__ src, const T* __restrict__ src2, int n,
                                          int lane) {
  for (int base = 0; base < n; base += WAVE * U) {
    T v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + lane + WAVE * u;
      v[u] = i < n ? (src2 ? src[i] + src2[i] : src[i]) : (T)0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + lane + WAVE * u;
      if (i < n) dst[i] = v[u];
    }
  }
}

// Positions (up then dn) and G^-1 into LDS by one wavefront, with every load of a U x 64 chunk of
// both issued before its stores: one memory round trip per chunk, one chunk for systems up to
// U x 64 elements per array.
template <int U = 4>
__device__ __forceinline__ void stage_walker(double* rr, const double* __restrict__ rup, int n_rup,
                                             const double* __restrict__ rdn, int n_rdn, double* gi,
                                             const double* __restrict__ Gi, int n_g, int lane) {
  const int n_r = n_rup + n_rdn;
  const int n_max = n_r > n_g ? n_r : n_g;
  for (int base = 0; base < n_max; base += WAVE * U) {
    double vr[U], vi[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + lane + WAVE * u;
      vr[u] = i < n_rup ? rup[i] : (i < n_r ? rdn[i - n_rup] : 0.0);
      vi[u] = i < n_g ? Gi[i] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + lane + WAVE * u;
      if (i < n_r) rr[i] = vr[u];
      if (i < n_g) gi[i] = vi[u];
    }
  }
}

// Elements of the mover's AO row and J3 field held in registers per lane (a = lane + 64 u); rows
// longer than 64 x PROP_RU are read from memory for the remaining entries.
constexpr int PROP_RU = 4;

// LDS of one wavefront in k_sweep_begin / k_sweep_propose (member names as SweepLds for the
// AS-factor helper): positions and G^-1, staged once per move, and the new AO and orbital rows.  G
// (Gm) and the pair rows of the other spin (pr) are read where they lie in the walker state (the
// kernels set the two pointers), which leaves room in LDS for more walkers per CU.  The moving
// electron's AO row and J3 field stay in registers.
template <typename T>
struct PropLds {
  double *rr, *Gi, *Gm, *vv, *xx, *yy, *phin, *dphi, *pr;
  T* anew;
  uintptr_t end;
  __host__ __device__ PropLds(char* base, const Sys& s) {
    const int ne = s.n_el, nu = s.n_up, na = s.n_ao, no = s.n_orb;
    Carve c{base};
    rr = c.take<double>(3 * ne);
    Gi = c.take<double>(nu * nu);
    Gm = nullptr;
    vv = c.take<double>(nu);
    xx = c.take<double>(nu);
    yy = c.take<double>(nu);
    anew = c.take<T>(na);
    phin = c.take<double>(no);
    dphi = c.take<double>(no);
    pr = nullptr;
    end = reinterpret_cast<uintptr_t>(c.p);
  }
};

template <typename T>
inline int64_t prop_lds_bytes(const Sys& s) {
  return (int64_t)PropLds<T>(0, s).end;
}

template <typename T>
__global__ void __launch_bounds__(256) k_sweep_begin(Sys s, int64_t W, WalkT<T> wk,
                                                     SweepWs<T> ws, int wpb, int64_t lds_per_wave) {
  extern __shared__ double smem[];
  const int wave = wave_id(), lane = lane_id();
  const int64_t w = (int64_t)blockIdx.x * wpb + wave;
  if (w >= W) return;
  PropLds<T> L(reinterpret_cast<char*>(smem) + wave * lds_per_wave, s);
  const int nu = s.n_up, na = s.n_ao;
  L.Gm = wk.G + w * nu * nu;
  for (int k = lane; k < nu * nu; k += WAVE) L.Gi[k] = wk.Ginv[w * nu * nu + k];
  for (int a = lane; a < na; a += WAVE) ws.Oup[w * na + a] = ws.Odn[w * na + a] = 0;
  wave_sync();
  const double R = sweep_as_factor(L, nu, lane, 0, 0, 1.0);
  if (lane == 0) {
    ws.Ro[w] = R;
    ws.mv[w] = -1;
  }
}

// Move m of the sweep for every walker (the body of k_vmc_sweep's move loop).
// A chain of dependent steps per walker, bound by latency while every wave has its place on the card at once and
// by the waves in flight beyond that, so there are two forms.  Up to PROP_MANY walkers (kMany false; 82 registers
// in FP32, 94 in FP64: five waves per SIMD) FP64 shells come from their records and eight loads are in flight in
// the orbital sums and, in FP64, in those of the new pair row.  More walkers take four loads and the shell loop (66
// and 69 registers, seven waves per SIMD), with the same bits.  Both find the nearest nucleus by a nucleus per lane.
// The few against one form of the shell loop with four loads and a serial nearest nucleus: 33 -> 26 us for 1024
// benzene walkers, 40.5 -> 36.8 for 2048 of 4 x H2O (FP32), 18.4 -> 17.1 for 256 of H2O.  A move of the whole sweep
// with eight loads and records for all -> with the many: benzene FP64 6144 walkers 146 -> 136 us, mixed 120 -> 103;
// 16384 357 -> 356 and 281 -> 268; 4 x H2O 16384 FP64 486 -> 466, mixed 351 -> 341; N2 16384 86.8 -> 82.1 and
// 85.0 -> 76.6; one H 6144 36.2 -> 33.7 and 37.5 -> 32.3.  Around 7168 walkers, where the many just fit in one go,
// FP64 takes up to 4 % longer (benzene 172 -> 176 us).  For 2048 walkers of 4 x H2O the many cost 2 of 66 us.
template <typename T, bool kMany>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
    k_sweep_propose(Sys s, int64_t W, WalkT<T> wk, SweepWs<T> ws, int m, double Dt, double eps_AS, uint64_t seed,
                    int64_t move_base, const int64_t* __restrict__ move_ctr, int wpb, int64_t lds_per_wave) {
  constexpr bool kF64 = std::is_same<T, double>::value;
  constexpr int kOrbLoads = kMany ? 4 : 8, kPairLoads = kF64 && !kMany ? 8 : 4;
  extern __shared__ double smem[];
  const RealTabs<T>& R = tabs<T>(s);
  const int wave = wave_id(), lane = lane_id();
  const int64_t w = (int64_t)blockIdx.x * wpb + wave;
  if (w >= W) return;
  PropLds<T> L(reinterpret_cast<char*>(smem) + wave * lds_per_wave, s);
  const int nu = s.n_up, nd = s.n_dn, ne = s.n_el, na = s.n_ao, no = s.n_orb;
  T* Aw = wk.ao + w * ne * na;
  double* Pw = wk.orb + w * ne * no;
  double* Qw = wk.pair + w * ne * no;
  const T* gw = s.j3_on ? wk.jfield + w * ne * na : nullptr;
  T* dAw = ws.dA + w * na;
  const uint64_t mvc = (uint64_t)(move_base + (move_ctr ? *move_ctr : 0) + m);

  // ---- draws in the reference order (jqmc_mcmc.py:4322-4500), before any walker load
  const U4 d0 = draw_words(seed, (uint32_t)w, mvc, STREAM_VMC, 0);
  const U4 d1 = draw_words(seed, (uint32_t)w, mvc, STREAM_VMC, 1);
  const U4 d2 = draw_words(seed, (uint32_t)w, mvc, STREAM_VMC, 2);
  const int rand_num = randint(d0.x, ne);
  const int up_index = randint(d0.y, nu > 0 ? nu : 1);
  const int dn_index = randint(d0.z, nd > 0 ? nd : 1);
  const int axis = randint(d0.w, 3);
  const double u1 = uniform01_open0(d1.x, d1.y), u2 = uniform01(d1.z, d1.w);
  const double gauss = sqrt(-2.0 * log(u1)) * cos(2.0 * M_PI * u2);
  const double bdraw = uniform01(d2.x, d2.y);
  const bool is_up = rand_num < nu;
  const int idx = is_up ? up_index : dn_index;
  const int e = is_up ? idx : nu + idx;

  // ---- load the walker data this move reads: the mover's AO row and J3 field (with its block
  // offset) into registers, positions and G^-1 into LDS, all loads in flight together; G and the
  // pair rows of the other spin (dn rows for an up move, up rows for a dn move) are read in place
  const T* Ae = Aw + (int64_t)e * na;
  const T* ge = gw ? gw + (int64_t)e * na : nullptr;
  const T* Oe = (is_up ? ws.Oup : ws.Odn) + w * na;
  T ae_r[PROP_RU], ge_r[PROP_RU];
#pragma unroll
  for (int u = 0; u < PROP_RU; ++u) {
    const int a = lane + WAVE * u;
    ae_r[u] = a < na ? Ae[a] : (T)0;
    ge_r[u] = (gw && a < na) ? ge[a] + Oe[a] : (T)0;
  }
  L.Gm = wk.G + w * nu * nu;
  L.pr = Qw + (is_up ? (int64_t)nu * no : 0);
  stage_walker(L.rr, wk.r_up + w * 3 * nu, 3 * nu, wk.r_dn + w * 3 * nd, 3 * nd, L.Gi, wk.Ginv + w * nu * nu,
               nu * nu, lane);
  const double R_o = ws.Ro[w];
  wave_sync();

  // ---- proposal with nearest-nucleus step size (jqmc_mcmc.py:4339-4401)
  const double ox = L.rr[3 * e], oy = L.rr[3 * e + 1], oz = L.rr[3 * e + 2];
  const int na0 = nearest_nucleus_wave<!kF64 || kMany>(s, ox, oy, oz, lane);
  const double Z0 = s.nuc_charge[na0];
  double dxn = ox - s.nuc_pos[3 * na0], dyn = oy - s.nuc_pos[3 * na0 + 1], dzn = oz - s.nuc_pos[3 * na0 + 2];
  const double f_l = step_factor(Z0, sqrt(dxn * dxn + dyn * dyn + dzn * dzn));
  const double g = gauss * (f_l * Dt);
  double nx = ox, ny = oy, nz = oz;
  if (axis == 0) nx += g;
  else if (axis == 1) ny += g;
  else nz += g;
  const int na1 = nearest_nucleus_wave<!kF64 || kMany>(s, nx, ny, nz, lane);
  const double Z1 = s.nuc_charge[na1];
  dxn = nx - s.nuc_pos[3 * na1];
  dyn = ny - s.nuc_pos[3 * na1 + 1];
  dzn = nz - s.nuc_pos[3 * na1 + 2];
  const double f_p = step_factor(Z1, sqrt(dxn * dxn + dyn * dyn + dzn * dzn));
  const double ddx = nx - ox, ddy = ny - oy, ddz = nz - oz;
  const double dist2 = ddx * ddx + ddy * ddy + ddz * ddz;
  const double T_ratio =
      (f_l / f_p) * exp(-dist2 * (1.0 / (2.0 * f_p * f_p * Dt * Dt) - 1.0 / (2.0 * f_l * f_l * Dt * Dt)));

  // ---- AO values at the new position, Jastrow log-ratio
  for (int sh = lane; sh < s.n_shell; sh += WAVE) {
    if constexpr (kF64 && !kMany)
      shell_record_values(s, sh, nx, ny, nz, L.anew);
    else
      shell_values<T>(s, sh, nx, ny, nz, L.anew);
  }
  wave_sync();
  double jpart = 0.0;
#pragma unroll
  for (int u = 0; u < PROP_RU; ++u) {
    const int a = lane + WAVE * u;
    if (a < na) {
      const T da = L.anew[a] - ae_r[u];
      dAw[a] = da;
      if (gw) jpart += (double)(da * ge_r[u]);
    }
  }
  for (int a = lane + WAVE * PROP_RU; a < na; a += WAVE) {
    const T da = L.anew[a] - Ae[a];
    dAw[a] = da;
    if (gw) jpart += (double)(da * (ge[a] + Oe[a]));
  }
  if (s.j1_type) {
    for (int n = lane; n < s.n_nuc; n += WAVE) {
      const double* Rn = s.nuc_pos + 3 * n;
      const double d1x = nx - Rn[0], d1y = ny - Rn[1], d1z = nz - Rn[2];
      const double d0x = ox - Rn[0], d0y = oy - Rn[1], d0z = oz - Rn[2];
      jpart += j1_term(s.j1_type, s.j1_param, s.j1_c[n], s.j1_A[n], sqrt(d1x * d1x + d1y * d1y + d1z * d1z)) -
               j1_term(s.j1_type, s.j1_param, s.j1_c[n], s.j1_A[n], sqrt(d0x * d0x + d0y * d0y + d0z * d0z));
    }
  }
  if (s.j2_type) {
    for (int f = lane; f < ne; f += WAVE) {
      if (f == e) continue;
      const double* q = L.rr + 3 * f;
      const double d1x = nx - q[0], d1y = ny - q[1], d1z = nz - q[2];
      const double d0x = ox - q[0], d0y = oy - q[1], d0z = oz - q[2];
      jpart += j2_u(s.j2_type, s.j2_param, sqrt(d1x * d1x + d1y * d1y + d1z * d1z)) -
               j2_u(s.j2_type, s.j2_param, sqrt(d0x * d0x + d0y * d0y + d0z * d0z));
    }
  }
  const double J_ratio = exp(wave_sum(jpart));
  wave_sync();

  // ---- orbitals at the new position (FP64 sums of the AO values) and their change
  const double* Pe = Pw + (int64_t)e * no;
  if (s.orb_is_mo) {
    wave_matvec_T<double, T, double, kOrbLoads>(is_up ? s.td.mo_upT : s.td.mo_dnT, L.anew, na, no, lane, L.phin);
    wave_sync();
  } else {
    for (int k = lane; k < no; k += WAVE) L.phin[k] = (double)L.anew[k];
  }
  for (int k = lane; k < no; k += WAVE) L.dphi[k] = L.phin[k] - Pe[k];
  wave_sync();

  // ---- changed geminal row (up) or column (dn) and the determinant ratio
  double part = 0.0;
  if (is_up) {
    for (int j = lane; j < nu; j += WAVE) {
      double v = 0.0;
      if (j < nd) {
        const double* pr = L.pr + (int64_t)j * no;
#pragma unroll 4
        for (int k = 0; k < no; ++k) v += L.dphi[k] * pr[k];
      } else {
        for (int k = 0; k < no; ++k) v += L.dphi[k] * s.td.lam_u[(int64_t)k * s.n_unp + (j - nd)];
      }
      L.vv[j] = v;
      part += v * L.Gi[j * nu + idx];
    }
  } else {
    for (int i = lane; i < nu; i += WAVE) {
      const double* pr = L.pr + (int64_t)i * no;
      double u = 0.0;
#pragma unroll 4
      for (int k = 0; k < no; ++k) u += pr[k] * L.dphi[k];
      L.vv[i] = u;
      part += L.Gi[idx * nu + i] * u;
    }
  }
  const double det_ratio = 1.0 + wave_sum(part);
  wave_sync();
  if (is_up) {
    for (int p = lane; p < nu; p += WAVE) {
      L.xx[p] = L.Gi[p * nu + idx];
      double y = 0.0;
#pragma unroll 4
      for (int j = 0; j < nu; ++j) y += L.vv[j] * L.Gi[j * nu + p];
      L.yy[p] = y;
    }
  } else {
    for (int p = lane; p < nu; p += WAVE) {
      double x = 0.0;
#pragma unroll 4
      for (int i = 0; i < nu; ++i) x += L.Gi[p * nu + i] * L.vv[i];
      L.xx[p] = x;
      L.yy[p] = L.Gi[idx * nu + p];
    }
  }
  wave_sync();

  // ---- AS-regularised acceptance (jqmc_mcmc.py:4484-4520)
  const double R_p = sweep_as_factor(L, nu, lane, is_up ? 1 : 2, idx, det_ratio);
  const double R_AS_ratio = (fmax(R_p, eps_AS) / R_p) / (fmax(R_o, eps_AS) / R_o);
  const double wr = R_AS_ratio * J_ratio * det_ratio;
  const bool accepted = bdraw < fmin(1.0, wr * wr * T_ratio);

  if (accepted) {
    if (lane == 0) {
      double* rp = is_up ? wk.r_up + w * 3 * nu + 3 * idx : wk.r_dn + w * 3 * nd + 3 * idx;
      rp[0] = nx;
      rp[1] = ny;
      rp[2] = nz;
      ws.Ro[w] = R_p;
      ws.mv[w] = e;
      wk.accepted[w] += 1;
    }
    T* Aem = Aw + (int64_t)e * na;
    for (int a = lane; a < na; a += WAVE) Aem[a] = L.anew[a];
    double* Pem = Pw + (int64_t)e * no;
    double* Qem = Qw + (int64_t)e * no;
    const double* Lm = is_up ? s.td.lam_p : s.td.lam_pT;
    for (int k = lane; k < no; k += WAVE) {
      Pem[k] = L.phin[k];
      double q = 0.0;
#pragma unroll kPairLoads
      for (int j = 0; j < no; ++j) q += Lm[(int64_t)j * no + k] * L.phin[j];
      Qem[k] = q;
    }
    for (int t = lane; t < nu * nu; t += WAVE) {
      const int p = t / nu, q = t - p * nu;
      wk.Ginv[w * nu * nu + t] = L.Gi[t] - L.xx[p] * L.yy[q] / det_ratio;
      double gm = L.Gm[t];
      if (is_up && p == idx) gm += L.vv[q];
      if (!is_up && q == idx) gm += L.vv[p];
      wk.G[w * nu * nu + t] = gm;
    }
  } else if (lane == 0) {
    ws.mv[w] = -1;
    wk.rejected[w] += 1;
  }
}

// Walkers up to which every wave of k_sweep_propose<T, false> is on the card at once: five on each of 4 x 256 SIMDs.
constexpr int64_t PROP_MANY = 5 * 4 * 256;

constexpr int JF_SEG = 64;      // walkers whose movers one block collects
constexpr int JF_KC = 16;       // AO columns per step
constexpr int64_t JF_WIDE_BLOCKS = 6 * 256;  // blocks of one AO tile from which a block takes two
constexpr int JF_LD = 17;       // words per LDS row of the staged changes: no conflict over 16 rows

// Matrix-core step of the J3 field products: D(16 x 16) += A(16 x 4) B(4 x 16) with A(i, k) from lane
// i + 16 k and B(k, j) from lane j + 16 k; row(q, ih) is the tile row that element q of lane
// il + 16 ih holds (column il).  FP64: v_mfma_f64_16x16x4f64, D(i, j) in lane j + 16 (i % 4), element
// i / 4.  FP32 (mixed form): v_mfma_f32_16x16x4f32, D(i, j) in lane j + 16 (i / 4), element i % 4.
template <typename T>
struct JfMfma;
template <>
struct JfMfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int q, int ih) { return 4 * q + ih; }
};
template <>
struct JfMfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int q, int ih) { return 4 * ih + q; }
};

// J3 fields of every electron of every walker from the prefix sums of k_init_jsums as one FP64 GEMM on
// the matrix cores: rows = the M = W n_el electrons, G[m, a] = j1[a] (NULL: 0) + sum_b S1[m, b] J3T[b, a] +
// sum_b S2[m, b] J3[b, a] (jastrow_factor.py:4121-4135); a symmetric J3 takes one product with S1 + S2.
// Bound by the FP64 matrix rate (4 n_ao^2 flops per electron): 64 x 64 output tiles, 16-deep slices of
// both operands through LDS with the next slice in registers, four waves of 2 x 2 MFMA tiles each.
// The column tiles of a row tile are eight blocks apart, so they run on one XCD and share the rows in
// its L2.  512 benzene walkers (15360 x 228): 1389 us with one thread per output and n_ao dependent
// steps, 98 us as this GEMM (33 TFLOP/s).
constexpr int JG_TILE = 64, JG_KC = 16, JG_FEW = 1024;
constexpr int JG_A_LD = JG_KC + 1;    // doubles per LDS row of S: 34 banks apart, no conflict over 16 rows
constexpr int JG_B_LD = JG_TILE + 8;  // the four 16-lane groups read rows 16 banks apart

__global__ void __launch_bounds__(256) k_init_jfield_mfma(Sys s, int64_t M, const double* __restrict__ S1,
                                                          const double* __restrict__ S2,
                                                          const double* __restrict__ j1, double* __restrict__ G,
                                                          int n_ct, int64_t n_rt) {
  using MF = JfMfma<double>;
  __shared__ double a_s[JG_TILE][JG_A_LD];
  __shared__ double b_s[JG_KC][JG_B_LD];
  const int64_t blk = blockIdx.x;
  const int64_t rt = (blk / (8 * n_ct)) * 8 + blk % 8;
  const int ct = (int)((blk / 8) % n_ct);
  if (rt >= n_rt) return;  // uniform across the block
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, il = lane & 15, ih = lane >> 4;
  const int na = s.n_ao, a0 = ct * JG_TILE;
  const int64_t m0 = rt * JG_TILE;
  const bool sym = s.j3_sym != 0;
  const int wr = 32 * (wave >> 1), wc = 32 * (wave & 1);
  const int n_k = (na + JG_KC - 1) / JG_KC, n_stage = sym ? n_k : 2 * n_k;
  double pa[4], pb[4];
  // thread t stages column b0 + t % 16 of rows t / 16 + 16 r of S, and column t % 64 of rows
  // t / 64 + 4 r of J
  auto fetch = [&](int st) {
    const bool second = st >= n_k;
    const int b0 = (second ? st - n_k : st) * JG_KC;
    const double* __restrict__ S = second ? S2 : S1;
    const double* __restrict__ J = second ? s.td.j3 : s.td.j3T;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t m = m0 + (t >> 4) + 16 * r;
      const int b = b0 + (t & 15);
      const bool ok = m < M && b < na;
      pa[r] = ok ? S[m * na + b] : 0.0;
      if (sym && ok) pa[r] += S2[m * na + b];
      const int bb = b0 + (t >> 6) + 4 * r, a = a0 + (t & 63);
      pb[r] = (bb < na && a < na) ? J[(int64_t)bb * na + a] : 0.0;
    }
  };
  MF::v4 acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) acc[x][y] = MF::v4{0, 0, 0, 0};
  fetch(0);
  for (int st = 0; st < n_stage; ++st) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      a_s[(t >> 4) + 16 * r][t & 15] = pa[r];
      b_s[(t >> 6) + 4 * r][t & 63] = pb[r];
    }
    __syncthreads();
    if (st + 1 < n_stage) fetch(st + 1);
#pragma unroll
    for (int kk = 0; kk < JG_KC; kk += 4) {
      double fa[2], fb[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        fa[x] = a_s[wr + 16 * x + il][kk + ih];
        fb[x] = b_s[kk + ih][wc + 16 * x + il];
      }
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = MF::mma(fa[x], fb[y], acc[x][y]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    const int a = a0 + wc + 16 * y + il;
    if (a >= na) continue;
    const double ja = j1 ? j1[a] : 0.0;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t m = m0 + wr + 16 * x + MF::row(q, ih);
        if (m < M) G[m * na + a] = ja + acc[x][y][q];
      }
  }
}

// The same bit for bit with a wave per 16 x 16 tile and the operands straight from L2, for small systems (at most
// JG_TILE AOs) up to JG_FEW row tiles of the form above, whose slices cost a memory latency each.  The whole set-up
// of N2 (24 AOs): 64 walkers 49 us with that form and 45 so, 2048 walkers 71 and 68, 8192 (1280 row tiles) 151 and
// 148; 256 walkers of H2 with 50 AOs 39 and 33.  Many AOs take it worse: 16 walkers of 4 x H2O (300) 289 and 316 us.
__global__ void __launch_bounds__(256) k_init_jfield_tile(Sys s, int64_t M, const double* __restrict__ S1,
                                                          const double* __restrict__ S2, const double* __restrict__ j1,
                                                          double* __restrict__ G) {
  using MF = JfMfma<double>;
  const int lane = lane_id(), il = lane & 15, ih = lane >> 4, na = s.n_ao, n_ct = (na + 15) / 16;
  const int64_t id = (int64_t)blockIdx.x * 4 + wave_id(), m0 = id / n_ct * 16;
  if (m0 >= M) return;
  const int a0 = (int)(id % n_ct) * 16, a = a0 + il < na ? a0 + il : na - 1;
  const bool sym = s.j3_sym != 0, row = m0 + il < M;
  const int64_t m = row ? m0 + il : M - 1;
  MF::v4 acc = {0, 0, 0, 0};
  for (int part = 0; part < (sym ? 1 : 2); ++part) {
    const double* __restrict__ S = (part ? S2 : S1) + m * na;
    const double* __restrict__ T = S2 + m * na;
    const double* __restrict__ J = (part ? s.td.j3 : s.td.j3T) + a;
    for (int b0 = 0; b0 < na; b0 += 16) {
      double fa[4], ft[4], fb[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int b = b0 + 4 * x + ih < na ? b0 + 4 * x + ih : na - 1;
        fa[x] = S[b];
        ft[x] = sym ? T[b] : 0.0;
        fb[x] = J[(int64_t)b * na];
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const bool ok = b0 + 4 * x + ih < na;
        if (sym) fa[x] += ft[x];
        acc = MF::mma(ok && row ? fa[x] : 0.0, ok ? fb[x] : 0.0, acc);
      }
    }
  }
  if (a0 + il >= na) return;
  const double ja = j1 ? j1[a] : 0.0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int64_t r = m0 + MF::row(q, ih);
    if (r < M) G[r * na + a] = ja + acc[q];
  }
}

// [T1 | T2] = [J3 dA | J3^T dA] of the walkers that accepted, then their field increments: an up move of
// e gives t1 to up f < e and t2 to every other electron; a dn move gives t1 to every up electron
// and to dn f < e, t2 to dn f > e.  The part shared by a spin block goes to its offset, the mover's
// own row is compensated, and the side of the mover's block with fewer electrons takes the
// individual correction (none for a symmetric J3).  With kDirect (the LRDMC move, whose fields are
// read by the next Hamiltonian launch), every row f != e of a moved walker takes its increment
// instead: t1 for f < e, t2 for f > e, no offsets.
//
// The four waves of a block share 64 walkers and 16 NT AOs: wave t takes the movers 16 t .. 16 t + 15 of the 64
// (in order; a wave without any leaves at once) as the rows of D(mover, a) = sum_b dA(mover, b) J(b, a).
// A(i, k) = dA of mover i at AO b0 + k through the wave's own LDS tile, B(k, j) = J3^T or J3 at (b0 + k, AO
// a0 + 16 y + j) straight from L2, both with the next sixteen b on their way during the current ones: no barrier, so
// that the products of some waves overlap the row updates of others, and many small blocks, so that small
// walker counts fill the chip.  The sums run over b in order in fours.  The AO tiles of a segment are eight
// blocks apart (one XCD): the lines that two tiles share meet in its L2.
// Bound by the row updates at large walker counts (104 bytes per AO and accepted move of benzene, 340 MB of
// 16384 walkers, at scattered rows) and by latency at small ones.  Blocks of 32 walkers x 64 AOs with barriers
// took 32.7 us for 1024 benzene walkers, 175 us for 16384, 38.5 us for 2048 of 4 x H2O in FP32 and 9.3 us for
// 256 of H2O; one tile (NT = 1) 20.8, 173, 27.7 and 7.7 us.  Two tiles keep those small launches waiting (31.4 and
// 36.0 us), 32 movers a wave give 171 us for 16384.
// NT = 2 is for launches that stay many blocks all the same (JF_WIDE_BLOCKS: six of one tile per CU, so at least
// three of two): then the pieces of rows bound, 64 bytes of FP32 or 128 of FP64 with one tile.  A move of the whole
// sweep, one tile -> two: 4 x H2O, FP32, 4096 walkers (1216 blocks) 97.7 -> 99.5 us, 8192 (2432) 197 -> 181 us,
// 16384 392 -> 350 us; benzene 8192 (1920) 152 -> 145 us; 30 electrons and 120 AOs 8192 (1024) 96.7 -> 99.9 us,
// 16384 (2048) 190 -> 185 us.  In FP64 4 x H2O 16384 504 -> 485 us, benzene 362 -> 358 us (three waves a SIMD; held
// to four it spills, 513 and 378 us).  Four tiles are slower (FP32 214 us for 8192 of 4 x H2O).  The LRDMC move
// keeps one tile (its other launches outweigh it: 4096 walkers of 4 x H2O 874 -> 863 us).
// A symmetric J3 takes the same product twice: a branch around the second put the operands in scratch (274 us for
// 16384).
template <typename T, bool kDirect, int NT>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(std::is_same<T, double>::value && NT == 2 ? 3 : 4)))
    k_sweep_jfield_mfma(Sys s, int64_t W, WalkT<T> wk, SweepWs<T> ws) {
  using M = JfMfma<T>;
  typedef typename M::v4 v4;
  __shared__ T da_sh[4][2][JF_KC * JF_LD];
  __shared__ int mv_sh[4][JF_SEG], at_sh[4][JF_SEG];
  const int lane = threadIdx.x & 63, wave = wave_id(), il = lane & 15, ih = lane >> 4;
  const int nu = s.n_up, ne = s.n_el, na = s.n_ao;
  constexpr int TA = 16 * NT, H = 4 / NT;  // AOs of a wave; rows of a pass of the epilogue
  const int n_ct = (na + TA - 1) / TA;
  const int64_t blk = blockIdx.x, w0 = (blk / (8 * n_ct) * 8 + blk % 8) * JF_SEG;
  const int a0 = (int)((blk / 8) % n_ct) * TA;
  if (w0 >= W) return;
  const int e_l = w0 + lane < W ? ws.mv[w0 + lane] : -1;
  const uint64_t movers = __ballot(e_l >= 0);
  const int n = __popcll(movers) - 16 * wave;  // movers of this wave and the later ones
  if (n <= 0) return;
  int* mv_s = mv_sh[wave];
  int* at_s = at_sh[wave];
  if (e_l >= 0) {
    const int r = __popcll(movers & ((1ull << lane) - 1ull)) - 16 * wave;
    if (r >= 0) {
      mv_s[r] = e_l;
      at_s[r] = lane;
    }
  }
  wave_sync();
  const T* __restrict__ JT = tabs<T>(s).j3T;
  const T* __restrict__ JJ = tabs<T>(s).j3;
  // staged change: columns (lane & 3) + 4 r of mover lane / 4 (past the last mover: zeros)
  const int sr = lane >> 2, sk = lane & 3;
  const bool s_on = sr < n;
  const T* __restrict__ DA = ws.dA + (w0 + at_s[s_on ? sr : 0]) * na;
  int a[NT];  // columns past the end are not used
  bool in[NT];
#pragma unroll
  for (int y = 0; y < NT; ++y) {
    in[y] = a0 + 16 * y + il < na;
    a[y] = in[y] ? a0 + 16 * y + il : na - 1;
  }
  T pa[4], pt[NT][4], pj[NT][4], ct[NT][4], cj[NT][4];
  auto fetch = [&](int b0) {  // without branches: AOs past the end repeat the last one
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int ba = b0 + sk + 4 * q < na ? b0 + sk + 4 * q : na - 1;
      const int b = b0 + 4 * q + ih < na ? b0 + 4 * q + ih : na - 1;
      pa[q] = DA[ba];
#pragma unroll
      for (int y = 0; y < NT; ++y) {
        pt[y][q] = JT[(int64_t)b * na + a[y]];
        pj[y][q] = JJ[(int64_t)b * na + a[y]];
      }
    }
  };
  v4 acc1[NT], acc2[NT];
#pragma unroll
  for (int y = 0; y < NT; ++y) acc1[y] = acc2[y] = v4{0, 0, 0, 0};
  fetch(0);
  for (int b0 = 0, st = 0; b0 < na; b0 += JF_KC, st ^= 1) {
    T* da = da_sh[wave][st];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      da[(sk + 4 * q) * JF_LD + sr] = s_on && b0 + sk + 4 * q < na ? pa[q] : (T)0;  // zero against repeated rows of J
#pragma unroll
      for (int y = 0; y < NT; ++y) {
        ct[y][q] = pt[y][q];
        cj[y][q] = pj[y][q];
      }
    }
    if (b0 + JF_KC < na) fetch(b0 + JF_KC);
    asm volatile("" ::: "memory");  // one wave's LDS accesses are taken in order
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const T fa = da[(4 * q + ih) * JF_LD + il];
#pragma unroll
      for (int y = 0; y < NT; ++y) {
        acc1[y] = M::mma(fa, ct[y][q], acc1[y]);
        acc2[y] = M::mma(fa, cj[y][q], acc2[y]);
      }
    }
  }
  if (!in[0]) return;  // no cross-lane work follows
  // epilogue: element q of this lane is mover row(q, ih) of the wave
  int ee[4];
  int64_t ww[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = M::row(q, ih);
    ee[q] = r < n ? mv_s[r] : -1;
    ww[q] = w0 + at_s[r < n ? r : 0];
  }
  if constexpr (kDirect) {
    static_assert(!kDirect || NT == 1);
    const int a1 = a[0];
    const v4 t1 = acc1[0], t2 = acc2[0];
    // four rows of the four walkers per pass, all 16 loads in flight together
    for (int f0 = 0; f0 < ne; f0 += 4) {
      T v[4][4];
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int f = f0 + h;
          v[h][q] = (f < ne && ee[q] >= 0 && f != ee[q]) ? wk.jfield[(ww[q] * ne + f) * na + a1] : (T)0;
        }
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int f = f0 + h;
          if (f < ne && ee[q] >= 0 && f != ee[q])
            wk.jfield[(ww[q] * ne + f) * na + a1] = v[h][q] + (f < ee[q] ? t1[q] : t2[q]);
        }
    }
    return;
  }
  const bool sym = s.j3_sym != 0;
  int cs[4], cn[4];
  bool upm[4], lw[4];
  T d4[NT][4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int e = ee[q];
    upm[q] = e < nu;
    const int f0 = upm[q] ? 0 : nu, f1 = upm[q] ? nu : ne;
    lw[q] = sym || (e - f0) <= (f1 - 1 - e);
    cs[q] = 0;
    cn[q] = 0;
    if (e >= 0 && !sym) {
      cs[q] = lw[q] ? f0 : e + 1;
      cn[q] = (lw[q] ? e : f1) - cs[q];
    }
    if constexpr (NT == 1) {
      d4[0][q] = lw[q] ? acc1[0][q] - acc2[0][q] : acc2[0][q] - acc1[0][q];
    } else {
#pragma unroll
      for (int y = 0; y < NT; ++y) d4[y][q] = lw[q] ? acc1[y][q] - acc2[y][q] : acc2[y][q] - acc1[y][q];
    }
  }
  if constexpr (std::is_same<T, double>::value && NT == 1) {
    // the updates below written without the loops over tiles, which take FP64 0.5 of 20 us more (1024 benzene walkers)
    const int a1 = a[0];
    const v4 t1 = acc1[0], t2 = acc2[0];
    T go[4], ou[4], od[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bool on = ee[q] >= 0;
      go[q] = on ? wk.jfield[(ww[q] * ne + ee[q]) * na + a1] : (T)0;
      ou[q] = on ? ws.Oup[ww[q] * na + a1] : (T)0;
      od[q] = on ? ws.Odn[ww[q] * na + a1] : (T)0;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (ee[q] < 0) continue;
      const T own = lw[q] ? t2[q] : t1[q];
      wk.jfield[(ww[q] * ne + ee[q]) * na + a1] = go[q] - own;
      ws.Oup[ww[q] * na + a1] = ou[q] + (upm[q] ? own : t1[q]);
      ws.Odn[ww[q] * na + a1] = od[q] + (upm[q] ? t2[q] : own);
    }
    int nmax = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) nmax = cn[q] > nmax ? cn[q] : nmax;
    for (int r = 0; r < nmax; r += 4) {
      T v[4][4];
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          v[h][q] = r + h < cn[q] ? wk.jfield[(ww[q] * ne + cs[q] + r + h) * na + a1] : (T)0;
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (r + h < cn[q]) wk.jfield[(ww[q] * ne + cs[q] + r + h) * na + a1] = v[h][q] + d4[0][q];
    }
    return;
  }
  {
    T go[4][NT], ou[4][NT], od[4][NT];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int y = 0; y < NT; ++y) {
        const bool on = ee[q] >= 0 && in[y];
        go[q][y] = on ? wk.jfield[(ww[q] * ne + ee[q]) * na + a[y]] : (T)0;
        ou[q][y] = on ? ws.Oup[ww[q] * na + a[y]] : (T)0;
        od[q][y] = on ? ws.Odn[ww[q] * na + a[y]] : (T)0;
      }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int y = 0; y < NT; ++y) {
        if (ee[q] < 0 || !in[y]) continue;
        const T own = lw[q] ? acc2[y][q] : acc1[y][q];
        wk.jfield[(ww[q] * ne + ee[q]) * na + a[y]] = go[q][y] - own;
        ws.Oup[ww[q] * na + a[y]] = ou[q][y] + (upm[q] ? own : acc1[y][q]);
        ws.Odn[ww[q] * na + a[y]] = od[q][y] + (upm[q] ? acc2[y][q] : own);
      }
  }
  // individual corrections: rows cs .. cs + cn - 1 of each walker get d, H rows per pass with all their
  // loads in flight together
  int nmax = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) nmax = cn[q] > nmax ? cn[q] : nmax;
  for (int r = 0; r < nmax; r += H) {
    T v[H][4][NT];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int y = 0; y < NT; ++y)
          v[h][q][y] = r + h < cn[q] && in[y] ? wk.jfield[(ww[q] * ne + cs[q] + r + h) * na + a[y]] : (T)0;
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int y = 0; y < NT; ++y)
          if (r + h < cn[q] && in[y])
            wk.jfield[(ww[q] * ne + cs[q] + r + h) * na + a[y]] = v[h][q][y] + d4[y][q];
  }
}

// The J3 field update of one move.
template <typename T, bool kDirect>
inline void launch_jfield_move(const Sys& s, int64_t W, const WalkT<T>& wk, const SweepWs<T>& ws, hipStream_t st) {
  const int64_t segs = (W + JF_SEG - 1) / JF_SEG;
  auto run = [&](auto N) {
    constexpr int NT = decltype(N)::value;
    const int64_t n_ct = (s.n_ao + 16 * NT - 1) / (16 * NT);
    k_sweep_jfield_mfma<T, kDirect, NT><<<(unsigned)((segs + 7) / 8 * 8 * n_ct), 256, 0, st>>>(s, W, wk, ws);
  };
  if constexpr (!kDirect)
    if (segs * ((s.n_ao + 15) / 16) >= JF_WIDE_BLOCKS) return run(std::integral_constant<int, 2>{});
  run(std::integral_constant<int, 1>{});
}

// Offsets into every field row and the AS factor into the walker state (one thread per element).
template <typename T>
__global__ void k_sweep_flush(int64_t W, WalkT<T> wk, SweepWs<T> ws, int n_el,
                              int n_ao, int n_up) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per_w = (int64_t)n_el * n_ao;
  if (idx < W * per_w && wk.jfield) {
    const int64_t w = idx / per_w;
    const int64_t r = idx - w * per_w;
    const int f = (int)(r / n_ao), a = (int)(r - (int64_t)f * n_ao);
    wk.jfield[idx] += f < n_up ? ws.Oup[w * n_ao + a] : ws.Odn[w * n_ao + a];
  }
  if (idx < W && wk.as_factor) wk.as_factor[idx] = ws.Ro[idx];
}

}  // namespace jqmc
