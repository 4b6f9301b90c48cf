// gfx950 kernels of the per-walker log-derivatives O_k = d ln|Psi| / d p_k (the SR inputs of
// jqmc_mcmc.py:854-873) for the variational blocks J1 b, J2 b, J3 matrix and Lambda:
//
//   k_rank_outer     out[w][m][n] = sum_k L[w][k][m] R[w][k][n] on the matrix cores: Z = G^-1 Phi_up, the J3
//                    block sum_{e<f} a_e a_f^T = sum_e a_e (sum_{f>e} a_f)^T and the Lambda_p block
//                    Z[:n_dn]^T Phi_dn
//   k_dlnpsi_small   J1 / J2 parameter derivatives, the J3 one-body column sum_e a_e and the
//                    Lambda_u block Z[n_dn:]^T, one block per walker
#pragma once

#include "jqmc_elp.hip"
#include "jqmc_lrdmc.hip"

namespace jqmc {

constexpr int RO_ROWS = 16, RO_TY = 5;                // output rows per block; column tiles per wave and step
constexpr int RO_COLS = 4 * 16 * RO_TY, RO_LD = RO_COLS + 1;

// out[w * out_ld + out_off + m * out_rs + n] = sum_{k < K} L[w * l_ld + k * l_rs + m * l_cs] R[w * r_ld + k * r_rs + n]
// for m < M, n < N.  A block owns 16 rows, its waves every fourth 16-column tile of 320 columns a step: operands
// straight from L2, products on the FP64 matrix cores, the result through LDS so that a wave writes whole rows.
// The row tiles of a walker are eight blocks apart (one XCD), so R is read from memory once.  Bound by writing
// the result, 0.56 GB each for the blocks of 777 walkers with 300 AOs, at 2.8 (Lambda, K = 16) and 2.2 TB/s (J3,
// K = 32): 201 and 257 us, and G^-1 Phi 25 us.  64 x 64 tiles of scalar FMAs took 249 us for each block and a
// thread per element 91 us for G^-1 Phi; 64 rows a block with whole-line stores 204, 270 and 35 us.
template <typename TL, typename TR>
__global__ void __launch_bounds__(256) k_rank_outer(int K, int M, int N, int64_t W, const TL* __restrict__ L, int64_t l_ld,
                                                    int64_t l_rs, int64_t l_cs, const TR* __restrict__ R, int64_t r_ld,
                                                    int64_t r_rs, double* __restrict__ out, int64_t out_ld,
                                                    int64_t out_rs, int64_t out_off) {
  using MF = JfMfma<double>;
  __shared__ double tile[RO_ROWS * RO_LD];
  const int n_mt = (M + RO_ROWS - 1) / RO_ROWS;
  const int64_t blk = blockIdx.x, w = blk / (8 * n_mt) * 8 + blk % 8;
  const int mt = (int)((blk / 8) % n_mt);
  const int wave = wave_id(), lane = lane_id(), il = lane & 15, ih = lane >> 4;
  if (w >= W) return;  // uniform across the block
  const int m0 = mt * RO_ROWS, m = m0 + il;
  const TL* Lw = L + w * l_ld + (m < M ? m : M - 1) * l_cs;
  const TR* Rw = R + w * r_ld;
  double* ow = out + w * out_ld + out_off + (int64_t)m0 * out_rs;
  const int rows = M - m0 < RO_ROWS ? M - m0 : RO_ROWS;
  for (int n0 = 0; n0 < N; n0 += RO_COLS) {
    const int n_t = (N - n0 + 15) / 16;  // column tiles left
    const int ty = n_t > wave ? (n_t - wave + 3) / 4 : 0;
    MF::v4 acc[RO_TY];
#pragma unroll
    for (int y = 0; y < RO_TY; ++y) acc[y] = MF::v4{0, 0, 0, 0};
    // sixteen k at a time, their loads in flight together; k and columns past the end repeat the last one
    for (int k0 = 0; k0 < K && ty > 0; k0 += 16) {
      double fa[4], fb[4][RO_TY];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int k = k0 + 4 * x + ih < K ? k0 + 4 * x + ih : K - 1;
        fa[x] = (double)Lw[(int64_t)k * l_rs];
#pragma unroll
        for (int y = 0; y < RO_TY; ++y) {
          const int n = n0 + 16 * (wave + 4 * y) + il;
          if (y < ty) fb[x][y] = (double)Rw[(int64_t)k * r_rs + (n < N ? n : N - 1)];
        }
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const bool ok = k0 + 4 * x + ih < K;
        const double a = ok && m < M ? fa[x] : 0.0;
#pragma unroll
        for (int y = 0; y < RO_TY; ++y)
          if (y < ty) acc[y] = MF::mma(a, ok ? fb[x][y] : 0.0, acc[y]);
      }
    }
    if (n0 > 0) __syncthreads();
#pragma unroll
    for (int y = 0; y < RO_TY; ++y)
#pragma unroll
      for (int q = 0; q < 4; ++q) tile[MF::row(q, ih) * RO_LD + 16 * (wave + 4 * y) + il] = acc[y][q];
    __syncthreads();
    for (int r = wave; r < rows; r += 4)
#pragma unroll
      for (int y = 0; y < RO_TY; ++y) {
        const int n = n0 + 64 * y + lane;
        if (n < N) ow[(int64_t)r * out_rs + n] = tile[r * RO_LD + 64 * y + lane];
      }
  }
}

// The same with a wave per 16 rows x 16 TY columns of the result (TY = 2; 1 up to 16 columns), stored straight from
// the registers: same sums in the same order.  For at most RO_NARROW columns, where the waves of the form above
// stand idle.  The whole call for 8192 walkers: N2 with 24 AOs 126 -> 55 us, 50 AOs 209 -> 115, 94 AOs 418 -> 316,
// 94 AO orbitals 717 -> 596 (TY = 1: 56, 138, 338, 634; TY = 4: 64, 113, 321, 604); 1024 walkers of C6H6 with 120
// AOs 99 us so and 89 with the form above.
constexpr int RO_NARROW = 112;
template <int TY, typename TL, typename TR>
__global__ void __launch_bounds__(256) k_rank_narrow(int K, int M, int N, int64_t W, const TL* __restrict__ L,
                                                     int64_t l_ld, int64_t l_rs, int64_t l_cs,
                                                     const TR* __restrict__ R, int64_t r_ld, int64_t r_rs,
                                                     double* __restrict__ out, int64_t out_ld, int64_t out_rs,
                                                     int64_t out_off) {
  using MF = JfMfma<double>;
  const int lane = lane_id(), il = lane & 15, ih = lane >> 4;
  const int n_ct = (N + 16 * TY - 1) / (16 * TY), n_t = (M + 15) / 16 * n_ct;
  const int64_t id = (int64_t)blockIdx.x * 4 + wave_id(), w = id / n_t;
  if (w >= W) return;
  const int t = (int)(id - w * n_t), m0 = t / n_ct * 16, n0 = (t - t / n_ct * n_ct) * 16 * TY;
  const int m = m0 + il < M ? m0 + il : M - 1;
  const TL* Lw = L + w * l_ld + m * l_cs;
  const TR* Rw = R + w * r_ld;
  int n[TY];
  MF::v4 acc[TY];
#pragma unroll
  for (int y = 0; y < TY; ++y) {
    n[y] = n0 + 16 * y + il < N ? n0 + 16 * y + il : N - 1;
    acc[y] = MF::v4{0, 0, 0, 0};
  }
  for (int k0 = 0; k0 < K; k0 += 16) {  // the last k again past the end, against a zero
    double fa[4], fb[4][TY];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int k = k0 + 4 * x + ih < K ? k0 + 4 * x + ih : K - 1;
      fa[x] = (double)Lw[(int64_t)k * l_rs];
#pragma unroll
      for (int y = 0; y < TY; ++y) fb[x][y] = (double)Rw[(int64_t)k * r_rs + n[y]];
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const bool ok = k0 + 4 * x + ih < K;
      const double a = ok && m0 + il < M ? fa[x] : 0.0;
#pragma unroll
      for (int y = 0; y < TY; ++y) acc[y] = MF::mma(a, ok ? fb[x][y] : 0.0, acc[y]);
    }
  }
  double* ow = out + w * out_ld + out_off + n0 + il;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = m0 + MF::row(q, ih);
    if (r >= M) continue;
#pragma unroll
    for (int y = 0; y < TY; ++y)
      if (n0 + 16 * y + il < N) ow[(int64_t)r * out_rs + 16 * y] = acc[y][q];
  }
}

// Offsets (in doubles, per walker) of the O_k blocks; -1 when a block is absent.
struct ParamLayout {
  int64_t j1, j2, j3, lam, total;
};

// d/db of the one- and two-body Jastrow sums (jastrow_factor.py:672-711, 1207-1230), the J3
// one-body column d/dj[a] = sum_e a_e[a] and the unpaired Lambda block
// d/dLambda_u[k][u] = Z[n_dn + u][k] (determinant.py:1379-1402); one block per walker, its waves (four, or one for
// at most 16 electrons and 64 AOs) sharing the pairs and columns.  Latency bound: 777 walkers of 4 x H2O 100 us with
// one wave and 31 with four; 8192 of H2 with 10 AOs, whole call, 81 us with four and 32 with one.
template <typename T>
__global__ void __launch_bounds__(256) k_dlnpsi_small(Sys s, int64_t W, WalkT<T> wk, const double* __restrict__ Z,
                                                      ParamLayout lay, double* __restrict__ out, int64_t out_ld) {
  __shared__ double part[4][2];
  const int wave = wave_id(), lane = lane_id(), tid = threadIdx.x, nt = blockDim.x, nw = nt / WAVE;
  const int64_t w = wide_block();
  if (w >= W) return;  // uniform across the block
  const int ne = s.n_el, na = s.n_ao, no = s.n_orb, nu = s.n_up, nd = s.n_dn;
  double* ow = out + w * out_ld;
  double acc[2] = {0.0, 0.0};
  if (lay.j1 >= 0) {
    const double b = s.j1_param;
    for (int t = tid; t < ne * s.n_nuc; t += nt) {
      const int e = t / s.n_nuc, n = t - e * s.n_nuc;
      const double* r = elec_pos(s, wk, w, e);
      const double dx = r[0] - s.nuc_pos[3 * n], dy = r[1] - s.nuc_pos[3 * n + 1], dz = r[2] - s.nuc_pos[3 * n + 2];
      const double d = sqrt(dx * dx + dy * dy + dz * dz);
      const double c = s.j1_c[n], A = s.j1_A[n], cd = c * d;
      if (s.j1_type == 1) {
        const double ex = exp_nonpos(-b * cd);
        acc[0] += -A * (-(1.0 - ex) / (2.0 * b * b) + cd * ex / (2.0 * b));
      } else {
        const double den = 1.0 + b * cd;
        acc[0] += A * d * cd / (2.0 * den * den);
      }
    }
  }
  if (lay.j2 >= 0) {
    const double b = s.j2_param;
    for (int e = lane; e < ne; e += WAVE) {
      const double* r = elec_pos(s, wk, w, e);
      for (int f = e + 1 + wave; f < ne; f += nw) {
        const double* q = elec_pos(s, wk, w, f);
        const double dx = r[0] - q[0], dy = r[1] - q[1], dz = r[2] - q[2];
        const double x = sqrt(dx * dx + dy * dy + dz * dz);
        if (s.j2_type == 2) {
          const double den = 1.0 + b * x;
          acc[1] += -x * x / (2.0 * den * den);
        } else {
          const double ex = exp_nonpos(-b * x);
          acc[1] += -(1.0 - ex) / (2.0 * b * b) + x * ex / (2.0 * b);
        }
      }
    }
  }
  wave_sum_k<2>(acc);
  if (lane == 0) {
    part[wave][0] = acc[0];
    part[wave][1] = acc[1];
  }
  __syncthreads();
  if (tid == 0) {
    for (int q = 1; q < nw; ++q) {
      acc[0] += part[q][0];
      acc[1] += part[q][1];
    }
    if (lay.j1 >= 0) ow[lay.j1] = acc[0];
    if (lay.j2 >= 0) ow[lay.j2] = acc[1];
  }
  if (lay.j3 >= 0) {
    const T* A = wk.ao + w * ne * na;
    for (int a = tid; a < na; a += nt) {
      double sa = 0.0;
#pragma unroll 8
      for (int e = 0; e < ne; ++e) sa += (double)A[(int64_t)e * na + a];
      ow[lay.j3 + (int64_t)a * (na + 1) + na] = sa;
    }
  }
  if (lay.lam >= 0 && nu > nd) {
    const int unp = nu - nd;
    const double* Zw = Z + w * nu * no;
    for (int t = tid; t < no * unp; t += nt) {
      const int k = t / unp, u = t - k * unp;
      ow[lay.lam + (int64_t)k * (no + unp) + no + u] = Zw[(int64_t)(nd + u) * no + k];
    }
  }
}

}  // namespace jqmc
