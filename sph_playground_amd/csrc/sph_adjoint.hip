// Differentiable anisotropic diffusion: the loop-2 diffusion operator with a
// global conduction tensor, its transpose and its tensor gradient (FP64).
//
// With particles at rest, h, rho and Omega are fixed after the Newton solve
// and loop 2's diffusion term (circuit2.f90:376-397) is linear in T and in the
// tensor K:
//     dT_a/dt = (A(K) T)_a = sum_{b in N_a} w_ab (T_b rho_b - T_a rho_a),
//     w_ab    = m_b / (rho_b rho_a) * (K : H(r_ab, h_a)),
// H the fab / fw / n2w Hessian of the kernel at h_a (kernel.f90:377-539).
// The adjoint needs (A^T lam)_b = rho_b sum_{a: b in N_a} lam_a w_ab
// - lam_b rho_b sum_c w_bc, a gather over the reverse neighbour list R_b, and
// dL/dK_k = sum_a lam_a sum_b m_b/(rho_b rho_a) (T_b rho_b - T_a rho_a) G_ab,k
// with G_ab,k = d(K:H_ab)/dK_k, K_k = (xx, yy, zz, xy, xz, yz).
//
// For one K every pair weight is fixed, so the weights are assembled once per
// K (k_diff_weights in list order, k_diff_rweights in reverse-list order) and
// each STS stage is a streaming sparse product with one gather per pair and
// the stage's vector arithmetic at its rows' end (k_batch_stage, k_adj_stage).
// The adjoint stages leave a record (lam, Zt) per particle, and k_diff_coef
// adds eight stages' records at a time to one coefficient per pair, S_t +=
// lam_a (Zt_b - Zt_a), which k_diff_gcontract contracts with G once per
// backward pass.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "sph_kernels.h"

namespace sph {

__device__ __forceinline__ int xcd_block_a(int b, int nb) {
  int x = b & 7, i = b >> 3, q = nb >> 3, r = nb & 7;
  return x * q + (x < r ? x : r) + i;
}
__device__ __forceinline__ int gtid_a() { return xcd_block_a(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x; }

// The row of this thread in a streaming product.  With rev each XCD runs its
// range of blocks from the far end: successive stages read the same lists and
// weights, and one that starts where the last ended finds the part the
// memory-side cache still holds (a 64^3 operator is 356 MB of the cache's 256).
__device__ __forceinline__ int stage_row(int rev) {
  const int b = blockIdx.x, nb = gridDim.x;
  const int x = b & 7, q = nb >> 3, r = nb & 7;
  const int i = rev ? q + (x < r ? 1 : 0) - 1 - (b >> 3) : b >> 3;
  return (x * q + (x < r ? x : r) + i) * blockDim.x + threadIdx.x;
}

// Basis contractions G_k of the Hessian operator at h_a: K:H = sum_k K_k G_k.
template <int DIM, int KT>
__device__ __forceinline__ void hess_basis(const DiffOpArgs &a, double rx, double ry, double rz, double inv_ha,
                                           double G[6]) {
  using Kf = KernelFn<KT, double>;
  const double r2 = rx * rx + ry * ry + rz * rz;
  const double inv_r2 = 1.0 / r2;
  const double dr = sqrt(r2);
  const double inv_dr = dr * inv_r2;
  const double q = dr * inv_ha;
  const double ihd1 = ipow<DIM + 1>(inv_ha);
  const double xx = rx * rx * inv_r2, yy = ry * ry * inv_r2, zz = rz * rz * inv_r2;
  const double xy = rx * ry * inv_r2, xz = rx * rz * inv_r2, yz = ry * rz * inv_r2;
  if (a.ddw == 401) {
    // hessian_ddw_cart (kernel.f90:377-417): cst (ddf rr + df/q (I - rr))
    double df, ddf;
    Kf::df_ddf(q, df, ddf);
    const double cst = a.wcv * ihd1 * inv_ha, dfq = df / q, e = ddf - dfq;
    G[0] = cst * (e * xx + dfq);
    G[1] = DIM >= 2 ? cst * (e * yy + dfq) : 0.0;
    G[2] = DIM == 3 ? cst * (e * zz + dfq) : 0.0;
    G[3] = DIM >= 2 ? 2.0 * cst * e * xy : 0.0;
    G[4] = DIM == 3 ? 2.0 * cst * e * xz : 0.0;
    G[5] = DIM == 3 ? 2.0 * cst * e * yz : 0.0;
  } else {
    // hessian_fab_cart / hessian_fw_cart (kernel.f90:460-539): half ((d+2) rr - I)
    double half;
    if (a.ddw == 402) {
      half = 0.5 * a.fwc * a.wcv * Kf::f(q) * ihd1 * inv_ha;
    } else {
      half = -a.wcv * Kf::df(q) * ihd1 * inv_dr;
    }
    const double d2 = DIM + 2.0;
    G[0] = half * (d2 * xx - 1.0);
    G[1] = DIM >= 2 ? half * (d2 * yy - 1.0) : 0.0;
    G[2] = DIM == 3 ? half * (d2 * zz - 1.0) : 0.0;
    G[3] = DIM >= 2 ? half * 2.0 * d2 * xy : 0.0;
    G[4] = DIM == 3 ? half * 2.0 * d2 * xz : 0.0;
    G[5] = DIM == 3 ? half * 2.0 * d2 * yz : 0.0;
  }
}

__device__ __forceinline__ double kdot(const double K[6], const double G[6]) {
  return K[0] * G[0] + K[1] * G[1] + K[2] * G[2] + K[3] * G[3] + K[4] * G[4] + K[5] * G[5];
}

// Z = Y rho (the j-side value the operator reads).
__global__ void k_zrho(int n, const double *Y, const double4 *q0, double *Z) {
  int s = gtid_a();
  if (s < n) Z[s] = Y[s] * q0[s].y;
}

// pxh = (x, y, z, 1 / h), rho and 1 / rho of the frozen geometry.
__global__ void k_diff_pack(int n, const double4 *pm, const double4 *q0, double4 *pxh, double *rho, double *irho) {
  int s = gtid_a();
  if (s < n) {
    const double4 p = pm[s];
    const double4 q = q0[s];
    pxh[s] = make_double4(p.x, p.y, p.z, q.x);
    rho[s] = q.y;
    irho[s] = 1.0 / q.y;
  }
}

// Pair weights of A(K) in list order: W_ab = (m_b / rho_b) K:H_ab at the
// pair's list slot, and dW_a = sum_b W_ab (A's diagonal times rho_a^2 / rho_a).
template <int DIM, int KT>
__global__ __launch_bounds__(256) void k_diff_weights(DiffOpArgs a, double *W, double *dW) {
  int s = gtid_a();
  if (s >= a.n || !a.real[s]) return;
  const double4 pa = a.pm[s];
  const double inv_ha = a.q0[s].x;
  double sum = 0.0;
  size_t widx = (size_t)s * 8;
  const size_t wstep = (size_t)a.npad * 8 - 7;
  int k = 0;
  struct J { double4 pb; double rb; uint32_t code; };
  auto load = [&](uint32_t e) {
    J d;
    const uint32_t j = nb_index(e);
    d.code = nb_code(e);
    d.pb = a.pm[j];
    d.rb = a.q0[j].y;
    return d;
  };
  for_neighbours<1, 4>(a.nb, s, 0, a.npad, a.cnt[s], load, [&](const J &d) {
    double xb = d.pb.x, yb = d.pb.y, zb = d.pb.z;
    if (d.code != kNoImage) image_shift(xb, yb, zb, d.code, a.b);
    double G[6];
    hess_basis<DIM, KT>(a, pa.x - xb, pa.y - yb, pa.z - zb, inv_ha, G);
    const double w = d.pb.w / d.rb * kdot(a.K, G);
    W[widx] = w;
    sum += w;
    k++;
    widx += (k & 7) ? 1 : wstep;
  });
  dW[s] = sum;
}

// Reverse weights R_t = m_s K:H(r_as, h_a) / rho_a for the entries t = (a -> s)
// of s's reverse list, stored like the lists (nb_slot layout).
template <int DIM, int KT>
__global__ __launch_bounds__(256) void k_diff_rweights(DiffOpArgs a, const double *irho, double *R) {
  int s = gtid_a();
  if (s >= a.n || !a.real[s]) return;
  const double4 ps = a.pm[s];
  const int nr = a.rcnt[s];
  for (int k0 = 0; k0 < nr; k0 += 8) {
    const size_t base = nb_slot(k0, s, a.npad);
    const uint4 *pe = reinterpret_cast<const uint4 *>(a.rent + base);
    const uint4 e0 = pe[0], e1 = pe[1];
    const uint32_t e8[8] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w};
    const int m = min(8, nr - k0);
#pragma unroll
    for (int h = 0; h < 8; h += 4) {
      if (h >= m) break;
      double4 pi[4];
      double ri[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const uint32_t i = h + u < m ? nb_index(e8[h + u]) : (uint32_t)s;
        pi[u] = a.pxh[i];
        ri[u] = irho[i];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (h + u >= m) break;
        const uint32_t cd = nb_code(e8[h + u]);
        double xb = ps.x, yb = ps.y, zb = ps.z;
        if (cd != kNoImage) image_shift(xb, yb, zb, cd, a.b);
        double G[6];
        hess_basis<DIM, KT>(a, pi[u].x - xb, pi[u].y - yb, pi[u].z - zb, pi[u].w, G);
        R[base + h + u] = ps.w * kdot(a.K, G) * ri[u];
      }
    }
  }
}

// Entries and weights of a row, eight at a time, the next eight read while
// fn(entries, weights, valid) works on these: a row's chunks otherwise follow
// each other at the latency of two loads (64^3 has a single round of blocks).
template <typename WT, typename Fn>
__device__ __forceinline__ void over_chunks(const uint32_t *nb, const WT *W, int s, int npad, int nn, Fn fn) {
  using V = std::conditional_t<std::is_same_v<WT, float>, float4, double4>;
  uint4 e0{}, e1{};
  V w0{}, w1{};
  auto read = [&](int k0) {
    const size_t base = nb_slot(k0, s, npad);
    const uint4 *pe = reinterpret_cast<const uint4 *>(nb + base);
    const V *pw = reinterpret_cast<const V *>(W + base);
    e0 = pe[0]; e1 = pe[1];
    w0 = pw[0]; w1 = pw[1];
  };
  if (nn > 0) read(0);
  for (int k0 = 0; k0 < nn; k0 += 8) {
    const uint32_t e8[8] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w};
    const double w8[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
    if (k0 + 8 < nn) read(k0 + 8);
    fn(e8, w8, min(8, nn - k0));
  }
}

// out = A(K) Y from Z = Y rho: out_a = (1 / rho_a) sum_b W_ab (Z_b - Z_a);
// weights stream in list order, Z_b is the one gather per pair.
__global__ __launch_bounds__(256) void k_diff_spmv(DiffOpArgs a, const double *W, const double *Z, double *out) {
  int s = gtid_a();
  if (s >= a.n || !a.real[s]) return;
  const double za = Z[s];
  double acc = 0.0;
  over_chunks(a.nb, W, s, a.npad, a.cnt[s], [&](const uint32_t *e, const double *w, int m) {
    double z8[8];
#pragma unroll
    for (int u = 0; u < 8; u++) z8[u] = Z[u < m ? nb_index(e[u]) : (uint32_t)s];
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (u < m) acc = fma(w[u], z8[u] - za, acc);
  });
  out[s] = acc / a.q0[s].y;
}

// One adjoint stage (AdjStage, sts_integrator.f90:111-115 transposed): U =
// A^T L over the reverse lists,
//   U_s = sum_t L_a R_t - L_s dW_s,  t = (a -> s),
// and the stage's vector updates.  Bound by memory (12 bytes per pair; 64^3:
// 72 us, 5.2 TB/s, where product, record and update took three launches and
// 88 us).
__global__ __launch_bounds__(256) void k_adj_stage(AdjStage a) {
  const int s = stage_row(a.rev);
  if (s >= a.n) return;
  const double l = a.lam[s];
  double acc = 0.0;
  over_chunks(a.rent, a.R, s, a.npad, a.rcnt[s], [&](const uint32_t *e, const double *r, int m) {
    double l8[8];
#pragma unroll
    for (int u = 0; u < 8; u++) l8[u] = a.lam[u < m ? nb_index(e[u]) : (uint32_t)s];
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (u < m) acc += l8[u] * r[u];
  });
  // each sum in the order its terms come in, one rounding per term
  const double u = fma(-l, a.dW[s], acc);
  double next;
  if (a.last) {
    next = fma(a.mh, u, a.A0 ? a.A0[s] + l : 0.0);
  } else {
    next = fma(a.mh, u, fma(a.mu, l, a.lam1 ? a.nu1 * a.lam1[s] : 0.0));
    a.A0[s] = fma(a.gh, u, fma(a.c0, l, fma(a.nu0, l, a.a0_add ? a.A0[s] : 0.0)));
  }
  a.out[s] = next;
}

// The records of stages [first, count) side by side per particle (with `fill`
// the rest zero): rec[s][q] = (lam^q, Zt^q).  Written by the stages themselves,
// 16 bytes of each particle's line at a time, they cost every stage some 12 us
// at 64^3; this pass takes 23 us per eight stages.
__global__ __launch_bounds__(256) void k_adj_pack(int n, AdjRecs a, int first, int count, int fill, const double *rho,
                                                  double2 *rec) {
  const int t = gtid_a(), s = t / kRecs, q = t % kRecs;
  if (s >= n || q < first || (q >= count && !fill)) return;
  double2 r = make_double2(0.0, 0.0);
  if (q < count) {
    const double yb = a.Yb[q] ? a.wb[q] * a.Yb[q][s] : 0.0;
    r = make_double2(a.lam[q][s], (a.wa[q] * a.Ya[q][s] + yb) * rho[s]);
  }
  rec[t] = r;
}

template <int CTRL>
__device__ __forceinline__ double swap_half(bool high, double low_v, double high_v) {
  // keep one of the two values and add the partner lane's copy of it
  return (high ? high_v : low_v) + dpp_mov<CTRL>(high ? low_v : high_v);
}

// Pair coefficients of the tensor gradient, eight stages at once:
//   S_t (+)= sum_q lam^q_a (Zt^q_s - Zt^q_a),  t = (a -> s).
// Four lanes share a particle, each on two stages, so the four read a
// neighbour's records as one 128-byte line; eight entries' products are then
// summed over the lanes by halves, which leaves entries 2 l and 2 l + 1 on
// lane l, and S moves once per eight stages in whole lines.  Bound by the
// records' lines out of the caches and by S (64^3: 0.26 ms per eight stages, 3.8
// and 0.6 GB; a lane per particle and four stages at a time took 0.18 ms per
// four; fewer blocks in flight change nothing).
__global__ __launch_bounds__(256) void k_diff_coef(const uint32_t *rent, const int *rcnt, const double2 *rec,
                                                   double *S, int add, int n, int npad) {
  const int t = gtid_a(), s = t >> 2, l = t & 3;
  if (s >= n) return;
  const double2 *own = rec + (size_t)s * kRecs + 2 * l;
  const double z0 = own[0].y, z1 = own[1].y;
  const int nr = rcnt[s];
  uint4 e0{}, e1{};
  auto read = [&](int k0) {
    const uint4 *pe = reinterpret_cast<const uint4 *>(rent + nb_slot(k0, s, npad));
    e0 = pe[0]; e1 = pe[1];
  };
  if (nr > 0) read(0);
  for (int k0 = 0; k0 < nr; k0 += 8) {
    double2 *ps = reinterpret_cast<double2 *>(S + nb_slot(k0, s, npad)) + l;
    const uint32_t e8[8] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w};
    const int m = min(8, nr - k0);
    double2 sum = make_double2(0.0, 0.0);
    if (add) sum = *ps;
    if (k0 + 8 < nr) read(k0 + 8);
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const uint32_t i = u < m ? nb_index(e8[u]) : (uint32_t)s;
      const double2 *g = rec + (size_t)i * kRecs + 2 * l;
      const double2 g0 = g[0], g1 = g[1];
      v[u] = g0.x * (z0 - g0.y) + g1.x * (z1 - g1.y);
    }
    double w[4];
#pragma unroll
    for (int u = 0; u < 4; u++) w[u] = swap_half<0x4E>((l & 2) != 0, v[u], v[4 + u]);  // quad_perm [2,3,0,1]
    sum.x += swap_half<0xB1>((l & 1) != 0, w[0], w[2]);                                // quad_perm [1,0,3,2]
    sum.y += swap_half<0xB1>((l & 1) != 0, w[1], w[3]);
    *ps = sum;  // slots past the list's end are never read
  }
}

// Tensor gradient from the accumulated coefficients over the reverse lists:
//   g_k = sum_s sum_t m_s / (rho_s rho_a) G_k(r_as, h_a) S_t
// as 6 partial sums per block into gpart[block * 12 + k].  S null: one stage,
// whose S_t = lam_a (Z_s - Z_a) are formed here (through k_diff_coef's records
// and S, made for eight stages, a transposed product with two gradients took
// 0.45 ms for 1M particles in 1D and 3.93 at 100^3, so 0.23 and 1.67).
template <int DIM, int KT>
__global__ __launch_bounds__(256) void k_diff_gcontract(DiffOpArgs a, const double *irho, const double *S,
                                                        const double *lam, const double *Z, double *gpart) {
  __shared__ double red[4][12];
  int s = gtid_a();
  double g[6] = {0, 0, 0, 0, 0, 0};
  if (s < a.n && a.real[s]) {
    const double4 ps = a.pm[s];
    const double ms = ps.w * irho[s], zs = S ? 0.0 : Z[s];
    const int nr = a.rcnt[s];
    for (int k0 = 0; k0 < nr; k0 += 8) {
      const size_t base = nb_slot(k0, s, a.npad);
      const uint4 *pe = reinterpret_cast<const uint4 *>(a.rent + base);
      const uint4 e0 = pe[0], e1 = pe[1];
      const uint32_t e8[8] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w};
      const int m = min(8, nr - k0);
#pragma unroll
      for (int h = 0; h < 8; h += 4) {
        if (h >= m) break;
        double4 pi[4];
        double ri[4], ci[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const uint32_t i = h + u < m ? nb_index(e8[h + u]) : (uint32_t)s;
          pi[u] = a.pxh[i];
          ri[u] = irho[i];
          ci[u] = S ? S[base + h + u] : lam[i] * (zs - Z[i]);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (h + u >= m) break;
          const uint32_t cd = nb_code(e8[h + u]);
          double xb = ps.x, yb = ps.y, zb = ps.z;
          if (cd != kNoImage) image_shift(xb, yb, zb, cd, a.b);
          double G[6];
          hess_basis<DIM, KT>(a, pi[u].x - xb, pi[u].y - yb, pi[u].z - zb, pi[u].w, G);
          const double c = ms * ri[u] * ci[u];
          for (int k = 0; k < 6; k++) g[k] += c * G[k];
        }
      }
    }
  }
  for (int c = 0; c < 12; c++) {
    double v = c < 6 ? g[c] : 0.0;
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][c] = v;
  }
  __syncthreads();
  if (threadIdx.x < 12) {
    double t = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += red[w][threadIdx.x];
    gpart[(size_t)xcd_block_a(blockIdx.x, gridDim.x) * 12 + threadIdx.x] = t;
  }
}

// gk[c] += wa * sum_blocks gpart[b*12 + c] + wb * sum_blocks gpart[b*12 + 6 + c]
// in a fixed order (one block of 256 threads).
__global__ __launch_bounds__(256) void k_gk_accum(const double *gpart, int nblk, double wa, double wb, double *gk) {
  __shared__ double sh[12][256];
  double v[12];
  for (int c = 0; c < 12; c++) v[c] = 0.0;
  for (int b = threadIdx.x; b < nblk; b += 256)
    for (int c = 0; c < 12; c++) v[c] += gpart[(size_t)b * 12 + c];
  for (int c = 0; c < 12; c++) sh[c][threadIdx.x] = v[c];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int c = 0; c < 12; c++) sh[c][threadIdx.x] += sh[c][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 6) gk[threadIdx.x] += wa * sh[threadIdx.x][0] + wb * sh[6 + threadIdx.x][0];
}

// Reverse neighbour lists in the list layout: every list pair (s, k) takes the
// next slot of its neighbour j's reverse list, whatever the order; k_rev_sort
// then puts each list in ascending order of owner and image code, so that the
// sums over them do not depend on scheduling.  rcnt[npad] collects the longest
// list; entries past `cap` are counted but not stored (the host makes room and
// fills again).  Eight lanes per particle, whose entries go to neighbouring
// lists.
__global__ __launch_bounds__(256) void k_rev_fill(const uint8_t *real, const uint32_t *nb, const int *cnt, int n,
                                                  int npad, int cap, int *rcnt, uint32_t *rent) {
  const int t = gtid_a(), s = t >> 3, sub = t & 7;
  int longest = 0;
  if (s < n && real[s]) {
    const int m = cnt[s];
    for (int k = sub; k < m; k += 8) {
      const uint32_t e = nb[nb_slot(k, s, npad)], j = nb_index(e);
      const int pos = atomicAdd(&rcnt[j], 1);
      longest = max(longest, pos + 1);
      if (pos < cap) rent[nb_slot(pos, (int)j, npad)] = nb_pack((uint32_t)s, nb_code(e));
    }
  }
  for (int o = 32; o > 0; o >>= 1) longest = max(longest, __shfl_xor(longest, o, 64));
  if ((threadIdx.x & 63) == 0 && longest > __hip_atomic_load(&rcnt[npad], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax(&rcnt[npad], longest);
}

// Each reverse list (at most kRevSort entries) into ascending order, one wave
// per particle: an entry's place is the number of smaller ones, counted from a
// copy in LDS (a list's entries are distinct).  40^3 takes 0.06 ms here and
// 0.16 ms in k_rev_fill (bound by its 7.2M atomics) where counting, listing,
// radix-sorting and laying out the pairs took 0.47 ms; lists past kRevSort
// still go that way, whose work grows with the pairs and not with the square
// of a list.
__global__ __launch_bounds__(256) void k_rev_sort(int n, int npad, const int *rcnt, uint32_t *rent) {
  __shared__ __align__(16) uint32_t lists[4][kRevSort];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int s = xcd_block_a(blockIdx.x, gridDim.x) * 4 + w;
  if (s >= n) return;
  uint32_t *list = lists[w];
  const int m = rcnt[s], m4 = (m + 3) & ~3;
  for (int k = lane; k < m4; k += 64) list[k] = k < m ? rent[nb_slot(k, s, npad)] : 0xFFFFFFFFu;
  // the wave's own LDS accesses complete in order
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  for (int k0 = 0; k0 < m; k0 += 128) {
    const int ka = k0 + lane, kb = ka + 64;
    const uint32_t ea = ka < m ? list[ka] : 0u, eb = kb < m ? list[kb] : 0u;
    int ra = 0, rb = 0;
    for (int i = 0; i < m4; i += 4) {
      const uint4 q = *reinterpret_cast<const uint4 *>(list + i);
      ra += (q.x < ea) + (q.y < ea) + (q.z < ea) + (q.w < ea);
      rb += (q.x < eb) + (q.y < eb) + (q.z < eb) + (q.w < eb);
    }
    if (ka < m) rent[nb_slot(ra, s, npad)] = ea;
    if (kb < m) rent[nb_slot(rb, s, npad)] = eb;
  }
}

// The same lists for long ones: the pairs (key j, value: a and the image code
// of j in a's list) enumerated owner-major at foff[a] + k; a stable radix sort
// on j then gives each reverse segment in (a, k) order.
__global__ void k_rev_count(const uint8_t *real, const uint32_t *nb, const int *cnt, int n, int npad, int *rcnt) {
  int s = gtid_a();
  if (s >= n || !real[s]) return;
  for (int k = 0; k < cnt[s]; k++) atomicAdd(&rcnt[nb_index(nb[nb_slot(k, s, npad)])], 1);
}

__global__ void k_pair_enum(const uint8_t *real, const uint32_t *nb, const int *cnt, int n, int npad,
                            const int *foff, uint32_t *keys, uint32_t *vals) {
  int s = gtid_a();
  if (s >= n || !real[s]) return;
  const int base = foff[s];
  for (int k = 0; k < cnt[s]; k++) {
    const uint32_t e = nb[nb_slot(k, s, npad)];
    keys[base + k] = nb_index(e);
    vals[base + k] = nb_pack((uint32_t)s, nb_code(e));
  }
}

// Sorted reverse entries (CSR by roff) into the list layout of rent.
__global__ void k_rev_chunk(const int *roff, const uint32_t *flat, int n, int npad, int *rcnt, uint32_t *rent) {
  int s = gtid_a();
  if (s >= n) return;
  const int b = roff[s], e = roff[s + 1];
  rcnt[s] = e - b;
  for (int k = 0; k < e - b; k++) rent[nb_slot(k, s, npad)] = flat[b + k];
}

// ------------------------------------------------------- batched problems
// Many prepared problems merged into one index space: problem p's row s is
// off_p + s, its list entries point to off_p + j and its pair weights are
// copied from its own list layout into the merged one (npad_g rows).  Every
// RKL2 stage of every problem is then one launch of k_batch_stage.
__global__ void k_batch_merge(int n, int npad, int64_t off, int pid, const int *cnt, const uint32_t *nb,
                              const double *W, const double4 *q0, const int64_t *orig, int npad_g, int *mcnt,
                              uint32_t *mnb, double *mW, float *mW32, double *mrho, int64_t *morig, int *mpid) {
  int s = gtid_a();
  if (s >= n) return;
  const int64_t g = off + s;
  const int c = cnt[s];
  mcnt[g] = c;
  mrho[g] = q0[s].y;
  morig[g] = off + orig[s];
  mpid[g] = pid;
  for (int k = 0; k < c; k++) {
    const size_t src = nb_slot(k, s, npad), dst = nb_slot(k, (int)g, npad_g);
    mnb[dst] = (uint32_t)(off + nb_index(nb[src]));
    if (mW32) mW32[dst] = (float)W[src];
    else mW[dst] = W[src];
  }
}

// A product that is never fused into a following add (Z = Y rho is rounded
// before the difference, as k_zrho stores it).
__device__ __forceinline__ double mul_rn(double x, double y) {
#pragma clang fp contract(off)
  return x * y;
}

// Super-step input: Y_0 in sorted (merged) order and its Z_0 = Y_0 rho; orig
// null: T0 is in that order already.
__global__ void k_batch_in(const double *T0, const int64_t *orig, const double *rho, int n, double *Y0,
                           double *Z0) {
  int s = gtid_a();
  if (s >= n) return;
  const double y = T0[orig ? orig[s] : s];
  if (Y0 != T0) Y0[s] = y;
  Z0[s] = mul_rn(y, rho[s]);
}

// One RKL2 stage j over all problems (sts_integrator.f90:105-118), fused:
//   D   = (A Y_{j-1})_s = (1 / rho_s) sum_b W_sb (Z_b - Z_s),  Z = Y_{j-1} rho
//   j=1: DY0 = D;  Y_1 = Y_0 + mhat dt DY0
//   j>1: Y_j = mu Y_{j-1} + nu Y_{j-2} + (1 - mu - nu) Y_0 + mhat dt D + ghat dt DY0
// and Z_j = Y_j rho for the next stage's gathers.  The per-row summation
// is k_diff_spmv's and the combination a rounded first product, then explicit
// fused multiply-adds, whatever the instantiation, so every problem's result
// is bitwise the unbatched super-step's.  Y_j may be Y_0's buffer: row s reads
// only its own Y_0 entry before writing it.
// ONE: one prepared problem on its own lists, whose entries carry image codes
// (sph_diff_forward), with one time step.
template <bool FIRST, typename WT, bool ONE>
__global__ __launch_bounds__(512) void k_batch_stage(BatchStage a) {
  const int s = stage_row(a.rev);
  if (s >= a.n) return;
  const double ya = a.Yjm1[s], rs = a.rho[s];
  const double za = mul_rn(ya, rs);
  double acc = 0.0;
  const WT *W;
  if constexpr (std::is_same_v<WT, float>) W = a.W32;  // FP32 weights, FP64 products and sums
  else W = a.W;
  over_chunks(a.nb, W, s, a.npad, a.cnt[s], [&](const uint32_t *e, const double *w, int m) {
    double z8[8];
#pragma unroll
    for (int u = 0; u < 8; u++) z8[u] = a.Zjm1[u < m ? (ONE ? nb_index(e[u]) : e[u]) : (uint32_t)s];
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (u < m) acc = fma(w[u], z8[u] - za, acc);
  });
  const double D = acc / rs;
  const double h = ONE ? a.h : a.dt[a.pid[s]];
  double v;
  if (FIRST) {
    a.DY0[s] = D;
    v = fma(a.mhat * h, D, ya);
  } else {
    v = a.mu * ya;
    v = fma(a.nu, a.Yjm2[s], v);
    v = fma(a.c0, a.Y0[s], v);
    v = fma(a.mhat * h, D, v);
    v = fma(a.ghat * h, a.DY0[s], v);
  }
  a.Yj[s] = v;
  a.Zj[s] = mul_rn(v, rs);
}

// Vectors in original particle order <-> sorted order.
__global__ void k_to_sorted(const double *src, const int64_t *orig, int n, double *dst) {
  int s = gtid_a();
  if (s < n) dst[s] = src[orig[s]];
}
__global__ void k_from_sorted(const double *src, const int64_t *orig, int n, double *dst) {
  int s = gtid_a();
  if (s < n) dst[orig[s]] = src[s];
}

// ---------------------------------------------------------------------------
// Operators that read grad T: the 2nw- + / 2nw+ - second derivatives
// (circuit2.f90:398-420) and flux-limited diffusion (circuit2.f90:177-190,
// 356-397), with the geometry (h, rho, Omega of the prepared step) frozen.
//
//   U = G(Y): loop 1's grad T (circuit1.f90:172-181) of a field Y,
//     mode 1  U_a = 1/(rho_a Om_a) sum_b m_b (Y_b rho_b - Y_a rho_a) nw(r_ab, h_a)
//     mode 2  U_a = sum_b m_b (Y_a/(Om_a rho_a) nw(r_ab, h_a) + Y_b rho_a/(Om_b rho_b^2) nw(r_ab, h_b))
//   2nw-+ : f_a = sum_b m_b ((K U_a).nw_a /(Om_a rho_a^2) + (K U_b).nw_b /(Om_b rho_b^2))   (mode 1)
//   2nw+- : f_a = 1/(Om_a rho_a^2) sum_b m_b (K U_b - K U_a).nw_a                          (mode 2)
//   FLD   : f_a = 1/rho_a sum_b (m_b/rho_b) tr H_ab(h_a) (D_a + D_b)/2 (Y_b rho_b - Y_a rho_a),
//           D_a = c lambda(R_a)/(kappa_a rho_a), R_a = |U_a|/(kappa_a rho_a Y_a rho_a),
//           lambda(R) = (2 + R)/(6 + 3R + R^2)                                            (mode 1)
// with nw(r, h) = wcv df(q) r / (h^(dim+2) q) (kernel.f90:189-197).  The 2nw
// operators are linear in Y and in K; FLD is not linear in Y, and its
// adjoint is the transposed Jacobian at a state.  Every adjoint sum is a
// gather over the reverse lists: no atomics, a fixed order.

// These operators are bound by the latency of their gathers (a list entry,
// then up to five records) and by FP64 divisions: 4 or 8 lanes share a
// particle (the host's NL_LAUNCH), and 1/|r| is the refined reciprocal square root (a few
// ulp, as in loop 2).  32^3 with one lane, one entry at a time and IEEE
// divisions: grad T 97 us, the FLD operator 105, its adjoint 191; now
// 19, 17 and 33.

// nw(r, h) / r-vector: wcv df(q) / (h^(dim+2) q), from 1/|r|
template <int DIM, int KT>
__device__ __forceinline__ double nw_coef(const DiffOpArgs &a, double r2, double inv_dr, double inv_h) {
  const double q = r2 * inv_dr * inv_h;
  return a.wcv * KernelFn<KT, double>::df(q) * ipow<DIM + 1>(inv_h) * inv_dr;
}

// tr H of the Hessian operator at h (hess_basis with K = I)
template <int DIM, int KT>
__device__ __forceinline__ double hess_trace(const DiffOpArgs &a, double r2, double inv_dr, double inv_h) {
  using Kf = KernelFn<KT, double>;
  const double q = r2 * inv_dr * inv_h, ihd1 = ipow<DIM + 1>(inv_h);
  if (a.ddw == 401) {
    double df, ddf;
    Kf::df_ddf(q, df, ddf);
    // df / q with 1/q = h / |r|
    return a.wcv * ihd1 * (inv_h * ddf + (DIM - 1) * df * inv_dr);
  }
  // half ((dim + 2) - dim)
  if (a.ddw == 402) return a.fwc * a.wcv * Kf::f(q) * ihd1 * inv_h;
  return -2.0 * a.wcv * Kf::df(q) * ihd1 * inv_dr;
}

__device__ __forceinline__ double3 kmul(const double K[6], double x, double y, double z) {
  return make_double3(K[0] * x + K[3] * y + K[4] * z, K[3] * x + K[1] * y + K[5] * z,
                      K[4] * x + K[5] * y + K[2] * z);
}

// Pair loop over s's list, G lanes: fn(j's record, rx, ry, rz, r^2, 1/|r|) with
// r = x_s - x_j(image); rec(j) gathers what fn reads of j.
template <int G, typename Rec, typename Fn>
__device__ __forceinline__ void over_list(const DiffOpArgs &a, int s, int sub, const double4 &ps, Rec rec, Fn fn) {
  struct J { double4 pb; decltype(rec(0u)) r; uint32_t code; };
  auto load = [&](uint32_t e) { const uint32_t j = nb_index(e); return J{a.pm[j], rec(j), nb_code(e)}; };
  for_neighbours<G, 1>(a.nb, s, sub, a.npad, a.cnt[s], load, [&](const J &d) {
    double xb = d.pb.x, yb = d.pb.y, zb = d.pb.z;
    if (d.code != kNoImage) image_shift(xb, yb, zb, d.code, a.b);
    const double rx = ps.x - xb, ry = ps.y - yb, rz = ps.z - zb;
    const double r2 = rx * rx + ry * ry + rz * rz;
    fn(d.r, d.pb.w, rx, ry, rz, r2, rsq_nr(r2));
  });
}

// Pair loop over s's reverse list, G lanes: fn(i's record, ...) with i the owner
// (s in i's list) and r = x_i - x_s(image as i sees it).
template <int G, typename Rec, typename Fn>
__device__ __forceinline__ void over_rlist(const DiffOpArgs &a, int s, int sub, const double4 &ps, Rec rec, Fn fn) {
  struct J { double4 pi; decltype(rec(0u)) r; uint32_t code; };
  auto load = [&](uint32_t e) { const uint32_t i = nb_index(e); return J{a.pxh[i], rec(i), nb_code(e)}; };
  for_neighbours<G, 1>(a.rent, s, sub, a.npad, a.rcnt[s], load, [&](const J &d) {
    double xb = ps.x, yb = ps.y, zb = ps.z;
    if (d.code != kNoImage) image_shift(xb, yb, zb, d.code, a.b);
    const double rx = d.pi.x - xb, ry = d.pi.y - yb, rz = d.pi.z - zb;
    const double r2 = rx * rx + ry * ry + rz * rz;
    fn(d.r, d.pi.w, rx, ry, rz, r2, rsq_nr(r2));
  });
}

// U = G(Y), and with F the geometry sum F_s = sum_b m_b nw(r_sb, h_s).  With D
// (FLD) also the conductivity at state Y: D, dD/dR and R per particle.
template <int DIM, int KT, int MODE, int G>
__global__ __launch_bounds__(256) void k_nl_grad(DiffOpArgs a, const double *Y, double4 *U, double4 *F, double *D,
                                                 double *dDdR, double *R) {
  const int t = gtid_a(), s = t / G, sub = t & (G - 1);
  if (s >= a.n || !a.real[s]) return;
  const double4 ps = a.pm[s];
  const double4 qa = a.q0[s];
  const double inv_ha = qa.x, rhoa = qa.y, oma = qa.z;
  const double ya = Y ? Y[s] : 0.0;
  double ux = 0, uy = 0, uz = 0, fx = 0, fy = 0, fz = 0;
  struct Rec { double y, rho; double4 q; };
  auto rec = [&](uint32_t j) {
    Rec r{};
    if (Y) {
      r.y = Y[j];
      if constexpr (MODE == 1) r.rho = a.rho[j];
      else r.q = a.q0[j];
    }
    return r;
  };
  over_list<G>(a, s, sub, ps, rec, [&](const Rec &j, double mb, double rx, double ry, double rz, double r2, double ir) {
    const double wa = nw_coef<DIM, KT>(a, r2, ir, inv_ha);
    if (F) { fx += mb * wa * rx; fy += mb * wa * ry; fz += mb * wa * rz; }
    if (!Y) return;
    if constexpr (MODE == 1) {
      const double t = mb * (j.y * j.rho - ya * rhoa) * wa;
      ux += t * rx; uy += t * ry; uz += t * rz;
    } else {
      const double wb = nw_coef<DIM, KT>(a, r2, ir, j.q.x);
      const double ca = mb * ya / (oma * rhoa) * wa, cb = mb * j.y * rhoa / (j.q.z * j.q.y * j.q.y) * wb;
      ux += (ca + cb) * rx; uy += (ca + cb) * ry; uz += (ca + cb) * rz;
    }
  });
  group_sum<G>(ux, uy, uz);
  if (F) group_sum<G>(fx, fy, fz);
  if (sub != 0) return;
  if (F) F[s] = make_double4(fx, fy, fz, 0.0);
  if (!Y) return;
  const double c = MODE == 1 ? 1.0 / (rhoa * oma) : 1.0;
  ux *= c; uy *= c; uz *= c;
  U[s] = make_double4(ux, uy, uz, 0.0);
  if (D) {
    const double kap = a.kap[s];
    const double un = sqrt(ux * ux + uy * uy + uz * uz);
    const double r = un / (kap * rhoa * ya * rhoa);
    const double den = 6. + 3. * r + r * r;
    D[s] = kLightspeed * ((2. + r) / den) / kap / rhoa;
    dDdR[s] = kLightspeed * (-r * (4. + r) / (den * den)) / kap / rhoa;
    R[s] = r;
  }
}

// The stages' vector sums are done where f and A^T lam are at hand: as vector
// operations of their own they were 184 launches of a gradient through 2 FLD
// super-steps of 4 stages (32^3 particles: 0.41 of 1.74 ms on the device, and
// a host round trip per stage, 3.68 ms in all).
// Each product and each sum is rounded by itself, as vector operations round
// them and a time step per particle still has them.
__device__ __forceinline__ void nl_stage(const NlStage &o, int s, double f) {
#pragma clang fp contract(off)
  if (o.orig) {
    o.out[o.orig[s]] = f;
  } else if (o.first) {
    o.dy0[s] = f;
    o.out[s] = o.y0[s] + o.cf * f;
  } else {
    o.out[s] = o.c1 * o.y1[s] + o.c2 * o.y2[s] + o.c0 * o.y0[s] + o.cf * f + o.cd * o.dy0[s];
  }
}
__device__ __forceinline__ void nl_adj_stage(const NlAdjStage &o, int s, double v) {
#pragma clang fp contract(off)
  if (o.orig) {
    o.out[o.orig[s]] = v;
    return;
  }
  if (o.close) {
    o.lam[s] = o.l0[s] + v;
    return;
  }
  const double l = o.lam[s], below = o.c2 * l;
  double lj = o.c1 * l + o.cf * v, l0 = 0.0, ldy0 = 0.0;
  if (!o.first) {
    lj += o.pend[s];
    l0 = o.l0[s];
    ldy0 = o.ldy0[s];
  }
  if (o.last) l0 += below;
  l0 += o.c0 * l;
  ldy0 += o.cd * l;
  if (o.last) {
    l0 += lj;
    ldy0 += o.c_1 * lj;
  }
  o.lam[s] = lj;
  o.pend[s] = below;
  o.l0[s] = l0;
  o.ldy0[s] = ldy0;
}

// f = A Y for the three operators (OP 3 = 2nw-+, 4 = 2nw+-, 5 = FLD).
template <int DIM, int KT, int OP, int G>
__global__ __launch_bounds__(256) void k_nl_apply(DiffOpArgs a, const double *Y, const double4 *U, const double *D,
                                                  NlStage o) {
  const int t = gtid_a(), s = t / G, sub = t & (G - 1);
  if (s >= a.n || !a.real[s]) return;
  const double4 ps = a.pm[s];
  const double4 qa = a.q0[s];
  const double inv_ha = qa.x, rhoa = qa.y, oma = qa.z;
  double acc = 0.0;
  if constexpr (OP == 5) {
    const double za = Y[s] * rhoa, da = D[s];
    struct Rec { double y, rho, d; };
    auto rec = [&](uint32_t j) { return Rec{Y[j], a.rho[j], D[j]}; };
    over_list<G>(a, s, sub, ps, rec, [&](const Rec &j, double mb, double, double, double, double r2, double ir) {
      acc += mb / j.rho * hess_trace<DIM, KT>(a, r2, ir, inv_ha) * (0.5 * (da + j.d)) * (j.y * j.rho - za);
    });
    group_sum<G>(acc);
    if (sub == 0) nl_stage(o, s, acc / rhoa);
  } else {
    const double4 ua = U[s];
    const double3 ka = kmul(a.K, ua.x, ua.y, ua.z);
    const double odda = 1.0 / (oma * rhoa * rhoa);
    struct Rec { double4 q, u; };
    auto rec = [&](uint32_t j) {
      Rec r{};
      if constexpr (OP == 3) r.q = a.q0[j];
      r.u = U[j];
      return r;
    };
    over_list<G>(a, s, sub, ps, rec, [&](const Rec &j, double mb, double rx, double ry, double rz, double r2, double ir) {
      const double3 kb = kmul(a.K, j.u.x, j.u.y, j.u.z);
      const double wa = nw_coef<DIM, KT>(a, r2, ir, inv_ha);
      if constexpr (OP == 3) {
        const double wb = nw_coef<DIM, KT>(a, r2, ir, j.q.x);
        const double oddb = 1.0 / (j.q.z * j.q.y * j.q.y);
        acc += mb * ((ka.x * rx + ka.y * ry + ka.z * rz) * wa * odda + (kb.x * rx + kb.y * ry + kb.z * rz) * wb * oddb);
      } else {
        acc += mb * ((kb.x - ka.x) * rx + (kb.y - ka.y) * ry + (kb.z - ka.z) * rz) * wa;
      }
    });
    group_sum<G>(acc);
    if (sub == 0) nl_stage(o, s, OP == 3 ? acc : acc * odda);
  }
}

// 2nw adjoint, the vector nu with <lam, A Y> = sum_s (K U_s) . nu_s:
//   2nw-+ : nu_s = (lam_s F_s + m_s sum_{a in R(s)} lam_a nw(r_as, h_s)) / (Om_s rho_s^2)
//   2nw+- : nu_s = m_s sum_{a in R(s)} lam_a nw(r_as, h_a)/(Om_a rho_a^2) - lam_s F_s/(Om_s rho_s^2)
template <int DIM, int KT, int OP, int G>
__global__ __launch_bounds__(256) void k_nl_nu(DiffOpArgs a, const double *lam, const double4 *F, double4 *nu) {
  const int t = gtid_a(), s = t / G, sub = t & (G - 1);
  if (s >= a.n || !a.real[s]) return;
  const double4 ps = a.pm[s];
  const double4 qs = a.q0[s];
  const double odds = 1.0 / (qs.z * qs.y * qs.y);
  double rx_ = 0, ry_ = 0, rz_ = 0;
  struct Rec { double lam; double4 q; };
  auto rec = [&](uint32_t i) {
    Rec r{};
    r.lam = lam[i];
    if constexpr (OP != 3) r.q = a.q0[i];
    return r;
  };
  over_rlist<G>(a, s, sub, ps, rec, [&](const Rec &i, double inv_hi, double rx, double ry, double rz, double r2, double ir) {
    double c;
    if constexpr (OP == 3) c = i.lam * nw_coef<DIM, KT>(a, r2, ir, qs.x);
    else c = i.lam / (i.q.z * i.q.y * i.q.y) * nw_coef<DIM, KT>(a, r2, ir, inv_hi);
    rx_ += c * rx; ry_ += c * ry; rz_ += c * rz;
  });
  group_sum<G>(rx_, ry_, rz_);
  if (sub != 0) return;
  const double4 f = F[s];
  const double ls = lam[s], ms = ps.w;
  if constexpr (OP == 3)
    nu[s] = make_double4((ls * f.x + ms * rx_) * odds, (ls * f.y + ms * ry_) * odds, (ls * f.z + ms * rz_) * odds, 0.0);
  else
    nu[s] = make_double4(ms * rx_ - ls * f.x * odds, ms * ry_ - ls * f.y * odds, ms * rz_ - ls * f.z * odds, 0.0);
}

// mu = K nu, and per block the tensor-gradient partials
// sum_s sym(U_s (x) nu_s)_k for U = UA (slots 0..5) and UB (6..11).
__global__ __launch_bounds__(256) void k_nl_mu(DiffOpArgs a, const double4 *nu, const double4 *UA, const double4 *UB,
                                               double4 *mu, double *gpart) {
  __shared__ double red[4][12];
  int s = gtid_a();
  double g[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (s < a.n && a.real[s]) {
    const double4 v = nu[s];
    const double3 m = kmul(a.K, v.x, v.y, v.z);
    mu[s] = make_double4(m.x, m.y, m.z, 0.0);
    const double4 *Us[2] = {UA, UB};
    for (int w = 0; w < 2; w++) {
      if (!Us[w]) continue;
      const double4 u = Us[w][s];
      double *o = g + 6 * w;
      o[0] = u.x * v.x; o[1] = u.y * v.y; o[2] = u.z * v.z;
      o[3] = u.x * v.y + u.y * v.x; o[4] = u.x * v.z + u.z * v.x; o[5] = u.y * v.z + u.z * v.y;
    }
  }
  for (int c = 0; c < 12; c++) {
    double v = g[c];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][c] = v;
  }
  __syncthreads();
  if (threadIdx.x < 12) {
    double t = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += red[w][threadIdx.x];
    gpart[(size_t)xcd_block_a(blockIdx.x, gridDim.x) * 12 + threadIdx.x] = t;
  }
}

// A^T lam = base + d<mu, G(Y)>/dY (base null: 0):
//   mode 1: rho_s m_s sum_{a in R(s)} mu_a.nw(r_as, h_a)/(rho_a Om_a) - mu_s.F_s/Om_s
//   mode 2: mu_s.F_s/(Om_s rho_s) + m_s/(Om_s rho_s^2) sum_{a in R(s)} rho_a mu_a.nw(r_as, h_s)
template <int DIM, int KT, int MODE, int G>
__global__ __launch_bounds__(256) void k_nl_gT(DiffOpArgs a, const double4 *mu, const double4 *F, const double *base,
                                               NlAdjStage o) {
  const int t = gtid_a(), s = t / G, sub = t & (G - 1);
  if (s >= a.n || !a.real[s]) return;
  const double4 ps = a.pm[s];
  const double4 qs = a.q0[s];
  double acc = 0.0;
  struct Rec { double4 q, m; };
  auto rec = [&](uint32_t i) { return Rec{a.q0[i], mu[i]}; };
  over_rlist<G>(a, s, sub, ps, rec, [&](const Rec &i, double, double rx, double ry, double rz, double r2, double ir) {
    const double dot = i.m.x * rx + i.m.y * ry + i.m.z * rz;
    if constexpr (MODE == 1) acc += dot * nw_coef<DIM, KT>(a, r2, ir, i.q.x) / (i.q.y * i.q.z);
    else acc += i.q.y * dot * nw_coef<DIM, KT>(a, r2, ir, qs.x);
  });
  group_sum<G>(acc);
  if (sub != 0) return;
  const double4 m = mu[s], f = F[s];
  const double mf = m.x * f.x + m.y * f.y + m.z * f.z;
  double v;
  if constexpr (MODE == 1) v = qs.y * ps.w * acc - mf / qs.z;
  else v = mf / (qs.z * qs.y) + ps.w / (qs.z * qs.y * qs.y) * acc;
  nl_adj_stage(o, s, base ? base[s] + v : v);
}

// FLD adjoint at state Y, the part with the conductivity held:
//   out_s = m_s sum_{a in R(s)} (lam_a/rho_a) trH_as (D_a + D_s)/2 - lam_s sum_b (m_b/rho_b) trH_sb (D_s + D_b)/2
// and sD_s = d<lam, f>/dD_s
//   = ((lam_s/rho_s) sum_b (m_b/rho_b) trH_sb (Z_b - Z_s) + (m_s/rho_s) sum_{a in R(s)} (lam_a/rho_a) trH_as (Z_s - Z_a)) / 2
// with Z = Y rho and trH at the list owner's h; then the conductivity's
// dependence on the state: p = sD dD/dR, the direct dR/dY = -R / Y into out and
// v = p dR/dU = p U / (|U| kappa rho^2 Y) (0 where U = 0) for k_nl_gT.
template <int DIM, int KT, int G>
__global__ __launch_bounds__(256) void k_fld_adj(DiffOpArgs a, const double *lam, const double *Y, const double *D,
                                                 const double *dDdR, const double *R, const double4 *U, double *out,
                                                 double4 *v) {
  const int t = gtid_a(), s = t / G, sub = t & (G - 1);
  if (s >= a.n || !a.real[s]) return;
  const double4 ps = a.pm[s];
  const double4 qs = a.q0[s];
  const double ys = Y[s], zs = ys * qs.y, ds = D[s], ls = lam[s];
  double s1 = 0, s2 = 0, s3 = 0, s4 = 0;
  struct Rec { double y, rho, d, lam; };
  auto rec = [&](uint32_t j) { return Rec{Y[j], a.rho[j], D[j], 0.0}; };
  over_list<G>(a, s, sub, ps, rec, [&](const Rec &j, double mb, double, double, double, double r2, double ir) {
    const double w = mb / j.rho * hess_trace<DIM, KT>(a, r2, ir, qs.x);
    s1 += w * (0.5 * (ds + j.d));
    s2 += w * (j.y * j.rho - zs);
  });
  auto rrec = [&](uint32_t i) { return Rec{Y[i], a.rho[i], D[i], lam[i]}; };
  over_rlist<G>(a, s, sub, ps, rrec, [&](const Rec &i, double inv_hi, double, double, double, double r2, double ir) {
    const double w = i.lam / i.rho * hess_trace<DIM, KT>(a, r2, ir, inv_hi);
    s3 += w * (0.5 * (i.d + ds));
    s4 += w * (zs - i.y * i.rho);
  });
  group_sum<G>(s1, s2, s3, s4);
  if (sub != 0) return;
  const double sD = 0.5 * (ls / qs.y * s2 + ps.w / qs.y * s4);
  const double p = sD * dDdR[s];
  const double4 u = U[s];
  const double un = sqrt(u.x * u.x + u.y * u.y + u.z * u.z);
  const double rho = qs.y;
  const double c = un > 0.0 ? p / (un * a.kap[s] * rho * rho * ys) : 0.0;
  v[s] = make_double4(c * u.x, c * u.y, c * u.z, 0.0);
  out[s] = ps.w * s3 - ls * s1 - p * R[s] / ys;
}

#define SPH_INST_NLG(DIM, KT, G)                                                                              \
  template __global__ void k_nl_grad<DIM, KT, 1, G>(DiffOpArgs, const double *, double4 *, double4 *, double *, \
                                                    double *, double *);                                      \
  template __global__ void k_nl_grad<DIM, KT, 2, G>(DiffOpArgs, const double *, double4 *, double4 *, double *, \
                                                    double *, double *);                                      \
  template __global__ void k_nl_apply<DIM, KT, 3, G>(DiffOpArgs, const double *, const double4 *, const double *, \
                                                     NlStage);                              \
  template __global__ void k_nl_apply<DIM, KT, 4, G>(DiffOpArgs, const double *, const double4 *, const double *, \
                                                     NlStage);                              \
  template __global__ void k_nl_apply<DIM, KT, 5, G>(DiffOpArgs, const double *, const double4 *, const double *, \
                                                     NlStage);                              \
  template __global__ void k_nl_nu<DIM, KT, 3, G>(DiffOpArgs, const double *, const double4 *, double4 *);    \
  template __global__ void k_nl_nu<DIM, KT, 4, G>(DiffOpArgs, const double *, const double4 *, double4 *);    \
  template __global__ void k_nl_gT<DIM, KT, 1, G>(DiffOpArgs, const double4 *, const double4 *, const double *, \
                                                  NlAdjStage);                                 \
  template __global__ void k_nl_gT<DIM, KT, 2, G>(DiffOpArgs, const double4 *, const double4 *, const double *, \
                                                  NlAdjStage);                                 \
  template __global__ void k_fld_adj<DIM, KT, G>(DiffOpArgs, const double *, const double *, const double *,  \
                                                 const double *, const double *, const double4 *, double *, double4 *);
#define SPH_INST_NL(DIM, KT) SPH_INST_NLG(DIM, KT, 4) SPH_INST_NLG(DIM, KT, 8)
SPH_INST_NL(1, 0) SPH_INST_NL(1, 1) SPH_INST_NL(1, 2)
SPH_INST_NL(2, 0) SPH_INST_NL(2, 1) SPH_INST_NL(2, 2)
SPH_INST_NL(3, 0) SPH_INST_NL(3, 1) SPH_INST_NL(3, 2)

template __global__ void k_batch_stage<true, double, false>(BatchStage);
template __global__ void k_batch_stage<false, double, false>(BatchStage);
template __global__ void k_batch_stage<true, float, false>(BatchStage);
template __global__ void k_batch_stage<false, float, false>(BatchStage);
template __global__ void k_batch_stage<true, double, true>(BatchStage);
template __global__ void k_batch_stage<false, double, true>(BatchStage);

#define SPH_INST_ADJ(DIM, KT)                                                                  \
  template __global__ void k_diff_weights<DIM, KT>(DiffOpArgs, double *, double *);                 \
  template __global__ void k_diff_rweights<DIM, KT>(DiffOpArgs, const double *, double *);          \
  template __global__ void k_diff_gcontract<DIM, KT>(DiffOpArgs, const double *, const double *, const double *, \
                                                     const double *, double *);
SPH_INST_ADJ(1, 0) SPH_INST_ADJ(1, 1) SPH_INST_ADJ(1, 2)
SPH_INST_ADJ(2, 0) SPH_INST_ADJ(2, 1) SPH_INST_ADJ(2, 2)
SPH_INST_ADJ(3, 0) SPH_INST_ADJ(3, 1) SPH_INST_ADJ(3, 2)

}  // namespace sph
