// Kernels of the all-pairs two-site reduced density matrices (TwoSiteExpVal and
// EvaluateMeasures, observables_module.f90:836-883,2286-2526, built from ThetaKernal,
// ThetaNext and TwoSiteRho, :704-832).  The host (tebd_capi.cpp) carries, for every right
// site l2, the environment Theta(a, i, j, b) of l2 with the sites between absorbed, and
// steps all of them over one left site l1 at a time with batched GEMMs; these kernels do
// the parts that are not GEMMs, for all right sites (k_cr_kernal, k_rho1_trace,
// k_rho_reduce) or all chains (k_cr_left) in one launch.
//
// One right site at a time, a table was a sequence of ten short launches per pair of sites:
// 27.8 ms for 276 pairs of a Fermi-Hubbard chain of 24 sites at chi = 64, whose products take
// 1.5 ms at the GEMM's rate; stepped together, 3.8 ms (k_rho_reduce 47 us for 23 pairs).
#include "tebd_device.h"
#include "tebd_kernels.h"

namespace {

// ThetaKernal's two factors (observables_module.f90:704-730) of a right site: the ket factor
// K((a, i), e) = lambda_l(a) G(a, i, e) lambda_r(e), a (chi_l d) x chi_r matrix, and the bra factor
// as a chi_r x (d chi_l) matrix with columns j + d b: B(e, j + d b) = conj(G(b, j, e)) lambda_l(b)
// lambda_r(e); Theta = K B has Theta(a, i, j, b) at a + chi_l (i + d (j + d b)).
__global__ void k_cr_kernal(const CrRight* __restrict__ sites) {
  const CrRight t = sites[blockIdx.y];
  const int m = t.chil * t.d;
  const size_t n = (size_t)m * t.chir;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const int row = (int)(e % m), eta = (int)(e / m);
    const int a = row % t.chil, i = row / t.chil;
    const zc g = t.G[e];
    const double w = t.ll[a] * t.lr[eta];
    t.K[e] = zmk(g.x * w, g.y * w);
    t.B[eta + (size_t)t.chir * (i + (size_t)t.d * a)] = zmk(g.x * w, -g.y * w);
  }
}

// The factors of a left site: A((a, i), b) = lambda(a) phase(i) G(a, i, b) (phase null: 1) for the
// ket, and the bra's conjugate transpose Gbar(b, a + chi_a l) = conj(G(a, l, b)) lambda(a).
__global__ void k_cr_left(const CrLeft* __restrict__ sites) {
  const CrLeft t = sites[blockIdx.y];
  const int m = t.chia * t.d;
  const size_t n = (size_t)m * t.chib;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const int row = (int)(e % m), b = (int)(e / m);
    const zc g = t.G[e];
    const double w = t.lam[row % t.chia], p = t.phase ? w * t.phase[row / t.chia] : w;
    t.A[e] = zmk(g.x * p, g.y * p);
    t.Gbar[b + (size_t)t.chib * row] = zmk(g.x * w, -g.y * w);
  }
}

// TwoSiteRho's final contraction (observables_module.f90:815-826):
//   rho[(i d + j) + d^2 (l d + k)] = sum_{a < chi_a, b < chi_b} A(a, i, b) T(b, j, k; a + chi_a l)
// A: the left site's scaled ket Gamma; T: (chi_b d^2) x (chi_a d), element b + chi_b (j + d k) +
// chi_b d^2 (a + chi_a l) (the environment with the left site's bra Gamma absorbed).  One
// workgroup per (j, k, l) and pair forms the d entries i from one pass over its part of T, the
// bulk of the bytes: lanes run over b, where T is contiguous, and each wave takes a range of a.
template <int D>
__global__ __launch_bounds__(256) void k_rho_reduce(const CrPair* __restrict__ pairs) {
  const CrPair t = pairs[blockIdx.y];
  const int jk = blockIdx.x % (D * D), l = blockIdx.x / (D * D);
  const int j = jk % D, k = jk / D;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int chi_a = t.chia, chi_b = t.chib;
  const int part = (chi_a + 3) / 4, a0 = wave * part, a1 = min(chi_a, a0 + part);
  const zc* T = t.T + (size_t)chi_b * jk + (size_t)chi_b * D * D * ((size_t)chi_a * l);
  double re[D], im[D];
#pragma unroll
  for (int i = 0; i < D; ++i) re[i] = im[i] = 0.0;
  for (int b = lane; b < chi_b; b += 64) {
    const zc* A = t.A + (size_t)chi_a * D * b;
    for (int a = a0; a < a1; ++a) {
      const zc x = T[b + (size_t)chi_b * D * D * a];
#pragma unroll
      for (int i = 0; i < D; ++i) {
        const zc g = A[a + (size_t)chi_a * i];
        re[i] += g.x * x.x - g.y * x.y;
        im[i] += g.x * x.y + g.y * x.x;
      }
    }
  }
  __shared__ double red[4][2 * D];
#pragma unroll
  for (int i = 0; i < D; ++i) {
    const double sr = wave_sum(re[i]), si = wave_sum(im[i]);
    if (lane == 0) {
      red[wave][2 * i] = sr;
      red[wave][2 * i + 1] = si;
    }
  }
  __syncthreads();
  if (threadIdx.x < D) {
    const int i = threadIdx.x;
    double sr = 0.0, si = 0.0;
    for (int w = 0; w < 4; ++w) {
      sr += red[w][2 * i];
      si += red[w][2 * i + 1];
    }
    t.rho[(i * D + j) + D * D * (l * D + k)] = zmk(sr, si);
  }
}

// The one-site density matrix as the trace of ThetaKernal over its bond index
// (FormSingleSiteRho, observables_module.f90:95-117): rho[i + d j] = sum_a Theta(a, i, j, a),
// Theta element a + chi (i + d (j + d b)).
__global__ __launch_bounds__(256) void k_rho1_trace(const CrRight* __restrict__ sites) {
  const CrRight t = sites[blockIdx.y];
  const int d = t.d, chi = t.chil, i = blockIdx.x % d, j = blockIdx.x / d;
  double re = 0.0, im = 0.0;
  for (int a = threadIdx.x; a < chi; a += 256) {
    const zc x = t.theta[a + (size_t)chi * (i + (size_t)d * (j + (size_t)d * a))];
    re += x.x;
    im += x.y;
  }
  __shared__ double red[4][2];
  re = wave_sum(re);
  im = wave_sum(im);
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6][0] = re;
    red[threadIdx.x >> 6][1] = im;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    t.rho1[blockIdx.x] = zmk(red[0][0] + red[1][0] + red[2][0] + red[3][0], red[0][1] + red[1][1] + red[2][1] + red[3][1]);
}

int blocks_for(size_t n) {
  const size_t b = (n + 255) / 256;
  return (int)(b < 1 ? 1 : (b < 1024 ? b : 1024));
}

}  // namespace

hipError_t launch_cr_kernal(const CrRight* d_sites, int n, size_t max_elems, hipStream_t st) {
  hipLaunchKernelGGL(k_cr_kernal, dim3(blocks_for(max_elems), n), dim3(256), 0, st, d_sites);
  return hipGetLastError();
}

hipError_t launch_cr_left(const CrLeft* d_sites, int n, size_t max_elems, hipStream_t st) {
  hipLaunchKernelGGL(k_cr_left, dim3(blocks_for(max_elems), n), dim3(256), 0, st, d_sites);
  return hipGetLastError();
}

hipError_t launch_rho_reduce(const CrPair* d_pairs, int n, int d, hipStream_t st) {
  const dim3 grid(d * d * d, n);
  switch (d) {
    case 2: hipLaunchKernelGGL(k_rho_reduce<2>, grid, dim3(256), 0, st, d_pairs); break;
    case 3: hipLaunchKernelGGL(k_rho_reduce<3>, grid, dim3(256), 0, st, d_pairs); break;
    case 4: hipLaunchKernelGGL(k_rho_reduce<4>, grid, dim3(256), 0, st, d_pairs); break;
    case 5: hipLaunchKernelGGL(k_rho_reduce<5>, grid, dim3(256), 0, st, d_pairs); break;
    case 6: hipLaunchKernelGGL(k_rho_reduce<6>, grid, dim3(256), 0, st, d_pairs); break;
    case 8: hipLaunchKernelGGL(k_rho_reduce<8>, grid, dim3(256), 0, st, d_pairs); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_rho1_trace(const CrRight* d_sites, int n, int d, hipStream_t st) {
  hipLaunchKernelGGL(k_rho1_trace, dim3(d * d, n), dim3(256), 0, st, d_sites);
  return hipGetLastError();
}
