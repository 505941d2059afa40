// One-sided block-Jacobi SVD of bond matrices of at most 32 columns (one pair of column blocks), the
// whole solve in one launch: one workgroup per task runs every sweep, Gram matrix, inner solve and
// rotation of tebd_jacobi.hip's method, with workgroup barriers where that file's large solve has
// kernel boundaries and with the convergence test on the device.
//
// A solve of this size is a chain of dependent small steps (3 to 12 sweeps of one pair): run as
// separate launches it spent a third of its time in launches, the queue between them and the
// host's wait after every sweep.  Step of a spin chain of 10 sites, chi = 8: 3.7 ms with one launch
// per step of the solve, 2.4 in one launch.  It is taken only where a whole batch has one pair:
//   * two pairs in one workgroup of 1024 threads share a CU, and a round took 2340 cycles there
//     instead of 1345; sweep by sweep they have a CU each.  Step of 30 spins 1 at chi = 20 (60 x 60
//     bonds): 13.4 ms so, 9.5 sweep by sweep; of 40 spins 1/2 at chi = 30: 6.6 and 5.3; of a ring of 13
//     at chi = 24: 16.4 and 15.7;
//   * beside larger bonds the launch is one more step in sequence, while the rounds of one more task
//     cost nothing: the same chains 8.7, 4.5 and 14.4 ms with all bonds sweep by sweep.
//
// The schedule is read from L2 one round ahead: its 34 KB in LDS left a CU one workgroup instead of two
// (step of 1024 chains of 10 spins, chi = 8: 13.6 ms, 11.2).
//
// Every number is formed by the same operations in the same order as sweep by sweep with
// BondTask::cyclic, so the results do not depend on the choice.
#include "tebd_device.h"
#include "tebd_jacobi_inner.h"
#include "tebd_kernels.h"

// Products and sums are fused where fma() is written and nowhere else, so that every number
// is rounded the same way whatever the compiler sees around it.
#pragma clang fp contract(off)

namespace {

// 16 rows of M's pair columns, from r0, times Q: (X Q)^T = Q^T X^T on the matrix cores.
__device__ __forceinline__ void rotate_rows(const zc (*Q)[JC + 1], zc* M, int rows, int ld, int r0, int bi, int bj,
                                            int lane) {
  const int lr = lane & 15, lk = lane >> 4;
  auto col_of = [&](int c) { return c < JB ? bi * JB + c : bj * JB + (c - JB); };
  const int r = r0 + lr;
  const bool in = r < rows;
  zc x[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) x[ks] = in ? M[(size_t)ld * col_of(4 * ks + lk) + r] : zmk(0.0, 0.0);
#pragma unroll 1
  for (int ct = 0; ct < 2; ++ct) {  // one half of the columns at a time keeps the registers below the spill limit
    d4 ore = d4{0.0, 0.0, 0.0, 0.0}, oim = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const zc q = Q[4 * ks + lk][16 * ct + lr];
      ore = mfma4(q.x, x[ks].x, ore);
      ore = mfma4(-q.y, x[ks].y, ore);
      oim = mfma4(q.x, x[ks].y, oim);
      oim = mfma4(q.y, x[ks].x, oim);
    }
    if (in) {
#pragma unroll
      for (int g = 0; g < 4; ++g) M[(size_t)ld * col_of(16 * ct + lk + 4 * g) + r] = zmk(ore[g], oim[g]);
    }
  }
}

// The whole SVD of every task; every task of the batch has one pair of column blocks.  W and V (global
// memory, tens of KB, in L2) are rotated in place.  counter[2] = sweeps run, counter[3] = those that
// rotated: all of them if the solve has not converged within max_sweeps.
__global__ __launch_bounds__(kPairThreads) void k_jacobi_small(const BondTask* __restrict__ tasks, double tol_rel,
                                                               double tol_abs, int max_sweeps) {
  const BondTask& t = tasks[blockIdx.x];
  __shared__ PairLds L;
  const int tid = threadIdx.x;
  zc* const W = t.W;
  zc* const V = t.V;
  const int R = t.R, NV = V ? t.NV : 0;
  const zc* Wi = W;
  const zc* Wj = W + (size_t)R * JB;
  const double floor = tol_abs * sqrt(t.result[2]);  // of the largest column norm
  int sweep = 0;
  bool done = false;
#pragma unroll 1
  for (;;) {
    // opaque per sweep: index arithmetic derived from it is done where it is used instead of
    // being held in registers across the whole solve (which spilled them)
    int pt = tid;
    asm volatile("" : "+v"(pt));
    const int lane = pt & 63, wave = pt >> 6;
    __syncthreads();
    if (pt == 0) L.need = 0;
    d4 gre, gim;
    double nx, ny;
    gram_block(Wi, Wj, R, wave, lane, gre, gim, nx, ny);
    reduce_block(L, gre, gim, pt, 0, JB, false);
    gram_block(Wi, Wi, R, wave, lane, gre, gim, nx, ny);
    reduce_block(L, gre, gim, pt, 0, 0, true);
    gram_block(Wj, Wj, R, wave, lane, gre, gim, nx, ny);
    reduce_block(L, gre, gim, pt, JB, JB, true);
    // does the pair need a rotation?  |A_pq| > tol_rel sqrt(A_pp A_qq) and |A_pq| > tol_abs
    // max_c|w_c| (|w_p| + |w_q|): the second bound is the rounding floor of the rotations
    int need = 0;
    for (int e = pt; e < JC * JC; e += kPairThreads) {
      const int pp = e % JC, qq = e / JC;
      if (pp >= qq) continue;
      const double g2 = abs2(L.A[pp][qq]);
      const double app = fmax(L.dg[pp], 0.0), aqq = fmax(L.dg[qq], 0.0);
      const double fl = floor * (sqrt(app) + sqrt(aqq));
      if (g2 > tol_rel * tol_rel * app * aqq && g2 > fl * fl) need = 1;
    }
    if (need) L.need = 1;
    __syncthreads();
    ++sweep;
    done = !L.need;
    if (done) break;
    inner_solve(L, kRing.rounds, pt);
    asm volatile("" : "+v"(pt));
    {
      const int lane = pt & 63, wave = pt >> 6;
#pragma unroll 1
      for (int r0 = 16 * wave; r0 < R; r0 += 16 * kPairWaves) rotate_rows(L.Q, W, R, R, r0, 0, 1, lane);
#pragma unroll 1
      for (int r0 = 16 * wave; r0 < NV; r0 += 16 * kPairWaves) rotate_rows(L.Q, V, NV, NV, r0, 0, 1, lane);
    }
    if (sweep == max_sweeps) break;
  }
  if (tid == 0) {
    t.counter[2] = sweep;
    t.counter[3] = done ? sweep - 1 : sweep;
  }
}

}  // namespace

hipError_t launch_jacobi_small(const BondTask* d_tasks, int ntasks, double tol_rel, double tol_abs, int max_sweeps,
                               hipStream_t st) {
  hipLaunchKernelGGL(k_jacobi_small, dim3(ntasks), dim3(kPairThreads), 0, st, d_tasks, tol_rel, tol_abs, max_sweeps);
  return hipGetLastError();
}
