// One-sided block-Jacobi SVD of bond matrices of at most 64 columns, the whole solve in one
// launch: one workgroup per task runs every sweep, round, Gram matrix, inner solve and
// rotation of tebd_jacobi.hip's method, with workgroup barriers where that file's large solve
// has kernel boundaries and with the convergence test on the device.
//
// A solve of this size is a chain of dependent small steps (P = 1 or 2 pairs of 16-column
// blocks, 1 or 3 rounds per sweep, 3 to 12 sweeps): run as separate launches it spent a third
// of its time in launches, the queue between them and the host's wait after every sweep.
// Step of a spin chain of 10 sites, chi = 8: 3.9 ms with one launch per step of the solve, 2.9
// in one launch; of a ring of 13 sites, chi = 24: 21.2 and 17.2; imaginary-time step and
// canonical form of 8 chains of 16 sites, chi = 24: 37.2 and 27.6.
//
// Every number is formed by the same operations in the same order as in the launch-per-step
// form, and each pair is still solved by up to three cyclic inner sweeps: bonds this small
// are not preconditioned by the pivoted QR, and their smallest Schmidt vectors (which the
// Vidal form divides by lambda ~ 1e-14) keep the accuracy they had.
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

// The whole SVD of every task with P == NP and no QR preconditioning: NP x 512 threads, one
// pair of column blocks per 512.  W and V (global memory, a few hundred KB at most, in L2) are
// rotated in place.  cnt[4] = sweeps run (0: not converged within max_sweeps), cnt[8 + s] =
// pairs rotated in sweep s (the last of kSweepBins entries: that sweep and later ones).
template <int NP>
__global__ __launch_bounds__(NP * kPairThreads) void k_jacobi_small(const BondTask* __restrict__ tasks, double tol_rel,
                                                                    double tol_abs, int max_sweeps) {
  const BondTask& t = tasks[blockIdx.x];
  if (!t.small || t.P != NP) return;
  __shared__ PairLds lds[NP];
  __shared__ InnerRounds<kAllRounds, 2 * kInnerPairs> table;
  __shared__ unsigned ver[2 * NP];
  __shared__ unsigned long long seen[2 * NP][2 * NP];
  __shared__ int s_rot, s_hist[kSweepBins], s_visits;
  const int tid = threadIdx.x, mine = tid / kPairThreads, pair_tid = tid % kPairThreads;
  PairLds& L = lds[mine];
  zc* const W = t.W;
  zc* const V = t.V;
  const int R = t.R, NV = V ? t.NV : 0;
  load_rounds(table, kRing.rounds, tid, NP * kPairThreads);
  if (tid < 2 * NP) ver[tid] = 0u;
  if (tid < 4 * NP * NP) seen[tid / (2 * NP)][tid % (2 * NP)] = ~0ull;
  if (tid < kSweepBins) s_hist[tid] = 0;
  if (tid == 0) s_visits = 0;
  const double fnorm = sqrt(t.result[2]);  // largest column norm
  int sweeps = 0;
#pragma unroll 1
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    if (tid == 0) s_rot = 0;
#pragma unroll 1
    for (int round = 0; round < 2 * NP - 1; ++round) {
      const bool full = round == 0;
      // opaque per round: index arithmetic derived from it is done where it is used instead of
      // being held in registers across the whole solve (which spilled them)
      int pt = pair_tid;
      asm volatile("" : "+v"(pt));
      const int lane = pt & 63, wave = pt >> 6;
      int bi, bj;
      rr_pair(2 * NP, round, mine, bi, bj);
      const int lo = bi < bj ? bi : bj, hi = bi < bj ? bj : bi;
      __syncthreads();
      const unsigned long long stamp = ((unsigned long long)ver[lo] << 32) | ver[hi];
      const bool on = full || seen[lo][hi] != stamp;  // else unchanged since it was found orthogonal
      if (pt == 0) L.need = 0;
      const zc* Wi = W + (size_t)R * (bi * JB);
      const zc* Wj = W + (size_t)R * (bj * JB);
      d4 gre{}, gim{};
      double nx = 0.0, ny = 0.0;
      if (on) gram_block(Wi, Wj, R, wave, lane, gre, gim, nx, ny);
      if (on && !full) {
        nx += __shfl_xor(nx, 16, 64);
        nx += __shfl_xor(nx, 32, 64);
        ny += __shfl_xor(ny, 16, 64);
        ny += __shfl_xor(ny, 32, 64);
        if (lane < 16) {
          L.g.nred[wave][0][lane] = nx;
          L.g.nred[wave][1][lane] = ny;
        }
        // within-block entries: zero (the blocks' columns are orthogonal)
        const int blk = pt / (JB * JB), r = (pt / JB) % JB, c = pt % JB;
        L.A[blk * JB + r][blk * JB + c] = zmk(0.0, 0.0);
      }
      reduce_block(L, on, gre, gim, pt, 0, JB, false);
      if (full) {
        gram_block(Wi, Wi, R, wave, lane, gre, gim, nx, ny);
        reduce_block(L, on, gre, gim, pt, 0, 0, true);
        gram_block(Wj, Wj, R, wave, lane, gre, gim, nx, ny);
        reduce_block(L, on, gre, gim, pt, JB, JB, true);
      } else {
        if (on && pt < JC) {
          const int side = pt / JB, col = pt % JB;
          double v = 0.0;
          for (int w = 0; w < kPairWaves; ++w) v += L.g.nred[w][side][col];
          L.dg[pt] = v;
        }
        __syncthreads();
      }
      // does the pair need a rotation?  |A_pq| > tol_rel sqrt(A_pp A_qq) and |A_pq| > tol_abs
      // max_c|w_c| (|w_p| + |w_q|): the second bound is the rounding floor of the rotations
      if (on) {
        int need = 0;
        for (int e = pt; e < JC * JC; e += kPairThreads) {
          const int pp = e % JC, qq = e / JC;
          if (pp >= qq) continue;
          const double g2 = abs2(L.A[pp][qq]);
          const double app = fmax(L.dg[pp], 0.0), aqq = fmax(L.dg[qq], 0.0);
          const double fl = tol_abs * fnorm * (sqrt(app) + sqrt(aqq));
          if (g2 > tol_rel * tol_rel * app * aqq && g2 > fl * fl) need = 1;
        }
        if (need) L.need = 1;
      }
      __syncthreads();
      const bool rot = on && L.need;
      if (pt == 0 && on) {
        atomicAdd(&s_visits, 1);
        if (rot) {
          atomicAdd(&s_rot, 1);
          atomicAdd(&s_hist[sweep < kSweepBins ? sweep : kSweepBins - 1], 1);
          ver[lo] += 1;
          ver[hi] += 1;
        } else {
          seen[lo][hi] = stamp;
        }
      }
      bool any = rot;
#pragma unroll
      for (int k = 0; k < NP; ++k) any = any || lds[k].need;  // uniform over the workgroup
      if (!any) continue;
      inner_solve<false>(L, table, pt, rot);
      asm volatile("" : "+v"(pt));
      if (rot) {
        const int lane = pt & 63, wave = pt >> 6;
#pragma unroll 1
        for (int r0 = 16 * wave; r0 < R; r0 += 16 * kPairWaves) rotate_rows(L.Q, W, R, R, r0, bi, bj, lane);
#pragma unroll 1
        for (int r0 = 16 * wave; r0 < NV; r0 += 16 * kPairWaves) rotate_rows(L.Q, V, NV, NV, r0, bi, bj, lane);
      }
    }
    __syncthreads();
    ++sweeps;
    const bool done = s_rot == 0;
    __syncthreads();
    if (done) {
      if (tid == 0) t.counter[4] = sweeps;
      break;
    }
    if (sweep + 1 == max_sweeps && tid == 0) t.counter[4] = 0;
  }
  if (tid < kSweepBins) t.counter[8 + tid] = s_hist[tid];
  if (tid == 0) {
    int rots = 0;
    for (int s = 0; s < kSweepBins; ++s) rots += s_hist[s];
    t.counter[2] = s_visits;
    t.counter[3] = rots;
  }
}

}  // namespace

hipError_t launch_jacobi_small(const BondTask* d_tasks, int ntasks, bool one_pair, bool two_pairs, double tol_rel,
                               double tol_abs, int max_sweeps, hipStream_t st) {
  if (one_pair) {
    hipLaunchKernelGGL(k_jacobi_small<1>, dim3(ntasks), dim3(kPairThreads), 0, st, d_tasks, tol_rel, tol_abs, max_sweeps);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (two_pairs) {
    hipLaunchKernelGGL(k_jacobi_small<2>, dim3(ntasks), dim3(2 * kPairThreads), 0, st, d_tasks, tol_rel, tol_abs,
                       max_sweeps);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}
