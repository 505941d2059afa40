// One-sided block-Jacobi SVD of the bond matrix (replaces ZGESVD in SVDTruncation,
// local_operations_module.f90:322-345).
//
// W (R x Cpad, column-major) is orthogonalised in place and V accumulates the right
// rotations.  The columns form 2P blocks of JB; a round pairs every block with one
// other (round-robin "circle" order, 2P-1 rounds per sweep).  A round is two kernels:
//   k_jacobi_round   one workgroup per pair: the pair's Gram matrix on FP64 MFMA
//                    (v_mfma_f64_16x16x4f64), the decision whether it needs a
//                    rotation, and rotations over its index pairs in LDS -> Q (32x32, to
//                    global memory): one pass (inner_jacobi) or the whole 32x32 problem by
//                    cyclic sweeps (inner_solve, tebd_jacobi_inner.h); rotated pairs are
//                    queued;
//   k_jacobi_rotate  [W; V](:, pair) <- [W; V](:, pair) Q for every queued pair, on
//                    MFMA, spread over 64-row slabs so a rotation costs one memory
//                    round trip of the whole GPU instead of one workgroup's stream.
// Only the first round of a sweep forms the full Gram of each pair and rotates the pairs
// within the blocks too; the other rounds form the 16x16 cross block and the 32 column norms
// (4x less Gram work), take the columns of a block as orthogonal and, where a visit is one
// pass, rotate the cross pairs once.  With a strongly graded spectrum the rounding of rotations
// lets the small columns of a block drift away from orthogonality, and the first round restores
// it (a cross-only iteration does not converge there).
//
// A pair visit is bound by the latency of its rounds of rotations: three cyclic sweeps over
// all index pairs per visit (93 rounds, two barriers each) took 59 us at 400 x 400
// (Fermi-Hubbard, chi = 100) and 54 at 225 x 225 (Bose-Hubbard, chi = 45); one pass over the
// cross pairs (16 rounds of one barrier) takes 16 and 14, for 6 to 7 outer sweeps instead of 5
// to 6.  Whole cyclic sweeps per visit stay for tasks that say so (BondTask::cyclic):
//   * CanonicalForm's matrices are not preconditioned: with a generic basis and singular values
//     over 13 decades one pass per visit does not converge within 40 sweeps at 192 columns
//     (cyclic: 36).
//   * the number blocks' Schmidt values are cut at 1e-10, where another rounding keeps another
//     state: with one pass a Fermi-Hubbard chain of 64 sites, chi = 128, gave lambda up to 8e-9 from
//     what cyclic sweeps give (its step takes 14.5 ms so and 19.6 with them).
// They also stay for bonds of more than kCyclicRows rows, see there.
//
// Work that cannot change the result is skipped exactly:
//   * a task whose previous sweep rotated nothing has converged: its workgroups exit;
//   * a pair whose two blocks have not been rotated since the pair was last found
//     orthogonal would produce the same Gram and the same decision: it is skipped.
// Per task, counter[0..1] count rotated pairs of the current / previous sweep (by
// sweep parity), counter[2] pairs whose Gram was formed and counter[3] rotated pairs
// over the whole SVD; blkver[b] counts rotations of block b and pairseen[lo*2P+hi]
// holds (blkver[lo], blkver[hi]) from the last time that pair was verified.
#include "tebd_device.h"
#include "tebd_jacobi_inner.h"
#include "tebd_kernels.h"

namespace {

// k_jacobi_round runs 8 waves: all of them form the Gram matrix; in the inner solve
// waves 0-3 update A and waves 4-7 the rotation accumulator Q.
constexpr int kRoundThreads = kPairThreads;
static_assert(kRoundThreads == 512 && JB == kInnerPairs, "the inner solve's thread roles");

// Index pair t (t < 16) of round r of level h (h = 1, 2, 4, 8 or 16): the 32 indices in
// groups of 2h, the lower half of a group against its upper half shifted by r.  Level 16
// pairs the two column blocks with each other; levels 8, 4, 2 and 1 pair each block within
// itself.  Over rounds 0 .. h-1 of every level each index pair meets exactly once.
__host__ __device__ constexpr int level_p(int h, int t) { return 2 * t - (t & (h - 1)); }
__host__ __device__ constexpr int level_q(int h, int r, int t) {
  return level_p(h, t) - (t & (h - 1)) + h + (((t & (h - 1)) + r) & (h - 1));
}

// Bonds of more rows solve each visited pair by cyclic sweeps: their Grams and rotations of W cost
// more than the rounds, which run side by side once a batch fills the GPU, so fewer outer sweeps
// pay.  Hubbard, exact SVDs, ms per step with one pass per visit and with cyclic sweeps, chains of
// 24 and of 96 sites: 560 rows 51 and 56, 111 and 98; 720 rows 75 and 84, 211 and 176; 800 rows 77
// and 82, 264 and 211; 912 rows 124 and 130, 452 and 341; 1024 rows 163 and 165, 673 and 537; 128
// sites, 1024 rows 235 and 186.  Below the bound, 64 sites of 512 rows 55 and 59, 24 sites of 400
// rows 26 and 32.  The bound looks at the bond alone, so that no result depends on the batch.
constexpr int kCyclicRows = 512;

// The schedules: kCross the 16 rounds of level 16 (pair t's next entry lies in block (t, t + 1),
// the last one's in block (0, 15)), kFull the 15 rounds of levels 8, 4, 2, 1 and then kCross.
constexpr int kWithinRounds = JB - 1;
using CrossTable = InnerTable<JB, 2 * kInnerPairs>;
using FullTable = InnerTable<kAllRounds, 2 * kOffBlocks>;
template <class Table>
constexpr Table level_table(int first_level) {
  Table t{};
  int rd = 0;
  for (int lv = 0; lv < 5; ++lv) {
    const int h = lv < 4 ? 8 >> lv : 16;
    if (lv < first_level) continue;
    for (int r = 0; r < h; ++r, ++rd)
      for (int x = 0; x < kInnerPairs; ++x) {
        t.p[rd][x] = (unsigned char)level_p(h, x);
        t.q[rd][x] = (unsigned char)level_q(h, r, x);
      }
  }
  int br[16] = {}, bk[16] = {};
  for (int x = 0; x < 16; ++x) {
    br[x] = x < 15 ? x : 0;
    bk[x] = x < 15 ? x + 1 : 15;
  }
  return complete_table(t, br, bk);
}
__device__ constexpr CrossTable kCross = level_table<CrossTable>(4);
__device__ constexpr FullTable kFull = level_table<FullTable>(0);

// Eigenvector rotations of a pair's Gram matrix A into Q.  A pair is visited once per outer
// sweep, so its eigenproblem need not be finished: the 256 index pairs across the two
// blocks are rotated once (16 rounds); in the first round of a sweep (FULL), whose Gram
// includes the blocks' own couplings, the pairs within the blocks too, in two passes.
// Measured on Hubbard and Bose-Hubbard bonds (numpy restatement, 225 x 225 and 256 x 256):
// 6 outer sweeps and 1300-1400 inner rounds in sequence per solve; three cyclic sweeps over
// all 496 pairs per visit take 5 outer sweeps but 4400-4650 rounds in sequence.
// Waves 0..3 update A; waves 4..7 apply the rotations to Q: in level 16 from registers (lane t
// of a 16-lane row has two rows' entries at p_t, which stays, and q_t, which comes from the next
// lane in every round), in the other levels in LDS.
template <bool FULL, class Rounds>
__device__ __forceinline__ void inner_jacobi(PairLds& L, const Rounds& T, int tid) {
  zc (*A)[kInnerLd] = L.A;
  zc (*Q)[JC + 1] = L.Q;
  double* dg = L.dg;
  RotBuf* rb = L.rb;
  constexpr int NN = FULL ? 2 * kOffBlocks : 2 * kInnerPairs, RW = FULL ? kWithinRounds : 0;
  const bool is_a = tid < 2 * kOffBlocks, is_q = tid >= 256;
  const int tr = is_a ? kCross.tr[tid] : 0, tk = is_a ? kCross.tk[tid] : 0, half = tid & 1;
  const int qt = tid & 15, qk = (tid >> 4) & 15;
  if (FULL) {
    for (int e = tid; e < JC * JC; e += kRoundThreads) Q[e / JC][e % JC] = zmk(e / JC == e % JC ? 1.0 : 0.0, 0.0);
    __syncthreads();
  }
  zc f[2], s[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    f[u] = zmk(qk + 16 * u == qt ? 1.0 : 0.0, 0.0);
    s[u] = zmk(qk + 16 * u == qt + 16 ? 1.0 : 0.0, 0.0);
  }
  int buf = 0;
#pragma unroll 1
  for (int pass = 0; pass < (FULL ? 2 : 1); ++pass) {
    if (tid < kInnerPairs) {
      const int p = level_p(FULL ? 8 : 16, tid), q = level_q(FULL ? 8 : 16, 0, tid);
      A[p][q] = make_rotation(rb[buf], dg[p], dg[q], &dg[p], &dg[q], nullptr, tid, A[p][q], jrot);
    }
    __syncthreads();
    if (FULL) {
      int rd = 0;
      unsigned entry = is_a ? T.entry[0][tid] : 0u, next = tid < NN ? T.next[0][tid] : 0u;
#pragma unroll 1
      for (int h = 8; h >= 1; h >>= 1)
#pragma unroll 1
        for (int r = 0; r < h; ++r, ++rd, buf ^= 1) {
          const RotBuf& R = rb[buf];
          if (is_a) {
            const unsigned e1 = T.entry[rd + 1][tid], n1 = T.next[rd + 1][tid];
            update_block(&A[0][0], dg, R, rb[buf ^ 1], nullptr, entry, next, tr, tk, half, jrot);
            entry = e1;
            next = n1;
          } else if (is_q) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              const zc sw = R.sw[qt];
              const double c = R.c[qt];
              const int k = qk + 16 * u, p = level_p(h, qt), q = level_q(h, r, qt);
              const zc xp = Q[k][p], xq = Q[k][q];
              Q[k][p] = zsub(zscale(xp, c), zmul(zconj(sw), xq));
              Q[k][q] = zadd(zmul(sw, xp), zscale(xq, c));
            }
          }
          __syncthreads();
        }
      if (is_q) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          f[u] = Q[qk + 16 * u][qt];
          s[u] = Q[qk + 16 * u][qt + 16];
        }
      }
    }
    unsigned entry = is_a ? T.entry[RW][tid] : 0u, next = tid < NN ? T.next[RW][tid] : 0u;
#pragma unroll 1
    for (int r = 0; r < JB; ++r, buf ^= 1) {
      const RotBuf& R = rb[buf];
      if (is_a) {
        const int ahead = RW + (r + 1 < JB ? r + 1 : 0);  // read now, used after the barrier
        unsigned e1, n1 = 0u;
        if (FULL) {
          e1 = T.entry[ahead][tid];
          n1 = T.next[ahead][tid];
        }
        update_block(&A[0][0], dg, R, rb[buf ^ 1], nullptr, entry, next, tr, tk, half, jrot);
        if (!FULL) {
          e1 = T.entry[ahead][tid];
          if (tid < NN) n1 = T.next[ahead][tid];
        }
        entry = e1;
        next = n1;
      } else if (is_q) {
        const double c = R.c[qt];
        const zc sw = R.sw[qt];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          // Q_:p <- c Q_:p - s conj(w) Q_:q ; Q_:q <- s w Q_:p + c Q_:q
          const zc xp = f[u], xq = s[u];
          f[u] = zsub(zscale(xp, c), zmul(zconj(sw), xq));
          const zc nq = zadd(zmul(sw, xp), zscale(xq, c));
          s[u] = zdpp<kDppRotate>(nq);
        }
      }
      __syncthreads();
    }
    if (is_q) {  // after 16 rounds every q is back at its lane
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        Q[qk + 16 * u][qt] = f[u];
        Q[qk + 16 * u][qt + 16] = s[u];
      }
    }
    __syncthreads();
  }
}

template <bool FULL>
__global__ __launch_bounds__(kRoundThreads) void k_jacobi_round(const BondTask* __restrict__ tasks, int sweep, int round,
                                                      double tol_rel, double tol_abs, double tol_pass,
                                                      int* __restrict__ wl_count, int2* __restrict__ wl_items, int wl_cap) {
  const BondTask t = tasks[blockIdx.y];
  const int p = blockIdx.x;
  if (p >= t.P || round >= 2 * t.P - 1) return;
  int* cnt = t.counter;
  if (sweep > 0 && cnt[(sweep - 1) & 1] == 0) return;  // converged in the previous sweep
  const int nblk = 2 * t.P;
  int bi, bj;
  rr_pair(nblk, round, p, bi, bj);
  const int lo = bi < bj ? bi : bj, hi = bi < bj ? bj : bi;
  const unsigned vlo = t.blkver[lo], vhi = t.blkver[hi];
  const unsigned long long stamp = ((unsigned long long)vlo << 32) | vhi;
  unsigned long long* seen = t.pairseen + (size_t)lo * nblk + hi;
  if (!FULL && *seen == stamp) return;  // unchanged since it was verified orthogonal

  // The schedules are read from L2 one round ahead: that of 16 rounds in LDS gave no time and its 17
  // KB kept the other lanes' kernels off the CU (96 sites, 1024 rows: 559 ms a step with it, 537).
  __shared__ PairLds L;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const zc* Wi = t.W + (size_t)t.R * (bi * JB);
  const zc* Wj = t.W + (size_t)t.R * (bj * JB);
  if (tid == 0) L.need = 0;
  const bool cyclic = t.cyclic || t.R > kCyclicRows;

  // ---- Gram: A = [Wi Wj]^H [Wi Wj]
  {
    d4 gre, gim;
    double nx, ny;
    gram_block(Wi, Wj, t.R, wave, lane, gre, gim, nx, ny);
    if (!FULL) {
      nx += __shfl_xor(nx, 16, 64);
      nx += __shfl_xor(nx, 32, 64);
      ny += __shfl_xor(ny, 16, 64);
      ny += __shfl_xor(ny, 32, 64);
      if (lane < 16) {
        L.g.nred[wave][0][lane] = nx;
        L.g.nred[wave][1][lane] = ny;
      }
      // within-block entries: zero (the blocks' columns are nearly orthogonal)
      {
        const int blk = tid / (JB * JB), r = (tid / JB) % JB, c = tid % JB;
        L.A[blk * JB + r][blk * JB + c] = zmk(0.0, 0.0);
      }
    }
    reduce_block(L, gre, gim, tid, 0, JB, false);
    if (FULL) {
      gram_block(Wi, Wi, t.R, wave, lane, gre, gim, nx, ny);
      reduce_block(L, gre, gim, tid, 0, 0, true);
      gram_block(Wj, Wj, t.R, wave, lane, gre, gim, nx, ny);
      reduce_block(L, gre, gim, tid, JB, JB, true);
    } else {
      if (tid < JC) {
        const int side = tid / JB, col = tid % JB;
        double v = 0.0;
        for (int w = 0; w < kPairWaves; ++w) v += L.g.nred[w][side][col];
        L.dg[tid] = v;
      }
      __syncthreads();
    }
  }

  // ---- does this pair need a rotation?  |A_pq| > tol_rel sqrt(A_pp A_qq) and
  // |A_pq| > tol max_c|w_c| (|w_p| + |w_q|), tol = tol_abs (cyclic) or tol_pass: the second bound
  // is the rounding floor of the rotations in the |w_c|-sized columns of W
  {
    const double floor = (cyclic ? tol_abs : tol_pass) * sqrt(t.result[2]);  // of the largest column norm
    int need = 0;
    for (int e = tid; e < (FULL ? JC * JC : JB * JB); e += kRoundThreads) {
      const int pp = FULL ? e % JC : e % JB, qq = FULL ? e / JC : JB + e / JB;
      if (pp >= qq) continue;
      const double g2 = abs2(L.A[pp][qq]);
      const double app = fmax(L.dg[pp], 0.0), aqq = fmax(L.dg[qq], 0.0);
      const double fl = floor * (sqrt(app) + sqrt(aqq));
      if (g2 > tol_rel * tol_rel * app * aqq && g2 > fl * fl) need = 1;
    }
    if (need) L.need = 1;
    __syncthreads();
    if (!L.need) {
      if (tid == 0) {
        *seen = stamp;
        atomicAdd(&cnt[2], 1);
      }
      return;
    }
  }

  // ---- rotations of A -> Q, to the pair's slot; queue the pair for rotation
  if (cyclic) inner_solve(L, kRing.rounds, tid);
  else if constexpr (FULL) inner_jacobi<true>(L, kFull.rounds, tid);
  else inner_jacobi<false>(L, kCross.rounds, tid);
  zc (*Q)[JC + 1] = L.Q;
  zc* qg = t.Qg + (size_t)p * JC * JC;
  for (int e = tid; e < JC * JC; e += kRoundThreads) qg[e] = Q[e / JC][e % JC];  // qg[k JC + c] = Q[k][c]
  if (tid == 0) {
    atomicAdd(&cnt[sweep & 1], 1);
    atomicAdd(&cnt[2], 1);
    atomicAdd(&cnt[3], 1);
    t.blkver[lo] = vlo + 1;
    t.blkver[hi] = vhi + 1;
    const int slot = atomicAdd(&wl_count[round & 1], 1);
    if (slot < wl_cap) wl_items[(size_t)(round & 1) * wl_cap + slot] = make_int2(blockIdx.y, p);
  }
}

constexpr int kRotRows = 64;  // rows of W or V per work item of k_jacobi_rotate

// Work item w = (queued pair w / nchunk, 64-row slab w % nchunk): slabs of W first,
// then of V.  The pair's Q comes from its slot; each wave rotates 16 rows as
// (X Q)^T = Q^T X^T: A operand Q^T (16 output columns x 4 k), B operand X^T (4 k x
// 16 rows), so every load and store touches 4 columns x 16 consecutive rows.
__global__ __launch_bounds__(256) void k_jacobi_rotate(const BondTask* __restrict__ tasks, int round,
                                                       int* __restrict__ wl_count, const int2* __restrict__ wl_items,
                                                       int wl_cap, int nchunk_w, int nchunk) {
  if (blockIdx.x == 0 && threadIdx.x == 0) wl_count[(round + 1) & 1] = 0;  // the next round's queue
  const int n = min(wl_count[round & 1], wl_cap);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  for (int w = blockIdx.x; w < n * nchunk; w += gridDim.x) {
    const int2 item = wl_items[(size_t)(round & 1) * wl_cap + w / nchunk];
    const int chunk = w % nchunk;
    const BondTask& t = tasks[item.x];
    const int p = item.y;
    int bi, bj;
    rr_pair(2 * t.P, round, p, bi, bj);
    zc* M;
    int rows, ld, r0;
    if (chunk < nchunk_w) {
      M = t.W; rows = t.R; ld = t.R; r0 = chunk * kRotRows;
    } else {
      M = t.V; rows = t.V ? t.NV : 0; ld = t.NV; r0 = (chunk - nchunk_w) * kRotRows;
    }
    if (r0 >= rows) continue;
    const zc* qg = t.Qg + (size_t)p * JC * JC;
    double qre[2][8], qim[2][8];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        const zc q = qg[(4 * ks + lk) * JC + 16 * ct + lr];
        qre[ct][ks] = q.x;
        qim[ct][ks] = q.y;
      }
    auto col_of = [&](int c) { return c < JB ? bi * JB + c : bj * JB + (c - JB); };
    const int r = r0 + 16 * wave + lr;
    const bool in = r < rows;
    zc x[8];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) x[ks] = in ? M[(size_t)ld * col_of(4 * ks + lk) + r] : zmk(0.0, 0.0);
    d4 ore[2], oim[2];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      ore[ct] = d4{0.0, 0.0, 0.0, 0.0};
      oim[ct] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        ore[ct] = mfma4(qre[ct][ks], x[ks].x, ore[ct]);
        ore[ct] = mfma4(-qim[ct][ks], x[ks].y, ore[ct]);
        oim[ct] = mfma4(qre[ct][ks], x[ks].y, oim[ct]);
        oim[ct] = mfma4(qim[ct][ks], x[ks].x, oim[ct]);
      }
    }
    if (in) {
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int g = 0; g < 4; ++g) M[(size_t)ld * col_of(16 * ct + lk + 4 * g) + r] = zmk(ore[ct][g], oim[ct][g]);
    }
  }
}

// Start of a Jacobi solve: zero the counters and block versions, invalidate the
// verified-pair stamps.  One workgroup per task.
__global__ void k_jacobi_begin(const BondTask* __restrict__ tasks) {
  const BondTask t = tasks[blockIdx.x];
  const int nblk = 2 * t.P;
  if (threadIdx.x < kCounters) t.counter[threadIdx.x] = 0;
  for (int e = threadIdx.x; e < nblk; e += blockDim.x) t.blkver[e] = 0u;
  for (int e = threadIdx.x; e < nblk * nblk; e += blockDim.x) t.pairseen[e] = ~0ull;
}

// Start of sweep `sweep`: clear that sweep's rotation counter (its parity slot last
// held sweep - 2, which is no longer read) and both rotation queues.
__global__ void k_jacobi_sweep_begin(const BondTask* __restrict__ tasks, int ntasks, int sweep, int* wl_count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < ntasks) tasks[i].counter[sweep & 1] = 0;
  if (i < 2) wl_count[i] = 0;
}

}  // namespace

hipError_t launch_jacobi_begin(const BondTask* d_tasks, int ntasks, hipStream_t st) {
  hipLaunchKernelGGL(k_jacobi_begin, dim3(ntasks), dim3(256), 0, st, d_tasks);
  return hipGetLastError();
}

hipError_t launch_jacobi_sweep_begin(const BondTask* d_tasks, int ntasks, int sweep, int* wl_count, hipStream_t st) {
  hipLaunchKernelGGL(k_jacobi_sweep_begin, dim3((ntasks + 255) / 256), dim3(256), 0, st, d_tasks, ntasks, sweep,
                     wl_count);
  return hipGetLastError();
}

hipError_t launch_jacobi_round(const BondTask* d_tasks, int ntasks, int max_pairs, int sweep, int round,
                               double tol_rel, double tol_abs, double tol_pass, int* wl_count, int2* wl_items,
                               int wl_cap, hipStream_t st) {
  const auto k = round == 0 ? k_jacobi_round<true> : k_jacobi_round<false>;
  hipLaunchKernelGGL(k, dim3(max_pairs, ntasks), dim3(kRoundThreads), 0, st, d_tasks, sweep, round, tol_rel, tol_abs,
                     tol_pass, wl_count, wl_items, wl_cap);
  return hipGetLastError();
}

hipError_t launch_jacobi_rotate(const BondTask* d_tasks, int round, int max_rows_w, int max_rows_v, int* wl_count,
                                int2* wl_items, int wl_cap, hipStream_t st) {
  const int nw = (max_rows_w + kRotRows - 1) / kRotRows, nv = (max_rows_v + kRotRows - 1) / kRotRows;
  hipLaunchKernelGGL(k_jacobi_rotate, dim3(1024), dim3(256), 0, st, d_tasks, round, wl_count, wl_items, wl_cap, nw,
                     nw + nv);
  return hipGetLastError();
}
