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

typedef double d4 __attribute__((ext_vector_type(4)));

// D(16x16) += A(16x4) B(4x16).  Lane l supplies A[l%16][l/16] and B[l/16][l%16];
// element g of the result in lane l is D[l/16 + 4g][l%16].
__device__ __forceinline__ d4 mfma4(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

constexpr int kPairThreads = 512;            // threads of one pair
constexpr int kPairWaves = kPairThreads / 64;
constexpr int kInnerSweepCap = 3;            // cyclic inner sweeps per pair visit

// Round-robin ("circle") schedule over nb = 2P blocks: block 0 stays, the others
// rotate; over nb-1 rounds every pair of blocks meets exactly once.
__device__ __forceinline__ void rr_pair(int nb, int round, int p, int& bi, int& bj) {
  auto pos = [&](int k) { return k == 0 ? 0 : 1 + (k - 1 + round) % (nb - 1); };
  bi = pos(p);
  bj = pos(nb - 1 - p);
}

// 1/sqrt(x) to full FP64 precision: the hardware estimate refined by two Newton-Raphson
// steps (y <- y (3 - x y^2) / 2).
__device__ __forceinline__ double rsqrt_nr(double x) {
  double y = __builtin_amdgcn_rsq(x);
  y = y * fma(-0.5 * x * y, y, 1.5);
  return y * fma(-0.5 * x * y, y, 1.5);
}

// Hermitian 2x2 Jacobi rotation J = [[c, s w], [-s conj(w), c]], w = g/|g|, that zeroes g in
// [[a, g], [conj(g), b]] via J^dagger H J, with the inner angle (|theta| <= pi/4).  With
// e = sqrt((b - a)^2 + 4|g|^2): cos 2theta = |b - a| / e, sin 2theta = 2|g| / e, c = (1 + cos
// 2theta) r and |s| = sin 2theta r with r = 1/sqrt(2 (1 + cos 2theta)); s takes the sign of
// b - a.  a and b become the rotated diagonal a - t|g|, b + t|g|, t = s / c.
__device__ __forceinline__ void jrot(double& a, double& b, zc g, double g2, double& c, zc& sw) {
  const double dd = b - a;
  const double inv = rsqrt_nr(g2);
  const double re = rsqrt_nr(fma(dd, dd, 4.0 * g2));
  const double h = fma(fabs(dd), re, 1.0);  // 1 + cos 2theta
  const double sin2 = (2.0 * g2 * inv) * re;
  const double r = rsqrt_nr(2.0 * h);
  const double sg = dd < 0.0 ? -sin2 : sin2;
  const double s = sg * r, x = g2 * inv, y = sg * (2.0 * r * r);
  c = h * r;
  sw = zmk(g.x * inv * s, g.y * inv * s);
  a = fma(-x, y, a);
  b = fma(x, y, b);
}

// The LDS of one pair.  Until the inner solve starts, Q's storage holds the Gram's reduction
// scratch and the column-norm partials.
struct PairLds {
  zc A[JC][kInnerLd];  // the pair's Gram matrix: its upper triangle; its diagonal is in dg
  double dg[JC];
  union {
    zc Q[JC][JC + 1];
    struct {
      double red[kPairWaves][512];
      double nred[kPairWaves][2][16];
    } g;
  };
  RotBuf rb[2];
  int need;       // the pair needs a rotation this round
  int swept[2];   // a rotation in inner sweep (parity)
  int more;       // another inner sweep would rotate something
};

// Element at position k of inner round rd (circle order over JC indices).
constexpr __host__ __device__ int ring(int rd, int k) {
  int x = k - 1 + rd;
  x = x >= JC - 1 ? x - (JC - 1) : x;
  return k == 0 ? 0 : 1 + x;
}

// Cyclic order: pair t of round rd is ring positions t and 31 - t.  The ring moves every element
// by one position per round, so pair t's next elements are now at positions 32 - t and t + 1: the
// next pairs' entries lie in the blocks (0, 1), (t - 1, t + 1) and (14, 15).
using RingTable = InnerTable<kAllRounds, 2 * kInnerPairs>;
constexpr RingTable ring_table() {
  RingTable t{};
  for (int rd = 0; rd < kAllRounds; ++rd)
    for (int x = 0; x < kInnerPairs; ++x) {
      const int a = ring(rd, x), b = ring(rd, JC - 1 - x);
      t.p[rd][x] = (unsigned char)(a < b ? a : b);
      t.q[rd][x] = (unsigned char)(a < b ? b : a);
    }
  int r[16] = {}, k[16] = {};
  for (int x = 0; x < 16; ++x) {
    r[x] = x == 0 ? 0 : x - 1;
    k[x] = x == 0 ? 1 : (x == 15 ? 15 : x + 1);
  }
  return complete_table(t, r, k);
}
__device__ constexpr RingTable kRing = ring_table();

// Gram block D = X^H Y (16 x 16) of two 16-column blocks over rows [0, R), as per-wave
// partial sums of kPairWaves waves (wave w takes rows 8 (w + kPairWaves m) .. +7), with the
// lane's partial squared norms of X and Y.
__device__ __forceinline__ void gram_block(const zc* X, const zc* Y, int R, int wave, int lane, d4& gre, d4& gim,
                                           double& nx, double& ny) {
  constexpr int U = 2;
  const int lr = lane & 15, lk = lane >> 4;
  gre = d4{0.0, 0.0, 0.0, 0.0};
  gim = d4{0.0, 0.0, 0.0, 0.0};
  nx = 0.0;
  ny = 0.0;
  const zc* xc = X + (size_t)R * lr;
  const zc* yc = Y + (size_t)R * lr;
  constexpr int PER = 8 * kPairWaves;
#pragma unroll 1
  for (int r0 = 8 * wave; r0 < R; r0 += PER * U) {
    zc a[2 * U], b[2 * U];
#pragma unroll
    for (int u = 0; u < 2 * U; ++u) {
      const int r = r0 + PER * (u >> 1) + 4 * (u & 1) + lk;
      a[u] = r < R ? xc[r] : zmk(0.0, 0.0);
      b[u] = r < R ? yc[r] : zmk(0.0, 0.0);
    }
#pragma unroll
    for (int u = 0; u < 2 * U; ++u) {
      gre = mfma4(a[u].x, b[u].x, gre);
      gre = mfma4(a[u].y, b[u].y, gre);
      gim = mfma4(a[u].x, b[u].y, gim);
      gim = mfma4(-a[u].y, b[u].x, gim);
      nx += abs2(a[u]);
      ny += fma(b[u].y, b[u].y, b[u].x * b[u].x);
    }
  }
}

// Sums the waves' partial blocks in wave order and stores the upper triangle's part of rows
// [ro, ro+16) x cols [co, co+16) of A (diagonal blocks: the real diagonal goes to dg).  Called
// by every thread; `on` is uniform per pair.
__device__ __forceinline__ void reduce_block(PairLds& L, bool on, d4 gre, d4 gim, int pt, int ro, int co, bool diag) {
  const int wave = pt >> 6, lane = pt & 63;
  if (on) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      L.g.red[wave][g * 64 + lane] = gre[g];
      L.g.red[wave][256 + g * 64 + lane] = gim[g];
    }
  }
  __syncthreads();
  if (on) {
    const int idx = pt & 255, l = idx & 63, im = pt >> 8;
    double v = L.g.red[0][pt];
    for (int w = 1; w < kPairWaves; ++w) v += L.g.red[w][pt];
    const int p = (l >> 4) + 4 * (idx >> 6), q = l & 15;
    if (!diag || p < q) reinterpret_cast<double*>(&L.A[ro + p][co + q])[im] = v;
    else if (p == q && !im) L.dg[ro + p] = v;
  }
  __syncthreads();
}

// The 32 x 32 eigenproblems of the workgroup's pairs, by cyclic Jacobi: at most
// kInnerSweepCap sweeps, ended when a sweep rotates nothing or the next one would.  Waves 0..3 of
// a pair update A; waves 4..7 apply the round's rotations to Q, held in registers: lane t of a
// 16-lane row has two rows' entries of Q at ring positions t and 31 - t, and the ring's move by
// one position per round is a move between neighbouring lanes.  All threads take part in every
// barrier; pairs that need no rotation, or have finished, only wait.
__device__ __forceinline__ void inner_solve(PairLds& L, const InnerRounds<kAllRounds, 2 * kInnerPairs>& T, int pt, bool on) {
  const bool is_q = pt >= 256, is_a = pt < 2 * kOffBlocks;
  const int tr = is_a ? kRing.tr[pt] : 0, tk = is_a ? kRing.tk[pt] : 0, half = pt & 1;
  // rows qk and qk + 16 of Q at ring positions qt (f) and 31 - qt (s), starting from the identity
  const int qt = pt & 15, qk = (pt >> 4) & 15;
  zc f[2], s[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    f[u] = zmk(qk + 16 * u == ring(0, qt) ? 1.0 : 0.0, 0.0);
    s[u] = zmk(qk + 16 * u == ring(0, JC - 1 - qt) ? 1.0 : 0.0, 0.0);
  }
  int buf = 0;
  bool live = on;
#pragma unroll 1
  for (int isw = 0; isw < kInnerSweepCap; ++isw) {
    if (pt == 0) L.swept[isw & 1] = 0;
    __syncthreads();
    if (live && pt < JC / 2) {
      const int p = kRing.p[0][pt], q = kRing.q[0][pt];
      L.A[p][q] = make_rotation(L.rb[buf], L.dg[p], L.dg[q], &L.dg[p], &L.dg[q], &L.swept[isw & 1], pt, L.A[p][q], jrot);
    }
    __syncthreads();
    unsigned entry = is_a ? T.entry[0][pt] : 0u, next = pt < 2 * kInnerPairs ? T.next[0][pt] : 0u;
#pragma unroll 1
    for (int rd = 0; rd < kAllRounds; ++rd, buf ^= 1) {
      const RotBuf& R = L.rb[buf];
      if (!live) {
      } else if (is_q) {
        // with p the lower of the pair's indices: Q_:p <- c Q_:p - s conj(w) Q_:q ; Q_:q <- s w Q_:p
        // + c Q_:q.  f and s take the two roles as fp says; the signs go into x, and only the
        // imaginary parts' products change their order of rounding with the roles.
        const bool fp = ring(rd, qt) < ring(rd, JC - 1 - qt);
        const double c = R.c[qt];
        const zc sw = R.sw[qt];
        if (__any(sw.x != 0.0 || sw.y != 0.0)) {
          const double x = fp ? -sw.x : sw.x, y = sw.y;
          const double u1 = fp ? x : y, m1 = fp ? y : x, u2 = fp ? y : -x, m2 = fp ? -x : y;
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const zc a = f[u], b = s[u];
            const double a1 = fp ? b.y : b.x, b1 = fp ? b.x : b.y, a2 = fp ? a.x : a.y, b2 = fp ? a.y : a.x;
            f[u] = zmk(fma(c, a.x, fma(x, b.x, -(y * b.y))), fma(c, a.y, fma(u1, a1, m1 * b1)));
            s[u] = zmk(fma(c, b.x, fma(-x, a.x, -(y * a.y))), fma(c, b.y, fma(u2, a2, m2 * b2)));
          }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {  // the ring moves on
          const zc nf = zdpp<kDppNext>(s[u], f[u]);
          s[u] = zdpp<kDppPrev>(nf, s[u]);
          f[u] = zsel(qt != 0, nf, f[u]);
        }
      } else if (is_a) {
        update_block(&L.A[0][0], L.dg, R, L.rb[buf ^ 1], &L.swept[isw & 1], entry, next, tr, tk, half, jrot);
        const int ahead = rd + 1 < kAllRounds ? rd + 1 : 0;  // read now, used after the barrier
        entry = T.entry[ahead][pt];
        if (pt < 2 * kInnerPairs) next = T.next[ahead][pt];
      }
      __syncthreads();
    }
    if (isw + 1 == kInnerSweepCap) break;
    // would the next sweep rotate anything?
    if (pt == 0) L.more = 0;
    __syncthreads();
    if (live && L.swept[isw & 1])
      for (int e = pt; e < JC * JC; e += kPairThreads) {
        const int pp = e % JC, qq = e / JC;
        if (pp < qq && needs_rotation(abs2(L.A[pp][qq]), L.dg[pp], L.dg[qq])) L.more = 1;
      }
    __syncthreads();
    if (live && !L.more) live = false;
  }
  // after whole sweeps the ring is back at its start
  if (on && is_q) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      L.Q[qk + 16 * u][ring(0, qt)] = f[u];
      L.Q[qk + 16 * u][ring(0, JC - 1 - qt)] = s[u];
    }
  }
  __syncthreads();
}

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
  if (t.qr || t.P != NP) return;
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
      inner_solve(L, table, pt, rot);
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
