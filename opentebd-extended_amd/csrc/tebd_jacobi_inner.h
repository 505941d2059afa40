// A Jacobi pair: its 32 x 32 Hermitian Gram matrix in LDS and rounds of 16 disjoint rotations on
// it.  Shared by the sweep-by-sweep solve (tebd_jacobi.hip) and the one-launch solve
// (tebd_jacobi_small.hip): the latter, and the former where the task asks for it, solve a pair's
// problem by whole cyclic sweeps (inner_solve); the former has schedules of its own for a single pass.
//
// What bounds a round: a wave64 instruction holds its SIMD for 4 cycles, so a round costs the
// instructions of its longest wave plus one LDS round trip and one barrier.  With the index
// arithmetic done in place, the rotations formed by all four waves and every entry read by
// two threads, a round took 1650 cycles (0.69 us), now 1345; hence
//   * one barrier per round: the thread that has updated the entry of one of the next round's
//     pairs forms that rotation at once, from the value in its registers;
//   * the threads that do so sit in one wave, the others skip the rotation's code;
//   * everything that depends only on the round and the thread (LDS offsets, signs, the next
//     pair) comes from a table, read one round ahead so that no barrier waits for L2;
//   * only the upper triangle of A is kept, each entry is read by one lane, and the two lanes
//     of a 2x2 block exchange their rows;
//   * every LDS read of a round is issued before its first product, so a round waits for LDS once
//     (1405 cycles without).
#pragma once
#include "tebd_device.h"

namespace {

constexpr int kInnerPairs = JC / 2;                               // 16 rotations per round
constexpr int kAllRounds = JC - 1;                                // rounds that visit every pair once
constexpr int kOffBlocks = kInnerPairs * (kInnerPairs - 1) / 2;   // 2x2 blocks above the diagonal
constexpr int kInnerLd = JC + 1;                                  // leading dimension of A in LDS
static_assert(JC == 32 && 2 * kOffBlocks <= 256, "four waves update A");

// Rotations of one round, pair t: c and s w (c = 1, s w = 0: the pair stays put).
struct RotBuf {
  double c[kInnerPairs];
  zc sw[kInnerPairs];
};

// A schedule of rounds as the threads 0 .. 239 that update A see it.  Thread th has row th & 1 of
// the block of the pairs tr[th] < tk[th]: the entries (own, p_k) and (own, q_k), own = p_r or q_r.
//   entry   byte offset of (own, p_k) in bits 0..14 and of (own, q_k) in bits 15..29, both in the
//           upper triangle; bit 30 / 31: that entry is stored as its conjugate;
//   next    bits 0..7 / 8..15: 8 x the indices p < q of the next round's pair whose entry this
//           thread updates, bit 16: there is one, bit 17: it is the entry at column p_k, bit 18:
//           the thread holds its conjugate, bits 20..23: the pair's number.
// NR rounds; only threads below NN have a next pair.
template <int NR, int NN>
struct InnerRounds {
  unsigned entry[NR][2 * kOffBlocks];
  unsigned next[NR][NN];
};
template <int NR, int NN>
struct InnerTable {
  InnerRounds<NR, NN> rounds;
  unsigned char tr[2 * kOffBlocks], tk[2 * kOffBlocks];
  unsigned char p[NR][kInnerPairs], q[NR][kInnerPairs];
};

// Completes a table whose p, q (p < q) are filled in; the blocks (first_tr[i], first_tk[i]), i <
// 16, are dealt to the first wave.
template <int NR, int NN>
constexpr InnerTable<NR, NN> complete_table(InnerTable<NR, NN> t, const int (&first_tr)[16], const int (&first_tk)[16]) {
  bool used[16][16] = {};
  int n = 0;
  for (int i = 0; i < 16; ++i) {
    used[first_tr[i]][first_tk[i]] = true;
    for (int h = 0; h < 2; ++h, ++n) {
      t.tr[n] = (unsigned char)first_tr[i];
      t.tk[n] = (unsigned char)first_tk[i];
    }
  }
  for (int r = 0; r < 16; ++r)
    for (int k = r + 1; k < 16; ++k) {
      if (used[r][k]) continue;
      for (int h = 0; h < 2; ++h, ++n) {
        t.tr[n] = (unsigned char)r;
        t.tk[n] = (unsigned char)k;
      }
    }
  for (int rd = 0; rd < NR; ++rd) {
    int mate[JC] = {}, num[JC] = {};  // the next round's partner and pair number of each index
    if (rd + 1 < NR)
      for (int x = 0; x < 16; ++x) {
        mate[t.p[rd + 1][x]] = t.q[rd + 1][x];
        mate[t.q[rd + 1][x]] = t.p[rd + 1][x];
        num[t.p[rd + 1][x]] = num[t.q[rd + 1][x]] = x;
      }
    for (int th = 0; th < 2 * kOffBlocks; ++th) {
      const int r = t.tr[th], k = t.tk[th];
      const int own = (th & 1) ? t.q[rd][r] : t.p[rd][r];
      const int c0 = t.p[rd][k], c1 = t.q[rd][k];
      const unsigned l0 = 16u * (unsigned)(own < c0 ? own * kInnerLd + c0 : c0 * kInnerLd + own);
      const unsigned l1 = 16u * (unsigned)(own < c1 ? own * kInnerLd + c1 : c1 * kInnerLd + own);
      t.rounds.entry[rd][th] = l0 | l1 << 15 | (own > c0 ? 1u << 30 : 0u) | (own > c1 ? 1u << 31 : 0u);
      unsigned nx = 0;
      if (rd + 1 < NR && (mate[own] == c0 || mate[own] == c1)) {
        const int m = mate[own];
        const unsigned lo = (unsigned)(own < m ? own : m), hi = (unsigned)(own < m ? m : own);
        nx = 8u * lo | (8u * hi) << 8 | 1u << 16 | (m == c0 ? 1u << 17 : 0u) | (own > m ? 1u << 18 : 0u) |
             (unsigned)num[own] << 20;
      }
      if (th < NN) t.rounds.next[rd][th] = nx;
    }
  }
  return t;
}

// Lane moves inside rows of 16 lanes (`edge`: what a lane without a source gets): from the next
// lane, from the previous one, from the next one cyclically, and between lanes 2k and 2k + 1.
constexpr int kDppNext = 0x101, kDppPrev = 0x111, kDppRotate = 0x12f, kDppSwap = 0xb1;
template <int CTRL>
__device__ __forceinline__ double dpp(double edge, double v) {
  const long long e = __double_as_longlong(edge), x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)e, (int)x, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(e >> 32), (int)(x >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int CTRL>
__device__ __forceinline__ zc zdpp(zc edge, zc v) {
  return zmk(dpp<CTRL>(edge.x, v.x), dpp<CTRL>(edge.y, v.y));
}
// The same where every lane has a source.
template <int CTRL>
__device__ __forceinline__ zc zdpp(zc v) {
  return zmk(dpp_mov<CTRL>(v.x), dpp_mov<CTRL>(v.y));
}
// a or b, part by part (a conditional of the two structs would keep them in memory)
__device__ __forceinline__ zc zsel(bool first, zc a, zc b) { return zmk(first ? a.x : b.x, first ? a.y : b.y); }
// v with its sign flipped when the top bit of m is set
__device__ __forceinline__ double flip(double v, unsigned m) {
  return __longlong_as_double(__double_as_longlong(v) ^ ((long long)(m & 0x80000000u) << 32));
}
__device__ __forceinline__ double abs2(zc a) { return fma(a.x, a.x, a.y * a.y); }

// The inner solve rotates a pair unless its entry is below a purely relative bound (a Gram
// entry is accurate relative to sqrt(A_pp A_qq)).
__device__ __forceinline__ bool needs_rotation(double g2, double a, double b) {
  return !(g2 <= 1e-30 * fabs(a * b) || g2 == 0.0);
}

// The rotation of pair t with entry g = A_pq and diagonal a, b: into rb; a rotated pair's
// diagonal goes to *da, *db.  Returns the entry after it (zero, or g when the pair stays put).
// rotate(a, b, g, |g|^2, c, s w) forms the rotation and the rotated diagonal; it is formed
// before the test on it is known, which takes the test off the dependent chain.
template <class Rotate>
__device__ __forceinline__ zc make_rotation(RotBuf& rb, double a, double b, double* da, double* db, int* swept, int t,
                                            zc g, Rotate rotate) {
  const double g2 = abs2(g);
  const bool need = needs_rotation(g2, a, b);
  double c;
  zc sw;
  rotate(a, b, g, g2, c, sw);
  rb.c[t] = need ? c : 1.0;
  rb.sw[t] = zmk(need ? sw.x : 0.0, need ? sw.y : 0.0);
  if (need) {
    *da = a;
    *db = b;
    if (swept) *swept = 1;
  }
  return zmk(need ? 0.0 : g.x, need ? 0.0 : g.y);
}

// One thread's part of a round on A (LDS, kInnerLd): the rotations R applied to its row of its
// block, and the next round's rotation into N if its pair's entry is among them.
template <class Rotate>
__device__ __forceinline__ void update_block(zc* A, double* dg, const RotBuf& R, RotBuf& N, int* swept, unsigned entry,
                                             unsigned next, int tr, int tk, int half, Rotate rotate) {
#pragma clang fp contract(off)
  char* const base = reinterpret_cast<char*>(A);
  zc* const l0 = reinterpret_cast<zc*>(base + (entry & 0x7fffu));
  zc* const l1 = reinterpret_cast<zc*>(base + ((entry >> 15) & 0x7fffu));
  const zc swr = R.sw[tr], swk = R.sw[tk];
  const double cr = R.c[tr], ck = R.c[tk];
  zc own0 = *l0, own1 = *l1;
  double* const da = reinterpret_cast<double*>(reinterpret_cast<char*>(dg) + (next & 0xffu));
  double* const db = reinterpret_cast<double*>(reinterpret_cast<char*>(dg) + ((next >> 8) & 0xffu));
  double a = *da, b = *db;
  // every LDS read of the round is under way before the first value is used
  asm volatile("" : "+v"(a), "+v"(b), "+v"(own0.x), "+v"(own0.y), "+v"(own1.x), "+v"(own1.y));
  const bool rot = swr.x != 0.0 || swr.y != 0.0 || swk.x != 0.0 || swk.y != 0.0 || next != 0u;
  if (!__any(rot)) return;
  const unsigned s0 = entry << 1, s1 = entry;  // the conjugation bits at the top
  own0.y = flip(own0.y, s0);
  own1.y = flip(own1.y, s1);
  const zc oth0 = zdpp<kDppSwap>(own0), oth1 = zdpp<kDppSwap>(own1);
  // this lane's row after the row rotation: A_p <- c A_p - s w A_q ; A_q <- s conj(w) A_p + c A_q;
  // then the column rotation: A_:p <- c A_:p - s conj(w) A_:q ; A_:q <- s w A_:p + c A_:q
  const double fx = half ? swr.x : -swr.x;
  const zc x0 = zmk(fma(cr, own0.x, fma(fx, oth0.x, swr.y * oth0.y)), fma(cr, own0.y, fma(fx, oth0.y, -(swr.y * oth0.x))));
  const zc x1 = zmk(fma(cr, own1.x, fma(fx, oth1.x, swr.y * oth1.y)), fma(cr, own1.y, fma(fx, oth1.y, -(swr.y * oth1.x))));
  zc n0 = zmk(fma(ck, x0.x, -fma(swk.x, x1.x, swk.y * x1.y)), fma(ck, x0.y, -fma(swk.x, x1.y, -(swk.y * x1.x))));
  zc n1 = zmk(fma(ck, x1.x, fma(swk.x, x0.x, -(swk.y * x0.y))), fma(ck, x1.y, fma(swk.y, x0.x, swk.x * x0.y)));
  if (next) {
    const bool first = next & (1u << 17);
    zc n = zsel(first, n0, n1);
    const unsigned sn = next << 13;  // bit 18 at the top
    n.y = flip(n.y, sn);
    n = make_rotation(N, a, b, da, db, swept, (int)(next >> 20), n, rotate);
    n.y = flip(n.y, sn);
    n0 = zsel(first, n, n0);
    n1 = zsel(first, n1, n);
  }
  n0.y = flip(n0.y, s0);
  n1.y = flip(n1.y, s1);
  *l0 = n0;
  *l1 = n1;
}

// ---- a pair's LDS, its Gram matrix and the whole 32 x 32 problem by cyclic sweeps ----
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
#pragma clang fp contract(off)
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
#pragma clang fp contract(off)
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
#pragma clang fp contract(off)
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
// by every thread.
__device__ __forceinline__ void reduce_block(PairLds& L, d4 gre, d4 gim, int pt, int ro, int co, bool diag) {
#pragma clang fp contract(off)
  const int wave = pt >> 6, lane = pt & 63;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    L.g.red[wave][g * 64 + lane] = gre[g];
    L.g.red[wave][256 + g * 64 + lane] = gim[g];
  }
  __syncthreads();
  {
    const int idx = pt & 255, l = idx & 63, im = pt >> 8;
    double v = L.g.red[0][pt];
    for (int w = 1; w < kPairWaves; ++w) v += L.g.red[w][pt];
    const int p = (l >> 4) + 4 * (idx >> 6), q = l & 15;
    if (!diag || p < q) reinterpret_cast<double*>(&L.A[ro + p][co + q])[im] = v;
    else if (p == q && !im) L.dg[ro + p] = v;
  }
  __syncthreads();
}

// The pair's 32 x 32 eigenproblem by cyclic Jacobi: at most kInnerSweepCap sweeps, ended when a sweep
// rotates nothing or the next one would not.  Waves 0..3 update A; waves 4..7 apply the round's
// rotations to Q, held in registers: lane t of a 16-lane row has two rows' entries of Q at ring
// positions t and 31 - t, and the ring's move by one position per round is a move between
// neighbouring lanes.
template <class Rounds>
__device__ __forceinline__ void inner_solve(PairLds& L, const Rounds& T, int pt) {
#pragma clang fp contract(off)
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
#pragma unroll 1
  for (int isw = 0; isw < kInnerSweepCap; ++isw) {
    if (pt == 0) L.swept[isw & 1] = 0;
    __syncthreads();
    if (pt < JC / 2) {
      const int p = kRing.p[0][pt], q = kRing.q[0][pt];
      L.A[p][q] = make_rotation(L.rb[buf], L.dg[p], L.dg[q], &L.dg[p], &L.dg[q], &L.swept[isw & 1], pt, L.A[p][q], jrot);
    }
    __syncthreads();
    unsigned entry = is_a ? T.entry[0][pt] : 0u, next = pt < 2 * kInnerPairs ? T.next[0][pt] : 0u;
#pragma unroll 1
    for (int rd = 0; rd < kAllRounds; ++rd, buf ^= 1) {
      const RotBuf& R = L.rb[buf];
      if (is_q) {
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
    if (L.swept[isw & 1])
      for (int e = pt; e < JC * JC; e += kPairThreads) {
        const int pp = e % JC, qq = e / JC;
        if (pp < qq && needs_rotation(abs2(L.A[pp][qq]), L.dg[pp], L.dg[qq])) L.more = 1;
      }
    __syncthreads();
    if (!L.more) break;
  }
  // after whole sweeps the ring is back at its start
  if (is_q) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      L.Q[qk + 16 * u][ring(0, qt)] = f[u];
      L.Q[qk + 16 * u][ring(0, JC - 1 - qt)] = s[u];
    }
  }
  __syncthreads();
}

}  // namespace
