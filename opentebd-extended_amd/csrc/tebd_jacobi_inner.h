// The inner solve of a Jacobi pair: rounds of 16 disjoint rotations on a 32 x 32 Hermitian
// Gram matrix in LDS.  Shared by the large solve (tebd_jacobi.hip) and the small one
// (tebd_jacobi_small.hip), which differ in the order of the rounds, the rotation formula and
// where the accumulated rotations are kept.
//
// What bounds a round: a wave64 instruction holds its SIMD for 4 cycles, so a round costs the
// instructions of its longest wave plus one LDS round trip and one barrier.  With the index
// arithmetic done in place, the rotations formed by all four waves and every entry read by
// two threads, a round took 1650 cycles (0.69 us), now 1345; hence
//   * one barrier per round: the thread that has updated the entry of one of the next round's
//     pairs forms that rotation at once, from the value in its registers;
//   * the threads that do so sit in one wave, the others skip the rotation's code;
//   * everything that depends only on the round and the thread (LDS offsets, signs, the next
//     pair) comes from a table in LDS (read from global memory in every round it made each
//     barrier wait for L2);
//   * only the upper triangle of A is kept, each entry is read by one lane, and the two lanes
//     of a 2x2 block exchange their rows;
//   * every LDS read of a round is issued before its first product, and the table's entries one
//     round ahead, so a round waits for LDS once (1405 cycles without).
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

// The table from constant memory to LDS, by all n threads of the workgroup.
template <int NR, int NN>
__device__ __forceinline__ void load_rounds(InnerRounds<NR, NN>& dst, const InnerRounds<NR, NN>& src, int tid, int n) {
  unsigned* d = &dst.entry[0][0];
  const unsigned* s = &src.entry[0][0];
  for (int e = tid; e < (int)(sizeof(dst) / sizeof(unsigned)); e += n) d[e] = s[e];
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

}  // namespace
