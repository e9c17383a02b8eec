// Banded NW DP in packed 16-bit arithmetic: two band positions of a pair per
// 32-bit register, the directions written out and traced back afterwards.
// Included only by the per-family sources nw_fam_pk*.hip.  Recurrence and tie
// rules: see the head of nw.hip (genCPU.cpp:348-464).
//
// Why: the DP is bound by VALU issue, and nw_reg_wave / nw_sliced_wave issue
// ~13.5 instructions per cell (4 selects and 2 compares of them carry the
// direction, match count and alignment length along every cell).  Here a
// cell's whole comparison is one integer maximum, and only the end cell's path
// is ever counted: 5.15 instructions per cell in the plain steps, the
// directions' 2 bits written once and the path read back by the wave that
// wrote it.  Counted over whole calls, with the boundary and last-column steps,
// the padding and the trace: 7.3 to 7.7 per in-band cell for 200-900 bp reads
// at bands 5 and 10, 9.1 for 2000-3200 bp (slices of at most 24 cells), 12 for
// 1,000 reads and 24 for full alignments, which are boundary steps mostly.
// Measured (the DP phase, before -> now): 0.84 M pairs of 200-300 bp at band 10
// 3.4 -> 2.03 ms; 3.27 M pairs of 150-550 bp 16.9 -> 10.2 ms; 0.24 M pairs of
// 400-900 bp at band 5 12.3 -> 7.0 ms; whole calls with 3000 full alignments of
// 200-300 bp, which had only the generic kernel, 26.0 -> 0.6 ms, and with reads
// of 300-500 bp, some with N, 18.2 -> 2.6 ms.
// The second bound at large calls is the traffic: 15 GB out and 20 GB back for
// 5.0e10 cells, of which the directions themselves are 12.5 GB each way (the
// rest is padding, spilled registers and partly used lines), 3.4 TB/s where a
// copy reaches 4.96.
//
// Key of a cell: 4 (M + 11 i - 7 j + off) + p in 16 bits, p = the direction's
// tie rank (diagonal 3, then 2 and 1: "up" before "left", or "left" before
// "up" in the transposed frame).  So max(diag, up, left) of the candidates'
// keys is the reference's choice, ties included, and its low bits are the
// direction.  The frame 11 i - 7 j makes a mismatch add nothing, and both gap
// offers one table look-up by p with 8-bit entries (v_perm_b32 does two):
//   offer to the right  K_h = W - TabH[p]   (pen_h, -7, rank "up")
//   offer below         K_v = W + TabV[p]   (pen_v, +11, rank "left")
//   diagonal            K_d = W | 3, + 36 on a match.
// 0 stands for out of band: every real key is at least 4 * 32.
//
// Layout: a pair's W = 2 kB + 1 band positions are cut into V = 2 G slices of
// C; virtual lane v = 2 g + h (lane g of the pair, h = low / high half) owns
// positions [C v, C v + C) and runs row t - v at step t, one row behind its
// left neighbour.  So a lane's two halves are two slices of one pair, and a
// slice needs per step only its left neighbour's last K_h (sent at the end of
// the step before) and its right neighbour's first K_v (computed first in the
// same step): the other half of the lane's own word, or a DPP shift.
//
// Per two cells 10.3 VALU instructions (11.3 where keys pass 0x7BFF), 5 of
// them at the 4-cycle rate of packed and three-operand forms, which no more
// waves hide (measured: half-and-half mixes issue one per 3.8 cycles and SIMD):
// the match bit masked out of a match word, v_pk_mad_u16, v_pk_maximum3_f16
// (or two v_pk_max_u16), the rank mask, two v_perm_b32, one subtract, one add,
// one or, and the direction shifted into a word of 8 cells x 2 halves.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "common.hpp"
#include "nw_fused.hpp"

namespace crispy {

typedef unsigned short pk_u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk_max(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(pk_u16x2, a),
                                                                __builtin_bit_cast(pk_u16x2, b)));
}

// The maximum of three keys per half.  F16: keys up to 0x7BFF are finite
// non-negative half-precision patterns, which order like the integers, and one
// v_pk_maximum3_f16 replaces two v_pk_max_u16.
typedef _Float16 pk_f16x2 __attribute__((ext_vector_type(2)));
template <bool F16>
__device__ __forceinline__ uint32_t pk_max3(uint32_t a, uint32_t b, uint32_t c) {
  if constexpr (F16)
    return __builtin_bit_cast(
        uint32_t, __builtin_elementwise_maximum(__builtin_elementwise_maximum(__builtin_bit_cast(pk_f16x2, a),
                                                                              __builtin_bit_cast(pk_f16x2, b)),
                                                __builtin_bit_cast(pk_f16x2, c)));
  else
    return pk_max(pk_max(a, b), c);
}

__device__ __forceinline__ uint32_t pk_mad(uint32_t a, unsigned short c, uint32_t b) {
  return __builtin_bit_cast(uint32_t,
                            __builtin_bit_cast(pk_u16x2, a) * (pk_u16x2){c, c} + __builtin_bit_cast(pk_u16x2, b));
}

__device__ __forceinline__ uint32_t pk_word(const uint32_t *s, int w, int nw) {
  return (w >= 0 && w < nw) ? s[w] : 0u;
}

// the 16 even bits of w, packed
__device__ __forceinline__ uint32_t pk_even(uint32_t w) {
  w &= 0x55555555u;
  w = (w | (w >> 1)) & 0x33333333u;
  w = (w | (w >> 2)) & 0x0F0F0F0Fu;
  w = (w | (w >> 4)) & 0x00FF00FFu;
  return (w | (w >> 8)) & 0xFFFFu;
}

// A stream of a read's bases, 16 at a time, from base index q on (any
// alignment, zeros outside the read).  One word is loaded per 16 bases, two
// blocks ahead of its use in the source; the loop that the compiler makes waits
// for it right after the load, and other waves cover that wait.
struct PkStream {
  const uint32_t *s;
  int nw, w, sh;        // next word to load, 2 (q mod 16)
  uint32_t w0, w1, w2;  // the next block's words and the one after
  __device__ __forceinline__ void open(const uint32_t *s_, int nw_, int q) {
    s = s_;
    nw = nw_;
    w = q >> 4;
    sh = 2 * (q & 15);
    w0 = pk_word(s, w, nw);
    w1 = pk_word(s, w + 1, nw);
    w2 = pk_word(s, w + 2, nw);
    w += 3;
  }
  __device__ __forceinline__ uint32_t next() {  // 16 bases, 2 bits each
    const uint32_t r = (uint32_t)((((uint64_t)w1 << 32) | w0) >> sh);
    w0 = w1;
    w1 = w2;
    w2 = pk_word(s, w, nw);
    ++w;
    return r;
  }
};

template <int A, class F, int... I>
__device__ __forceinline__ void static_for_pk_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, A + I>{}), ...);
}
// f(integral_constant<int, A>) ... f(integral_constant<int, B - 1>), unrolled
template <int A, int B, class F>
__device__ __forceinline__ void static_for_pk(F &&f) {
  static_for_pk_impl<A>(f, std::make_integer_sequence<int, (B > A ? B - A : 0)>{});
}

// tables indexed by rank, byte p (byte 0 is unused): first the untransposed
// frame (rank 2 up, 1 left), then the transposed one (rank 2 left, 1 up)
constexpr uint32_t kPkTabH[2] = {(27u << 8) | (32u << 16) | (69u << 24), (32u << 8) | (29u << 16) | (70u << 24)};
constexpr uint32_t kPkTabV[2] = {(40u << 8) | (43u << 16) | (2u << 24), (45u << 8) | (40u << 16) | (3u << 24)};

// One wave: 64 / G pairs of bucket KB starting at order[wave * (64 / G)].
// `dirs`: this block's slot of direction words, [step][word of 8 cells][lane].
// `stage`: kPkTraceSteps * pk_dir_words(C) * 64 words of LDS.
template <int C, bool EXT, bool F16>
__device__ __forceinline__ void nw_pk_wave(const uint32_t *__restrict__ pack, const uint32_t *__restrict__ pack_hi,
                                           const int64_t *__restrict__ poff,
                                           const int32_t *__restrict__ len, const int2 *__restrict__ pairs,
                                           const uint32_t *__restrict__ order, const int32_t count, const int KB,
                                           const int G, const int wave, uint32_t *__restrict__ dirs,
                                           uint32_t *__restrict__ stage, float *__restrict__ out) {
  constexpr int ND = pk_dir_words(C);
  constexpr int NB = (2 * C - 1 + 31) / 32;  // window words per plane
  constexpr int NLO = (C + 31) / 32;         // of them: the low half's cells
  constexpr int NQ = (C + 15) / 16;          // match words, 16 cells of each half
  const int lane = threadIdx.x & 63;
  const int groups = 64 / G;
  const int grp = lane / G;
  const int g = lane - grp * G;
  const int slot = wave * groups + grp;
  const bool has_pair = grp < groups && slot < count;
  const uint32_t pidx = order[has_pair ? slot : count - 1];
  const int2 pr = pairs[pidx];
  const int La = len[pr.x], Lb = len[pr.y];
  // rows over the shorter read; with rows over the reference's read 1 the
  // frame is transposed: "left" (previous row) wins gap ties
  const bool tr = La <= Lb;
  const int64_t o1 = poff[tr ? pr.y : pr.x], o2 = poff[tr ? pr.x : pr.y];  // columns, rows
  const int L1 = tr ? Lb : La;
  const int R = tr ? La : Lb;  // the shorter read: every row of it has in-band cells
  const uint32_t tabH = tr ? kPkTabH[1] : kPkTabH[0], tabV = tr ? kPkTabV[1] : kPkTabV[0];
  const uint32_t rank_left = tr ? 2u : 1u;
  const int W = 2 * KB + 1;
  const int V = 2 * G;  // V C >= W + 1: W is odd
  const int off = 7 * (V * C - KB) + 32;  // keys of every computed cell are positive
  const bool is_end = g == G - 1;
  const int nw1 = (L1 + 15) >> 4, nw2 = (R + 15) >> 4;

  // wave-uniform step ranges
  int tm = has_pair ? R + 2 * g + 1 : 0;
  int l1m = has_pair ? L1 : 0x7fffffff, rm = has_pair ? R : 0x7fffffff;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    tm = max(tm, __shfl_xor(tm, o, 64));
    l1m = min(l1m, __shfl_xor(l1m, o, 64));
    rm = min(rm, __shfl_xor(rm, o, 64));
  }
  const int tmax = __builtin_amdgcn_readfirstlane(tm);
  const int L1min = __builtin_amdgcn_readfirstlane(l1m);
  const int Rmin = __builtin_amdgcn_readfirstlane(rm);

  // masks: 0 from the left neighbour of the pair's first lane and the right
  // neighbour of its last, and on the first position past the band (position W,
  // virtual lane W / C), where the last real cell has no "left"
  const uint32_t first_mask = g > 0 ? ~0u : 0u, last_mask = is_end ? 0u : ~0u;
  const int dead_v = W / C, dead_k = W - dead_v * C;
  // (its lanes by execution mask and its cell by masks in scalar registers: a
  // vector mask was spilled, and its reload in every step waited for the
  // direction stores; choosing the cell by branches moved the row's registers.
  // Of the same kind and still there: the plain steps of the 1-16 and 25-32
  // families reload the store's 64-bit address from scratch.)
  const bool dead_lane = g == dead_v >> 1;
  const uint32_t dead_half = dead_v & 1 ? 0x0000FFFFu : 0xFFFF0000u;
  uint32_t dead_near[4];  // cells C - 1, - 3, - 5, - 7: where W / (2 G) leaves it mostly
#pragma unroll
  for (int o = 0; o < 4; ++o)
    dead_near[o] = (uint32_t)__builtin_amdgcn_readfirstlane((int)(C - dead_k == 2 * o + 1 ? dead_half : ~0u));
  const bool dead_far = (C - dead_k) % 2 == 0 || C - dead_k > 7;

  // row 0: M 0 at every position (positions with j < 0 are computed but never
  // read by a cell of the matrix: the boundary cells are set below)
  uint32_t Kd[C], Kv[C];
  auto row0 = [&](const int d) -> uint32_t { return (uint32_t)(4 * (off - 7 * (d - KB))); };
  const int dlo = 2 * g * C, dhi = dlo + C;
#pragma unroll
  for (int k = 0; k < C; ++k) {
    const uint32_t b = row0(dlo + k) | (row0(dhi + k) << 16);
    Kd[k] = b | 0x00030003u;
    Kv[k] = b + 0x00010001u * (44u + rank_left);
  }
  auto mask_dead = [&]() {
    if (dead_lane)
      static_for_pk<0, 4>([&](auto O) {
        constexpr int k = C - 1 - 2 * decltype(O)::value;
        if constexpr (k >= 0) Kv[k >= 0 ? k : 0] &= dead_near[decltype(O)::value];
      });
    if (dead_far) {  // wave-uniform
      asm volatile("");  // a branch, not selects in every step
      static_for_pk<0, C>([&](auto K) {
        constexpr int k = decltype(K)::value;
        if constexpr ((C - k) % 2 == 0 || C - k > 7)
          if (dead_lane) Kv[k] &= k == dead_k ? dead_half : ~0u;
      });
    }
  };
  mask_dead();

  // Column window, two bit planes: bit b at step t is base t - 2g + 2gC - kB -
  // 1 + b of the column read; the low half's cell k reads bit k, the high
  // half's (one row behind, C positions on) bit C - 1 + k.  Row bases: step t's
  // low row t - 2g; the high half's row is the low half's of the step before.
  // EXT: two more planes, the upper code bits of reads with other bytes.
  constexpr int NP = EXT ? 4 : 2;
  uint32_t B[NP][NB];
  PkStream cs[NP / 2], rs[NP / 2];
#pragma unroll
  for (int p = 0; p < NP / 2; ++p) {
    const uint32_t *src = p ? pack_hi : pack;
    cs[p].open(src + o1, has_pair ? nw1 : 0, dlo - 2 * g - KB);
    rs[p].open(src + o2, has_pair ? nw2 : 0, -2 * g);
#pragma unroll
    for (int w = 0; w < NB; ++w) {
      const uint32_t a = cs[p].next(), b = cs[p].next();
      B[2 * p][w] = pk_even(a) | (pk_even(b) << 16);
      B[2 * p + 1][w] = pk_even(a >> 1) | (pk_even(b >> 1) << 16);
    }
  }
  uint32_t F[NP], Rw[NP];  // the next bases of both streams
  uint32_t rm_[NP];        // the low row's base, a mask per plane
#pragma unroll
  for (int p = 0; p < NP; ++p) F[p] = Rw[p] = rm_[p] = 0;
  uint32_t upw = 0;                         // "up" of the first cells
  int bestJ = kNeg, bestJr = 0;             // last column: M (in the column's frame), row

  // boundary cell (i, 0) of step t: position kB - i in virtual lane vt, cell
  // kt = (kB - t) mod (C - 1), vt = (kB - t) / (C - 1)
  int kt = 0, vt = -1;
  if (C > 1 && KB >= 1) {
    vt = (KB - 1) / (C - 1 > 0 ? C - 1 : 1);
    kt = (KB - 1) % (C - 1 > 0 ? C - 1 : 1);
  }
  uint32_t *dst = dirs;  // wave-uniform

  auto step = [&](const int t, auto top_tag, auto cap_tag) {
    constexpr bool TOP = decltype(top_tag)::value, CAP = decltype(cap_tag)::value;
    if (((t - 1) & 15) == 0) {
#pragma unroll
      for (int p = 0; p < NP / 2; ++p) {
        const uint32_t c = cs[p].next(), r = rs[p].next();
        F[2 * p] = pk_even(c);
        F[2 * p + 1] = pk_even(c >> 1);
        Rw[2 * p] = pk_even(r);
        Rw[2 * p + 1] = pk_even(r >> 1);
      }
    }
    const int ilo = t - 2 * g, ihi = ilo - 1;
    uint32_t hm[NP];  // the high half's row base
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      hm[p] = rm_[p];
      rm_[p] = (uint32_t)__builtin_amdgcn_sbfe((int)Rw[p], 0, 1);
      Rw[p] >>= 1;
    }
    // match words: 16 cells of the low half below 16 of the high half
    uint32_t ml[NLO], mh[NB], mm[NQ];
    auto match = [&](const int w, const uint32_t (&r)[NP]) {
      uint32_t x = (B[0][w] ^ r[0]) | (B[1][w] ^ r[1]);
      if constexpr (EXT) x |= (B[2][w] ^ r[2]) | (B[3][w] ^ r[3]);
      return ~x;
    };
#pragma unroll
    for (int w = 0; w < NLO; ++w) ml[w] = match(w, rm_);
#pragma unroll
    for (int w = (C - 1) / 32; w < NB; ++w) mh[w] = match(w, hm);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int b = C - 1 + 16 * q, w = b / 32, o = b % 32;
      uint32_t h;
      if (o == 0)
        h = mh[w];
      else if (o > 16 && w + 1 < NB)
        h = __builtin_amdgcn_alignbit(mh[w + 1 < NB ? w + 1 : w], mh[w], o);
      else
        h = mh[w] >> o;
      mm[q] = __builtin_amdgcn_perm(h, ml[q / 2], q & 1 ? 0x05040302u : 0x05040100u);
    }
    const bool active = has_pair && ilo >= 1 && ihi <= R;
    const uint32_t keep_lo = CAP && ilo > R ? 0x0000FFFFu : 0u;  // the low half has ended: its last row stays
    const int kc_lo = CAP ? L1 - ilo + KB - dlo : 0, kc_hi = CAP ? kc_lo + 1 - C : 0;
    uint32_t up = upw, acc = 0, grpw = 0;
    auto cell = [&](auto K, const uint32_t left) {
      constexpr int k = decltype(K)::value;
      constexpr int r = (k & 15) == 15 ? 0 : (k & 15) % 3;
      if constexpr (r == 0) grpw = mm[k >> 4] >> (k & 15);
      const uint32_t dg = pk_mad(grpw & (0x00010001u << r), (unsigned short)(36 >> r), Kd[k]);
      uint32_t Wk = pk_max3<F16>(dg, left, up);
      if constexpr (TOP) {
        if (k == kt || (k == C - 1 && kt == 0)) {  // wave-uniform
          const int v = k == kt ? vt : vt - 1;
          if (v >= 0 && g == v >> 1) {
            const uint32_t b = (uint32_t)(4 * (11 * (t - v) + off)) + rank_left;  // (i, 0): M 0, no gap penalty
            Wk = v & 1 ? (Wk & 0x0000FFFFu) | (b << 16) : (Wk & 0xFFFF0000u) | b;
          }
        }
      }
      const uint32_t x = Wk & 0x00030003u;
      up = Wk - __builtin_amdgcn_perm(0u, tabH, x);
      Kv[k] = Wk + __builtin_amdgcn_perm(0u, tabV, x);
      if constexpr (CAP)
        Kd[k] = (Kd[k] & keep_lo) | ((Wk | 0x00030003u) & ~keep_lo);
      else
        Kd[k] = Wk | 0x00030003u;
      // here, not sunk into the next row (which would keep W and the rank
      // alive beside them) nor hoisted over the other cells
      asm volatile("" : "+v"(Kv[k]), "+v"(Kd[k]));
      acc = k & 7 ? (acc << 2) | x : x;
      asm volatile("" : "+v"(acc));  // one v_lshl_or_b32 per cell
      if constexpr ((k & 7) == 7 || k == C - 1) dst[(k >> 3) * 64 + lane] = acc;
    };
    const uint32_t kv0_old = Kv[0];
    if (active) {
      cell(std::integral_constant<int, 0>{}, C > 1 ? Kv[C > 1 ? 1 : 0] : 0u);
      if constexpr (TOP) {
        // the high half starts a step later: its row 0 stays
        if (ihi == 0) Kv[0] = (Kv[0] & 0x0000FFFFu) | (kv0_old & 0xFFFF0000u);
      }
      // the left neighbour reads it in this step
      if (dead_k == 0 && dead_lane) Kv[0] &= dead_half;
    }
    // "left" of the last cells: the high half's first offer for the low half,
    // the next lane's low half's for the high half
    const uint32_t nk = (uint32_t)__builtin_amdgcn_update_dpp((int)Kv[0], (int)Kv[0], 0x130, 0xF, 0xF, false);
    const uint32_t leftw = __builtin_amdgcn_alignbit(nk & last_mask, Kv[0], 16);
    if (active) {
      static_for_pk<1, C>([&](auto K) {
        constexpr int k = decltype(K)::value;
        if constexpr (k == C - 1)
          cell(K, leftw);
        else
          cell(K, Kv[k + 1 < C ? k + 1 : k]);
      });
      mask_dead();
      if constexpr (TOP) {
        if (ihi == 0) {  // the high half's row 0 again
          uint32_t b0 = row0(dhi);
          asm volatile("" : "+v"(b0));  // opaque: 2 C hoisted constants would spill
#pragma unroll
          for (int k = 0; k < C; ++k) {
            const uint32_t b = b0 - 28u * k;
            Kd[k] = (Kd[k] & 0x0000FFFFu) | ((b | 3u) << 16);
            Kv[k] = (Kv[k] & 0x0000FFFFu) | ((b + 44u + rank_left) << 16);
          }
          mask_dead();
        }
      }
      if constexpr (CAP) {
        // the cells of column L1, by a per-lane index: the row goes through LDS
        // (bank = lane, no VALU work), where selecting them in registers cost
        // a compare per cell
#pragma unroll
        for (int k = 0; k < C; ++k) stage[k * 64 + lane] = Kd[k];
        if (kc_lo >= 0 && kc_lo < C && ilo <= R && ilo >= L1 - KB) {
          const int m = (int)((stage[kc_lo * 64 + lane] >> 2) & 0x3FFFu) - 11 * ilo;
          if (m > bestJ || (m == bestJ && ilo > bestJr)) {
            bestJ = m;
            bestJr = ilo;
          }
        }
        if (kc_hi >= 0 && kc_hi < C && ihi >= 1 && ihi >= L1 - KB) {
          const int m = (int)(stage[kc_hi * 64 + lane] >> 18) - 11 * ihi;
          if (m > bestJ || (m == bestJ && ihi > bestJr)) {
            bestJ = m;
            bestJr = ihi;
          }
        }
      }
    }
    // "up" of the next step's first cells: the low half's last offer for the
    // high half, the previous lane's high half's for the low half
    const uint32_t nu = (uint32_t)__builtin_amdgcn_update_dpp((int)up, (int)up, 0x138, 0xF, 0xF, false);
    upw = __builtin_amdgcn_alignbit(up, nu & first_mask, 16);
    dst += ND * 64;
    // slide both windows by one base
#pragma unroll
    for (int p = 0; p < NP; ++p) {
#pragma unroll
      for (int w = 0; w < NB - 1; ++w) B[p][w] = __builtin_amdgcn_alignbit(B[p][w + 1], B[p][w], 1);
      B[p][NB - 1] = __builtin_amdgcn_alignbit(F[p], B[p][NB - 1], 1);
      F[p] >>= 1;
    }
    if constexpr (TOP) {
      if (--kt < 0) {
        kt = C - 2;
        --vt;
      }
    }
  };
  // Steps 1..kB hold a boundary cell (and the first 2G the lanes' starts);
  // column L1 enters the band at row L1 - kB in the virtual lane of the last
  // position, and the first low half passes its last row at step Rmin + 1.
  const int top_end = min(max(KB, V), tmax);
  const int cap_from = min(max(L1min - KB + (W - 1) / C, 1), Rmin + 1);
  const int top_plain_end = min(top_end, cap_from - 1);
  const int mid_end = max(top_end, min(tmax, cap_from - 1));
  int t = 1;
  for (; t <= top_plain_end; ++t) step(t, std::true_type{}, std::false_type{});
  for (; t <= top_end; ++t) step(t, std::true_type{}, std::true_type{});
  for (; t <= mid_end; ++t) step(t, std::false_type{}, std::false_type{});
  for (; t <= tmax; ++t) step(t, std::false_type{}, std::true_type{});

  // Last row (both halves still hold row R): the last maximum over 1 <= j <= L1
  int bestI = kNeg, bestIj = 0;
  if (has_pair) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int j0 = R - KB + dlo + h * C;
#pragma unroll
      for (int k = 0; k < C; ++k) {
        const int j = j0 + k;
        const int m = (int)((Kd[k] >> (16 * h + 2)) & 0x3FFFu) + 7 * j;
        if (j >= 1 && j <= L1 && dlo + h * C + k < W && m >= bestI) {
          bestI = m;
          bestIj = j;
        }
      }
    }
  }
  // the pair's G lanes: the last maximum has the larger j (row)
  int mI = bestI, mIj = bestIj, mJ = bestJ, mJr = bestJr;
  for (int q = 1; q < G; ++q) {
    const int src = grp * G + (g + q) % G;
    const int oI = __shfl(bestI, src, 64), oj = __shfl(bestIj, src, 64);
    const int oJ = __shfl(bestJ, src, 64), orow = __shfl(bestJr, src, 64);
    if (oI > mI || (oI == mI && oj > mIj)) mI = oI, mIj = oj;
    if (oJ > mJ || (oJ == mJ && orow > mJr)) mJ = oJ, mJr = orow;
  }
  // M of both: last row M = m - 11 R - off, last column M = m + 7 L1 - off
  if (mI > kNeg) mI -= 11 * R + off;
  if (mJ > kNeg) mJ += 7 * L1 - off;
  // the reference takes its last row's best only when it beats its last
  // column's (genCPU.cpp:461-464); transposed, those are this frame's last
  // column and last row
  const bool row_end = tr ? !(mJ > mI) : mI > mJ;
  const int ei = row_end ? R : mJr, ej = row_end ? mIj : L1, eM = row_end ? mI : mJ;

  // ---- trace: lane q walks pair q's path from its end cell to the boundary,
  // counting the vertical steps and the gap cost; the path's score then gives
  // its matches.  The directions come back in blocks of kPkTraceSteps steps
  // (coalesced, the next block requested before this one is walked); they were
  // written by this wave, so a wait makes them visible past the vector cache.
  const int from = min(lane, groups - 1) * G;
  const int ti = __shfl(ei, from, 64), tj = __shfl(ej, from, 64), tM = __shfl(eM, from, 64);
  const bool ttr = __shfl((int)tr, from, 64) != 0;
  const uint32_t tpidx = (uint32_t)__shfl((int)pidx, from, 64);
  const int has = __shfl((int)has_pair, from, 64);  // not in the condition: every lane takes part
  bool act = lane < groups && has != 0;
  const bool mine = act;
  const int rank_up = ttr ? 1 : 2;
  int i = ti, j = tj, vert = 0, cost = 0, prev = 0;  // prev: the move that left this cell, 1 up, 2 left
  int v = (tj - ti + KB) / C, k = (tj - ti + KB) - v * C;
  int tt = act ? ti + v : 0;
  int top = tt;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) top = max(top, __shfl_xor(top, o, 64));
  const int tlast = __builtin_amdgcn_readfirstlane(top);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  constexpr int NW = kPkTraceSteps * ND;
  uint32_t pre[NW];
  auto fetch = [&](const int tb) {
#pragma unroll
    for (int q = 0; q < NW; ++q)
      pre[q] = __hip_atomic_load(dirs + (size_t)(tb * ND + q) * 64 + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  int tb = (tlast - 1) / kPkTraceSteps * kPkTraceSteps;
  fetch(tb);
  for (; tb >= 0; tb -= kPkTraceSteps) {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // the wave's own LDS: its operations are in order
#pragma unroll
    for (int q = 0; q < NW; ++q) stage[q * 64 + lane] = pre[q];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (tb > 0) fetch(tb - kPkTraceSteps);
    while (__ballot(act && tt > tb)) {
      if (act && tt > tb) {
        const int c = k >> 3;
        const int nc = c == ND - 1 ? C - 8 * (ND - 1) : 8;
        const int sh = 2 * (nc - 1 - (k & 7)) + 16 * (v & 1);
        const uint32_t *w = stage + ((tt - 1 - tb) * ND + c) * 64 + from + (v >> 1);
        // the diagonal run from here: up to 4 cells of this position, read at once
        const int most = min(min(i, j), tt - tb);
        uint32_t x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = q < most ? w[-q * ND * 64] : 0u;
        const int dir = (int)(x[0] >> sh) & 3;
        if (dir == 3) {
          int n = 1;
          bool on = true;
#pragma unroll
          for (int q = 1; q < 4; ++q) {
            on = on && ((x[q] >> sh) & 3u) == 3u;
            n += on;
          }
          cost += prev ? 10 : 0;
          prev = 0;
          i -= n;
          j -= n;
        } else if (dir == rank_up) {
          cost += prev == 1;
          prev = 1;
          --j;
          if (--k < 0) k = C - 1, --v;
        } else {
          cost += prev == 2;
          prev = 2;
          --i;
          ++vert;
          if (++k == C) k = 0, ++v;
        }
        tt = i + v;
        act = i > 0 && j > 0;
      }
    }
  }
  if (mine) {
    const int diag = ti - i - vert;
    const int match = (tM + cost + 4 * diag) / 9;  // M = 5 match - 4 (diag - match) - cost
    const int AL = vert + i + tj;
    const int ML = AL - (i + j) - match;
    out[tpidx] = (float)ML / (float)AL;
  }
}

template <int HI, int C, bool EXT, bool F16>
__device__ __forceinline__ void pk_dispatch(const int c, const NwFusedArgs &a, const PkLaunchArgs &x,
                                            const uint32_t *order, int32_t count, int kb, int G, int wave,
                                            uint32_t *dirs, uint32_t *stage) {
  if constexpr (C <= HI) {
    if (c == C) {
      nw_pk_wave<C, EXT, F16>(a.pack, x.pack_hi, a.poff, a.len, a.pairs, order, count, kb, G, wave, dirs, stage, a.out);
      return;
    }
    pk_dispatch<HI, C + 1, EXT, F16>(c, a, x, order, count, kb, G, wave, dirs, stage);
  }
}

// Packed kernel for slice widths LO..HI (family F).  The grid is the number
// of direction slots (about the waves the chip holds), so the scratch is
// bounded whatever the pair count: a wave keeps its slot and takes the
// family's tasks one after the other, longest first: its slot's number, then
// what a device counter gives out.
// Blocks of one wave, or of kPkBlockWaves = 4 independent ones (pk_plan in nw.hip).
template <int LO, int HI, int WAVES, int F, bool EXT, bool F16>
__global__ __launch_bounds__(64 * kPkBlockWaves, WAVES) void nw_pk_fused_kernel(const NwFusedArgs a,
                                                                                const PkLaunchArgs x) {
  constexpr int kStage = kPkTraceSteps * pk_dir_words(HI) * 64;
  extern __shared__ uint32_t stages[];  // kStage words per wave
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const uint32_t slot = blockIdx.x * (blockDim.x >> 6) + (uint32_t)wv;
  uint32_t *stage = stages + wv * kStage;
  uint32_t *dirs = x.dirs + (int64_t)slot * x.words;
  NwPlan *plan = a.plan;
  const uint32_t ntasks = plan->ntasks[F];
  const int nbk = (int)plan->nbuckets[F];
  const uint2 *list = plan->list[F];
  uint32_t t = slot;
  while (t < ntasks) {
    int k = 0;
    for (int base = 0; base < nbk; base += 64) {
      const int e = base + (int)(threadIdx.x & 63);
      k += __popcll(__ballot(e < nbk && list[e].y <= t));
    }
    const uint2 e = list[k - 1];
    const int kb = __builtin_amdgcn_readfirstlane((int)e.x);
    const uint2 bk = plan->btab[kb];
    const int G = pk_lanes(kb, x.cap);
    const uint32_t per = 64u / (uint32_t)G;
    const uint32_t waves = (bk.y + per - 1) / per;
    const int wave = __builtin_amdgcn_readfirstlane((int)(waves - 1 - (t - e.y)));
    pk_dispatch<HI, LO, EXT, F16>(pk_cells(kb, x.cap), a, x, a.order + bk.x, (int32_t)bk.y, kb, G, wave, dirs, stage);
    uint32_t n = 0;
    if ((threadIdx.x & 63) == 0) n = atomicAdd(&plan->next[F], 1u);
    t = gridDim.x * (blockDim.x >> 6) + (uint32_t)__builtin_amdgcn_readfirstlane((int)n);
  }
}

template <int P>
inline void launch_nw_pk_family(hipStream_t s, unsigned slots, const NwFusedArgs &a, const PkLaunchArgs &k) {
  constexpr PkFamily fam = kPkFamilies[P];
  const unsigned blocks = slots / k.block_waves, threads = 64 * k.block_waves;
  const size_t lds = sizeof(uint32_t) * kPkTraceSteps * pk_dir_words(fam.hi) * 64 * k.block_waves;
  if (k.pack_hi)
    nw_pk_fused_kernel<fam.lo, fam.hi, fam.ext_waves, kFirstPkFamily + P, true, false>
        <<<blocks, threads, lds, s>>>(a, k);
  else if (k.f16)
    nw_pk_fused_kernel<fam.lo, fam.hi, fam.waves, kFirstPkFamily + P, false, true><<<blocks, threads, lds, s>>>(a, k);
  else
    nw_pk_fused_kernel<fam.lo, fam.hi, fam.waves, kFirstPkFamily + P, false, false><<<blocks, threads, lds, s>>>(a, k);
}

}  // namespace crispy
