// Producer / consumer kernel for small and mid-size numbers of activation rows (1 .. ~700) on gfx950.
//
// Orientation, operands and epilogue values are those of kernels_tiled.hip: the MFMA A operand is fed with weight rows, the B
// operand with activation rows. The gated kernel keeps W13's interleaved rows as they lie: of the four consecutive weight rows
// that an accumulator lane owns two are "up" and two "gate" rows of the same two features, so the gating (swiglu.cu:380-381) is
// per-lane arithmetic without a de-interleave, and a tile may hold any multiple of 32 weight rows.
//
// What bounds it: the copies. A compute unit fetches 136 bytes per ns from the L2, but 45 .. 57 when an activation line and a weight line
// from HBM are asked for in turn: its loads return in order through its 32 KB L1, whose 256 lines are all it can have under way, so a
// line that the L2 has at once holds its place for as long as the weight line ahead of it takes. (Copies alone, 64 weight rows from HBM and
// 224 activation rows from the L2 a step, 8 KB rows: 42 us for 64 steps; weights two steps at a time 32 us; four 32 us. Without the 224
// rows 20 us.) So weight lines are asked for in PAIRS where a tile holds more than 64 activation rows, and what the chip shares once a
// line of weights takes longer than its activations is HBM. The tile follows from both: any height of 32 weight rows and any multiple of
// 32 activation rows, chosen by an estimate (mid_plan) so that one round of compute units shares the work with as few lines each as
// possible.
//   * Four waves copy (global -> LDS, buffer_load ... lds) and four multiply. A copying wave may stall on a full memory queue
//     without holding back an MFMA, and the multiplying waves need no wait for copies of their own: one barrier per K tile of 64
//     hands a line over and its predecessor's slot back.
//   * LINES, not K tiles. A row is fetched in whole, aligned 128-byte lines wherever it starts. With rows that are no multiple of
//     128 bytes long (K % 64 != 0) a K tile of a row lies in two lines, at a shift that depends on the row; the slot of a line
//     keeps the line as it is, and a fragment read picks, per lane, the slot of this line or the next (ph = 1: one more line has
//     to be there). Fetched by K tiles instead every line crosses L2 -> L1 twice, and twice from HBM when non-temporal: gate/up
//     38880 x 5800, 40 rows 139.7 -> 69.5 us; 16016 x 3000, 100 rows 36.6 -> 23.7, 20 rows 26.4 -> 18.9; down 19440 -> 5800, 20
//     rows 74.1 -> 38.2, 130 rows 76.7 -> 58.6. Aligned rows gain by the tile: gate/up 22016 x 4096, 130 rows 50.4 -> 42.9;
//     16384 x 2048, 40 rows 20.3 -> 12.9; down 13824 -> 5120, 16 rows 37.5 -> 26.0, 200 rows 61.9 -> 51.8.
//   * Two rings, NW weight lines and NA activation lines. Step kt takes line kt of both; activation line kt + NA - 1 is asked for at its
//     start, weight lines kt + NW - 2 and kt + NW - 1 together at every second one (G = 2; G = 1: line kt + NW - 1). Against one ring of both,
//     line by line, same values bit for bit, us: gate/up 22016 x 4096, 160 rows 43.4 -> 38.8, 16016 x 3000, 200 rows 34.4 -> 29.2, 28672 x
//     4096, 128 rows 46.8 -> 43.6, 46128 x 8096, 162 rows 187 -> 163; down 8008 -> 3000, 200 rows 26.0 -> 24.4. Two rings line by line:
//     level. Up to 64 activation rows, where few lines wait behind the weights, pairs gain on whole K (27648 x 5120, 40 rows 47.2 ->
//     46.4) and lose on parts of it (13824 -> 5120, 40 rows 28.9 -> 29.4; 2816 -> 1024, 130 rows 13.4 -> 14.8): G = 1.
//   * The copying waves' own instructions count: lines that lie whole inside K take the row's offset from a register and the line's as the
//     scalar offset, two instructions a copy, against a bounds check and three additions (down 2816 -> 1024, 512 rows 14.3 -> 12.4).
//   * LDS: slots of [rows][128 bytes]; chunk c of row r of a line at position c ^ ((r >> 1) &
//     7). The 16 rows that a fragment read touches cover the 64 banks once, shifted or not: for even (and for odd) rows the
//     position ((c + shift of the row) & 7) ^ (r >> 1) is a permutation, since the shift grows by an even number of chunks from
//     one such row to the next.
// Measured and not taken: eight multiplying waves, fragments of the next K tile read while this one is multiplied, two waves of a
// block with half of every K tile each (all level within 2 % or slower), weight lines of a pair ahead of the activation line (3 .. 10 %
// slower), weight lines brought to the L2 by scalar loads first (twice the time).
#pragma once
#include <type_traits>

#include "fsw_internal.h"
#include "fsw_device.h"

namespace fsw {

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((ext_vector_type(2))) float f32x2;

// Wait until at most N copies are outstanding (the counter holds 63).
template <int N>
__device__ __forceinline__ void wait_copies() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 0 ? 0 : N < 63 ? N : 63) : "memory");
}

// four packed 16-bit features n .. n + 3 of a row of the output
__device__ __forceinline__ void store4(int n, int nout, bool vec, unsigned lo, unsigned hi, unsigned short* row) {
  if (vec && n + 3 < nout) {
    *(u32x2*)(row + n) = u32x2{lo, hi};
  } else {
    if (n < nout) row[n] = (unsigned short)lo;
    if (n + 1 < nout) row[n + 1] = (unsigned short)(lo >> 16);
    if (n + 2 < nout) row[n + 2] = (unsigned short)hi;
    if (n + 3 < nout) row[n + 3] = (unsigned short)(hi >> 16);
  }
}

// Copies that a wave has asked for by the end of step kt (kt % 2 == parity) behind the last line that step kt + 1 reads: line kt + 1, or
// kt + 2 with rows that are no whole lines (ph). lp, lq: the wave's copies of a weight and of an activation line.
constexpr int copies_behind(int parity, int ph, int g, int nw, int na, int lp, int lq) {
  const int kt = 64 + parity, need = kt + 1 + ph;
  int behind = 0;
  for (int s = 0; s <= kt; ++s) {
    behind += lq;
    if (lq > 0 && s + na - 1 == need) behind = 0;
    for (int j = g; s % g == 0 && j >= 1; --j) {
      behind += lp;
      if (lp > 0 && s + nw - j == need) behind = 0;
    }
  }
  return behind;
}

// bits of the kernel's `how`
constexpr int MID_STREAM = 1;  // weight lines are non-temporal
constexpr int MID_SPREAD = 2;  // workgroups start their walk over K at different lines

template <class E, bool GATED, int FP, int FQ, int PAIRS, int NW, int NA>
__global__ void __launch_bounds__(512)
mid_kernel(const GemmArgs a, const int tiles_p, const int tiles_q, const int group, const int ph, const int how) {
  constexpr int NC = 4;
  constexpr int WP = 2, WQ = 2, BP = WP * FP * 16, BQ = WQ * FQ * 16;
  constexpr int LP = BP / 32, LQ = BQ / 32;
  constexpr int WLINE = BP * 128, ALINE = BQ * 128;
  constexpr int ABASE = NW * WLINE;
  static_assert(NW >= 4 && NA >= 3 && NW * WLINE + NA * ALINE <= 160 * 1024, "LDS budget of a gfx950 CU");
  static_assert(BP % 32 == 0 && BQ % 32 == 0, "copy mapping");
  __shared__ __align__(1024) unsigned char lds[NW * WLINE + NA * ALINE];

  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int tp, tq;
  tile_coords(blockIdx.x, tiles_p, tiles_q, group, tp, tq);
  const int step_p = (a.tile_p > 0 && a.tile_p < BP) ? a.tile_p : BP;
  const int p0 = tp * step_p;
  const int p_end = p0 + step_p < a.np ? p0 + step_p : a.np;
  const int q0 = tq * BQ;
  if (GATED && blockIdx.x == 0 && blockIdx.y == 0)
    for (int i = t; i < a.n_zero_words; i += (NC + 4) * 64) a.zero_words[i] = 0u;
  const int nkt_all = (a.k + 63) / 64;
  const int kt_per = (nkt_all + a.splits - 1) / a.splits;
  const int kt0 = (int)blockIdx.y * kt_per;
  const int nkt = nkt_all - kt0 < kt_per ? (nkt_all - kt0 > 0 ? nkt_all - kt0 : 0) : kt_per;
  const int rot = (how & MID_SPREAD) && nkt > 1 ? (int)(((unsigned)blockIdx.x * 2654435761u >> 12) % (unsigned)nkt) : 0;
  const unsigned char* pbase = (const unsigned char*)a.P + (long long)p0 * a.ldp * 2;
  const unsigned char* qbase = (const unsigned char*)a.Q + (long long)q0 * a.ldq * 2;

  // The copies start the launch: where few rows leave little else to do their code goes first, next to the prologue (behind the epilogue it
  // is fetched into the instruction cache later: gate/up 9216 x 1280, 22 rows 8.1 -> 7.9 us). Not on wider tiles (5632 x 1024, 130 rows 8.8 ->
  // 9.2, 512 rows 10.1 -> 10.4).
  if (FQ <= 2 ? __builtin_expect(wave >= NC, 1) : wave >= NC) {
    // ---- producers
    const int u = t - NC * 64;
    const int rb = u >> 3, pos = (u & 7) ^ ((rb >> 1) & 7);
    const __amdgpu_buffer_rsrc_t prs = make_rsrc(pbase, ((long long)(p_end - p0 - 1) * a.ldp + a.k) * 2);
    const __amdgpu_buffer_rsrc_t qrs = make_rsrc(qbase, ((long long)(a.nq - q0 - 1) * a.ldq + a.k) * 2);
    const int ap = ph ? (int)((((uintptr_t)pbase >> 4) + (unsigned)rb * ((unsigned)a.ldp >> 3)) & 7) : 0;
    const int aq = ph ? (int)((((uintptr_t)qbase >> 4) + (unsigned)rb * ((unsigned)a.ldq >> 3)) & 7) : 0;
    const int cp = pos - ap, cq = pos - aq;  // logical chunk of line 0 this lane fetches
    const int c_lo = kt0 * 8, c_all = a.k >> 3;
    const int c_hi = (kt0 + nkt) * 8 < c_all ? (kt0 + nkt) * 8 : c_all;
    unsigned char* const lw = lds + (wave - NC) * 1024;
    const int nline = nkt + ph;
    auto line_of = [&](int l) -> int {
      int r = l + rot;
      if (r >= nkt && rot > 0) r -= nkt;
      return kt0 + r;
    };
    // CP, CQ: copies of a weight and of an activation line that this wave has rows for
    auto produce = [&](auto cp_c, auto cq_c, auto g_c) __attribute__((always_inline)) {
      constexpr int CP = decltype(cp_c)::value, CQ = decltype(cq_c)::value, G = decltype(g_c)::value;
      // Line by line on a ring made for pairs (short K): five lines ahead. The first lines of a launch wait for the copies asked for beside
      // them (six lines -> five, us: gate/up 5632 x 1024, 189 rows 9.1 -> 8.8; down 2816 -> 1024, 540 rows 14.0 -> 13.5; 120 calls 0.989).
      constexpr int LW = PAIRS == 2 && G == 1 && NW > 5 ? 5 : NW;
      // A lane's offsets of line `ph` (the row's part and the chunk's), which stay; a line adds its distance from that one as the scalar offset
      unsigned poff[CP + 1], qoff[CQ + 1];
#pragma unroll
      for (int i = 0; i < CP; ++i)
        poff[i] = rb + 32 * i < p_end - p0 ? (unsigned)(rb + 32 * i) * (unsigned)a.ldp * 2u + (unsigned)(cp * 16 + ph * 128) : OOB_OFFSET;
#pragma unroll
      for (int i = 0; i < CQ; ++i)
        qoff[i] = rb + 32 * i < a.nq - q0 ? (unsigned)(rb + 32 * i) * (unsigned)a.ldq * 2u + (unsigned)(cq * 16 + ph * 128) : OOB_OFFSET;
      // masked: lines that have chunks out of the range of K (the first and last of a row) or lie past the end; others are whole
      auto issue_w = [&](int l, int slot, auto masked) __attribute__((always_inline)) {
        const int L = line_of(l);
        const bool in = l < nline && 8 * L + cp >= c_lo && 8 * L + cp < c_hi;
        const int rel = (L - ph) * 128;
        unsigned char* const st = lw + slot * WLINE;
#define FSW_MID_COPY(RSRC, OFF, I, AUX)                                                                                      \
  if constexpr (decltype(masked)::value)                                                                                     \
    __builtin_amdgcn_raw_ptr_buffer_load_lds(RSRC, (lds_void*)(st + (I) * 32 * 128), 16,                                     \
                                             (int)(in ? (OFF) + (unsigned)rel : OOB_OFFSET), 0, 0, AUX);                     \
  else                                                                                                                       \
    __builtin_amdgcn_raw_ptr_buffer_load_lds(RSRC, (lds_void*)(st + (I) * 32 * 128), 16, (int)(OFF), rel, 0, AUX)
        if (how & MID_STREAM) {
#pragma unroll
          for (int i = 0; i < CP; ++i) { FSW_MID_COPY(prs, poff[i], i, 2); }
        } else {
#pragma unroll
          for (int i = 0; i < CP; ++i) { FSW_MID_COPY(prs, poff[i], i, 0); }
        }
      };
      auto issue_a = [&](int l, int slot, auto masked) __attribute__((always_inline)) {
        const int L = line_of(l);
        const bool in = l < nline && 8 * L + cq >= c_lo && 8 * L + cq < c_hi;
        const int rel = (L - ph) * 128;
        unsigned char* const st = lw + ABASE + slot * ALINE;
#pragma unroll
        for (int i = 0; i < CQ; ++i) { FSW_MID_COPY(qrs, qoff[i], i, 0); }
#undef FSW_MID_COPY
      };
      int ws = LW % NW, as = 0;  // slots that the next weight and activation lines take
      if (nkt > 0) {
        // the issues of the steps before the first, in the order of the loop
#pragma unroll
        for (int s = -(NA > LW ? NA : LW); s <= 0; ++s) {
          if (s + NA - 1 >= 0) issue_a(s + NA - 1, s + NA - 1, std::true_type{});
#pragma unroll
          for (int j = G; s % G == 0 && j >= 1; --j)
            if (s + LW - j >= 0) issue_w(s + LW - j, s + LW - j, std::true_type{});
        }
        if (ph) wait_copies<copies_behind(1, 1, G, LW, NA, CP, CQ) + CQ + G * CP>();
        else wait_copies<copies_behind(1, 0, G, LW, NA, CP, CQ) + CQ + G * CP>();
      }
      int kt = 0;
      // step kt + u (u = 0, 1): line kt + u - 1 has been multiplied: its slots take later lines, weights G lines at once
      auto step = [&](int u, auto masked) __attribute__((always_inline)) {
        asm volatile("s_barrier" ::: "memory");
        if (u == 1 || kt > 0) {
          issue_a(kt + u + NA - 1, as, masked);
          as = as + 1 == NA ? 0 : as + 1;
#pragma unroll
          for (int j = G; u % G == 0 && j >= 1; --j) {
            issue_w(kt + u + LW - j, ws, masked);
            ws = ws + 1 == NW ? 0 : ws + 1;
          }
        }
        if (u == 0) {
          if (ph) wait_copies<copies_behind(0, 1, G, LW, NA, CP, CQ)>();
          else wait_copies<copies_behind(0, 0, G, LW, NA, CP, CQ)>();
        } else {
          if (ph) wait_copies<copies_behind(1, 1, G, LW, NA, CP, CQ)>();
          else wait_copies<copies_behind(1, 0, G, LW, NA, CP, CQ)>();
        }
      };
      // Lines behind the prologue's and before this one are whole: all, or those before the line that K ends in (ph: before the last, too)
      const int whole = ph ? nkt - 1 : (a.k & 63) != 0 && kt0 + nkt == nkt_all ? nkt - 1 - rot : nkt;
      constexpr int AHEAD = NA > LW - 1 + (G == 1) ? NA : LW - 1 + (G == 1);
      for (; kt + AHEAD < whole; kt += 2) {
        step(0, std::false_type{});
        step(1, std::false_type{});
      }
      for (; kt < nkt; kt += 2) {
        step(0, std::true_type{});
        if (kt + 1 < nkt) step(1, std::true_type{});
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    // A copy covers 8 rows. Where the matrix or the piece ends before them the wave leaves its last copy of a line out: out of range it would
    // write zeros, which only products that nobody stores take, in the time of a line that the L2 has (130 rows in a tile of 160: 2 us of 40).
    const int r8 = (wave - NC) * 8 + 32 * (LP - 1), q8 = (wave - NC) * 8 + 32 * (LQ - 1);
    const bool fewer_p = r8 >= p_end - p0, fewer_q = q8 >= a.nq - q0;
    using std::integral_constant;
    auto rows = [&](auto g) __attribute__((always_inline)) {
      if (!fewer_p && !fewer_q) produce(integral_constant<int, LP>{}, integral_constant<int, LQ>{}, g);
      else if (!fewer_p) produce(integral_constant<int, LP>{}, integral_constant<int, LQ - 1>{}, g);
      else if (!fewer_q) produce(integral_constant<int, LP - 1>{}, integral_constant<int, LQ>{}, g);
      else produce(integral_constant<int, LP - 1>{}, integral_constant<int, LQ - 1>{}, g);
    };
    // Two weight lines at once where the tile says so and there are enough to fill the rings a few times (11008 -> 4096 in parts of 22 lines,
    // 75 rows 25.4 us with pairs 26.2, 149 rows 30.6 and 31.9; 8008 -> 3000 in parts of 32, 200 rows 26.0 and 24.4). 22 .. 31 lines, line by
    // line -> pairs: tiles of 128 and more activation rows 0.94 (25 problems, 0.87 .. 1.00; gate/up 16336 x 1520 176 rows 19.4 -> 16.9), of 96
    // 1.01 (19, 0.95 .. 1.04; 31696 x 1976 87 rows 25.5 -> 26.6): one bound for both lies on the safe side. A launch whose last part of K is
    // the only one below it runs that part line by line. Not on rings of four weight lines with rows that are no whole lines: the step before
    // needs the second pair's first line then, one step after it was asked for (40736 x 6928, 349 rows 229 and 271).
    if constexpr (PAIRS == 2) {
      if (nkt >= 32 && (NW > 4 || !ph)) rows(integral_constant<int, 2>{});
      else rows(integral_constant<int, 1>{});
    } else {
      rows(integral_constant<int, 1>{});
    }
    return;
  }

  // ---- consumers
  const int lane = t & 63, r16 = lane & 15, c4 = lane >> 4;
  const int wq = wave % WQ, wp = wave / WQ;
  const int ap = ph ? (int)((((uintptr_t)pbase >> 4) + (unsigned)r16 * ((unsigned)a.ldp >> 3)) & 7) : 0;
  const int aq = ph ? (int)((((uintptr_t)qbase >> 4) + (unsigned)r16 * ((unsigned)a.ldq >> 3)) & 7) : 0;
  unsigned po[2], qo[2];
  bool pn[2], qn[2];  // the chunk lies in the next line
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int pp = 4 * h + c4 + ap, qq = 4 * h + c4 + aq;
    pn[h] = pp >= 8;
    qn[h] = qq >= 8;
    po[h] = (unsigned)(wp * FP * 16 + r16) * 128u + (unsigned)(((pp & 7) ^ ((r16 >> 1) & 7)) * 16);
    qo[h] = (unsigned)(ABASE + (wq * FQ * 16 + r16) * 128) + (unsigned)(((qq & 7) ^ ((r16 >> 1) & 7)) * 16);
  }
  f32x4 acc[FP][FQ];
#pragma unroll
  for (int f = 0; f < FP; ++f)
#pragma unroll
    for (int g = 0; g < FQ; ++g) acc[f][g] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 pf[2][FP], qf[2][FQ];
  unsigned wcur = 0, acur = 0;
  auto read_half = [&](int h, unsigned wnxt, unsigned anxt) {
    const unsigned char* pb = lds + po[h] + (pn[h] ? wnxt : wcur);
    const unsigned char* qb = lds + qo[h] + (qn[h] ? anxt : acur);
#pragma unroll
    for (int f = 0; f < FP; ++f) pf[h][f] = *(const u32x4*)(pb + f * 16 * 128);
#pragma unroll
    for (int g = 0; g < FQ; ++g) qf[h][g] = *(const u32x4*)(qb + g * 16 * 128);
  };
  auto mul_half = [&](int h) {
#pragma unroll
    for (int f = 0; f < FP; ++f)
#pragma unroll
      for (int g = 0; g < FQ; ++g) acc[f][g] = E::mfma16(pf[h][f], qf[h][g], acc[f][g]);
  };
  auto multiply = [&](int from, int to) {
    for (int kt = from; kt < to; ++kt) {
      const unsigned wnxt = wcur + WLINE == NW * WLINE ? 0u : wcur + WLINE;
      const unsigned anxt = acur + ALINE == NA * ALINE ? 0u : acur + ALINE;
      // every read of the line before is complete (its slot is refilled behind the barrier), line kt has landed
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      read_half(0, wnxt, anxt);
      read_half(1, wnxt, anxt);
      mul_half(0);
      mul_half(1);
      wcur = wnxt;
      acur = anxt;
    }
  };
  if constexpr (FQ <= 2) {
    // GemmArgs::short_sums (few rows, where a second set of accumulators fits): every four K tiles the sums so far go to the totals and
    // start again, so that no value is the end of one chain of K / 32 sums. Off float64, gate/up unrounded, one chain -> this (skinny_kernel):
    // 27648 x 5120 6.6e-7 -> 2.0e-7 (3.1e-7), 16384 x 2048 4.2e-7 -> 1.6e-7 (1.6e-7). The four is a constant: with chains of an eighth of K the
    // compiler (ROCm 7.2) let the 32 x 32 tile add the sums two wait states behind the last MFMA, which needs seven, and they were wrong.
    f32x4 total[FP][FQ];
#pragma unroll
    for (int f = 0; f < FP; ++f)
#pragma unroll
      for (int g = 0; g < FQ; ++g) total[f][g] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int chain = a.short_sums ? 4 : nkt;
    for (int kt = 0; kt < nkt; kt += chain) {
      multiply(kt, kt + chain < nkt ? kt + chain : nkt);
#pragma unroll
      for (int f = 0; f < FP; ++f)
#pragma unroll
        for (int g = 0; g < FQ; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            total[f][g][e] += acc[f][g][e];
            acc[f][g][e] = 0.f;
          }
    }
#pragma unroll
    for (int f = 0; f < FP; ++f)
#pragma unroll
      for (int g = 0; g < FQ; ++g) acc[f][g] = total[f][g];
  } else {
    multiply(0, nkt);
  }

  // ---- epilogue: a lane owns activation row r16 of each block column and 4 consecutive weight rows (4 c4 ..)
#pragma unroll
  for (int g = 0; g < FQ; ++g) {
    const int m = q0 + (wq * FQ + g) * 16 + r16;
    if constexpr (GATED) {
      const int nout = p_end / 2;
      if (a.out_f32) {
        if (m >= a.nq) continue;
        const bool vec = ((a.ldo & 1) == 0) && ((((uintptr_t)a.O) & 7) == 0);
#pragma unroll
        for (int f = 0; f < FP; ++f) {
          const int n = p0 / 2 + (wp * FP + f) * 8 + c4 * 2;
          const float v0 = acc[f][g][0] * silu_f32(acc[f][g][1]), v1 = acc[f][g][2] * silu_f32(acc[f][g][3]);
          float* o = (float*)a.O + (long long)m * a.ldo + n;
          if (vec && n + 1 < nout) {
            *(f32x2*)o = f32x2{v0, v1};
          } else {
            if (n < nout) o[0] = v0;
            if (n + 1 < nout) o[1] = v1;
          }
        }
      } else {
        const bool vec = ((a.ldo & 3) == 0) && ((((uintptr_t)a.O) & 7) == 0);
        unsigned h[FP];
#pragma unroll
        for (int f = 0; f < FP; ++f)
          h[f] = E::pack2(acc[f][g][0] * silu_f32(acc[f][g][1]), acc[f][g][2] * silu_f32(acc[f][g][3]));
        // Two features (4 bytes) to a lane and block of 8 features: the odd 16-lane rows of one block change places with the even
        // rows of the next, after which a lane holds four features of one block and a store covers 32 bytes of a row of H.
#pragma unroll
        for (int f = 0; f + 1 < FP; f += 2) {
          const auto sw = __builtin_amdgcn_permlane16_swap(h[f], h[f + 1], false, false);
          const int n = p0 / 2 + (wp * FP + f + (c4 & 1)) * 8 + (c4 >> 1) * 4;
          if (m < a.nq) store4(n, nout, vec, sw[0], sw[1], (unsigned short*)a.O + (long long)m * a.ldo);
        }
        if (FP % 2 != 0) {
          const int n = p0 / 2 + (wp * FP + FP - 1) * 8 + c4 * 2;
          unsigned short* o = (unsigned short*)a.O + (long long)m * a.ldo + n;
          if (m < a.nq) {
            if (vec && n + 1 < nout) {
              *(unsigned*)o = h[FP - 1];
            } else {
              if (n < nout) o[0] = (unsigned short)h[FP - 1];
              if (n + 1 < nout) o[1] = (unsigned short)(h[FP - 1] >> 16);
            }
          }
        }
      }
    } else if (m >= a.nq) {
      continue;
    } else if (a.splits > 1) {
      float* row = a.partial + ((long long)blockIdx.y * a.nq + m) * a.np;
#pragma unroll
      for (int f = 0; f < FP; ++f) {
        const int n = p0 + (wp * FP + f) * 16 + c4 * 4;
        if (((a.np & 3) == 0) && n + 3 < p_end) {
          *(f32x4*)(row + n) = acc[f][g];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < p_end) row[n + e] = acc[f][g][e];
        }
      }
    } else {
      unsigned short* orow = (unsigned short*)a.O + (long long)m * a.ldo;
      const bool vec_ok = ((a.ldo & 3) == 0) && ((((uintptr_t)a.O) & 7) == 0);
#pragma unroll
      for (int f = 0; f < FP; ++f) {
        const int n = p0 + (wp * FP + f) * 16 + c4 * 4;
        if (vec_ok && n + 3 < p_end) {
          u32x2 pk = {E::pack2(acc[f][g][0], acc[f][g][1]), E::pack2(acc[f][g][2], acc[f][g][3])};
          *(u32x2*)(orow + n) = pk;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < p_end) orow[n + e] = E::cvt1(acc[f][g][e]);
        }
      }
    }
  }
}

// ---- tiles, launch ------------------------------------------------------------------------------------------------
struct MidTile {
  int fp, fq, g, nw, na;  // 32 fp weight rows x 32 fq activation rows; weight lines asked for g at a time, rings of nw weight and na activation lines
};
#define FSW_MID_TILES(X)                                                                                              \
  X(1, 1, 1, 8, 8) X(1, 2, 1, 8, 8) X(2, 1, 1, 5, 5) X(3, 1, 1, 5, 5) X(4, 1, 1, 5, 5) X(5, 1, 1, 5, 5) X(6, 1, 1, 5, 5) X(8, 1, 1, 4, 4) \
  X(2, 2, 1, 5, 5) X(3, 2, 1, 5, 5) X(4, 2, 1, 5, 5) X(5, 2, 1, 5, 5) X(6, 2, 1, 5, 5) X(8, 2, 1, 4, 4) \
  X(2, 3, 2, 6, 5) X(3, 3, 2, 6, 5) X(4, 3, 2, 6, 4) X(5, 3, 2, 5, 4) X(6, 3, 2, 4, 4) X(2, 4, 2, 6, 5) X(3, 4, 2, 6, 5) X(4, 4, 2, 5, 5) \
  X(5, 4, 2, 4, 5) X(6, 4, 2, 4, 4) X(2, 5, 2, 6, 5) X(3, 5, 2, 6, 4) X(4, 5, 2, 5, 4) X(2, 6, 2, 6, 4) X(3, 6, 2, 5, 4) X(4, 6, 2, 4, 4) \
  X(2, 7, 2, 6, 4) X(3, 7, 2, 4, 4) X(4, 7, 2, 4, 3) X(2, 8, 2, 4, 4) X(3, 8, 2, 5, 3) X(4, 8, 2, 4, 3)
#define FSW_MID_ENTRY(FP, FQ, G, NW, NA) {FP, FQ, G, NW, NA},
constexpr MidTile kMidTiles[] = {FSW_MID_TILES(FSW_MID_ENTRY)};

template <class E, bool GATED, int FP, int FQ, int G, int NW, int NA>
hipError_t launch_mid_tile(const MidPlan& p, const GemmArgs& a, int ph, hipStream_t stream) {
  const int tiles_p = (a.np + p.step - 1) / p.step;
  const int tiles_q = (a.nq + 32 * FQ - 1) / (32 * FQ);
  GemmArgs b = a;
  b.tile_p = p.step;
  // whole lines are non-temporal when at most two tiles of activation rows share them
  int how = tiles_q <= 2 ? MID_STREAM : 0;
  // Where one tile holds all activation rows, the walks over K start at different lines, so that workgroups do not meet on the same memory
  // channels. Padded rows whose K ends inside a line do that only with weight rows a multiple of 4 KB apart, which all start on one channel
  // (all from line 0 -> spread, us: gate/up 47040 x 6096 in rows of 6144 7 rows 112 -> 84, 31648 x 4080 15 rows 53 -> 41, down 14328 -> 5600 35
  // rows 38.7 -> 31.3; 92 such problems 0.96, 49 with other strides 1.02), and while the activations fit an XCD's 4 MB L2, for all their lines
  // are in use at once then (down 20464 -> 7496 174 rows, 7 MB, 74 and 100; 16344 -> 4464 161 rows, 5 MB, 41 and 51).
  const bool line_tail = (a.k & 63) != 0;
  if (!ph && tiles_q == 1 && (!line_tail || ((a.ldp & 2047) == 0 && (long long)a.nq * a.k <= 1 << 21))) how |= MID_SPREAD;
  hipLaunchKernelGGL((mid_kernel<E, GATED, FP, FQ, G, NW, NA>), dim3((unsigned)(tiles_p * tiles_q), (unsigned)a.splits), dim3(512),
                     0, stream, b, tiles_p, tiles_q, GATED ? 4 : 2, ph, how);
  return hipGetLastError();
}

template <class E, bool GATED>
hipError_t launch_mid_typed(const MidPlan& p, const GemmArgs& a, int ph, hipStream_t stream) {
#define FSW_MID_CASE(FP, FQ, G, NW, NA) \
  if (kMidTiles[p.tile].fp == FP && kMidTiles[p.tile].fq == FQ) return launch_mid_tile<E, GATED, FP, FQ, G, NW, NA>(p, a, ph, stream);
  FSW_MID_TILES(FSW_MID_CASE)
#undef FSW_MID_CASE
  return hipErrorInvalidValue;
}

// One translation unit each (kernels_mid_*.hip): the instances compile side by side.
hipError_t launch_mid_bf16_gateup(const MidPlan& p, const GemmArgs& a, int ph, hipStream_t stream);
hipError_t launch_mid_bf16_down(const MidPlan& p, const GemmArgs& a, int ph, hipStream_t stream);
hipError_t launch_mid_fp16_gateup(const MidPlan& p, const GemmArgs& a, int ph, hipStream_t stream);
hipError_t launch_mid_fp16_down(const MidPlan& p, const GemmArgs& a, int ph, hipStream_t stream);

}  // namespace fsw
