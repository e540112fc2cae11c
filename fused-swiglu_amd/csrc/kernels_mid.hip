// Producer / consumer kernel for small and mid-size numbers of activation rows (1 .. ~700) on gfx950.
//
// Orientation, operands and epilogue values are those of kernels_tiled.hip: the MFMA A operand is fed with weight rows, the B
// operand with activation rows. The gated kernel keeps W13's interleaved rows as they lie: of the four consecutive weight rows
// that an accumulator lane owns two are "up" and two "gate" rows of the same two features, so the gating (swiglu.cu:380-381) is
// per-lane arithmetic without a de-interleave, and a tile may hold any multiple of 32 weight rows.
//
// What bounds it: the copies. A compute unit fetches 45 .. 60 bytes per ns when some of the lines come from HBM (62 .. 76 on the 256-row
// kernel's larger tiles, where the L2 serves more of them; 30 where all do and half the compute units fetch), whatever the
// number of lines asked for ahead (copy loops of 2 .. 8 stages of 24 KB measure the same): the loads of a compute unit return in
// order through its 32 KB L1, so an activation line that the L2 has at once waits behind the weight lines ahead of it. Time is
// therefore bytes per compute unit, and the tile follows from it: any height of 32 weight rows and any multiple of 32 activation
// rows, chosen by an estimate (mid_plan) so that one round of compute units shares the work with as few lines each as possible.
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
//   * LDS: NS slots of [BP weight rows, then BQ activation rows][128 bytes]; chunk c of row r of a line at position c ^ ((r >> 1) &
//     7). The 16 rows that a fragment read touches cover the 64 banks once, shifted or not: for even (and for odd) rows the
//     position ((c + shift of the row) & 7) ^ (r >> 1) is a permutation, since the shift grows by an even number of chunks from
//     one such row to the next.
// Measured and not taken: eight multiplying waves, fragments of the next K tile read before the barrier, pairs of lines issued
// together (all level within 2 %, the last slower where it costs a slot).
#include <math.h>
#include <stdio.h>

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

template <class E, bool GATED, int WP, int WQ, int FP, int FQ, int NS>
__global__ void __launch_bounds__((WP * WQ + 4) * 64)
mid_kernel(const GemmArgs a, const int tiles_p, const int tiles_q, const int group, const int ph, const int stream_w) {
  constexpr int NC = WP * WQ;
  constexpr int BP = WP * FP * 16, BQ = WQ * FQ * 16;
  constexpr int LINE = (BP + BQ) * 128;
  constexpr int LP = BP / 32, LQ = BQ / 32, NL = LP + LQ;
  static_assert(NS >= 3 && NS * LINE <= 160 * 1024, "LDS budget of a gfx950 CU");
  static_assert(BP % 32 == 0 && BQ % 32 == 0, "copy mapping");
  __shared__ __align__(1024) unsigned char lds[NS * LINE];

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
  const int rot = (!ph && tiles_q == 1 && nkt > 1) ? (int)(((unsigned)blockIdx.x * 2654435761u >> 12) % (unsigned)nkt) : 0;
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
    const unsigned poff = (unsigned)rb * (unsigned)a.ldp * 2u + (unsigned)(cp * 16);
    const unsigned qoff = (unsigned)rb * (unsigned)a.ldq * 2u + (unsigned)(cq * 16);
    const unsigned pstep = 32u * (unsigned)a.ldp * 2u, qstep = 32u * (unsigned)a.ldq * 2u;
    const int c_lo = kt0 * 8, c_all = a.k >> 3;
    const int c_hi = (kt0 + nkt) * 8 < c_all ? (kt0 + nkt) * 8 : c_all;
    unsigned char* const lw = lds + (wave - NC) * 1024;
    const int nline = nkt + ph;
    auto line_of = [&](int l) -> int {
      int r = l + rot;
      if (r >= nkt && rot > 0) r -= nkt;
      return kt0 + r;
    };
    auto issue_line = [&](int l, int slot) {
      const int L = line_of(l);
      const int kp = 8 * L + cp, kq = 8 * L + cq;
      const bool pin = l < nline && kp >= c_lo && kp < c_hi, qin = l < nline && kq >= c_lo && kq < c_hi;
      const unsigned po = poff + (unsigned)L * 128u, qo = qoff + (unsigned)L * 128u;
      unsigned char* const st = lw + slot * LINE;
      // activations first: they are in the L2 and need not wait behind weight lines that come from HBM (1 .. 2 %)
#pragma unroll
      for (int i = 0; i < LQ; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(qrs, (lds_void*)(st + (BP + i * 32) * 128), 16,
                                                 (int)(qin ? qo + i * qstep : OOB_OFFSET), 0, 0, 0);
      if (stream_w) {
#pragma unroll
        for (int i = 0; i < LP; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(prs, (lds_void*)(st + i * 32 * 128), 16,
                                                   (int)(pin ? po + i * pstep : OOB_OFFSET), 0, 0, 2);
      } else {
#pragma unroll
        for (int i = 0; i < LP; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(prs, (lds_void*)(st + i * 32 * 128), 16,
                                                   (int)(pin ? po + i * pstep : OOB_OFFSET), 0, 0, 0);
      }
    };
    if (nkt > 0) {
#pragma unroll
      for (int l = 0; l < NS; ++l) issue_line(l, l);
      if (ph) wait_copies<(NS - 2) * NL>();
      else wait_copies<(NS - 1) * NL>();
    }
    int slot = 0;
    for (int kt = 0; kt < nkt; ++kt) {
      asm volatile("s_barrier" ::: "memory");
      if (kt > 0) {  // line kt - 1 has been multiplied: its slot takes line kt - 1 + NS
        issue_line(kt - 1 + NS, slot);
        slot = slot + 1 == NS ? 0 : slot + 1;
      }
      if (ph) wait_copies<(NS - 3) * NL>();
      else wait_copies<(NS - 2) * NL>();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
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
    qo[h] = (unsigned)(BP + wq * FQ * 16 + r16) * 128u + (unsigned)(((qq & 7) ^ ((r16 >> 1) & 7)) * 16);
  }
  f32x4 acc[FP][FQ];
#pragma unroll
  for (int f = 0; f < FP; ++f)
#pragma unroll
    for (int g = 0; g < FQ; ++g) acc[f][g] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 pf[2][FP], qf[2][FQ];
  auto read_half = [&](int h, unsigned cur, unsigned nxt) {
    const unsigned char* pb = lds + po[h] + (pn[h] ? nxt : cur);
    const unsigned char* qb = lds + qo[h] + (qn[h] ? nxt : cur);
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
  unsigned cur = 0;
  auto multiply = [&](int from, int to) {
    for (int kt = from; kt < to; ++kt) {
      const unsigned nxt = cur + LINE == NS * LINE ? 0u : cur + LINE;
      // every read of the line before is complete (its slot is refilled behind the barrier), line kt has landed
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      read_half(0, cur, nxt);
      read_half(1, cur, nxt);
      mul_half(0);
      mul_half(1);
      cur = nxt;
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


// ---- tiles, plan, launch ------------------------------------------------------------------------------------------
namespace {

struct MidTile {
  int fp, fq, ns;  // tile of 32 fp weight rows x 32 fq activation rows, ring of ns lines (five or what 160 KB hold, eight of the two smallest)
};
#define FSW_MID_TILES(X)                                                                                              \
  X(1, 1, 8) X(1, 2, 8) X(2, 1, 5) X(3, 1, 5) X(4, 1, 5) X(5, 1, 5) X(6, 1, 5) X(8, 1, 4) X(2, 2, 5) X(3, 2, 5) X(4, 2, 5) X(5, 2, 5)         \
  X(6, 2, 5) X(8, 2, 4) X(2, 3, 5) X(3, 3, 5) X(4, 3, 5) X(5, 3, 5) X(6, 3, 4) X(2, 4, 5) X(3, 4, 5) X(4, 4, 5)         \
  X(5, 4, 4) X(6, 4, 4) X(2, 5, 5) X(3, 5, 5) X(4, 5, 4) X(2, 6, 5) X(3, 6, 4) X(4, 6, 4) X(2, 7, 4) X(3, 7, 4)         \
  X(4, 7, 3) X(2, 8, 4) X(3, 8, 3) X(4, 8, 3)
#define FSW_MID_ENTRY(FP, FQ, NS) {FP, FQ, NS},
const MidTile kTiles[] = {FSW_MID_TILES(FSW_MID_ENTRY)};
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);
struct TileSet {
  bool v[kNumTiles];
  bool operator[](int i) const { return v[i]; }
};
// whether there is a tile of as many weight rows and 32 activation rows fewer
const TileSet kNarrower = [] {
  TileSet s;
  for (int i = 0; i < kNumTiles; ++i) {
    s.v[i] = false;
    for (int u = 0; u < kNumTiles; ++u) s.v[i] |= kTiles[u].fp == kTiles[i].fp && kTiles[u].fq == kTiles[i].fq - 1;
  }
  return s;
}();

// Estimated time, us, of one launch (and the summing kernel of a split one): fitted to 2300 timings of 230 problems (gate/up and
// down, 1 .. 900 rows, d 1024 .. 8192, aligned and ragged rows, weights from memory), 4 % rms; the tile it picks is 1.3 % slower
// than the best of them on average. A K tile of 64 costs the copies of its weight and activation rows (0.00256 us = 128 bytes at
// 50 bytes per ns) or the LDS reads and MFMAs, whichever is more, plus a part of the other; a part that fills the chip shares
// HBM; a second round overlaps with the first where it is partly filled.
double mid_time(int np, int nq, int k, bool ragged, const MidTile& t, int step, int splits) {
  const int tq = (nq + 32 * t.fq - 1) / (32 * t.fq);
  const long long tp = (np + step - 1) / step;
  const long long wgs = tp * tq * splits;
  const int kt = ((k + 63) / 64 + splits - 1) / splits;
  const int rows = nq < 32 * t.fq ? nq : 32 * t.fq;
  double copy = (0.672 * step + 0.464 * rows) * 0.00256;
  if (wgs >= 200) copy += 0.153 * 0.00256 * step / tq;
  const double mul = 0.0227 * (t.fp + t.fq) + 0.01178 * t.fp * t.fq;
  const double tile = (copy > mul ? copy + 0.397 * mul : mul + 0.397 * copy) + 0.05;
  const double rounds = wgs <= 256 ? 1.0 : 0.787 * (double)((wgs + 255) / 256) + 0.213 * (double)wgs / 256.0;
  double us = rounds * (kt + 2.36 + (ragged ? 1.0 : 0.0)) * tile;
  const double hbm = 2.0 * np * (double)k / 7.305e6;
  us = us * us;
  us = sqrt(sqrt(us * us + hbm * hbm * hbm * hbm)) + 3.12;
  if (splits > 1) us += 1.19 + 0.078 * splits + 8.0 * splits * (double)nq * np / 4.53e6;
  return us;
}

template <class E, bool GATED, int FP, int FQ, int NS>
hipError_t launch_mid_tile(const MidPlan& p, const GemmArgs& a, int ph, hipStream_t stream) {
  const int tiles_p = (a.np + p.step - 1) / p.step;
  const int tiles_q = (a.nq + 32 * FQ - 1) / (32 * FQ);
  GemmArgs b = a;
  b.tile_p = p.step;
  // whole lines are non-temporal when at most two tiles of activation rows share them
  hipLaunchKernelGGL((mid_kernel<E, GATED, 2, 2, FP, FQ, NS>), dim3((unsigned)(tiles_p * tiles_q), (unsigned)a.splits), dim3(512),
                     0, stream, b, tiles_p, tiles_q, GATED ? 4 : 2, ph, tiles_q <= 2 ? 1 : 0);
  return hipGetLastError();
}

template <class E, bool GATED>
hipError_t launch_mid_typed(const MidPlan& p, const GemmArgs& a, int ph, hipStream_t stream) {
#define FSW_MID_CASE(FP, FQ, NS) \
  if (kTiles[p.tile].fp == FP && kTiles[p.tile].fq == FQ) return launch_mid_tile<E, GATED, FP, FQ, NS>(p, a, ph, stream);
  FSW_MID_TILES(FSW_MID_CASE)
#undef FSW_MID_CASE
  return hipErrorInvalidValue;
}

}  // namespace

static MidPlan find_plan(bool gated, int np, int nq, int k, bool ragged, int splits, int max_splits) {
  MidPlan best = {-1, 0, 1, 0.0};
  const int q32 = (nq + 31) / 32;
  for (int tile = 0; tile < kNumTiles; ++tile) {
    const MidTile& t = kTiles[tile];
    if (ragged && t.ns < 4) continue;  // one line of the ring is taken by the shift: three lines leave no copy in flight
    const int tq = (q32 + t.fq - 1) / t.fq;
    if (t.fq > 1 && (q32 + t.fq - 2) / (t.fq - 1) == tq) {
      // a narrower tile needs no more columns of tiles: this one holds padding only
      if (kNarrower[tile]) continue;
    }
    const int full = 32 * t.fp;
    const long long tp = (np + full - 1) / full;
    int steps[2] = {full, 0};
    const long long rounds = (tp * tq + 255) / 256;
    // As many pieces as whole rounds hold. Aligned 128-row tiles of up to 64 activation rows stay whole where they leave less than an
    // eighth of a round empty: the pieces' wasted MFMA and LDS work costs what those compute units give, and K is then walked from the same
    // start (mid_kernel's `rot`) for all these row counts. us, pieces -> whole: 28672 x 4096 (224 tiles) 16 rows 37.1 -> 36.5, 48 rows 38.4
    // -> 37.9; 28928 x 5568 (226) 11 rows 53.3 -> 51.2; 29056 x 5760 (227) 40 rows 53.7 -> 55.0. With fewer tiles, 27648 x 5120 (216), 16
    // rows 45.2 whole, 43.9 in pieces, 48 rows 51.4 and 49.7.
    const bool whole = !ragged && nq <= 64 && t.fp == 4 && 8 * tp >= 7 * 256 * rounds;
    if (gated && tp * tq <= 1024 && !whole) {
      const long long pieces = rounds * 256 / tq;
      const int step = (int)(((np + pieces - 1) / pieces + 7) / 8 * 8);
      if (step < full && step > full - 32) steps[1] = step;
    }
    for (int s = 0; s < 2 && steps[s] > 0; ++s) {
      const long long tps = (np + steps[s] - 1) / steps[s];
      int sps[3] = {1, 0, 0};
      if (splits > 0) {
        sps[0] = splits;
      } else {
        const int deep = k / 256 < 16 ? k / 256 : 16;
        for (int r = 1; r <= 2; ++r) {
          long long sp = 256LL * r / (tps * tq);
          if (sp > deep) sp = deep;
          if (sp > max_splits) sp = max_splits;
          if (sp > 1 && 4.0 * sp * (double)nq * np <= 256e6 && (r == 1 || sp != sps[1])) sps[r] = (int)sp;
        }
      }
      for (int i = 0; i < 3; ++i) {
        if (sps[i] < 1) continue;
        double us = mid_time(np, nq, k, ragged, t, steps[s], sps[i]);
        // The estimate flatters fewer parts on lower tiles, which fetch every activation row for fewer weight rows (11008 -> 4096,
        // 200 rows: four parts on 64 x 224 38.4 us, eight on 128 x 224 34.5; 14336 -> 4096, 256 rows 48.8 and 45.6).
        if (splits == 0 && !gated && nq > 64 && tq == 1 && t.fp == 4) us *= 0.92;
        if (best.tile < 0 || us < best.us) best = {tile, steps[s], sps[i], us};
      }
    }
  }
  return best;
}

// A search takes a few microseconds of host time and one call asks for its plans several times (workspace query, launch), so each
// thread keeps the last few plans by the sizes they follow from.
MidPlan mid_plan(bool gated, int np, int nq, int k, bool ragged, int splits, int max_splits) {
  struct Entry {
    int np, nq, k, rest;
    MidPlan plan;
  };
  static thread_local Entry memo[32];  // zero-initialised: np 0 is never asked for
  const int rest = (gated ? 1 : 0) | (ragged ? 2 : 0) | splits << 2 | max_splits << 8;
  const unsigned h = (((unsigned)np * 31u + (unsigned)nq) * 31u + (unsigned)k) * 31u + (unsigned)rest;
  Entry& e = memo[(h ^ (h >> 7) ^ (h >> 15)) % 32];
  if (e.np != np || e.nq != nq || e.k != k || e.rest != rest)
    e = {np, nq, k, rest, find_plan(gated, np, nq, k, ragged, splits, max_splits)};
  return e.plan;
}

// static storage: "mid_<weight rows>x<activation rows>"
const char* mid_name(const MidPlan& p) {
  static char names[kNumTiles][16];
  static const bool done = [] {
    for (int i = 0; i < kNumTiles; ++i) snprintf(names[i], sizeof(names[i]), "mid_%dx%d", kTiles[i].fp * 32, kTiles[i].fq * 32);
    return true;
  }();
  (void)done;
  return p.tile >= 0 ? names[p.tile] : "none";
}

int mid_tile_count() { return kNumTiles; }
int mid_tile_rows(int tile) { return 32 * kTiles[tile].fp; }
int mid_tile_index(int bp, int bq) {
  for (int i = 0; i < kNumTiles; ++i)
    if (kTiles[i].fp * 32 == bp && kTiles[i].fq * 32 == bq) return i;
  return -1;
}

hipError_t launch_mid(int dtype, bool gated, const MidPlan& p, const GemmArgs& a, hipStream_t stream) {
  if (p.tile < 0 || p.tile >= kNumTiles || p.step <= 0 || p.step > 32 * kTiles[p.tile].fp || p.step % 8 != 0)
    return hipErrorInvalidValue;
  if (a.np <= 0 || a.nq <= 0) return hipSuccess;
  const int ph = mid_ragged(a) ? 1 : 0;
  hipError_t e = dtype == 0 ? (gated ? launch_mid_typed<Bf16, true>(p, a, ph, stream) : launch_mid_typed<Bf16, false>(p, a, ph, stream))
                            : (gated ? launch_mid_typed<Fp16, true>(p, a, ph, stream) : launch_mid_typed<Fp16, false>(p, a, ph, stream));
  if (e != hipSuccess || a.splits <= 1) return e;
  return launch_splitk_reduce(dtype, a, stream);
}

}  // namespace fsw
