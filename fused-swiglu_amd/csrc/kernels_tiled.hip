// LDS-tiled MFMA kernels (v_mfma_f32_32x32x16) for small and mid-size problems on gfx950, the split-K reduction and
// the row-major -> panel-blocked copy. The 256 x 256 prefill kernel lives in kernels_pair16.hip.
//
// One kernel template covers both GEMMs of the MLP forward:
//   GATED : H[m, j] = up * silu(gate), up = X[m,:].W13[2j,:], gate = X[m,:].W13[2j+1,:]
//           (the computation of swiglu.cu:111-394: main loop :290-343, gating epilogue :345-393)
//   plain : Y[m, n] = H[m,:].W2[n,:]   (no counterpart in the reference)
//
// Orientation. The MFMA "A" operand (rows of the 32x32 result) is fed with WEIGHT rows and the "B" operand
// (columns of the result) with ACTIVATION rows, so an accumulator lane owns one activation row m and runs of 4
// consecutive output features. That makes the stores 8-byte vectors along the contiguous dimension of the
// output, and, for the gated kernel, lets the de-interleave of W13 happen while the tile is copied into LDS:
// LDS rows [0, BP/2) receive the even ("up") rows of the weight tile and rows [BP/2, BP) the odd ("gate")
// rows. A wave then runs two accumulator sets over the same activation fragments, and up/gate of one (m, j)
// land in the same lane and register index: the gating is plain per-lane fp32 math, no cross-lane traffic.
#include <math.h>

#include <type_traits>

#include "fsw_internal.h"
#include "fsw_device.h"

namespace fsw {

// Epilogue shared by the tiled kernels. A lane owns activation row m = l32 of each Q fragment and, per group
// of 4 accumulator registers, 4 consecutive output features: feature = 8 * (i / 4) + 4 * hi + (i % 4) within
// the fragment. Gating (fp32 multiply and SiLU, swiglu.cu:380-381) happens here, then ONE rounding and an
// 8-byte store (GemmArgs::out_f32: no rounding and a 16-byte store).
template <class E, bool GATED, int WP, int WQ, int FP, int FQ>
__device__ __forceinline__ void store_tile(f32x16 (&acc)[FP][FQ], const GemmArgs& a, int p0, int q0, int wp, int wq,
                                           int l32, int hi, int p_end) {
  unsigned short* O = (unsigned short*)a.O;
  const int nout = GATED ? p_end / 2 : p_end;  // p_end: first weight row this workgroup does not own
  const bool vec_ok = ((a.ldo & 3) == 0) && ((((uintptr_t)a.O) & 7) == 0);
  const bool vec32_ok = ((a.ldo & 3) == 0) && ((((uintptr_t)a.O) & 15) == 0);
  constexpr int FO = GATED ? FP / 2 : FP;
#pragma unroll
  for (int g = 0; g < FQ; ++g) {
    const int m = q0 + (wq * FQ + g) * 32 + l32;
    if (m >= a.nq) continue;
    unsigned short* orow = O + (long long)m * a.ldo;
#pragma unroll
    for (int f = 0; f < FO; ++f) {
      const int nb = (GATED ? p0 / 2 + (wp * FO + f) * 32 : p0 + (wp * FO + f) * 32) + hi * 4;
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (GATED) {
            v[e] = acc[f][g][i4 * 4 + e] * silu_f32(acc[f + FO][g][i4 * 4 + e]);
          } else {
            v[e] = acc[f][g][i4 * 4 + e];
          }
        }
        const int n = nb + i4 * 8;
        if (GATED && a.out_f32) {
          float* o32 = (float*)a.O + (long long)m * a.ldo + n;
          if (vec32_ok && n + 3 < nout) {
            *(f32x4*)o32 = f32x4{v[0], v[1], v[2], v[3]};
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < nout) o32[e] = v[e];
          }
        } else if (vec_ok && n + 3 < nout) {
          u32x2 pk = {E::pack2(v[0], v[1]), E::pack2(v[2], v[3])};
          *(u32x2*)(orow + n) = pk;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < nout) orow[n + e] = E::cvt1(v[e]);
        }
      }
    }
  }
}

// Split-K epilogue of the plain kernel: fp32 partial sums to partial[split][m][n], 16 bytes per lane.
template <int WP, int WQ, int FP, int FQ>
__device__ __forceinline__ void store_partial(f32x16 (&acc)[FP][FQ], const GemmArgs& a, int split, int p0, int q0,
                                              int wp, int wq, int l32, int hi) {
  float* base = a.partial + (long long)split * a.nq * a.np;
#pragma unroll
  for (int g = 0; g < FQ; ++g) {
    const int m = q0 + (wq * FQ + g) * 32 + l32;
    if (m >= a.nq) continue;
    float* row = base + (long long)m * a.np;
#pragma unroll
    for (int f = 0; f < FP; ++f) {
      const int nb = p0 + (wp * FP + f) * 32 + hi * 4;
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const int n = nb + i4 * 8;
        if (((a.np & 3) == 0) && n + 3 < a.np) {
          f32x4 v = {acc[f][g][i4 * 4], acc[f][g][i4 * 4 + 1], acc[f][g][i4 * 4 + 2], acc[f][g][i4 * 4 + 3]};
          *(f32x4*)(row + n) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < a.np) row[n + e] = acc[f][g][i4 * 4 + e];
        }
      }
    }
  }
}

// O[m, n] = round(sum over splits of partial[s][m][n]); one thread per 4 consecutive n. The number of parts is a template
// parameter so that the loads of all parts are in flight at once (bound: latency; a loop over the parts waits for each load
// before it asks for the next). Forward 60 rows of 1888 x 5504 37.2 -> 35.1 us, 100 rows of 1928 x 5640 49.1 -> 46.9, 40 rows of 5120 x
// 13824 80.2 -> 79.1; where the sums are a small part of the call: level.
template <class E, int SPLITS>
__global__ void __launch_bounds__(256)
splitk_reduce_kernel(const float* __restrict__ partial, int nq, int np, unsigned short* __restrict__ O, long long ldo) {
  const int groups = (np + 3) >> 2;
  const long long id = (long long)blockIdx.x * 256 + threadIdx.x;
  if (id >= (long long)nq * groups) return;
  const int m = (int)(id / groups);
  const int n = (int)(id - (long long)m * groups) * 4;
  const long long plane = (long long)nq * np;
  const float* src = partial + (long long)m * np + n;
  const bool full = (np & 3) == 0;
  f32x4 part[SPLITS];
#pragma unroll
  for (int s = 0; s < SPLITS; ++s) {
    if (full) {
      part[s] = *(const f32x4*)(src + s * plane);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) part[s][e] = n + e < np ? src[s * plane + e] : 0.f;
    }
  }
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SPLITS; ++s)
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += part[s][e];
  unsigned short* orow = O + (long long)m * ldo;
  if (full && ((ldo & 3) == 0) && ((((uintptr_t)O) & 7) == 0)) {
    u32x2 pk = {E::pack2(v[0], v[1]), E::pack2(v[2], v[3])};
    *(u32x2*)(orow + n) = pk;
  } else {
    for (int e = 0; e < 4; ++e)
      if (n + e < np) orow[n + e] = E::cvt1(v[e]);
  }
}

// ---- direct-to-LDS variant ---------------------------------------------------------------------------------
// Same tiling and epilogue, but the operand tiles go from global memory straight into LDS with
// buffer_load_dwordx4 ... lds (no staging registers, no ds_write: LDS writes by ds_write_b128 run at roughly a
// third of the read rate on this chip and were the largest single cost of the register-staged loop).
// An LDS-DMA instruction writes lane i's 16 bytes at base + 16 i, so a wave instruction fills 8 consecutive
// 128-byte rows; the swizzle is applied on the global side: the lane that lands on chunk position p of row r
// fetches logical chunk p ^ ((r >> 1) & 7). With that function any 16 consecutive rows at one logical chunk
// cover all 64 banks once (the LDS serves ds_read_b128 sixteen lanes per clock), so operand reads are
// conflict-free. The two stages are separate __shared__ objects so that the compiler's counter tracking can
// tell reads of the live stage from DMA writes into the other one.
typedef __attribute__((address_space(3))) void lds_void;

template <class E, bool GATED, bool KTAIL, int WP, int WQ, int FP, int FQ, bool STREAM_W = false, int NS = 2>
__global__ void __launch_bounds__(WP* WQ * 64)
tiled_dma_kernel(const GemmArgs a, const int tiles_p, const int tiles_q, const int group) {
  constexpr int NT = WP * WQ * 64;
  constexpr int BP = WP * FP * 32;
  constexpr int BQ = WQ * FQ * 32;
  constexpr int BK = 64;
  constexpr int ROWB = BK * 2;
  constexpr int RSTEP = NT / 8;
  constexpr int LP = BP / RSTEP;
  constexpr int LQ = BQ / RSTEP;
  constexpr int STAGE = (BP + BQ) * ROWB;
  static_assert(BP % RSTEP == 0 && BQ % RSTEP == 0 && RSTEP % 16 == 0, "copy mapping");
  static_assert(!GATED || (FP % 2 == 0), "gated kernel pairs fragments");
  static_assert(NS >= 2 && NS <= 4 && NS * STAGE <= 160 * 1024, "LDS budget of a gfx950 CU");

  __shared__ __align__(1024) unsigned char lds0[STAGE];
  __shared__ __align__(1024) unsigned char lds1[STAGE];
  __shared__ alignas(NS > 2 ? 1024 : 16) unsigned char lds2[NS > 2 ? STAGE : 16];
  __shared__ alignas(NS > 3 ? 1024 : 16) unsigned char lds3[NS > 3 ? STAGE : 16];

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // wave-uniform: LDS-DMA bases live in SGPRs
  const int wq = wave % WQ;
  const int wp = wave / WQ;
  const int l32 = lane & 31;
  const int hi = lane >> 5;

  int tp, tq;
  tile_coords(blockIdx.x, tiles_p, tiles_q, group, tp, tq);
  const int step_p = (a.tile_p > 0 && a.tile_p < BP) ? a.tile_p : BP;  // weight rows this workgroup owns
  const int p0 = tp * step_p;
  const int p_end = p0 + step_p < a.np ? p0 + step_p : a.np;
  const int q0 = tq * BQ;
  if (GATED && blockIdx.x == 0 && blockIdx.y == 0)  // counters of the kernel that follows in fsw_mlp (GemmArgs::zero_words)
    for (int i = t; i < a.n_zero_words; i += NT) a.zero_words[i] = 0u;

  // ---- global -> LDS copy mapping: lane lands on chunk position pc of row rb (+ i * RSTEP)
  const int pc = t & 7;
  const int rb = t >> 3;
  const int lc = pc ^ ((rb >> 1) & 7);  // logical chunk this lane fetches (RSTEP % 16 == 0 keeps (row >> 1) & 7)
  const unsigned char* pbase = (const unsigned char*)a.P + (long long)p0 * a.ldp * 2;
  const unsigned char* qbase = (const unsigned char*)a.Q + (long long)q0 * a.ldq * 2;
  const __amdgpu_buffer_rsrc_t prs = make_rsrc(pbase, ((long long)(p_end - p0 - 1) * a.ldp + a.k) * 2);
  const __amdgpu_buffer_rsrc_t qrs = make_rsrc(qbase, ((long long)(a.nq - q0 - 1) * a.ldq + a.k) * 2);
  unsigned poff[LP], qoff[LQ];
#pragma unroll
  for (int i = 0; i < LP; ++i) {
    const int r = rb + i * RSTEP;
    const int grow = GATED ? (r < BP / 2 ? 2 * r : 2 * (r - BP / 2) + 1) : r;
    poff[i] = (unsigned)grow * (unsigned)a.ldp * 2u + (unsigned)lc * 16u;
  }
#pragma unroll
  for (int i = 0; i < LQ; ++i) {
    const int r = rb + i * RSTEP;
    qoff[i] = (unsigned)r * (unsigned)a.ldq * 2u + (unsigned)lc * 16u;
  }

  // ---- LDS -> MFMA fragment read mapping
  unsigned xo[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) xo[ks] = (unsigned)((((ks << 1) | hi) ^ ((l32 >> 1) & 7)) * 16);
  const unsigned rd_p = (unsigned)((GATED ? wp * (FP / 2) * 32 : wp * FP * 32) + l32) * ROWB;
  const unsigned rd_q = (unsigned)(BP + wq * FQ * 32 + l32) * ROWB;
  auto p_frag_off = [](int f) -> unsigned {
    if (GATED) return (unsigned)((f < FP / 2 ? f * 32 : BP / 2 + (f - FP / 2) * 32) * ROWB);
    return (unsigned)(f * 32 * ROWB);
  };

  f32x16 acc[FP][FQ];
#pragma unroll
  for (int f = 0; f < FP; ++f)
#pragma unroll
    for (int g = 0; g < FQ; ++g)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[f][g][i] = 0.0f;

  // K range of this workgroup: everything, or one of a.splits contiguous runs of K tiles (blockIdx.y)
  const int nkt_all = (a.k + BK - 1) / BK;
  const int kt_per = (nkt_all + a.splits - 1) / a.splits;
  const int kt0 = (int)blockIdx.y * kt_per;
  const int nkt = nkt_all - kt0 < kt_per ? (nkt_all - kt0 > 0 ? nkt_all - kt0 : 0) : kt_per;

  // With a single tile of activation rows no two workgroups share a weight panel, every weight byte comes from
  // HBM, and workgroups that walk K in step all ask for the same column offset of rows a power of two apart: the
  // same few memory channels at any moment (measured 2.2 TB/s). Each workgroup therefore starts its walk at its own
  // K tile and wraps around; only the order of the fp32 summation changes. (With several activation tiles the
  // workgroups that share a panel must stay in step for the L2 to serve them, so there rot = 0.)
  const int rot = (tiles_q == 1 && nkt > 1) ? (int)(((unsigned)blockIdx.x * 2654435761u >> 12) % (unsigned)nkt) : 0;

  // STREAM_W: the weight copies carry the non-temporal cache policy, for launches with one or two tiles of activation rows,
  // where a weight line has at most two users: the single-use stream then neither displaces the activations nor has
  // to evict whatever the previous kernels left dirty in the L2s and the Infinity Cache. Measured at 4096 x 28672,
  // M = 128, caches filled with freshly written data before each call: gate/up 94 -> 67 us, down 63 -> 44 us;
  // back-to-back forwards 110 -> 106 us.
  // DMA of K tile `kt` into `stage`: wave-uniform LDS base per instruction, loop-invariant per-lane offset in a
  // VGPR, the K offset in an SGPR. Rows beyond the matrix are out of range for the buffer descriptor and arrive
  // as zeros. A prefetch past the last tile is out of range as a whole: no memory traffic (with three stages and
  // a dozen K tiles a re-read of the last tile would be a sixth of it all), never consumed. When K is not a multiple of
  // 64 (KTAIL) lanes whose chunk lies at or beyond K redirect their offset out of range as well.
  auto dma = [&](unsigned char* stage, int kt) {
    int ktr = kt + rot;
    if (ktr >= nkt) ktr -= nkt;
    const int ktc = kt0 + ktr;
    const int kb = kt < nkt ? ktc * (BK * 2) : 0;
    const bool in = kt < nkt && (!KTAIL || (ktc * BK + lc * 8) < a.k);
#pragma unroll
    for (int i = 0; i < LP; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(prs, (lds_void*)(stage + i * RSTEP * ROWB + wave * 1024), 16,
                                               (int)(in ? poff[i] : OOB_OFFSET), kb, 0, STREAM_W ? 2 : 0);
#pragma unroll
    for (int i = 0; i < LQ; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(qrs, (lds_void*)(stage + (BP + i * RSTEP) * ROWB + wave * 1024), 16,
                                               (int)(in ? qoff[i] : OOB_OFFSET), kb, 0, 0);
  };

  u32x4 pf[2][FP], qf[2][FQ];
  auto f_read = [&](int fb, const unsigned char* base, int ks) {
    pf[fb][0] = *(const u32x4*)(base + rd_p + p_frag_off(0) + xo[ks]);
#pragma unroll
    for (int g = 0; g < FQ; ++g) qf[fb][g] = *(const u32x4*)(base + rd_q + g * 32 * ROWB + xo[ks]);
#pragma unroll
    for (int f = 1; f < FP; ++f) pf[fb][f] = *(const u32x4*)(base + rd_p + p_frag_off(f) + xo[ks]);
  };
  auto mma = [&](int fb, int f_lo, int f_hi) {
#pragma unroll
    for (int f = f_lo; f < f_hi; ++f)
#pragma unroll
      for (int g = 0; g < FQ; ++g) acc[f][g] = E::mfma32(pf[fb][f], qf[fb][g], acc[f][g]);
  };

  constexpr int NM = FP * FQ;
  constexpr int NR = FP + FQ;
  constexpr int NL = LP + LQ;
  constexpr int HF = FP / 2 > 0 ? FP / 2 : 1;
  constexpr int MPR = NM / NR > 0 ? NM / NR : 1;

  // One K tile. On entry: stage `cur` holds tile kt (made visible by the previous barrier) and its step-0
  // fragments are in pf[0]/qf[0]; every wave is done reading `oth`. The DMA of tile kt+1 into `oth` is issued
  // in step 0 and has the whole iteration to land before the barrier in step 3.
  auto iteration = [&](unsigned char* cur, unsigned char* oth, int kt) {
    dma(oth, kt + 1);
    f_read(1, cur, 1);
    mma(0, 0, FP);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, MPR, 0);
      __builtin_amdgcn_sched_group_barrier(0x010, (NL + NR - 1) / NR, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    f_read(0, cur, 2);
    mma(1, 0, FP);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, MPR, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    f_read(1, cur, 3);
    mma(0, 0, FP);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, MPR, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    mma(1, 0, HF);
    // This wave's copy of tile kt + 1 has landed (vmcnt) and its reads of `cur` are complete (lgkmcnt), then the
    // workgroup barrier publishes every wave's part. Written out: the fences of __syncthreads() need not wait for
    // vmcnt, and nothing else orders another wave's direct-to-LDS copy against this wave's reads after the barrier.
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    f_read(0, oth, 0);
    mma(1, HF, FP);
#pragma unroll
    for (int i = 0; i < (FP - HF) * FQ; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, (NR + (FP - HF) * FQ - 1) / ((FP - HF) * FQ), 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
  };

  // NS stages: two where two workgroups share a compute unit; three or four where a workgroup has it to itself (see
  // launch_dma_kernel): the copy of tile kt + NS - 1 is issued while tile kt is multiplied, which multiplies the
  // bytes in flight per workgroup. Measured at 4096 x 28672, gate/up, two -> three: M = 65: 67.6 -> 43.9 us, M = 128:
  // 67.0 -> 49.0 us (a fourth stage: level).
  if constexpr (NS == 2) {
    if (nkt > 0) dma(lds0, 0);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (nkt > 0) f_read(0, lds0, 0);
    int kt = 0;
    for (; kt + 1 < nkt; kt += 2) {
      iteration(lds0, lds1, kt);
      iteration(lds1, lds0, kt + 1);
    }
    if (kt < nkt) iteration(lds0, lds1, kt);
  } else {
    unsigned char* const ring[4] = {lds0, lds1, lds2, lds3};
    constexpr int VM = (NS - 2) * NL;
    static_assert(VM <= 63, "vmcnt is a 6-bit counter");
    constexpr int WAIT_IMM = (VM & 15) | ((VM >> 4) << 14) | (7 << 4) | (0 << 8);
    auto ring_iteration = [&](unsigned char* cur, unsigned char* nxt, unsigned char* fill, int kt) {
      dma(fill, kt + NS - 1);
      f_read(1, cur, 1);
      mma(0, 0, FP);
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, MPR, 0);
        __builtin_amdgcn_sched_group_barrier(0x010, (NL + NR - 1) / NR, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      f_read(0, cur, 2);
      mma(1, 0, FP);
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, MPR, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      f_read(1, cur, 3);
      mma(0, 0, FP);
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, MPR, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      mma(1, 0, HF);
      asm volatile("s_waitcnt %0\n\ts_barrier" ::"n"(WAIT_IMM) : "memory");
      f_read(0, nxt, 0);
      mma(1, HF, FP);
#pragma unroll
      for (int i = 0; i < (FP - HF) * FQ; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, (NR + (FP - HF) * FQ - 1) / ((FP - HF) * FQ), 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
    };
    if (nkt > 0) {
#pragma unroll
      for (int j = 0; j < NS - 1; ++j) dma(ring[j], j);
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 2) * NL) : "memory");
      f_read(0, lds0, 0);
    }
    int kt = 0;
    for (; kt + NS - 1 < nkt; kt += NS) {
#pragma unroll
      for (int j = 0; j < NS; ++j) ring_iteration(ring[j], ring[(j + 1) % NS], ring[(j + NS - 1) % NS], kt + j);
    }
#pragma unroll
    for (int j = 0; j < NS - 1; ++j) {
      if (kt < nkt) {
        ring_iteration(ring[j], ring[(j + 1) % NS], ring[(j + NS - 1) % NS], kt);
        ++kt;
      }
    }
  }

  if constexpr (!GATED) {
    if (a.splits > 1) {
      store_partial<WP, WQ, FP, FQ>(acc, a, (int)blockIdx.y, p0, q0, wp, wq, l32, hi);
      return;
    }
  }
  store_tile<E, GATED, WP, WQ, FP, FQ>(acc, a, p0, q0, wp, wq, l32, hi, p_end);
}

// ---- row-major -> panel-blocked copy ---------------------------------------------------------------------------
// dst block (panel, kt) = [256 rows][64 bytes]: rows 256 panel .. 256 panel + 255 of src, K elements 32 kt .. 32 kt + 31;
// rows past `rows` and elements past `k` are written as zeros. A workgroup copies four K tiles of one panel: reads
// are 256 contiguous bytes per row (16 lanes), writes 1 KB contiguous per 16 rows of a block.
// gated_order (W13): block row r < 128 is source row 2r of the panel (the "up" row of feature r), block row
// r >= 128 is source row 2(r - 128) + 1 (its "gate" row): the order the gated kernel keeps a weight tile in LDS.
__global__ void __launch_bounds__(256)
block_rows_kernel(const unsigned short* __restrict__ src, long long ld, int rows, int k, unsigned char* __restrict__ dst,
                  int nkt, int gated_order) {
  const int t = threadIdx.x;
  const int c16 = t & 15;
  const int r0 = t >> 4;
  const int panel = blockIdx.y;
  const int kt = (int)blockIdx.x * 4 + (c16 >> 2);
  if (kt >= nkt) return;
  const int k0 = (int)blockIdx.x * 128 + c16 * 8;
  unsigned char* block = dst + ((long long)panel * nkt + kt) * (256 * 64) + (c16 & 3) * 16;
#pragma unroll 4
  for (int pass = 0; pass < 16; ++pass) {
    const int row = pass * 16 + r0;
    const int srow = gated_order ? (row < 128 ? 2 * row : 2 * (row - 128) + 1) : row;
    const long long gr = (long long)panel * 256 + srow;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (gr < rows && k0 < k) v = *(const u32x4*)(src + gr * ld + k0);
    *(u32x4*)(block + row * 64) = v;
  }
}


// ---- variant table ------------------------------------------------------------------------------------
namespace {

const TiledVariant kVariants[] = {
    {"dma_128x128", 128, 128, 256},    // two- or three-stage direct-to-LDS copies, 4 waves of 64 x 64
    {"dma8w_128x256", 128, 256, 512},  // id 3 under an older number (a form on 4 waves had it: 72 against 64 us)
    {"dma_128x192", 128, 192, 256},    // 129 .. 192 activation rows in ONE tile: every weight byte is read once
    {"dma8w_128x256", 128, 256, 512},  // the same for 193 .. 256 rows, on 8 waves (two per SIMD), wave tile 64 x 64
    {"dma_128x64", 128, 64, 256},      // up to 64 activation rows in one tile
    {"pair16_256x256", 256, 256, 256}, // v_mfma_f32_16x16x32 prefill kernel (kernels_pair16.hip), row-major operands
};
constexpr int kPair16Variant = 5;

}  // namespace

// Activation-row tiles per raster band of the 256 x 256 kernel (the 128-row kernels above use 4 for the gate/up and
// 2 for the down product): 4, i.e. the 32 tiles an XCD runs at once are 4 activation panels x 8 weight
// panels (12 operand panels through its L2 per round). The down product of tall problems (32 activation tiles or
// more, 16 weight panels, 14336-deep K) measures level to 1 % slower that way and keeps bands of 2; with fewer
// activation tiles bands of 4 win (4096 x 4096 x 11008: 244 -> 236 us, 2048 x 8192 x 28672 fp16: 639 -> 633 us).
int raster_group(bool gated, int tiles_q) { return gated ? 4 : (tiles_q >= 32 ? 2 : 4); }

namespace {

// The 128-row instances stream their weights non-temporally when at most two tiles of activation rows share them and weight
// rows are whole 128-byte lines (ldp a multiple of 64, the matrix on a line). Otherwise a line at the edge of a 128-byte piece of a
// row serves two consecutive K tiles and has to stay in the cache between them: non-temporal -> default policy, us, weights that
// repeat from call to call: gate/up 3000 x 16016 at 130 rows 51.7 -> 31.5, 4104 x 28000 at 100 rows 66.1 -> 41.7, 5000 x 32016 at
// 64 rows 82.2 -> 71.6; down 8008 -> 3000 at 64 rows 23.3 -> 17.2, 28680 -> 8192 at 100 rows 153 -> 129. Weights that come from
// memory, the matrix 16 bytes past a line: gate/up 5120 x 27648 at 40 rows 69.8 -> 63.8, 4096 x 28672 at 64 rows 56.3 -> 52.4 and
// at 200 rows 80.4 -> 76.4; down 14336 -> 4096 at 64 rows 38.4 -> 33.4.
// Ring length: a launch of at most 256 workgroups has a compute unit to itself per workgroup, so nothing else hides
// the latency of its copies and the LDS is free: three stages (four of the small 128 x 64 ones), copies two (three) K
// tiles ahead. Two stages -> three, us: gate/up fp16 3000 x 16016 at 200 rows (252 workgroups) 68 -> 57, whole forward
// 92.1 -> 82.9; forward 512 rows of 1024 x 2816 29.8 -> 24.2; gate/up 250 rows of 1024 x 5632 17.7 -> 12.9; a fourth and
// fifth stage of 32 KB: level. 128 x 64, three -> four stages: gate/up 64 rows of 4096 x 22016 34.3 -> 32.2.
// More workgroups than compute units keep two stages and two workgroups per compute unit (8192 x 57344 at 65 rows,
// 448 workgroups: 168 us with three stages, 158 with two).
template <class E, bool GATED, bool KTAIL, int WP, int WQ, int FP, int FQ>
void launch_dma_kernel(const dim3 grid, hipStream_t stream, const GemmArgs& a, int tiles_p, int tiles_q, int group) {
  constexpr int DEEP = WQ * FQ == 2 ? 4 : 3;
  const dim3 block(WP * WQ * 64);
  const bool deep = (long long)grid.x * grid.y <= 256;
  if (tiles_q <= 2 && a.ldp % 64 == 0 && ((uintptr_t)a.P & 127) == 0) {
    if (deep) {
      hipLaunchKernelGGL((tiled_dma_kernel<E, GATED, KTAIL, WP, WQ, FP, FQ, true, DEEP>), grid, block, 0, stream, a,
                         tiles_p, tiles_q, group);
    } else {
      hipLaunchKernelGGL((tiled_dma_kernel<E, GATED, KTAIL, WP, WQ, FP, FQ, true>), grid, block, 0, stream, a, tiles_p,
                         tiles_q, group);
    }
  } else if (deep) {
    hipLaunchKernelGGL((tiled_dma_kernel<E, GATED, KTAIL, WP, WQ, FP, FQ, false, DEEP>), grid, block, 0, stream, a, tiles_p,
                       tiles_q, group);
  } else {
    hipLaunchKernelGGL((tiled_dma_kernel<E, GATED, KTAIL, WP, WQ, FP, FQ>), grid, block, 0, stream, a, tiles_p, tiles_q,
                       group);
  }
}

template <class E, bool GATED, int WP, int WQ, int FP, int FQ>
hipError_t launch_dma(const GemmArgs& a, hipStream_t stream) {
  constexpr int BP = WP * FP * 32, BQ = WQ * FQ * 32;
  const int step_p = (a.tile_p > 0 && a.tile_p < BP) ? a.tile_p : BP;
  const int tiles_p = (a.np + step_p - 1) / step_p;
  const int tiles_q = (a.nq + BQ - 1) / BQ;
  if (tiles_p <= 0 || tiles_q <= 0) return hipSuccess;
  const dim3 grid((unsigned)(tiles_p * tiles_q));
  if (a.k % 64 == 0) {
    launch_dma_kernel<E, GATED, false, WP, WQ, FP, FQ>(grid, stream, a, tiles_p, tiles_q, GATED ? 4 : 2);
  } else {
    launch_dma_kernel<E, GATED, true, WP, WQ, FP, FQ>(grid, stream, a, tiles_p, tiles_q, GATED ? 4 : 2);
  }
  return hipGetLastError();
}

template <class E, bool GATED>
hipError_t launch_variant(int variant, const GemmArgs& a, hipStream_t stream) {
  switch (variant) {
    case 0: return launch_dma<E, GATED, 2, 2, 2, 2>(a, stream);
    case 2: return launch_dma<E, GATED, 2, 2, 2, 3>(a, stream);
    case 1:
    case 3: return launch_dma<E, GATED, 2, 4, 2, 2>(a, stream);
    case 4: return launch_dma<E, GATED, 2, 2, 2, 1>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

// Rounds of one-workgroup-per-compute-unit launches, as time. A partly filled round takes 0.75 .. 0.8 of a full one up to
// 160 workgroups (its compute units run at a higher clock) and grows from there to 1 (down 11008 -> 4096 in 256 x 256 tiles:
// 64 workgroups 162.7 us, 128 167.7, 160 173, 192 191, 224 208; in 256 x 160 tiles 64 112.7, 160 121.6, 208 139, 240 148.5,
// 256 152.7, 432 282).
static double pair16_rounds(long long wgs) {
  const double r = (double)(wgs % 256);
  const double part = r == 0.0 ? 0.0 : (r <= 160.0 ? 0.75 + 0.05 * r / 160.0 : 0.8 + 0.2 * (r - 160.0) / 96.0);
  return (double)(wgs / 256) + part;
}

// Time of a 256 x rows tile as a share of a 256 x 256 one (full rounds of the down product above: 216, 200.5, 177, 152.7
// us; gate/up 4096 x 28672, 224 tiles: 79.2, 70.5, 62.9, 57.9): per FLOP the narrow tile costs up to 14 % more.
struct NarrowTile {
  int rows;
  double cost;
};
static const NarrowTile kNarrow[] = {{256, 1.0}, {224, 0.91}, {192, 0.81}, {160, 0.715}};

// Activation rows per tile of the 256-weight-row kernel: 256, or 224, 192, 160 where these fit the rows and the compute
// units better, by the two measurements above. Only up to 512 large tiles (two rounds; gate/up, with seven times
// as many, four): beyond, the padding of the last tile and the last round weigh little against the dearer tiles and against
// blocked H, which these tiles do not read. A narrow tile must be ahead by 1 - `need`.
// 256 -> best, us: gate/up 4096 x 28672: 300 rows 78 -> 57 (160), 333 rows 79 -> 63 (192), 448 rows 85 -> 77 (224),
// 640 rows 150 -> 112 (160), 1000 rows stay (168, narrow 193 or more); 8192 x 57344, 520 rows 472 -> 412 (192); down
// 11008 -> 4096: 2500 rows 173 -> 153 (160), 3000 rows 191 -> 177 (192), 4300 rows 379 -> 282 (160); inputs that repeat from
// call to call. With inputs that come from memory: 2500 rows 195 -> 175, 4351 rows 408 -> 323.
// Rounds decide, not only padding, so row counts that 256 divides gain as well (from memory, too): 11008 -> 4096: 2304 rows
// 210 -> 169 (160), 2560 rows 212 -> 180 (160), 3072 rows 217 -> 199 (192), 4352 rows 408 -> 322 (160); 8192 x 28672, forward of
// 1280 rows 1328 -> 1293.
int pair16_tile_rows(bool gated, long long np, long long nq, double need) {
  const long long tp = (np + 255) / 256;
  if (tp * ((nq + 255) / 256) > (gated ? 1024 : 512)) return 256;
  int rows = 256;
  double best = pair16_rounds(tp * ((nq + 255) / 256)) * need;
  for (const NarrowTile& t : kNarrow) {
    const double cost = t.cost * pair16_rounds(tp * ((nq + t.rows - 1) / t.rows));
    if (t.rows < 256 && cost < best) {
      best = cost;
      rows = t.rows;
    }
  }
  return rows;
}

// Down projection of more than 256 rows with fewer than 129 large tiles: estimated time, us, of K split into `sp` parts
// (1: no split) on 128 x 128 tiles (tile_q 128) or 256 x tile_q ones of relative cost `tile_cost`. Every term was fitted to
// 2400 timings: the better plans of 346 problems (layers of common width and random ones; d 500 .. 8192, ff 1.5 .. 5 d,
// 257 .. 6000 rows, bf16 and fp16, weights rotated so that they come from memory): 5 % rms, and the plan it picks is 0.7 % slower
// than the fastest one on average, 12 % at worst.
//   * a workgroup's K tiles of 64: 1.19 us on 256 x 256 plus 1.9 us to fill and drain the pipeline (what shallow parts pay
//     for: 1996 rows of 2088 -> 736 in two parts of 17 tiles 34.4 us on 256 x 160, 22.2 on 128 x 128), 0.6 us on 128 x 128
//     alone on a compute unit (three stages), 1.6 .. 1.83 times that where 257 .. 512 workgroups share them two by two;
//   * a round costs the same whether 100 or 256 compute units are in it, but 256 workgroups of eight parts and more take
//     a fifth longer (4096 x 11008, 426 rows on 256 x 224: seven parts 53.7 us, eight 65.7);
//   * K no multiple of 64: rows share cache lines, all tiles take 1.22 times as long;
//   * the weights once from memory at 4.5 TB/s: combined with the above so that the larger one counts;
//   * parts: fp32 sums written and read back at 5 TB/s, and the summing kernel's launch and one dependent load per part.
static double split_time(int np, int nq, int k, int tile_q, double tile_cost, int sp) {
  const long long rows_p = tile_q == 128 ? 128 : 256;
  const long long wgs = ((np + rows_p - 1) / rows_p) * ((nq + tile_q - 1) / tile_q) * sp;
  const int kt = ((k + 63) / 64 + sp - 1) / sp;
  double t;
  if (tile_q == 128) {
    t = 0.6 * kt * (wgs <= 256 ? 1.0 : 1.6 + 0.23 * (double)(wgs - 257) / 255.0);
  } else {
    t = tile_cost * (1.9 + 1.19 * kt) * (wgs == 256 && sp >= 8 ? 1.2 : 1.0);
  }
  if (k % 64 != 0) t *= 1.22;
  const double w = 2.0 * (double)np * (double)k / 4.5e6;  // us
  t = sqrt(sqrt(t * t * t * t + w * w * w * w));
  if (sp > 1) t += 1.6 + 0.34 * sp + 8.0 * sp * (double)nq * (double)np / 5.0e6;
  return t;
}

// The fastest plan by split_time() among those that are resident at once (two 128 x 128 workgroups or one large one per
// compute unit: a second, partly filled round costs a whole one), whose parts are 8 (16) K tiles deep at least and whose
// partial sums stay under 256 MB. Tiles half filled with rows and row counts that are multiples of 256 need no rule of their own.
// Down projection, us, with 128 x 128 and 256 x 256 tiles only / with an estimate that knew neither the fill of short parts nor
// the three-stage ring and left half-filled tiles out / with this one: 28672 -> 8192, 264 rows 170 / 239 / 144; 8192 -> 2048,
// 371 rows 30.7 / 35.0 / 27.3; 2088 -> 736, 1996 rows 26.0 / 34.5 / 22.5; 3408 -> 1352, 910 rows 28.4 / 34.0 / 27.8; 11104 -> 5904,
// 479 rows 76.5 / 86.8 / 76.5; 11008 -> 4096, 333 rows 61.7 / 51.9 / 48.4, 1536 rows 133 / 133 / 120; 14336 -> 4096, 1024 rows
// level at 102. On 302 random problems none of these were fitted to: 0.896 of the first on average (95 % of them below 0.99, worst
// 1.06), 0.931 of the second (worst 1.02); on 260 with d of 64 .. 768 or ff of up to 12 d 0.869 (worst 1.11) and 0.881 (worst 1.09).
static SplitPlan mid_split_plan(int np, int nq, int k) {
  static const struct {
    int rows;
    double cost;  // of a K tile against 256 x 256
  } kTiles[] = {{128, 0.0}, {256, 1.0}, {224, 0.926}, {192, 0.863}, {160, 0.797}};
  SplitPlan p = {128, 1};
  double best = split_time(np, nq, k, 128, 0.0, 1);
  for (const auto& t : kTiles) {
    const bool small = t.rows == 128;
    const long long rows_p = small ? 128 : 256;
    const long long nt = ((np + rows_p - 1) / rows_p) * ((nq + t.rows - 1) / t.rows);
    long long smax = (small ? 512 : 256) / nt;
    const long long deep = small ? k / 512 : k / 1024;
    if (smax > deep) smax = deep;
    if (smax > 16) smax = 16;
    for (int sp = 2; sp <= (int)smax; ++sp) {
      if (4.0 * sp * (double)nq * (double)np > 256e6) break;
      const double cost = split_time(np, nq, k, t.rows, t.cost, sp);
      if (cost < best) {
        best = cost;
        p.tile = t.rows;
        p.splits = sp;
      }
    }
  }
  return p;
}

SplitPlan tiled_split_plan(int np, int nq, int k) {
  const long long t128 = (long long)((np + 127) / 128) * ((nq + 127) / 128);
  const long long t256 = (long long)((np + 255) / 256) * ((nq + 255) / 256);
  SplitPlan p = {256, 1};
  // One or two activation tiles with more large tiles than half the compute units: no split (see pick_tiled).
  // More rows: splitting can still pay by evening out rounds (288 tiles are two rounds of K, 288 x 3 are four
  // rounds of K / 3), up to 512 tiles.
  if (t128 <= 0 || t256 > (nq > 256 ? 512 : 128)) return p;
  if (nq > 256 && t256 < 129) return mid_split_plan(np, nq, k);
  if (nq > 256) {
    // From 129 large tiles up: the unsplit alternative is the 16x16x32 kernel on blocked H (~8 % faster than on row-major
    // H, which the split kernel reads), so a split, over several rounds if need be, must win by 15 %; its partials stay under
    // 256 MB. Estimated time in us on 256 compute units: MFMA work of the busiest one at 5.1 / 0.77 TFLOP/s (see
    // pair16_rounds() for partly filled rounds) plus the fp32 partials at ~5 TB/s.
    // Unsplit tiles of fewer rows need no place in the comparison: of 35 problems that split here (256 x 256, us) 34 are
    // slower on the best of them (28672 -> 8192: 2079 rows 839 -> 888 on 256 x 160, 2419 rows 907 -> 916; 31856 -> 5408, 3060
    // rows 1078 -> 1165; the forward of 2079 rows of 8192 x 28672 2257 -> 2300), one is faster (31400 -> 6648, 1170 rows 638 -> 581).
    const int nkt = (k + 63) / 64;
    double best = 0.0, unsplit = 0.0;
    p.splits = 1;
    for (int sp = 1; sp <= 16 && (sp == 1 || sp <= k / 1024); ++sp) {
      if (sp > 1 && 4.0 * sp * (double)nq * (double)np > 256e6) break;
      const double kper = 64.0 * ((nkt + sp - 1) / sp);
      const double mfma = 2.0 * kper * 256 * 256 * 0.77 * pair16_rounds(t256 * sp) / 5.1e6;
      const double cost = mfma + (sp > 1 ? 8.0 * sp * (double)nq * (double)np / 5.0e6 : 0.0);
      if (sp == 1) unsplit = mfma;
      if (best == 0.0 || cost < best) {
        best = cost;
        p.splits = sp;
      }
    }
    if (p.splits > 1 && best > 0.85 * unsplit) p.splits = 1;
    return p;
  }
  int by_k;
  long long tiles;
  if (t128 < 256) {
    p.tile = 128;
    tiles = t128;
    by_k = k / 512;  // at least 8 K tiles of 64 per partition
  } else {
    tiles = t256;
    by_k = k / 1024;
  }
  // One tile of activation rows: three-stage workgroups, one per compute unit, beat two two-stage ones (less
  // partial-sum traffic as well); 129..256 rows take one 128 x 256 tile per workgroup for the same reason.
  int target = 512;
  if (nq <= 128) {
    target = 256;
  } else if (nq <= 256) {
    // ... as long as that still fills most compute units (narrow outputs: 1024 x 2816 at 256 rows, 40 wide
    // workgroups 18.3 us, unsplit 128 x 128 tiles 21.4 us)
    const long long wide = (np + 127) / 128;
    long long sw = (256 + wide - 1) / wide;
    if (sw > by_k) sw = by_k;
    if (sw > 16) sw = 16;
    if (wide * sw >= 192) {
      p.tile = nq <= 192 ? 130 : 129;  // 128 x 192 does a quarter less MFMA work where 192 rows are enough
      tiles = wide;
      target = 256;
    }
  }
  // all workgroups resident at once: rounding up put 40 tiles x 7 splits on 256 one-workgroup compute units
  // (5120 x 13824 at 256 rows: 86 us, against 68 us at 257 rows)
  int splits = (int)(target / tiles);
  if (splits > by_k) splits = by_k;
  if (splits > 16) splits = 16;
  p.splits = splits < 1 ? 1 : splits;
  if (p.splits == 1 && p.tile == 256) p.tile = 128;  // unsplit mid-size problems keep the smaller tile
  return p;
}


namespace {
template <class E, int SPLITS>
hipError_t launch_splitk_reduce_n(const GemmArgs& a, hipStream_t stream) {
  if constexpr (SPLITS > 16) {
    return hipErrorInvalidValue;  // no plan splits K into more parts
  } else {
    if (a.splits != SPLITS) return launch_splitk_reduce_n<E, SPLITS + 1>(a, stream);
    const long long work = (long long)a.nq * ((a.np + 3) / 4);
    hipLaunchKernelGGL((splitk_reduce_kernel<E, SPLITS>), dim3((unsigned)((work + 255) / 256)), dim3(256), 0, stream, a.partial,
                       a.nq, a.np, (unsigned short*)a.O, a.ldo);
    return hipGetLastError();
  }
}
template <class E>
hipError_t launch_splitk_reduce(const GemmArgs& a, hipStream_t stream) {
  return launch_splitk_reduce_n<E, 2>(a, stream);
}

template <class E, int WP, int WQ, int FP, int FQ>
hipError_t launch_splitk_one(const GemmArgs& a, hipStream_t stream) {
  constexpr int BP = WP * FP * 32, BQ = WQ * FQ * 32;
  const int tiles_p = (a.np + BP - 1) / BP;
  const int tiles_q = (a.nq + BQ - 1) / BQ;
  if (tiles_p <= 0 || tiles_q <= 0) return hipSuccess;
  const dim3 grid((unsigned)(tiles_p * tiles_q), (unsigned)a.splits);
  const int group = 2;
  if (a.k % 64 == 0) {
    launch_dma_kernel<E, false, false, WP, WQ, FP, FQ>(grid, stream, a, tiles_p, tiles_q, group);
  } else {
    launch_dma_kernel<E, false, true, WP, WQ, FP, FQ>(grid, stream, a, tiles_p, tiles_q, group);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.splits <= 1) return e;
  return launch_splitk_reduce<E>(a, stream);
}
}  // namespace

hipError_t launch_tiled_splitk(int dtype, int tile, const GemmArgs& a, hipStream_t stream) {
  // up to 64 rows the 128 x 64 form of the same split: half the LDS reads and MFMAs per weight byte and four stages instead of
  // three (down 11008 -> 4096, 33 rows 22.7 -> 21.3 us, 64 rows 25.5 -> 24.6; forward 5120 x 13824 fp16, 40 rows 79.0 -> 77.2)
  if (tile == 128 && a.nq <= 64) {
    return dtype == 0 ? launch_splitk_one<Bf16, 2, 2, 2, 1>(a, stream) : launch_splitk_one<Fp16, 2, 2, 2, 1>(a, stream);
  }
  if (tile == 128) {
    return dtype == 0 ? launch_splitk_one<Bf16, 2, 2, 2, 2>(a, stream) : launch_splitk_one<Fp16, 2, 2, 2, 2>(a, stream);
  }
  if (tile == 130) {  // 128 output features x 192 activation rows
    return dtype == 0 ? launch_splitk_one<Bf16, 2, 2, 2, 3>(a, stream) : launch_splitk_one<Fp16, 2, 2, 2, 3>(a, stream);
  }
  if (tile == 129) {  // 128 output features x 256 activation rows, 8 waves
    return dtype == 0 ? launch_splitk_one<Bf16, 2, 4, 2, 2>(a, stream) : launch_splitk_one<Fp16, 2, 4, 2, 2>(a, stream);
  }
  // 256 x tile on the 16x16x32 kernel, then the reduction
  GemmArgs b = a;
  b.tile_q = tile;
  const hipError_t e = launch_pair16_splitk(dtype, b, stream);
  if (e != hipSuccess || a.splits <= 1) return e;
  return dtype == 0 ? launch_splitk_reduce<Bf16>(a, stream) : launch_splitk_reduce<Fp16>(a, stream);
}

hipError_t launch_block_rows(const void* src, long long ld, int rows, int k, void* dst, bool gated_order,
                             hipStream_t stream) {
  const int nkt = (k + 31) / 32;
  const int panels = (rows + 255) / 256;
  if (nkt <= 0 || panels <= 0) return hipSuccess;
  hipLaunchKernelGGL(block_rows_kernel, dim3((unsigned)((nkt + 3) / 4), (unsigned)panels), dim3(256), 0, stream,
                     (const unsigned short*)src, ld, rows, k, (unsigned char*)dst, nkt, gated_order ? 1 : 0);
  return hipGetLastError();
}

int tiled_variant_count() { return (int)(sizeof(kVariants) / sizeof(kVariants[0])); }
int pair16_variant() { return kPair16Variant; }
const TiledVariant& tiled_variant(int variant) { return kVariants[variant]; }

// row-major operands; the 256 x 256 variant is the 16x16x32 kernel with GemmArgs::layout 0
hipError_t launch_tiled(int variant, int dtype, bool gated, const GemmArgs& a, hipStream_t stream) {
  if (variant == kPair16Variant) return launch_pair16(dtype, gated, a, stream);
  if (dtype == 0) {
    return gated ? launch_variant<Bf16, true>(variant, a, stream) : launch_variant<Bf16, false>(variant, a, stream);
  }
  return gated ? launch_variant<Fp16, true>(variant, a, stream) : launch_variant<Fp16, false>(variant, a, stream);
}

}  // namespace fsw
