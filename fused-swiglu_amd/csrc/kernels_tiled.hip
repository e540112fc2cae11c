// Plans of the tiled kernels (which tile, how many K parts), the split-K reduction and the row-major -> panel-blocked copy. The
// kernels live in kernels_pair16.hip (256 weight rows a tile, prefill) and mid_kernel.h (smaller tiles).
//
// Orientation of both. The MFMA "A" operand (rows of the result block) is fed with WEIGHT rows and the "B" operand (columns of
// the result) with ACTIVATION rows, so an accumulator lane owns one activation row m and runs of consecutive output features,
// which makes the stores vectors along the contiguous dimension of the output, and the gating of the gated product
//   H[m, j] = up * silu(gate), up = X[m,:].W13[2j,:], gate = X[m,:].W13[2j+1,:]   (swiglu.cu:111-394)
// plain per-lane fp32 math with no cross-lane traffic; the plain product is Y[m, n] = H[m,:].W2[n,:] (no counterpart there).
#include <math.h>

#include "fsw_internal.h"
#include "fsw_device.h"

namespace fsw {

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
    // the first five name ranges of rows of the producer / consumer kernel (mid_kernel.h) and, forced, its tile
    {"dma_128x128"},
    {"dma8w_128x256"},  // id 3 under an older number
    {"dma_128x192"},
    {"dma8w_128x256"},
    {"dma_128x64"},
    {"pair16_256x256"}, // the prefill kernel (kernels_pair16.hip), row-major operands
};

}  // namespace

// Activation-row tiles per raster band of the 256 x 256 kernel (mid_kernel uses 4 for the gate/up and 2 for the down
// product): 4, i.e. the 32 tiles an XCD runs at once are 4 activation panels x 8 weight
// panels (12 operand panels through its L2 per round). The down product of tall problems (32 activation tiles or
// more, 16 weight panels, 14336-deep K) measures level to 1 % slower that way and keeps bands of 2; with fewer
// activation tiles bands of 4 win (4096 x 4096 x 11008: 244 -> 236 us, 2048 x 8192 x 28672 fp16: 639 -> 633 us).
int raster_group(bool gated, int tiles_q) { return gated ? 4 : (tiles_q >= 32 ? 2 : 4); }

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

// Gate/up of rows that are no whole 128-byte lines: a K pair of 64 columns is two lines of every row of the tile, and these copies,
// not the MFMAs, are the time: 62 bytes per ns and compute unit where all weight lines come from HBM (one tile of activation
// rows), 76 where the L2 serves some (48 problems of 130 .. 700 rows: -18 .. +10 %).
double pair16_ragged_time(int np, int nq, int k, int rows) {
  double cost = 1.0;
  for (const NarrowTile& t : kNarrow)
    if (t.rows == rows) cost = t.cost;
  const long long tq = (nq + rows - 1) / rows;
  const double copy = (256 + rows) * 0.256 / (tq == 1 ? 62.0 : 76.0), mul = 1.19 * cost;
  return 3.5 + pair16_rounds((long long)((np + 255) / 256) * tq) * ((k + 63) / 64 + 2) * (copy > mul ? copy : mul);
}

// Down projection of more than 256 rows with fewer than 129 large tiles: estimated time, us, of K split into `sp` parts
// (1: no split) on 128 x 128 tiles (tile_q 128) or 256 x tile_q ones of relative cost `tile_cost`. Every term was fitted to
// 2400 timings: the better plans of 346 problems (layers of common width and random ones; d 500 .. 8192, ff 1.5 .. 5 d,
// 257 .. 6000 rows, bf16 and fp16, weights rotated so that they come from memory): 5 % rms, and the plan it picks is 0.7 % slower
// than the fastest one on average, 12 % at worst.
//   * a workgroup's K tiles of 64: 1.19 us on 256 x 256 plus 1.9 us to fill and drain the pipeline (what shallow parts pay
//     for: 1996 rows of 2088 -> 736 in two parts of 17 tiles 34.4 us on 256 x 160, 22.2 on 128 x 128), 0.6 us on 128 x 128
//     alone on a compute unit, 1.6 .. 1.83 times that with 257 .. 512 workgroups. The 128 x 128 terms are those of the kernel that mid_kernel
//     replaced there; they still draw the line between the 256-row kernel and mid_kernel, which then plans its own tile and parts by
//     mid_plan() and is faster than they say (down 2816 -> 1024, 512 rows 15.9 -> 13.5; 8192 -> 2048, 371 rows 27.0 -> 25.7);
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

static const struct {
  int rows;
  double cost;  // of a K tile against 256 x 256
} kSplitTiles[] = {{128, 0.0}, {256, 1.0}, {224, 0.926}, {192, 0.863}, {160, 0.797}};

// The fastest plan by split_time() among those of one round (256 large workgroups, 512 of 128 x 128: a second, partly filled round costs
// a whole one; mid_kernel's own plan takes these parts as the most it may have), whose parts are 8 (16) K tiles deep at least and whose
// partial sums stay under 256 MB. Tiles half filled with rows and row counts that are multiples of 256 need no rule of their own.
// Down projection, us, with 128 x 128 and 256 x 256 tiles only / with an estimate that knew neither the fill of short parts nor
// the three-stage ring and left half-filled tiles out / with this one: 28672 -> 8192, 264 rows 170 / 239 / 144; 8192 -> 2048,
// 371 rows 30.7 / 35.0 / 27.3; 2088 -> 736, 1996 rows 26.0 / 34.5 / 22.5; 3408 -> 1352, 910 rows 28.4 / 34.0 / 27.8; 11104 -> 5904,
// 479 rows 76.5 / 86.8 / 76.5; 11008 -> 4096, 333 rows 61.7 / 51.9 / 48.4, 1536 rows 133 / 133 / 120; 14336 -> 4096, 1024 rows
// level at 102. On 302 random problems none of these were fitted to: 0.896 of the first on average (95 % of them below 0.99, worst
// 1.06), 0.931 of the second (worst 1.02); on 260 with d of 64 .. 768 or ff of up to 12 d 0.869 (worst 1.11) and 0.881 (worst 1.09).
static SplitPlan mid_split_plan(int np, int nq, int k) {
  SplitPlan p = {128, 1};
  double best = split_time(np, nq, k, 128, 0.0, 1);
  for (const auto& t : kSplitTiles) {
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

double pair16_split_time(int np, int nq, int k, const SplitPlan& plan) {
  double cost = 1.0;
  for (const auto& t : kSplitTiles)
    if (t.rows == plan.tile) cost = t.cost;
  return split_time(np, nq, k, plan.tile, cost, plan.splits);
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
  // Up to 256 rows mid_plan() plans what runs; these parts name the range and are the least scratch that a call of 49 .. 256 rows has to
  // bring (down_least). One tile of activation rows: one workgroup per compute unit.
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

}  // namespace

hipError_t launch_splitk_reduce(int dtype, const GemmArgs& a, hipStream_t stream) {
  return dtype == 0 ? launch_splitk_reduce<Bf16>(a, stream) : launch_splitk_reduce<Fp16>(a, stream);
}

// 256 x tile on the 16x16x32 kernel, then the reduction
hipError_t launch_tiled_splitk(int dtype, int tile, const GemmArgs& a, hipStream_t stream) {
  GemmArgs b = a;
  b.tile_q = tile;
  const hipError_t e = launch_pair16_splitk(dtype, b, stream);
  return e != hipSuccess || a.splits <= 1 ? e : launch_splitk_reduce(dtype, a, stream);
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
const TiledVariant& tiled_variant(int variant) { return kVariants[variant]; }

}  // namespace fsw
