// C-ABI dispatcher: argument validation (host only), regime selection by activation-row count, launches.
// Replaces the host launcher swiglu_fwd<TA,TB,TC> (swiglu.cu:397-525) and the convenience op's shape
// derivation (swiglu.cu:538-553); the public contract is include/fsw.h.
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>

#include "fsw.h"
#include "fsw_internal.h"

namespace {

thread_local int g_last_hip_error = 0;
// Kernel override of fsw_set_variant, per calling thread: a thread's workspace queries and launches always agree,
// and no thread can change another's kernel choice. family 0 = gate/up, 1 = down.
thread_local int g_forced_variant[2] = {-1, -1};

constexpr int VARIANT_SKINNY = 100;          // id of the weight-streaming kernel in fsw_set_variant
constexpr int VARIANT_DECODE_STREAM = 102;   // M <= 16: the streaming kernel of kernels_decode.hip, one phase per launch
constexpr int VARIANT_DECODE_FUSED = 101;    // fsw_mlp only: single-launch decode forward (family 0)
constexpr int VARIANT_DECODE_FUSED_FAIL = 103;  // 101 with a device-wide barrier that cannot complete (failure-path test)
constexpr int VARIANT_STREAM_SPLIT = 104;    // family 1, fsw_mlp only: split-K streaming down projection for M <= 32
// the 256 x 256 kernel with narrower tiles: VARIANT_NARROW + 5, 6, 7 = 160, 192, 224 activation rows per tile
constexpr int VARIANT_NARROW = 110;
constexpr int VARIANT_MID = 200;             // VARIANT_MID + i: tile i of the producer / consumer kernel, whole tiles, unsplit
constexpr int64_t MAX_DIM = 1LL << 30;       // every size is cast to int inside the kernels
constexpr int64_t MAX_LD = 1LL << 21;        // keeps tile-relative byte offsets below 2^31

bool aligned16(const void* p) { return (((uintptr_t)p) & 15) == 0; }

// gfx950 check, cached per device ordinal.
int check_device() {
  static std::atomic<int> ok_mask[64];  // 0 unknown, 1 ok, 2 not gfx950 (zero-initialised; racing writers agree)
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    g_last_hip_error = (int)e;
    return FSW_E_DEVICE;
  }
  if (dev < 0 || dev >= 64) return FSW_E_DEVICE;
  int state = ok_mask[dev].load(std::memory_order_relaxed);
  if (state == 0) {
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, dev);
    if (e != hipSuccess) {
      g_last_hip_error = (int)e;
      return FSW_E_DEVICE;
    }
    state = (strncmp(prop.gcnArchName, "gfx950", 6) == 0) ? 1 : 2;
    ok_mask[dev].store(state, std::memory_order_relaxed);
  }
  return state == 1 ? FSW_OK : FSW_E_DEVICE;
}

// indices of the tiled kernels (tiled_variant() of kernels_tiled.hip)
constexpr int V_128x128 = 0, V_128x192 = 2, V_8W_128x256 = 3, V_128x64 = 4, V_256x256 = 5;

// Range of rows of a tiled launch. The 128-row names stand for the producer / consumer kernel (mid_kernel.h), which chooses its
// tile by an estimate of its own; they tell the rows that one of its launches shares the weights between (128 x 64: up to 64, 128 x
// 128 and so on) and are what fsw_set_variant forces. The others are the 256-row kernel.
// `narrow_need`: a narrower large tile is taken only if its estimated time is below this share of 256 x 256's
int pick_tiled(int family, int64_t m, int64_t np, int64_t k, double narrow_need = 0.95) {
  const int64_t tiles256 = ((np + 255) / 256) * ((m + 255) / 256);
  // 256 x 256 tiles down to half-filled compute units (129 tiles); up to 128 activation rows are one weight stream whatever the
  // tile count.
  if (tiles256 < 129 || m <= 128) {
    const int64_t tp = (np + 127) / 128;
    if (family == 0 && m > 128 && tp * ((m + 127) / 128) > 256) {
      if (m <= 256) return m <= 192 ? V_128x192 : V_8W_128x256;
      const int64_t w192 = tp * ((m + 191) / 192), w256 = tp * ((m + 255) / 256);
      if (k >= 2048 && w192 >= 224 && w192 <= 256) return V_128x192;
      if (k >= 2048 && w256 >= 224 && w256 <= 256) return V_8W_128x256;
    }
    return (family == 0 && m <= 64) ? V_128x64 : V_128x128;
  }
  const int rows = fsw::pair16_tile_rows(family == 0, np, m, narrow_need);
  if (rows != 256) return VARIANT_NARROW + rows / 32;
  if (family == 0 && tiles256 > 256 && tiles256 <= 512) {
    // A few large tiles more than compute units: the second round is nearly empty, while smaller tiles come in shorter rounds.
    const int64_t tiles128 = ((np + 127) / 128) * ((m + 127) / 128);
    if (((tiles128 + 255) / 256) * 44 < ((tiles256 + 255) / 256) * 100) return V_128x128;
  }
  return V_256x256;
}

// Most activation rows of the decode range, whose launches are weight streaming by skinny_kernel or, where that is faster
// (mid_wanted), by the producer / consumer kernel: fewer the larger the weights. K == 0 stays with the weight-streaming kernels,
// which write the all-zero result.
int64_t decode_rows(int family, int64_t np, int64_t k) {
  if (k <= 0) return 64;
  const int64_t d_ff = family == 0 ? (np / 2) * k : np * k;
  return d_ff < ((int64_t)1 << 25) ? 48 : d_ff < ((int64_t)1 << 27) ? 32 : 16;
}

// whether these rows are in the decode range
bool few_rows(int family, int64_t m, int64_t np, int64_t k) {
  if (m > decode_rows(family, np, k)) return false;
  // from a dozen rows on a gate/up matrix of 200 .. 256 pieces of 128 rows is past that range
  const int64_t tiles = (np + 127) / 128;
  return !(family == 0 && m >= 12 && k > 0 && tiles >= 200 && tiles <= 256);
}

int resolve_variant(int family, int64_t m, int64_t np, int64_t k) {
  const int forced = g_forced_variant[family];
  if (forced == VARIANT_DECODE_FUSED || forced == VARIANT_DECODE_FUSED_FAIL || forced == VARIANT_DECODE_STREAM ||
      forced == VARIANT_STREAM_SPLIT)
    return m <= 64 ? VARIANT_SKINNY : pick_tiled(family, m, np, k);
  if (forced >= 0 && !(forced == VARIANT_SKINNY && m > 64)) return forced;
  if (few_rows(family, m, np, k)) return VARIANT_SKINNY;  // decode and small batches: weight streaming, HBM bound
  return pick_tiled(family, m, np, k);
}

// the weight-streaming kernels need no scratch and no blocked operands
bool streams_weights(int family, int64_t m, int64_t np, int64_t k) {
  return m <= 64 && resolve_variant(family, m, np, k) == VARIANT_SKINNY;
}

// M <= 16 with very large weight matrices runs on the persistent streaming kernel of kernels_decode.hip (one phase
// per launch) unless the caller forces the skinny kernel. Measured whole forwards at M = 16, skinny vs streaming:
// 8192 x 28672: 254 vs 233 us; 5120 x 13824: 87.6 vs 90.3; 4096 x 14336: 61.1 vs 63.4; 4096 x 11008: 50.0 vs 54.5;
// 2048 x 8192: 26.9 vs 31.6: the streaming kernel needs many tiles per CU to balance and to amortise its single
// reduction. K == 0 stays with the skinny kernel, which writes the all-zero result.
bool decode_stream_wanted(int family, int64_t m, int64_t rows, int64_t k) {
  if (m > 16 || k <= 0 || g_forced_variant[family] == VARIANT_SKINNY) return false;
  if (g_forced_variant[family] == VARIANT_DECODE_STREAM) return true;
  return rows * k >= (family == 0 ? (int64_t)1 << 28 : (int64_t)1 << 27);  // = d * ff >= 2^27 for either projection
}

int finish(hipError_t e) {
  if (e != hipSuccess) {
    g_last_hip_error = (int)e;
    return FSW_E_LAUNCH;
  }
  return FSW_OK;
}

bool narrow_variant(int v) { return v >= VARIANT_NARROW + 5 && v <= VARIANT_NARROW + 7; }

bool mid_variant(int v) { return v >= VARIANT_MID && v < VARIANT_MID + fsw::mid_tile_count(); }
bool dma_variant(int v) { return (v >= 0 && v < V_256x256) || mid_variant(v); }

// Rows of a dense operand of `k` columns that are no whole 128-byte lines.
bool ragged(int64_t k) { return k % 64 != 0; }

// Estimated time, us, of skinny_kernel's down projection of up to 48 rows and a K of up to 8192: 7 % rms over 448 timings. Rounds of one
// workgroup of 16 features per compute unit, the activations (in blocks of 16 rows) that they all fetch from the L2, and more of these in
// pieces of lines with ragged rows.
double skinny_down_time(int64_t np, int64_t m, int64_t k, bool rag) {
  const double tiles = (double)((np + 15) / 16), rounds = (double)(((np + 15) / 16 + 255) / 256);
  const double over = tiles > 256 ? tiles / 256 : 1.0, fill = tiles / (256 * rounds);
  const double blocks = 0.3 * (double)((m + 15) / 16) + 0.7 * (double)m / 16;
  return 2.412 + (double)k / 1024 * (1.088 * rounds + blocks * over * (0.487 * fill + (rag ? 0.36 : 0.0)));
}

// Whether a launch that the rules above give to the kernels for few rows (`v`: VARIANT_SKINNY or a 128-row tile) runs the
// producer / consumer kernel. skinny_kernel (one launch, one workgroup per 32 weight rows, 16 in the down projection) stays
// where its workgroups fit the compute units at once and the call is short. Gate/up, us, skinny -> mid: 5632 x 1024 (176
// workgroups) 16 rows 5.1 -> 6.4; 8192 x 1536 (256) 24 rows 7.4 -> 8.1; 11264 x 2048 (352) 4 rows 10.5 -> 10.8, 16 rows 11.7 ->
// 10.9, 24 rows 15.4 -> 11.0; 7808 x 1320 (244, ragged) 4 rows 6.7 -> 7.2, 24 rows 8.0 -> 7.3; 16016 x 3000 (ragged) 1 row 22.0 ->
// 19.4. Down, where K is split and a summing launch follows: 8192 -> 3072 16 rows 12.4 -> 13.1, 24 rows 15.2 -> 13.4; 13824 ->
// 5120 (320 workgroups, two rounds) 1 row 31.3 -> 25.2; 16416 -> 4880 (ragged) 1 row 40.5 -> 28.7; up to 2048 features, where
// skinny_kernel has 4 or 8 a workgroup, 2816 -> 1024 16 rows 4.7 -> 6.4, 8192 -> 2048 16 rows 10.1 -> 10.7, 16384 -> 2048 1 row
// 16.2 -> 14.2, 16 rows 19.6 -> 15.2; ragged 5360 -> 1344 1 row 6.3 -> 8.1, 12 rows 8.2 -> 8.4, 16 rows 9.0 -> 8.4. Matrices of the
// persistent streaming kernel (decode_stream_wanted): gate/up 57344 x 8192 1 row 144.1 -> 142.4, 16 rows 147.4 -> 136.5; 46336 x 7000
// (ragged) 1 row 124.0 -> 98.8; down 28672 -> 8192 1 and 4 rows level, 16 rows 84.1 -> 72.1; 23168 -> 7000 1 row 55.5 -> 52.1.
// The 256-row kernel fetches rows that are no whole lines by K tiles, every line twice; the gate/up product of such rows takes the
// kernel whose estimated time is less (47 problems of 130 .. 700 rows: it chose the slower one four times, by 7 % at most; 38880 x
// 5800 130 rows 150.4 -> 119.0, 256 rows 189.6 -> 138.1; 43680 x 7592 279 rows 348 -> 241; 24160 x 3448 409 rows stays, 93.6 and 105).
bool mid_wanted(int family, int v, int64_t m, int64_t np, int64_t k, bool rag) {
  // what resolve_variant() makes of the forced id: a weight-streaming id takes up to 64 rows, more run the range's own kernel
  if (g_forced_variant[family] >= 0) return dma_variant(v);
  if (k <= 0) return false;
  if (family == 0 && rag && (v == V_256x256 || narrow_variant(v)) && m <= 1024) {
    const int rows = narrow_variant(v) ? 32 * (v - VARIANT_NARROW) : 256;
    return fsw::mid_plan(true, (int)np, (int)m, (int)k, true, 1, 1).us < fsw::pair16_ragged_time((int)np, (int)m, (int)k, rows);
  }
  if (!(v == VARIANT_SKINNY || dma_variant(v))) return false;
  if (v != VARIANT_SKINNY) return true;
  const int64_t bytes = 2 * np * k;
  if (family == 0) {
    const int64_t tiles = (np + 31) / 32;
    // Ragged rows of few workgroups, us, skinny -> mid: 17 rows 2048 x 1160 6.1 -> 6.8, 2672 x 1336 6.5 -> 7.1, 4096 x 1640 8.3 -> 8.1, 6016 x
    // 2008 9.9 -> 9.4; 32 rows 4096 x 1000 5.9 -> 6.4, 7808 x 1320 8.2 -> 7.7; 48 rows 1024 x 392 4.2 -> 4.6, 6000 x 968 6.9 -> 7.2, 4096 x 1000
    // 6.6 -> 6.4, 2832 x 1096 7.1 -> 6.8.
    if (m > 16) return tiles > 256 || (rag && (m <= 32 ? bytes >= (int64_t)12 << 20 : k >= 1000));
    if (tiles <= 256 || (m <= 8 && bytes < (int64_t)56 << 20)) return false;
    // 9 .. 16 rows, 9 / 16 rows, us, skinny -> mid: 8704 x 512 4.5 -> 5.0 / 4.6 -> 5.0, 8704 x 1024 6.5 -> 6.8 / 6.7 -> 6.8, 12800 x 1024 level / 7.4
    // -> 7.1, 24576 x 512 6.4 -> 6.6 / level; ragged 10000 x 520 5.3 -> 5.6 / 5.4 -> 5.7, 10000 x 1000 7.5 -> 7.7 / 7.9 -> 7.7, 8800 x 1320 9.3 ->
    // 8.8 / 9.9 -> 8.9.
    if (m > 8 && !(rag ? k * m >= 11000 : k >= 1024 && bytes >= (int64_t)22 << 20)) return false;
    // Up to 8 rows skinny_kernel is as fast where its workgroups leave less than an eighth of their rounds of compute units empty (less than a
    // sixteenth above four rounds). us, 1 / 8 rows, skinny -> mid: 28672 x 4096 (896 workgroups) 37.6 -> 36.9 / 38.0 -> 36.6; 32768 x 4096
    // (1024) 41.5 -> 41.5 / 40.9 -> 41.4; 24576 x 4608 (768) 35.9 -> 35.4 / level; 40960 x 5120 (1280) 62.5 -> 63.4 / level; 22016 x 4096
    // (688) 29.8 -> 29.2 / 29.7 -> 29.1; 16128 x 2880 (504) 16.3 -> 16.9; 39424 x 5568 (1232) 65.1 -> 65.6. With more of them empty:
    // 27648 x 5120 (864) 46.2 -> 43.4 / 48.2 -> 43.6; 20480 x 2560 (640) 18.9 -> 18.3; 37760 x 6336 (1180) 73.9 -> 71.3. Rows a multiple
    // of 2 KB apart are the exception: its eight-wave workgroups walk K in step and meet on the same memory channels (16384 x 4096 25.9 ->
    // 21.9, 16384 x 2048 13.4 -> 12.4, 16384 x 3072 18.2 -> 17.5).
    // Up to 4 rows with 257 .. 448 workgroups, which share the compute units unevenly but run at once, us, skinny -> mid: 8448 x 4800 1 row 19.1 ->
    // 23.3, 10240 x 3776 16.1 -> 16.8, 12288 x 6016 25.1 -> 27.7, 13824 x 4800 21.4 -> 22.8, 15872 x 4800 level; 8 rows 10240 x 3776 17.5 -> 16.6.
    if (m <= 4 && !rag && tiles <= 448 && k % 1024 != 0) return false;
    const int64_t rounds = (tiles + 255) / 256, empty = 256 * rounds - tiles;
    if (m <= 8 && !rag && !decode_stream_wanted(0, m, np, k) && empty <= (rounds <= 4 ? 32 : 16) * rounds)
      return tiles <= 640 && k % 1024 == 0;
    return true;
  }
  const int64_t tiles = (np + 15) / 16;
  // K of up to 8192, where the second launch weighs most: only where the estimated time is less than skinny_kernel's (448 timings: the pair
  // of estimates picks a kernel 0.3 % slower than the faster one on average, 12 % at worst; the rules below alone 11 % and 90 %). Not for ragged
  // rows of more than 256 workgroups, where it flatters skinny_kernel (3800 -> 6000 1 row 12.9 -> 11.8); for up to 4 ragged rows it is too high
  // (7312 -> 2376 1 row 10.1 -> 11.2). us, skinny -> mid: 17 rows 1000 -> 512
  // 3.2 -> 6.1, 2048 -> 4096 5.9 -> 8.5, 6144 -> 2048 11.2 -> 10.2; 48 rows 2048 -> 2048 6.7 -> 8.0, 4104 -> 4096 15.1 -> 13.0; 1 row 1024 -> 5120
  // 4.3 -> 6.2, 4096 -> 8192 12.9 -> 17.1, 6144 -> 5120 15.1 -> 14.0; ragged 1 row 3080 -> 4096 6.8 -> 9.2, 4104 -> 4880 13.0 -> 11.1, 16 rows
  // 4744 -> 3104 10.9 -> 10.3.
  if (k <= 8192 && (m > 16 || tiles > 128) && !(rag && tiles > 256 && k >= 3400) &&
      fsw::mid_plan(false, (int)np, (int)m, (int)k, rag, 0, 16).us >= (rag && m <= 4 ? 0.86 : 0.98) * skinny_down_time(np, m, k, rag))
    return false;
  if (m > 16) return rag || bytes >= (int64_t)8 << 20;
  if (tiles <= 128) return k > 12288 ? m > 4 || np > 1024 : rag && m > 12 && bytes >= (int64_t)12 << 20;
  if (rag) return bytes >= (int64_t)14 << 20 || (m >= 8 && bytes >= (int64_t)7 << 20);
  if (bytes >= (int64_t)1 << 28) return m > 4;
  return tiles > 256;
}

// tile of a forced variant
fsw::MidPlan forced_mid_plan(int v) {
  if (mid_variant(v)) return {v - VARIANT_MID, fsw::mid_tile_rows(v - VARIANT_MID), 1, 0.0};
  const int bq = v == V_128x64 ? 64 : v == V_128x192 ? 192 : v == V_128x128 ? 128 : 256;
  return {fsw::mid_tile_index(128, bq), 128, 1, 0.0};
}

// the 256-row kernel, row-major operands (GemmArgs::layout 0)
hipError_t launch_large(int v, int dtype, bool gated, fsw::GemmArgs& a, hipStream_t stream) {
  if (narrow_variant(v)) a.tile_q = 32 * (v - VARIANT_NARROW);
  return fsw::launch_pair16(dtype, gated, a, stream);
}

}  // namespace

extern "C" {

int fsw_version(void) { return 2000; }

const char* fsw_strerror(int code) {
  switch (code) {
    case FSW_OK: return "ok";
    case FSW_E_NULL: return "fsw: a required pointer is NULL";
    case FSW_E_DTYPE: return "fsw: unsupported element type (expected bf16 or fp16)";
    case FSW_E_SHAPE: return "fsw: bad shape (negative size, odd N, or size out of range)";
    case FSW_E_LD: return "fsw: leading dimension smaller than the row it strides";
    case FSW_E_ALIGN: return "fsw: K/FF and leading dimensions must be multiples of 8 and inputs 16-byte aligned";
    case FSW_E_WORKSPACE: return "fsw: workspace missing or too small";
    case FSW_E_LAUNCH: return "fsw: the HIP runtime rejected the kernel launch";
    case FSW_E_DEVICE: return "fsw: the current device is not a gfx950 GPU";
    case FSW_E_VARIANT: return "fsw: unknown kernel variant";
    case FSW_E_STATIC_LIMIT: return "fsw: the problem needs more scratch than the library's static 64 MiB; use fsw_mlp";
    default: return "fsw: unknown error code";
  }
}

int fsw_last_hip_error(void) { return g_last_hip_error; }

int fsw_decode_barrier_failures(void) {
  const int drc = check_device();
  if (drc != FSW_OK) return drc;
  int count = 0;
  const int rc = finish(fsw::decode_barrier_failures(&count));
  return rc != FSW_OK ? rc : count;
}

int fsw_set_variant(int family, int variant) {
  if (family < 0 || family > 1) return FSW_E_VARIANT;
  // the barrier that cannot complete exists for the failure-path test only: refused unless the process's
  // environment holds FSW_TEST_HOOKS=1, so a caller cannot leave it set by accident and get forwards without Y
  if (variant == VARIANT_DECODE_FUSED_FAIL) {
    const char* hooks = getenv("FSW_TEST_HOOKS");
    if (!hooks || strcmp(hooks, "1") != 0) return FSW_E_VARIANT;
  }
  if (variant >= 0 && variant != VARIANT_SKINNY && variant != VARIANT_DECODE_STREAM &&
      !(family == 0 && (variant == VARIANT_DECODE_FUSED || variant == VARIANT_DECODE_FUSED_FAIL)) &&
      !(family == 1 && variant == VARIANT_STREAM_SPLIT) &&
      !narrow_variant(variant) && !mid_variant(variant) && variant >= fsw::tiled_variant_count())
    return FSW_E_VARIANT;
  g_forced_variant[family] = variant < 0 ? -1 : variant;
  return FSW_OK;
}

static fsw::StreamPlan mlp_stream_plan(int64_t M, int64_t D, int64_t FF);
static const char* running_name(int family, int64_t M, int64_t N_or_D, int64_t K_or_FF);
static bool blocked_regime(int64_t M, int64_t D, int64_t FF, size_t scratch);

const char* fsw_variant_name(int family, int dtype, int64_t M, int64_t N_or_D, int64_t K_or_FF) {
  (void)dtype;
  if (family >= 3 && family <= 5) return running_name(family, M, N_or_D, K_or_FF);
  if (family == 2) {  // the down projection inside fsw_mlp
    if (mlp_stream_plan(M, N_or_D, K_or_FF).splits > 1) return "stream_split";
    if (blocked_regime(M, N_or_D, K_or_FF, SIZE_MAX)) return fsw::tiled_variant(V_256x256).name;
    family = 1;
  }
  if (family < 0 || family > 1) return "invalid";
  const int v = resolve_variant(family, M, N_or_D, K_or_FF);
  if (v == VARIANT_SKINNY) return decode_stream_wanted(family, M, N_or_D, K_or_FF) ? "decode_stream" : "skinny";
  if (family == 1 && g_forced_variant[1] < 0 && M <= MAX_DIM && N_or_D > 0 && N_or_D <= MAX_DIM && K_or_FF > 0 &&
      K_or_FF <= MAX_DIM) {
    const fsw::SplitPlan plan = fsw::tiled_split_plan((int)N_or_D, (int)M, (int)K_or_FF);
    if (plan.splits > 1) {
      if (plan.tile == 128) return M <= 64 ? "splitk_dma_128x64" : "splitk_dma_128x128";  // see launch_tiled_splitk
      if (plan.tile == 129) return "splitk_dma_128x256";
      if (plan.tile == 130) return "splitk_dma_128x192";
      if (plan.tile == 160) return "splitk_pair16_256x160";
      if (plan.tile == 192) return "splitk_pair16_256x192";
      if (plan.tile == 224) return "splitk_pair16_256x224";
      return "splitk_pair16_256x256";
    }
  }
  if (narrow_variant(v)) {
    static const char* const names[3] = {"pair16_256x160", "pair16_256x192", "pair16_256x224"};
    return names[v - VARIANT_NARROW - 5];
  }
  if (mid_variant(v)) return fsw::mid_name(forced_mid_plan(v));
  return fsw::tiled_variant(v).name;
}

int fsw_validate_gateup(int dtype, int64_t M, int64_t N, int64_t K, const void* X, int64_t ldx, const void* W13,
                        int64_t ldw, const void* H, int64_t ldh) {
  if (dtype != FSW_BF16 && dtype != FSW_FP16) return FSW_E_DTYPE;
  if (M < 0 || N < 0 || K < 0 || (N & 1)) return FSW_E_SHAPE;
  if (M > MAX_DIM || N > MAX_DIM || K > MAX_DIM) return FSW_E_SHAPE;
  if (M == 0 || N == 0) return FSW_OK;  // nothing to read or write
  if (!H || (K > 0 && (!X || !W13))) return FSW_E_NULL;  // K == 0: X and W13 are never read
  if (ldx < K || ldw < K || ldh < N / 2) return FSW_E_LD;
  if (ldx > MAX_LD || ldw > MAX_LD || ldh > MAX_DIM) return FSW_E_SHAPE;
  if ((((uintptr_t)H) & 1)) return FSW_E_ALIGN;
  if (K == 0) return FSW_OK;
  if ((K & 7) || (ldx & 7) || (ldw & 7)) return FSW_E_ALIGN;
  if (!aligned16(X) || !aligned16(W13)) return FSW_E_ALIGN;
  return FSW_OK;
}

int fsw_validate_down(int dtype, int64_t M, int64_t D, int64_t FF, const void* H, int64_t ldh, const void* W2,
                      int64_t ldw2, const void* Y, int64_t ldy) {
  if (dtype != FSW_BF16 && dtype != FSW_FP16) return FSW_E_DTYPE;
  if (M < 0 || D < 0 || FF < 0) return FSW_E_SHAPE;
  if (M > MAX_DIM || D > MAX_DIM || FF > MAX_DIM) return FSW_E_SHAPE;
  if (M == 0 || D == 0) return FSW_OK;
  if (!Y || (FF > 0 && (!H || !W2))) return FSW_E_NULL;  // FF == 0: H and W2 are never read
  if (ldh < FF || ldw2 < FF || ldy < D) return FSW_E_LD;
  if (ldh > MAX_LD || ldw2 > MAX_LD || ldy > MAX_DIM) return FSW_E_SHAPE;
  if ((((uintptr_t)Y) & 1)) return FSW_E_ALIGN;
  if (FF == 0) return FSW_OK;
  if ((FF & 7) || (ldh & 7) || (ldw2 & 7)) return FSW_E_ALIGN;
  if (!aligned16(H) || !aligned16(W2)) return FSW_E_ALIGN;
  return FSW_OK;
}

static hipError_t launch_gateup_mid(int v, int dtype, const fsw::GemmArgs& a, hipStream_t stream) {
  const fsw::MidPlan p = g_forced_variant[0] >= 0 ? forced_mid_plan(v)
                                                  : fsw::mid_plan(true, a.np, a.nq, a.k, fsw::mid_ragged(a), 1, 1);
  fsw::GemmArgs b = a;
  b.short_sums = few_rows(0, a.nq, a.np, a.k) ? 1 : 0;
  return fsw::launch_mid(dtype, true, p, b, stream);
}

// zero_words / n_zero_words: see GemmArgs (only the decode-regime kernels honour them; the caller checks that)
static int gateup_impl(int dtype, int64_t M, int64_t N, int64_t K, const void* X, int64_t ldx, const void* W13,
                       int64_t ldw, void* H, int64_t ldh, void* stream, unsigned* zero_words, int n_zero_words) {
  const int rc = fsw_validate_gateup(dtype, M, N, K, X, ldx, W13, ldw, H, ldh);
  if (rc != FSW_OK) return rc;
  if (M == 0 || N == 0) return FSW_OK;
  const int drc = check_device();
  if (drc != FSW_OK) return drc;
  fsw::GemmArgs a;
  a.P = W13;
  a.Q = X;
  a.O = H;
  a.ldp = ldw;
  a.ldq = ldx;
  a.ldo = ldh;
  a.np = (int)N;
  a.nq = (int)M;
  a.k = (int)K;
  a.zero_words = zero_words;
  a.n_zero_words = n_zero_words;
  const int v = resolve_variant(0, M, N, K);
  if (mid_wanted(0, v, M, N, K, fsw::mid_ragged(a))) return finish(launch_gateup_mid(v, dtype, a, (hipStream_t)stream));
  if (v == VARIANT_SKINNY) {
    if (decode_stream_wanted(0, M, N, K)) {  // at most 16 rows: one 8-wave workgroup per CU, X held in registers
      fsw::DecodeArgs da = {};
      da.X = X;
      da.W13 = W13;
      da.H = H;
      da.ldx = ldx;
      da.ldw13 = ldw;
      da.ldh = ldh;
      da.nq = (int)M;
      da.d = (int)K;
      da.ff = (int)(N / 2);
      if (fsw::decode_mlp_supported(da, 1)) return finish(fsw::launch_decode_mlp(dtype, da, (hipStream_t)stream, 1));
    }
    return finish(fsw::launch_skinny(dtype, true, a, nullptr, (hipStream_t)stream));
  }
  return finish(launch_large(v, dtype, true, a, (hipStream_t)stream));
}

int fsw_gateup(int dtype, int64_t M, int64_t N, int64_t K, const void* X, int64_t ldx, const void* W13, int64_t ldw,
               void* H, int64_t ldh, void* stream) {
  return gateup_impl(dtype, M, N, K, X, ldx, W13, ldw, H, ldh, stream, nullptr, 0);
}

// The reference's other build (C_TYPE float, constants.cuh:9-14; "C can work with either bf16 or fp32",
// swiglu.cu:470-471): H is float and receives the gated fp32 value without a rounding. From 2^21 gated weight pairs on
// (a layer of 1024 x 2816 has 2.9 million) it runs the kernel that the 16-bit output runs, but for the decode range (few_rows), which
// skinny_kernel keeps whole (the persistent streaming kernel has no float store). Against the weight-streaming kernel (up to 64 rows) and
// the 256 x 256 kernel (above), us: 4096 x 11008: 40 rows 38.4 -> 30.0, 130 rows 66.0 -> 42.0; 4608 x 9216: 65 rows 33.5; 1024 x 2816: 65 rows
// 21.0 -> 10.1, 300 rows 23.5 -> 9.4.
// Smaller layers keep those two kernels: others add the products in another order, and the results of such layers, of which rounding gives
// the 16-bit output of these kernels bit for bit, would change in their last bits.
int fsw_gateup_f32out(int dtype, int64_t M, int64_t N, int64_t K, const void* X, int64_t ldx, const void* W13,
                      int64_t ldw, float* H, int64_t ldh, void* stream) {
  const int rc = fsw_validate_gateup(dtype, M, N, K, X, ldx, W13, ldw, H, ldh);
  if (rc != FSW_OK) return rc;
  if (M == 0 || N == 0) return FSW_OK;
  if ((((uintptr_t)H) & 3)) return FSW_E_ALIGN;
  const int drc = check_device();
  if (drc != FSW_OK) return drc;
  fsw::GemmArgs a;
  a.P = W13;
  a.Q = X;
  a.O = H;
  a.ldp = ldw;
  a.ldq = ldx;
  a.ldo = ldh;
  a.np = (int)N;
  a.nq = (int)M;
  a.k = (int)K;
  a.out_f32 = 1;
  int v = M <= 64 ? VARIANT_SKINNY : V_256x256;
  if ((N / 2) * K >= (int64_t)1 << 21) {
    v = resolve_variant(0, M, N, K);
    // The decode range stays on skinny_kernel, whose waves sum a quarter or less of K each: 1.6e-7 off float64 at 16384 x 2048. The rows past
    // it have all of K in one chain of sums, as they had on the 128-row tiles that mid_kernel replaced (6.9e-7 at 27648 x 5120, 16 rows).
    if (v != VARIANT_SKINNY && mid_wanted(0, v, M, N, K, fsw::mid_ragged(a)))
      return finish(launch_gateup_mid(v, dtype, a, (hipStream_t)stream));
  }
  if (v == VARIANT_SKINNY) return finish(fsw::launch_skinny(dtype, true, a, nullptr, (hipStream_t)stream));
  return finish(launch_large(v, dtype, true, a, (hipStream_t)stream));
}

// Rows of fsw_mlp (17 .. 32, large layers) that have the name "stream_split", and the plan of the split-K streaming kernel for them.
// That kernel runs only when variant 104 asks for it (then any shape it supports), and where the gate/up product before it runs a
// kernel that zeroes the ticket counters (skinny_kernel or mid_kernel): K parts of mid_kernel and a summing launch are faster
// everywhere (whole forwards, us, stream_split -> mid: 4096 x 11008 24 rows 52.1 -> 48.9; 4096 x 14336 17 rows 60.3 -> 59.2, 32 rows
// 63.5 -> 61.3; 5120 x 13824 24 rows 83.7 -> 72.4; 2048 x 8192 32 rows 28.3 -> 24.6; 4880 x 16416 24 rows 102 -> 83).
static fsw::StreamPlan mlp_stream_plan(int64_t M, int64_t D, int64_t FF) {
  const fsw::StreamPlan none = {0, 0, 0, 0};
  if (M < 1 || M > 32 || D <= 0 || FF <= 0 || D > MAX_DIM || FF > MAX_DIM / 2) return none;
  const int f1 = g_forced_variant[1];
  if (f1 >= 0 && f1 != VARIANT_STREAM_SPLIT) return none;
  const int f0 = g_forced_variant[0];
  if (f0 == VARIANT_DECODE_FUSED || f0 == VARIANT_DECODE_FUSED_FAIL) return none;
  const int v0 = resolve_variant(0, M, 2 * FF, D);
  const bool zeroes = (v0 == VARIANT_SKINNY && !decode_stream_wanted(0, M, 2 * FF, D)) || v0 == V_128x64;
  if (!zeroes) return none;
  if (f1 == VARIANT_STREAM_SPLIT) return fsw::stream_split_plan((int)D, (int)M, (int)FF, true);
  if (!streams_weights(1, M, D, FF) || decode_stream_wanted(1, M, D, FF)) return none;
  return fsw::stream_split_plan((int)D, (int)M, (int)FF, false);
}
static bool stream_split_runs(int64_t M, int64_t D, int64_t FF) {
  return g_forced_variant[1] == VARIANT_STREAM_SPLIT && mlp_stream_plan(M, D, FF).splits > 1;
}
static size_t stream_scratch_bytes(const fsw::StreamPlan& p) {
  return (p.partial_bytes + (size_t)p.ticket_words * 4 + 255) & ~(size_t)255;
}

// How the down projection runs. Parts of K: fp32 partial sums of parts * M * D floats in the workspace.
//   mid:  the producer / consumer kernel (any number of parts)
//   else: parts > 1: launch_tiled_splitk on `plan.tile`; 1: the unsplit kernel of resolve_variant()
// `limit`: most bytes the partial sums may take; a plan that wants more splits K less often (fsw_mlp_static, whose scratch is
// fixed, keeps the shapes that any plan fits).
struct DownPlan {
  bool mid;
  fsw::SplitPlan plan;
};
static DownPlan down_plan(int64_t M, int64_t D, int64_t FF, size_t limit, bool rag) {
  DownPlan r = {false, {128, 1}};
  if (M <= 0 || M > MAX_DIM || D <= 0 || D > MAX_DIM || FF <= 0 || FF > MAX_DIM) return r;
  const int v = resolve_variant(1, M, D, FF);
  const size_t part = (size_t)M * (size_t)D * sizeof(float);
  const int64_t most = (int64_t)(limit / part < 16 ? limit / part : 16);
  if (g_forced_variant[1] >= 0) {  // a forced kernel runs unsplit
    r.mid = dma_variant(v);
    return r;
  }
  if (v == VARIANT_SKINNY || M <= 256) {
    r.mid = mid_wanted(1, v, M, D, FF, rag);
    if (r.mid) r.plan.splits = fsw::mid_plan(false, (int)D, (int)M, (int)FF, rag, 0, most < 1 ? 1 : (int)most).splits;
    if (r.mid || v == VARIANT_SKINNY) return r;
  }
  r.plan = fsw::tiled_split_plan((int)D, (int)M, (int)FF);
  if (r.plan.splits > most) r.plan.splits = most < 1 ? 1 : (int)most;
  r.mid = r.plan.splits > 1 ? r.plan.tile <= 130 : dma_variant(v);
  // The same parts or fewer on whichever kernel takes them faster by the estimates. Outputs of up to 3072 features, whole lines: mid_kernel's
  // is 8 % high where the 256-row kernel's is right. Down, us, 256-row kernel -> mid_kernel: 8192 -> 2048 656 rows 41.8 -> 35.9, 700 rows
  // 39.3 -> 34.3, 768 rows 45.3 -> 39.2; 9792 -> 2776 328 rows 34.1 -> 31.0; 12288 -> 3064 295 rows 39.0 -> 34.2; 25 problems of 1024 .. 2304
  // features 0.91 (worst 1.025), 25 of 2304 .. 3072 0.91 (worst 0.98). Left out are tiles of 224 and 256 activation rows, which the estimate
  // does not tell apart there: 20 problems that would take 96 x 224 0.94 (0.86 .. 1.03). Wider outputs are level within what one call differs
  // from run to run (11008 -> 4096 359 rows 52 and 57, 384 rows 48.5 and 45.0; 14336 -> 4096 333 rows 55.7 and 52.2, the forward 135 either
  // way). The plan is that of dense rows, as the scratch is: K of whole lines in rows that are none gains more, as the 256-row kernel fetches
  // their lines twice (20 problems, rows 8 elements longer: 0.76, 0.67 .. 0.82). Fewer parts are longer chains of sums in fp32: 6144 -> 1536
  // 1024 rows in two parts where six were, 3.3e-4 of the bf16 results are not the nearest to the exact one, 2.4e-4 before (fp16 2.2e-3 and
  // 1.6e-3), and the error of the result is the same to five digits (1.6539e-3, fp16 2.0704e-4).
  // Other rows: 8008 -> 3000 300 rows 39.6 -> 28.8, 900 rows 62.9 -> 58.8; 23568 -> 6168 499 rows stays, 152 and 189.
  if (!r.mid && r.plan.splits > 1 && M <= 1024) {
    const bool narrow = !rag && D <= 3072;
    const fsw::MidPlan p = fsw::mid_plan(false, (int)D, (int)M, (int)FF, rag, 0, r.plan.splits);
    r.mid = (rag || (narrow && fsw::mid_tile_cols(p.tile) <= 192)) &&
            p.us < (narrow ? 1.05 : 0.95) * fsw::pair16_split_time((int)D, (int)M, (int)FF, r.plan);
  }
  return r;
}

// bytes of the partial sums; planned for dense operands (FF columns to a row)
static size_t down_split(int64_t M, int64_t D, int64_t FF, size_t limit, DownPlan* plan) {
  *plan = down_plan(M, D, FF, limit, ragged(FF));
  return plan->plan.splits > 1 ? plan->plan.splits * (size_t)M * (size_t)D * sizeof(float) : 0;
}

// Least scratch that the down projection accepts: more than that only buys K parts on the producer / consumer kernel, which runs with
// as many of them as there is room for. What the 128-row tiles asked for is still asked for: a call that was refused stays refused.
static size_t down_least(int64_t M, int64_t D, int64_t FF, size_t limit) {
  if (M <= 0 || D <= 0 || FF <= 0 || g_forced_variant[1] >= 0 || streams_weights(1, M, D, FF)) return 0;
  const size_t part = (size_t)M * (size_t)D * sizeof(float);
  size_t parts = (size_t)fsw::tiled_split_plan((int)D, (int)M, (int)FF).splits;
  if (parts > limit / part) parts = limit / part;
  return parts > 1 ? parts * part : 0;
}

size_t fsw_down_workspace_bytes(int dtype, int64_t M, int64_t D, int64_t FF) {
  (void)dtype;
  DownPlan plan;
  return down_split(M, D, FF, SIZE_MAX, &plan);
}

static int down_impl(int dtype, int64_t M, int64_t D, int64_t FF, const void* H, int64_t ldh, const void* W2, int64_t ldw2,
                     void* Y, int64_t ldy, void* workspace, size_t workspace_bytes, size_t limit, void* stream) {
  const int rc = fsw_validate_down(dtype, M, D, FF, H, ldh, W2, ldw2, Y, ldy);
  if (rc != FSW_OK) return rc;
  if (M == 0 || D == 0) return FSW_OK;
  DownPlan plan;
  size_t need = down_split(M, D, FF, limit, &plan);
  const int v = resolve_variant(1, M, D, FF);
  const size_t room = workspace && aligned16(workspace) ? workspace_bytes : 0;
  if (need > room) {
    const size_t least = down_least(M, D, FF, limit);
    if (least > 0 && (!workspace || workspace_bytes < least)) return FSW_E_WORKSPACE;
    if (least > 0 && !aligned16(workspace)) return FSW_E_ALIGN;
    need = down_split(M, D, FF, room < limit ? room : limit, &plan);
    if (need == 0 && v == VARIANT_SKINNY) plan.mid = false;  // few rows: the weight-streaming kernel needs no scratch
  }
  const int drc = check_device();
  if (drc != FSW_OK) return drc;
  fsw::GemmArgs a;
  a.P = W2;
  a.Q = H;
  a.O = Y;
  a.ldp = ldw2;
  a.ldq = ldh;
  a.ldo = ldy;
  a.np = (int)D;
  a.nq = (int)M;
  a.k = (int)FF;
  if (plan.mid) {
    a.splits = need > 0 ? plan.plan.splits : 1;
    a.partial = (float*)workspace;
    // Above 256 rows the plan's parts are the most there is scratch for: fewer, or none, where smaller tiles fill the chip without
    // them. us: 2088 -> 736 1996 rows 17.8 -> 14.1; 2816 -> 1024 512 rows 14.8 -> 13.4, 900 rows 17.6 -> 15.3; 8192 -> 2048 371 rows
    // 27.0 -> 25.7; 12680 -> 3304 (ragged) 368 rows 60.3 -> 48.3; 50 problems 0.940 on average, worst 1.012.
    const fsw::MidPlan p = g_forced_variant[1] >= 0
                               ? forced_mid_plan(v)
                               : fsw::mid_plan(false, (int)D, (int)M, (int)FF, fsw::mid_ragged(a), M > 256 ? 0 : a.splits, a.splits);
    a.splits = p.splits;
    a.short_sums = few_rows(1, M, D, FF) ? 1 : 0;
    return finish(fsw::launch_mid(dtype, false, p, a, (hipStream_t)stream));
  }
  if (v == VARIANT_SKINNY) {
    if (decode_stream_wanted(1, M, D, FF)) {
      fsw::DecodeArgs da = {};
      da.W2 = W2;
      da.H = const_cast<void*>(H);
      da.Y = Y;
      da.ldw2 = ldw2;
      da.ldy = ldy;
      da.ldh = ldh;
      da.nq = (int)M;
      da.d = (int)D;
      da.ff = (int)FF;
      if (fsw::decode_mlp_supported(da, 2)) return finish(fsw::launch_decode_mlp(dtype, da, (hipStream_t)stream, 2));
    }
    return finish(fsw::launch_skinny(dtype, false, a, workspace, (hipStream_t)stream));
  }
  if (need > 0) {  // few output tiles, deep K: split K across workgroups
    a.splits = plan.plan.splits;
    a.partial = (float*)workspace;
    return finish(fsw::launch_tiled_splitk(dtype, plan.plan.tile, a, (hipStream_t)stream));
  }
  return finish(launch_large(v, dtype, false, a, (hipStream_t)stream));
}

int fsw_down(int dtype, int64_t M, int64_t D, int64_t FF, const void* H, int64_t ldh, const void* W2, int64_t ldw2,
             void* Y, int64_t ldy, void* workspace, size_t workspace_bytes, void* stream) {
  return down_impl(dtype, M, D, FF, H, ldh, W2, ldw2, Y, ldy, workspace, workspace_bytes, SIZE_MAX, stream);
}

static size_t h_bytes(int64_t M, int64_t ldh) {
  const size_t raw = (size_t)M * (size_t)ldh * 2;
  return (raw + 255) & ~(size_t)255;
}

// Row stride of row-major H between the two kernels of fsw_mlp: whole 128-byte lines above 256 rows, where the caller's scratch has
// room for them beside the `need` bytes of dense H and the partial sums. The 256-row kernel fetches a row that starts inside a line by
// K tiles that lie in two lines. Forward, us, dense -> whole lines: 4096 x 14344 5000 rows 1480 -> 1394, 1200 rows 400 -> 383; 3488 x
// 11656 2500 rows 554 -> 532; 3000 x 8008 600 rows 120.1 -> 117.3. Up to 256 rows, where mid_kernel copies whole lines anyway, level.
static int64_t h_stride(int64_t M, int64_t FF, size_t need, size_t workspace_bytes) {
  const int64_t lines = (FF + 63) / 64 * 64;
  return M > 256 && need - h_bytes(M, FF) + h_bytes(M, lines) <= workspace_bytes ? lines : FF;
}

// what row-major H leaves of `scratch` bytes (SIZE_MAX: no limit) for the down projection's partial sums
static size_t beside_h(int64_t M, int64_t FF, size_t scratch) {
  const size_t h = h_bytes(M, FF);
  return scratch == SIZE_MAX ? SIZE_MAX : scratch > h ? (scratch - h) & ~(size_t)255 : 0;
}

// Large-tile regime of fsw_mlp: both projections run 256 x 256 tiles, and H never exists row-major: the gate/up
// epilogue writes it panel-blocked (whole 1 KB runs) and the down projection reads it blocked. Against row-major H
// the whole forward measures 0.8 % (8192 x 4096 x 14336) to 1.3 % (4096 x 4096 x 11008) faster; X is read row-major.
static bool blocked_regime(int64_t M, int64_t D, int64_t FF, size_t scratch) {
  if (M <= 64 || D <= 0 || FF <= 0 || g_forced_variant[0] >= 0 || g_forced_variant[1] >= 0) return false;
  if (M > MAX_DIM || D > MAX_DIM || FF > MAX_DIM / 2) return false;
  // a down projection on narrower tiles reads row-major H; it has to gain more than H blocked does (3000 rows of 4096 x
  // 11008: 7 % of the down kernel, a third of the forward, is not enough; 2500 rows: 11 %)
  DownPlan plan;  // a split-K down projection reads row-major H
  return pick_tiled(0, M, 2 * FF, D) == V_256x256 && pick_tiled(1, M, D, FF, 0.9) == V_256x256 &&
         (size_t)fsw::blocked_bytes(M, FF) <= scratch && down_split(M, D, FF, beside_h(M, FF, scratch), &plan) == 0;
}

// fsw_variant_name families 3 .. 5: the kernel that runs, for dense operands on whole lines where the rows are
static const char* running_name(int family, int64_t M, int64_t N_or_D, int64_t K_or_FF) {
  if (M <= 0 || M > MAX_DIM || N_or_D <= 0 || N_or_D > MAX_DIM || K_or_FF <= 0 || K_or_FF > MAX_DIM) return "none";
  if (family == 5) {
    if (stream_split_runs(M, N_or_D, K_or_FF)) return "stream_split";
    if (blocked_regime(M, N_or_D, K_or_FF, SIZE_MAX)) return fsw::tiled_variant(V_256x256).name;
  }
  const bool gated = family == 3, rag = ragged(K_or_FF);
  const int f = gated ? 0 : 1, v = resolve_variant(f, M, N_or_D, K_or_FF);
  const DownPlan d = gated ? DownPlan{false, {0, 1}} : down_plan(M, N_or_D, K_or_FF, SIZE_MAX, rag);
  if (gated ? mid_wanted(0, v, M, N_or_D, K_or_FF, rag) : d.mid)
    return fsw::mid_name(g_forced_variant[f] >= 0 ? forced_mid_plan(v)
                                                  : fsw::mid_plan(gated, (int)N_or_D, (int)M, (int)K_or_FF, rag,
                                                                !gated && M > 256 ? 0 : d.plan.splits, d.plan.splits));
  return fsw_variant_name(f, FSW_BF16, M, N_or_D, K_or_FF);
}

size_t fsw_blocked_bytes(int64_t rows, int64_t k) {
  if (rows <= 0 || k <= 0 || rows > MAX_DIM || k > MAX_DIM) return 0;
  return (size_t)fsw::blocked_bytes(rows, k);
}

// src: row-major [rows, k], 16-byte aligned, ld and k multiples of 8; dst: fsw_blocked_bytes(rows, k) bytes
static int block_rows_impl(int dtype, int64_t rows, int64_t k, const void* src, int64_t ld, void* dst, bool gated_order,
                           void* stream) {
  if (dtype != FSW_BF16 && dtype != FSW_FP16) return FSW_E_DTYPE;
  if (rows < 0 || k < 0 || rows > MAX_DIM || k > MAX_DIM || (gated_order && (rows & 1))) return FSW_E_SHAPE;
  if (rows == 0 || k == 0) return FSW_OK;
  if (!src || !dst) return FSW_E_NULL;
  if (ld < k) return FSW_E_LD;
  if (ld > MAX_LD) return FSW_E_SHAPE;
  if ((k & 7) || (ld & 7) || !aligned16(src) || !aligned16(dst)) return FSW_E_ALIGN;
  const int drc = check_device();
  if (drc != FSW_OK) return drc;
  return finish(fsw::launch_block_rows(src, ld, (int)rows, (int)k, dst, gated_order, (hipStream_t)stream));
}

int fsw_block_rows(int dtype, int64_t rows, int64_t k, const void* src, int64_t ld, void* dst, void* stream) {
  return block_rows_impl(dtype, rows, k, src, ld, dst, false, stream);
}

int fsw_prepack_w13(int dtype, int64_t N, int64_t K, const void* W13, int64_t ldw, void* dst, void* stream) {
  return block_rows_impl(dtype, N, K, W13, ldw, dst, true, stream);
}

int fsw_prepack_w2(int dtype, int64_t D, int64_t FF, const void* W2, int64_t ldw2, void* dst, void* stream) {
  return block_rows_impl(dtype, D, FF, W2, ldw2, dst, false, stream);
}

int fsw_gateup_blocked(int dtype, int64_t M, int64_t N, int64_t K, const void* Xb, const void* W13, int64_t ldw,
                       int w_blocked, void* Hb, int64_t ldh, void* stream) {

  if (dtype != FSW_BF16 && dtype != FSW_FP16) return FSW_E_DTYPE;
  if (M < 0 || N < 0 || K < 0 || (N & 1) || M > MAX_DIM || N > MAX_DIM || K > MAX_DIM) return FSW_E_SHAPE;
  if (M == 0 || N == 0) return FSW_OK;
  if (K == 0) return FSW_E_SHAPE;  // a blocked matrix with no columns has no representation
  if (!Xb || !W13 || !Hb) return FSW_E_NULL;
  if (!w_blocked && ldw < K) return FSW_E_LD;
  if (!w_blocked && ldw > MAX_LD) return FSW_E_SHAPE;
  if (ldh != 0 && ldh < N / 2) return FSW_E_LD;
  if (ldh > MAX_DIM) return FSW_E_SHAPE;
  if ((K & 7) || (!w_blocked && (ldw & 7))) return FSW_E_ALIGN;
  if (!aligned16(Xb) || !aligned16(W13) || (ldh == 0 ? !aligned16(Hb) : ((((uintptr_t)Hb) & 1) != 0))) return FSW_E_ALIGN;
  const int drc = check_device();
  if (drc != FSW_OK) return drc;
  fsw::GemmArgs a;
  a.P = W13;
  a.Q = Xb;
  a.O = Hb;
  a.ldp = ldw;
  a.ldq = 0;
  a.ldo = ldh;
  a.np = (int)N;
  a.nq = (int)M;
  a.k = (int)K;
  a.layout = 1 | (ldh == 0 ? 2 : 0) | (w_blocked ? 4 : 0);
  return finish(fsw::launch_pair16(dtype, true, a, (hipStream_t)stream));
}

int fsw_gateup_hblocked(int dtype, int64_t M, int64_t N, int64_t K, const void* X, int64_t ldx, const void* W13,
                        int64_t ldw, int w_blocked, void* Hb, void* stream) {
  // blocked weights have no leading dimension: validated as if their rows were K long
  const int rc = fsw_validate_gateup(dtype, M, N, K, X, ldx, W13, w_blocked ? K : ldw, Hb, N / 2);
  if (rc != FSW_OK) return rc;
  if (M == 0 || N == 0) return FSW_OK;
  if (K == 0) return FSW_E_SHAPE;  // a blocked matrix with no columns has no representation
  if (!aligned16(Hb)) return FSW_E_ALIGN;
  const int drc = check_device();
  if (drc != FSW_OK) return drc;
  fsw::GemmArgs a;
  a.P = W13;
  a.Q = X;
  a.O = Hb;
  a.ldp = ldw;
  a.ldq = ldx;
  a.ldo = 0;
  a.np = (int)N;
  a.nq = (int)M;
  a.k = (int)K;
  a.layout = w_blocked ? 6 : 2;
  return finish(fsw::launch_pair16(dtype, true, a, (hipStream_t)stream));
}

int fsw_down_blocked(int dtype, int64_t M, int64_t D, int64_t FF, const void* Hb, const void* W2, int64_t ldw2,
                     int w_blocked, void* Y, int64_t ldy, void* stream) {
  if (dtype != FSW_BF16 && dtype != FSW_FP16) return FSW_E_DTYPE;
  if (M < 0 || D < 0 || FF < 0 || M > MAX_DIM || D > MAX_DIM || FF > MAX_DIM) return FSW_E_SHAPE;
  if (M == 0 || D == 0) return FSW_OK;
  if (FF == 0) return FSW_E_SHAPE;
  if (!Hb || !W2 || !Y) return FSW_E_NULL;
  if ((!w_blocked && ldw2 < FF) || ldy < D) return FSW_E_LD;
  if ((!w_blocked && ldw2 > MAX_LD) || ldy > MAX_DIM) return FSW_E_SHAPE;
  if ((FF & 7) || (!w_blocked && (ldw2 & 7)) || (((uintptr_t)Y) & 1)) return FSW_E_ALIGN;
  if (!aligned16(Hb) || !aligned16(W2)) return FSW_E_ALIGN;
  const int drc = check_device();
  if (drc != FSW_OK) return drc;
  fsw::GemmArgs a;
  a.P = W2;
  a.Q = Hb;
  a.O = Y;
  a.ldp = ldw2;
  a.ldq = 0;
  a.ldo = ldy;
  a.np = (int)D;
  a.nq = (int)M;
  a.k = (int)FF;
  a.layout = w_blocked ? 5 : 1;
  return finish(fsw::launch_pair16(dtype, false, a, (hipStream_t)stream));
}

// fsw_gateup never needs scratch: the large-tile kernel reads row-major X in whole cache lines (K pairs), which
// measures level with a blocked copy of X (8192 x 4096 x 28672: 1.2515 vs 1.2530 ms) and saves the copy. The two
// entry points stay for callers written against them.
size_t fsw_gateup_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t K) {
  (void)dtype;
  (void)M;
  (void)N;
  (void)K;
  return 0;
}

int fsw_gateup_ws(int dtype, int64_t M, int64_t N, int64_t K, const void* X, int64_t ldx, const void* W13, int64_t ldw,
                  void* H, int64_t ldh, void* workspace, size_t workspace_bytes, void* stream) {
  (void)workspace;
  (void)workspace_bytes;
  return fsw_gateup(dtype, M, N, K, X, ldx, W13, ldw, H, ldh, stream);
}

// `scratch`: the bytes there are, which the plan keeps to if H alone fits (SIZE_MAX: no limit)
static size_t mlp_workspace(int64_t M, int64_t D, int64_t FF, size_t scratch) {
  if (M <= 0 || D <= 0 || FF <= 0) return 0;
  if (blocked_regime(M, D, FF, scratch)) return (size_t)fsw::blocked_bytes(M, FF);  // H, panel-blocked
  if (stream_split_runs(M, D, FF))
    return h_bytes(M, FF) + stream_scratch_bytes(mlp_stream_plan(M, D, FF));  // [H row-major][partials][ticket counters]
  // otherwise [H row-major][split-K scratch of the down projection]
  DownPlan plan;
  return h_bytes(M, FF) + ((down_split(M, D, FF, beside_h(M, FF, scratch), &plan) + 255) & ~(size_t)255);
}

// The least scratch the forward accepts, `need` bytes being what its plan asks for: see down_least().
static size_t mlp_least(int64_t M, int64_t D, int64_t FF, size_t scratch, size_t need) {
  if (blocked_regime(M, D, FF, scratch) || stream_split_runs(M, D, FF)) return need;
  const fsw::StreamPlan sp = mlp_stream_plan(M, D, FF);
  const size_t least = h_bytes(M, FF) + (sp.splits > 1 ? stream_scratch_bytes(sp)
                                                       : (down_least(M, D, FF, beside_h(M, FF, scratch)) + 255) & ~(size_t)255);
  return least < need ? least : need;
}

size_t fsw_mlp_workspace_bytes(int dtype, int64_t M, int64_t D, int64_t FF) {
  (void)dtype;
  return mlp_workspace(M, D, FF, SIZE_MAX);
}

// single_launch_ok: whether the opt-in single-launch decode forward may be used (it creates events on first use,
// which the entry point that must not allocate cannot afford); scratch: see mlp_workspace
static int mlp_impl(int dtype, int64_t M, int64_t D, int64_t FF, const void* X, int64_t ldx, const void* W13,
                    int64_t ldw13, const void* W2, int64_t ldw2, void* Y, int64_t ldy, void* workspace,
                    size_t workspace_bytes, void* stream, bool single_launch_ok, size_t scratch) {
  if (dtype != FSW_BF16 && dtype != FSW_FP16) return FSW_E_DTYPE;
  if (M < 0 || D < 0 || FF < 0 || M > MAX_DIM || D > MAX_DIM || FF > MAX_DIM / 2) return FSW_E_SHAPE;
  if (M == 0 || D == 0) return FSW_OK;  // Y is empty: nothing to read or write
  size_t need = mlp_workspace(M, D, FF, scratch);
  if (workspace_bytes < need) need = mlp_least(M, D, FF, scratch, need);
  if (need > 0 && (!workspace || workspace_bytes < need)) return FSW_E_WORKSPACE;
  if (need > 0 && !aligned16(workspace)) return FSW_E_ALIGN;
  // FF == 0 needs no H: any non-NULL pointer satisfies the validators and is never dereferenced
  void* Hbuf = need > 0 ? workspace : (void*)Y;
  // validate both halves before launching either, so a bad down-projection argument leaves nothing enqueued
  int rc = fsw_validate_gateup(dtype, M, 2 * FF, D, X, ldx, W13, ldw13, Hbuf, FF);
  if (rc != FSW_OK) return rc;
  rc = fsw_validate_down(dtype, M, D, FF, Hbuf, FF, W2, ldw2, Y, ldy);
  if (rc != FSW_OK) return rc;
  if (single_launch_ok && M <= 16 && FF > 0 &&
      (g_forced_variant[0] == VARIANT_DECODE_FUSED || g_forced_variant[0] == VARIANT_DECODE_FUSED_FAIL)) {
    // opt-in: one persistent launch does both projections with a device-wide barrier in between. Measured
    // slower than the two weight-streaming launches so far (stragglers before the barrier), so not the default.
    // Without a free barrier slot, or on a stream that is being captured, it is the two launches below.
    fsw::DecodeArgs da;
    da.X = X;
    da.W13 = W13;
    da.W2 = W2;
    da.H = Hbuf;
    da.Y = Y;
    da.ldx = ldx;
    da.ldw13 = ldw13;
    da.ldw2 = ldw2;
    da.ldy = ldy;
    da.ldh = FF;
    da.nq = (int)M;
    da.d = (int)D;
    da.ff = (int)FF;
    if (fsw::decode_mlp_supported(da, 3)) {
      const int drc = check_device();
      if (drc != FSW_OK) return drc;
      bool launched = false;
      const int lrc = finish(fsw::launch_decode_mlp(dtype, da, (hipStream_t)stream, 3, &launched,
                                                    g_forced_variant[0] == VARIANT_DECODE_FUSED_FAIL));
      if (lrc != FSW_OK || launched) return lrc;
    }
  }
  if (blocked_regime(M, D, FF, scratch)) {  // workspace = H, panel-blocked
    rc = fsw_gateup_hblocked(dtype, M, 2 * FF, D, X, ldx, W13, ldw13, 0, workspace, stream);
    if (rc != FSW_OK) return rc;
    return fsw_down_blocked(dtype, M, D, FF, workspace, W2, ldw2, 0, Y, ldy, stream);
  }
  const int64_t ldh = FF > 0 ? h_stride(M, FF, need, workspace_bytes) : 0;
  unsigned char* ws2 = (unsigned char*)workspace + h_bytes(M, ldh);
  if (stream_split_runs(M, D, FF)) {
    const fsw::StreamPlan sp = mlp_stream_plan(M, D, FF);
    // the gate/up kernel zeroes the ticket counters of the split-K streaming down projection
    unsigned* tickets = (unsigned*)(ws2 + sp.partial_bytes);
    rc = gateup_impl(dtype, M, 2 * FF, D, X, ldx, W13, ldw13, Hbuf, ldh, stream, tickets, sp.ticket_words);
    if (rc != FSW_OK) return rc;
    fsw::GemmArgs a;
    a.P = W2;
    a.Q = Hbuf;
    a.O = Y;
    a.ldp = ldw2;
    a.ldq = ldh;
    a.ldo = ldy;
    a.np = (int)D;
    a.nq = (int)M;
    a.k = (int)FF;
    return finish(fsw::launch_stream_split(dtype, a, sp, ws2, (hipStream_t)stream));
  }
  const size_t hb = h_bytes(M, ldh), down_ws = workspace_bytes > hb ? workspace_bytes - hb : 0;
  rc = fsw_gateup(dtype, M, 2 * FF, D, X, ldx, W13, ldw13, Hbuf, ldh, stream);
  if (rc != FSW_OK) return rc;
  return down_impl(dtype, M, D, FF, Hbuf, ldh, W2, ldw2, Y, ldy, ws2, down_ws, beside_h(M, FF, scratch), stream);
}

int fsw_mlp(int dtype, int64_t M, int64_t D, int64_t FF, const void* X, int64_t ldx, const void* W13, int64_t ldw13,
            const void* W2, int64_t ldw2, void* Y, int64_t ldy, void* workspace, size_t workspace_bytes,
            void* stream) {
  return mlp_impl(dtype, M, D, FF, X, ldx, W13, ldw13, W2, ldw2, Y, ldy, workspace, workspace_bytes, stream, true,
                  SIZE_MAX);
}

// ---- the entry point that allocates nothing ------------------------------------------------------------------
// fsw_mlp with its workspace inside the library: a file-scope device array that every GPU the library runs on
// holds until the process ends. The array's name is a host-side stand-in, not a device address; its address on a
// device comes from hipGetSymbolAddress, asked once per device with that device current, and only that pointer is
// handed to kernels.
#define FSW_STATIC_SCRATCH_BYTES (64u << 20)
static __device__ __align__(256) unsigned char scratch[FSW_STATIC_SCRATCH_BYTES];

// device address of `scratch` on the current device (looked up on the first call per device, then cached)
static int static_scratch_ptr(void** out) {
  static std::atomic<void*> ptr_of_device[64];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= 64) {
    g_last_hip_error = (int)e;
    return FSW_E_DEVICE;
  }
  void* p = ptr_of_device[dev].load(std::memory_order_acquire);
  if (!p) {
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      g_last_hip_error = (int)e;
      return FSW_E_LAUNCH;
    }
    ptr_of_device[dev].store(p, std::memory_order_release);  // racing first calls on one device store the same address
  }
  *out = p;
  return FSW_OK;
}

size_t fsw_mlp_static_max_bytes(void) { return FSW_STATIC_SCRATCH_BYTES; }

int fsw_mlp_static(int dtype, int64_t M, int64_t D, int64_t FF, const void* X, int64_t ldx, const void* W13,
                   int64_t ldw13, const void* W2, int64_t ldw2, void* Y, int64_t ldy, void* stream) {
  if (dtype != FSW_BF16 && dtype != FSW_FP16) return FSW_E_DTYPE;
  if (M < 0 || D < 0 || FF < 0 || M > MAX_DIM || D > MAX_DIM || FF > MAX_DIM / 2) return FSW_E_SHAPE;
  if (M == 0 || D == 0) return FSW_OK;
  if (mlp_workspace(M, D, FF, FSW_STATIC_SCRATCH_BYTES) > FSW_STATIC_SCRATCH_BYTES) return FSW_E_STATIC_LIMIT;
  const int drc = check_device();
  if (drc != FSW_OK) return drc;
  void* ws = nullptr;
  const int rc = static_scratch_ptr(&ws);
  if (rc != FSW_OK) return rc;
  return mlp_impl(dtype, M, D, FF, X, ldx, W13, ldw13, W2, ldw2, Y, ldy, ws, FSW_STATIC_SCRATCH_BYTES, stream, false,
                  FSW_STATIC_SCRATCH_BYTES);
}

}  // extern "C"
