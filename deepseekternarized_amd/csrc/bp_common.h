// Shared declarations for the gfx950 ternary kernels: error reporting, dtype helpers, launch
// argument blocks. Host and device code of libbp_ternary_hip.so include this.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <type_traits>

#include "../../include/bp_ternary.h"
#include "bp_xcd.h"

namespace bp {

// ---- host-side error plumbing (thread local, surfaced through bp_last_error) ----
int fail(int code, const char* fmt, ...);
void note_kernel(const char* name);
void note_kernel_suffix(const char* suffix);  // ... appended to the name noted last
int check_launch(const char* what);

// ---- argument block of one grouped GEMM call (validated by the C entry point) ----
struct GemmArgs {
  float* out;
  const void* x;
  const float* x_scale;
  const int64_t* offsets;
  const uint8_t* packed[BP_MAX_TERMS];
  const void* w_scale[BP_MAX_TERMS];
  int x_dtype, scale_dtype, n_terms, fmt;
  int64_t T, N, K, Kp, G, group, E, max_rows;
  // Tile-list mode of the token-tile kernels, with tiles of 32 or 64 rows (set by callers that keep the routing on the device, where
  // the widest expert's row count is unknown to the host): tiles = (expert, first row) pairs of the token tiles that exist, in
  // expert order, tile_count[0] of them (device memory, written by a kernel earlier on the stream); the launch covers
  // tile_cap entries and workgroups past the count leave at once. NULL: token tiles are counted by blockIdx.z up to max_rows.
  const int32_t* tiles;
  const int32_t* tile_count;
  int64_t tile_cap;
  int row_grid;   // decode launches: one blockIdx.y per token row instead of one per expert (expert_of_block; set by launch_mfma)
  int overwrite;  // the results replace `out` instead of being added to it
  // Workspace of the caller for kernels that convert the activations in a pass of their own (NULL: those kernels are not used).
  unsigned char* stage;
  int64_t stage_bytes;
  // Row gather in the conversion pass of the grouped GEMMs over converted activations (x_index != NULL): row r of the launch is
  // row x_index[r] / x_div of x, which has x_rows rows (the routed copy of the activations is never materialised).
  const int64_t* x_index;
  int64_t x_div, x_rows;
  int quant;  // x is bf16 and the conversion pass of the kernel for 64-token tiles quantises its rows (x_scale unused)
  // bf16 out16[T, N] is written instead of float32 `out` (one launch that covers all of K and all terms; a kernel that
  // takes several passes over an output returns ERR_NO_OUT16 instead).
  uint16_t* out16;
  // SwiGLU in the epilogue of the same GEMMs (glu_h != NULL; tile-list mode with overwrite): the N output rows are N / 2 gate
  // rows followed by N / 2 up rows, and the kernel writes bf16 glu_h[T, N / 2] instead of `out`, with the rounding points of
  // bp_swiglu_bf16 (glu_v4 = 0) or of bp_swiglu_v4 (glu_v4 = 1: clamp by glu_limit when positive, float32 product times
  // glu_weights[glu_order[row]] when glu_weights is set, one rounding to bf16).
  uint16_t* glu_h;
  int glu_v4;
  float glu_limit;
  const float* glu_weights;
  const int64_t* glu_order;
  int64_t glu_pairs;
};

__device__ __forceinline__ int64_t clamp_i64(int64_t v, int64_t lo, int64_t hi) { return v < lo ? lo : (v > hi ? hi : v); }

// The expert of a decode launch's blockIdx.y. With many fewer token rows than experts (one token of a routed layer: 6 of 64)
// the grid holds one y per row, and y = j is the j-th expert that has rows - every wave looks for it in the offsets - rather than
// one y per expert, most of whose workgroups would only take a CU's LDS, read two offsets and leave.
// The search is another trip to memory ahead of everything else, so only from eight experts per row on: one token of the
// 64-expert layer 49.2 -> 40.2 us, but 25 rows of 50 experts 25.1 -> 26.8.
inline bool rows_in_grid(int64_t T, int64_t E) { return 8 * T <= E; }  // (GemmArgs::row_grid)
inline unsigned grid_experts(const GemmArgs& a) { return (unsigned)(a.row_grid ? a.T : a.E); }
constexpr unsigned NO_EXPERT = 0xffffffffu;
__device__ __forceinline__ unsigned expert_of_block(const GemmArgs& a, unsigned j) {
  if (__builtin_expect(!a.row_grid, 1)) return j;
  const int lane = threadIdx.x & 63;
  for (int64_t base = 0; base < a.E; base += 256) {
    unsigned long long has[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t x = base + 64 * i + lane;
      bool rows = false;
      if (x < a.E) rows = clamp_i64(a.offsets[x + 1], 0, a.T) > clamp_i64(a.offsets[x], 0, a.T);
      has[i] = __ballot(rows);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned n = (unsigned)__popcll(has[i]);
      if (j < n) {
        for (; j > 0; --j) has[i] &= has[i] - 1;
        return (unsigned)base + 64u * (unsigned)i + (unsigned)(__ffsll((long long)has[i]) - 1);
      }
      j -= n;
    }
  }
  return NO_EXPERT;  // fewer experts with rows
}

// Which token tile of ROWS rows a workgroup takes: `slot` is its expert (list entry in tile-list mode), z its token tile.
struct TileRef {
  int64_t e, tok0, o1;
  bool live;
};
template <int ROWS = 32>
__device__ __forceinline__ TileRef tile_ref(const GemmArgs& a, int64_t slot, unsigned z) {
  TileRef r = {0, 0, 0, false};
  if (a.tiles) {
    if (slot >= a.tile_count[0] || slot >= a.tile_cap) return r;
    r.e = a.tiles[2 * slot];
    r.tok0 = a.tiles[2 * slot + 1];
    r.o1 = clamp_i64(a.offsets[r.e + 1], 0, a.T);
  } else {
    if (slot >= a.E) return r;
    r.e = slot;
    r.o1 = clamp_i64(a.offsets[slot + 1], 0, a.T);
    r.tok0 = clamp_i64(a.offsets[slot], 0, a.T) + (int64_t)z * ROWS;
  }
  r.live = r.tok0 < r.o1;
  return r;
}

// Which token tile and which block of output rows a workgroup of a token-tile kernel takes, from its linear index: bp_xcd.h.
template <int ROWS = 32>
__device__ __forceinline__ TileRef tile_of_workgroup(const GemmArgs& a, const TileSplit& split, unsigned linear, int& row_block) {
  unsigned expert = 0, tile = 0, block = 0;
  if (a.tiles) {
    const unsigned slot = list_item(split, ROWS, linear, block);
    row_block = (int)block;
    return tile_ref<ROWS>(a, slot, 0);
  }
  if (!tile_item(split, linear, expert, tile, block)) return {0, 0, 0, false};
  row_block = (int)block;
  return tile_ref<ROWS>(a, expert, tile);
}
// Workgroups of such a launch and its split (-1: more than a grid's x extent holds).
template <int ROWS = 32>
inline int64_t split_tiles(TileSplit& split, const GemmArgs& a, int64_t row_blocks) {
  split = tile_split(a.E, a.max_rows, ROWS, row_blocks);
  const int64_t wgs = a.tiles ? list_items(ROWS, a.tile_cap, row_blocks) : tile_items(split);
  split.eighth = (unsigned)(wgs / 8);
  return wgs;
}

// Development overrides of the kernel selection (environment variables BP_TUNE_*), read once when the library is first
// used; bp_reload_tuning() reads them again (the tests switch kernels that way). 0 / unset = automatic.
struct Tuning {
  int r;       // BP_TUNE_R: 16-row tiles per wave of the TQ2 kernel (1, 2)
  int waves;   // BP_TUNE_WAVES: waves per workgroup (8, 16)
  char tq1;    // BP_TUNE_TQ1: 'l' table-lookup GEMV, 'm' 16-token MFMA kernel, 'c' the chunk-per-wave GEMV wherever it can run, 'r' never (first letter of the value)
  char tq2g;   // BP_TUNE_TQ2G: 'b' (bf16) never the fp8 x fp4 grouped GEMM over converted activations, 'f' (fp4) wherever it can run
  char tq2v;   // BP_TUNE_TQ2V: 'k' the K-split fp8 x fp4 TQ2 GEMV wherever it can run, 'n' never
  int f4w;     // BP_TUNE_F4W: waves per workgroup of the fp8 x fp4 GEMV (8, 16)
  int f4t;     // BP_TUNE_F4T: routed rows per expert up to which launches of 8 rows are used (-1 = default)
  int cpt;     // BP_TUNE_CPT: chunks per table pass of the table-lookup GEMV
  int tiles;   // BP_TUNE_TILES: tokens from which bp_moe_layer_* runs its GEMMs over the device-side list of token tiles (-1 = default)
  int f4;      // BP_TUNE_F4: token rows (per expert on average) from which TQ2 layers and linears run on the GEMM over tiles of 64 (-1 = default)
  int f4q;     // BP_TUNE_F4Q: routed rows from which TQ1 layers run on that kernel (-1 = default)
  char glu;    // BP_TUNE_GLU: 'n' bp_moe_layer_* never lets the gate | up GEMM apply SwiGLU itself (a launch of its own instead), 'g' it does but the row gather stays a launch of its own
};
const Tuning& tuning();

// Raises a kernel's dynamic LDS limit, once per device and kernel (thread-safe).
template <auto Kernel>
int raise_lds_limit(int bytes) {
  static std::mutex m;
  static bool done[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return fail(BP_ERR_LAUNCH, "cannot identify the current device");
  std::lock_guard<std::mutex> lock(m);
  if (!done[dev]) {
    const hipError_t rc = hipFuncSetAttribute((const void*)Kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (rc != hipSuccess) return fail(BP_ERR_LAUNCH, "cannot raise the dynamic LDS limit of a kernel: %s", hipGetErrorString(rc));
    done[dev] = true;
  }
  return BP_OK;
}

// Internal result of a launcher whose kernel cannot write GemmArgs::out16 for this call: the caller takes float32 sums of
// the whole call and rounds them in a pass of its own.
constexpr int ERR_NO_OUT16 = -100;

// Kernel selection for a validated argument block (the body of bp_ternary_grouped_gemm after its checks).
int run_gemm(const GemmArgs& a, hipStream_t s);
// True when a launch in tile-list mode would run on one of the 32-token-tile kernels (which honour tiles / overwrite).
bool gemm_tiles_supported(const GemmArgs& a);
// Workspace bytes of the TQ1 grouped GEMM over converted activations (GemmArgs::stage) for T rows in all; 0: not available.
size_t gemm_tq2f_workspace_bytes(int64_t T, int64_t K, int64_t E);
// ... of the GEMM on the 32 x 32 x 64 instruction (act: BP_BF16 or BP_I8).
size_t gemm_f4_workspace_bytes(int act, int64_t T, int64_t K, int64_t E, int fmt);
int launch_general(const GemmArgs& a, hipStream_t s);
// bp_route.hip: where a sort by expert also lists the token tiles of `rows` rows: (expert, first row) of each in expert order, count[0]
// their number, at most `cap`. tiles NULL: no list.
struct SortTiles {
  int32_t* tiles;
  int32_t* count;
  int64_t cap;
  int rows;
};
// bp_repack.hip: TQ1 rows as TQ2 rows
int launch_tq1_to_tq2(uint8_t* out, const uint8_t* in, int64_t rows, int64_t K, hipStream_t s);
// Returns BP_ERR_UNSUPPORTED (without setting an error message) when the shape is outside the
// tuned kernels' preconditions.
int launch_mfma(const GemmArgs& a, hipStream_t s);
bool mfma_supports(const GemmArgs& a);

// ---- device helpers ----
__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }

__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {  // round to nearest even, NaN kept quiet
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_bit_cast(uint16_t, (__bf16)f);  // v_cvt_pk_bf16_f32: one instruction, the same bits for every float32 value
#else
  const uint32_t u = __builtin_bit_cast(uint32_t, f);
  return (uint16_t)(f != f ? (u >> 16) | 0x0040u : (u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
#endif
}

__device__ __forceinline__ float f16_bits_to_f32(uint16_t b) {
  _Float16 h = __builtin_bit_cast(_Float16, b);
  return (float)h;
}

__device__ __forceinline__ float load_scale(const void* p, int dtype, int64_t i) {
  if (dtype == BP_F32) return ((const float*)p)[i];
  const uint16_t b = ((const uint16_t*)p)[i];
  return dtype == BP_F16 ? f16_bits_to_f32(b) : bf16_bits_to_f32(b);
}

// SwiGLU of one pair of gate and up sums with the rounding points of bp_swiglu_bf16 or (V4) of bp_swiglu_v4, as bf16 bits.
template <bool V4>
__device__ __forceinline__ uint16_t swiglu_bits(float gate, float up, bool weighted, float weight, float limit) {
  float g = bf16_bits_to_f32(f32_to_bf16_bits(gate)), u = bf16_bits_to_f32(f32_to_bf16_bits(up));
  if (V4) {
    if (limit > 0.f) {  // torch.clamp: a NaN stays a NaN
      u = u < -limit ? -limit : (u > limit ? limit : u);
      g = g > limit ? limit : g;
    }
    const float v = (g / (1.0f + expf(-g))) * u;
    return f32_to_bf16_bits(weighted ? weight * v : v);
  }
  return f32_to_bf16_bits(bf16_bits_to_f32(f32_to_bf16_bits(g / (1.0f + expf(-g)))) * u);
}

// What happens to the outputs. A source is compiled for both cases where its kernels feel the difference (build.py,
// BP_REPLACES): launches that add to float32 `out`, the grouped entry point's contract, and launches of a linear or a layer
// that replace it or write bf16 `out16` instead. Elsewhere GemmArgs::overwrite decides. Tested at run time in every kernel, the
// second case cost the first: spilled scalar registers in the streaming TQ1 kernels (192 against 185 with six loads per loader, two
// tokens 43 against 24), and 2 - 15 % of a grouped launch's time (int8, 64 experts x 32 rows x 2048 x 2048: TQ1 61.0 -> 70.2 us).
namespace {
#ifdef BP_REPLACES
constexpr int OUTPUTS = BP_REPLACES;  // 0: added to, 1: replaced
#else
constexpr int OUTPUTS = -1;  // by GemmArgs::overwrite
#endif
__device__ __forceinline__ bool replaces(const GemmArgs& a) { return OUTPUTS < 0 ? a.overwrite != 0 : OUTPUTS == 1; }
// Where a kernel's epilogue writes: copies of the arguments, not a reference, through which every output would load them again.
struct Output {
  float* out;
  uint16_t* out16;
  bool replace;
};
__device__ __forceinline__ Output output_of(const GemmArgs& a) { return {a.out, OUTPUTS == 0 ? nullptr : a.out16, replaces(a)}; }
// An epilogue f(OUT16): once for bf16 outputs and once for float32 ones, so that the branch is outside its loops (inside, it kept the
// compiler from grouping an epilogue's loads).
template <class F>
__device__ __forceinline__ void with_output(const Output& o, F&& f) {
  if (OUTPUTS != 0 && o.out16) f(std::true_type{});
  else f(std::false_type{});
}
// One finished output.
template <bool OUT16>
__device__ __forceinline__ void store_out(const Output& o, int64_t i, float v) {
  if (OUT16) o.out16[i] = f32_to_bf16_bits(v);
  else o.out[i] = (o.replace ? 0.f : o.out[i]) + v;
}
}  // namespace

__device__ __forceinline__ float load_act_f32(const void* p, int dtype, int64_t i) {
  if (dtype == BP_F32) return ((const float*)p)[i];
  if (dtype == BP_I8) return (float)((const int8_t*)p)[i];
  const uint16_t b = ((const uint16_t*)p)[i];
  return dtype == BP_F16 ? f16_bits_to_f32(b) : bf16_bits_to_f32(b);
}


// TQ1 digit i of byte v as a trit (boilerplate/ternary/pack.py:62-67): bytes >= 243 decode to 0.
__device__ __host__ __forceinline__ int tq1_trit(unsigned v, int i) {
  if (v >= 243u) return 0;
  const unsigned p = i == 0 ? 1u : i == 1 ? 3u : i == 2 ? 9u : i == 3 ? 27u : 81u;
  return (int)((v / p) % 3u) - 1;
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

}  // namespace bp
