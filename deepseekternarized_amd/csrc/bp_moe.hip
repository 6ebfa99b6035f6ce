// One routed-expert MoE layer as one call: sort of the routing, row gather, gate|up grouped GEMM, SwiGLU, down grouped
// GEMM, weighted combine - the per-expert loop of boilerplate/engine/standard.py:156-176 after the router's top-k, with
// the same rounding points (every linear rounded to bf16, products with the routing weight rounded to bf16, the sum
// over a token's experts accumulated in bf16 in ascending expert order).
//
// Nothing is read back to the host. The reference sizes its grouped launch from `int(offsets.diff().max())`
// (boilerplate/kernels/ternary_cuda.py:97), a device-to-host copy in the middle of the layer; here a kernel writes
// the list of token tiles that exist (made by the sort; 32 or 64 rows each), and the grouped GEMMs run over it. Up to 64 tokens
// no expert can have more than 64 rows, and the launch is sized by that bound instead (the small-batch kernels).
//
// All intermediate tensors live in a workspace the caller provides (bp_moe_layer_workspace_bytes): the library
// allocates nothing, so the call can be captured in a HIP graph.
#include <string.h>

#include "bp_mfma.h"

namespace bp {
int kernel_policy();  // bp_api.hip
int sort_with_inverse(int64_t* order, int64_t* offsets, int64_t* inv, const int64_t* ids, int64_t n, int64_t E, int32_t* workspace,
                      int32_t* bad, hipStream_t stream, const SortTiles& t);  // bp_route.hip
int64_t sort_with_inverse_ints(int64_t n, int64_t E);  // its workspace
int moe_combine(void* out, const void* y, bool y16, const int64_t* inv, const void* w, const int64_t* experts, int64_t T, int64_t k, int64_t H,
                void* stream);  // bp_route.hip
int moe_combine_v4(void* out, int out_dtype, const void* y, bool y16, const int64_t* inv, const int64_t* experts, int64_t T, int64_t k, int64_t H,
                   void* stream);
// bp_general.hip
int quant_gathered(int8_t* q, float* s, const void* x, const int64_t* index, int64_t div, int64_t src_rows, int64_t M, int64_t K, hipStream_t st);
int swiglu_quant(bool v4, int8_t* q, float* s, const float* gate, const float* up, const float* weights, const int64_t* order, int64_t pairs, float limit,
                 int64_t rows, int64_t I, int64_t ld, hipStream_t st);
namespace {

constexpr int TILE_ROWS = 32;  // token tile of k_gemm_tq1 / k_gemm_tq2

// (expert, first row) of every token tile of `tile_rows` rows, in expert order; count[0] = their number: a second list beside the sort's, for
// layers whose two products run over tiles of different sizes. One workgroup; experts in chunks of 1024 with a running total.
__global__ __launch_bounds__(1024) void k_tile_list(int32_t* __restrict__ tiles, int32_t* __restrict__ count, const int64_t* __restrict__ offsets,
                                                    int64_t E, int64_t T, int64_t cap, int tile_rows) {
  __shared__ int part[16];
  __shared__ int carry;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int64_t base = 0; base < E; base += 1024) {
    const int64_t e = base + threadIdx.x;
    int64_t o0 = 0, rows = 0;
    if (e < E) {
      o0 = clamp_i64(offsets[e], 0, T);
      const int64_t o1 = clamp_i64(offsets[e + 1], 0, T);
      rows = o1 > o0 ? o1 - o0 : 0;
    }
    const int mine = (int)((rows + tile_rows - 1) / tile_rows);
    int incl = mine;  // inclusive prefix sum within the wave
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(incl, d, 64);
      if (lane >= d) incl += up;
    }
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    int before = carry;
    for (int w = 0; w < wave; ++w) before += part[w];
    int64_t at = before + incl - mine;
    for (int j = 0; j < mine; ++j, ++at) {
      if (at < cap) {
        tiles[2 * at] = (int32_t)e;
        tiles[2 * at + 1] = (int32_t)(o0 + (int64_t)j * tile_rows);
      }
    }
    __syncthreads();
    if (threadIdx.x == 1023) carry = before + incl;
    __syncthreads();
  }
  if (threadIdx.x == 0) count[0] = carry < cap ? carry : (int)cap;
}

// The row gather xg[r] = x[order[r] / k] (rows of 16-byte pieces).
__global__ __launch_bounds__(256) void k_gather16(u32x4* __restrict__ xg, const u32x4* __restrict__ x, const int64_t* __restrict__ order, int64_t n,
                                                  int64_t k, int64_t T, int64_t row16) {
  const int64_t gtid = (int64_t)blockIdx.x * 256 + threadIdx.x, gsz = (int64_t)gridDim.x * 256;
  for (int64_t w = gtid; w < n * row16; w += gsz) {
    const int64_t r = w / row16, c = w - r * row16;
    const int64_t src = clamp_i64(order[r] / k, 0, T - 1);
    xg[r * row16 + c] = x[src * row16 + c];
  }
}

// A few routed rows (n <= ROUTE_SMALL_N): the layer's whole preparation in one launch instead of five - stable sort of
// the expert ids (every workgroup ranks the ids for itself in LDS: element i goes to slot #(ids below id_i) + #(equal
// ids before i); workgroup 0 writes order, offsets and the inverse permutation), the row gather xg[r] = x[order[r] / k]
// and, where the GEMMs run over the list of token tiles, that list (position r of the order starts a tile when it is a
// multiple of tile_rows, 32 or 64, into its expert; the tiles come out in expert order).
constexpr int ROUTE_SMALL_N = 256, ROUTE_SMALL_THREADS = 256;
__global__ __launch_bounds__(ROUTE_SMALL_THREADS) void k_route_small(int64_t* __restrict__ order, int64_t* __restrict__ offsets, int64_t* __restrict__ inv,
                                                                     const int64_t* __restrict__ ids, int n, int64_t E, int32_t* __restrict__ bad,
                                                                     u32x4* __restrict__ xg, const u32x4* __restrict__ x, int k, int64_t T, int64_t row16,
                                                                     int32_t* __restrict__ tiles, int32_t* __restrict__ tile_count, int64_t tile_cap, int tile_rows) {
  __shared__ __attribute__((aligned(16))) int32_t sid[ROUTE_SMALL_N];  // (entries from n on: 0x7fffffff, "no expert")
  __shared__ int32_t ord[ROUTE_SMALL_N];
  __shared__ __attribute__((aligned(16))) int32_t tstart[ROUTE_SMALL_N];  // position r of the order starts a token tile
  const int i = threadIdx.x;
  int32_t mine = 0x7fffffff;  // an id outside [0, E) is left out of the order, as in bp_sort_by_expert
  if (i < n) {
    const int64_t id = ids[i];
    if (id >= 0 && id < E) mine = (int32_t)id;
    else if (bad && blockIdx.x == 0) *bad = 1;
  }
  sid[i] = mine;
  ord[i] = -1;
  tstart[i] = 0;
  __syncthreads();
  int rank = 0;
  if (i < n && mine != 0x7fffffff) {
    int lower = 0;  // rows of the experts before this one
    for (int j = 0; j < n; j += 4) {  // (four ids per LDS read; the padding compares as "after every expert")
      const int4 v = *(const int4*)&sid[j];
      lower += (v.x < mine ? 1 : 0) + (v.y < mine ? 1 : 0) + (v.z < mine ? 1 : 0) + (v.w < mine ? 1 : 0);
      rank += (v.x == mine && j < i ? 1 : 0) + (v.y == mine && j + 1 < i ? 1 : 0) + (v.z == mine && j + 2 < i ? 1 : 0) + (v.w == mine && j + 3 < i ? 1 : 0);
    }
    rank += lower;
    ord[rank] = i;
    if (((rank - lower) & (tile_rows - 1)) == 0) tstart[rank] = 1;
    if (blockIdx.x == 0) {
      order[rank] = i;
      inv[i] = rank;
    }
  }
  if (blockIdx.x == 0) {
    for (int64_t e = i; e <= E; e += ROUTE_SMALL_THREADS) {
      int cnt = 0;
      for (int j = 0; j < n; j += 4) {
        const int4 v = *(const int4*)&sid[j];
        cnt += (v.x < e ? 1 : 0) + (v.y < e ? 1 : 0) + (v.z < e ? 1 : 0) + (v.w < e ? 1 : 0);
      }
      offsets[e] = cnt;
    }
  }
  __syncthreads();
  if (tiles && blockIdx.x == 0) {
    if (i < n && mine != 0x7fffffff && tstart[rank]) {
      int at = 0;  // tiles that start before this one
      for (int q = 0; q < rank; q += 4) {
        const int4 v = *(const int4*)&tstart[q];
        at += v.x + (q + 1 < rank ? v.y : 0) + (q + 2 < rank ? v.z : 0) + (q + 3 < rank ? v.w : 0);
      }
      if (at < tile_cap) {
        tiles[2 * at] = mine;
        tiles[2 * at + 1] = rank;
      }
    }
    if (i == ROUTE_SMALL_THREADS - 1) {
      int total = 0;
      for (int q = 0; q < n; q += 4) {  // (entries from n on are 0)
        const int4 v = *(const int4*)&tstart[q];
        total += v.x + v.y + v.z + v.w;
      }
      tile_count[0] = total < tile_cap ? total : (int)tile_cap;
    }
  }
  const int64_t gtid = (int64_t)blockIdx.x * ROUTE_SMALL_THREADS + i, gsz = (int64_t)gridDim.x * ROUTE_SMALL_THREADS;
  for (int64_t w = gtid; w < (int64_t)n * row16; w += gsz) {  // 16 bytes of a gathered row
    const int64_t r = w / row16, c = w - r * row16;
    const int o = ord[r];
    if (o >= 0) {
      int64_t src = o / k;
      src = src < T ? src : T - 1;
      xg[r * row16 + c] = x[src * row16 + c];
    }
  }
}

// A product of N output rows of a TQ2 layer with bf16 activations: on fp8 pieces where it would be as a grouped call (f4_pays_bf16; launches
// sized by the tokens with few rows per expert stay on the 16-token tiles). The two products of a layer are held to it one by one: the
// one below stays on bf16 matrix instructions, which sum more exactly.
bool f4_product(int64_t T, int64_t n, int64_t N, int64_t E) { return f4_pays_bf16(n, N) && (T > 64 || n > 8 * E || tuning().tq2g == 'f'); }

// Layers whose GEMMs run on the kernel for token tiles of 64 (32 for TQ1).
// TQ2, int8: from 16 rows per expert on average. Whole layer on it / on the 32-token tiles, us: 2048 / 1024 (hidden / intermediate), 64
// experts, 16 rows each 73 / 82, 50 rows 112 / 146; 4096 / 2048, 64 experts, 12 rows 164 / 163, 37 rows 203 / 305; 384 experts, 6 rows
// 733 / 739, 19 rows 750 / 920, 62 rows 1350 / 2194. Few experts leave its larger workgroups short of the device: with at most 1024 output
// columns of gate and up it takes over where the 32-token kernel needs more than one workgroup per CU (by the average rows: half a tile
// per expert is padding), with more from 128 rows on; up to 64 tokens, where the other kernels' launches are sized by the tokens, where all experts
// together have 384 blocks of 128 columns. On it / off it: 2048 / 1024, 8 experts, 300 rows 64 / 54, 800 rows 65 / 59, 1200 rows 70 / 84; 16 experts,
// 600 rows 66 / 56, 900 rows 67 / 79; 4096 / 2048, 4 experts, 66 rows 73 / 61, 160 rows 86 / 102; 2048 / 1280, 2 experts, 66 rows 65 / 52, 200 rows
// 66 / 63; 64 tokens: 7168 / 2048, 4 experts 112 / 76, 8 experts (256 rows) 112 / 86, 16 experts (512) 117 / 133; 2048 / 1024, 32 experts (512) 63 / 59;
// 2816 / 1536, 32 experts (512) 81 / 88; 2048 / 1024, 64 experts (1024) 81 / 91. bf16: layers of which a product does (f4_product).
// TQ1, int8: from 129 routed rows, where all experts together have 512 workgroups (two to a CU) or there are more than 64 tokens (the old
// kernels' grids are bounded by the tokens up to there). Whole layer, us: 4096 / 2048, 64 experts of 6, 16 tokens 194 / 181, 32 205 / 316, 64
// 204 / 221, 251 241 / 372, 1500 765 / 1274; 384 experts, 400 tokens 1038 / 1188, 2000 1357 / 2033; 2048 / 1024, 64 experts of 8, 16 tokens
// 86 / 86, 64 86 / 89, 200 112 / 182. With fewer workgroups: 7168 / 2048, 16 experts of 8, 17 tokens 188 / 163, 100 179 / 252; 2816 / 1536, 32
// experts of 4, 34 tokens 99 / 91, 192 130 / 203.
// TQ1, bf16: from 16 rows per expert, with stacked terms from 44. 4096 / 2048, 64 experts, 6 rows 207 / 199, 12 rows 212 / 209, 23 rows
// 248 / 295, 37 rows 359 / 402; 384 experts, 6 rows 1080 / 1023, 19 rows 1098 / 1129; 2048 / 1024, 8 rows 84 / 85, 25 rows 111 / 149; in two
// terms, 64 experts, 37 rows 658 / 622, 47 rows 711 / 730.
bool moe_f4(int act, int fmt, int64_t T, int64_t n, int64_t H, int64_t I, int64_t E, int n_terms, bool rewritten) {
  if (tuning().tq2g == 'b') return false;
  if (fmt == BP_TQ1 && tuning().f4q >= 0) return n >= tuning().f4q;
  if (fmt == BP_TQ1) return act == BP_I8 ? n > 128 && (T > 64 || E * I >= 512 * 128) : n >= (n_terms == 1 ? 16 : 44) * E;
  if (act == BP_I8) {
    if (tuning().f4 >= 0) return n >= tuning().f4 * E;
    if (rewritten || n < 16 * E) return rewritten;
    if (T <= 64) return E * I >= 384 * 128;
    return (I > 1024 && n >= 128) || (n + 16 * E) * ((2 * I + 255) / 256) > 280 * 32;
  }
  return rewritten || f4_product(T, n, 2 * I, E) || f4_product(T, n, H, E);  // (a TQ1 layer that isn't rewritten runs on fp8 pieces as well)
}

// TQ1 layers whose weights are rewritten as TQ2 ones first (k_tq1_to_tq2, 0.45 bytes of traffic per weight), in memory that the caller
// brings beyond bp_moe_layer_workspace_bytes: tiles of 64 tokens and no byte table in the products of such a layer then. int8 from 48 rows
// per expert on average, with stacked terms from 56, bf16 from 64 and 84. Whole layer with / without, us, int8: 4096 / 2048 (hidden /
// intermediate), 64 experts, 37 rows each 352 / 341, 56 rows 391 / 430, 94 rows 463 / 560, 375 rows 1133 / 1820; 384 experts, 37 rows
// 1734 / 1690, 56 rows 1904 / 2000; 2048 / 1024, 37 rows 126 / 129, 75 rows 165 / 173. bf16: 64 experts, 47 rows 380 / 362, 66 rows
// 481 / 480, 94 rows 525 / 580; 384 experts, 56 rows 2197 / 2120, 78 rows 2713 / 2840; 2048 / 1024, 56 rows 162 / 156, 100 rows 186 / 212;
// in two terms, 64 experts, 75 rows 896 / 890, 94 rows 921 / 1020.
bool moe_repacks(int act, int fmt, int64_t n, int64_t H, int64_t I, int64_t E, int64_t group, int n_terms) {
  if (fmt != BP_TQ1 || kernel_policy() == 1 || H % 256 != 0 || I % 256 != 0 || H < 1024 || I < 1024 || H > 65536 || I > 65536) return false;
  if (group != 128 && !(group == 256 && H % 512 == 0 && I % 512 == 0 && H >= 2048 && I >= 2048)) return false;
  return tuning().tq2g != 'b' && n >= (tuning().f4 >= 0 ? tuning().f4 : act == BP_I8 ? (n_terms == 1 ? 48 : 56) : n_terms == 1 ? 64 : 84) * E;
}
size_t rewritten_bytes(int64_t rows, int64_t K) { return ((size_t)rows * (size_t)(K / 4) + 255) & ~(size_t)255; }
size_t repack_bytes(int64_t H, int64_t I, int64_t E, int n_terms) { return (size_t)n_terms * (rewritten_bytes(E * 2 * I, H) + rewritten_bytes(E * H, I)); }
constexpr size_t REPACK_LIMIT = (size_t)8 << 30;

struct Carve {
  unsigned char* base;
  size_t used;
  void* take(size_t bytes) {
    void* p = base ? base + used : nullptr;
    used += (bytes + 255) & ~(size_t)255;
    return p;
  }
};

struct Plan {
  int64_t* order;
  int64_t* offsets;
  int64_t* inv;
  int32_t* sort_ws;
  int32_t* tiles;
  int32_t* tile_count;
  int32_t* tiles64;  // ... of 64 rows and their number, where `tiles` holds those of 32 for the other product
  void* xg;       // gathered rows, bf16 [T k, H]
  int8_t* q;      // int8 activations of the wider of the two GEMM inputs
  float* q_scale;
  float* gu;      // f32 [T k, 2 I]
  void* h;        // bf16 [T k, I]
  float* y;       // f32 [T k, H]
  unsigned char* stage;  // converted activations of the GEMM in flight (bf16 activations)
  size_t stage_bytes;
  int64_t tile_cap;
  size_t bytes;
};

Plan plan(void* workspace, int64_t T, int64_t H, int64_t I, int64_t E, int64_t k, int act, int fmt, int n_terms, bool rewritten = false) {
  Carve c = {(unsigned char*)workspace, 0};
  Plan p;
  const int64_t n = T * k;
  p.order = (int64_t*)c.take(8 * (size_t)n);
  p.offsets = (int64_t*)c.take(8 * (size_t)(E + 1));
  p.inv = (int64_t*)c.take(8 * (size_t)n);
  p.sort_ws = (int32_t*)c.take(4 * (size_t)sort_with_inverse_ints(n, E));
  p.tile_cap = (n + TILE_ROWS - 1) / TILE_ROWS + E;
  p.tiles = (int32_t*)c.take(8 * (size_t)p.tile_cap);
  p.tile_count = (int32_t*)c.take(4);
  p.tiles64 = (int32_t*)c.take(act == BP_BF16 ? 8 * (size_t)((n + F4_TOK - 1) / F4_TOK + E) + 4 : 0);
  p.xg = c.take(2 * (size_t)n * H);
  p.q = (int8_t*)c.take(act == BP_I8 ? (size_t)n * (H > I ? H : I) : 0);
  p.q_scale = (float*)c.take(act == BP_I8 ? 4 * (size_t)n : 0);
  p.gu = (float*)c.take(4 * (size_t)n * 2 * I);
  p.h = c.take(2 * (size_t)n * I);
  p.y = (float*)c.take(4 * (size_t)n * H);
  p.stage_bytes = 0;
  if (act == BP_BF16) {
    const size_t a = gemm_tq2f_workspace_bytes(n, H, E), b = gemm_tq2f_workspace_bytes(n, I, E);
    p.stage_bytes = a > b ? a : b;
  }
  if (moe_f4(act, fmt, T, n, H, I, E, n_terms, rewritten)) {
    const size_t a = gemm_f4_workspace_bytes(act, n, H, E, fmt), b = gemm_f4_workspace_bytes(act, n, I, E, fmt), more = a > b ? a : b;
    p.stage_bytes = more > p.stage_bytes ? more : p.stage_bytes;
  }
  p.stage = (unsigned char*)c.take(p.stage_bytes);
  p.bytes = c.used;
  return p;
}

}  // namespace
}  // namespace bp

using namespace bp;

extern "C" size_t bp_moe_layer_workspace_bytes(int64_t T, int64_t H, int64_t I, int64_t E, int64_t k, int act, int fmt) {
  if (T < 0 || H <= 0 || I <= 0 || E <= 0 || k <= 0) return 0;
  return plan(nullptr, T, H, I, E, k, act, fmt, 1).bytes;  // (of any count of terms: one has the lowest lines)
}

extern "C" size_t bp_moe_layer_workspace_bytes_terms(int64_t T, int64_t H, int64_t I, int64_t E, int64_t k, int64_t group, int n_terms, int act, int fmt) {
  if (T <= 0 || H <= 0 || I <= 0 || E <= 0 || k <= 0 || n_terms < 1 || n_terms > BP_MAX_TERMS) return 0;
  const size_t base = plan(nullptr, T, H, I, E, k, act, fmt, 1).bytes;
  if (!moe_repacks(act, fmt, T * k, H, I, E, group, n_terms) || repack_bytes(H, I, E, n_terms) > REPACK_LIMIT) return base;
  const size_t more = plan(nullptr, T, H, I, E, k, act, BP_TQ2, n_terms, true).bytes + repack_bytes(H, I, E, n_terms);
  return more > base ? more : base;
}

// `v4`: the rounding points of the V4 engine (boilerplate/engine/model.py:376-387, 407-422) instead of the standard
// decoder's: float32 routing weights applied to the float32 SwiGLU product before the down projection, `limit` clamps,
// float32 accumulation over a token's experts, output float32 or cast once to bf16 (out_dtype).
static int moe_layer(bool v4, void* out, int out_dtype, float limit, const void* x, const int64_t* experts, const void* weights,
                     const uint8_t* const* gate_up_packed, const void* const* gate_up_scale,
                     const uint8_t* const* down_packed, const void* const* down_scale, int scale_dtype,
                     int n_terms, int64_t T, int64_t H, int64_t I, int64_t E, int64_t k, int64_t group, int fmt,
                     int act, void* workspace, size_t workspace_bytes, int32_t* bad, void* stream, bool rewritten = false) {
  if (T < 0 || H <= 0 || I <= 0 || E <= 0 || E > 65535 || k <= 0 || k > 64 || k > E) return fail(BP_ERR_ARG, "invalid MoE layer dimensions (experts up to 65535, top-k up to 64)");
  if (T * k > ((int64_t)1 << 31) - 1 - 32 * E) return fail(BP_ERR_ARG, "too many routed rows for one call");
  if (fmt != BP_TQ1 && fmt != BP_TQ2) return fail(BP_ERR_ARG, "fmt must be 1 (TQ1) or 2 (TQ2)");
  if (act != BP_BF16 && act != BP_I8) return fail(BP_ERR_ARG, "act must be BP_BF16 or BP_I8");
  if (scale_dtype != BP_F32 && scale_dtype != BP_F16 && scale_dtype != BP_BF16) return fail(BP_ERR_ARG, "unexpected scale dtype");
  if (n_terms < 1 || n_terms > BP_MAX_TERMS) return fail(BP_ERR_ARG, "n_terms must be in 1..%d", BP_MAX_TERMS);
  if (group <= 0 || group > ((int64_t)1 << 24)) return fail(BP_ERR_ARG, "invalid group");
  if ((H % 8) != 0 || (I % 8) != 0) return fail(BP_ERR_ARG, "hidden and intermediate sizes must be multiples of 8 (16-byte rows)");
  if (T == 0) return BP_OK;
  if (!out || !x || !experts || !weights || !gate_up_packed || !gate_up_scale || !down_packed || !down_scale) return fail(BP_ERR_ARG, "null pointer");
  for (int t = 0; t < n_terms; ++t)
    if (!gate_up_packed[t] || !gate_up_scale[t] || !down_packed[t] || !down_scale[t]) return fail(BP_ERR_ARG, "null packed or scale pointer in term %d", t);
  const Plan p = plan(workspace, T, H, I, E, k, act, fmt, n_terms, rewritten);
  if (!workspace || workspace_bytes < p.bytes) return fail(BP_ERR_ARG, "the workspace must hold bp_moe_layer_workspace_bytes() = %zu bytes", p.bytes);
  if (((uintptr_t)workspace & 255) != 0) return fail(BP_ERR_ARG, "the workspace must be 256-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  const int64_t n = T * k;
  // bf16 TQ1 layers on fp8 pieces, rewritten or not: those that k_gemm_tq2f has on pieces too. The others keep the kernel that multiplies bf16.
  bool pieces = act != BP_BF16 || fmt != BP_TQ1 || (T > 24 && scale_dtype != BP_F32 && (group != 256 || (((H + 255) / 256) % 2 == 0 && ((I + 255) / 256) % 2 == 0)));
  if (act == BP_BF16 && fmt == BP_TQ1)
    for (int t = 1; t < n_terms; ++t)
      pieces = pieces && ((((uintptr_t)gate_up_packed[t] ^ (uintptr_t)gate_up_packed[0]) | ((uintptr_t)down_packed[t] ^ (uintptr_t)down_packed[0])) & 3) == 0;
  if (pieces && moe_repacks(act, fmt, n, H, I, E, group, n_terms) && (((uintptr_t)x | (uintptr_t)out) & 15) == 0) {
    const size_t own = plan(nullptr, T, H, I, E, k, act, BP_TQ2, n_terms, true).bytes, weights2 = repack_bytes(H, I, E, n_terms);
    bool fits = weights2 <= REPACK_LIMIT && workspace_bytes >= own + weights2;
    for (int t = 0; t < n_terms; ++t) fits = fits && (((uintptr_t)gate_up_scale[t] | (uintptr_t)down_scale[t]) & 15) == 0;
    if (fits) {
      const uint8_t *gu[BP_MAX_TERMS], *dn[BP_MAX_TERMS];
      unsigned char* at = (unsigned char*)workspace + own;
      for (int t = 0; t < n_terms; ++t) {
        gu[t] = at;
        dn[t] = at + rewritten_bytes(E * 2 * I, H);
        if (const int rc = launch_tq1_to_tq2(at, gate_up_packed[t], E * 2 * I, H, s)) return rc;
        if (const int rc = launch_tq1_to_tq2(at + rewritten_bytes(E * 2 * I, H), down_packed[t], E * H, I, s)) return rc;
        at += rewritten_bytes(E * 2 * I, H) + rewritten_bytes(E * H, I);
      }
      return moe_layer(v4, out, out_dtype, limit, x, experts, weights, gu, gate_up_scale, dn, down_scale, scale_dtype, n_terms, T, H, I, E, k, group, BP_TQ2, act,
                       workspace, own, bad, stream, true);
    }
  }
  const int per = fmt == BP_TQ2 ? 4 : 5;

  int rc = BP_OK;
  // Tokens beyond which the GEMMs run over the tile list. Up to 64 no expert can have more than 64 rows and the small-batch
  // kernels take the launch by that bound; TQ1 with bf16 activations changes over at 24 already: the launches of 8 rows
  // cost what their widest expert costs (an expert with 9 rows means a second pass over few CUs), the tile kernel a flat
  // 0.23 ms from 24 to 64 tokens on config 2's layer, where the small-batch kernels take 0.25 - 0.26 (and 0.18 - 0.21 below).
  const int64_t tiles_from = tuning().tiles >= 0 ? tuning().tiles : (fmt == BP_TQ1 && act == BP_BF16 ? 24 : 64);
  const bool tiles = T > tiles_from;
  const bool aligned16 = (((uintptr_t)x | (uintptr_t)p.xg) & 15) == 0;
  // int8 activations: the rows are quantised where they are gathered, and SwiGLU's result where it is made, when the rows'
  // lengths suit those kernels - two launches and two copies of the rows less
  const bool quant_in = act == BP_I8 && aligned16 && H <= 8192;
  // The gate | up projection as the grouped GEMM over converted activations with SwiGLU in its epilogue (bf16 h written,
  // no float32 gate | up rows), where that kernel takes the call: over the tile list, bf16 activations. Its conversion
  // pass then also does the row gather (rows read through `order`): no routed copy of the activations is written.
  GemmArgs fused;
  memset(&fused, 0, sizeof(fused));
  bool fuse = false;
  if (tiles && fmt == BP_TQ1 && act == BP_BF16 && p.stage_bytes && kernel_policy() != 1 && tuning().glu != 'n' && tuning().tq2g != 'b') {
    GemmArgs& a = fused;
    a.out = p.gu; a.x = p.xg; a.offsets = p.offsets; a.x_dtype = act;
    for (int t = 0; t < n_terms; ++t) { a.packed[t] = gate_up_packed[t]; a.w_scale[t] = gate_up_scale[t]; }
    a.scale_dtype = scale_dtype; a.n_terms = n_terms; a.fmt = fmt;
    a.T = n; a.N = 2 * I; a.K = H; a.Kp = (H + per - 1) / per; a.G = (H + group - 1) / group; a.group = group; a.E = E;
    a.stage = p.stage; a.stage_bytes = (int64_t)p.stage_bytes;
    a.tiles = p.tiles; a.tile_count = p.tile_count; a.tile_cap = p.tile_cap;
    a.overwrite = 1; a.max_rows = TILE_ROWS;
    a.glu_h = (uint16_t*)p.h; a.glu_v4 = v4 ? 1 : 0; a.glu_limit = limit;
    a.glu_weights = v4 ? (const float*)weights : nullptr; a.glu_order = p.order; a.glu_pairs = n;
    if (aligned16 && tuning().glu != 'g') {  // (development: BP_TUNE_GLU=g keeps the gather a launch of its own)
      a.x = x; a.x_index = p.order; a.x_div = k; a.x_rows = T;
    }
    fuse = gemm_tiles_supported(a) && gemm_tq2f_applies(a) == BP_OK;
  }
  // Token tiles of 64 (TQ1: 32), either activation type: the conversion passes gather (int8: the token rows are quantised once) and
  // quantise h; gate | up applies SwiGLU and the down projection writes bf16 rows. A down projection that the kernel does not take runs
  // elsewhere, unless it would need the list of 32-row tiles. TQ2 with bf16 activations: each product by its own line, with two lists.
  GemmArgs f4_gu, f4_down;
  const int f4_tok = fmt == BP_TQ1 ? F4_TOK1 : F4_TOK;
  const bool f4_each = act == BP_BF16 && fmt == BP_TQ2 && !rewritten;
  bool f4 = false, f4_first = false, f4_second = false, two_lists = false;  // (of gate | up and down; any of them)
  const bool f4_glu = tuning().glu != 'n', f4_gather = f4_glu && tuning().glu != 'g';
  if (moe_f4(act, fmt, T, n, H, I, E, n_terms, rewritten) && pieces && aligned16 && kernel_policy() != 1 && (f4_gather || act == BP_BF16)) {
    memset(&f4_gu, 0, sizeof(f4_gu));
    GemmArgs& a = f4_gu;
    a.offsets = p.offsets; a.x_dtype = act; a.scale_dtype = scale_dtype; a.n_terms = n_terms; a.fmt = fmt; a.group = group;
    a.T = n; a.E = E; a.max_rows = f4_tok; a.overwrite = 1;
    a.stage = p.stage; a.stage_bytes = (int64_t)p.stage_bytes;
    a.tiles = p.tiles; a.tile_count = p.tile_count; a.tile_cap = (n + f4_tok - 1) / f4_tok + E;
    f4_down = a;
    for (int t = 0; t < n_terms; ++t) { a.packed[t] = gate_up_packed[t]; a.w_scale[t] = gate_up_scale[t]; }
    a.x = p.xg;
    if (f4_gather) { a.x = act == BP_I8 ? (const void*)p.q : x; a.x_scale = p.q_scale; a.x_index = p.order; a.x_div = k; a.x_rows = T; }
    a.N = 2 * I; a.K = H; a.Kp = (H + per - 1) / per; a.G = (H + group - 1) / group;
    a.out = p.gu;
    if (f4_glu) {
      a.glu_h = (uint16_t*)p.h; a.glu_v4 = v4 ? 1 : 0; a.glu_limit = limit;
      a.glu_weights = v4 ? (const float*)weights : nullptr; a.glu_order = p.order; a.glu_pairs = n;
    }
    GemmArgs& d = f4_down;
    for (int t = 0; t < n_terms; ++t) { d.packed[t] = down_packed[t]; d.w_scale[t] = down_scale[t]; }
    d.x = p.h; d.x_dtype = BP_BF16; d.quant = act == BP_I8 ? 1 : 0;
    d.N = H; d.K = I; d.Kp = (I + per - 1) / per; d.G = (I + group - 1) / group;
    d.out = p.y;
    d.out16 = f4_glu ? (uint16_t*)p.y : nullptr;
    GemmArgs probe = d;  // (mfma_supports knows the product's own activation type)
    probe.x_dtype = act;
    f4_first = mfma_supports(a) && gemm_f4_applies(a) == BP_OK && (!f4_each || f4_product(T, n, 2 * I, E));
    f4_second = mfma_supports(probe) && gemm_f4_applies(d) == BP_OK && (!f4_each || f4_product(T, n, H, E));
    if (!f4_each && (!f4_first || (!f4_second && gemm_tiles_supported(probe)))) f4_first = f4_second = false;
    f4 = f4_first || f4_second;
    two_lists = f4_each && tiles && f4_first != f4_second;
    if (two_lists) {
      a.tiles = d.tiles = p.tiles64;
      a.tile_count = d.tile_count = p.tiles64 + 2 * a.tile_cap;
    }
  }
  const bool f4_reads = f4_first && f4_gather;  // gate | up reads its rows through `order`
  const int list_rows = f4 && !two_lists ? f4_tok : TILE_ROWS;
  const int64_t row16 = f4_reads || (fuse && fused.x_index) || (quant_in && !f4) ? 0 : H / 8;  // (no rows to copy where they are read through `order`)
  // A few routed rows in one launch: up to 256 where it gathers, which the sort doesn't, and up to 64 else (every thread reads all ids: 4 us for
  // 6 rows, 12 for 192, where k_sort takes 5.4 for 384; its histograms grow with the experts. 64 experts of 4096 / 2048, TQ1 bf16, 32 tokens x 6: 198.8 -> 193.5 us).
  const bool small = n <= (row16 || E > 512 ? ROUTE_SMALL_N : 64) && (((uintptr_t)x | (uintptr_t)p.xg) & 15) == 0;
  if (small) {
    int64_t g = ((int64_t)n * row16 + ROUTE_SMALL_THREADS - 1) / ROUTE_SMALL_THREADS;
    g = g < 1 ? 1 : (g > 256 ? 256 : g);
    hipLaunchKernelGGL(k_route_small, dim3((unsigned)g), dim3(ROUTE_SMALL_THREADS), 0, s, p.order, p.offsets, p.inv, experts, (int)n, E, bad,
                       (u32x4*)p.xg, (const u32x4*)x, (int)k, T, row16, tiles || f4 ? p.tiles : nullptr, p.tile_count,
                       p.tile_cap, list_rows);
    if ((rc = check_launch("route_small")) != BP_OK) return rc;
  } else {
    const SortTiles list = {tiles || f4 ? p.tiles : nullptr, p.tile_count, p.tile_cap, list_rows};
    if ((rc = sort_with_inverse(p.order, p.offsets, p.inv, experts, n, E, p.sort_ws, bad, s, list)) != BP_OK) return rc;
    if (f4_reads || (fuse && fused.x_index) || (quant_in && !f4)) {
      // (no routed copy of the activations: the gate | up launch's conversion pass reads them through `order`)
    } else if (aligned16) {
      int64_t g = (n * (H / 8) + 255) / 256;
      g = g < 1 ? 1 : (g > 4096 ? 4096 : g);
      hipLaunchKernelGGL(k_gather16, dim3((unsigned)g), dim3(256), 0, s, (u32x4*)p.xg, (const u32x4*)x, p.order, n, k, T, H / 8);
      if ((rc = check_launch("gather")) != BP_OK) return rc;
    } else if ((rc = bp_gather_rows(p.xg, x, p.order, k, n, T, 2 * H, s)) != BP_OK) return rc;
  }

  // `o16`: the caller takes bf16 rows (the combine rounds the down projection's rows to bf16 first); set to whether
  // the launch wrote them, into the same buffer. `quantised`: p.q and p.q_scale hold the int8 rows already. Every launch
  // replaces what its output held.
  auto gemm = [&](float* o, const void* in, const uint8_t* const* packed, const void* const* scale, int64_t N, int64_t K, bool tiles, bool* o16, bool quantised) -> int {
    const bool want16 = o16 && *o16;
    if (o16) *o16 = false;
    GemmArgs a;
    memset(&a, 0, sizeof(a));
    a.out = o;
    a.x = in;
    a.offsets = p.offsets;
    a.x_dtype = act;
    a.overwrite = 1;
    if (act == BP_I8) {
      if (quantised) {
      } else if (const int q = bp_quant_act_int8(p.q, p.q_scale, in, BP_BF16, n, K, s)) return q;
      a.x = p.q;
      a.x_scale = p.q_scale;
    }
    for (int t = 0; t < n_terms; ++t) { a.packed[t] = packed[t]; a.w_scale[t] = scale[t]; }
    a.scale_dtype = scale_dtype; a.n_terms = n_terms; a.fmt = fmt;
    a.T = n; a.N = N; a.K = K; a.Kp = (K + per - 1) / per; a.G = (K + group - 1) / group; a.group = group; a.E = E;
    a.max_rows = T < n ? T : n;  // an expert has at most one row per token
    if (p.stage_bytes) {
      a.stage = p.stage;
      a.stage_bytes = (int64_t)p.stage_bytes;
    }
    if (tiles) {
      a.tiles = p.tiles; a.tile_count = p.tile_count; a.tile_cap = p.tile_cap;
      if (kernel_policy() != 1 && gemm_tiles_supported(a)) {
        a.max_rows = TILE_ROWS;
        if (want16 && tuning().glu != 'n' && tuning().tq2g != 'b') {
          a.out16 = (uint16_t*)o;
          if (gemm_tq2f_applies(a) == BP_OK) {
            *o16 = true;
            return launch_gemm_tq2f(a, s);
          }
          a.out16 = nullptr;
        }
        return run_gemm(a, s);
      }
      a.tiles = nullptr;  // no tile kernel for this shape: the launch covers the bound (every expert up to T rows)
    }
    if (want16) {
      a.out16 = (uint16_t*)o;
      const int got = run_gemm(a, s);
      if (got != ERR_NO_OUT16) {
        *o16 = true;
        return got;
      }
      a.out16 = nullptr;
    }
    return run_gemm(a, s);
  };
  if (f4) {
    if (act == BP_I8 && (rc = bp_quant_act_int8(p.q, p.q_scale, x, BP_BF16, T, H, s)) != BP_OK) return rc;
    if (two_lists) {
      hipLaunchKernelGGL(k_tile_list, dim3(1), dim3(1024), 0, s, p.tiles64, p.tiles64 + 2 * f4_gu.tile_cap, p.offsets, E, n, f4_gu.tile_cap, F4_TOK);
      if ((rc = check_launch("tile_list")) != BP_OK) return rc;
    }
    rc = f4_first ? launch_gemm_f4(f4_gu, s, rewritten) : gemm(p.gu, p.xg, gate_up_packed, gate_up_scale, 2 * I, H, tiles, nullptr, false);
    if (rc != BP_OK) return rc;
    const bool glu_done = f4_first && f4_glu;
    if (!glu_done) rc = v4 ? bp_swiglu_v4(p.h, p.gu, p.gu + I, (const float*)weights, p.order, n, limit, n, I, 2 * I, s) : bp_swiglu_bf16(p.h, p.gu, p.gu + I, n, I, 2 * I, s);
    if (rc != BP_OK) return rc;
    bool y16 = f4_glu;
    rc = f4_second ? launch_gemm_f4(f4_down, s, rewritten) : gemm(p.y, p.h, down_packed, down_scale, H, I, two_lists, &y16, false);
    if (rc != BP_OK) return rc;
    if (glu_done) note_kernel_suffix(f4_gather ? "+glu+gather" : "+glu");
    if (y16) note_kernel_suffix("+y16");
    if (v4) return moe_combine_v4(out, out_dtype, p.y, y16, p.inv, experts, T, k, H, s);
    return moe_combine(out, p.y, y16, p.inv, weights, experts, T, k, H, s);
  }
  bool quant_h = false;
  if (fuse) {
    rc = launch_gemm_tq2f(fused, s);
  } else {
    if (quant_in && (rc = quant_gathered(p.q, p.q_scale, x, p.order, k, T, n, H, s)) != BP_OK) return rc;
    if ((rc = gemm(p.gu, p.xg, gate_up_packed, gate_up_scale, 2 * I, H, tiles, nullptr, quant_in)) != BP_OK) return rc;
    rc = BP_ERR_UNSUPPORTED;
    if (act == BP_I8) rc = swiglu_quant(v4, p.q, p.q_scale, p.gu, p.gu + I, v4 ? (const float*)weights : nullptr, p.order, n, limit, n, I, 2 * I, s);
    quant_h = rc == BP_OK;
    if (quant_h) {
    } else if (v4) rc = bp_swiglu_v4(p.h, p.gu, p.gu + I, (const float*)weights, p.order, n, limit, n, I, 2 * I, s);
    else rc = bp_swiglu_bf16(p.h, p.gu, p.gu + I, n, I, 2 * I, s);
  }
  if (rc != BP_OK) return rc;
  bool y16 = true;
  if ((rc = gemm(p.y, p.h, down_packed, down_scale, H, I, tiles, &y16, quant_h)) != BP_OK) return rc;
  if (fuse) note_kernel_suffix(fused.x_index ? "+glu+gather" : "+glu");  // (bp_last_kernel: the down projection's kernel, and that the gate | up one applied SwiGLU)
  if (y16) note_kernel_suffix("+y16");  // (... and that the down projection wrote bf16 rows)
  if (v4) return moe_combine_v4(out, out_dtype, p.y, y16, p.inv, experts, T, k, H, s);
  return moe_combine(out, p.y, y16, p.inv, weights, experts, T, k, H, s);
}

extern "C" int bp_moe_layer_bf16(void* out, const void* x, const int64_t* experts, const void* weights,
                                 const uint8_t* const* gate_up_packed, const void* const* gate_up_scale,
                                 const uint8_t* const* down_packed, const void* const* down_scale, int scale_dtype,
                                 int n_terms, int64_t T, int64_t H, int64_t I, int64_t E, int64_t k, int64_t group, int fmt,
                                 int act, void* workspace, size_t workspace_bytes, int32_t* bad, void* stream) {
  return moe_layer(false, out, BP_BF16, 0.f, x, experts, weights, gate_up_packed, gate_up_scale, down_packed, down_scale, scale_dtype,
                   n_terms, T, H, I, E, k, group, fmt, act, workspace, workspace_bytes, bad, stream);
}

extern "C" int bp_moe_layer_v4(void* out, int out_dtype, const void* x, const int64_t* experts, const float* weights, float swiglu_limit,
                               const uint8_t* const* gate_up_packed, const void* const* gate_up_scale,
                               const uint8_t* const* down_packed, const void* const* down_scale, int scale_dtype,
                               int n_terms, int64_t T, int64_t H, int64_t I, int64_t E, int64_t k, int64_t group, int fmt,
                               int act, void* workspace, size_t workspace_bytes, int32_t* bad, void* stream) {
  if (out_dtype != BP_F32 && out_dtype != BP_BF16) return fail(BP_ERR_ARG, "the layer's output is float32 or bf16");
  if (!(swiglu_limit == swiglu_limit) || swiglu_limit < 0.f) return fail(BP_ERR_ARG, "swiglu_limit must be 0 (no clamp) or positive");
  return moe_layer(true, out, out_dtype, swiglu_limit, x, experts, weights, gate_up_packed, gate_up_scale, down_packed, down_scale, scale_dtype,
                   n_terms, T, H, I, E, k, group, fmt, act, workspace, workspace_bytes, bad, stream);
}
