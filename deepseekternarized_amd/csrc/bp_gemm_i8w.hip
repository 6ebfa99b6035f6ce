// TQ2 grouped GEMM for int8 activations and token tiles of 128 rows (prompts, experts with many token rows each).
//
// Contract as everywhere (boilerplate/kernels/ternary_cuda.py:52-64): exact int32 group sums, then in float32
// total += sum * scale[n, g] over the groups in ascending order and the stacked terms, then x_scale[t].
//
// What bounds it: the matrix cores and, beside them, the vector ALU. A group's 16 x 16 tile is two
// v_mfma_i32_16x16x64_i8, and turning its int32 sums into scaled float32 ones (a conversion and an FMA per sum) takes the
// vector ALU about as long as the two instructions take the matrix core; decoding the packed weights comes on top and is
// what the tile sizes are about: a wave decodes 64 rows for 64 tokens (k_gemm_tq2: 32 rows for 32 tokens), and the
// 8 waves of a workgroup (4 x 64 rows, 2 x 64 tokens) share the activations of 128 tokens, so that a weight is
// read from the L2 for 64 tokens at a time and an activation for 256 rows. 64 x 64 float32 totals are 64 registers of a
// wave's 256 (two waves per SIMD: one's vector work beside the other's matrix instructions).
//
// The activations are laid out beforehand (k_stage_i8w): the KiB that a wave reads as operand A of one instruction is
// contiguous in lane order, every 16 of its bytes are transposed to the decode's code order, and the group sums that take
// the codes' offset off again are made there, so that the GEMM only copies them to LDS (two windows of 256 k, one barrier
// per window). The pass also gathers routed rows through an index, and quantises bf16 rows on the way (the arithmetic of
// bp_quant_act_int8), which saves the routed copy of the activations and the int8 rows.
// 8192 x 2048 x 6144 from bf16 rows to bf16 rows, both launches: 441 us on the 32-token tiles; 263 with the compiler's own schedule, 207
// with the interleaving pinned, 184 with two small workgroups per CU, 174 with the quantisation in the conversion pass (22 us of it) and
// the epilogue through LDS. 1.36 Pop/s of the rest; by itself under a tracer this kernel takes 175 to 199 us as the clock falls. The
// vector ALU is active in 61 % of the SIMDs' cycles, the matrix cores in 26 %, the waves wait half of their time.
#include <type_traits>

#include "bp_mfma.h"
#include "bp_tq2_decode.h"

namespace bp {
namespace {

typedef __attribute__((address_space(3))) float lds_f32;

constexpr int W_WAVES = 8, W_THREADS = W_WAVES * 64;  // of the conversion
constexpr int W_RT = 4, W_TT = 4;                  // 16-row tiles and 16-token tiles of a wave
constexpr int W_WT = 2;                            // waves along the tokens; along the rows: the kernel's WR, 2 or 4
constexpr int i8w_rows(int WR) { return WR * W_RT * 16; }  // output rows per workgroup: 128 or 256
constexpr int W_TOK = W_WT * W_TT * 16;            // 128 tokens
constexpr int W_OPS = 2 * 2 * (W_TOK / 16) * 1024; // operands of a window: 2 groups x 2 instructions x 8 token tiles x 1 KiB
constexpr int W_SUM = 2 * W_TOK * 4;               // ... and the offset sums: [group][token] int32
constexpr int W_FB = W_OPS + W_SUM;
static_assert(W_OPS % (4 * 16 * 2 * W_WT * 64) == 0 && W_SUM <= 16 * 2 * W_WT * 64, "a staged window: four or eight 16-byte pieces per thread and a tail");
static_assert(W_TOK == I8W_TOK && W_FB % W_TOK == 0, "");
constexpr int W_SC = 2 * W_FB;                     // LDS: two staged windows, then the rows' scales, float32 [term][row][groups + 2]

// The staged windows of token tile (expert e, first row tok0): tiles never overlap whatever the experts' row counts are.
// The rows' activation scales, float32 [T], come first.
__host__ __device__ __forceinline__ int64_t scales_bytes(int64_t T) { return (4 * T + 255) & ~(int64_t)255; }
__device__ __forceinline__ unsigned char* staged_tile(const GemmArgs& a, int64_t e, int64_t tok0) {
  return a.stage + scales_bytes(a.T) + (tok0 + W_TOK * e) * (a.K / 256) * (W_FB / W_TOK);
}

// ---- the conversion: one workgroup per 16 tokens of a token tile. Wave = every eighth group; lane = (token t of 16,
// quarter q of the group): the 16-element units 2 q and 2 q + 1, which instructions 0 and 1 take in lane block kb.
// SRC = BP_I8: rows and their scales are copied. SRC = BP_BF16: a row is quantised, operation for operation as k_quant16.
// KEEP: groups per wave whose bf16 activations stay in registers between the two passes (K up to 1024 KEEP; more are read
// again), no more than K needs: at K = 1024, 4 of them left room for one workgroup per CU (116 us for 65,536 rows).
template <int SRC, int KEEP>
__global__ __launch_bounds__(W_THREADS) void k_stage_i8w(GemmArgs a) {
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const TileRef tr = tile_ref<W_TOK>(a, blockIdx.x, blockIdx.z);
  if (!tr.live) return;  // uniform for the workgroup
  const int ntok = (int)(tr.o1 - tr.tok0 < W_TOK ? tr.o1 - tr.tok0 : W_TOK);
  const int mt = blockIdx.y;
  if (16 * mt >= ntok) return;  // uniform (the GEMM reads what lies there and stores none of it)
  const int t = lane & 15, q = lane >> 4;
  const int kb = ((q & 1) << 1) | (q >> 1);
  const int tok = 16 * mt + t;
  const int64_t row = tr.tok0 + (tok < ntok ? tok : ntok - 1);  // rows past the expert's tokens repeat its last one
  int64_t src = row;
  if (a.x_index) src = clamp_i64(a.x_index[row] / a.x_div, 0, a.x_rows - 1);
  unsigned char* dst = staged_tile(a, tr.e, tr.tok0);
  const int groups = (int)(a.K / 128);
  auto put = [&](int g, const u32x4& u0, const u32x4& u1) {
    unsigned char* w = dst + (int64_t)(g >> 1) * W_FB;
    unsigned char* f = w + ((g & 1) * 2 * (W_TOK / 16) + mt) * 1024 + (kb * 16 + t) * 16;
    *(u32x4*)f = tq2_permute_i8(u0);
    *(u32x4*)(f + (W_TOK / 16) * 1024) = tq2_permute_i8(u1);
    int n = 0;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      n = __builtin_amdgcn_sdot4((int)u0[d], 0x01010101, n, false);
      n = __builtin_amdgcn_sdot4((int)u1[d], 0x01010101, n, false);
    }
    n += __shfl_xor(n, 16, 64);
    n += __shfl_xor(n, 32, 64);
    if (q == 0) *(int*)(w + W_OPS + ((g & 1) * W_TOK + tok) * 4) = -n;
  };
  float* scales = (float*)a.stage;
  if constexpr (SRC == BP_I8) {
    const u32x4* xp = (const u32x4*)((const unsigned char*)a.x + src * a.K) + 2 * q;
    if (wave == 0 && q == 0 && tok < ntok) scales[row] = a.x_scale[src];
    int g = wave;
    for (; g + W_WAVES < groups; g += 2 * W_WAVES) {  // (two groups' loads on their way)
      const u32x4 u0 = xp[8 * g], u1 = xp[8 * g + 1], v0 = xp[8 * (g + W_WAVES)], v1 = xp[8 * (g + W_WAVES) + 1];
      put(g, u0, u1);
      put(g + W_WAVES, v0, v1);
    }
    if (g < groups) put(g, xp[8 * g], xp[8 * g + 1]);
  } else {
    const u32x4* xp = (const u32x4*)((const uint16_t*)a.x + src * a.K) + 4 * q;
    u32x4 kept[KEEP][4];
    float amax = 0.f;
    bool nan = false;
    auto look = [&](const u32x4& v) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const float lo = __uint_as_float(v[d] << 16), hi = __uint_as_float(v[d] & 0xffff0000u);
        nan |= lo != lo || hi != hi;
        amax = fmaxf(amax, fmaxf(fabsf(lo), fabsf(hi)));
      }
    };
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
      const int g = wave + i * W_WAVES;
#pragma unroll
      for (int d = 0; d < 4; ++d) kept[i][d] = g < groups ? xp[16 * g + d] : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
#pragma unroll
      for (int d = 0; d < 4; ++d) look(kept[i][d]);
    for (int g = wave + KEEP * W_WAVES; g < groups; g += W_WAVES)
#pragma unroll
      for (int d = 0; d < 4; ++d) look(xp[16 * g + d]);
    if (nan) amax = __builtin_nanf("");
    auto join = [](float x, float y) { return (x != x || y != y) ? __builtin_nanf("") : fmaxf(x, y); };
    amax = join(amax, __shfl_xor(amax, 16, 64));
    amax = join(amax, __shfl_xor(amax, 32, 64));
    if (q == 0) *(lds_f32*)(unsigned)((wave * 16 + t) * 4) = amax;
    __syncthreads();
    amax = 0.f;
#pragma unroll
    for (int w = 0; w < W_WAVES; ++w) amax = join(amax, *(const lds_f32*)(unsigned)((w * 16 + t) * 4));
    float sc = __fdiv_rn(amax, 127.0f);
    sc = sc != sc ? sc : fmaxf(sc, 1e-8f);
    if (wave == 0 && q == 0 && tok < ntok) scales[row] = sc;
    auto quant8 = [&](const u32x4& v, unsigned& lo4, unsigned& hi4) {  // 8 activations -> 8 bytes
      unsigned o[2] = {0u, 0u};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const unsigned h = v[j >> 1];
        const float x = __uint_as_float((j & 1) ? (h & 0xffff0000u) : (h << 16));
        float r = rintf(__fdiv_rn(x, sc));
        r = fminf(fmaxf(r, -127.f), 127.f);
        o[j >> 2] |= ((unsigned)(r != r ? 0 : (int)r) & 0xffu) << (8 * (j & 3));
      }
      lo4 = o[0];
      hi4 = o[1];
    };
    auto put16 = [&](int g, const u32x4 (&v)[4]) {
      u32x4 u0, u1;
      unsigned x, y;
      quant8(v[0], x, y); u0.x = x; u0.y = y;
      quant8(v[1], x, y); u0.z = x; u0.w = y;
      quant8(v[2], x, y); u1.x = x; u1.y = y;
      quant8(v[3], x, y); u1.z = x; u1.w = y;
      put(g, u0, u1);
    };
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
      if (wave + i * W_WAVES < groups) put16(wave + i * W_WAVES, kept[i]);
    for (int g = wave + KEEP * W_WAVES; g < groups; g += W_WAVES) {
      const u32x4 v[4] = {xp[16 * g], xp[16 * g + 1], xp[16 * g + 2], xp[16 * g + 3]};
      put16(g, v);
    }
  }
}

// WR = 2: workgroups of four waves, 128 rows x 128 tokens, two of them to a CU where a workgroup's LDS is no more than half
// of it (K up to 3328 with one term): one loads its first windows and writes its results while the other multiplies, which
// is a third of a workgroup's time at K = 2048. WR = 4: eight waves, 256 x 128, for longer rows.
template <int WR>
__global__ __launch_bounds__(WR * W_WT * 64, 2) void k_gemm_i8w(GemmArgs a, TileSplit split) {
  constexpr int W_WR = WR, W_ROWS = i8w_rows(WR), W_THREADS = WR * W_WT * 64;
  constexpr int NB = W_OPS / (4 * 16 * W_THREADS);  // batches of four pieces per thread in a staged window
  static_assert(NB == 1 || NB == 2, "");
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int r16 = lane & 15, b = lane >> 4;
  const int wr = wave % W_WR, wt = wave / W_WR;
  // SwiGLU in the epilogue: a wave's four row tiles are two of the gate and the same two of the up projection
  const bool glu = a.glu_h != nullptr;
  const int64_t NH = glu ? a.N / 2 : a.N;
  int wg_block;
  const TileRef tr = tile_of_workgroup<W_TOK>(a, split, blockIdx.x, wg_block);
  if (!tr.live) return;  // uniform for the workgroup
  const int64_t e = tr.e, tok0 = tr.tok0;
  const int ntok = (int)(tr.o1 - tok0 < W_TOK ? tr.o1 - tok0 : W_TOK);
  const bool live = 64 * wt < ntok;  // (uniform for the wave) the wave's half of the tile holds tokens
  auto tile_row = [&](int w, int r) -> int64_t {  // first row of row tile r of row wave w (-1: past the rows)
    if (glu) {
      const int64_t c = (int64_t)wg_block * (W_ROWS / 2) + w * 32 + 16 * (r & 1);
      return c < NH ? (r >> 1) * NH + c : -1;
    }
    const int64_t row = (int64_t)wg_block * W_ROWS + w * 64 + 16 * r;
    return row < a.N ? row : -1;
  };
  const int nwin = (int)(a.K / 256), NW = nwin * a.n_terms, groups = 2 * nwin, gs = a.group == 256 ? 1 : 0;
  const unsigned pitch = (unsigned)(groups + 2) * 4u;

  // ---- the load stream: per window the thread's pieces of the staged activations and the wave's weights
  const unsigned voff = (unsigned)r16 * (unsigned)a.Kp + 16u * b;
  unsigned wrow[W_RT];
#pragma unroll
  for (int r = 0; r < W_RT; ++r) {  // (a row tile past N repeats the wave's first one, or row 0, and is not stored)
    int64_t row = tile_row(wr, r);
    if (row < 0) row = tile_row(wr, 0) < 0 ? 0 : tile_row(wr, 0);
    wrow[r] = (unsigned)(row * a.Kp);
  }
  const __amdgpu_buffer_rsrc_t xrs = make_rsrc(staged_tile(a, e, tok0), (int64_t)nwin * W_FB);
  const unsigned tail_off = threadIdx.x < W_SUM / 16 ? (unsigned)(W_OPS + 16 * threadIdx.x) : 0xfffffff0u;  // (past the range: no memory access)
  u32x4 W[2][W_RT], xa[5];
  auto term_rsrc = [&](int term) { return make_rsrc(a.packed[term] + e * a.N * a.Kp, (a.E - e) * a.N * a.Kp); };
  int wterm = 0, ws = 0;  // the next window of weights to request
  __amdgpu_buffer_rsrc_t wrs = term_rsrc(0);
  auto request_w = [&](u32x4 (&dst)[W_RT]) {
#pragma unroll
    for (int r = 0; r < W_RT; ++r) dst[r] = buf_load16(wrs, voff, wrow[r] + 64u * (unsigned)ws);
    if (ws + 1 < nwin) ++ws;
    else if (wterm + 1 < a.n_terms) {
      ++wterm;
      ws = 0;
      wrs = term_rsrc(wterm);
    }
  };
  // (batch 0 goes with the tail: the offset sums)
  int xs_next[2] = {0, 0};  // the window that a batch is requested of next
  auto request_x = [&](int batch) {
#pragma unroll
    for (int i = 0; i < 4; ++i) xa[i] = buf_load16(xrs, 16u * threadIdx.x + 16u * W_THREADS * (4 * batch + i), (unsigned)W_FB * (unsigned)xs_next[batch]);
    if (batch == 0) xa[4] = buf_load16(xrs, tail_off, (unsigned)W_FB * (unsigned)xs_next[batch]);
    xs_next[batch] = xs_next[batch] + 1 < nwin ? xs_next[batch] + 1 : 0;
  };
  auto store_x = [&](int batch, unsigned buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *(lds_u32x4*)(buf + 16u * threadIdx.x + 16u * W_THREADS * (4 * batch + i)) = xa[i];
    if (batch == 0 && threadIdx.x < W_SUM / 16) *(lds_u32x4*)(buf + (unsigned)W_OPS + 16u * threadIdx.x) = xa[4];
  };
  // a window's two places for them: the next window's first batch is stored, and in the second place, before the barrier,
  // its second one; the registers are requested again at once
  auto carry_early = [&](unsigned buf) {
    store_x(0, buf);
    request_x(NB == 2 ? 1 : 0);
  };
  auto carry_late = [&](unsigned buf) {
    if (NB == 2) {
      store_x(1, buf);
      request_x(0);
    }
  };

  request_x(0);
  request_w(W[0]);
  request_w(W[1]);
  // the rows' scales of all terms, widened to float32 and one per 128 weights: 16-row tiles of contiguous bytes, 8 (16-bit)
  // or 4 scales per thread at a time where they come in whole aligned pieces
  const int sb = a.scale_dtype == BP_F32 ? 4 : 2, spp = 16 / sb;
  const int tile_pieces = (int)a.G * sb;  // 16-byte pieces of a row tile's scales: 16 G sb / 16
  for (int term = 0; term < a.n_terms; ++term) {
    const unsigned char* sbase = (const unsigned char*)a.w_scale[term];
    const unsigned lds = (unsigned)W_SC + (unsigned)(term * W_ROWS) * pitch;
    if (a.G % spp == 0) {  // (a piece stays in one row)
#pragma unroll 2
      for (int i = threadIdx.x; i < W_ROWS / 16 * tile_pieces; i += W_THREADS) {
        const int tile = i / tile_pieces, pc = i - tile * tile_pieces;
        const int64_t at = tile_row(tile >> 2, tile & 3);
        u32x4 v = {0u, 0u, 0u, 0u};
        if (at >= 0) v = *(const u32x4*)(sbase + (e * a.N + at) * a.G * sb + 16 * (int64_t)pc);
        const int row = pc * spp / (int)a.G, g0 = pc * spp - row * (int)a.G;
        const unsigned dst = lds + (unsigned)(16 * tile + row) * pitch;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (j >= spp) break;
          const uint16_t h = (uint16_t)(v[j >> 1] >> (16 * (j & 1)));
          const float f = sb == 4 ? __uint_as_float(v[j & 3]) : a.scale_dtype == BP_F16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
          if (gs) *(lds_f32*)(dst + 8u * (unsigned)(g0 + j)) = f;
          *(lds_f32*)(dst + (gs ? 8u * (unsigned)(g0 + j) + 4u : 4u * (unsigned)(g0 + j))) = f;
        }
      }
    } else {
      for (int i = threadIdx.x; i < W_ROWS * groups; i += W_THREADS) {
        const int row = i / groups, g = i - row * groups;
        const int64_t at = tile_row(row >> 6, (row >> 4) & 3);
        *(lds_f32*)(lds + (unsigned)row * pitch + 4u * (unsigned)g) =
            at < 0 ? 0.f : load_scale(sbase, a.scale_dtype, (e * a.N + at + (row & 15)) * a.G + (g >> gs));
      }
    }
  }
  carry_early(0u);
  carry_late(0u);
  __syncthreads();

  // ---- The windows. A step = (group g, row tile r): eight matrix instructions, and between them the vector work of its
  // neighbours - the step before is scaled and added to the totals, the step after is decoded - so that neither unit
  // waits for the other; the last row tile's step reloads every operand A and starting value behind its last use. The
  // workgroup's one barrier per window comes after the second group's first step: before it the next window's
  // activations go to LDS, and the reads of this window's have returned; after it the next window's are read.
  f32x4 total[W_RT][W_TT];
#pragma unroll
  for (int r = 0; r < W_RT; ++r)
#pragma unroll
    for (int m = 0; m < W_TT; ++m) total[r][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (!live) {  // (uniform) this wave only carries activations
    for (int w = 0; w < NW; ++w) {
      carry_early((unsigned)(((w & 1) ^ 1) * W_FB));
      carry_late((unsigned)(((w & 1) ^ 1) * W_FB));
      __syncthreads();
    }
  } else {
    const unsigned xlane = (unsigned)(4 * wt * 1024 + lane * 16), olane = (unsigned)(W_OPS + (64 * wt + 4 * b) * 4);
    u32x4 x[2][W_TT], wd[2][2];
    i32x4 base[W_TT], acc[2][W_TT];
    u32x2 s[2][W_RT];
    float sp = 0.f;
#pragma unroll
    for (int m = 0; m < W_TT; ++m) acc[1][m] = i32x4{0, 0, 0, 0};
    auto read_x = [&](unsigned buf, int g, int j, int m) { x[j][m] = *(const lds_u32x4*)(buf + xlane + (unsigned)(((g * 2 + j) * (W_TOK / 16) + m) * 1024)); };
    auto read_base = [&](unsigned buf, int g, int m) { base[m] = __builtin_bit_cast(i32x4, *(const lds_u32x4*)(buf + olane + (unsigned)((g * W_TOK + 16 * m) * 4))); };
    unsigned sc_at = (unsigned)W_SC + (unsigned)(wr * 64 + r16) * pitch;
    int ss = 0;
    auto read_scales = [&](u32x2 (&d)[W_RT]) {  // of the window after the one read last
#pragma unroll
      for (int r = 0; r < W_RT; ++r) d[r] = *(const lds_u32x2*)(sc_at + 16u * r * pitch);
      if (++ss == nwin) {  // (uniform) on to the next term's scales; after the last term's the first again, not used
        ss = 0;
        sc_at += (unsigned)W_ROWS * pitch - 8u * (unsigned)(nwin - 1);
        if (sc_at >= (unsigned)W_SC + (unsigned)(a.n_terms * W_ROWS) * pitch) sc_at = (unsigned)W_SC + (unsigned)(wr * 64 + r16) * pitch;
      } else {
        sc_at += 8u;
      }
    };
    auto regroup = [&](u32x4 (&w)[W_RT]) {  // .x/.y = the lane's 8 bytes of the window's first group, .z/.w = of its second
#pragma unroll
      for (int r = 0; r < W_RT; ++r) {
        const auto s0 = __builtin_amdgcn_permlane32_swap(w[r].x, w[r].z, false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(w[r].y, w[r].w, false, false);
        w[r] = u32x4{s0[0], s1[0], s0[1], s1[1]};
      }
    };
    auto step = [&](auto h_c, auto g_c, auto r_c) {
      constexpr int H = decltype(h_c)::value, g = decltype(g_c)::value, r = decltype(r_c)::value, P = r & 1, pr = (r + W_RT - 1) % W_RT;
      constexpr bool last = r == W_RT - 1;
      constexpr unsigned nbuf = (unsigned)((g == 0 ? H : H ^ 1) * W_FB);  // where the next group's operands are
      constexpr int ng = g ^ 1;
      const u32x4& nd = last ? W[g == 0 ? H : H ^ 1][0] : W[H][last ? 0 : r + 1];  // the next step's bytes
      const int gd = last ? ng : g;
      auto scaled = [&](int m, int i0) {  // two of the step before's sums of token tile m
#pragma unroll
        for (int i = i0; i < i0 + 2; ++i) total[pr][m][i] += (float)acc[P ^ 1][m][i] * sp;
        asm volatile("" : "+v"(total[pr][m]));
      };
#pragma unroll
      for (int m = 0; m < W_TT; ++m) {
        acc[P][m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, x[0][m]), __builtin_bit_cast(i32x4, wd[P][0]), base[m], 0, 0, 0);
        asm volatile("" : "+v"(acc[P][m]) : : "memory");
        if (last) {
          read_x(nbuf, ng, 0, m);
          read_base(nbuf, ng, m);
        }
        scaled(m / 2, 2 * (m & 1));
        if (m == 1) {
          wd[P ^ 1][0] = tq2_decode_i8(gd == 0 ? nd.x : nd.z);
          asm volatile("" : "+v"(wd[P ^ 1][0]));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int m = 0; m < W_TT; ++m) {
        acc[P][m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, x[1][m]), __builtin_bit_cast(i32x4, wd[P][1]), acc[P][m], 0, 0, 0);
        asm volatile("" : "+v"(acc[P][m]) : : "memory");
        if (last) read_x(nbuf, ng, 1, m);
        scaled(2 + m / 2, 2 * (m & 1));
        if (m == 1) {
          wd[P ^ 1][1] = tq2_decode_i8(gd == 0 ? nd.y : nd.w);
          asm volatile("" : "+v"(wd[P ^ 1][1]));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      sp = __uint_as_float(s[H][r][g]);
    };
    auto window = [&](auto h_c) {
      constexpr int H = decltype(h_c)::value;
      typedef std::integral_constant<int, 0> C0;
      typedef std::integral_constant<int, 1> C1;
      typedef std::integral_constant<int, 2> C2;
      typedef std::integral_constant<int, 3> C3;
      step(h_c, C0{}, C0{});
      carry_early((unsigned)((H ^ 1) * W_FB));  // (the next window's buffer was last read before the barrier)
      step(h_c, C0{}, C1{});
      step(h_c, C0{}, C2{});
      step(h_c, C0{}, C3{});
      step(h_c, C1{}, C0{});
      carry_late((unsigned)((H ^ 1) * W_FB));
      __syncthreads();
      read_scales(s[H ^ 1]);
      step(h_c, C1{}, C1{});
      regroup(W[H ^ 1]);
      step(h_c, C1{}, C2{});
      step(h_c, C1{}, C3{});
      request_w(W[H]);
      __builtin_amdgcn_sched_barrier(0);
    };
    regroup(W[0]);
    read_scales(s[0]);
#pragma unroll
    for (int m = 0; m < W_TT; ++m) {
      read_x(0u, 0, 0, m);
      read_x(0u, 0, 1, m);
      read_base(0u, 0, m);
    }
    wd[0][0] = tq2_decode_i8(W[0][0].x);
    wd[0][1] = tq2_decode_i8(W[0][0].y);
    __builtin_amdgcn_sched_barrier(0);
    int w = 0;
    for (; w + 1 < NW; w += 2) {
      window(std::integral_constant<int, 0>{});
      window(std::integral_constant<int, 1>{});
    }
    if (w < NW) window(std::integral_constant<int, 0>{});  // uniform
#pragma unroll
    for (int m = 0; m < W_TT; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) total[W_RT - 1][m][i] += (float)acc[1][m][i] * sp;
  }

  // ---- epilogue: lane holds tokens 4 b + i of each token tile, output row tile_row(wr, r) + r16. bf16 rows leave through a
  // transposition in LDS, of the wave's own 64 tokens x 64 (SwiGLU: 32) columns, as 16-byte pieces of whole lines.
  __syncthreads();  // (the staged windows' place)
  if (!live) return;
  const unsigned area = (unsigned)(wave * 8192);
  static_assert(WR * W_WT * 8192 <= W_SC, "a wave's 64 x 64 bf16 results fit its share of the staged windows");
  const int np = glu ? 4 : 8;  // 16-byte pieces of a token's columns; piece pc of token t lies at pc ^ (t % np)
  uint16_t* dst16 = glu ? a.glu_h : a.out16;
  float xs[W_TT][4], wgt[W_TT][4];  // (all loads on their way together)
  {
    const float* scales = (const float*)a.stage;
    int64_t at[W_TT][4];
#pragma unroll
    for (int m = 0; m < W_TT; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tk = 64 * wt + 16 * m + 4 * b + i;
        at[m][i] = tok0 + (tk < ntok ? tk : ntok - 1);
        xs[m][i] = scales[at[m][i]];
        wgt[m][i] = 1.f;
      }
    if (glu && a.glu_v4 && a.glu_weights) {
      if (a.glu_order) {
#pragma unroll
        for (int m = 0; m < W_TT; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) at[m][i] = a.glu_order[at[m][i]];
      }
#pragma unroll
      for (int m = 0; m < W_TT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) wgt[m][i] = a.glu_weights[a.glu_order ? clamp_i64(at[m][i], 0, a.glu_pairs - 1) : at[m][i]];
    }
  }
  auto park = [&](int tl, int c, uint16_t v) {  // token tl and column c of the wave's
    *(lds_u16*)(area + (unsigned)(tl * 16 * np + (((c >> 3) ^ (tl & (np - 1))) << 4) + 2 * (c & 7))) = v;
  };
  if (glu) {  // (uniform) h = SwiGLU of the lane's gate and up sums
#pragma unroll
    for (int m = 0; m < W_TT; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          park(16 * m + 4 * b + i, 16 * p + r16, swiglu_value(a, total[p][m][i] * xs[m][i], total[p + 2][m][i] * xs[m][i], wgt[m][i]));
  } else if (dst16) {
#pragma unroll
    for (int m = 0; m < W_TT; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < W_RT; ++r) park(16 * m + 4 * b + i, 16 * r + r16, f32_to_bf16_bits(total[r][m][i] * xs[m][i]));
  } else {
    const Output o = output_of(a);
#pragma unroll
    for (int r = 0; r < W_RT; ++r) {
      const int64_t row = tile_row(wr, r);
      if (row < 0) continue;
#pragma unroll
      for (int m = 0; m < W_TT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int tk = 64 * wt + 16 * m + 4 * b + i;
          if (tk < ntok) store_out<false>(o, (tok0 + tk) * NH + row + r16, total[r][m][i] * xs[m][i]);
        }
    }
  }
  if (!dst16) return;
  // (the wave's own writes: in order in the LDS pipeline, and the compiler sees the dependence)
  const int64_t col0 = glu ? (int64_t)wg_block * (W_ROWS / 2) + wr * 32 : (int64_t)wg_block * W_ROWS + wr * 64;
  for (int q = lane; q < 64 * np; q += 64) {
    const int tl = q / np, pc = q % np, tk = 64 * wt + tl;
    const u32x4 v = *(const lds_u32x4*)(area + (unsigned)(tl * 16 * np + ((pc ^ (tl & (np - 1))) << 4)));
    if (tk < ntok && tile_row(wr, pc >> 1) >= 0) *(u32x4*)(dst16 + (tok0 + tk) * NH + col0 + 8 * pc) = v;
  }
}

int64_t i8w_row_blocks(const GemmArgs& a, int WR) {
  const int64_t rows = a.glu_h ? a.N / 2 : a.N, per = a.glu_h ? i8w_rows(WR) / 2 : i8w_rows(WR);
  return (rows + per - 1) / per;
}
static_assert(W_SC == I8W_STAGED && i8w_rows(2) == 64 * 2, "i8w_lds_bytes");
template <int WR>
int launch_i8w(const GemmArgs& a, hipStream_t s) {
  if (const int rc = raise_lds_limit<k_gemm_i8w<WR>>(160 * 1024)) return rc;
  TileSplit split;
  const int64_t wgs = split_tiles<W_TOK>(split, a, i8w_row_blocks(a, WR));
  if (wgs < 0) return BP_ERR_UNSUPPORTED;  // (gemm_i8w_applies)
  note_kernel("gemm_tq2_i8w");
  hipLaunchKernelGGL(k_gemm_i8w<WR>, dim3((unsigned)wgs), dim3(WR * W_WT * 64), (size_t)i8w_lds_bytes(a.K, a.n_terms, WR), s, a, split);
  return check_launch("gemm_tq2_i8w");
}

}  // namespace

size_t gemm_i8w_workspace_bytes(int64_t T, int64_t K, int64_t E) {
  if (T <= 0 || K % 256 != 0 || K < 1024 || E <= 0) return 0;
  return (size_t)scales_bytes(T) + (size_t)(T + W_TOK * E + W_TOK) * (size_t)(K / 256) * (W_FB / W_TOK);
}

// Preconditions (beyond mfma_supports): TQ2; int8 activations, or bf16 ones to be quantised per row (a.quant); a workspace
// of gemm_i8w_workspace_bytes in a.stage (256-byte aligned); the rows' scales of all terms fit LDS beside the activations;
// offsets into an expert's rows and a staged tile fit 32 bits. BP_ERR_UNSUPPORTED (no message): another kernel's call.
int gemm_i8w_applies(const GemmArgs& a) {
  if (a.fmt != BP_TQ2 || (a.quant ? a.x_dtype != BP_BF16 : a.x_dtype != BP_I8)) return BP_ERR_UNSUPPORTED;
  if (!a.stage || ((uintptr_t)a.stage & 255) != 0) return BP_ERR_UNSUPPORTED;
  const size_t need = gemm_i8w_workspace_bytes(a.T, a.K, a.E);
  if (need == 0 || (size_t)a.stage_bytes < need) return BP_ERR_UNSUPPORTED;
  if (!i8w_takes(a.N, a.K, a.group, a.n_terms, a.max_rows)) return BP_ERR_UNSUPPORTED;
  const int WR = i8w_wr(a.K, a.n_terms);
  if (a.glu_h && a.N % 32 != 0) return BP_ERR_UNSUPPORTED;
  if ((((uintptr_t)a.glu_h | (uintptr_t)a.out16) & 15) != 0) return BP_ERR_UNSUPPORTED;  // (16-byte pieces of bf16 rows)
  TileSplit split;
  return split_tiles<W_TOK>(split, a, i8w_row_blocks(a, WR)) < 0 ? BP_ERR_UNSUPPORTED : BP_OK;
}

int launch_gemm_i8w(const GemmArgs& a, hipStream_t s) {
  if (const int rc = gemm_i8w_applies(a)) return rc;
  const int64_t slots = a.tiles ? a.tile_cap : a.E;
  const unsigned z = a.tiles ? 1u : (unsigned)((a.max_rows + W_TOK - 1) / W_TOK);
  const dim3 sgrid((unsigned)slots, W_TOK / 16, z);
  const int red = W_WAVES * 16 * 4;  // bytes of LDS for the row maxima
  if (!a.quant) hipLaunchKernelGGL((k_stage_i8w<BP_I8, 1>), sgrid, dim3(W_THREADS), 0, s, a);
  else if (a.K <= 1024) hipLaunchKernelGGL((k_stage_i8w<BP_BF16, 1>), sgrid, dim3(W_THREADS), red, s, a);
  else if (a.K <= 2048) hipLaunchKernelGGL((k_stage_i8w<BP_BF16, 2>), sgrid, dim3(W_THREADS), red, s, a);
  else hipLaunchKernelGGL((k_stage_i8w<BP_BF16, 4>), sgrid, dim3(W_THREADS), red, s, a);
  if (const int rc = check_launch("stage_i8w")) return rc;
  return i8w_wr(a.K, a.n_terms) == 2 ? launch_i8w<2>(a, s) : launch_i8w<4>(a, s);
}

}  // namespace bp
