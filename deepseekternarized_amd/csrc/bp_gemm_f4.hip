// Grouped GEMM over token tiles of 64 rows (TQ2) or 32 (TQ1) on v_mfma_scale_f32_32x32x64_f8f6f4: ternary weights as fp4, activations
// as two pieces, int8 ones in fp6 (exact) and bf16 ones in fp8 (exact down to 2^-9 of a block's largest), converted beforehand.
//
// Contract as everywhere (boilerplate/kernels/ternary_cuda.py:52-64, boilerplate/kernels/csrc/ternary_cuda_kernel.cu:44-99):
// out[t, n] += sum_g scale[n, g] * sum_{k in g} x[t, k] * trit[n, k] over the groups in ascending order and the stacked terms, in float32.
//
// What bounds it: the matrix cores' power and, for int8, the issue of the vector instructions beside them. The 32 x 32 x 64 form does in
// one instruction what the 16 x 16 x 128 one does in two, and up to six vector instructions behind each one cost nearly nothing: 31.2 ns
// for fp8 pieces (two 16 x 16 x 128 with four each: 35), 19.9 for fp6 ones (31.5), 2 waves per SIMD. So every choice is about vector
// instructions: signed codes that need three for 16 weights (decode) and no offset sums; int8 as fp6 pieces, whose sums come as exact
// floats (the int32 sums of v_mfma_i32 need a conversion each); one FMA per sum and group is what remains. Four waves per workgroup, 64 rows
// x 64 tokens each, two workgroups to a CU. 8192 tokens x 2048 x 6144, whole call: bf16 250 -> 183 us (the library's own bf16 product of
// that size runs 163 us at the 1.26 PFLOP/s that it reaches on this card, whose clock falls to 1.8 GHz under such load), int8 174 -> 154;
// matrix cores busy in 61 % and 47 % of the cycles. Loads straight to LDS, with the waits counted by hand, ran 1 - 2 % faster in one run
// and level in another; s_setprio around the matrix instructions and the barrier left out changed nothing.
//
// Tiles with one token tile of 32, all of TQ1's, are bound by how long the weights take to arrive and, TQ1, by the vector instructions that
// turn bytes into codes (245 per 128 k and wave, 104 for TQ2; LDS active in 32 % of the cycles, the matrix cores in 11 %). Two windows of
// weights and four steps of operands are on their way, a piece requested as soon as the one before it has been taken: 64 experts of
// 4096 / 2048, 251 tokens x 6, TQ1 bf16 264 -> 248 us against loads at a window's end; without the table's reads 5 %, without all of the
// decode 20 % less.
//
// The conversion lays the operands out as the instruction takes them, so that a step's operands (128 k) are contiguous.
//  * fp8: a block of 32 k shares an E8M0 scale 2^(e - 7), e the exponent of its largest magnitude, which the instruction applies; y = x /
//    scale = p0 + p1, p1 the remainder in E4M3. The instruction adds the products of 8 consecutive k aligned to the largest of them, and
//    drops what lies more than 13 bits below its leading one (found with single products in bounds; between blocks of 8 it keeps float32's
//    width). p0 is therefore rounded to a multiple of 2^-5 as well as to E4M3: below 2^-10 of the block's largest its low bits go to p1
//    instead of being lost. Error of a float32 output against 64 bits, normally distributed activations: 4.4e-6 -> 5e-7.
//  * fp6: q = 8 p0 + p1 with whole p0, p1 of at most 16, exact in E2M3 as n / 8; sums of a group stay below 2^24: exact, the same bits as
//    the integer kernels'.
#include <type_traits>

#include "bp_mfma.h"

namespace bp {
namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x32 __attribute__((ext_vector_type(32)));
typedef int i32x6 __attribute__((ext_vector_type(6)));
typedef __attribute__((address_space(3))) float lds_f32;
template <int V>
using FC = std::integral_constant<int, V>;
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(FC<N - 1>{});
  }
}

constexpr int P_WAVES = 4, P_THREADS = P_WAVES * 64;
constexpr int P_ROWS = P_WAVES * 64;  // output rows of a workgroup: a wave has two row tiles of 32
// ... and the tile's tokens, two token tiles of 32 (TQ2) or one (TQ1, whose weights are decoded for it once more)
constexpr int p_tok(int fmt) { return fmt == BP_TQ1 ? F4_TOK1 : F4_TOK; }
// Operands of 32 tokens x 128 k: two instructions x two pieces x 64 lanes of 32 (fp8) or 24 (fp6) bytes.
constexpr int p_unit(int act) { return act == BP_I8 ? 6144 : 8192; }
constexpr int p_stage(int act, int fmt) { return p_tok(fmt) / 32 * p_unit(act); }  // ... of the tile's tokens: what a step of 128 k takes
constexpr int P_W = P_ROWS * 64;                            // a window's weights (256 k), 64 bytes of a row as TQ2 codes
constexpr int P_TABLE = 256 * 64 * 2;                       // TQ1: byte -> five 2-bit codes, a copy per lane
// LDS: two steps' operands, two windows' weights (TQ1: one, and the table)
constexpr int p_lds_w(int act, int fmt) { return 2 * p_stage(act, fmt); }
constexpr int p_lds_t(int act, int fmt) { return p_lds_w(act, fmt) + (fmt == BP_TQ1 ? 1 : 2) * P_W; }
constexpr int p_lds(int act, int fmt) { return p_lds_t(act, fmt) + (fmt == BP_TQ1 ? P_TABLE : 0); }
static_assert(p_lds(BP_BF16, BP_TQ2) <= 80 * 1024 && p_lds(BP_BF16, BP_TQ1) <= 80 * 1024, "two workgroups to a CU");
static_assert(P_WAVES * 8192 <= p_lds(BP_I8, BP_TQ2) && P_WAVES * 4096 <= p_lds(BP_I8, BP_TQ1), "the epilogue's transposition");

// The workspace: the rows' activation scales (int8; float32 [T]), the tiles' operands, the block scales (bf16). The tile of expert e
// that starts at row tok0 lies tok0 + TOK e tokens into both, so tiles never overlap whatever the experts' row counts are.
__host__ __device__ __forceinline__ int64_t p_tokens(int64_t T, int64_t E, int tok) { return T + tok * E + tok; }
__host__ __device__ __forceinline__ int64_t p_scales_bytes(int64_t T) { return (4 * T + 255) & ~(int64_t)255; }
__host__ __device__ __forceinline__ int64_t p_row_bytes(int act, int64_t K) { return K / 128 * (p_unit(act) / 32); }
__host__ __device__ __forceinline__ int64_t p_block_bytes(int64_t K) { return K / 256 * 8; }
template <int ACT, int TOK>
__device__ __forceinline__ unsigned char* p_tile(const GemmArgs& a, int64_t e, int64_t tok0) {
  return a.stage + (ACT == BP_I8 ? p_scales_bytes(a.T) : 0) + (tok0 + TOK * e) * p_row_bytes(ACT, a.K);
}
template <int TOK>
__device__ __forceinline__ unsigned char* p_blocks(const GemmArgs& a, int64_t e, int64_t tok0) {
  return a.stage + p_tokens(a.T, a.E, TOK) * p_row_bytes(BP_BF16, a.K) + (tok0 + TOK * e) * p_block_bytes(a.K);
}

// ---- bf16 rows as two E4M3 pieces under an E8M0 scale per 32 k. One workgroup per (32 tokens, window of 256 k): wave = (group g of the
// window, eight tokens), lane = (token of eight, quarter kbA, instruction h, half kb): 16 consecutive activations, which fill registers
// 4 kb .. 4 kb + 3 of lane (m, kbA) of instruction h.
template <int TOK>
__global__ __launch_bounds__(512) void k_stage_f4_bf16(GemmArgs a) {
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  constexpr int SUBS = TOK / 32;
  const TileRef tr = tile_ref<TOK>(a, blockIdx.x, blockIdx.z / SUBS);
  if (!tr.live) return;  // uniform for the workgroup
  const int sub = blockIdx.z % SUBS;
  const int ntok = (int)(tr.o1 - tr.tok0 < TOK ? tr.o1 - tr.tok0 : TOK);
  if (32 * sub >= ntok) return;  // uniform
  const int s = blockIdx.y, g = wave & 1;
  const int m = 8 * (wave >> 1) + (lane & 7), kbA = (lane >> 3) & 1, h = (lane >> 4) & 1, kb = lane >> 5;
  int srow = 32 * sub + m;
  if (srow >= ntok) srow = ntok - 1;  // rows past the expert's tokens repeat its last one (their results are not stored)
  int64_t xrow = tr.tok0 + srow;
  if (a.x_index) xrow = clamp_i64(a.x_index[xrow] / a.x_div, 0, a.x_rows - 1);
  const uint16_t* xp = (const uint16_t*)a.x + xrow * a.K + 256 * (int64_t)s + 128 * g + 64 * kb + 32 * h + 16 * kbA;
  const u32x4 raw[2] = {*(const u32x4*)xp, *(const u32x4*)(xp + 8)};
  float y[16];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const unsigned v = raw[i >> 2][i & 3];
    y[2 * i] = __uint_as_float(v << 16);
    y[2 * i + 1] = __uint_as_float(v & 0xffff0000u);
  }
  unsigned mx = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const unsigned v = __float_as_uint(y[i]) & 0x7fffffffu;
    mx = mx > v ? mx : v;
  }
  {  // the block of 32: this lane's 16 and those of the lane with the other kbA
    const unsigned other = (unsigned)__shfl_xor((int)mx, 8, 64);
    mx = mx > other ? mx : other;
  }
  const int ex = (int)(mx >> 23);
  int sh = 134 - ex;  // brings the block's largest magnitude into [128, 256)
  sh = sh > 126 ? 126 : sh;
  float mult = __uint_as_float((unsigned)(127 + sh) << 23);
  if (ex == 255) mult = __uint_as_float(0x7fc00000u);  // a NaN or an infinity in the block: every slot becomes NaN
  const float R = 393216.f;  // (1.5 x 2^18: a float near it is a multiple of 2^-5)
  u32x4 p0, p1;
#pragma unroll
  for (int d = 0; d < 4; ++d) {  // register d of the lane's four: activations 8 (d % 2) + (d / 2), + 2, + 4, + 6
    const int v0 = d & 1, v1 = d >> 1;
    int c0 = 0, c1 = 0;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const float f0 = y[8 * v0 + 4 * q + v1] * mult, f1 = y[8 * v0 + 4 * q + 2 + v1] * mult;
      const float g0 = (f0 + R) - R, g1 = (f1 + R) - R;
      c0 = q == 0 ? __builtin_amdgcn_cvt_pk_fp8_f32(g0, g1, c0, false) : __builtin_amdgcn_cvt_pk_fp8_f32(g0, g1, c0, true);
      const float b0 = q == 0 ? __builtin_amdgcn_cvt_f32_fp8(c0, 0) : __builtin_amdgcn_cvt_f32_fp8(c0, 2);
      const float b1 = q == 0 ? __builtin_amdgcn_cvt_f32_fp8(c0, 1) : __builtin_amdgcn_cvt_f32_fp8(c0, 3);
      c1 = q == 0 ? __builtin_amdgcn_cvt_pk_fp8_f32(f0 - b0, f1 - b1, c1, false) : __builtin_amdgcn_cvt_pk_fp8_f32(f0 - b0, f1 - b1, c1, true);
    }
    p0[d] = (unsigned)c0;
    p1[d] = (unsigned)c1;
  }
  unsigned char* ob = p_tile<BP_BF16, TOK>(a, tr.e, tr.tok0) + (int64_t)(2 * s + g) * (SUBS * p_unit(BP_BF16)) + sub * p_unit(BP_BF16) + h * 4096 + kb * 1024 + (kbA * 32 + m) * 16;
  *(u32x4*)ob = p0;
  *(u32x4*)(ob + 2048) = p1;
  // the block scales of (m, kb): bytes 2 g + h of the window's dword
  const unsigned mine = (unsigned)(127 - sh), pair = mine | ((unsigned)__shfl_xor((int)mine, 16, 64) << 8);
  if (kbA == 0 && h == 0)
    *(uint16_t*)(p_blocks<TOK>(a, tr.e, tr.tok0) + (int64_t)s * (SUBS * 256) + sub * 256 + (kb * 32 + m) * 4 + 2 * g) = (uint16_t)pair;
}

// ---- int8 rows, or bf16 ones quantised as bp_quant_act_int8 does, as two E2M3 pieces: q = 8 p0 + p1, p0 = round(q / 8), |p0| <= 16,
// |p1| <= 4, both exact as n / 8. One workgroup per 16 tokens; wave = every eighth group; lane = (token t, quarter q of the group):
// the 32 activations of lane (token, q / 2) of instruction q % 2.
// KEEP: groups per wave whose bf16 activations stay in registers between the two passes (K up to 1024 KEEP; more are read again).
template <int TOK, int SRC, int KEEP>
__global__ __launch_bounds__(512) void k_stage_f4_i8(GemmArgs a) {
  constexpr int NWV = 8;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const TileRef tr = tile_ref<TOK>(a, blockIdx.x, blockIdx.z);
  if (!tr.live) return;  // uniform for the workgroup
  const int ntok = (int)(tr.o1 - tr.tok0 < TOK ? tr.o1 - tr.tok0 : TOK);
  const int mt = blockIdx.y;
  if (32 * (mt >> 1) >= ntok) return;  // uniform
  const int t = lane & 15, q = lane >> 4, tok = 16 * mt + t;
  const int64_t row = tr.tok0 + (tok < ntok ? tok : ntok - 1);  // rows past the expert's tokens repeat its last one
  int64_t src = row;
  if (a.x_index) src = clamp_i64(a.x_index[row] / a.x_div, 0, a.x_rows - 1);
  unsigned char* dst = p_tile<BP_I8, TOK>(a, tr.e, tr.tok0) + (mt >> 1) * p_unit(BP_I8);
  const int groups = (int)(a.K / 128);
  const int at = (q >> 1) * 32 + 16 * (mt & 1) + t, h = q & 1;
  auto put = [&](int g, const float (&v)[32]) {  // v: whole numbers -127 .. 127 in k order
    unsigned char* u = dst + (int64_t)g * (TOK / 32 * p_unit(BP_I8));
    f32x16 e0, e1, f0, f1;  // the instruction's order: even, odd activations of the first 16, of the second 16
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      const int k = 16 * (j >> 4) + 2 * (j & 7) + ((j >> 3) & 1);
      const float p0 = rintf(v[k] * 0.125f), p1 = fmaf(-8.f, p0, v[k]);
      if (j & 1) { e1[j >> 1] = p0; f1[j >> 1] = p1; }  // (the conversion takes its two sources in turn)
      else { e0[j >> 1] = p0; f0[j >> 1] = p1; }
    }
    const i32x6 c0 = __builtin_bit_cast(i32x6, __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(e0, e1, 8.f));
    const i32x6 c1 = __builtin_bit_cast(i32x6, __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(f0, f1, 8.f));
    unsigned char* b = u + (h * 2) * 1024 + at * 16;
    *(u32x4*)b = u32x4{(unsigned)c0[0], (unsigned)c0[1], (unsigned)c0[2], (unsigned)c0[3]};
    *(u32x4*)(b + 1024) = u32x4{(unsigned)c1[0], (unsigned)c1[1], (unsigned)c1[2], (unsigned)c1[3]};
    unsigned char* c = u + 4096 + (h * 2) * 512 + at * 8;
    *(u32x2*)c = u32x2{(unsigned)c0[4], (unsigned)c0[5]};
    *(u32x2*)(c + 512) = u32x2{(unsigned)c1[4], (unsigned)c1[5]};
  };
  float* scales = (float*)a.stage;
  if constexpr (SRC == BP_I8) {
    const u32x4* xp = (const u32x4*)((const unsigned char*)a.x + src * a.K) + 2 * q;
    if (wave == 0 && q == 0 && tok < ntok) scales[row] = a.x_scale[src];
    auto put8 = [&](int g, const u32x4& u0, const u32x4& u1) {
      float v[32];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        v[j] = (float)(int8_t)(u0[j >> 2] >> (8 * (j & 3)));
        v[16 + j] = (float)(int8_t)(u1[j >> 2] >> (8 * (j & 3)));
      }
      put(g, v);
    };
    int g = wave;
    for (; g + NWV < groups; g += 2 * NWV) {  // (two groups' loads on their way)
      const u32x4 u0 = xp[8 * g], u1 = xp[8 * g + 1], w0 = xp[8 * (g + NWV)], w1 = xp[8 * (g + NWV) + 1];
      put8(g, u0, u1);
      put8(g + NWV, w0, w1);
    }
    if (g < groups) put8(g, xp[8 * g], xp[8 * g + 1]);
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
      const int g = wave + i * NWV;
#pragma unroll
      for (int d = 0; d < 4; ++d) kept[i][d] = g < groups ? xp[16 * g + d] : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
#pragma unroll
      for (int d = 0; d < 4; ++d) look(kept[i][d]);
    for (int g = wave + KEEP * NWV; g < groups; g += NWV)
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
    for (int w = 0; w < NWV; ++w) amax = join(amax, *(const lds_f32*)(unsigned)((w * 16 + t) * 4));
    float sc = __fdiv_rn(amax, 127.0f);
    sc = sc != sc ? sc : fmaxf(sc, 1e-8f);
    if (wave == 0 && q == 0 && tok < ntok) scales[row] = sc;
    auto put16 = [&](int g, const u32x4 (&v)[4]) {
      float f[32];
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        const unsigned w = v[j >> 3][(j >> 1) & 3];
        float r = rintf(__fdiv_rn(__uint_as_float((j & 1) ? (w & 0xffff0000u) : (w << 16)), sc));
        r = fminf(fmaxf(r, -127.f), 127.f);
        f[j] = r != r ? 0.f : r;
      }
      put(g, f);
    };
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
      if (wave + i * NWV < groups) put16(wave + i * NWV, kept[i]);
    for (int g = wave + KEEP * NWV; g < groups; g += NWV) {
      const u32x4 v[4] = {xp[16 * g], xp[16 * g + 1], xp[16 * g + 2], xp[16 * g + 3]};
      put16(g, v);
    }
  }
}

// The workgroup's barrier: its LDS reads and writes have been done, its loads to registers go on.
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int ACT, int SDT, int GS, int FMT>
__global__ __launch_bounds__(P_THREADS, 2) void k_gemm_f4(GemmArgs a, TileSplit split) {
  constexpr bool I8 = ACT == BP_I8;
  constexpr int SB = SDT == BP_F32 ? 4 : 2;
  constexpr bool Q1 = FMT == BP_TQ1;
  constexpr int TOK = p_tok(FMT), UNIT = p_unit(ACT), STAGE = p_stage(ACT, FMT), LW = p_lds_w(ACT, FMT), LT = p_lds_t(ACT, FMT);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int n = lane & 31, kb = lane >> 5;
  // SwiGLU in the epilogue: a wave's two row tiles are one of the gate and the same one of the up projection
  const bool glu = a.glu_h != nullptr;
  const int64_t NH = glu ? a.N / 2 : a.N;
  int wg_block;
  const TileRef tr = tile_of_workgroup<TOK>(a, split, blockIdx.x, wg_block);
  if (!tr.live) return;  // uniform for the workgroup
  const int64_t e = tr.e, tok0 = tr.tok0;
  const int ntok = (int)(tr.o1 - tok0 < TOK ? tr.o1 - tok0 : TOK);
  const int64_t col0 = glu ? (int64_t)wg_block * (P_ROWS / 2) + wave * 32 : (int64_t)wg_block * P_ROWS + wave * 64;  // the wave's first column of the output
  const unsigned row0 = (unsigned)col0, row1 = (unsigned)(glu ? NH + col0 : col0 + 32);                             // first rows of its row tiles
  const int nwin = (int)(a.K / 256);

  // ---- the load stream. A step is 128 k of one term; (xterm, xg) and (wterm, ww): the next step of the activations and the next window
  // of the weights to request. Past the last one the offsets lie outside the buffers: such loads bring zeros that nobody reads.
  const unsigned Kp = (unsigned)a.Kp, scale_pitch = (unsigned)a.G * SB;
  constexpr unsigned NOWHERE = 0xfffffff0u;
  // a load brings 16 rows x 64 codes x 4, lane L a piece of row L / 4; a row's pieces lie in the order that lets the eight lanes which
  // read together meet all banks
  const unsigned piece = (lane & 3) ^ ((lane >> 3) & 3), wrow = (unsigned)(lane >> 2) * Kp;
  unsigned vw = wrow + 16u * piece, vx = 16u * lane;
  const unsigned vs = (unsigned)(lane & 31) * scale_pitch + (lane >= 32 ? row1 : row0) * scale_pitch;
  const __amdgpu_buffer_rsrc_t xrs = make_rsrc(p_tile<ACT, TOK>(a, e, tok0), (int64_t)2 * nwin * STAGE);
  const __amdgpu_buffer_rsrc_t ers = make_rsrc(I8 ? a.stage : p_blocks<TOK>(a, e, tok0), TOK * p_block_bytes(a.K));
  // (TQ1 rows begin at any byte: the buffer at the dword that holds their first one, up to the dword that holds the tensor's last)
  auto misaligned = [&](int term) { return Q1 ? (unsigned)((uintptr_t)(a.packed[term] + e * a.N * a.Kp) & 3) : 0u; };
  auto weights_of = [&](int term) {
    const unsigned mis = misaligned(term);
    const int64_t bytes = (a.E - e) * a.N * a.Kp + mis;
    return make_rsrc(a.packed[term] + e * a.N * a.Kp - mis, Q1 ? whole_dwords(bytes) : bytes);
  };
  auto scales_of = [&](int term) {
    const unsigned char* sbeg = (const unsigned char*)a.w_scale[term];
    return make_rsrc(sbeg + e * a.N * a.G * SB, (a.E - e) * a.N * a.G * SB);
  };
  int xterm = 0, xg = 0, wterm = 0, ww = 0;
  __amdgpu_buffer_rsrc_t wrs = weights_of(0);
  unsigned wmis = misaligned(0);
  if constexpr (Q1) {  // the byte table, a byte value per thread
    unsigned c = 0;
#pragma unroll
    for (int i = 0; i < 5; ++i) c |= (unsigned)(tq1_trit(threadIdx.x, i) + 1) << (2 * i);
    c |= c << 16;
#pragma unroll
    for (unsigned i = 0; i < 8; ++i) *(lds_u32x4*)((unsigned)LT + 128u * threadIdx.x + 16u * ((i + threadIdx.x) & 7)) = u32x4{c, c, c, c};  // (neighbours on different banks)
  }

  auto all_steps = [&](auto tt_c) {
    constexpr int TT = decltype(tt_c)::value;                   // token tiles that hold tokens
    constexpr int CHUNKS = TT * UNIT / 1024;                    // KiB of a step's operands
    constexpr int MINE = (CHUNKS + P_WAVES - 1) / P_WAVES;      // ... that a wave brings, at most
    // One token tile: the weights are what the time goes to, so two windows of them are on their way (wq; 64 KB of a CU) while a third is
    // multiplied, and four steps of the operands (xa): loads return in order, and a wait for a young one is a wait for all before it.
    // Two token tiles: a row tile of the next window (wa) and a step, which leaves the registers for the sums.
    constexpr bool DEEP = TT == 1;
    constexpr int XD = DEEP ? 4 : 1;
    u32x4 xa[XD][MINE], wa[2], wq[2][4];
    unsigned wq4[2][4], walign[2], wshift[2];  // TQ1: a piece's fifth dword; where its digits start in its bytes and in its first byte
    auto has = [&](int j) { return CHUNKS % P_WAVES == 0 || j + 1 < MINE || wave + j * P_WAVES < CHUNKS; };  // uniform
    auto load_x = [&](auto d_c, int j) { if (has(j)) xa[decltype(d_c)::value % XD][j] = buf_load16(xrs, vx, (unsigned)xg * (unsigned)STAGE + 1024u * (unsigned)(wave + j * P_WAVES)); };
    auto store_x = [&](auto d_c, int j, unsigned buf) { if (has(j)) *(lds_u32x4*)(buf * (unsigned)STAGE + 1024u * (unsigned)(wave + j * P_WAVES) + 16u * lane) = xa[decltype(d_c)::value % XD][j]; };
    auto next_x = [&]() {
      if (++xg == 2 * nwin) {
        xg = 0;
        if (++xterm >= a.n_terms) vx = NOWHERE;
      }
    };
    // half a row tile (16 rows) of window ww
    auto load_w = [&](int r, int half) { wa[half] = buf_load16(wrs, vw, ((r ? row1 : row0) + 16u * half) * Kp + 64u * (unsigned)ww); };
    auto put_w = [&](unsigned buf, int j, const u32x4& v) { *(lds_u32x4*)((unsigned)(LW + wave * 4096 + j * 1024) + buf * (unsigned)P_W + 16u * lane) = v; };  // j = 2 r + half
    auto next_w = [&]() {
      if (++ww == nwin) {
        ww = 0;
        ++wterm;
        const int t = wterm < a.n_terms ? wterm : 0;
        wrs = weights_of(t);
        wmis = misaligned(t);
        vw = wterm < a.n_terms ? vw : NOWHERE;
      }
    };
    auto load_pieces = [&](auto p_c, auto h_c) {  // window ww, a row tile's two pieces of a lane
      constexpr int P = decltype(p_c)::value, H = decltype(h_c)::value;
      if constexpr (Q1) {
        const unsigned q = (256u * (unsigned)ww) / 5u, x = 256u * (unsigned)ww - 5u * q + 64u * piece, b = (x * 205u) >> 10;  // (x < 1024: x / 5)
        const unsigned off = wmis + wrow + q + b;
        if constexpr (H == 1) {  // (row tile 1 of the window before has been looked up by then)
          walign[P] = off;
          wshift[P] = 2u * (x - 5u * b);
        }
#pragma unroll
        for (int j = 2 * H; j < 2 * H + 2; ++j) {
          const unsigned so = ((H ? row1 : row0) + 16u * (j & 1)) * Kp, at = vw == NOWHERE ? NOWHERE - 16u : off & ~3u;  // (16 rows: a multiple of 4 bytes)
          wq[P][j] = buf_load16(wrs, at, so);
          wq4[P][j] = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(wrs, (int)(at + 16u), (int)so, 0);
        }
      } else {
#pragma unroll
        for (int j = 2 * H; j < 2 * H + 2; ++j) wq[P][j] = buf_load16(wrs, vw, ((H ? row1 : row0) + 16u * (j & 1)) * Kp + 64u * (unsigned)ww);
      }
      if constexpr (H == 1) next_w();
    };
    auto load_window = [&](auto p_c) {
      load_pieces(p_c, FC<0>{});
      load_pieces(p_c, FC<1>{});
    };
    // TQ1: a lane's 13 or 14 bytes -> 10 bits each -> strung together, shifted by the digits that the first byte holds of the codes before
    const unsigned lane2 = (unsigned)LT + 2u * lane;
    auto look_up = [&](unsigned (&c)[14], auto p_c, int j) {
      constexpr int P = decltype(p_c)::value;
      const u32x4& w = wq[P][j];
      const unsigned d[4] = {__builtin_amdgcn_alignbyte(w.y, w.x, walign[P]), __builtin_amdgcn_alignbyte(w.z, w.y, walign[P]),
                             __builtin_amdgcn_alignbyte(w.w, w.z, walign[P]), __builtin_amdgcn_alignbyte(wq4[P][j], w.w, walign[P])};
#pragma unroll
      for (int i = 0; i < 14; ++i) {
        const unsigned v = d[i >> 2];
        c[i] = *(const lds_u16*)(((v >> (8 * (i & 3))) & 0xffu) * 128u + lane2);
      }
    };
    auto string = [&](const unsigned (&c)[14], auto p_c) {
      const unsigned sh = wshift[decltype(p_c)::value];
      const unsigned s0 = c[0] | c[1] << 10 | c[2] << 20 | c[3] << 30, s1 = c[3] >> 2 | c[4] << 8 | c[5] << 18 | c[6] << 28;
      const unsigned s2 = c[6] >> 4 | c[7] << 6 | c[8] << 16 | c[9] << 26, s3 = c[9] >> 6 | c[10] << 4 | c[11] << 14 | c[12] << 24, s4 = c[12] >> 8 | c[13] << 2;
      return u32x4{__builtin_amdgcn_alignbit(s1, s0, sh), __builtin_amdgcn_alignbit(s2, s1, sh), __builtin_amdgcn_alignbit(s3, s2, sh),
                   __builtin_amdgcn_alignbit(s4, s3, sh)};
    };
    // scales: 16 bytes of each row at a time, lane L's row of its row tile (L / 32); windows that these cover
    constexpr int CW = (16 / SB) >> (GS ? 0 : 1);
    u32x4 sfar;
    __amdgpu_buffer_rsrc_t srs = scales_of(0);
    auto load_scales = [&](__amdgpu_buffer_rsrc_t rs, int win) { sfar = buf_load16(rs, vs, (unsigned)((2 * win) >> GS) * SB); };

    f32x16 total[2][TT], C[2];
    i32x8 A[TT][2][2], B[2][2];
    u32x4 raw[2], sq[2];
    int sa[TT], sn[DEEP ? 2 : 1][TT];
    float sc[2][2], sp = 0.f;  // [row tile][group of the window]
    int one_half = 0x7e7e7e7e, hi8 = 0x85858585, lo8 = 0x82828282;  // (E8M0: 2^-1, 2^6, 2^3)
    asm volatile("" : "+v"(one_half), "+v"(hi8), "+v"(lo8));
    unsigned mC = 0xccccccccu, m4 = 0x44444444u;
    asm volatile("" : "+v"(mC), "+s"(m4));
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) total[r][t][i] = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) C[1][i] = 0.f;

    // where the lane reads a step's operands and weights (opaque: an address is this register and a constant in the instruction)
    unsigned at16, at8, atw;
    auto read_from = [&](unsigned buf, unsigned wbuf, int g) {
      at16 = buf * (unsigned)STAGE + 16u * lane;
      at8 = buf * (unsigned)STAGE + 8u * lane;
      atw = (unsigned)(LW + wave * 4096) + wbuf * (unsigned)P_W + 64u * n + 16u * ((2 * g + kb) ^ ((n >> 1) & 3));
      asm volatile("" : "+v"(at16), "+v"(at8), "+v"(atw));
    };
    auto read_a = [&](auto t_c, auto h_c, auto p_c) {
      constexpr int t = decltype(t_c)::value, h = decltype(h_c)::value, p = decltype(p_c)::value;
      if constexpr (I8) {
        const u32x4 lo = *(const lds_u32x4*)(at16 + (unsigned)(t * UNIT + (h * 2 + p) * 1024));
        const u32x2 hi = *(const lds_u32x2*)(at8 + (unsigned)(t * UNIT + 4096 + (h * 2 + p) * 512));
        A[t][h][p] = i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, 0, 0};
      } else {
        const u32x4 lo = *(const lds_u32x4*)(at16 + (unsigned)(t * UNIT + (h * 2 + p) * 2048)), hi = *(const lds_u32x4*)(at16 + (unsigned)(t * UNIT + (h * 2 + p) * 2048 + 1024));
        A[t][h][p] = i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
      }
    };
    auto read_w = [&](int r) { raw[r] = *(const lds_u32x4*)(atw + 2048u * r); };
    auto load_blocks = [&](auto h_c, int win) {
#pragma unroll
      for (int t = 0; t < TT; ++t) sn[decltype(h_c)::value][t] = I8 ? 0 : (int)__builtin_amdgcn_raw_buffer_load_b32(ers, 4 * lane, win * (TOK / 32 * 256) + t * 256, 0);
    };
    // A packed dword's 16 codes u = trit + 1 as two operand dwords: with a code in a nibble's upper two bits, flipping the lower of them
    // and clearing the nibble's other half leaves the E2M1 number -2 (u - 1) (0100, 0000 or 1000, 1100; the code 3, never written, -0).
    auto decode = [&](int r, int d) {
      const unsigned w = raw[r][d], x = w << 2;
      B[r][d >> 1][2 * (d & 1)] = (int)((x ^ m4) & mC);
      B[r][d >> 1][2 * (d & 1) + 1] = (int)((w ^ m4) & mC);
    };
    auto take_scales = [&](int win) {  // of window `win` of its term
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        if constexpr (SDT == BP_F32) {
          sc[r][0] = -__uint_as_float(sq[r].x);
          sc[r][1] = GS ? sc[r][0] : -__uint_as_float(sq[r].y);
          sq[r] = GS ? u32x4{sq[r].y, sq[r].z, sq[r].w, 0u} : u32x4{sq[r].z, sq[r].w, 0u, 0u};
        } else {
          unsigned v = sq[r].x;
          if (GS && (win & 1)) v >>= 16;  // uniform
          const uint16_t lo = (uint16_t)v, hi = GS ? lo : (uint16_t)(v >> 16);
          sc[r][0] = SDT == BP_F16 ? -f16_bits_to_f32(lo) : -bf16_bits_to_f32(lo);
          sc[r][1] = SDT == BP_F16 ? -f16_bits_to_f32(hi) : -bf16_bits_to_f32(hi);
          if (!GS || (win & 1)) sq[r] = u32x4{sq[r].y, sq[r].z, sq[r].w, 0u};
        }
        asm volatile("" : "+v"(sc[r][0]), "+v"(sc[r][1]));
      }
    };

    // ---- prologue: step 0 and window 0 into LDS, step 1 and the weights that follow on their way
    if constexpr (Q1) meet();  // (the table)
    load_scales(srs, 0);
    load_blocks(FC<0>{}, 0);
    if constexpr (DEEP) load_blocks(FC<1>{}, 1);
#pragma unroll
    for (int j = 0; j < MINE; ++j) load_x(FC<0>{}, j);
    next_x();
    load_window(FC<0>{});
    if constexpr (DEEP) load_window(FC<1>{});
#pragma unroll
    for (int j = 0; j < MINE; ++j) store_x(FC<0>{}, j, 0u);
    static_for<XD>([&](auto d_c) {  // steps 1 .. XD
#pragma unroll
      for (int j = 0; j < MINE; ++j) load_x(FC<decltype(d_c)::value + 1>{}, j);
      next_x();
    });
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (Q1) {
        unsigned c[14];
        look_up(c, FC<0>{}, j);
        put_w(0u, j, string(c, FC<0>{}));
      } else {
        put_w(0u, j, wq[0][j]);
      }
    }
    if constexpr (DEEP) {
      load_window(FC<0>{});
    } else {
      load_w(0, 0);
      load_w(0, 1);
    }
    meet();
    read_from(0u, 0u, 0);
    read_w(0);
    read_w(1);
    static_for<4 * TT>([&](auto i) {
      constexpr int I = decltype(i)::value;
      read_a(FC<(I >> 2)>{}, FC<((I >> 1) & 1)>{}, FC<(I & 1)>{});
    });
    // step 1's operands go to the other buffer, which nobody has read yet
#pragma unroll
    for (int j = 0; j < MINE; ++j) store_x(FC<1>{}, j, 1u);
#pragma unroll
    for (int j = 0; j < MINE; ++j) load_x(FC<XD + 1>{}, j);
    next_x();
#pragma unroll
    for (int d = 0; d < 4; ++d) decode(0, d);

    // The step's operands are in registers when it begins. Its first half multiplies row tile 0; then all waves have taken theirs, the
    // step after the next may go to this step's place in LDS, and the next step's are read behind the second half's instructions.
    int term = 0, win = 0;       // the window being multiplied
    unsigned wb = 0;             // TQ2: the place of its weights
    unsigned look[2][14];        // TQ1: two pieces of the next window on their way through the table
    u32x4 made[2];
    auto step = [&](auto h_c, auto g_c) {  // h: the window's parity
      constexpr int g = decltype(g_c)::value, NP = decltype(h_c)::value ^ 1;
      auto slot = [&](auto q_c) {
        constexpr int q = decltype(q_c)::value, c = q / 4, r = c / TT, t = c % TT, s = q % 4, h = s / 2, p = s % 2;
        constexpr int pc = (c + 2 * TT - 1) % (2 * TT), pr = pc / TT, pt = pc % TT;  // the chain before
        constexpr int half = 4 * TT;
        if constexpr (I8) {
          C[c & 1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A[t][h][p], B[r][h], s == 0 ? f32x16{} : C[c & 1], 2, 4, 0, p ? lo8 : hi8, 0, one_half);
        } else {
          C[c & 1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A[t][h][p], B[r][h], s == 0 ? f32x16{} : C[c & 1], 0, 4, 2 * g + h, sa[t], 0, one_half);
        }
        asm volatile("" : "+v"(C[c & 1]) : : "memory");
        // the chain before's sums under the rows' scales
#pragma unroll
        for (int i = 4 * s; i < 4 * s + 4; ++i) total[pr][pt][i] += sp * C[(c & 1) ^ 1][i];
        asm volatile("" : "+v"(total[pr][pt]));
        if constexpr (q < 4) decode(1, q);
        if constexpr (Q1 && q < 2) look_up(look[q], FC<NP>{}, 2 * g + q);
        if constexpr (Q1 && q >= 2 && q < 4) made[q - 2] = string(look[q - 2], FC<NP>{});
        if constexpr (q >= half) {  // this step's operands and weights have been read by all waves: the next ones come
          constexpr int k = q - half;
          if constexpr (k == 0) {
            // A row tile of the next window's weights per step goes to LDS, the wave's own, whose accesses stay in order. TQ1 has one
            // place: row tile 0 behind the reads of this window's second group, row tile 1 ahead of the next one's first.
            auto put_row_tile = [&]() {
#pragma unroll
              for (int half = 0; half < 2; ++half) put_w(Q1 ? 0u : wb ^ 1u, 2 * g + half, Q1 ? made[half] : DEEP ? wq[NP][2 * g + half] : wa[half]);
            };
            if constexpr (!Q1 || g == 1) put_row_tile();
            read_from(g ^ 1, Q1 ? 0u : g == 0 ? wb : wb ^ 1u, g ^ 1);
            read_w(0);
            read_w(1);
            if constexpr (Q1 && g == 0) put_row_tile();
          }
          read_a(FC<t>{}, FC<h>{}, FC<p>{});
          if constexpr (k == 1 && !DEEP) {
            load_w(g ^ 1, 0);
            load_w(g ^ 1, 1);
          }
          if constexpr (k == 1 && DEEP) load_pieces(FC<NP>{}, FC<g>{});
          // the step after the next to LDS, a later one requested
          if constexpr (TT == 2) {
            if constexpr (k >= 1 && k <= MINE) store_x(FC<0>{}, k - 1, g);
            if constexpr (k >= 2 && k <= MINE + 1) load_x(FC<0>{}, k - 2);
          } else {
            constexpr int S = 2 * (NP ^ 1) + g + 2;  // (the step after the next, of four)
            if constexpr (k >= 1 && k <= MINE) store_x(FC<S>{}, k - 1, g);
            if constexpr (k == 3) {
#pragma unroll
              for (int j = 0; j < MINE; ++j) load_x(FC<S>{}, j);
            }
          }
          if constexpr (q == 2 * half - 1) next_x();
          constexpr int d = q - (2 * half - 4);
          if constexpr (TT == 2 && d >= 0) decode(0, d);
          if constexpr (TT == 1 && d >= 2) {
            decode(0, 2 * (d - 2));
            decode(0, 2 * (d - 2) + 1);
          }
        }
        if constexpr (s == 3) sp = sc[r][g];
        __builtin_amdgcn_sched_barrier(0);
      };
      static_for<4 * TT>(slot);
      meet();
      if constexpr (g == 1 && !DEEP) next_w();
      static_for<4 * TT>([&](auto i) { slot(FC<4 * TT + decltype(i)::value>{}); });
    };
    auto window = [&](auto h_c) {
      const int next = win + 1 < nwin ? win + 1 : 0;
      if (win % CW == 0) {  // uniform
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          unsigned v = sfar[i];
          // (a copy that isn't the same register: the load below goes straight to sfar's, without a move that waits for it)
          if constexpr (DEEP) asm volatile("v_mov_b32 %0, %1" : "=&v"(v) : "v"(sfar[i]));
          const auto s2 = __builtin_amdgcn_permlane32_swap(v, v, false, false);
          sq[0][i] = s2[0];
          sq[1][i] = s2[1];
        }
        const bool more = win + CW < nwin;
        if constexpr (DEEP) {
          if (!more && term + 1 < a.n_terms) srs = scales_of(term + 1);  // uniform
          load_scales(srs, more ? win + CW : 0);
        } else {
          load_scales(scales_of(more || term + 1 == a.n_terms ? term : term + 1), more ? win + CW : 0);
        }
      }
      take_scales(win);
#pragma unroll
      for (int t = 0; t < TT; ++t) sa[t] = sn[decltype(h_c)::value][t];
      load_blocks(h_c, !DEEP ? next : win + 2 < nwin ? win + 2 : win + 2 - nwin);
      step(h_c, FC<0>{});
      step(h_c, FC<1>{});
      win = next;
      wb ^= 1u;
      if (next == 0) ++term;
    };
    const int NW = nwin * a.n_terms;
    if constexpr (DEEP) {
      int w = 0;
      for (; w + 1 < NW; w += 2) {
        window(FC<0>{});
        window(FC<1>{});
      }
      if (w < NW) window(FC<0>{});  // uniform
    } else {
      for (int w = 0; w < NW; ++w) window(FC<0>{});
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) total[1][TT - 1][i] += sp * C[1][i];

    // ---- epilogue: lane (n, kb) holds tokens 8 (i / 4) + 4 kb + i % 4 of each token tile, column n of each row tile. bf16 rows leave
    // through a transposition in LDS, of the wave's own tokens, as 16-byte pieces of whole lines.
    meet();  // (the operands' place)
    float xs[TT][16], wgt[TT][16];  // (all loads on their way together)
    {
      const float* scales = (const float*)a.stage;
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int tk = 32 * t + 8 * (i / 4) + 4 * kb + i % 4;
          const int64_t at = tok0 + (tk < ntok ? tk : ntok - 1);
          xs[t][i] = I8 ? scales[at] : 1.f;
          wgt[t][i] = 1.f;
          if (glu && a.glu_v4 && a.glu_weights) wgt[t][i] = a.glu_weights[a.glu_order ? clamp_i64(a.glu_order[at], 0, a.glu_pairs - 1) : at];
        }
    }
    uint16_t* dst16 = glu ? a.glu_h : a.out16;
    const int np = glu ? 4 : 8;  // 16-byte pieces of a token's columns; piece pc of token t lies at pc ^ (t % np)
    const unsigned area = (unsigned)(wave * 4096 * TT);
    auto park = [&](int tl, int c, uint16_t v) {  // token tl and column c of the wave's
      *(lds_u16*)(area + (unsigned)(tl * 16 * np + (((c >> 3) ^ (tl & (np - 1))) << 4) + 2 * (c & 7))) = v;
    };
    if (glu) {  // (uniform)
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          park(32 * t + 8 * (i / 4) + 4 * kb + i % 4, n, swiglu_value(a, total[0][t][i] * xs[t][i], total[1][t][i] * xs[t][i], wgt[t][i]));
    } else if (dst16) {
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
          for (int r = 0; r < 2; ++r) park(32 * t + 8 * (i / 4) + 4 * kb + i % 4, 32 * r + n, f32_to_bf16_bits(total[r][t][i] * xs[t][i]));
    } else {
      const Output o = output_of(a);
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int tk = 32 * t + 8 * (i / 4) + 4 * kb + i % 4;
#pragma unroll
          for (int r = 0; r < 2; ++r)
            if (tk < ntok && col0 + 32 * r + n < NH) store_out<false>(o, (tok0 + tk) * NH + col0 + 32 * r + n, total[r][t][i] * xs[t][i]);
        }
    }
    if (!dst16) return;
    // (the wave's own writes: in order in the LDS pipeline, and the compiler sees the dependence)
    for (int q = lane; q < 32 * TT * np; q += 64) {
      const int tl = q / np, pc = q % np;
      const u32x4 v = *(const lds_u32x4*)(area + (unsigned)(tl * 16 * np + ((pc ^ (tl & (np - 1))) << 4)));
      if (tl < ntok && col0 + 8 * pc < NH) *(u32x4*)(dst16 + (tok0 + tl) * NH + col0 + 8 * pc) = v;
    }
  };
  if constexpr (!Q1) {
    if (ntok > 32) {
      all_steps(FC<2>{});
      return;
    }
  }
  all_steps(FC<1>{});
}

int64_t f4_row_blocks(const GemmArgs& a) { return a.glu_h ? (a.N / 2 + P_ROWS / 2 - 1) / (P_ROWS / 2) : (a.N + P_ROWS - 1) / P_ROWS; }

template <int ACT, int SDT, int GS, int FMT>
int launch_f4_g(const GemmArgs& a, hipStream_t s, const char* name) {
  constexpr int LDS = p_lds(ACT, FMT);
  if (const int rc = raise_lds_limit<k_gemm_f4<ACT, SDT, GS, FMT>>(LDS)) return rc;
  TileSplit split;
  const int64_t wgs = split_tiles<p_tok(FMT)>(split, a, f4_row_blocks(a));
  if (wgs < 0) return BP_ERR_UNSUPPORTED;  // (gemm_f4_applies)
  note_kernel(name);
  hipLaunchKernelGGL((k_gemm_f4<ACT, SDT, GS, FMT>), dim3((unsigned)wgs), dim3(P_THREADS), (size_t)LDS, s, a, split);
  return check_launch(name);
}
template <int ACT, int FMT>
int launch_f4(const GemmArgs& a, hipStream_t s, const char* name) {
  const bool g = a.group == 256;
  if (a.scale_dtype == BP_F16) return g ? launch_f4_g<ACT, BP_F16, 1, FMT>(a, s, name) : launch_f4_g<ACT, BP_F16, 0, FMT>(a, s, name);
  if (a.scale_dtype == BP_BF16) return g ? launch_f4_g<ACT, BP_BF16, 1, FMT>(a, s, name) : launch_f4_g<ACT, BP_BF16, 0, FMT>(a, s, name);
  return g ? launch_f4_g<ACT, BP_F32, 1, FMT>(a, s, name) : launch_f4_g<ACT, BP_F32, 0, FMT>(a, s, name);
}

// The conversion, then the product.
template <int FMT>
int launch_f4_all(const GemmArgs& a, hipStream_t s, const char* name) {
  constexpr int TOK = p_tok(FMT);
  const int64_t slots = a.tiles ? a.tile_cap : a.E;
  const unsigned z = a.tiles ? 1u : (unsigned)((a.max_rows + TOK - 1) / TOK);
  if (a.x_dtype == BP_BF16 && !a.quant) {
    hipLaunchKernelGGL(k_stage_f4_bf16<TOK>, dim3((unsigned)slots, (unsigned)(a.K / 256), TOK / 32 * z), dim3(512), 0, s, a);
    if (const int rc = check_launch("stage_f4")) return rc;
    return launch_f4<BP_BF16, FMT>(a, s, name);
  }
  const dim3 sgrid((unsigned)slots, TOK / 16, z);
  const int red = 8 * 16 * 4;  // bytes of LDS for the row maxima
  if (!a.quant) hipLaunchKernelGGL((k_stage_f4_i8<TOK, BP_I8, 1>), sgrid, dim3(512), 0, s, a);
  else if (a.K <= 1024) hipLaunchKernelGGL((k_stage_f4_i8<TOK, BP_BF16, 1>), sgrid, dim3(512), red, s, a);
  else if (a.K <= 2048) hipLaunchKernelGGL((k_stage_f4_i8<TOK, BP_BF16, 2>), sgrid, dim3(512), red, s, a);
  else hipLaunchKernelGGL((k_stage_f4_i8<TOK, BP_BF16, 4>), sgrid, dim3(512), red, s, a);
  if (const int rc = check_launch("stage_f4")) return rc;
  return launch_f4<BP_I8, FMT>(a, s, name);
}

}  // namespace

size_t gemm_f4_workspace_bytes(int act, int64_t T, int64_t K, int64_t E, int fmt) {
  if (T <= 0 || K % 256 != 0 || K < 1024 || E <= 0) return 0;
  const int64_t per = p_row_bytes(act, K) + (act == BP_I8 ? 0 : p_block_bytes(K));
  return (size_t)(act == BP_I8 ? p_scales_bytes(T) : 0) + (size_t)p_tokens(T, E, p_tok(fmt)) * (size_t)per;
}

// Preconditions (beyond mfma_supports): bf16 activations, int8 ones, or bf16 ones to be quantised per row (a.quant); a workspace of
// gemm_f4_workspace_bytes in a.stage (256-byte aligned); offsets into an expert's rows and a staged tile fit 32 bits.
// BP_ERR_UNSUPPORTED (no message): another kernel's call.
int gemm_f4_applies(const GemmArgs& a) {
  if (a.quant ? a.x_dtype != BP_BF16 : a.x_dtype != BP_I8 && a.x_dtype != BP_BF16) return BP_ERR_UNSUPPORTED;
  if (!a.stage || ((uintptr_t)a.stage & 255) != 0) return BP_ERR_UNSUPPORTED;
  const int act = a.quant ? BP_I8 : a.x_dtype;
  const int64_t tok = p_tok(a.fmt);
  const size_t need = gemm_f4_workspace_bytes(act, a.T, a.K, a.E, a.fmt);
  if (need == 0 || (size_t)a.stage_bytes < need) return BP_ERR_UNSUPPORTED;
  if (a.K > ((int64_t)1 << 20) || a.N * a.Kp > ((int64_t)1 << 31) - 4096 || (a.max_rows + tok - 1) / tok > 32767) return BP_ERR_UNSUPPORTED;
  if (a.fmt == BP_TQ1 && a.Kp != (a.K + 4) / 5) return BP_ERR_UNSUPPORTED;
  if (a.tiles && a.max_rows != tok) return BP_ERR_UNSUPPORTED;  // (a list of other tiles)
  if (!a.tiles && (a.max_rows + tok - 1) / tok * tok * a.E > 4 * a.T + tok * a.E) return BP_ERR_UNSUPPORTED;  // (a loose bound on the rows per expert: mostly tiles that do not exist)
  if (a.glu_h && (!a.overwrite || a.N % 32 != 0)) return BP_ERR_UNSUPPORTED;
  if ((((uintptr_t)a.glu_h | (uintptr_t)a.out16) & 15) != 0) return BP_ERR_UNSUPPORTED;  // (16-byte pieces of bf16 rows)
  TileSplit split;
  const int64_t wgs = a.fmt == BP_TQ1 ? split_tiles<F4_TOK1>(split, a, f4_row_blocks(a)) : split_tiles<F4_TOK>(split, a, f4_row_blocks(a));
  return wgs < 0 ? BP_ERR_UNSUPPORTED : BP_OK;
}

int launch_gemm_f4(const GemmArgs& a, hipStream_t s, bool rewritten) {
  if (const int rc = gemm_f4_applies(a)) return rc;
  const bool i8 = a.quant || a.x_dtype == BP_I8;
  if (a.fmt == BP_TQ1) return launch_f4_all<BP_TQ1>(a, s, i8 ? "gemm_tq1f4_i8" : "gemm_tq1f4_bf16");
  return launch_f4_all<BP_TQ2>(a, s, rewritten ? (i8 ? "gemm_tq1_as_tq2f4_i8" : "gemm_tq1_as_tq2f4_bf16") : i8 ? "gemm_tq2f4_i8" : "gemm_tq2f4_bf16");
}

}  // namespace bp
