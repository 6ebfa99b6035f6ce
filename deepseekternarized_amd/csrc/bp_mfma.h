// Shared pieces of the tuned gfx950 MFMA kernels (bp_mfma_tq2.hip, bp_mfma_tq1.hip).
//
// Packed trits are decoded in registers straight into MFMA operands, one 16-row x 16-token tile per
// instruction (v_mfma_f32_16x16x32_bf16 for bf16 activations, v_mfma_i32_16x16x64_i8 for int8).
// Accumulators are flushed at every 128-wide K group: total += acc * scale[n, g] in float32, so the
// scale multiplies the group sum exactly as in the reference contract
// (boilerplate/kernels/ternary_cuda.py:58-63, boilerplate/kernels/csrc/boilerplate_cpu.cpp:114-124).
// Stacked terms share one staging of the activations and one output write.
//
// Operand A = activations (row i = token), operand B = weights (column j = output row), so a lane
// ends with 4 tokens x 1 output row and needs one scale per group.
//
// The kernels address LDS absolutely: they declare no static LDS, so the dynamic allocation requested
// at launch starts at LDS address 0.
#pragma once
#include <cstdlib>

#include "bp_common.h"

namespace bp {

// A launcher whose source is compiled twice (BP_REPLACES in bp_common.h): NAME_add for launches that add to their outputs,
// NAME_set for those that replace them.
#define BP_LAUNCHER(NAME, PARAMS, ARGS) \
  int NAME##_add PARAMS;                \
  int NAME##_set PARAMS;                \
  inline int NAME PARAMS { return a.overwrite ? NAME##_set ARGS : NAME##_add ARGS; }
#if defined(BP_REPLACES) && BP_REPLACES
#define BP_OUTPUTS(NAME) NAME##_set
#else
#define BP_OUTPUTS(NAME) NAME##_add
#endif

// implemented in bp_mfma_tq2.hip / bp_mfma_tq1.hip; R, MT, waves: the tiling chosen by launch_mfma
BP_LAUNCHER(launch_mfma_tq2, (const GemmArgs& a, hipStream_t s, int R, int MT, int waves), (a, s, R, MT, waves))
BP_LAUNCHER(launch_mfma_tq1, (const GemmArgs& a, hipStream_t s, int waves), (a, s, waves))
// bp_gemm_tq2.hip: TQ2 with token tiles of 32 (experts with more than 16 token rows)
BP_LAUNCHER(launch_gemm_tq2, (const GemmArgs& a, hipStream_t s), (a, s))
int launch_gemm_tq2f(const GemmArgs& a, hipStream_t s);
int gemm_tq2f_applies(const GemmArgs& a);  // BP_OK where launch_gemm_tq2f takes the call (nothing is launched)
// bp_gemm_i8w.hip: TQ2 with int8 activations (or bf16 ones that it quantises: GemmArgs::quant) and token tiles of 128
constexpr int I8W_TOK = 128;
constexpr int I8W_STAGED = 2 * (2 * 2 * (I8W_TOK / 16) * 1024 + 2 * I8W_TOK * 4);  // LDS: two staged windows of the activations
int launch_gemm_i8w(const GemmArgs& a, hipStream_t s);
int gemm_i8w_applies(const GemmArgs& a);  // BP_OK where launch_gemm_i8w takes the call (nothing is launched)
// LDS of a workgroup of 64 WR rows: the staged windows and the rows' scales of all terms, float32. WR = 2 where two workgroups
// fit a CU, else 4, or 0 where that does not fit either.
inline int64_t i8w_lds_bytes(int64_t K, int n_terms, int WR) { return I8W_STAGED + (int64_t)n_terms * 64 * WR * (K / 128 + 2) * 4; }
inline int i8w_wr(int64_t K, int n_terms) { return i8w_lds_bytes(K, n_terms, 2) <= 80 * 1024 ? 2 : i8w_lds_bytes(K, n_terms, 4) <= 160 * 1024 ? 4 : 0; }
// Sizes that the kernel takes (beside them: alignments and workspace, gemm_i8w_applies and mfma_supports).
inline bool i8w_takes(int64_t N, int64_t K, int64_t group, int n_terms, int64_t max_rows) {
  return (group == 128 || (group == 256 && K >= 2048)) && K % 256 == 0 && K >= 1024 && K <= ((int64_t)1 << 20) && N % 16 == 0 && i8w_wr(K, n_terms) != 0 &&
         N * (K / 4) <= ((int64_t)1 << 31) - 4096 && (max_rows + I8W_TOK - 1) / I8W_TOK <= 65535;
}
// Calls that run on it when the caller brings a workspace, by their blocks of 128 tokens x 256 rows.
// One expert: from 96 tokens (64 / 96 tokens x 2048 x 32768, 128 blocks each, 1.50 / 0.94 of the time on the 32-token tiles, x 65536 1.12 /
// 0.87; a second tile may be nearly empty: 140 tokens x 2048 x 16384 0.94) and 128 blocks on as two small workgroups per CU (WR = 2), from 192 as one of eight waves, which takes as long for 64
// blocks as for 256. us on it / on the 32-token tiles: 2048 x 2048 x 2048 (128 blocks) 32.8 / 35.5, 512 x 2048 x 6144 (96) 31.1 / 31.9,
// 1024 x 2048 x 2048 (64) 30.9 / 20.4; eight waves: 3072 x 4096 x 2048 (192) 65.7 / 73.5, 2048 x 4096 x 2048 (128) 63.7 / 51.8, in two
// terms 2048 x 2048 x 2048 (128) 56.8 / 51.2, 3072 x 2048 x 2048 (192) 60.0 / 73.3, 1024 x 7168 x 6144 (192) 100.6 / 103.9.
// Several experts, whose last tiles are partly empty: from 112 rows per expert and 384 blocks on. 64 experts x 2048 x 2048, 64 / 80 / 96 /
// 112 / 128 rows each: 1.26 / 1.03 / 1.02 / 0.86 / 0.80 of the time on the 32-token tiles (with 0 to twice as many rows: 1.04 / 1.01 / 0.99 /
// 0.91 / 0.88); 16 experts x 2048 x 4096 at 256 rows (256 blocks) 0.91 and 1.09, 16 x 4096 x 1024 at 192 (384) 1.05 and 0.94.
inline bool i8w_pays(int64_t T, int64_t N, int64_t K, int64_t E, int n_terms) {
  const int64_t blocks = (T + I8W_TOK - 1) / I8W_TOK * ((N + 255) / 256);
  return E == 1 ? T >= 96 && blocks >= (i8w_wr(K, n_terms) == 2 ? 128 : 192) : T >= 112 * E && blocks >= 384;
}
// bp_gemm_tq1.hip: TQ1 with token tiles of 32 on the fp8 x fp4 matrix instruction (experts with more than 8 token rows);
// BP_ERR_UNSUPPORTED without a message when the call is outside its preconditions
BP_LAUNCHER(launch_gemm_tq1, (const GemmArgs& a, hipStream_t s), (a, s))
// TQ1 calls of seven or eight token rows per expert that run on the tile kernel over converted activations when the
// caller brings a workspace, rather than as two launches of the four-row decode kernel: dense batches (four rows per
// expert on average) of at least 512 blocks of 512 output rows. Measured with 8 rows per expert: 128 experts x 2048 x
// 7168 204 against 230 us, 64 x 4096 x 4096 113 against 130 us, 128 x 7168 x 2048 268 against 272 us; 16 experts x
// 2048 x 7168 (64 blocks) 82 against 79 us; six rows per expert 203 against 198 us.
inline bool tq1_rows_on_tiles(int64_t max_rows, int64_t E, int64_t T, int64_t N) {
  return max_rows >= 7 && max_rows <= 8 && T >= 4 * E && (E < T ? E : T) * ((N + 511) / 512) >= 512;
}
// bp_tq1_gemv.hip: TQ1, one token row per expert (max_rows == 1), bf16 activations, table-lookup GEMV
int launch_tq1_gemv(const GemmArgs& a, hipStream_t s, int waves);
// bp_tq1_gemv_fp4.hip: the same through the fp8 x fp4 matrix instruction (16-bit and int8 activations), and small
// batches: up to 8 token rows per expert, or up to 64 in launches of 8 when the experts average at most 4 rows;
// BP_ERR_UNSUPPORTED without a message when the call is outside its preconditions
BP_LAUNCHER(launch_tq1_gemv_fp4, (const GemmArgs& a, hipStream_t s), (a, s))
// bp_tq2_gemv_fp4.hip: TQ2, one to four token rows per expert, on the fp8 x fp4 matrix instruction with K split over the waves;
// BP_ERR_UNSUPPORTED without a message when the call is outside its preconditions
BP_LAUNCHER(launch_tq2_gemv_fp4, (const GemmArgs& a, hipStream_t s), (a, s))

namespace {

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) unsigned lds_u32;
typedef __attribute__((address_space(3))) unsigned short lds_u16;

// Weights and scales are read with raw buffer loads: a wave-uniform descriptor (base, byte range) in
// scalar registers, a 32-bit lane offset and a scalar step offset, so a load needs no vector address
// arithmetic, and a read past the range returns zeros instead of touching memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, int64_t bytes) {
  const int n = bytes > 0x7fffffff ? 0x7fffffff : (int)bytes;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, n, 0x00020000);
}
// A buffer load returns zero for a dword that straddles the end of its range, valid bytes included. Ranges over tensors
// that may start at any byte (the base is aligned down to a dword by the caller) therefore end with the dword that holds
// the tensor's last byte: up to 3 bytes behind the tensor are read with it - inside a dword of which the tensor owns a
// byte - and never used.
__device__ __forceinline__ int64_t whole_dwords(int64_t bytes) { return (bytes + 3) & ~(int64_t)3; }
__device__ __forceinline__ u32x4 buf_load16(__amdgpu_buffer_rsrc_t r, unsigned lane_off, unsigned wave_off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)lane_off, (int)wave_off, 0));
}

template <int ACT>
struct Acc;
template <>
struct Acc<BP_BF16> { typedef f32x4 type; };
template <>
struct Acc<BP_I8> { typedef i32x4 type; };

template <int SDT>
__device__ __forceinline__ float scale_at(const u32x4 (&raw)[2], int i) {  // i-th of the 8 scales held in raw
  if (SDT == BP_F32) return __uint_as_float(raw[i >> 2][i & 3]);
  const unsigned v = raw[i >> 3][(i >> 1) & 3];
  if (SDT == BP_F16) return f16_bits_to_f32((uint16_t)((i & 1) ? (v >> 16) : (v & 0xffffu)));
  return __uint_as_float((i & 1) ? (v & 0xffff0000u) : (v << 16));
}

// SwiGLU in a GEMM's epilogue (GemmArgs::glu_h).
__device__ __forceinline__ uint16_t swiglu_value(const GemmArgs& a, float gate, float up, float weight) {
  if (a.glu_v4) return swiglu_bits<true>(gate, up, a.glu_weights != nullptr, weight, a.glu_limit);
  return swiglu_bits<false>(gate, up, false, 1.f, 0.f);
}

}  // namespace
}  // namespace bp
