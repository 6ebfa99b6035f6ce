// TQ1 rows as TQ2 rows: five base-3 digits per byte become 2-bit codes, four to a byte.
//
// The TQ2 token-tile kernels turn 16 weights into matrix operands with four vector instructions; a TQ1 one takes a table
// read per five weights and strings the pieces together, again for every token tile that meets the weights, and that is
// what it spends its time on. A linear over a whole prompt meets each weight with many token tiles, so its weights are
// rewritten once, in the workspace, and the call continues as a TQ2 one: the same digits, the same scales.
// Bound by the memory: 1/5 + 1/4 byte per weight.
#include "bp_common.h"

namespace bp {
namespace {

constexpr int RP_THREADS = 256;
constexpr int RP_BYTES = 32 * 1024;  // packed bytes of the rows that a workgroup takes, staged in LDS

// Rows of K digits (K a multiple of 64), Kp = ceil(K / 5) bytes each, at any byte address; out rows of K / 4 bytes, 16-byte aligned.
// A thread makes 16 bytes = 64 codes at a time: the 13 or 14 bytes that hold them through a table byte -> 10 bits, strung
// together and shifted by the digits that the first byte holds of the codes before.
__global__ __launch_bounds__(RP_THREADS) void k_tq1_to_tq2(uint4* __restrict__ out, const uint8_t* __restrict__ in, int64_t rows, int K, int Kp,
                                                           int rows_per_wg) {
  __shared__ unsigned table[256];
  __shared__ __attribute__((aligned(16))) unsigned staged[RP_BYTES / 4 + 8];
  {
    const unsigned v = threadIdx.x;  // (RP_THREADS = 256 entries)
    unsigned c = 0;
#pragma unroll
    for (int i = 0; i < 5; ++i) c |= (unsigned)(tq1_trit(v, i) + 1) << (2 * i);
    table[v] = c;
  }
  const int64_t row0 = (int64_t)blockIdx.x * rows_per_wg;
  const int n = (int)(rows - row0 < rows_per_wg ? rows - row0 : rows_per_wg);
  const uint8_t* src = in + row0 * Kp;
  // (whole dwords: the first and the last one hold a byte of the rows)
  const int mis = (int)((uintptr_t)src & 3);
  const unsigned* src4 = (const unsigned*)(src - mis);
  const int words = (mis + n * Kp + 3) / 4;
  for (int i = threadIdx.x; i < words; i += RP_THREADS) staged[i] = src4[i];
  __syncthreads();
  const uint8_t* bytes = (const uint8_t*)staged + mis;
  const int pieces = K / 64;
  for (int i = threadIdx.x; i < n * pieces; i += RP_THREADS) {
    const int r = i / pieces, p = i - r * pieces;
    const int first = (64 * p) / 5, sh = 2 * (64 * p - 5 * first);
    const uint8_t* b = bytes + r * Kp + first;  // (up to 14 bytes: past the row's last one only where no code comes from them)
    unsigned c[14];
#pragma unroll
    for (int j = 0; j < 14; ++j) c[j] = table[b[j]];
    const unsigned w0 = c[0] | c[1] << 10 | c[2] << 20 | c[3] << 30;
    const unsigned w1 = c[3] >> 2 | c[4] << 8 | c[5] << 18 | c[6] << 28;
    const unsigned w2 = c[6] >> 4 | c[7] << 6 | c[8] << 16 | c[9] << 26;
    const unsigned w3 = c[9] >> 6 | c[10] << 4 | c[11] << 14 | c[12] << 24;
    const unsigned w4 = c[12] >> 8 | c[13] << 2;
    out[(row0 + r) * pieces + p] = make_uint4(__builtin_amdgcn_alignbit(w1, w0, sh), __builtin_amdgcn_alignbit(w2, w1, sh),
                                              __builtin_amdgcn_alignbit(w3, w2, sh), __builtin_amdgcn_alignbit(w4, w3, sh));
  }
}

}  // namespace

// `rows` TQ1 rows of K digits as TQ2 rows at `out` (16-byte aligned). K a multiple of 64, up to 5 * RP_BYTES.
int launch_tq1_to_tq2(uint8_t* out, const uint8_t* in, int64_t rows, int64_t K, hipStream_t s) {
  const int64_t Kp = (K + 4) / 5;
  if (K % 64 != 0 || Kp > RP_BYTES || ((uintptr_t)out & 15) != 0) return BP_ERR_UNSUPPORTED;
  int64_t per = RP_BYTES / Kp;
  const int64_t spread = (rows + 1023) / 1024;  // (at least four workgroups per CU where there are rows enough)
  per = per < spread ? per : spread;
  if ((rows + per - 1) / per > 0x7fffffff) return BP_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(k_tq1_to_tq2, dim3((unsigned)((rows + per - 1) / per)), dim3(RP_THREADS), 0, s, (uint4*)out, in, rows, (int)K, (int)Kp, (int)per);
  return check_launch("tq1_to_tq2");
}

}  // namespace bp
