// TQ1 rows as TQ2 rows: five base-3 digits per byte become 2-bit codes, four to a byte.
//
// The TQ2 token-tile kernels turn 16 weights into matrix operands with three or four vector instructions; a TQ1 one takes a table
// read per five weights and strings the pieces together, again for every token tile that meets the weights, and that is
// what it spends its time on. A linear or a layer over a whole prompt meets each weight with many token tiles, so its weights are
// rewritten once, in the workspace, and the call continues as a TQ2 one: the same digits, the same scales.
// Bound by the memory: 1/5 + 1/4 byte per weight. What kept an earlier version from it was LDS: bytes and a table of one copy, 28
// conflicting reads for 64 codes. Now a lane loads its 13 or 14 bytes as dwords and has its own copy of the table (64 experts x 3 x
// 4096 x 2048 weights: 0.73 GB in 280 -> 140 us). The loads are on their way before the table is made.
#include "bp_mfma.h"

namespace bp {
namespace {

constexpr int RP_THREADS = 256;

// Pieces of 64 codes, `P` to a row (K = 64 P digits, Kp bytes each, at any byte address). The 13 or 14 bytes that hold a piece's digits
// through a table byte -> 10 bits, strung together and shifted by the digits that the first byte holds of the codes before. EACH: pieces
// that a thread makes.
template <int EACH>
__global__ __launch_bounds__(RP_THREADS) void k_tq1_to_tq2(uint4* __restrict__ out, const uint8_t* __restrict__ in, unsigned pieces, unsigned P, Divisor by_P,
                                                           unsigned Kp, int64_t bytes) {
  __shared__ __attribute__((aligned(16))) uint16_t table[256 * 64];  // entry v, copy of lane L at 64 v + L
  const unsigned mis = (unsigned)((uintptr_t)in & 3);
  // (whole dwords: the first and the last one hold a byte of the rows; zeros past them)
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(in - mis, whole_dwords(bytes + mis));
  const unsigned first_piece = blockIdx.x * (RP_THREADS * EACH) + threadIdx.x;
  u32x4 w[EACH];
  unsigned w4[EACH], off[EACH];
#pragma unroll
  for (int j = 0; j < EACH; ++j) {
    const unsigned i = first_piece + RP_THREADS * j, r = quotient(i < pieces ? i : 0u, by_P), p = (i < pieces ? i : 0u) - r * P;
    off[j] = mis + r * Kp + ((64 * p * 52429u) >> 18);  // (x / 5 for x < 81920)
    w[j] = buf_load16(rs, off[j] & ~3u, 0u);
    w4[j] = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(rs, (int)((off[j] & ~3u) + 16u), 0, 0);
  }
  {
    const unsigned v = threadIdx.x;  // (RP_THREADS = 256 entries)
    unsigned c = 0;
#pragma unroll
    for (int i = 0; i < 5; ++i) c |= (unsigned)(tq1_trit(v, i) + 1) << (2 * i);
    c |= c << 16;
    uint4* row = (uint4*)(table + 64 * v);
#pragma unroll
    for (unsigned i = 0; i < 8; ++i) row[(i + v) & 7] = make_uint4(c, c, c, c);  // (neighbouring threads on different banks)
  }
  __syncthreads();
  const uint16_t* mine = table + (threadIdx.x & 63);
#pragma unroll
  for (int j = 0; j < EACH; ++j) {
    const unsigned i = first_piece + RP_THREADS * j;
    if (i >= pieces) break;
    const unsigned p = i - quotient(i, by_P) * P, sh = 2 * (64 * p - 5 * ((64 * p * 52429u) >> 18));
    const unsigned d[4] = {__builtin_amdgcn_alignbyte(w[j].y, w[j].x, off[j]), __builtin_amdgcn_alignbyte(w[j].z, w[j].y, off[j]),
                           __builtin_amdgcn_alignbyte(w[j].w, w[j].z, off[j]), __builtin_amdgcn_alignbyte(w4[j], w[j].w, off[j])};
    unsigned c[14];
#pragma unroll
    for (int b = 0; b < 14; ++b) c[b] = mine[64 * ((d[b >> 2] >> (8 * (b & 3))) & 255u)];
    const unsigned s0 = c[0] | c[1] << 10 | c[2] << 20 | c[3] << 30;
    const unsigned s1 = c[3] >> 2 | c[4] << 8 | c[5] << 18 | c[6] << 28;
    const unsigned s2 = c[6] >> 4 | c[7] << 6 | c[8] << 16 | c[9] << 26;
    const unsigned s3 = c[9] >> 6 | c[10] << 4 | c[11] << 14 | c[12] << 24;
    const unsigned s4 = c[12] >> 8 | c[13] << 2;
    out[i] = make_uint4(__builtin_amdgcn_alignbit(s1, s0, sh), __builtin_amdgcn_alignbit(s2, s1, sh), __builtin_amdgcn_alignbit(s3, s2, sh),
                        __builtin_amdgcn_alignbit(s4, s3, sh));
  }
}

}  // namespace

// `rows` TQ1 rows of K digits as TQ2 rows at `out` (16-byte aligned). K a multiple of 64, up to 65536.
int launch_tq1_to_tq2(uint8_t* out, const uint8_t* in, int64_t rows, int64_t K, hipStream_t s) {
  const int64_t Kp = (K + 4) / 5, P = K / 64;
  if (K % 64 != 0 || K > 65536 || ((uintptr_t)out & 15) != 0) return BP_ERR_UNSUPPORTED;
  const int64_t most = ((int64_t)1 << 30) / Kp;  // rows of a launch (32-bit offsets)
  for (int64_t r = 0; r < rows; r += most) {
    const int64_t n = rows - r < most ? rows - r : most;
    // Eight pieces per thread, whose workgroups have more loads on their way and a table for more of them, where that leaves a CU
    // four workgroups; two where the rows are few (a two-term int8 linear of 37 x 4096 x 4096, which rewrites 2 x 128 workgroups of eight:
    // 37.6 -> 32.3 us).
    const int64_t pieces = n * P;
    const bool many = pieces >= (int64_t)1024 * RP_THREADS * 8;
    const auto kernel = many ? k_tq1_to_tq2<8> : k_tq1_to_tq2<2>;
    const int64_t per = RP_THREADS * (many ? 8 : 2);
    hipLaunchKernelGGL(kernel, dim3((unsigned)((pieces + per - 1) / per)), dim3(RP_THREADS), 0, s, (uint4*)(out + r * (K / 4)), in + r * Kp, (unsigned)pieces, (unsigned)P,
                       divisor((unsigned)P), (unsigned)Kp, n * Kp);
    if (const int rc = check_launch("tq1_to_tq2")) return rc;
  }
  return BP_OK;
}

}  // namespace bp
