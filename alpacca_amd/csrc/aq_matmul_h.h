// aq_matmul_h.h - what the kernels of the exact fp16 matmul share
// (aq_matmul_h.hip states the scheme): vector types, the B operand of the
// K-quants, the super-block scales and the stores.
#pragma once

#include "aq_internal.h"

namespace aq {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// The prepared X of a call, in the stream's workspace: fp16 piece planes of
// M x K halves (`plane` halves apart), the rows' exponents and the sub-block
// sums.
struct MmhX {
  const uint16_t *xp;
  int64_t plane;
  const int32_t *xe;
  const uint16_t *xs;
};

// ---- the B operand: sc * code as fp16 subnormals, from packed code bytes ---
// sc * code of a Q4_K weight is an integer m below 1024 (6-bit scale, 4-bit
// code), and the fp16 half whose bits are m is the subnormal m 2^-24: exact,
// and exactly multiplied by the matrix core (fp16 subnormal inputs are
// kept).  A byte permute puts two codes (low nibbles, or high nibbles
// shifted down) into the low bytes of two halves with zero high bytes, and
// one packed 16-bit integer multiply by (sc, sc) gives the two B values.
// The 2^24 goes with the super-block scale d.
__device__ __forceinline__ uint32_t fma_h2(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_bit_cast(
      uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(h2, a), __builtin_bit_cast(h2, b),
                                          __builtin_bit_cast(h2, c)));
}
__device__ __forceinline__ uint32_t mul_u16x2(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b));
}
// 8 values from two words of codes (one per byte, below 16), in byte order,
// times sc2 = (sc, sc)
__device__ __forceinline__ void sc_codes8(uint32_t c0, uint32_t c1, uint32_t sc2, uint32_t *o) {
  o[0] = mul_u16x2(__builtin_amdgcn_perm(0u, c0, 0x0C010C00u), sc2);
  o[1] = mul_u16x2(__builtin_amdgcn_perm(0u, c0, 0x0C030C02u), sc2);
  o[2] = mul_u16x2(__builtin_amdgcn_perm(0u, c1, 0x0C010C00u), sc2);
  o[3] = mul_u16x2(__builtin_amdgcn_perm(0u, c1, 0x0C030C02u), sc2);
}

// What the end of a K-quant super-block needs from its header h = (d | dmin,
// 12 scale bytes): d in the units of the products (2^24), -32 dmin (the sums
// S carry 2^(e-5)), and the mins of sub-blocks 4 (g & 1) .. +3 as the B
// operand of the min product.
__device__ __forceinline__ void kquant_block_scales(const uint4 &h, int g, float &d, float &dm32,
                                                    h4 &bm) {
  d = f16_bits_to_f32(h.x) * 16777216.f;
  dm32 = -32.f * f16_bits_to_f32(h.x >> 16);
  uint32_t sc0, mn0, sc1, mn1;
  kquant_scale_pair(h.y, h.z, h.w, 2 * (g & 1), sc0, mn0);
  kquant_scale_pair(h.y, h.z, h.w, 2 * (g & 1) + 1, sc1, mn1);
  const uint32_t mn4 = mn0 | (mn1 << 16);
  bm = __builtin_bit_cast(
      h4, uint2{fma_h2(__builtin_amdgcn_perm(0x64646464u, mn4, 0x05010400u), 0x3c003c00u,
                       0xe400e400u),
                fma_h2(__builtin_amdgcn_perm(0x64646464u, mn4, 0x05030402u), 0x3c003c00u,
                       0xe400e400u)});
}

// The SwiGLU of a (gate, up) pair, rounded operation by operation as the
// reference's NumPy expression (model.py:513) and the library's elementwise
// SwiGLU kernel are.
__device__ __forceinline__ float swiglu_pair(float g, float u) {
#pragma clang fp contract(off)
  return g / (1.0f + expf(-g)) * u;
}

// Store a lane's four outputs of one 16 x 16 tile: rows row0 .. row0 + 3 of
// column n (the lane's column l % 16 of the tile), Y = acc 2^-ex; rows past M
// and columns past N are not stored.  Ysw (a launch over interleaved gate/up
// rows without a split of K, N even): the pair of columns 2p, 2p+1 sits in
// neighbouring lanes of one row, and the M x N/2 output takes silu(gate) *
// up at column p instead.  Of each two rows rr, rr + 1 the even lane forms
// row rr's pair and the odd lane row rr + 1's, one exchanged value each (gate
// of rr + 1 one way, up of rr the other).
__device__ __forceinline__ void store_tile(const f32x4 &acc, const int *ex, int64_t row0,
                                           int64_t n, int64_t M, int64_t N, bool odd,
                                           float *__restrict__ Y, float *__restrict__ Ysw) {
  float v[4];
#pragma unroll
  for (int rr = 0; rr < 4; ++rr) v[rr] = __builtin_amdgcn_ldexpf(acc[rr], -ex[rr]);
  if (Ysw) {
#pragma unroll
    for (int rr = 0; rr < 4; rr += 2) {
      const float mine = odd ? v[rr] : v[rr + 1];  // what the partner lane needs
      const float got = __shfl_xor(mine, 1);
      const int r = odd ? rr + 1 : rr;
      const float out = odd ? swiglu_pair(got, v[rr + 1]) : swiglu_pair(v[rr], got);
      if (row0 + r < M && n < N) Ysw[(row0 + r) * (N >> 1) + (n >> 1)] = out;
    }
  } else {
#pragma unroll
    for (int rr = 0; rr < 4; ++rr)
      if (row0 + rr < M && n < N) Y[(row0 + rr) * N + n] = v[rr];
  }
}

// The tile kernel (aq_matmul_hd.hip) over prepared X: shape 0 = 128 x 256, 1 =
// 128 x 128, 2 = 64 x 128, 3 = 32 x 128, 4 = 16 x 128.
hipError_t launch_mm_hd(int shape, const aq_matrix *m, const MmhX &x, int64_t M, float *dst,
                        int splits, int per, float *ysw, hipStream_t s);

}  // namespace aq
