// aq_matmul_h.hip - batched Y = X W^T on fp16 matrix cores with the weights
// kept as exact integers: the X preparation, the kernel of up to 16 rows of X
// (Q4_K, Q5_K) and the choice of tiles.  aq_matmul_hd.hip holds the tile
// kernel and how each format enters the products.
//
// Replaces QuantMatrix.matmul_t (alpacca/qmatrix.py:184-211) at float32
// accuracy.  The reference dequantizes f32 row tiles (w = d*sc*code -
// dmin*mn) and multiplies them with SGEMM.  Here the decode stops before
// the fp32 scales: per 32-element sub-block the product sc*code of a Q4_K
// weight is an integer of at most 945 (6-bit scale, 4-bit code), exact in
// fp16 as the subnormal sc*code * 2^-24, and the 6-bit min mn is exact too.
// The super-block scales d and dmin (fp16 fields, exact in fp32) are applied
// once per 256 weights in fp32:
//
//   Y[m][n] = sum_b  d[n][b] * P[m][n][b] - dmin[n][b] * Q[m][n][b]
//   P = sum_{k in b} (sc*code)[n][k] * x[m][k]     (v_mfma_f32_16x16x32_f16)
//   Q = sum_{sb in b} mn[n][sb] * S[m][sb]         (v_mfma_f32_16x16x16f16)
//
// with S the sub-block sums of x.  x itself is cut into fp16 pieces after a
// per-row power-of-two scale 2^e (the row maximum lands in [2^14, 2^15), so
// nothing overflows fp16): NP = 2 pieces carry 22 bits of every element
// (hi = fp16(x 2^e), lo = fp16(x 2^e - hi)).  The products of 10-bit integers
// with fp16 pieces are exact in fp32, so the only roundings are the fp32 sums
// inside the matrix core, the scale products and the final 2^-e (exact).  The
// sub-block sums are formed in fp32 from the unscaled x and carried as two
// fp16 pieces at 2^(e-5).
#include <stdlib.h>

#include <algorithm>

#include "aq_matmul_h.h"
#include "aq_matmul_tiles.h"

namespace aq {
namespace {

constexpr int NP = 2;           // pieces of X
constexpr int kXsStages = 16;   // 64-column stages a whole-split X staging holds
constexpr int kLdA = 64 + 16;   // halves per staged row (160 B)

// ---- X preparation ---------------------------------------------------------
// One workgroup per row of X.  e[m] = 15 - E with max|x| = f 2^E, f in
// [0.5, 1) (0 for an all-zero row); piece planes xp[0] (hi) and xp[1] (lo),
// M x K halves each; xs[(m * (K / 256) + b) * 16 + j] = hi (j < 8) and lo
// (j >= 8) of the sum of sub-block j of super-block b, times 2^(e - 5).
// Sums are formed per 8 elements ((x0 + x1) + (x2 + x3)) + (...) and then
// over the four 8-element runs of a sub-block in pairs - one fixed order, the
// same for every M.  Thread t takes the 8-element runs j = 8 t + 2048 i.
// CH > 0 (K <= 2048 CH): all of the thread's runs are loaded at once and kept
// in registers, so the row is read in one memory round trip; CH = 0 reads
// the row twice (the maximum, then the pieces).
__device__ __forceinline__ float wave_max(float v) {
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
  return v;
}
__device__ __forceinline__ float run_max(const float (&v)[8]) {
  float mx = 0.f;
  bool nan = false;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    mx = fmaxf(mx, fabsf(v[i]));
    nan = nan || !(v[i] == v[i]);
  }
  // a NaN anywhere makes the row's scale NaN-safe below (isfinite test)
  return nan ? INFINITY : mx;
}
__device__ __forceinline__ void load_run(const float *p, float (&v)[8]) {
  const float4 a = *reinterpret_cast<const float4 *>(p);
  const float4 b = *reinterpret_cast<const float4 *>(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
// pieces and the sub-block sum of the run at column j
__device__ __forceinline__ void emit_run(const float (&v)[8], int64_t m, int64_t j, int64_t K,
                                         int e, int t, uint16_t *__restrict__ xp, int64_t plane,
                                         uint16_t *__restrict__ xs) {
  uint32_t hi[4], lo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float s0 = __builtin_amdgcn_ldexpf(v[2 * i], e);
    const float s1 = __builtin_amdgcn_ldexpf(v[2 * i + 1], e);
    const _Float16 h0 = (_Float16)s0, h1 = (_Float16)s1;
    const _Float16 l0 = (_Float16)(s0 - (float)h0), l1 = (_Float16)(s1 - (float)h1);
    hi[i] = (uint32_t)__builtin_bit_cast(uint16_t, h0) |
            ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16);
    lo[i] = (uint32_t)__builtin_bit_cast(uint16_t, l0) |
            ((uint32_t)__builtin_bit_cast(uint16_t, l1) << 16);
  }
  *reinterpret_cast<uint4 *>(xp + m * K + j) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
  *reinterpret_cast<uint4 *>(xp + plane + m * K + j) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
  if (xs) {
    // sub-block sum: this thread's 8 elements, then the four threads of
    // the sub-block (lanes 4q .. 4q+3 hold one sub-block: j = 8t)
    float s = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    const float s1 = __shfl_xor(s, 1);
    s = (t & 1) ? s1 + s : s + s1;  // (s0 + s1) in both lanes of the pair
    const float s2 = __shfl_xor(s, 2);
    s = (t & 2) ? s2 + s : s + s2;  // (s01 + s23) in all four lanes
    if ((t & 3) == 0) {
      const int64_t nsb = K / 256;
      const float ss = __builtin_amdgcn_ldexpf(s, e - 5);
      const _Float16 h = (_Float16)ss, l = (_Float16)(ss - (float)h);
      const int64_t sb = j / 32, b = sb / 8, r = sb % 8;
      xs[(m * nsb + b) * 16 + r] = __builtin_bit_cast(uint16_t, h);
      xs[(m * nsb + b) * 16 + 8 + r] = __builtin_bit_cast(uint16_t, l);
    }
  }
}
template <int CH>
__global__ void __launch_bounds__(256)
    k_x_h_pieces(const float *__restrict__ X, int64_t K, uint16_t *__restrict__ xp,
                 int64_t plane, int32_t *__restrict__ xe, uint16_t *__restrict__ xs) {
  __shared__ float red[4];
  const int64_t m = blockIdx.x;
  const float *xr = X + m * K;
  const int t = threadIdx.x;
  float v[CH > 0 ? CH : 1][8];
  float mx = 0.f;
  if constexpr (CH > 0) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int64_t j = 8 * (int64_t)t + 2048 * c;
      if (j < K) load_run(xr + j, v[c]);
    }
#pragma unroll
    for (int c = 0; c < CH; ++c)
      if (8 * (int64_t)t + 2048 * c < K) mx = fmaxf(mx, run_max(v[c]));
  } else {
    for (int64_t j = 8 * (int64_t)t; j < K; j += 2048) {
      load_run(xr + j, v[0]);
      mx = fmaxf(mx, run_max(v[0]));
    }
  }
  mx = wave_max(mx);
  if ((t & 63) == 0) red[t >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  // a non-finite row keeps e = 0: its infinities and NaNs reach the outputs
  const int e = (mx > 0.f && mx < INFINITY) ? 15 - __builtin_amdgcn_frexp_expf(mx) : 0;
  if (t == 0) xe[m] = e;
  if constexpr (CH > 0) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int64_t j = 8 * (int64_t)t + 2048 * c;
      if (j < K) emit_run(v[c], m, j, K, e, t, xp, plane, xs);
    }
  } else {
    for (int64_t j = 8 * (int64_t)t; j < K; j += 2048) {
      load_run(xr + j, v[0]);
      emit_run(v[0], m, j, K, e, t, xp, plane, xs);
    }
  }
}

// X pieces of an M x K matrix (K a multiple of 256)
void launch_x_h_pieces(const float *X, int64_t M, int64_t K, uint16_t *xp, int64_t plane,
                       int32_t *xe, uint16_t *xs, hipStream_t s) {
#define AQ_XH(ch) \
  hipLaunchKernelGGL((k_x_h_pieces<ch>), dim3((unsigned)M), dim3(256), 0, s, X, K, xp, plane, xe, xs)
  if (K <= 2048) AQ_XH(1);
  else if (K <= 4096) AQ_XH(2);
  else if (K <= 8192) AQ_XH(4);
  else if (K <= 16384) AQ_XH(8);
  else AQ_XH(0);
#undef AQ_XH
}

// byte-granular buffer loads (offsets past the resource read zeros)
__device__ __forceinline__ uint2 rsrc_u2(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}
// Lane group g holds chunk (0, 2, 1, 3)[g] of a 64-byte run as (v.x, v.y,
// v.z, v.w); afterwards (v.x, v.y) are bytes 8 g .. 8 g + 7 of the run's
// first 32 bytes and (v.z, v.w) those of its second 32: two 16-lane row
// swaps (odd lane groups' first words for even groups' second words).
// Every lane of the wave must be active.
__device__ __forceinline__ void pair_words(uint4 &v) {
  const auto a = __builtin_amdgcn_permlane16_swap(v.x, v.z, false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(v.y, v.w, false, false);
  v.x = a[0];
  v.z = a[1];
  v.y = b[0];
  v.w = b[1];
}
// the chunk of a 64-byte run that lane group g loads for pair_words
__device__ __forceinline__ uint32_t pair_chunk(int g) {
  return 16u * (uint32_t)(((g & 1) << 1) | (g >> 1));
}

__device__ __forceinline__ uint4 rsrc_u4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}

// ---- up to 16 rows of X (Q4_K, Q5_K) ---------------------------------------------
// One 16 x 128 tile: eight waves of one 16 x 16 tile each.  Lane l: A row l%16
// and B column l%16 with k = 8 (l/16) .. +7 of each 32-column sub-block (the
// same k set for A and B, so the matrix core sums over every k), D rows 4
// (l/16) .. +3 of column l%16.  Q4_K sub-block 2c is the low nibbles of
// qs[32c, 32c + 32), 2c+1 the high nibbles (quants.py:136-161): lane group g
// takes bytes 32c + 8g .. +7, i.e. elements 8g .. 8g+7 of both sub-blocks, in
// natural order.  One loop iteration is a super-block (four stages c = 0..3,
// each two sub-blocks), so every index into the register sets is a
// compile-time one.  Weights go from memory straight into registers.
//
// The workgroup makes its X pieces itself from the fp32 rows X, for the whole
// split (at most kXsStages stages) before the loop, which then has neither X
// loads nor barriers.  The power-of-two scale e per row is over the split's
// own columns (the split's maximum in [2^14, 2^15)), and the partial is
// written as acc 2^-e: no preparation launch.  The pieces of an element are
// its pieces under the whole-row scale shifted by a power of two (exact
// unless the element falls among fp16 subnormals, where the split's larger
// scale keeps more of its bits), and the sub-block sums are formed in the
// preparation kernel's order, so the outputs are those of the tile kernel.
// The sub-block sums and the exponents live in the padding columns 64..79 of
// the staged rows, which the matrix-core reads never touch: super-block bb's
// sums at As[4 bb][0][r][64..79] (hi 0..7, lo 8..15), row r's exponent at
// As[0][1][r][64..65].
//
// Q5 (Q5_K): the same kernel with a fifth code bit from the qh plane: bit 2c
// (low nibbles) and 2c+1 (high nibbles) of qh byte l for element l of
// sub-blocks 2c, 2c+1 (quants.py:164-193), so a lane's bits for a whole
// super-block are qh bytes 8g .. 8g+7, loaded with the header.  sc*code is
// then at most 63 * 31 = 1953: below 2048, the fp16 half whose bits are that
// integer m is still m 2^-24 exactly (a normal half from 1024 on).
//
// M = 8 / 16 on 14336 x 4096: 16.7 / 17.3 us a call in 4 splits; the tile
// kernel behind its preparation launch 16.9 / 17.8, and 0.8 - 2 us more on
// smaller matrices.
template <bool Q5>
__global__ void __launch_bounds__(512)
    k_mm_h_16(const uint8_t *qs, const uint8_t *hd, uint32_t qs_stride, uint32_t hd_stride,
              int64_t N, int nb_row, const float *__restrict__ X, int64_t M,
              float *__restrict__ Y, int sb_per_split, const uint8_t *qhp, uint32_t qh_stride,
              float *__restrict__ Ysw) {
  constexpr int XS = kXsStages, BN = 128;
  __shared__ __attribute__((aligned(16))) uint16_t As[XS][NP][16 * kLdA];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const int64_t n = (int64_t)blockIdx.x * BN + 16 * wave + c16;
  const int64_t K = (int64_t)nb_row * 256;
  const int b_begin = (int)blockIdx.z * sb_per_split;
  const int b_end = std::min(b_begin + sb_per_split, nb_row);
  Y += (int64_t)blockIdx.z * M * N;

  // weights: one buffer resource per plane, over the rows that exist (the
  // launcher keeps them below 2^31 bytes)
  const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t *>(qs), 0, (int)(N * nb_row * qs_stride), kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t *>(hd), 0, (int)(N * nb_row * hd_stride), kRsrcWord3);
  const __amdgpu_buffer_rsrc_t r5 = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t *>(qhp), 0, Q5 ? (int)(N * nb_row * qh_stride) : 0, kRsrcWord3);
  constexpr uint32_t kNone = 0x7fffffffu;  // an offset past every resource
  // byte offsets of this lane's row (block 0; + the 16-byte chunk this lane
  // group loads of a stage pair: w_load)
  const uint32_t rowq = n < N ? (uint32_t)(n * nb_row * qs_stride) + pair_chunk(g) : kNone;
  const uint32_t rowh = n < N ? (uint32_t)(n * nb_row * hd_stride) : kNone;
  const uint32_t row5 = Q5 && n < N ? (uint32_t)(n * nb_row * qh_stride) + 8 * g : kNone;

  const int n_st = 4 * (b_end - b_begin);
  // code bytes of split stages 2 pr and 2 pr + 1 (zeros past the split): the
  // pair's 64 bytes of a row are four 16-byte chunks, lane group g loads
  // chunk (0, 2, 1, 3)[g], and two 16-lane row swaps (pair_words) leave each
  // lane group its 8 bytes of either stage (bytes 8 g .. 8 g + 7 of each
  // stage's 32) in place of two 8-byte loads per pair
  auto w_load = [&](int pr) {
    const int stg = 2 * pr, b = b_begin + stg / 4, c = stg % 4;
    return rsrc_u4(rq, stg < n_st && rowq != kNone ? rowq + (uint32_t)b * qs_stride + 32 * c
                                                   : kNone);
  };
  auto h_load = [&](int b, uint4 &h, uint2 &q5) {  // header (and Q5's qh bytes)
    h = rsrc_u4(rh, b < b_end && rowh != kNone ? rowh + (uint32_t)b * hd_stride : kNone);
    if constexpr (Q5)
      q5 = rsrc_u2(r5, b < b_end && row5 != kNone ? row5 + (uint32_t)b * qh_stride : kNone);
  };

  // The code bytes of stages s + 3, s + 4 are issued as soon as stages s - 1,
  // s have turned theirs into B operands (two register sets of a stage pair
  // each), the next super-block's header at this one's first stage.
  uint4 hdr, hdn, wq[2];
  uint2 q5r, q5n;
  h_load(b_begin, hdr, q5r);
  wq[0] = w_load(0);
  wq[1] = w_load(1);
  {
    // thread t: row t / 16 % 16, columns 4 (t % 16) .. +3 of stages 2 i + t / 256
    const int r = (tid >> 4) & 15, q = tid & 15, hs = tid >> 8;
    const __amdgpu_buffer_rsrc_t rf = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(X), 0, (int)(M * K * 4), kRsrcWord3);
    constexpr int XT = XS / 2;  // stages per thread
    f32x4 xv[XT];
#pragma unroll
    for (int i = 0; i < XT; ++i) {
      const int st = 2 * i + hs;
      xv[i] = __builtin_bit_cast(
          f32x4, rsrc_u4(rf, st < n_st && r < M
                                 ? (uint32_t)(4 * (r * K + (int64_t)b_begin * 256 + 64 * st + 4 * q))
                                 : kNone));
    }
    float mx = 0.f;
    bool nan = false;
#pragma unroll
    for (int i = 0; i < XT; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        mx = fmaxf(mx, fabsf(xv[i][k]));
        nan = nan || !(xv[i][k] == xv[i][k]);
      }
    if (nan) mx = INFINITY;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    // the row's two halves meet in a padding slot of stage 1's lo piece
    float *slot = reinterpret_cast<float *>(&As[1][1][r * kLdA + 64]);
    if (q == 0) slot[hs] = mx;
    __syncthreads();
    mx = fmaxf(slot[0], slot[1]);
    // a non-finite row keeps e = 0: its infinities and NaNs reach the outputs
    const int e = (mx > 0.f && mx < INFINITY) ? 15 - __builtin_amdgcn_frexp_expf(mx) : 0;
    if (q == 0 && hs == 0) *reinterpret_cast<int32_t *>(&As[0][1][r * kLdA + 64]) = e;
#pragma unroll
    for (int i = 0; i < XT; ++i) {  // (stages past the split: zeros, never read)
      const int st = 2 * i + hs;
      uint32_t hi[2], lo[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const float s0 = __builtin_amdgcn_ldexpf(xv[i][2 * k], e);
        const float s1 = __builtin_amdgcn_ldexpf(xv[i][2 * k + 1], e);
        const _Float16 h0 = (_Float16)s0, h1 = (_Float16)s1;
        const _Float16 l0 = (_Float16)(s0 - (float)h0), l1 = (_Float16)(s1 - (float)h1);
        hi[k] = (uint32_t)__builtin_bit_cast(uint16_t, h0) |
                ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16);
        lo[k] = (uint32_t)__builtin_bit_cast(uint16_t, l0) |
                ((uint32_t)__builtin_bit_cast(uint16_t, l1) << 16);
      }
      *reinterpret_cast<uint2 *>(&As[st][0][r * kLdA + 4 * q]) = make_uint2(hi[0], hi[1]);
      *reinterpret_cast<uint2 *>(&As[st][1][r * kLdA + 4 * q]) = make_uint2(lo[0], lo[1]);
      // sub-block sum in the preparation kernel's order: per 8-element run
      // ((x0 + x1) + (x2 + x3)) + ((x4 + x5) + (x6 + x7)) (two threads), then
      // the four runs in pairs (threads q ^ 2, then q ^ 4)
      float a = (xv[i][0] + xv[i][1]) + (xv[i][2] + xv[i][3]);
      a = a + __shfl_xor(a, 1);
      a = a + __shfl_xor(a, 2);
      a = a + __shfl_xor(a, 4);
      if ((q & 7) == 0) {
        const float ss = __builtin_amdgcn_ldexpf(a, e - 5);
        const _Float16 h = (_Float16)ss, l = (_Float16)(ss - (float)h);
        const int r8 = 2 * (st % 4) + (q >> 3);
        As[st & ~3][0][r * kLdA + 64 + r8] = __builtin_bit_cast(uint16_t, h);
        As[st & ~3][0][r * kLdA + 72 + r8] = __builtin_bit_cast(uint16_t, l);
      }
    }
  }
  __syncthreads();

  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  // one super-block; hdr holds its header, hdn receives the next one (the
  // loop runs two super-blocks per iteration with the two sets swapped, so
  // no copy ties a pending load to the loop edge)
  auto superblock = [&](int b, uint4 &hdr, uint4 &hdn, uint2 &q5r, uint2 &q5n) {
    h_load(b + 1, hdn, q5n);
    const uint2 xsv =
        *reinterpret_cast<const uint2 *>(&As[4 * (b - b_begin)][0][c16 * kLdA + 64 + 4 * g]);
    f32x4 P;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int stg = 4 * (b - b_begin) + c;
      // B operands of the two sub-blocks 2c, 2c+1
      uint32_t bop[2][4];
      if (c % 2 == 0) pair_words(wq[c >> 1]);
      uint32_t sc, mn;
      kquant_scale_pair(hdr.y, hdr.z, hdr.w, c, sc, mn);
      const uint4 &wp = wq[c >> 1];
      const uint2 w = c % 2 == 0 ? uint2{wp.x, wp.y} : uint2{wp.z, wp.w};
      const uint32_t sl = sc & 0xFFu, sh = sc >> 8;
      uint32_t l0 = w.x & 0x0F0F0F0Fu, l1 = w.y & 0x0F0F0F0Fu;
      uint32_t h0 = (w.x >> 4) & 0x0F0F0F0Fu, h1 = (w.y >> 4) & 0x0F0F0F0Fu;
      if constexpr (Q5) {  // the fifth bit: 16 when set
        l0 |= ((q5r.x >> (2 * c)) & 0x01010101u) << 4;
        l1 |= ((q5r.y >> (2 * c)) & 0x01010101u) << 4;
        h0 |= ((q5r.x >> (2 * c + 1)) & 0x01010101u) << 4;
        h1 |= ((q5r.y >> (2 * c + 1)) & 0x01010101u) << 4;
      }
      sc_codes8(l0, l1, sl | (sl << 16), bop[0]);
      sc_codes8(h0, h1, sh | (sh << 16), bop[1]);
      if (c % 2 == 1) wq[c >> 1] = w_load((stg + 3) / 2);  // stages stg + 3, stg + 4
      h8 a[2][NP];  // the stage's fragments, read before its first product
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int p = 0; p < NP; ++p)
          a[e][p] = *reinterpret_cast<const h8 *>(&As[stg][p][c16 * kLdA + 32 * e + 8 * g]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int p = 0; p < NP; ++p)
          P = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              a[e][p], __builtin_bit_cast(h8, u32x4{bop[e][0], bop[e][1], bop[e][2], bop[e][3]}),
              (c == 0 && e == 0 && p == 0) ? f32x4{0.f, 0.f, 0.f, 0.f} : P, 0, 0, 0);
    }
    // super-block end: the min term and the fp32 scales
    float d, dm32;
    h4 bm;
    kquant_block_scales(hdr, g, d, dm32, bm);
    const f32x4 q = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h4, xsv), bm,
                                                          f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      acc[rr] = fmaf(d, P[rr], acc[rr]);
      acc[rr] = fmaf(dm32, q[rr], acc[rr]);
    }
  };
  int b = b_begin;
  for (; b + 1 < b_end; b += 2) {
    superblock(b, hdr, hdn, q5r, q5n);
    superblock(b + 1, hdn, hdr, q5n, q5r);
  }
  if (b < b_end) superblock(b, hdr, hdn, q5r, q5n);
  int ex[4];
#pragma unroll
  for (int rr = 0; rr < 4; ++rr)
    ex[rr] = *reinterpret_cast<const int32_t *>(&As[0][1][(4 * g + rr) * kLdA + 64]);
  store_tile(acc, ex, 4 * g, n, M, N, c16 & 1, Y, Ysw);
}

// ---- the choice of tiles ----------------------------------------------------------
// Shapes of the tile kernel; kinds: Q4_K / Q5_K, Q6_K, the per-32 formats.  The
// constants are a fit to 4,028 timed calls (Q4_K, Q6_K, Q8_0, Q5_0; N 512 -
// 14336, K 2048 - 14336, M 5 - 1500, every shape with up to eight splits): the
// call they pick is 0.5 % slower than the fastest on average, 10 % at worst.
// Q5_K goes by Q4_K's: 128 x 256 is its fastest too where they choose it (14336 x
// 4096 at M = 512 131 us against 150 with 128 x 128, M = 2048 514 / 549), its worst
// picks 12 - 13 % (M = 768 251 / 225, unsplit M = 128 59.9 / 52.8).
constexpr TileCost kTiles[] = {
    {128, 256, {1.86f, 0.f, 0.f}, {0.f, 0.f, 0.f}, 3.6f},
    {128, 128, {1.15f, 1.55f, 1.33f}, {0.f, 0.f, 0.f}, 1.2f},
    {64, 128, {0.74f, 0.97f, 0.80f}, {1.14f, 0.f, 1.56f}, 0.9f},
    {32, 128, {0.57f, 0.58f, 0.565f}, {0.69f, 0.92f, 1.59f}, 0.7f},
    {16, 128, {0.496f, 0.595f, 0.494f}, {0.513f, 0.92f, 0.75f}, 0.f},
};
constexpr int kTileShapes = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr TileModel kModel = {kTiles, kTileShapes, 0.89f, 1.f / 4.6f};
}  // namespace

// Workspace bytes of the X pieces of an M x K matrix (the piece planes, the
// exponents and the sub-block sums), each 256-B aligned.
size_t mm_h_x_bytes(int64_t M, int64_t K) {
  auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
  return al((size_t)NP * M * K * 2) + al((size_t)M * 4) + al((size_t)M * (K / 256) * 32);
}

bool mm_h_supported(const aq_matrix *m) {
  // 32-bit buffer offsets over each plane
  const double nblk = (double)m->rows * m->nb_row;
  if (m->nb_pitch != m->nb_row) return false;
  if (m->dtype == AQ_Q4_K || m->dtype == AQ_Q5_K) {
    const int np = m->dtype == AQ_Q4_K ? 2 : 3;
    for (int k = 0; k < np; ++k)
      if (nblk * (double)m->planes.stride[k] >= 2147483648.0) return false;
    return true;
  }
  // per-32 block formats: the dense planes of the SPLIT layout (codes, then
  // qh for Q5_0/Q5_1, then d or d|m), whole 256-column groups
  const int dt = m->dtype;
  if (dt == AQ_Q8_0 || dt == AQ_Q4_0 || dt == AQ_Q4_1 || dt == AQ_Q5_0 || dt == AQ_Q5_1) {
    const bool high = dt == AQ_Q5_0 || dt == AQ_Q5_1, mn = dt == AQ_Q4_1 || dt == AQ_Q5_1;
    const int64_t qsb = dt == AQ_Q8_0 ? 32 : 16;
    return m->layout == AQ_LAYOUT_SPLIT && m->cols % 256 == 0 && m->planes.stride[0] == qsb &&
           (!high || m->planes.stride[1] == 4) && m->planes.stride[high ? 2 : 1] == (mn ? 4 : 2) &&
           nblk * (double)qsb < 2147483648.0;
  }
  // Q6_K: the dense planes of the SPLIT layout (ql, qh, scales, d)
  return m->dtype == AQ_Q6_K && m->layout == AQ_LAYOUT_SPLIT && m->planes.stride[0] == 128 &&
         m->planes.stride[1] == 64 && m->planes.stride[2] == 16 && m->planes.stride[3] == 2 &&
         nblk * 128.0 < 2147483648.0;
}

// Y (M x rows) = X W^T with X in two fp16 pieces.  m_invariant: no split
// of the 256-column groups, so every output is the same sequence of
// operations for any M (the batched prefill step gives the same bits in any
// chunk size); otherwise the groups are split over workgroups where that is
// estimated faster, and the partials added in split order.
hipError_t launch_matmul_h(const aq_matrix *m, const float *X, int64_t M, float *Y,
                           bool m_invariant, hipStream_t s, float *ysw, bool *fused_sw) {
  if (M == 0 || m->rows == 0) return hipSuccess;
  if (!mm_h_supported(m)) return hipErrorInvalidValue;
  // the X pieces through 32-bit offsets: callers split larger batches
  if ((double)M * m->cols * 2 * NP >= 2147483648.0) return hipErrorInvalidValue;
  const int64_t K = m->cols, N = m->rows;
  const int units = (int)(K / 256);
  const int dt = m->dtype;
  const bool q5 = dt == AQ_Q5_K, kq = dt == AQ_Q4_K || q5, q6 = dt == AQ_Q6_K;
  const int cus = device_info(m->device).cus;
  // Up to 16 rows at AQ_PREC_AUTO the K-quants take the 16-row kernel, K
  // split over up to two workgroups per CU (M = 16 on 14336 x 4096: 4 splits
  // 24.9 us, 8 splits 27.2 us), where the split's X fits the staging.
  // AQ_MATMUL_X_PREP (tests compare the two) takes the tile kernel at the
  // same split instead.
  bool rows16 = false;
  int shape = 4, splits = 1;
  if (kq && !m_invariant && M <= 16) {
    const int64_t tiles = (N + 127) / 128;
    if (tiles < 2 * cus) splits = (int)std::min<int64_t>(2 * cus / tiles, 16);
    splits = std::min(splits, std::max(1, units / 2));
    rows16 = 4 * ((units + splits - 1) / splits) <= kXsStages;
  }
  const bool prep = rows16 && getenv("AQ_MATMUL_X_PREP");
  const int kind = kq ? 0 : q6 ? 1 : 2;
  if (!rows16)
    choose_tile(kModel, kind, M, N, units, 4, 2, cus, m_invariant ? 1 : 16, shape, splits);
  rows16 = rows16 && !prep;
  // AQ_MATMUL_TILE (tests): the shape itself, where the kind has it
  if (const char *env = rows16 ? nullptr : getenv("AQ_MATMUL_TILE")) {
    const int v = atoi(env);
    if (v >= 0 && v < kTileShapes && kTiles[v].one[kind] > 0.f) shape = v;
  }
  const int per = (units + splits - 1) / splits;
  splits = (units + per - 1) / per;

  auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
  const size_t xb = rows16 ? 0 : mm_h_x_bytes(M, K);
  const size_t part = splits > 1 ? (size_t)splits * M * N * 4 : 0;
  uint8_t *ws = nullptr;
  if (xb + part) {
    ws = static_cast<uint8_t *>(workspace(m->device, s, xb + part));
    if (!ws) return hipErrorOutOfMemory;
  }
  float *dst = splits > 1 ? reinterpret_cast<float *>(ws + xb) : Y;
  // the SwiGLU pairs in the store: launches without a split
  float *sw = ysw && splits == 1 && N % 2 == 0 ? ysw : nullptr;
  if (fused_sw) *fused_sw = sw != nullptr;
  hipError_t e;
  if (rows16) {
    // planes: Q4_K qs, header; Q5_K qs, qh, header
    const Planes &P = m->planes;
    const int h = q5 ? 2 : 1;
    const dim3 grid((unsigned)((N + 127) / 128), 1, (unsigned)splits);
    hipLaunchKernelGGL(q5 ? k_mm_h_16<true> : k_mm_h_16<false>, grid, dim3(512), 0, s, P.p[0],
                       P.p[h], (uint32_t)P.stride[0], (uint32_t)P.stride[h], N, units, X, M, dst,
                       per, P.p[1], (uint32_t)P.stride[1], sw);
    e = hipGetLastError();
  } else {
    uint16_t *xp = reinterpret_cast<uint16_t *>(ws);
    int32_t *xe = reinterpret_cast<int32_t *>(ws + al((size_t)NP * M * K * 2));
    uint16_t *xs = reinterpret_cast<uint16_t *>(ws + al((size_t)NP * M * K * 2) + al((size_t)M * 4));
    const bool sums = kq || dt == AQ_Q4_1 || dt == AQ_Q5_1;
    launch_x_h_pieces(X, M, K, xp, M * K, xe, sums ? xs : nullptr, s);
    e = launch_mm_hd(shape, m, MmhX{xp, M * K, xe, xs}, M, dst, splits, per, sw, s);
  }
  if (e != hipSuccess || splits == 1) return e;
  return sum_splits(dst, splits, M * N, Y, s);
}

}  // namespace aq
