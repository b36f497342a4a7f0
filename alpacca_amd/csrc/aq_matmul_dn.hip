// aq_matmul_dn.hip - batched Y = X W^T of dense F16 / BF16 / F32 weights on
// 16-bit matrix cores at float32 accuracy.
//
// Replaces the dense products of the reference (alpacca/model.py:276-281
// keeps such weights as float32 arrays, alpacca/tensor.py:91-97 multiplies
// them with SGEMM).  Every operand enters the products exactly or in pieces:
//   F16   W as stored (11 bits); x in two fp16 pieces after a per-row
//         power-of-two scale, the second with 2^12 more and an accumulator of
//         its own (22 bits from 2^-28 of the row's largest on): 2 products;
//   BF16  W as stored (8 bits); x in three bf16 pieces (24 bits): 3;
//   F32   W and x in three bf16 pieces each: the 6 piece products of index
//         sum at most 2 (what is dropped is below 2^-25 of a product).
// Products are exact in fp32, the small ones of a sub-block are summed first,
// and one accumulator (F16: one per piece) runs over K.  Behind the stores,
// what the pieces of a row lack is added (F16: up to eight values below that
// range), or the row's outputs are formed again from plain fp32 products (more
// of them; else: rows with an infinity, a NaN or a value below 2^-110).  Weights
// with an infinity or a NaN, and F32 weights below 2^-110, stay on the fp32
// matrix cores (aq_matmul.hip): a piece of x that is zero times an infinity
// would be a NaN, and three pieces hold 24 bits from 2^-110 on.
//
// One workgroup: BM rows of X, BN rows of W, stages of 64 columns of both in
// LDS by DMA a stage ahead (rows of 128 bytes, 256 for F32, the 16-byte chunks
// swizzled by row).  An output is the same sequence of operations in every
// tile shape.
//
// 4096 x 4096 at M = 512 on the fp32 matrix cores (16x16x4 products at 1/16 of
// the rate) and here: F16 248 -> 50 us a call, BF16 247 -> 63, F32 244 -> 114,
// error against float64 8.1e-7 -> 2.9e-7, 6.9e-7 and 7.1e-7.  The fp32 kernel's
// 128-row tiles also left small batches on few workgroups: 5414 x 12800 at M =
// 2 F16 1198 -> 38 us (the weights alone: 29), F32 1311 -> 71.  What bounds it:
// a stage's products and fragment reads (0.5 us of matrix cores in the 1.0 -
// 1.4 us of a 128 x 128 stage), two waves per SIMD.  F16 rows with values below
// the pieces' range, 4096 x 14336 at M = 512, 141 us for normal ones: SwiGLU
// outputs (0.7 % of rows have one) 143, every row with a few 203, every row
// formed again 1264 (the fp32 kernel: 919).
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "aq_internal.h"
#include "aq_matmul_dma.h"
#include "aq_matmul_tiles.h"

namespace aq {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

enum Kind { kF16 = 0, kBF16 = 1, kF32 = 2 };
constexpr int pieces_of(int kind) { return kind == kF16 ? 2 : 3; }

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, b2));
}
__device__ __forceinline__ uint32_t pack_f16(float a, float b) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)a) |
         ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)b) << 16);
}
// x less its first piece; 0 for an infinity (NaN stays in the first piece)
__device__ __forceinline__ float rest_of(float x, float piece) {
  return __builtin_isinf(x) ? 0.f : x - piece;
}
// x, or for a finite x that would round to a bf16 infinity its bf16 below
__device__ __forceinline__ float bf16_finite(float x) {
  return fabsf(x) >= 3.38e38f && !__builtin_isinf(x)
             ? __uint_as_float(__float_as_uint(x) & 0xFFFF0000u) : x;
}

// ---- X preparation -----------------------------------------------------------
// One workgroup per row: NX piece planes of M x Kp 16-bit values (zeros from
// column K to Kp), `plane` values apart, and xe[m] = 16 e + mark.
//   F16: e = 15 - E for the largest finite |x| = f 2^E, f in [0.5, 1) (0 without
//     one); hi = fp16(x 2^e), lo = fp16((x 2^e - hi) 2^12).  The products of hi
//     and of lo have an accumulator each, so lo's own 2^12 costs nothing and
//     every x from 2^-28 of the largest on keeps 22 bits (hi is normal from
//     2^-14 on, and lo's last bit there is 2^-36).  What the pieces lack of
//     smaller values other than zero is listed, xl[m] (a row of SwiGLU outputs
//     14,336 wide has one in 0.7 % of cases): mark = entries, or kAgain for more
//     than kList of them.
//   Else the pieces are bf16, e is 0 and the mark of rows with an infinity, a NaN
//     or a value below kPieceMin other than zero kAgain.
// Marked rows are corrected, or formed again, after the stores.

// The smallest magnitude whose 24 bits three bf16 pieces hold: its last bit is
// bf16's smallest subnormal, 2^-133 (the matrix cores keep subnormal inputs)
constexpr float kPieceMin = 0x1p-110f;
constexpr int kLoExp = 12, kList = 8, kAgain = 15;
struct Lacking {
  int32_t k;
  float x;
};
// the exponent of a row from its largest finite |x|
__device__ __forceinline__ int row_exp(float mx) {
  return mx > 0.f ? 15 - __builtin_amdgcn_frexp_expf(mx) : 0;
}
// largest finite |x| and smallest |x| other than zero so far
__device__ __forceinline__ void row_range(float x, float &mx, float &mn) {
  mx = fmaxf(mx, __builtin_isfinite(x) ? fabsf(x) : 0.f);
  mn = fminf(mn, x == 0.f ? INFINITY : fabsf(x));
}
// what the two fp16 pieces of x lack, 0 unless x is below their range
__device__ __forceinline__ float lacking(float x, int e) {
  const float y = __builtin_amdgcn_ldexpf(x, e);
  if (x == 0.f || !(fabsf(y) < 0x1p-14f)) return 0.f;
  const float hi = (float)(_Float16)y;
  const float lo = (float)(_Float16)((y - hi) * (1 << kLoExp));
  // (exact: the pieces hold 22 bits next to x's own)
  return x - __builtin_amdgcn_ldexpf(fmaf(lo, 1.f / (1 << kLoExp), hi), -e);
}
// whether the three bf16 pieces of x cannot stand for it
__device__ __forceinline__ bool no_pieces(float x) {
  return !__builtin_isfinite(x) || (x != 0.f && fabsf(x) < kPieceMin);
}
// the pieces of four values (F16: scaled by 2^e), packed
template <int KIND>
__device__ __forceinline__ void cut4(float (&a)[4], uint32_t (&o)[pieces_of(KIND)][2]) {
#pragma unroll
  for (int p = 0; p < pieces_of(KIND); ++p)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float &x = a[2 * i], &y = a[2 * i + 1];
      if constexpr (KIND == kF16) {
        o[p][i] = pack_f16(x, y);
        x = rest_of(x, (float)(_Float16)x) * (float)(1 << kLoExp);
        y = rest_of(y, (float)(_Float16)y) * (float)(1 << kLoExp);
      } else {
        o[p][i] = pack_bf16(bf16_finite(x), bf16_finite(y));
        x = rest_of(x, __uint_as_float(o[p][i] << 16));
        y = rest_of(y, __uint_as_float(o[p][i] & 0xFFFF0000u));
      }
    }
}
template <int KIND>
__global__ void __launch_bounds__(256)
    k_x_pieces(const float *__restrict__ X, int64_t K, int64_t Kp, uint16_t *__restrict__ xp,
               int64_t plane, int32_t *__restrict__ xe, Lacking *__restrict__ xl) {
  const int64_t m = blockIdx.x;
  const float *xr = X + m * K;
  const int t = threadIdx.x;
  int e = 0;
  bool again = false;  // F16: some of the row's values are to be listed
  __shared__ int n_list;
  __shared__ Lacking list[kList];
  if constexpr (KIND == kF16) {
    __shared__ float red[2][4];
    if (t == 0) n_list = 0;
    float mx = 0.f, mn = INFINITY;  // of the finite values, mn without zeros
#pragma unroll 4
    for (int64_t j = 4 * (int64_t)t; j < K; j += 1024) {
      const float4 v = *reinterpret_cast<const float4 *>(xr + j);
      const float a[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) row_range(a[i], mx, mn);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      mx = fmaxf(mx, __shfl_xor(mx, off));
      mn = fminf(mn, __shfl_xor(mn, off));
    }
    if ((t & 63) == 0) {
      red[0][t >> 6] = mx;
      red[1][t >> 6] = mn;
    }
    __syncthreads();
    mx = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    mn = fminf(fminf(red[1][0], red[1][1]), fminf(red[1][2], red[1][3]));
    e = row_exp(mx);
    again = __builtin_amdgcn_ldexpf(mn, e) < 0x1p-14f;
  }
  for (int64_t j = 4 * (int64_t)t; j < Kp; j += 1024) {
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (j < K) v = *reinterpret_cast<const float4 *>(xr + j);
    float a[4] = {v.x, v.y, v.z, v.w};
    if (KIND == kF16 && again)
      for (int i = 0; i < 4; ++i) {
        const float d = lacking(i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w, e);
        if (d == 0.f) continue;
        const int slot = atomicAdd(&n_list, 1);
        if (slot < kList) list[slot] = Lacking{(int32_t)j + i, d};
      }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (KIND == kF16) a[i] = __builtin_amdgcn_ldexpf(a[i], e);
      else again = again || no_pieces(a[i]);
    }
    uint32_t w[pieces_of(KIND)][2];
    cut4<KIND>(a, w);
#pragma unroll
    for (int p = 0; p < pieces_of(KIND); ++p)
      *reinterpret_cast<uint2 *>(xp + p * plane + m * Kp + j) = make_uint2(w[p][0], w[p][1]);
  }
  int mark = 0;
  if constexpr (KIND != kF16) {
    mark = __syncthreads_or(again) ? kAgain : 0;
  } else if (again) {  // the same for the whole workgroup
    __syncthreads();
    mark = n_list <= kList ? n_list : kAgain;
    if (t < mark && mark <= kList) {  // in column order
      int at = 0;
      for (int i = 0; i < mark; ++i) at += list[i].k < list[t].k;
      xl[m * kList + at] = list[t];
    }
  }
  if (t == 0) xe[m] = 16 * e + mark;
}

// ---- tile kernel -----------------------------------------------------------------
template <int KIND, int MT, int NT, int WGM, int WGN>
struct DnTile {
  static constexpr int kWaves = WGM * WGN, kThreads = 64 * kWaves;
  static constexpr int BM = WGM * MT * 16, BN = WGN * NT * 16;
  static constexpr int kRow = KIND == kF32 ? 256 : 128;  // bytes of a W row's stage
  static constexpr int kX = pieces_of(KIND) * BM * 128, kW = BN * kRow;
  static constexpr int kLds = 2 * (kX + kW);
};

template <int KIND>
__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (KIND == kF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b),
                                                  c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a),
                                                   __builtin_bit_cast(b8, b), c, 0, 0, 0);
}

// NT tiles of plain fp32 products over columns k_begin .. k_end (a multiple of
// 32 long, not none): 16 rows of X (this lane's: `row`) by 16 rows of W each
// (this lane's of tile j: n + 16 j, row N - 1 past the last).  Lane group g takes
// columns 4 g .. +3 of every 16; the next 32 columns are loaded during the
// products of these.
template <int KIND, int NT>
__device__ __forceinline__ void plain_tile(const float *X, int64_t row, const uint8_t *W, int64_t n,
                                           int64_t N, int64_t K, int64_t k_begin, int64_t k_end,
                                           int g, f32x4 (&o)[NT]) {
  constexpr int ESZ = KIND == kF32 ? 4 : 2;
  using Raw = std::conditional_t<KIND == kF32, f32x4, uint2>;  // four weights
  const float *xr = X + row * K + 4 * g;
  const uint8_t *wr[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    wr[j] = W + ((n + 16 * j < N ? n + 16 * j : N - 1) * K + 4 * g) * ESZ;
    o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  f32x4 x[2], xn[2];
  Raw w[2][NT], wn[2][NT];
  auto load = [&](int64_t k, f32x4 (&xd)[2], Raw (&wd)[2][NT]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      xd[h] = *reinterpret_cast<const f32x4 *>(xr + k + 16 * h);
#pragma unroll
      for (int j = 0; j < NT; ++j)
        wd[h][j] = *reinterpret_cast<const Raw *>(wr[j] + (k + 16 * h) * ESZ);
    }
  };
  load(k_begin, x, w);
  for (int64_t k = k_begin; k < k_end; k += 32) {
    load(k + 32 < k_end ? k + 32 : k, xn, wn);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          float v;
          if constexpr (KIND == kF32) {
            v = w[h][j][t];
          } else {
            const uint32_t b = (t < 2 ? w[h][j].x : w[h][j].y) >> (16 * (t & 1)) & 0xFFFFu;
            v = KIND == kF16 ? (float)__builtin_bit_cast(_Float16, (uint16_t)b)
                             : __uint_as_float(b << 16);
          }
          o[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[h][t], v, o[j], 0, 0, 0);
        }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      x[h] = xn[h];
#pragma unroll
      for (int j = 0; j < NT; ++j) w[h][j] = wn[h][j];
    }
  }
}

// BARE: for calls that have no scratch for pieces of X.  The workgroup reads its
// rows of X once for their exponents and marks and cuts each stage's pieces into
// LDS itself, without a split of K: the same pieces, and bits, as otherwise
// (14336 x 4096 at M = 512 F16 265 us, BF16 538, F32 825 against 117, 148 and
// 332 with scratch and 650 on the fp32 kernel; at M = 2 85, 119, 152 against 42,
// 44, 78 and 370 - 390).
template <int KIND, int MT, int NT, int WGM, int WGN, bool BARE>
__global__ void __launch_bounds__(64 * WGM * WGN)
    k_mm_dn(const uint8_t *W, int64_t N, int64_t K, const uint16_t *xp, int64_t plane, int64_t Kp,
            const int32_t *__restrict__ xe, const Lacking *__restrict__ xl,
            const float *__restrict__ X, int64_t M, float *__restrict__ Y, int per_split, int m_tiles,
            int n_tiles) {
  using T = DnTile<KIND, MT, NT, WGM, WGN>;
  constexpr int BM = T::BM, BN = T::BN, WAVES = T::kWaves, NX = pieces_of(KIND);
  constexpr int NB = KIND == kF32 ? 3 : 1;           // pieces of W
  constexpr int ESZ = KIND == kF32 ? 4 : 2;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  const int g = lane >> 4, c16 = lane & 15;
  int mt, nt;
  if (!xcd_tile((int)blockIdx.x, m_tiles, n_tiles, mt, nt)) return;
  const int64_t m0 = (int64_t)mt * BM, n0 = (int64_t)nt * BN;
  const int n_st = (int)(Kp / 64);
  const int s_begin = (int)blockIdx.z * per_split;
  const int s_end = std::min(s_begin + per_split, n_st);
  Y += (int64_t)blockIdx.z * M * N;
  const uint32_t lds0 = lds_offset(smem);
  constexpr uint32_t oW = 2 * T::kX;

  // X stage: NX x BM rows of 128 bytes, chunk c of row r in slot c ^ (r & 7);
  // rows past M repeat row M - 1
  constexpr int XI = NX * BM / 8 / WAVES, XP = BM / 8, XR = XP / WAVES;
  static_assert(XP % WAVES == 0 && MT * 16 <= 64, "whole DMAs per wave and piece; a lane per row");
  uint32_t vx[XR];
#pragma unroll
  for (int i = 0; i < XR; ++i) {
    const int64_t r = m0 + 8 * (i * WAVES + wave) + (lane >> 3);
    vx[i] = (uint32_t)(2 * (r < M ? r : M - 1) * Kp) + 16 * ((lane & 7) ^ (lane >> 3));
  }
  // BARE: exponents and marks of the rows (rows past M: of row M - 1, unused)
  int *tab = reinterpret_cast<int *>(smem + T::kLds);
  if constexpr (BARE) {
    for (int r = wave; r < BM; r += WAVES) {
      const float *xr = X + (m0 + r < M ? m0 + r : M - 1) * K;
      float mx = 0.f, mn = INFINITY;
      bool bad = false;
      for (int64_t j = 4 * (int64_t)lane; j < K; j += 256) {
        const f32x4 v = *reinterpret_cast<const f32x4 *>(xr + j);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          row_range(v[i], mx, mn);
          bad = bad || no_pieces(v[i]);
        }
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        mx = fmaxf(mx, __shfl_xor(mx, off));
        mn = fminf(mn, __shfl_xor(mn, off));
      }
      int e = 0, mark = 0;
      if constexpr (KIND == kF16) {
        e = row_exp(mx);
        if (__builtin_amdgcn_ldexpf(mn, e) < 0x1p-14f) {
          for (int64_t j = lane; j < K; j += 64) mark += lacking(xr[j], e) != 0.f;
#pragma unroll
          for (int off = 32; off > 0; off >>= 1) mark += __shfl_xor(mark, off);
          if (mark > kList) mark = kAgain;
        }
      } else if (__any(bad)) {
        mark = kAgain;
      }
      if (lane == 0) tab[r] = 16 * e + mark;
    }
    __syncthreads();
  }
  // BARE: the pieces of X of a stage, laid out as the DMAs lay them out
  auto cut_stage = [&](int st, int buf) {
    for (int q = tid; q < BM * 8; q += T::kThreads) {
      const int r = q >> 3, c = q & 7;
      const int64_t col = (int64_t)st * 64 + 8 * c;
      float a[2][4] = {};
      if (col < K) {
        const float *p = X + (m0 + r < M ? m0 + r : M - 1) * K + col;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) a[h][i] = p[4 * h + i];
      }
      if constexpr (KIND == kF16) {
        const int e = tab[r] >> 4;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) a[h][i] = __builtin_amdgcn_ldexpf(a[h][i], e);
      }
      uint32_t w0[NX][2], w1[NX][2];
      cut4<KIND>(a[0], w0);
      cut4<KIND>(a[1], w1);
#pragma unroll
      for (int p = 0; p < NX; ++p)
        *reinterpret_cast<u32x4 *>(smem + buf * T::kX + p * BM * 128 + r * 128 + 16 * (c ^ (r & 7))) =
            u32x4{w0[p][0], w0[p][1], w1[p][0], w1[p][1]};
    }
  };
  // W stage: BN rows of kRow bytes, chunk c of row r in slot c ^ (r & 7); rows
  // past N repeat row N - 1.  Where K ends inside a stage (K is a multiple of
  // 32), the chunks past it repeat the stage's first half: x is zero there.
  constexpr int WC = T::kRow / 16, RPD = 64 / WC;  // chunks per row, rows per DMA
  constexpr int WI = BN / RPD / WAVES;
  static_assert(BN % (RPD * WAVES) == 0, "whole DMAs per wave");
  uint32_t vw[WI], tail = 0;
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int r = RPD * (i * WAVES + wave) + lane / WC;
    const int ck = (lane % WC) ^ (r & 7);
    const int64_t n = n0 + r < N ? n0 + r : N - 1;
    vw[i] = (uint32_t)(n * K * ESZ) + 16 * ck;
    // (the rows of a wave's DMAs agree modulo 8: RPD WAVES is a multiple of 8)
    if (16 * ck >= 32 * ESZ) tail = 32 * ESZ;
  }
  static_assert(RPD * WAVES % 8 == 0, "one swizzle per lane");
  auto dma_stage = [&](int st, int buf) {
    if constexpr (BARE) cut_stage(st, buf);
#pragma unroll
    for (int i = 0; i < (BARE ? 0 : XI); ++i)
      dma16(lds0 + buf * T::kX + 1024 * (i * WAVES + wave), vx[i % XR],
            reinterpret_cast<const uint8_t *>(xp) + 2 * plane * ((i * WAVES) / XP) + 128 * (int64_t)st);
    const uint32_t back = (int64_t)st * 64 + 64 > K ? tail : 0;
#pragma unroll
    for (int i = 0; i < WI; ++i)
      dma16(lds0 + oW + buf * T::kW + 1024 * (i * WAVES + wave), vw[i] - back,
            W + (int64_t)st * 64 * ESZ);
  };

  // fragments: A (row tile i, piece p) and B (column tile j) of sub-block e
  constexpr int STEPS = MT * NX;
  const uint8_t *pa = smem + 128 * (wm * MT * 16 + c16);
  const uint8_t *pb = smem + oW + T::kRow * (wn * NT * 16 + c16);
  const int sw = c16 & 7;
  auto read_a = [&](int buf, int e, int k) {
    // small pieces first
    return lds_read<u32x4>(pa + buf * T::kX + (NX - 1 - k / MT) * BM * 128 + (k % MT) * 16 * 128 +
                           16 * ((4 * e + g) ^ sw));
  };
  auto read_b = [&](int buf, int e, int j, u32x4 (&o)[NB]) {
    const uint8_t *p = pb + buf * T::kW + j * 16 * T::kRow;
    if constexpr (KIND == kF32) {
      uint32_t w[4][3];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f32x4 v = lds_read<f32x4>(p + 16 * ((8 * e + 2 * g + h) ^ sw));
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            const uint32_t u = pack_bf16(v[2 * i], v[2 * i + 1]);
            w[2 * h + i][q] = u;
            v[2 * i] -= __uint_as_float(u << 16);
            v[2 * i + 1] -= __uint_as_float(u & 0xFFFF0000u);
          }
      }
#pragma unroll
      for (int q = 0; q < NB; ++q) o[q] = u32x4{w[0][q], w[1][q], w[2][q], w[3][q]};
    } else {
      o[0] = lds_read<u32x4>(p + 16 * ((4 * e + g) ^ sw));
    }
  };

  // F16: acc[0] takes the products of hi, acc[1] those of lo
  constexpr int NA = KIND == kF16 ? 2 : 1;
  f32x4 acc[NA][MT][NT];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[a][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // A fragments are read two steps ahead (ring A), B a sub-block ahead.  At
  // step STEPS - 2 of a stage's second sub-block every fragment of the stage
  // is in registers: the barrier there publishes the next stage, issued a
  // stage ago, and frees this one's buffer.
  u32x4 A[4], B[2][NT][NB];
  // exponents and marks of the wave's rows, row i in lane i: loaded here and pinned
  // behind a stage's barrier (in the stores their latency would be 0.3 us of every
  // call)
  const int64_t my_row = m0 + wm * MT * 16 + lane;
  int mark = 0;
  if (lane < MT * 16 && my_row < M) mark = BARE ? tab[wm * MT * 16 + lane] : xe[my_row];
  dma_stage(s_begin, 0);
  if (s_begin + 1 < s_end) {
    dma_stage(s_begin + 1, 1);
    dma_barrier<(BARE ? 0 : XI) + WI>();
  } else {
    dma_barrier<0>();
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) read_b(0, 0, j, B[0][j]);
  A[0] = read_a(0, 0, 0);
  A[1] = read_a(0, 0, 1);
  for (int st = s_begin; st < s_end; ++st) {
    const int buf = (st - s_begin) & 1;
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int k = 0; k < STEPS; ++k) {
        const int step = e * STEPS + k;
        if (e == 1 && k == STEPS - 2 && st + 1 < s_end) {
          dma_barrier<0>();
          asm volatile("" : "+v"(mark));
          if (st + 2 < s_end) dma_stage(st + 2, buf);
        }
        // (past the last stage: whatever the other buffer holds, not used)
        A[(step + 2) % 4] = k + 2 < STEPS ? read_a(buf, e, k + 2)
                            : e == 0      ? read_a(buf, 1, k + 2 - STEPS)
                                          : read_a(buf ^ 1, 0, k + 2 - STEPS);
        const int i = k % MT, p = NX - 1 - k / MT;
        // pieces of W with index sum at most 2, small ones first
#pragma unroll
        for (int q = NB - 1; q >= 0; --q)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            if (p + q <= 2)
              acc[p % NA][i][j] = mfma<KIND>(A[step % 4], B[e][j][q], acc[p % NA][i][j]);
        if (e == 0) {
#pragma unroll
          for (int j = k * NT / STEPS; j < (k + 1) * NT / STEPS; ++j) read_b(buf, 1, j, B[1][j]);
        } else if (k >= STEPS - 2) {
          constexpr int H = NT / 2;
#pragma unroll
          for (int j = 0; j < H; ++j)
            read_b(buf ^ 1, 0, j + (k - STEPS + 2) * H, B[0][j + (k - STEPS + 2) * H]);
        }
      }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      const int64_t row = m0 + (wm * MT + i) * 16 + 4 * g + rr;
      int ex = 0;
      if constexpr (KIND == kF16) ex = __shfl(mark, i * 16 + 4 * g + rr) >> 4;
      if (row >= M) continue;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int64_t n = n0 + (wn * NT + j) * 16 + c16;
        if (n >= N) continue;
        float v = acc[0][i][j][rr];
        if constexpr (KIND == kF16)
          v = __builtin_amdgcn_ldexpf(fmaf(acc[NA - 1][i][j][rr], 1.f / (1 << kLoExp), v), -ex);
        Y[row * N + n] = v;
      }
    }
  // Marked rows, over what was stored (at the end: code that the stores jump over
  // costs every call 0.5 us of instruction fetches)
  if (__builtin_expect(__any(mark & 15), 0)) {
    const int64_t k_begin = 64 * (int64_t)s_begin, k_end = std::min(64 * (int64_t)s_end, K);
#pragma unroll 1
    for (int i = 0; i < MT; ++i) {
      const int64_t row0 = m0 + (wm * MT + i) * 16;
      int todo[4];
#pragma unroll
      for (int rr = 0; rr < 4; ++rr)  // (rows past M have no mark)
        todo[rr] = __shfl(mark, i * 16 + 4 * g + rr) & 15;
      if constexpr (KIND == kF16) {
#pragma unroll 1
        for (int rr = 0; rr < 4; ++rr) {
          const int64_t row = row0 + 4 * g + rr;
          const int count = todo[rr] == kAgain ? 0 : todo[rr];
          auto add = [&](int64_t k, float x) {
            for (int j = 0; j < NT; ++j) {
              const int64_t n = n0 + (wn * NT + j) * 16 + c16;
              if (n < N)
                Y[row * N + n] = fmaf(x, (float)reinterpret_cast<const _Float16 *>(W)[n * K + k],
                                      Y[row * N + n]);
            }
          };
          if constexpr (BARE) {
            const int e = __shfl(mark, i * 16 + 4 * g + rr) >> 4;
#pragma unroll 1
            for (int64_t k = 0; count > 0 && k < K; ++k) {
              const float d = lacking(X[row * K + k], e);
              if (d != 0.f) add(k, d);
            }
          } else {
#pragma unroll 1
            for (int c = 0; c < count; ++c) {
              const Lacking l = xl[row * kList + c];
              if (l.k >= k_begin && l.k < k_end) add(l.k, l.x);  // (else another split's)
            }
          }
        }
      }
      if (!__any(todo[0] == kAgain || todo[1] == kAgain || todo[2] == kAgain || todo[3] == kAgain))
        continue;
      f32x4 plain[NT];
      plain_tile<KIND, NT>(X, row0 + c16 < M ? row0 + c16 : M - 1, W, n0 + wn * NT * 16 + c16, N, K,
                           k_begin, k_end, g, plain);
#pragma unroll
      for (int rr = 0; rr < 4; ++rr)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const int64_t n = n0 + (wn * NT + j) * 16 + c16;
          if (todo[rr] == kAgain && n < N) Y[(row0 + 4 * g + rr) * N + n] = plain[j][rr];
        }
    }
  }
}

struct DnLaunch {
  const aq_matrix *m;
  const uint16_t *xp;
  int64_t plane, Kp;
  const int32_t *xe;
  const Lacking *xl;
  const float *X;
  int64_t M;
  float *dst;
  int splits, per;
  hipStream_t s;
};
template <int KIND, int MT, int NT, int WGM, int WGN, bool BARE = false>
hipError_t launch_tile(const DnLaunch &a) {
  using T = DnTile<KIND, MT, NT, WGM, WGN>;
  const int mt = (int)((a.M + T::BM - 1) / T::BM), nt = (int)((a.m->rows + T::BN - 1) / T::BN);
  const dim3 grid((unsigned)(((int64_t)mt * nt + 7) / 8 * 8), 1, (unsigned)a.splits);
  constexpr int lds = T::kLds + (BARE ? T::BM * 4 : 0);
  auto kern = k_mm_dn<KIND, MT, NT, WGM, WGN, BARE>;
  if (hipError_t e = set_dynamic_lds(reinterpret_cast<const void *>(kern), lds)) return e;
  hipLaunchKernelGGL(kern, grid, dim3(T::kThreads), lds, a.s, a.m->planes.p[0], a.m->rows,
                     a.m->cols, a.xp, a.plane, a.Kp, a.xe, a.xl, a.X, a.M, a.dst, a.per, mt, nt);
  return hipGetLastError();
}
template <int KIND>
hipError_t launch_shape(int shape, const DnLaunch &a) {
  if (!a.xp) {
    // without scratch: 14336 x 4096, 32 against 64 rows a tile, M = 64 F16 104
    // against 111 us, F32 175 / 207, M = 512 322 / 265, 1173 / 825 (BF16 538 / 621)
    if constexpr (KIND != kBF16) {
      if (a.M > 128) return launch_tile<KIND, 2, 2, 2, 4, true>(a);
    }
    return launch_tile<KIND, 2, 2, 1, 4, true>(a);
  }
  switch (shape) {
    case 0:
      if constexpr (KIND != kF32) return launch_tile<KIND, 4, 4, 2, 4>(a);
      return hipErrorInvalidValue;
    case 1: return launch_tile<KIND, 4, 2, 2, 4>(a);
    case 2: return launch_tile<KIND, 2, 2, 2, 4>(a);
    default: return launch_tile<KIND, 2, 2, 1, 4>(a);
  }
}

// Shapes of the tile kernel; kinds: F16, BF16, F32.  A fit to 3,387 timed calls
// (N 512 - 14336, K 2048 - 14336, M 2 - 1500, every shape with up to eight
// splits): 0.3 % slower than the fastest on average, 8 % at worst.
constexpr TileCost kTiles[] = {
    {128, 256, {1.70f, 2.40f, 0.f}, {0.f, 0.f, 0.f}, 4.2f},
    {128, 128, {1.39f, 1.98f, 2.63f}, {0.f, 0.f, 0.f}, 2.2f},
    {64, 128, {0.76f, 0.98f, 1.87f}, {0.954f, 1.42f, 0.f}, 0.8f},
    {32, 128, {0.56f, 0.63f, 1.17f}, {0.745f, 0.893f, 0.f}, 0.36f},
};
constexpr int kTileShapes = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr TileModel kModel = {kTiles, kTileShapes, 1.f, 1.f / 3.6f};

// A value among n 16- or 32-bit ones with a magnitude (as its bits) of at least
// `high`, or below `low` and not zero
template <class W>
__global__ void k_out_of_range(const W *__restrict__ p, int64_t n, W low, W high, int *flag) {
  bool bad = false;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const W u = p[i] & (W)((W)~(W)0 >> 1);
    bad = bad || u >= high || (u != 0 && u < low);
  }
  if (bad) *flag = 1;
}
}  // namespace

hipError_t dense_in_range(const aq_matrix *m, bool *in_range) {
  *in_range = true;
  const int64_t n = m->rows * m->cols;
  if (n == 0) return hipSuccess;
  int *flag = nullptr, host = 0;
  hipError_t e = hipMalloc(reinterpret_cast<void **>(&flag), sizeof(int));
  if (e != hipSuccess) return e;
  e = hipMemcpy(flag, &host, sizeof(int), hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    const unsigned wg = (unsigned)std::min<int64_t>((n + 255) / 256, 4096);
    if (m->dtype == AQ_F32)  // (from 2^127 on a bf16 piece may round to infinity)
      hipLaunchKernelGGL((k_out_of_range<uint32_t>), dim3(wg), dim3(256), 0, nullptr,
                         reinterpret_cast<const uint32_t *>(m->planes.p[0]), n,
                         __builtin_bit_cast(uint32_t, kPieceMin), 0x7F000000u, flag);
    else
      hipLaunchKernelGGL((k_out_of_range<uint16_t>), dim3(wg), dim3(256), 0, nullptr,
                         reinterpret_cast<const uint16_t *>(m->planes.p[0]), n, (uint16_t)0,
                         (uint16_t)(m->dtype == AQ_F16 ? 0x7C00u : 0x7F80u), flag);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(&host, flag, sizeof(int), hipMemcpyDeviceToHost);
  (void)hipFree(flag);
  *in_range = host == 0;
  return e;
}

bool mm_dn_supported(const aq_matrix *m) {
  // 32-bit offsets into W
  return is_dense(m->dtype) && m->in_range && m->nb_pitch == m->nb_row && m->cols > 0 &&
         (double)m->rows * (double)m->cols * (m->dtype == AQ_F32 ? 4.0 : 2.0) < 4294967296.0;
}

hipError_t launch_matmul_dn(const aq_matrix *m, const float *X, int64_t M, float *Y,
                            bool m_invariant, hipStream_t s) {
  if (M == 0 || m->rows == 0) return hipSuccess;
  const int kind = m->dtype == AQ_F16 ? kF16 : m->dtype == AQ_BF16 ? kBF16 : kF32;
  const int64_t K = m->cols, N = m->rows, Kp = (K + 63) / 64 * 64;
  if (!mm_dn_supported(m) || (double)M * Kp * 2 >= 2147483648.0) return hipErrorInvalidValue;
  const int units = (int)(Kp / 64), cus = device_info(m->device).cus;
  auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
  const int64_t plane = M * Kp;
  const size_t xb = al((size_t)pieces_of(kind) * plane * 2), eb = al((size_t)M * 4),
               lb = kind == kF16 ? al((size_t)M * kList * sizeof(Lacking)) : 0;
  DnLaunch a{m, nullptr, plane, Kp, nullptr, nullptr, X, M, Y, 1, units, s};
  int shape = 0;
  uint8_t *ws = nullptr;
  // with a split of K, without one (whose partials the scratch may not hold)
  for (int most = m_invariant ? 1 : 16;; most = 1) {
    int splits = 1;
    choose_tile(kModel, kind, M, N, units, 1, 4, cus, most, shape, splits);
    // AQ_MATMUL_TILE (tests): the shape itself, where the kind has it
    if (const char *env = getenv("AQ_MATMUL_TILE")) {
      const int v = atoi(env);
      if (v >= 0 && v < kTileShapes && kTiles[v].one[kind] > 0.f) shape = v;
    }
    a.per = (units + splits - 1) / splits;
    a.splits = (units + a.per - 1) / a.per;
    const size_t part = a.splits > 1 ? (size_t)a.splits * M * N * 4 : 0;
    ws = static_cast<uint8_t *>(workspace(m->device, s, xb + eb + lb + part));
    if (ws || most == 1) break;
    workspace_forgo();
  }
  if (ws) {
    uint16_t *xp = reinterpret_cast<uint16_t *>(ws);
    int32_t *xe = reinterpret_cast<int32_t *>(ws + xb);
    Lacking *xl = reinterpret_cast<Lacking *>(ws + xb + eb);
    if (a.splits > 1) a.dst = reinterpret_cast<float *>(ws + xb + eb + lb);
    a.xp = xp;
    a.xe = xe;
    a.xl = xl;
#define AQ_XP(k) \
  hipLaunchKernelGGL(k_x_pieces<k>, dim3((unsigned)M), dim3(256), 0, s, X, K, Kp, xp, plane, xe, xl)
    if (kind == kF16) AQ_XP(kF16);
    else AQ_XP(kBF16);  // (the same pieces for F32)
#undef AQ_XP
  } else {
    // Few weight rows have always needed scratch (the fp32 kernel splits K for
    // them): refused without, as before.
    if (matmul_t_fp32_splits(m) > 1) return hipErrorOutOfMemory;
    workspace_forgo();
  }
  const hipError_t e = kind == kF16    ? launch_shape<kF16>(shape, a)
                       : kind == kBF16 ? launch_shape<kBF16>(shape, a)
                                       : launch_shape<kF32>(shape, a);
  if (e != hipSuccess || a.splits == 1) return e;
  return sum_splits(a.dst, a.splits, M * N, Y, s);
}

}  // namespace aq
