// aq_matmul_hd.hip - the tile kernel of the exact fp16 matmul: Y = X W^T on
// fp16 matrix cores with the weights kept as exact integers and X in two fp16
// pieces (aq_matmul_h.hip prepares X and chooses the tiles).
//
// Replaces QuantMatrix.matmul_t (alpacca/qmatrix.py:184-211) at float32
// accuracy.  A workgroup owns BM rows of X and BN rows of W; K runs in
// groups of 256 columns, four stages of 64 (two sub-blocks of 32) each.
// Everything the products read comes into LDS by DMA (global_load_lds, 16
// bytes per lane): the X pieces of a stage XB - 1 stages ahead, the packed
// bytes of a whole 256-column group of the BN weight rows a group ahead.  A
// wave decodes the B operands of its own columns from LDS, one sub-block
// ahead, between the products of the current one.
//
// Per format (decoding as alpacca/quants.py:50-224):
//   Q4_K, Q5_K  B = sc * code, an integer below 2048 as the half whose bits
//               it is (m 2^-24 exactly); 16 products (8 sub-blocks x 2 pieces)
//               chain in one accumulator P, then acc += d P - dmin Q with Q
//               = sum mn S over the sub-block sums S of x
//               (v_mfma_f32_16x16x16f16).
//   Q6_K        B = sc * (q - 32), up to 13 bits: hi = fp16(B) and, where |B|
//               passes 2048, lo = B - hi in {-1, 0, 1}, both exact.  x_hi hi
//               chains over the block in P, x_lo hi + x_hi lo in P2 (so the
//               large sums round once per sub-block), then acc += d (P + P2);
//               the dropped x_lo lo is below 2^-22 of the element's term, as
//               x's own rounding.
//   per 32      B = code (Q8_0, Q4_0, Q5_0: with its offset; Q4_1, Q5_1: the
//               subnormal half code 2^-24): one block is two products, G +=
//               d P per block in fp32 and acc += G per group (shorter sums
//               than one accumulator over K: Q8_0 at K = 4096 2.1e-7 ->
//               1.2e-7 relative); the m term of Q4_1 / Q5_1 once per group from
//               the block sums of x, as Q above.
// An output is the same sequence of operations in every tile shape.
//
// What bounds it: a 128 x 256 tile as eight waves of 64 x 64 issues 64
// products per wave and stage for 16 A fragment reads, so LDS (72 bytes per
// clock) and VALU (two instructions per product) both stay under the matrix
// cores; Q4_K 28672 x 4096 at M = 2048 runs 1.1 PFLOP/s of fp16 products
// (hipBLASLt's fp16 GEMM of 8192^3 on the same card: 1.2 - 1.3), and with
// every load, the decode and the scales left out 1.5.  The register-staged
// kernel before it, each wave with its weights in registers and 64 x 256
// tiles, read the X fragments twice as often: Q4_K 14336 x 4096 at M = 512
// 155 -> 121 us per call, M = 128 53 -> 47, 16384 x 2048 at M = 2048 331 ->
// 264 us.
#include <algorithm>
#include <type_traits>

#include "aq_internal.h"
#include "aq_matmul_dma.h"
#include "aq_matmul_h.h"

namespace aq {
namespace {

// ---- formats -------------------------------------------------------------------
// The packed bytes of a 256-column group of one row in LDS: three fields one
// after the other, kF0, kF1, kF2 16-byte chunks (kPad more to spread 16 rows
// over the banks), each from its own plane.  kNB B operands per sub-block;
// kChain: products chain over the group (scales at its end) or per 32; kSums:
// needs the sub-block sums of X; kD2: the group's fp16 d comes apart (2 bytes
// per row and group).  fetch() reads what stage c's two sub-blocks need,
// decode() makes the B operands of sub-block e (lane group g: elements 8 g ..
// 8 g + 7) and its scale.

// Q4_K / Q5_K: header (d, dmin, 12 scale bytes), qh, qs.  Sub-blocks 2c and
// 2c+1 are the low and high nibbles of qs[32c, 32c + 32) (quants.py:136-193).
template <bool Q5>
struct HdKq {
  static constexpr int kF0 = 1, kF1 = Q5 ? 2 : 0, kF2 = 8, kPad = 0, kNB = 1;
  static constexpr bool kChain = true, kSums = true, kD2 = false;
  struct Words {
    uint2 w, q5;
    uint32_t sc;
  };
  __device__ static void fetch(const uint8_t *p, int c, int g, Words &r) {
    r.w = lds_read<uint2>(p + (Q5 ? 48 : 16) + 32 * c + 8 * g);
    if constexpr (Q5) r.q5 = lds_read<uint2>(p + 16 + 8 * g);
    const uint4 h = lds_read<uint4>(p);
    uint32_t mn;
    kquant_scale_pair(h.y, h.z, h.w, c, r.sc, mn);
  }
  __device__ static void decode(const Words &r, int c, int e, int, u32x4 *o, float &) {
    uint32_t x = (r.w.x >> (4 * e)) & 0x0F0F0F0Fu, y = (r.w.y >> (4 * e)) & 0x0F0F0F0Fu;
    if constexpr (Q5) {  // the fifth bit: 16 when set
      x |= ((r.q5.x >> (2 * c + e)) & 0x01010101u) << 4;
      y |= ((r.q5.y >> (2 * c + e)) & 0x01010101u) << 4;
    }
    uint32_t v[4];
    sc_codes8(x, y, __builtin_amdgcn_perm(0u, r.sc, e ? 0x0C010C01u : 0x0C000C00u), v);
    o[0] = u32x4{v[0], v[1], v[2], v[3]};
  }
  __device__ static void group_end(const uint8_t *p, uint32_t, int g, float &d, float &dm, h4 &bm) {
    kquant_block_scales(lds_read<uint4>(p), g, d, dm, bm);
  }
};

// Q6_K: ql, qh, 16 int8 scales, d apart.  Sub-block 4 hf + 2 h + e takes ql
// bytes 64 hf + 32 e .., nibble h, and qh bytes 32 hf .. at shift 4 h + 2 e
// (quants.py:196-224), so stage c is hf = c / 2, h = c % 2; the scale of lane
// group g's elements is byte 4c + 2e + g / 2.
struct HdQ6 {
  static constexpr int kF0 = 8, kF1 = 4, kF2 = 1, kPad = 0, kNB = 2;
  static constexpr bool kChain = true, kSums = false, kD2 = true;
  struct Words {
    uint2 w[2], qh;
    uint32_t sc;
  };
  __device__ static void fetch(const uint8_t *p, int c, int g, Words &r) {
    r.w[0] = lds_read<uint2>(p + 64 * (c >> 1) + 8 * g);
    r.w[1] = lds_read<uint2>(p + 64 * (c >> 1) + 32 + 8 * g);
    r.qh = lds_read<uint2>(p + 128 + 32 * (c >> 1) + 8 * g);
    r.sc = lds_read<uint32_t>(p + 192 + 4 * c) >> (8 * (g >> 1));  // bytes 0 and 2 are this lane's
  }
  __device__ static void decode(const Words &r, int c, int e, int, u32x4 *o, float &) {
    const int h = c & 1;
    const uint32_t x = ((r.w[e].x >> (4 * h)) & 0x0F0F0F0Fu) |
                       (((r.qh.x >> (4 * h + 2 * e)) & 0x03030303u) << 4);
    const uint32_t y = ((r.w[e].y >> (4 * h)) & 0x0F0F0F0Fu) |
                       (((r.qh.y >> (4 * h + 2 * e)) & 0x03030303u) << 4);
    const h2 s1 = (h2)(_Float16)(float)((int32_t)(r.sc << (24 - 16 * e)) >> 24);
    const uint32_t cw[2] = {x, y};
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // the halves 1024 + q, less 1056
      const h2 t = __builtin_bit_cast(
          h2, fma_h2(__builtin_amdgcn_perm(0x64646464u, cw[q >> 1],
                                           (q & 1) ? 0x05030402u : 0x05010400u),
                     0x3c003c00u, 0xe420e420u));
      const h2 a = t * s1;
      hi[q] = __builtin_bit_cast(uint32_t, a);
      lo[q] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t, s1, -a));
    }
    o[0] = u32x4{hi[0], hi[1], hi[2], hi[3]};
    o[1] = u32x4{lo[0], lo[1], lo[2], lo[3]};
  }
  __device__ static void group_end(const uint8_t *, uint32_t d2, int, float &d, float &, h4 &) {
    d = f16_bits_to_f32(d2);
  }
};

// Q8_0, Q4_0, Q4_1, Q5_0, Q5_1: codes, fifth bits, d (or d | m).  QSB code
// bytes per block; OFF: code offset (0 with a min).  B from the code under
// 0x64 (the half 1024 + code; Q8_0: q + 128 after flipping its sign bit) and
// one packed fma by (1, -(1024 + OFF)), or the code as a subnormal half.
template <int QSB, bool HIGH, bool MIN, int OFF>
struct HdB32 {
  static constexpr int SB = MIN ? 4 : 2;  // scale bytes per block
  static constexpr int kF0 = QSB / 2, kF1 = HIGH ? 2 : 0, kF2 = SB / 2, kNB = 1;
  static constexpr int kPad = HIGH && MIN ? 1 : 0;
  static constexpr bool kChain = false, kSums = MIN, kD2 = false, kNib = QSB == 16;
  static constexpr int kScales = 16 * (kF0 + kF1);
  struct Words {
    uint2 w[2];
    uint32_t s[2], hb[2];
  };
  __device__ static void fetch(const uint8_t *p, int c, int g, Words &r) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int blk = 2 * c + e;
      r.w[e] = lds_read<uint2>(p + QSB * blk + (kNib ? 8 * (g & 1) : 8 * g));
      if constexpr (HIGH) r.hb[e] = p[16 * kF0 + 4 * blk + g];
      if constexpr (MIN) r.s[e] = lds_read<uint32_t>(p + kScales + 4 * blk);
    }
    if constexpr (!MIN) {
      const uint32_t s = lds_read<uint32_t>(p + kScales + 4 * c);
      r.s[0] = s & 0xFFFFu;
      r.s[1] = s >> 16;
    }
  }
  __device__ static void decode(const Words &r, int, int e, int g, u32x4 *o, float &dsc) {
    uint32_t c0 = r.w[e].x, c1 = r.w[e].y;
    if constexpr (kNib) {
      const int sh = 4 * (g >> 1);
      c0 = (c0 >> sh) & 0x0F0F0F0Fu;
      c1 = (c1 >> sh) & 0x0F0F0F0Fu;
    } else {
      c0 ^= 0x80808080u;
      c1 ^= 0x80808080u;
    }
    if constexpr (HIGH) {
      c0 |= spread4_to_bit4(r.hb[e] & 15u);
      c1 |= spread4_to_bit4(r.hb[e] >> 4);
    }
    uint32_t v[4];
    if constexpr (OFF == 0) {
      v[0] = __builtin_amdgcn_perm(0u, c0, 0x0C010C00u);
      v[1] = __builtin_amdgcn_perm(0u, c0, 0x0C030C02u);
      v[2] = __builtin_amdgcn_perm(0u, c1, 0x0C010C00u);
      v[3] = __builtin_amdgcn_perm(0u, c1, 0x0C030C02u);
      dsc = f16_bits_to_f32(r.s[e]) * 16777216.f;
    } else {
      constexpr uint32_t kSub = (0xE400u | OFF) * 0x10001u;  // -(1024 + offset), twice
      v[0] = fma_h2(__builtin_amdgcn_perm(0x64646464u, c0, 0x05010400u), 0x3c003c00u, kSub);
      v[1] = fma_h2(__builtin_amdgcn_perm(0x64646464u, c0, 0x05030402u), 0x3c003c00u, kSub);
      v[2] = fma_h2(__builtin_amdgcn_perm(0x64646464u, c1, 0x05010400u), 0x3c003c00u, kSub);
      v[3] = fma_h2(__builtin_amdgcn_perm(0x64646464u, c1, 0x05030402u), 0x3c003c00u, kSub);
      dsc = f16_bits_to_f32(r.s[e]);
    }
    o[0] = u32x4{v[0], v[1], v[2], v[3]};
  }
  // m of blocks 4 (g & 1) .. +3 (the sums of x carry 2^(e-5))
  __device__ static void group_end(const uint8_t *p, uint32_t, int g, float &, float &dm, h4 &bm) {
    if constexpr (MIN) {
      const uint4 s = lds_read<uint4>(p + kScales + 16 * (g & 1));
      bm = __builtin_bit_cast(h4, uint2{__builtin_amdgcn_perm(s.y, s.x, 0x07060302u),
                                        __builtin_amdgcn_perm(s.w, s.z, 0x07060302u)});
      dm = 32.f;
    }
  }
};

// ---- tile kernel -----------------------------------------------------------------
constexpr int NP = 2;  // pieces of X

// XB: X stages in LDS.  A group is four stages and stage c of any group uses
// buffer c % XB, so XB divides four.
template <class F, int MT, int NT, int WGM, int WGN, int XB>
struct HdTile {
  static_assert(XB == 2 || XB == 4, "whole turns of the X buffers per group");
  static constexpr int kWaves = WGM * WGN, kThreads = 64 * kWaves;
  static constexpr int BM = WGM * MT * 16, BN = WGN * NT * 16;
  static constexpr int kParts = F::kF0 + F::kF1 + F::kF2 + F::kPad;  // 16-byte chunks of a row
  static constexpr int kPitch = 16 * kParts;
  static constexpr int kX = NP * BM * 128;  // LDS bytes of one X stage
  static constexpr int kW = BN * kPitch;    // of one group of BN weight rows
  static constexpr int kS = F::kSums ? std::max(BM, 32) * 32 : 0;  // of its sums of X
  static constexpr int kD = F::kD2 ? BN * 4 : 0;                   // of its d
  static constexpr int kLds = XB * kX + 2 * (kW + kS + kD);
};

// off / st: byte offset of each field's plane from wbase, and its bytes per
// group (off3: the d plane of kD2); ng groups per row.
struct HdPlanes {
  uint32_t off[4], st[3];
};

template <class F, int MT, int NT, int WGM, int WGN, int XB>
__global__ void __launch_bounds__(64 * WGM * WGN)
    k_mm_hd(const uint8_t *wbase, HdPlanes pl, int64_t N, int ng, const uint16_t *xp,
            int64_t plane, const int32_t *__restrict__ xe, const uint16_t *xs, int64_t M,
            float *__restrict__ Y, int per_split, int m_tiles, int n_tiles,
            float *__restrict__ Ysw) {
  using T = HdTile<F, MT, NT, WGM, WGN, XB>;
  constexpr int BM = T::BM, BN = T::BN, WAVES = T::kWaves, PARTS = T::kParts, PITCH = T::kPitch;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  const int g = lane >> 4, c16 = lane & 15;
  int mt, nt;
  if (!xcd_tile((int)blockIdx.x, m_tiles, n_tiles, mt, nt)) return;
  const int64_t m0 = (int64_t)mt * BM, n0 = (int64_t)nt * BN;
  const int64_t K = (int64_t)ng * 256;
  const int b_begin = (int)blockIdx.z * per_split;
  const int b_end = std::min(b_begin + per_split, ng);
  Y += (int64_t)blockIdx.z * M * N;

  const uint32_t lds0 = lds_offset(smem);
  constexpr uint32_t oW = XB * T::kX, oS = oW + 2 * T::kW, oD = oS + 2 * T::kS;

  // X stage: NP x BM rows of 128 bytes, 16-byte chunk c of row r in slot
  // c ^ (r & 7) (the reads of 16 rows at one chunk then meet no bank twice).
  // A DMA covers 8 rows; those of one piece come first.  Rows past M repeat
  // row M - 1 (their outputs are not stored).
  constexpr int XI = NP * BM / 8 / WAVES;  // DMAs per wave and stage
  constexpr int XP = BM / 8;               // DMAs per piece
  static_assert(NP * BM % (8 * WAVES) == 0 && (XP % WAVES == 0 || WAVES % XP == 0), "whole DMAs");
  constexpr int XR = XP >= WAVES ? XP / WAVES : 1;  // different rows of a wave's DMAs
  uint32_t vx[XR];
#pragma unroll
  for (int i = 0; i < XR; ++i) {
    const int64_t r = m0 + 8 * ((i * WAVES + wave) % XP) + (lane >> 3);
    vx[i] = (uint32_t)(2 * (r < M ? r : M - 1) * K) + 16 * ((lane & 7) ^ (lane >> 3));
  }
  const uint8_t *xbase = reinterpret_cast<const uint8_t *>(xp) + 512 * (int64_t)b_begin;
  auto x_dma = [&](int stg, int buf) {  // stage stg of the split
#pragma unroll
    for (int i = 0; i < XI; ++i)
      dma16(lds0 + buf * T::kX + 1024 * (i * WAVES + wave), vx[i % XR],
            xbase + 2 * plane * ((i * WAVES + wave) / XP) + 128 * (int64_t)stg);
  };
  // W: the chunks of a group of the tile's BN rows, row by row; rows past N
  // repeat row N - 1.  WF DMAs of every wave, one more of the first WV.
  constexpr int WD = BN * PARTS / 64, WF = WD / WAVES, WV = WD % WAVES;
  static_assert(BN * PARTS % 64 == 0, "whole DMAs");
  uint32_t vw[WF + 1], sw[WF + 1];
#pragma unroll
  for (int i = 0; i <= WF; ++i) {
    const int q = (i * WAVES + wave) * 64 + lane;
    const int col = std::min(q / PARTS, BN - 1), part = q % PARTS;
    const int64_t n = n0 + col < N ? n0 + col : N - 1;
    const uint32_t grp = (uint32_t)(n * ng + b_begin);
    const bool f0 = part < F::kF0, f1 = part < F::kF0 + F::kF1;
    const bool f2 = part < F::kF0 + F::kF1 + F::kF2;  // (padding repeats chunk 0 of field 0)
    const int first = f0 || !f2 ? (f0 ? 0 : part) : f1 ? F::kF0 : F::kF0 + F::kF1;
    const int f = f0 || !f2 ? 0 : f1 ? 1 : 2;
    sw[i] = f == 0 ? pl.st[0] : f == 1 ? pl.st[1] : pl.st[2];
    vw[i] = (f == 0 ? pl.off[0] : f == 1 ? pl.off[1] : pl.off[2]) + grp * sw[i] +
            16 * (part - first);
  }
  auto w_dma = [&](int i, int buf) {
    dma16(lds0 + oW + buf * T::kW + 1024 * (i * WAVES + wave), vw[i], wbase);
    vw[i] += sw[i];
  };
  // the small parts of a group: sub-block sums of X, 32 bytes a row (waves 0 ..
  // SI - 1), d of the BN rows (waves 0 .. DI - 1: the aligned word that holds it)
  constexpr int SI = F::kSums ? (BM + 31) / 32 : 0, DI = F::kD2 ? BN / 64 : 0;
  static_assert(SI <= WAVES && DI <= WAVES && (!F::kD2 || BN % 64 == 0), "one DMA per wave");
  uint32_t vs = 0, vd = 0;
  if constexpr (F::kSums) {
    const int64_t r = m0 + 32 * wave + (lane >> 1);
    vs = (uint32_t)((r < M ? r : M - 1) * ng * 32) + 16 * (lane & 1);
  }
  if constexpr (F::kD2) {
    const int64_t n = n0 + 64 * wave + lane;
    vd = (uint32_t)((n < N ? n : N - 1) * ng);
  }
  auto s_dma = [&](int b, int buf) {
    if (F::kSums && wave < SI)
      dma16(lds0 + oS + buf * T::kS + 1024 * wave, vs,
            reinterpret_cast<const uint8_t *>(xs) + 32 * (int64_t)b);
    if (F::kD2 && wave < DI)
      dma4(lds0 + oD + buf * T::kD + 256 * wave, pl.off[3] + ((2 * (vd + (uint32_t)b)) & ~3u),
           wbase);
  };

  // fragment addresses
  const uint8_t *pa[2];
  {
    const int r = wm * MT * 16 + c16, s0 = g ^ (c16 & 7);
    pa[0] = smem + 128 * r + 16 * s0;
    pa[1] = smem + 128 * r + 16 * (s0 ^ 4);
  }
  const uint8_t *pw0 = smem + oW + (wn * NT * 16 + c16) * PITCH;
  const uint8_t *ps0 = smem + oS + (wm * MT * 16 + c16) * 32 + 8 * g;
  const uint8_t *pd0 = smem + oD + (wn * NT * 16 + c16) * 4;

  // kChain: P (and P2, the small products of kNB = 2) chain the group's
  // products of every tile; else P holds those of two row tiles in turn and
  // G the group's scaled sums
  constexpr int PR = F::kChain ? MT : 2;
  constexpr int GR = F::kChain ? (F::kNB > 1 ? MT : 1) : MT;
  f32x4 acc[MT][NT], P[PR][NT], G[GR][NT];
  auto &P2 = G;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // The products of a sub-block run as STEPS steps, one A fragment (row tile
  // i, piece p) against the NT column tiles each.  A fragments are read two
  // steps ahead (ring A), B operands and scales are decoded a sub-block
  // ahead, a part of them per step.
  constexpr int STEPS = MT * NP;
  h8 A[4];
  auto read_a = [&](int c, int e, int k, h8 &dst) {
    dst = lds_read<h8>(pa[e] + (c % XB) * T::kX + (k % NP) * BM * 128 + (k / NP) * 16 * 128);
  };
  typename F::Words w[NT];
  u32x4 B[2][NT][F::kNB];
  float dsc[2][NT];

  // prologue: group b_begin, the first XB stages of X and the first part of
  // the next group
  constexpr int W0 = (WF + 1) / 2, W1 = WF - W0;  // W DMAs issued with two X stages
#pragma unroll
  for (int i = 0; i < WF; ++i) w_dma(i, 0);
  if (WV && wave < WV) w_dma(WF, 0);
  s_dma(b_begin, 0);
  x_dma(0, 0);
  if (b_begin + 1 < b_end) {
    if (WV && wave < WV) w_dma(WF, 1);
    s_dma(b_begin + 1, 1);
  }
#pragma unroll
  for (int i = 1; i < XB; ++i) x_dma(i, i);
  if (b_begin + 1 < b_end) {
#pragma unroll
    for (int i = 0; i < W0; ++i) w_dma(i, 1);
    dma_barrier<(XB - 1) * XI + W0>();
  } else {
    dma_barrier<(XB - 1) * XI>();
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    F::fetch(pw0 + j * 16 * PITCH, 0, g, w[j]);
    F::decode(w[j], 0, 0, g, B[0][j], dsc[0][j]);
  }
  read_a(0, 0, 0, A[0]);
  read_a(0, 0, 1, A[1]);

  // One group.  MORE: another one follows in the split.  At step S - 2 of a
  // stage's second sub-block every fragment of the stage is in registers:
  // the barrier there publishes the next stage's X and frees this stage's
  // buffer for the X after it.
  auto group = [&](int b, auto more_c) {
    constexpr bool MORE = decltype(more_c)::value;
    const int par = (b - b_begin) & 1;
    const uint8_t *pw = pw0 + par * T::kW, *pwn = pw0 + (par ^ 1) * T::kW;
    const uint8_t *ps = ps0 + par * T::kS, *pd = pd0 + par * T::kD;
    const int st0 = 4 * (b - b_begin);
    float d[NT], dm[NT];
    h4 bm[NT], as[MT];
    // per 32: the scaled product of row tile i of sub-block sb.  The empty
    // assembly keeps the sums here: the compiler would sink those of a whole
    // group to its end, with every product kept until then (256 registers
    // and 0.4 - 1.8 KB of spills).
    auto add32 = [&](int i, int sb) {
      const int e = sb & 1;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const float v = P[(i + e * MT) & 1][j][rr];
          G[i % GR][j][rr] = sb ? fmaf(dsc[e][j], v, G[i % GR][j][rr]) : dsc[e][j] * v;
        }
        asm volatile("" : "+v"(G[i % GR][j]));
      }
    };
    // the end of a group for one tile: its products and the min term
    auto finish = [&](int i, int j) {
      f32x4 q;
      if constexpr (F::kSums)
        q = __builtin_amdgcn_mfma_f32_16x16x16f16(as[i], bm[j], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        if constexpr (!F::kChain) acc[i][j][rr] += G[i % GR][j][rr];
        else if constexpr (F::kNB > 1)
          acc[i][j][rr] = fmaf(d[j], P[i % PR][j][rr] + P2[i % GR][j][rr], acc[i][j][rr]);
        else acc[i][j][rr] = fmaf(d[j], P[i % PR][j][rr], acc[i][j][rr]);
        if constexpr (F::kSums) acc[i][j][rr] = fmaf(dm[j], q[rr], acc[i][j][rr]);
      }
    };
    auto stage = [&](auto cc) {
      constexpr int c = decltype(cc)::value;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
#pragma unroll
        for (int k = 0; k < STEPS; ++k) {
          const int i = k / NP, p = k % NP;
          const int step = (2 * c + e) * STEPS + k;
          if (e == 1 && k == STEPS - 2 && (c < 3 || MORE)) {
            // X of the next stage has landed: the XB - 2 stages after it
            // may be in flight, and the W DMAs issued since (the first part
            // with the last X stage of a group, the rest with the next one).
            // W, sums and d of the next group have landed by stage 2's
            // barrier.
            constexpr int XF = (XB - 2) * XI;
            if constexpr (!MORE) dma_barrier<std::max(0, std::min(XB - 2, 2 - c)) * XI>();
            else if (c == 0) dma_barrier<XF + W0>();
            else if (c == 1) dma_barrier<XF + (XB > 2 ? W0 : 0) + W1>();
            else if (c == 2) dma_barrier<std::min(XF, XI)>();
            else dma_barrier<XF>();
            const bool next = c == 3 && b + 2 < b_end;
            if (next) {
              if (WV && wave < WV) w_dma(WF, par);
              s_dma(b + 2, par);
            }
            if (c + XB < 4 || MORE) x_dma(st0 + c + XB, c % XB);
            if (next) {
#pragma unroll
              for (int q = 0; q < W0; ++q) w_dma(q, par);
            }
            if (c == 0 && MORE) {
#pragma unroll
              for (int q = W0; q < WF; ++q) w_dma(q, par ^ 1);
            }
          }
          // fragment two steps ahead
          if (k + 2 < STEPS) read_a(c, e, k + 2, A[(step + 2) % 4]);
          else if (e == 0) read_a(c, 1, k + 2 - STEPS, A[(step + 2) % 4]);
          else if (c < 3 || MORE) read_a((c + 1) & 3, 0, k + 2 - STEPS, A[(step + 2) % 4]);
          const int pi = F::kChain ? i : (i + e * MT) & 1;
          const bool first = F::kChain ? c == 0 && e == 0 && p == 0 : p == 0;
          const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            const h8 b0 = __builtin_bit_cast(h8, B[e][j][0]);
            if constexpr (F::kNB == 1) {
              P[pi][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[step % 4], b0,
                                                                first ? zero : P[pi][j], 0, 0, 0);
            } else if (p == 0) {
              P[pi][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[step % 4], b0,
                                                                first ? zero : P[pi][j], 0, 0, 0);
              P2[i % GR][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                  A[step % 4], __builtin_bit_cast(h8, B[e][j][F::kNB - 1]),
                  first ? zero : P2[i % GR][j], 0, 0, 0);
            } else {
              P2[i % GR][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[step % 4], b0,
                                                                     P2[i % GR][j], 0, 0, 0);
            }
          }
          if constexpr (!F::kChain) {
            if (p == 0 && i > 0) add32(i - 1, 2 * c + e);
            if (k == 0 && c + e > 0) add32(MT - 1, 2 * c + e - 1);
          }
          // the next sub-block's operands, column tile by column tile
#pragma unroll
          for (int j = k * NT / STEPS; j < (k + 1) * NT / STEPS; ++j) {
            if (e == 0) {
              F::decode(w[j], c, 1, g, B[1][j], dsc[1][j]);
              if (c < 3 || MORE)
                F::fetch((c < 3 ? pw : pwn) + j * 16 * PITCH, (c + 1) & 3, g, w[j]);
            } else if (c < 3 || MORE) {
              F::decode(w[j], (c + 1) & 3, 0, g, B[0][j], dsc[0][j]);
            }
            if (c == 3 && e == 0) {
              uint32_t d2 = 0;
              if constexpr (F::kD2) {
                const int64_t n = n0 + (wn * NT + j) * 16 + c16;
                const uint32_t odd = (uint32_t)((n < N ? n : N - 1) * ng + b) & 1u;
                d2 = lds_read<uint32_t>(pd + j * 64) >> (16 * odd);
              }
              F::group_end(pw + j * 16 * PITCH, d2, g, d[j], dm[j], bm[j]);
            }
          }
          if (F::kSums && c == 3 && e == 0 && p == 0) as[i] = lds_read<h4>(ps + i * 16 * 32);
          if (F::kChain && c == 3 && e == 1 && i > 0) {  // row tile i - 1, a part per step
#pragma unroll
            for (int j = p * NT / NP; j < (p + 1) * NT / NP; ++j) finish(i - 1, j);
          }
        }
      }
    };
    stage(std::integral_constant<int, 0>{});
    stage(std::integral_constant<int, 1>{});
    stage(std::integral_constant<int, 2>{});
    stage(std::integral_constant<int, 3>{});
    if constexpr (!F::kChain) add32(MT - 1, 7);
#pragma unroll
    for (int i = F::kChain ? MT - 1 : 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) finish(i, j);
  };
  int b = b_begin;
  for (; b + 1 < b_end; ++b) group(b, std::true_type{});
  group(b, std::false_type{});
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int64_t row0 = m0 + (wm * MT + i) * 16 + 4 * g;
    int ex[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) ex[rr] = row0 + rr < M ? xe[row0 + rr] : 0;
#pragma unroll
    for (int j = 0; j < NT; ++j)
      store_tile(acc[i][j], ex, row0, n0 + (wn * NT + j) * 16 + c16, M, N, c16 & 1, Y, Ysw);
  }
}

struct HdLaunch {
  const aq_matrix *m;
  HdPlanes pl;
  int ng;
  MmhX x;
  int64_t M;
  float *dst;
  int splits, per;
  float *ysw;
  hipStream_t s;
};

template <class F, int MT, int NT, int WGM, int WGN, int XB>
hipError_t launch_tile(const HdLaunch &a) {
  using T = HdTile<F, MT, NT, WGM, WGN, XB>;
  const int mt = (int)((a.M + T::BM - 1) / T::BM), nt = (int)((a.m->rows + T::BN - 1) / T::BN);
  const dim3 grid((unsigned)(((int64_t)mt * nt + 7) / 8 * 8), 1, (unsigned)a.splits);
  auto kern = k_mm_hd<F, MT, NT, WGM, WGN, XB>;
  if (hipError_t e = set_dynamic_lds(reinterpret_cast<const void *>(kern), T::kLds)) return e;
  hipLaunchKernelGGL(kern, grid, dim3(T::kThreads), T::kLds, a.s, a.m->dev, a.pl, a.m->rows, a.ng,
                     a.x.xp, a.x.plane, a.x.xe, a.x.xs, a.M, a.dst, a.per, mt, nt, a.ysw);
  return hipGetLastError();
}

template <class F>
hipError_t launch_shape(int shape, const HdLaunch &a) {
  switch (shape) {
    case 0:
      if constexpr (F::kChain && F::kNB == 1)
        return launch_tile<F, 4, 4, 2, 4, 2>(a);
      return hipErrorInvalidValue;
    case 1: return launch_tile<F, 4, 2, 2, 4, 2>(a);
    case 2: return launch_tile<F, 2, 2, 2, 4, 2>(a);
    case 3: return launch_tile<F, 2, 2, 1, 4, 2>(a);
    default: {
      // A stage of 16 rows is shorter than an X stage's way into LDS, so three are
      // under way at a time where the LDS for it costs no second workgroup on a
      // CU: always but for Q8_0, there where the launch has none (4096 x 14336
      // unsplit, M = 16: Q8_0 90.2 us with one, 77.3 with three, Q4_K 90.8 / 75.8;
      // split, two Q8_0 workgroups to a CU: 23.8 / 27.2).
      using T4 = HdTile<F, 1, 2, 1, 4, 4>;
      constexpr bool pair = 2 * T4::kLds <= 160 * 1024;
      if constexpr (!pair) {
        const int64_t wgs = (a.M + T4::BM - 1) / T4::BM * ((a.m->rows + T4::BN - 1) / T4::BN) * a.splits;
        if (wgs > device_info(a.m->device).cus) return launch_tile<F, 1, 2, 1, 4, 2>(a);
      }
      return launch_tile<F, 1, 2, 1, 4, 4>(a);
    }
  }
}

}  // namespace

hipError_t launch_mm_hd(int shape, const aq_matrix *m, const MmhX &x, int64_t M, float *dst,
                        int splits, int per, float *ysw, hipStream_t s) {
  HdLaunch a{m, {}, (int)(m->cols / 256), x, M, dst, splits, per, ysw, s};
  const int blocks = (int)(m->nb_row / a.ng);  // blocks per group
  auto field = [&](int f, int pl) {
    a.pl.off[f] = (uint32_t)(m->planes.p[pl] - m->dev);
    a.pl.st[f] = (uint32_t)(blocks * m->planes.stride[pl]);
  };
  switch (m->dtype) {
    case AQ_Q4_K:
      field(0, 1);
      field(2, 0);
      return launch_shape<HdKq<false>>(shape, a);
    case AQ_Q5_K:
      field(0, 2);
      field(1, 1);
      field(2, 0);
      return launch_shape<HdKq<true>>(shape, a);
    case AQ_Q6_K:
      field(0, 0);
      field(1, 1);
      field(2, 2);
      a.pl.off[3] = (uint32_t)(m->planes.p[3] - m->dev);
      return launch_shape<HdQ6>(shape, a);
    case AQ_Q8_0:
      field(0, 0);
      field(2, 1);
      return launch_shape<HdB32<32, false, false, 128>>(shape, a);
    case AQ_Q4_0:
      field(0, 0);
      field(2, 1);
      return launch_shape<HdB32<16, false, false, 8>>(shape, a);
    case AQ_Q4_1:
      field(0, 0);
      field(2, 1);
      return launch_shape<HdB32<16, false, true, 0>>(shape, a);
    case AQ_Q5_0:
      field(0, 0);
      field(1, 1);
      field(2, 2);
      return launch_shape<HdB32<16, true, false, 16>>(shape, a);
    case AQ_Q5_1:
      field(0, 0);
      field(1, 1);
      field(2, 2);
      return launch_shape<HdB32<16, true, true, 0>>(shape, a);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace aq
