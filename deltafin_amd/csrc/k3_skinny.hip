// Skinny products y[p, r] = sum_c W[r, c] x[p, c] on the BF16 matrix cores
// (v_mfma_f32_16x16x32_bf16) for a few activation rows and a resident weight
// matrix stored as BF16 bits, row-scaled int8 or MXFP4, in one launch with no
// scratch memory: the spine projections, one expert or one MXFP4 matrix against a
// batch of rows.  An output is summed in one order whatever the number of rows
// beside it: the split and the order of a row's lines follow from its length.
//
// Exactness.  An fp32 activation is split in registers into three BF16 terms
// by truncation (the top 8 significant bits, the next 8, the last 8).  The two
// lower terms are kept times 2^16 (kLowScale), which the sums' last step takes
// back: unscaled they fall under BF16's smallest subnormal (2^-133) from
// |x| < 2^-110 on, which lost 7e-5 of the result at 2^-120 (the multiply costs
// 7168 x 6144 int8 at 16 positions 16.2 -> 16.7 us).  Scaled, the terms
// sum to every finite fp32 value below 2^119 exactly, subnormals included (above,
// the scaled remainder may overflow: see below).  BF16, int8 and scaled E2M1
// weights are exact in BF16 and BF16 x BF16 products are exact in fp32 (the
// matrix cores keep subnormal operands and sums), so only the summation order
// differs from an fp32 FMA kernel.  Where a term product is not finite although
// the fp32 sum may be (an infinite activation has a NaN remainder, an infinite
// weight meets a zero term, a scaled code or remainder overflows), the output
// comes out non-finite and the epilogue forms it again in plain fp32.
//
// Layout.  A wave reads whole 128-byte lines: one dwordx4 load covers 8 weight
// rows x one line (lane l: row (l % 16) / 2 of the 8, 16-byte piece 4 (l % 2) +
// l / 16), which streams at 7.0 TB/s on MI355X against 3.7 TB/s for 16 rows x
// half a line.  Two such loads are one tile of 16 rows; neighbouring lanes
// exchange halves (one DPP step) so that the first register holds the first
// half line of all 16 rows and the second the second.  MFMA row m of a tile is
// then weight row (m % 2) 8 + m / 2.  A lane's 16 bytes are 8, 16 or 32
// columns; for int8 and MXFP4 permlane swaps hand lane group g = l / 16 the
// columns 32 q + 8 g .. + 7 of operand q, so that every operand meets a
// contiguous run of 32 activation columns and the activation loads touch one
// 128-byte line per row.
//
// Split.  A workgroup owns TL tiles of rows (with kGlu, of both gate and up)
// and its S waves split the lines of a row; the activation columns a wave
// needs come from the L2 with the weights, two lines in flight each, and the
// S partial tiles meet in LDS.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "k3_device.h"
#include "k3_internal.h"
#include "k3_launch.h"
#include "k3_skinny.h"

namespace k3 {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint64_t u64_unaligned __attribute__((aligned(1)));

constexpr int kMaxWaves = 8;
constexpr float kLowScale = 65536.0f;  // of an fp32 activation's two lower terms

// 32-column operands of a half line.
template <int kW>
constexpr int operands() {
  return kW == SKINNY_BF16 ? 1 : kW == SKINNY_INT8 ? 2 : 4;
}

struct SkinnyArgs {
  const uint8_t* w[2];   // weights; [1] = up with kGlu
  const uint8_t* sc[2];  // MXFP4 scale planes
  const float* rs[2];    // int8 row scales
  const void* x;
  void* y;
  float* y_up;       // kGlu: receives up . x when non-null
  const float* add;  // added to an fp32 result when non-null
  int rows, cols, P;
  int lines;      // 128-byte lines of a row, the last one possibly partial
  int tail;       // bytes of the last line
  int S, per;     // waves splitting the lines, lines of a wave
  int out_bf16, act;
};

// Activation blocks: 256 bytes of each row, operands of one block and blocks
// of one weight line.
template <typename XT>
constexpr int block_operands() {
  return 8 / (int)sizeof(XT);
}
template <int kW, typename XT>
constexpr int line_blocks() {
  return 2 * operands<kW>() / block_operands<XT>();
}

// A block goes to LDS as loaded (BF16 activations; fp32 ones of four row quads
// or more) or as its three terms: splitting before the store splits every value
// once instead of once per 16 columns of the operand read, which pays while the
// rows are fewer than those columns; a split row costs 6 bytes of LDS traffic
// each way instead of 4.
template <typename XT, int RQ>
constexpr bool raw_blocks() {
  return sizeof(XT) == 2 || RQ >= 4;
}
// 16-byte LDS slots of a block.
template <typename XT, int RQ>
constexpr int block_f4() {
  return RQ * 4 * 16 * (raw_blocks<XT, RQ>() ? 2 : 3) / 2;
}

// One line's worth of loads.
template <int kW, typename XT, int RQ, int TLT>
struct Stage {
  u32x4 a[TLT][2];
  u32x4 x[line_blocks<kW, XT>()][RQ];
  uint64_t s[kW == SKINNY_FP4 ? TLT : 1];
};

__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

__device__ __forceinline__ bf16x8 pack8(const uint32_t (&d)[4]) {
  return __builtin_bit_cast(bf16x8, u32x4{d[0], d[1], d[2], d[3]});
}

// High halves of two fp32 values as a BF16 pair (b in the high half).
__device__ __forceinline__ uint32_t hi_pair(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// The weight operands of one half line: o[q] = columns 32 q + 8 g .. + 7.
__device__ __forceinline__ void weight_operands(u32x4 w, uint32_t, bf16x8 (&o)[1]) {
  o[0] = __builtin_bit_cast(bf16x8, w);
}

__device__ __forceinline__ void weight_operands(u32x4 w, uint32_t, bf16x8 (&o)[2]) {
  uint32_t d[4] = {w.x, w.y, w.z, w.w};
  swap16(d[0], d[2]);
  swap16(d[1], d[3]);
  swap32(d[0], d[2]);
  swap32(d[1], d[3]);
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    uint32_t p[4];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint32_t v = d[2 * q + e];
      uint32_t f[4];
#pragma unroll
      for (int b = 0; b < 4; ++b)
        f[b] = __float_as_uint((float)((int32_t)(v << (24 - 8 * b)) >> 24));
      p[2 * e] = hi_pair(f[0], f[1]);
      p[2 * e + 1] = hi_pair(f[2], f[3]);
    }
    o[q] = pack8(p);
  }
}

// s: the four E8M0 bytes of the row's half line, byte q that of operand q.
// The convert takes the exponent field of its scale operand: byte 255 there is
// NaN, and byte 0, whose value is +0, zeroes the codes instead.
__device__ __forceinline__ void weight_operands(u32x4 w, uint32_t s, bf16x8 (&o)[4]) {
  uint32_t d[4] = {w.x, w.y, w.z, w.w};
  swap32(d[0], d[2]);
  swap32(d[1], d[3]);
  swap16(d[0], d[1]);
  swap16(d[2], d[3]);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float f = __uint_as_float((q < 3 ? s << (23 - 8 * q) : s >> 1) & 0x7f800000u);
    const uint32_t v = __float_as_uint(f) == 0u ? 0u : d[q];
    const v2bf c0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, f, 0);
    const v2bf c1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, f, 1);
    const v2bf c2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, f, 2);
    const v2bf c3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, f, 3);
    o[q] = bf16x8{c0.x, c0.y, c1.x, c1.y, c2.x, c2.y, c3.x, c3.y};
  }
}

// Four fp32 values -> three truncated BF16 terms each, the second and third
// times kLowScale.
__device__ __forceinline__ void split4(u32x4 v, uint2 (&t)[3]) {
  uint32_t w[3][2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const uint32_t u0 = v[2 * e], u1 = v[2 * e + 1];
    const float r0 = (__uint_as_float(u0) - __uint_as_float(u0 & 0xffff0000u)) * kLowScale;
    const float r1 = (__uint_as_float(u1) - __uint_as_float(u1 & 0xffff0000u)) * kLowScale;
    const uint32_t m0 = __float_as_uint(r0), m1 = __float_as_uint(r1);
    const float l0 = r0 - __uint_as_float(m0 & 0xffff0000u);
    const float l1 = r1 - __uint_as_float(m1 & 0xffff0000u);
    w[0][e] = hi_pair(u0, u1);
    w[1][e] = hi_pair(m0, m1);
    w[2][e] = hi_pair(__float_as_uint(l0), __float_as_uint(l1));
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) t[i] = make_uint2(w[i][0], w[i][1]);
}

// Up to four outputs of one activation row x in plain fp32 (see Exactness above),
// by a whole wave: lane l takes the rows' 16-byte pieces l, l + 64, ..., so that x
// is read once for the four rows and every load is a run of whole lines.  A
// position with an infinity or NaN forms all of its outputs here: 7168 x 6144 at
// 16 such positions takes 175 us (BF16) and 113 (int8), 21 and 17 being the
// finite call's; one thread per output took 1.46 ms.
template <int kW, typename XT>
__device__ __forceinline__ void plain_dots(const uint8_t* w, const uint8_t* sc, const XT* x,
                                           const int (&row)[4], int cols, int lane,
                                           float (&sum)[4]) {
  constexpr int C = 32 * operands<kW>() / 4;  // columns of a piece
  const int pieces = cols / C;
#pragma unroll
  for (int r = 0; r < 4; ++r) sum[r] = 0.0f;
  constexpr int kUnroll = kW == SKINNY_FP4 ? 1 : 2;  // within the main loop's registers
#pragma unroll kUnroll
  for (int c = lane; c < pieces; c += 64) {
    u32x4 wv[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) wv[r] = load_chunk(w + ((uint64_t)row[r] * pieces + c) * 16);
    float xv[C];
    constexpr int E = 16 / (int)sizeof(XT);  // activations of a 16-byte load
#pragma unroll
    for (int i = 0; i < C / E; ++i) {
      const u32x4 v = *(gu32x4*)(x + (uint64_t)C * c + E * i);
#pragma unroll
      for (int e = 0; e < E; ++e)
        xv[E * i + e] = sizeof(XT) == 4 ? __uint_as_float(v[e % 4])
                        : e % 2         ? __uint_as_float(v[e / 2] & 0xffff0000u)
                                        : __uint_as_float(v[e / 2] << 16);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (kW == SKINNY_FP4) {
        float part = 0.0f;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const v2f v0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wv[r][d], 1.0f, 0);
          const v2f v1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wv[r][d], 1.0f, 1);
          const v2f v2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wv[r][d], 1.0f, 2);
          const v2f v3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wv[r][d], 1.0f, 3);
          const float f[8] = {v0.x, v0.y, v1.x, v1.y, v2.x, v2.y, v3.x, v3.y};
#pragma unroll
          for (int e = 0; e < 8; ++e) part = fmaf(f[e], xv[8 * d + e], part);
        }
        sum[r] = fmaf(part, e8m0_scale(sc[(uint64_t)row[r] * pieces + c]), sum[r]);
      } else {
#pragma unroll
        for (int e = 0; e < C; ++e) {
          float f;
          if constexpr (kW == SKINNY_BF16)
            f = __uint_as_float(e % 2 ? wv[r][e / 2] & 0xffff0000u : wv[r][e / 2] << 16);
          else
            f = (float)((int32_t)(wv[r][e / 4] << (24 - 8 * (e % 4))) >> 24);
          sum[r] = fmaf(f, xv[e], sum[r]);
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) sum[r] = wave_sum(sum[r]);
}

// RQ quads of activation rows per workgroup: 4 RQ positions (1..16 of a
// 16-column block, or 32).
template <int kW, typename XT, int RQ, int TL, bool kGlu, int D>
__global__ __launch_bounds__(64 * kMaxWaves) void k_skinny(const SkinnyArgs args) {
  constexpr int Q = operands<kW>();
  constexpr int TLT = kGlu ? 2 * TL : TL;
  constexpr int NB = RQ > 4 ? RQ / 4 : 1;       // 16-position column blocks
  constexpr int NT = sizeof(XT) == 4 ? 3 : 1;   // terms of an activation
  constexpr int OB = block_operands<XT>();
  constexpr int NBK = line_blocks<kW, XT>();
  constexpr int XC = 256 / (int)sizeof(XT);     // columns of a block
  constexpr int kRegions = NBK > 1 ? 2 : 1;
  constexpr bool kRaw = raw_blocks<XT, RQ>();
  constexpr int kTermF4 = RQ * 4 * XC / 8;      // 16-byte slots of a block's term
  constexpr int kWaveF4 = kRegions * block_f4<XT, RQ>();
  extern __shared__ f32x4 part[];  // [S][kWaveF4] blocks, then [S][TLT][NB][64] sums
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i16 = lane & 15, g = lane >> 4;
  const bool odd = (i16 & 1) != 0;
  const int r0 = blockIdx.x * 16 * TL;
  const int p0 = blockIdx.y * 4 * RQ;
  const int rows = args.rows, P = args.P, S = args.S;
  const uint32_t row_bytes = kW == SKINNY_BF16   ? 2u * args.cols
                             : kW == SKINNY_INT8 ? (uint32_t)args.cols
                                                 : (uint32_t)args.cols >> 1;
  const int G = args.cols >> 5;  // MXFP4 scales of a row
  // this wave's lines [j0, j1)
  const int j0 = min(wave * args.per, args.lines);
  const int j1 = min(j0 + args.per, args.lines);

  // Lane offsets from wave-uniform bases: rows past the last one re-read it,
  // positions past the last one re-read it (neither is stored).
  const uint32_t piece = 64u * (i16 & 1) + 16u * g;
  uint32_t aoff[TL][2], soff[kW == SKINNY_FP4 ? TL : 1];
  const int last = rows - 1 - r0;
#pragma unroll
  for (int t = 0; t < TL; ++t) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      aoff[t][h] = (uint32_t)min(16 * t + 8 * h + (i16 >> 1), last) * row_bytes + piece;
    if constexpr (kW == SKINNY_FP4)
      soff[t] = (uint32_t)min(16 * t + 8 * (i16 & 1) + (i16 >> 1), last) * (uint32_t)G;
  }
  // Activation loads: a quarter wave reads one row's 256 bytes of a block.
  uint32_t xoff[RQ];
#pragma unroll
  for (int n = 0; n < RQ; ++n)
    xoff[n] = (uint32_t)min(p0 + 4 * n + g, P - 1) * (uint32_t)args.cols * (uint32_t)sizeof(XT);
  const uint8_t* xb = static_cast<const uint8_t*>(args.x);
  const uint8_t* wb[2];
  const uint8_t* sb[2];
#pragma unroll
  for (int m = 0; m < (kGlu ? 2 : 1); ++m) {
    wb[m] = args.w[m] + (uint64_t)r0 * row_bytes;
    if constexpr (kW == SKINNY_FP4) sb[m] = args.sc[m] + (uint64_t)r0 * (uint32_t)G;
  }
  const int tail_line = args.tail < 128 ? args.lines - 1 : -1;
  const bool tail_out = piece >= (uint32_t)args.tail;  // a piece past a partial line

  typedef Stage<kW, XT, RQ, TLT> St;
  // Pieces past the row's end (a partial last line) read the row's first piece
  // and meet zero weights.
  auto load_x = [&](St& s, int j) {
#pragma unroll
    for (int b = 0; b < NBK; ++b) {
      const uint32_t k = (uint32_t)(j * NBK + b) * XC + (16 / sizeof(XT)) * i16;
      const uint32_t ko = j == tail_line && k >= (uint32_t)args.cols ? 0u : k * sizeof(XT);
#pragma unroll
      for (int n = 0; n < RQ; ++n) s.x[b][n] = *(gu32x4*)(xb + (xoff[n] + ko));
    }
  };
  auto load_a = [&](St& s, int j) {
    const uint32_t back = j == tail_line && tail_out ? piece : 0u;
    if constexpr (kW == SKINNY_FP4) {
      const uint32_t so = min(8u * (uint32_t)j, (uint32_t)G - 8u);
#pragma unroll
      for (int t = 0; t < TLT; ++t)
        s.s[t] = *(__attribute__((address_space(1))) const u64_unaligned*)(sb[t / TL] + so +
                                                                            soff[t % TL]);
    }
#pragma unroll
    for (int t = 0; t < TLT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        s.a[t][h] = load_chunk(wb[t / TL] + 128u * (uint32_t)j + (aoff[t % TL][h] - back));
  };
  // Block b of a stage into the wave's LDS region.  16-byte piece c of row r is
  // at slot 16 r + (c ^ r % 16) (raw) or, of each term, 8 r + (c ^ (r / 2) % 8), so
  // that both the row-wise stores and the column-wise operand reads spread over
  // all banks.  A wave's LDS operations run in order, so no barrier is needed.
  f32x4* mine = part + wave * kWaveF4;
  auto slot = [](int r, int c) {
    return kRaw ? 16 * r + (c ^ (r & 15)) : 8 * r + (c ^ ((r >> 1) & 7));
  };
  auto put_block = [&](const St& s, int b) {
    f32x4* r = mine + (b & (kRegions - 1)) * block_f4<XT, RQ>();
#pragma unroll
    for (int n = 0; n < RQ; ++n) {
      if constexpr (kRaw) {
        r[slot(4 * n + g, i16)] = __builtin_bit_cast(f32x4, s.x[b][n]);
      } else {
        uint2 t[3];
        split4(s.x[b][n], t);
#pragma unroll
        for (int i = 0; i < 3; ++i)
          reinterpret_cast<uint2*>(r + i * kTermF4 + slot(4 * n + g, i16 >> 1))[i16 & 1] = t[i];
      }
    }
    __builtin_amdgcn_wave_barrier();
  };

  // Sums: fp32 activations keep the leading terms of a line's two halves and
  // the lower terms apart, BF16 ones the even and odd operands of each half, so
  // that each sum rounds a few times only (one sum for all: 3.3e-7 of the
  // result at 3584 x 7168 against 1.3e-7, and 2.0e-7 for the fp32 kernels).
  constexpr int NA = NT > 1 ? 3 : 4;
  f32x4 acc[TLT][NB][NA];
#pragma unroll
  for (int t = 0; t < TLT; ++t)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int c = 0; c < NA; ++c) acc[t][nb][c] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](St& s, int j) {
    if (j == tail_line && tail_out) {
#pragma unroll
      for (int t = 0; t < TLT; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) s.a[t][h] = u32x4{0u, 0u, 0u, 0u};
    }
    put_block(s, 0);
#pragma unroll
    for (int t = 0; t < TLT; ++t) pair_halves(s.a[t], odd);
    uint64_t sw[TLT];
    if constexpr (kW == SKINNY_FP4) {
      // the clamped scale load of a partial line starts up to 7 bytes early
      const int early = 8 * max(8 * j - (G - 8), 0);
#pragma unroll
      for (int t = 0; t < TLT; ++t) sw[t] = s.s[t] >> early;
    }
    bf16x8 wo[TLT][Q];
#pragma unroll
    for (int b = 0; b < NBK; ++b) {
      if (b + 1 < NBK) put_block(s, b + 1);
      const f32x4* r = mine + (b & (kRegions - 1)) * block_f4<XT, RQ>();
#pragma unroll
      for (int o = 0; o < OB; ++o) {
        const int h = (b * OB + o) / Q, q = (b * OB + o) % Q;
        if (q == 0) {
#pragma unroll
          for (int t = 0; t < TLT; ++t)
            weight_operands(s.a[t][h], kW == SKINNY_FP4 ? (uint32_t)(sw[t] >> (32 * h)) : 0u,
                            wo[t]);
        }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          // rows past the staged ones repeat an earlier one (not stored)
          const int row = RQ < 4 ? i16 & (4 * RQ - 1) : i16;
          bf16x8 xt[NT];
          if constexpr (kRaw && NT == 3) {
            uint2 lo[3], hi[3];
            split4(__builtin_bit_cast(u32x4, r[slot(16 * nb + row, 8 * o + 2 * g)]), lo);
            split4(__builtin_bit_cast(u32x4, r[slot(16 * nb + row, 8 * o + 2 * g + 1)]), hi);
#pragma unroll
            for (int i = 0; i < NT; ++i)
              xt[i] = __builtin_bit_cast(bf16x8, u32x4{lo[i].x, lo[i].y, hi[i].x, hi[i].y});
          } else {
#pragma unroll
            for (int i = 0; i < NT; ++i)
              xt[i] = __builtin_bit_cast(bf16x8, r[i * kTermF4 + slot(16 * nb + row, 4 * o + g)]);
          }
#pragma unroll
          for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int t = 0; t < TLT; ++t) {
              f32x4& d = acc[t][nb][NT > 1 ? (i > 0 ? 2 : h) : 2 * h + (q & 1)];
              d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wo[t][q], xt[i], d, 0, 0, 0);
            }
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  };

  if (j0 < j1) {
    // D lines in flight; a stage is refilled with the line D further on as soon
    // as it is used (past the wave's range: its last line again, so that every
    // load is unconditional and the wait counts stay exact).
    St st[D];
    auto load_stage = [&](St& s, int j) {
      load_x(s, j);
      load_a(s, j);
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load_stage(st[d], min(j0 + d, j1 - 1));
    int j = j0;
    for (; j + D < j1; j += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        compute(st[d], j + d);
        __builtin_amdgcn_sched_barrier(0);
        load_stage(st[d], min(j + d + D, j1 - 1));
      }
    }
    // the last 1..D lines (no exits inside the loop above: their paths, which
    // load nothing more, would merge into the wait counts at its head)
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (j + d < j1) compute(st[d], j + d);
  }

  f32x4* sums = part + S * kWaveF4;
#pragma unroll
  for (int t = 0; t < TLT; ++t)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      f32x4 v = acc[t][nb][0] + acc[t][nb][1];
#pragma unroll
      for (int c = 2; c < NA; ++c) v += NT > 1 ? acc[t][nb][c] * (1.0f / kLowScale) : acc[t][nb][c];
      sums[((wave * TLT + t) * NB + nb) * 64 + lane] = v;
    }
  __syncthreads();
  const int np = min(4 * RQ, P - p0);
  const float* pf = reinterpret_cast<const float*>(sums);
  const int n_out = 16 * TL * np;
  for (int o0 = 64 * wave; o0 < n_out; o0 += 64 * S) {
    const int o = min(o0 + lane, n_out - 1);
    const int rt = o % (16 * TL), p = o / (16 * TL);
    const int row = r0 + rt;
    const bool stored = o0 + lane < n_out && row < rows;
    const int t = rt >> 4, wr = rt & 15;
    const int m = wr < 8 ? 2 * wr : 2 * wr - 15;  // MFMA row of weight row wr
    const int at = (t * NB + (p >> 4)) * 256 + (16 * (m >> 2) + (p & 15)) * 4 + (m & 3);
    float v[kGlu ? 2 : 1];
#pragma unroll
    for (int k = 0; k < (kGlu ? 2 : 1); ++k) {
      const float* pk = pf + at + k * TL * NB * 256;
      float sum = 0.0f;
#pragma unroll
      for (int w = 0; w < kMaxWaves; ++w)  // wave order; all reads in flight at once
        if (w < S) sum += pk[w * TLT * NB * 256];
      // non-finite sums again, by the whole wave, four rows of one position at a time
      uint64_t left = __ballot(stored && !(fabsf(sum) < INFINITY));
      while (left != 0) {
        const int first = __builtin_ctzll(left);
        const int bp = (o0 + first) / (16 * TL);
        int bit[4], brow[4];
        float again[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int b = left != 0 ? __builtin_ctzll(left) : first;
          bit[i] = (o0 + b) / (16 * TL) == bp ? b : first;
          brow[i] = r0 + (o0 + bit[i]) % (16 * TL);
          left &= ~(1ull << bit[i]);
        }
        plain_dots<kW, XT>(args.w[k], args.sc[k],
                           static_cast<const XT*>(args.x) + (uint64_t)(p0 + bp) * args.cols, brow,
                           args.cols, lane, again);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (lane == bit[i]) sum = again[i];
      }
      if constexpr (kW == SKINNY_INT8) sum *= stored ? args.rs[k][row] : 0.0f;
      v[k] = sum;
    }
    if (!stored) continue;
    const uint64_t yi = (uint64_t)(p0 + p) * rows + row;
    float out = v[0];
    if constexpr (kGlu) {
      if (args.y_up) args.y_up[yi] = v[1];
      out = activate(args.act, v[0], v[1]);
    }
    if (args.out_bf16) {
      static_cast<uint16_t*>(args.y)[yi] = f32_to_bf16_bits(out);
    } else {
      if (!kGlu && args.add) out = args.add[yi] + out;
      static_cast<float*>(args.y)[yi] = out;
    }
  }
}

template <int kW, typename XT, int RQ, int TL, bool kGlu, int D>
bool go(const SkinnyArgs& a, hipStream_t st, TimedLaunch& tl) {
  constexpr int TLT = kGlu ? 2 * TL : TL;
  constexpr int NB = RQ > 4 ? RQ / 4 : 1;
  constexpr int kRegions = line_blocks<kW, XT>() > 1 ? 2 : 1;
  const unsigned lds = (unsigned)(a.S * (TLT * NB * 64 + kRegions * block_f4<XT, RQ>()) *
                                  sizeof(f32x4));
  const void* fn = reinterpret_cast<const void*>(k_skinny<kW, XT, RQ, TL, kGlu, D>);
  if (!lds_fits(fn, 64 * a.S, lds)) return false;
  const dim3 grid((a.rows + 16 * TL - 1) / (16 * TL), (a.P + 4 * RQ - 1) / (4 * RQ));
  launch_timed(tl, (k_skinny<kW, XT, RQ, TL, kGlu, D>), grid, dim3(64 * a.S), lds, st, a);
  return true;
}

// Lines in flight per wave: two, except for MXFP4 from two tiles up, whose lines
// bring four times the columns of BF16 ones: there one is as fast or faster (7168
// x 2048, 7 rows: 5.8 us against 6.7; one expert at 7 rows with one / two in its
// gate/up: 3584 / 3072 16.4 / 16.5, 7168 / 2048 21.0 / 20.5, 7168 / 7168 37.4 /
// 41.7).  Three, four and six lines of one BF16 or int8 tile measured the same or
// slower than two (896 x 7168, 8 rows, BF16: 11.2 at two, 12.4 at four, 13.7 at
// six), one line slower at few workgroups (3584 x 7168 BF16, 1 row: 14.4 against
// 10.5).  Four tiles, and two of gate and two of up, need 158 to 231 registers:
// one workgroup per CU.
template <int kW, int TL>
constexpr int depth() {
  return kW == SKINNY_FP4 && TL > 1 ? 1 : 2;
}

template <int kW, typename XT, int RQ>
bool go_tiles(int TL, const SkinnyArgs& a, hipStream_t st, TimedLaunch& tl) {
  if (TL == 1) return go<kW, XT, RQ, 1, false, depth<kW, 1>()>(a, st, tl);
  if (TL == 2) return go<kW, XT, RQ, 2, false, depth<kW, 2>()>(a, st, tl);
  return go<kW, XT, RQ, 4, false, depth<kW, 4>()>(a, st, tl);
}

template <int kW, typename XT>
bool go_rows(int TL, const SkinnyArgs& a, hipStream_t st, TimedLaunch& tl) {
  if (a.P <= 4) return go_tiles<kW, XT, 1>(TL, a, st, tl);
  if (a.P <= 8) return go_tiles<kW, XT, 2>(TL, a, st, tl);
  if constexpr (kW == SKINNY_BF16)
    // 32 positions per workgroup where four tiles of 16 would be next: 12288 x
    // 7168 at 64 positions 90.9 us against 108.8 (int8 and MXFP4 lines, with
    // more columns, would spill)
    if (a.P > 16 && TL == 4) return go<kW, XT, 8, 2, false, depth<kW, 2>()>(a, st, tl);
  return go_tiles<kW, XT, 4>(TL, a, st, tl);
}

// Tiles of gate and as many of up: two of each where one would leave more
// workgroups than CUs (MXFP4, with its longer lines, always one).
template <int kW, int RQ>
bool go_glu_tiles(int TL, const SkinnyArgs& a, hipStream_t st, TimedLaunch& tl) {
  if constexpr (kW != SKINNY_FP4)
    if (TL > 1) return go<kW, float, RQ, 2, true, 2>(a, st, tl);
  return go<kW, float, RQ, 1, true, depth<kW, 2>()>(a, st, tl);
}

template <int kW>
bool go_glu(int TL, const SkinnyArgs& a, hipStream_t st, TimedLaunch& tl) {
  if (a.P <= 4) return go_glu_tiles<kW, 1>(TL, a, st, tl);
  if (a.P <= 8) return go_glu_tiles<kW, 2>(TL, a, st, tl);
  return go_glu_tiles<kW, 4>(TL, a, st, tl);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace

bool skinny_fits(const SkinnyOp& op) {
  const int per = op.kind == SKINNY_BF16 ? 8 : op.kind == SKINNY_INT8 ? 16 : 32;
  const uint64_t row_bytes = op.kind == SKINNY_BF16   ? 2ull * op.cols
                             : op.kind == SKINNY_INT8 ? (uint64_t)op.cols
                                                      : (uint64_t)op.cols / 2;
  return op.rows > 0 && op.positions > 0 && op.cols > 0 && op.cols % per == 0 &&
         row_bytes >= (op.kind == SKINNY_FP4 ? 128u : 64u) && op.cols <= 65536 &&
         op.positions <= (1 << 19) && (uint64_t)op.positions * op.cols <= (1u << 28) &&
         (uint64_t)op.positions * op.rows <= INT32_MAX && aligned16(op.w) && aligned16(op.x) &&
         (!op.w2 || (aligned16(op.w2) && op.x_dtype == K3_DTYPE_F32)) &&
         !(op.add && (op.w2 || op.out_bf16));
}

int launch_skinny(const SkinnyOp& op, int kernel_class, hipStream_t st) {
  SkinnyArgs a{};
  a.w[0] = static_cast<const uint8_t*>(op.w);
  a.w[1] = static_cast<const uint8_t*>(op.w2);
  a.sc[0] = op.scales;
  a.sc[1] = op.scales2;
  a.rs[0] = op.row_scales;
  a.rs[1] = op.row_scales2;
  a.add = op.add;
  a.x = op.x;
  a.y = op.y;
  a.y_up = op.y_up;
  a.rows = op.rows;
  a.cols = op.cols;
  a.P = op.positions;
  a.out_bf16 = op.out_bf16;
  a.act = op.act;
  const int row_bytes = op.kind == SKINNY_BF16 ? 2 * op.cols : op.kind == SKINNY_INT8 ? op.cols
                                                                                  : op.cols / 2;
  a.lines = (row_bytes + 127) / 128;
  a.tail = row_bytes - 128 * (a.lines - 1);
  // Eight waves split a row's lines (16 measured the same or slower, also at few
  // rows: 896 x 7168 BF16 at 1 / 8 / 16 positions 9.2 / 12.7 / 16.3 us against 9.0 /
  // 11.2 / 15.0; 4 slower at long rows).
  a.per = (a.lines + kMaxWaves - 1) / kMaxWaves;
  a.S = (a.lines + a.per - 1) / a.per;
  // The fewest tiles per workgroup that leave no more workgroups than CUs, up to
  // four: every workgroup reads and splits all of its positions' activation,
  // and a second workgroup on some CUs only lengthens the launch.  BF16, 16
  // positions, us at 1 / 2 / 4 tiles: 3584 x 7168 16.7 / 20.3 / 29.4 (224
  // workgroups at 1), 4352 x 7168 27.6 / 20.9 / 29.7 (136 at 2), 7168 x 6144
  // 26.0 / 20.7 / 28.1 (224 at 2), 8704 x 7168 40.7 / 38.8 / 32.0 (136 at 4).
  const int cus = std::max(1, device_cu_count());
  const int pb = (a.P + 15) / 16;
  int TL = 1;
  while (TL < 4 && (int64_t)((a.rows + 16 * TL - 1) / (16 * TL)) * pb > cus) TL *= 2;
  TimedLaunch tl(kernel_class, st);
  bool ok;
  const bool glu = op.w2 != nullptr;
  if (op.kind == SKINNY_BF16)
    ok = glu ? go_glu<SKINNY_BF16>(TL, a, st, tl) : go_rows<SKINNY_BF16, float>(TL, a, st, tl);
  else if (op.kind == SKINNY_INT8)
    ok = glu ? go_glu<SKINNY_INT8>(TL, a, st, tl) : go_rows<SKINNY_INT8, float>(TL, a, st, tl);
  else if (op.x_dtype == K3_DTYPE_F32)
    ok = glu ? go_glu<SKINNY_FP4>(TL, a, st, tl) : go_rows<SKINNY_FP4, float>(TL, a, st, tl);
  else
    ok = go_rows<SKINNY_FP4, uint16_t>(TL, a, st, tl);
  if (!ok) {
    tl.failed();
    return fail(K3_HIP_E_EXEC, "skinny product: %d waves of partial tiles do not fit in LDS", a.S);
  }
  return launched(tl, "skinny product launch");
}

}  // namespace k3
