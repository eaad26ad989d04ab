// q1_digits.h — the N-column Q1_0 products (prefill, speculative verify) on gfx950's scaled 4/6-bit
// matrix instruction: matvec_batch_into_slice / matvec_add_batch_into_slice
// (Daiza-engine/src/model/weights.rs:475-682, 976-980).
//
// Numerics.  A weight is ±scale with one f16 scale per row and 128-column group, so the group's sum
// is scale · Σ ±x.  The signs are f4 (e2m1) operands, ±1 exactly.  An activation is a fixed-point
// number of six balanced base-32 digits relative to its block of 32 columns: with 2^e > max|x| >=
// 2^(e-1) over the block, v = x · 2^(4-e) lies in [-16, 16] and
//   v = d0 + d1/32 + ... + d5/32^5 + rest,   |d_i| <= 16 whole, |rest| <= 2^-26 (at most 2^-29 of the largest v)
// An integer d of that range is an f6 (e2m3) value in units of 1/8 exactly (codes 0..16 of the
// magnitude are the integers 0..16), and the power of two of a digit is the block scale (e8m0) of
// the matrix instruction.  v_mfma_scale_f32_16x16x128_f8f6f4 therefore sums 128 exact products per
// digit into an f32 accumulator; digits go in from the smallest to the largest, then the group's sum
// is multiplied by the f16 scale as it is added (one fma per group, where a three-part f16 split of
// the activations takes twelve f32 additions per group).  Six digits carry every bit of an f32 whose
// exponent is within 5 of its block's largest; smaller values are rounded to a grid of 2^-29 of the
// block's largest, beneath the rounding of an f32 dot product.  Errors of a 2048 x 5120 product against 64
// bits (2-norm; n = 2, 8 and 128 columns) with three f16 parts and with digits:
//   standard normal columns                            1.6e-7  1.6e-7  2.2e-7    0.8e-7  0.8e-7  0.8e-7
//   normal · e^(3 normal)                              1.7e-7  2.0e-7  2.1e-7    0.8e-7  0.7e-7  0.8e-7
//   two of about 2^14 that cancel in every group       2.2e-4  2.2e-4  2.6e-4    0.8e-7  1.2e-5  2.4e-4
// A block that holds an infinity or a NaN gets the NaN scale (0xFF), so its token's results are NaN.
//
// Rate.  The instruction runs at four times the f16 rate (measured 9.1 ns per 16x16x128 per SIMD,
// 7.4 PFLOP/s over the device); six of them replace the twelve f16 ones (4 steps of 32 columns x 3
// parts) of the same group, at half their cycles each: a quarter of the matrix time, and a quarter of
// the sign expansion (7 VALU operations per 32 signs).  Measured at n = 1024 against the f16 form it
// replaced: 34816 x 5120 865 -> 447 us, 16480 x 5120 457 -> 248, 5120 x 17408 565 -> 267 (with the
// split sum), 5120 x 6144 204 -> 135; error against 64 bits of a four-layer block 4.3e-6 -> 0.9e-6.
#pragma once
#include "q1_gemv.h"

namespace dz {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x6 __attribute__((ext_vector_type(6)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kDigits = 6;

// The signs' block scale, 2^-7: a group's 128 terms then sum without overflow whatever they are, as they do when
// the f16 scale comes first; kSignUp takes it back where the row's sum is stored (both exact).
constexpr int kSignScale = 0x78;
constexpr float kSignUp = 128.0f;

// 32 signs (bit 4j + k of w = element 8k + j) as f4 values: bit set -> +1 (0x2), clear -> -1 (0xA).
__device__ __forceinline__ void expand_f4(unsigned w, i32x8& a) {
#pragma unroll
  for (int k = 0; k < 4; ++k) a[k] = (int)(((w << (3 - k)) & 0x88888888u) ^ 0xAAAAAAAAu);
}

// Digit 0's block scale of a block whose largest |value| has the bits mb, and the exponent e its values are
// taken by (v = x · 2^(4-e)).  The scales go down to the last of the D digits', 5 (D - 1) below digit 0's,
// and have to stay block scales (>= 0): a block whose largest value is below 2^(5D - 132) is held to 2^-131 absolute.
template <int D>
__device__ __forceinline__ unsigned digit_scale(unsigned mb, int& e) {
  constexpr int lo = 5 * (D - 1) - 126;
  e = 0;
  if (mb >= 0x7F800000u) return 0xFFu;  // an infinity or a NaN in the block
  (void)frexpf(__builtin_bit_cast(float, mb), &e);
  e = mb == 0 ? 0 : (e < lo ? lo : e);
  return (unsigned)(126 + e);
}

// 32 whole numbers of at most 16 as f6 codes: element 2i is ra[i], 2i + 1 is rb[i], each over 8 (code n for n).
// The conversion writes its result while it still reads its sources, and the compiler does not keep them apart: where
// the last digit's result took its sources' registers, that digit came out wrong for a wave now and then (up to 2^-24 of
// the block's largest value, from one run to the next).  The statement below needs all three at once.
__device__ __forceinline__ u32x6 digit_codes(const f32x16& ra, const f32x16& rb) {
  u32x6 d = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(ra, rb, 8.0f);
  asm("" : "+v"(d) : "v"(ra), "v"(rb));
  return d;
}

// The six digit operands and digit 0's block scale of 32 values (column order).
__device__ __forceinline__ unsigned pack_digits(const float (&x)[32], u32x6 (&d)[kDigits]) {
  unsigned mb = 0;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const unsigned b = __builtin_bit_cast(unsigned, x[i]) & 0x7FFFFFFFu;
    mb = b > mb ? b : mb;
  }
  int e;
  const unsigned b0 = digit_scale<kDigits>(mb, e);
  const bool finite = b0 != 0xFFu;
  f32x16 a, b;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int c = 8 * (i & 3) + (i >> 2);
    a[i] = finite ? ldexpf(x[c], 4 - e) : 0.f;
    b[i] = finite ? ldexpf(x[c + 4], 4 - e) : 0.f;
  }
#pragma unroll
  for (int k = 0; k < kDigits; ++k) {
    f32x16 ra, rb;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      ra[i] = __builtin_rintf(a[i]);
      rb[i] = __builtin_rintf(b[i]);
      a[i] = (a[i] - ra[i]) * 32.0f;
      b[i] = (b[i] - rb[i]) * 32.0f;
    }
    d[k] = digit_codes(ra, rb);
  }
  return b0;
}

// ---- few columns (n <= 16): every workgroup packs the tiles it needs itself ----
//
// The 16 rows of the token operand hold T tokens x P = 16/T digits (row ρ = p·T + token, digit f·P + p of
// operand f), so a group of 128 columns takes F operands and F matrix instructions per 16 weight rows:
//   n <= 2: T = 2, P = 8, F = 1;  n <= 4: T = 4, P = 4, F = 2;  n <= 8: T = 8, P = 2, F = 3;  else T = 16, F = 6
// The first two have room for eight digits and hold eight (activations to 2^-39 of their block's largest), the others
// six.  A weight row's sums of the slots are kept apart until the end and then added.
template <int T>
struct FewForm {
  static constexpr int P = 16 / T;
  static constexpr int F = (kDigits + P - 1) / P;
  static constexpr int D = F * P;  // digits
  // LDS of a tile: [group][operand][block q: 416 B][row ρ: 24 B], the block and group strides chosen so that the
  // writes of the packing (16 blocks at once) meet few banks twice
  static constexpr int kBlk = 16 * 24 + 32;
  static constexpr int kOp = 4 * kBlk;
  static constexpr int kGrp = F * kOp + 32;
  static constexpr int kEx = 4 * kGrp;                            // the block scales: [lane] a byte per group
  static constexpr int kTile = kEx + 256;
};
constexpr int kFewStage = 16 * 36 * 4;  // a wave's 512 staged columns, blocks of 32 padded to 36

template <int CTRL>
__device__ __forceinline__ unsigned dpp_umax(unsigned v) {
  const unsigned o = (unsigned)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, false);
  return o > v ? o : v;
}

// A wave's 512 columns of a token (lane: columns 4·lane and 256 + 4·lane as x0, x1) to the staging area st.
__device__ __forceinline__ void few_stage(float* st, unsigned lane, float4 x0, float4 x1) {
  *reinterpret_cast<float4*>(st + 36 * (lane >> 3) + 4 * (lane & 7u)) = x0;
  *reinterpret_cast<float4*>(st + 36 * (8 + (lane >> 3)) + 4 * (lane & 7u)) = x1;
  __builtin_amdgcn_wave_barrier();  // LDS accesses of one wave complete in order
}

// The value of the next lane of the quad (the last one's own).
__device__ __forceinline__ unsigned dpp_next(unsigned v) {
  return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xF9, 0xF, 0xF, false);  // quad_perm [1,2,3,3]
}

// 512 staged columns split into digits: lane (block blk = lane >> 2, quarter kq) takes columns 4j + kq of its block, elements
// 8kq .. 8kq + 7 of a digit operand: 48 bits.  A block's 24 bytes of a digit leave as three aligned 8-byte pieces,
// each formed with the next lane's bits: put(digit, piece), of which piece kq of the block is lane kq's (kq < 3).
// Returns digit 0's block scale (slot p of an operand lies 5p below its slot 0).
// The packing is a chain of a wave (about 1700 cycles).  Written in parts of 16 and 32 bits at byte 6·kq, misaligned for
// half the lanes, the digits bound the CU's LDS: 2450 cycles per task and wave with four waves packing, 1960 with pieces.
template <int T, class Put>
__device__ __forceinline__ unsigned few_digits(const float* st, unsigned lane, Put&& put) {
  using FF = FewForm<T>;
  const unsigned blk = lane >> 2, kq = lane & 3u;
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = st[36 * blk + 4 * j + kq];
  __builtin_amdgcn_wave_barrier();
  unsigned mb = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const unsigned b = __builtin_bit_cast(unsigned, v[j]) & 0x7FFFFFFFu;
    mb = b > mb ? b : mb;
  }
  mb = dpp_umax<0xB1>(mb);  // the block's four quarters: quad xor 1, xor 2
  mb = dpp_umax<0x4E>(mb);
  int e;
  const unsigned b0 = digit_scale<FF::D>(mb, e);
  // 2^(4-e); 0 for a block that is not finite (its digits do not matter beside the NaN scale, but are formed)
  const float up = __builtin_bit_cast(float, (unsigned)(131 - e) << 23);
  const bool finite = b0 != 0xFFu;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = finite ? v[j] * up : 0.f;
#pragma unroll
  for (int k0 = 0; k0 < FF::D; k0 += 4) {
    // digit k0 + i takes elements 8i .. 8i + 7 of the conversion: element 2m is ra[m], 2m + 1 is rb[m]
    f32x16 ra = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, rb = ra;
#pragma unroll
    for (int i = 0; i < 4 && k0 + i < FF::D; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        // the nearest whole number of v·32^k (|.| <= 16): what adding 3·2^22 leaves
        const float r = __builtin_fmaf(v[j], (float)(1ull << (5 * (k0 + i))), 12582912.f) - 12582912.f;
        v[j] = __builtin_fmaf(r, -1.0f / (float)(1ull << (5 * (k0 + i))), v[j]);
        if (j & 1) rb[4 * i + (j >> 1)] = r;
        else ra[4 * i + (j >> 1)] = r;
      }
    const u32x6 d = digit_codes(ra, rb);
#pragma unroll
    for (int i = 0; i < 4 && k0 + i < FF::D; ++i) {
      const int h = 3 * (i >> 1);
      const unsigned lo = i & 1 ? d[h + 1] >> 16 | d[h + 2] << 16 : d[h], hi = i & 1 ? d[h + 2] >> 16 : d[h + 1] & 0xFFFFu;
      const unsigned nlo = dpp_next(lo), nhi = dpp_next(hi);
      const unsigned w1 = hi | nlo << 16, w2 = nlo >> 16 | nhi << 16;  // lo, w1, w2: this lane's and the next one's
      put(k0 + i, u32x2{kq == 0 ? lo : kq == 1 ? lo >> 16 | w1 << 16 : w1, kq == 0 ? w1 : kq == 1 ? w1 >> 16 | w2 << 16 : w2});
    }
  }
  return b0;
}

// Packs the 512 staged columns of token tok into the LDS tile.
template <int T>
__device__ __forceinline__ void few_pack(unsigned char* tile, const float* st, unsigned lane, int tok) {
  using FF = FewForm<T>;
  const unsigned g = lane >> 4, q = (lane >> 2) & 3u, kq = lane & 3u;
  unsigned char* o = tile + g * FF::kGrp + q * FF::kBlk + 24 * tok + 8 * kq;
  const unsigned b0 = few_digits<T>(st, lane, [&](int k, u32x2 piece) {
    if (kq < 3) *reinterpret_cast<u32x2*>(o + (k / FF::P) * FF::kOp + 24 * (k % FF::P) * T) = piece;
  });
  if (kq == 0) {
#pragma unroll
    for (int p = 0; p < FF::P; ++p) tile[FF::kEx + 4 * (16 * q + p * T + tok) + g] = (unsigned char)(b0 - 5 * p);
  }
}

// A unit's weights in a wave: the signs of (16-row block sb0 + sb, group g) and the rows' four scales.  A wave takes the
// four 16-row blocks of a row-block (SB = 4, sb0 = 0) or two of them (SB = 2, sb0 = 0 or 2).
template <int SB>
struct FewUnit {
  unsigned s[4][SB];  // [g][sb]
  u32x2 sc[SB];
};
template <int SB>
__device__ __forceinline__ void few_load(const __amdgpu_buffer_rsrc_t& wr, int woff, int soff, int unit, int sb0, FewUnit<SB>& u) {
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int sb = 0; sb < SB; ++sb)
      u.s[g][sb] = __builtin_amdgcn_raw_buffer_load_b32(wr, woff, unit + 1024 * (g ^ (sb0 + sb)) + 256 * (sb0 + sb), 0);
#pragma unroll
  for (int sb = 0; sb < SB; ++sb)
    u.sc[sb] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(wr, soff, unit + 128 * (sb0 + sb), 0));
}

// acc[sb] += the unit's products with the tile's digits: slot rows 4q + i of weight row 16·(sb0 + sb) + r.
template <int T, int SB>
__device__ __forceinline__ void few_unit(const unsigned char* tile, unsigned lane, unsigned psel, int sb0, const FewUnit<SB>& u,
                                         f32x4 (&acc)[SB]) {
  using FF = FewForm<T>;
  const unsigned ex = *reinterpret_cast<const unsigned*>(tile + FF::kEx + 4 * lane);
  // operand f's slots: P digits further down than operand f - 1's (no borrow: digit 0's scales are >= 5 (D - 1))
  constexpr unsigned drop = 0x05050505u * (unsigned)FF::P;
  const unsigned char* fl = tile + (lane >> 4) * FF::kBlk + 24 * (lane & 15u);
  // step i: operand F - 1 - i % F of group i / F.  Its digits are read a step before the matrix instructions that use
  // them: read where they are used, every step waited out the LDS (one wave per SIMD; T = 16, four instructions per
  // step: 4900 cycles a unit, with the reads ahead 3600)
  constexpr int STEPS = 4 * FF::F;
  auto read = [&](int i) {
    const u32x2* p = reinterpret_cast<const u32x2*>(fl + (i / FF::F) * FF::kGrp + (FF::F - 1 - i % FF::F) * FF::kOp);
    const u32x2 p0 = p[0], p1 = p[1], p2 = p[2];
    return i32x8{(int)p0.x, (int)p0.y, (int)p1.x, (int)p1.y, (int)p2.x, (int)p2.y, 0, 0};
  };
  // T = 4 and 8: operand 0's sums (the largest digits) start from 0 too and join by an fma.  Added onto the others' in the
  // accumulator, large values that cancel would round those away, to 2^-24 of the values before they cancel (the third
  // line of the errors above: 2.5e-4 at eight columns).
  constexpr bool kApart = T == 4 || T == 8;
  i32x8 a = read(0), b[SB];
  f32x4 d[SB], top[SB];
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int g = i / FF::F, f = FF::F - 1 - i % FF::F;
    const i32x8 an = i + 1 < STEPS ? read(i + 1) : a;
    __builtin_amdgcn_sched_barrier(0);
    if (f == FF::F - 1) {
#pragma unroll
      for (int sb = 0; sb < SB; ++sb) expand_f4(__builtin_amdgcn_perm(u.s[g][sb], u.s[g][sb], psel), b[sb]);
    }
    const int sx = (int)(ex - drop * (unsigned)f);
#pragma unroll
    for (int sb = 0; sb < SB; ++sb) {
      const f32x4 c = f == FF::F - 1 || (kApart && f == 0) ? f32x4{0.f, 0.f, 0.f, 0.f} : d[sb];
      f32x4& o = kApart && f == 0 ? top[sb] : d[sb];
      if (g == 0) o = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[sb], c, 2, 4, 0, sx, 0, kSignScale);
      else if (g == 1) o = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[sb], c, 2, 4, 1, sx, 0, kSignScale);
      else if (g == 2) o = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[sb], c, 2, 4, 2, sx, 0, kSignScale);
      else o = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[sb], c, 2, 4, 3, sx, 0, kSignScale);
    }
    a = an;
    if (f == 0) {
#pragma unroll
      for (int sb = 0; sb < SB; ++sb) {
        const unsigned slot = (unsigned)(g ^ (sb0 + sb));
        const unsigned h = (unsigned)(__builtin_bit_cast(unsigned long long, u.sc[sb]) >> (16 * slot));
        const float sf = (float)__builtin_bit_cast(_Float16, (unsigned short)h);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          acc[sb][v] = __builtin_fmaf(sf, d[sb][v], acc[sb][v]);
          if constexpr (kApart) acc[sb][v] = __builtin_fmaf(sf, top[sb][v], acc[sb][v]);
        }
      }
    }
  }
}

// Adds a weight row's slots: afterwards lane (r, q), register i holds token (4q + i) mod T of row r (T < 4:
// registers 0 and 1 of every lane the two tokens).
template <int T>
__device__ __forceinline__ void few_slots(f32x4& a) {
  if constexpr (T == 2) {
    a[0] += a[2];
    a[1] += a[3];
    a[0] += __shfl_xor(a[0], 16);
    a[1] += __shfl_xor(a[1], 16);
    a[0] += __shfl_xor(a[0], 32);
    a[1] += __shfl_xor(a[1], 32);
  } else if constexpr (T == 4) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      a[v] += __shfl_xor(a[v], 16);
      a[v] += __shfl_xor(a[v], 32);
    }
  } else if constexpr (T == 8) {
#pragma unroll
    for (int v = 0; v < 4; ++v) a[v] += __shfl_xor(a[v], 32);
  }
}

// Activations of the few-column product: x[n][K] f32 with row stride ldx.
struct FewX {
  const float* xf;
  int64_t ldx, K;
  const uint8_t* dig;  // PRE: packed tiles [ntiles][FewForm<T>::kTile] instead (x, nw and ssq unused)
  // with RMSNorm (rmsnorm_into, rmsnorm.rs:17-200): the digits are those of x·nw, and y = inv · W (x·nw) with
  // inv = 1/sqrt(Σx²/K + eps): applied by the kernel when its workgroups see every tile, else by the consumer
  // of the split partials, from the per-split sums of squares ssq[z][ssq_ld] that the first row chunk's
  // workgroups write
  const float* nw;
  float* ssq;
  int ssq_ld;
  float eps;
};
// Packing tasks of a wave whose inputs are requested and staged at once.  Requested one by one behind the weights, each
// task waited a memory round trip: 3300 cycles per task (64 x 128 by 16: four tasks a wave, 8.8 us the launch).
template <int T>
constexpr int kFewAhead = T <= 4 ? 1 : 2;
// (a packed product's tiles come as they are and need no staging area)
template <int T, bool PRE>
__host__ __device__ constexpr size_t few_shmem(int nw, int tps) {
  return (size_t)tps * FewForm<T>::kTile + (PRE ? 0 : (size_t)nw * kFewAhead<T> * kFewStage);
}
// K tiles of a workgroup (its LDS)
constexpr int few_max_tiles(int T) { return T == 16 ? 2 : 4; }

// Grid (ceil(nrb / RB), splits, blocks of 16 tokens), 64·NW threads: workgroup (chunk, z) takes K tiles [z·tps, min(ntiles, (z+1)·tps))
// of RB row-blocks, one per wave, or two waves to a row-block (RB = NW / 2).  The inputs are requested first, the first unit's
// weights behind them, and the packing runs while the weights arrive; one barrier, then every wave goes its own way.  With more
// than one split, workgroup z writes its partial to y + z·zstride.
// At eight tokens a product is bound by latencies: of 34816 x 5120's 15.2 us (packed tiles) about 7 are launch, digits
// and the stores of the partials, 5 the weights (25 MB) and 3 the signs' expansion and the matrix instructions.  The
// f16 form it replaced (three parts, K tiles packed one by one with a barrier each) against this one with packed
// tiles, us per launch in the verify forward: 34816 x 5120 22.7 -> 15.9, 16480 x 5120 15.7 -> 11.7, 5120 x 17408
// 14.2 -> 11.3, 5120 x 6144 7.5 -> 6.6.
//
// PRE: the digits come packed by the kernel that formed the activations: at eight tokens the packing costs 2 to
// 4 us of each product.
// (Registers: about kFewWaves waves run, so a CU rarely holds two of these workgroups; the larger forms that pack their
// own tiles take a few more than two would leave them.)
template <int T, int NW, int RB, bool PRE>
__global__ __launch_bounds__(64 * NW, NW < 8 ? 3 : T >= 4 && RB == 8 && !PRE ? 2 : 4) void q1_few_kernel(const uint8_t* __restrict__ W, int64_t rows, int64_t nrb,
                                                                     int ntiles, int tps, const FewX x, int n_tok,
                                                                     float* __restrict__ y, int64_t ldy, int64_t zstride,
                                                                     int accumulate) {
  using FF = FewForm<T>;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ float ssqs[few_max_tiles(T)][T];
  const unsigned tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, q = lane >> 4;
  const int wave = (int)__builtin_amdgcn_readfirstlane(tid >> 6);
  // token block blockIdx.z: 16 columns of a product with more
  const int tb = 16 * (int)blockIdx.z;
  n_tok = min(n_tok - tb, 16);
  const int t0 = (int)blockIdx.y * tps, nt = min(ntiles - t0, tps);
  constexpr int SB = 4 * RB / NW;  // 16-row blocks of a wave
  const int64_t rb = (int64_t)blockIdx.x * RB + wave * SB / 4;
  const int sb0 = wave * SB % 4;
  constexpr int MT = kFewAhead<T>;
  float* st = reinterpret_cast<float*>(smem + (size_t)tps * FF::kTile) + wave * (MT * kFewStage / 4);
  // packing task i of the wave: (token, tile) number wave + NW·i, tokens first.  MT at a time: the first ones' inputs
  // are requested before any weights (the CU returns loads in issue order) and staged behind a wait for them alone
  const int tasks = n_tok * nt;
  struct In {
    float4 x0, x1, w0, w1;
  };
  auto load_x = [&](int k) {  // (a task past the last reloads it)
    const int kc = min(k, tasks - 1), tok = kc % n_tok;
    const int64_t c0 = (int64_t)(t0 + kc / n_tok) * kTileCols + 4 * lane, c1 = c0 + 256;
    // K is a multiple of 128, so a float4 is wholly in or out; past it, column 0 is read and dropped
    const bool i0 = c0 < x.K, i1 = c1 < x.K;
    const float* p = x.xf + (size_t)(tb + tok) * x.ldx;
    In v;
    v.x0 = *reinterpret_cast<const float4*>(p + (i0 ? c0 : 0));
    v.x1 = *reinterpret_cast<const float4*>(p + (i1 ? c1 : 0));
    if (x.nw) {
      v.w0 = *reinterpret_cast<const float4*>(x.nw + (i0 ? c0 : 0));
      v.w1 = *reinterpret_cast<const float4*>(x.nw + (i1 ? c1 : 0));
    }
    return v;
  };
  In in[MT];
  // PRE: the tiles as 16-byte pieces, the first MP per thread requested before the weights
  constexpr int MP = PRE ? (NW == 8 ? 8 : 10) : 1;
  u32x4 pc[MP];
  const int pieces = nt * (FF::kTile / 16);
  const u32x4* psrc = reinterpret_cast<const u32x4*>(PRE ? x.dig + (size_t)t0 * FF::kTile : nullptr);
  if constexpr (PRE) {
#pragma unroll
    for (int i = 0; i < MP; ++i) pc[i] = psrc[min((int)tid + 64 * NW * i, pieces - 1)];
  } else {
#pragma unroll
    for (int i = 0; i < MT; ++i) in[i] = load_x(wave + NW * i);
  }
  const size_t wbytes = (size_t)(nrb - (int64_t)blockIdx.x * RB) * ntiles * kUnitBytes;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(W) + (size_t)blockIdx.x * RB * ntiles * kUnitBytes, 0, (int)(wbytes < 0x7FFFFFFFu ? wbytes : 0x7FFFFFFFu), 0x00027000);
  const int woff = (int)(16u * r + 4u * (q ^ (r >> 2))), soff = kUnitSignBytes + 8 * (int)r;
  const unsigned psel = 0x03020100u ^ (0x01010101u * (r & 3u));
  const int unit0 = (wave * SB / 4 * ntiles + t0) * kUnitBytes;
  FewUnit<SB> u;
  if (rb < nrb) few_load(wr, woff, soff, unit0, sb0, u);
  auto stage = [&](int k, int i, const In& v) {
    const int tok = k % n_tok, t = k / n_tok;
    const int64_t c0 = (int64_t)(t0 + t) * kTileCols + 4 * lane;
    const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 x0 = c0 < x.K ? v.x0 : z, x1 = c0 + 256 < x.K ? v.x1 : z;
    if (x.nw) {
      const float s = wave_sum(((x0.x * x0.x + x0.y * x0.y) + (x0.z * x0.z + x0.w * x0.w)) +
                               ((x1.x * x1.x + x1.y * x1.y) + (x1.z * x1.z + x1.w * x1.w)));
      if (lane == 0 && k < tasks) ssqs[t][tok] = s;
      x0 = make_float4(x0.x * v.w0.x, x0.y * v.w0.y, x0.z * v.w0.z, x0.w * v.w0.w);
      x1 = make_float4(x1.x * v.w1.x, x1.y * v.w1.y, x1.z * v.w1.z, x1.w * v.w1.w);
    }
    few_stage(st + i * (kFewStage / 4), lane, x0, x1);
  };
  if constexpr (PRE) {
    u32x4* dst = reinterpret_cast<u32x4*>(smem);
#pragma unroll
    for (int i = 0; i < MP; ++i)
      if ((int)tid + 64 * NW * i < pieces) dst[tid + 64 * NW * i] = pc[i];
    for (int i = (int)tid + 64 * NW * MP; i < pieces; i += 64 * NW) dst[i] = psrc[i];
  } else {
    for (int k0 = wave; k0 < tasks; k0 += MT * NW) {
#pragma unroll
      for (int i = 0; i < MT; ++i) stage(k0 + NW * i, i, in[i]);
      if (k0 + MT * NW < tasks) {
#pragma unroll
        for (int i = 0; i < MT; ++i) in[i] = load_x(k0 + NW * (MT + i));
      }
      // (one copy of the packing code, which a call that is alone on the device fetches cold)
#pragma unroll 1
      for (int i = 0; i < MT; ++i) {
        const int k = k0 + NW * i;
        if (k < tasks) few_pack<T>(smem + (size_t)(k / n_tok) * FF::kTile, st + i * (kFewStage / 4), lane, k % n_tok);
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  lds_barrier();  // the weights stay in flight
  if (!PRE && x.nw && gridDim.y > 1 && blockIdx.x == 0 && tid < (unsigned)n_tok) {
    float s = ssqs[0][tid];
    for (int t = 1; t < nt; ++t) s += ssqs[t][tid];
    x.ssq[(size_t)blockIdx.y * x.ssq_ld + tb + tid] = s;
  }
  if (rb >= nrb) return;
  f32x4 acc[SB];
#pragma unroll
  for (int sb = 0; sb < SB; ++sb) acc[sb] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int t = 0; t < nt; ++t) {
    FewUnit<SB> nx = u;
    if (t + 1 < nt) few_load(wr, woff, soff, unit0 + (t + 1) * kUnitBytes, sb0, nx);
    few_unit<T>(smem + (size_t)t * FF::kTile, lane, psel, sb0, u, acc);
    u = nx;
  }
  y += (size_t)blockIdx.y * zstride;
  if (gridDim.y > 1) accumulate = 0;
#pragma unroll
  for (int sb = 0; sb < SB; ++sb) few_slots<T>(acc[sb]);
#pragma unroll
  for (int v = 0; v < (T == 2 ? 2 : 4); ++v) {
    const int tok = T == 2 ? v : (4 * (int)q + v) % T;
    if (tok >= n_tok || (T == 2 && q) || (T == 4 && q) || (T == 8 && q > 1)) continue;
    float inv = kSignUp;
    if (!PRE && x.nw && gridDim.y == 1) {
      float s = ssqs[0][tok];
      for (int t = 1; t < nt; ++t) s += ssqs[t][tok];
      inv = kSignUp / sqrtf(s / (float)x.K + x.eps);
    }
    float* yr = y + (size_t)(tb + tok) * ldy + rb * kRowBlock + 16 * sb0 + r;
#pragma unroll
    for (int sb = 0; sb < SB; ++sb)
      if (rb * kRowBlock + 16 * (sb0 + sb) + r < rows) {
        const float val = acc[sb][v] * inv;
        yr[16 * sb] = accumulate ? yr[16 * sb] + val : val;
      }
  }
}

}  // namespace dz
