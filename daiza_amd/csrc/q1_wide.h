// q1_wide.h — the many-token (n > 16) Q1_0 product on digits (q1_digits.h): packing, product, split sum.
#pragma once
#include "q1_digits.h"

namespace dz {

constexpr int kFragBytes = 1536;                       // one digit operand: 64 lanes x 24 B (16 B plane, 8 B plane)
constexpr int kHalfBytes = 2 * kDigits * kFragBytes;   // two groups (256 columns) of 16 tokens
constexpr int kWideTokBlocks = 2;                      // 16-token blocks per workgroup
constexpr int kWideTok = 16 * kWideTokBlocks;
constexpr int kWideRb = 8;                             // row-blocks per workgroup (two per wave)
constexpr int kWideStage = kWideTokBlocks * kHalfBytes;  // bytes of one staged half tile
constexpr size_t kWideShmem = 2 * (size_t)kWideStage;

// Digit operands of a batch of activations.
//   dig: [16-token block][half tile h][group 2][digit 6][plane 0: 64 lanes x 16 B | plane 1: 64 x 8 B],
//        lane (r = lane & 15, q = lane >> 4) holding token r's block q of the group; element 8k + j of
//        a lane's 32 is column 4j + k of the block (expand_f4's order).
//   ex:  [16-token block][tile][lane]: byte g = digit 0's block scale of group g.
//   ssq: [tile][Np] sums of squares of the unweighted x (with an RMSNorm only).
struct DigitX {
  const uint8_t* dig;
  const uint32_t* ex;
  const float* ssq;
  int Np;
  int64_t K;
  float eps;
};

// Grid (Np / 16, ntiles), 256 threads: wave g packs group g of the tile for 16 tokens, one block of 32
// columns per lane; tokens past n_tok and columns past K are zero.  With w, the digits are those of
// x ⊙ w and ssq gets the tile's sums of squares of x (rmsnorm_into, rmsnorm.rs:17-200, with 1/rms
// applied to the product).  Bound by HBM: 4 B in and 4.5 B out per value.
__global__ __launch_bounds__(256) void digit_pack_kernel(const float* __restrict__ x, int64_t ldx, int64_t K, int n_tok,
                                                         const float* __restrict__ w, uint8_t* __restrict__ dig,
                                                         uint32_t* __restrict__ ex, float* __restrict__ ssq, int Np) {
  __shared__ unsigned sb[4][64];
  __shared__ float ss[4][16];
  const unsigned tid = threadIdx.x, lane = tid & 63u, g = tid >> 6, r = lane & 15u, q = lane >> 4;
  const int tb = blockIdx.x, t = blockIdx.y;
  const int tok = 16 * tb + (int)r;
  const int64_t col = (int64_t)t * kTileCols + kGroup * g + 32 * q;
  const bool live = tok < n_tok && col < K;
  const float4* xp = reinterpret_cast<const float4*>(x + (live ? (size_t)tok * ldx + col : 0));
  const float4* wp = reinterpret_cast<const float4*>(w + (live ? col : 0));
  float v[32];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float4 f = xp[j];
    v[4 * j] = live ? f.x : 0.f;
    v[4 * j + 1] = live ? f.y : 0.f;
    v[4 * j + 2] = live ? f.z : 0.f;
    v[4 * j + 3] = live ? f.w : 0.f;
  }
  if (w) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) s = __builtin_fmaf(v[i], v[i], s);
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    if (q == 0) ss[g][r] = s;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float4 f = wp[j];
      v[4 * j] *= f.x;
      v[4 * j + 1] *= f.y;
      v[4 * j + 2] *= f.z;
      v[4 * j + 3] *= f.w;
    }
  }
  u32x6 d[kDigits];
  sb[g][lane] = pack_digits(v, d);
  uint8_t* o = dig + (((size_t)tb * gridDim.y + t) * 2 + (g >> 1)) * kHalfBytes + (size_t)(g & 1u) * kDigits * kFragBytes;
#pragma unroll
  for (int k = 0; k < kDigits; ++k) {
    *reinterpret_cast<u32x4*>(o + k * kFragBytes + 16 * lane) = u32x4{d[k][0], d[k][1], d[k][2], d[k][3]};
    *reinterpret_cast<u32x2*>(o + k * kFragBytes + 1024 + 8 * lane) = u32x2{d[k][4], d[k][5]};
  }
  __syncthreads();
  if (tid < 64) ex[((size_t)tb * gridDim.y + t) * 64 + tid] = sb[0][tid] | sb[1][tid] << 8 | sb[2][tid] << 16 | sb[3][tid] << 24;
  if (w && tid < 16) ssq[(size_t)t * Np + 16 * tb + tid] = (ss[0][tid] + ss[1][tid]) + (ss[2][tid] + ss[3][tid]);
}

// N KiB (N <= 4) from g + voff (g wave-uniform, voff = 16·lane and whole KiB) to LDS lds_base + 16·lane:
// 16 bytes per lane and KiB, without passing through registers.  The compiler does not count these
// loads: the reader waits with lds_dma_wait before the barrier that publishes them.  m0 holds the LDS
// base: one statement sets it, issues the loads and puts its old value back, so that the compiler's use of
// m0 (it cannot be named as changed) and this one do not meet.
template <int N>
__device__ __forceinline__ void lds_dma(const void* g, unsigned voff, unsigned lds_base) {
  static_assert(N == 1 || N == 4, "the instruction offset holds three KiB");
  unsigned old;
  if constexpr (N == 1)
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(old) : "v"(voff), "s"(g), "s"(lds_base) : "memory");
  else
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\t"
                 "global_load_lds_dwordx4 %1, %2 offset:1024\n\tglobal_load_lds_dwordx4 %1, %2 offset:2048\n\t"
                 "global_load_lds_dwordx4 %1, %2 offset:3072\n\ts_mov_b32 m0, %0"
                 : "=&s"(old) : "v"(voff), "s"(g), "s"(lds_base) : "memory");
}
__device__ __forceinline__ void lds_dma_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Ends one step of the product: the sums are formed before it and the next step's loads stay after it.
// Without it the compiler reads all of a half tile's digit operands first, which takes more registers
// than there are.
__device__ __forceinline__ void step_fence(f32x4 (&d)[8]) {
  asm volatile("" : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]), "+v"(d[4]), "+v"(d[5]), "+v"(d[6]), "+v"(d[7])::"memory");
}

// A digit operand from LDS: the 16-byte plane, then the 8-byte plane.
__device__ __forceinline__ i32x8 read_frag(const unsigned char* f, unsigned lane) {
  const u32x4 lo = *reinterpret_cast<const u32x4*>(f + 16 * lane);
  const u32x2 hi = *reinterpret_cast<const u32x2*>(f + 1024 + 8 * lane);
  return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], 0, 0};
}

// Workgroup tile of the wide product: 512 rows x 32 tokens; the K loop goes by half tiles (two groups,
// 256 columns).  Four waves, each holding 128 rows (eight 16-row blocks) x 32 tokens of f32 sums.
//   A operand (lane & 15 = token): digit k of the token block, read from LDS and used for eight
//     matrix instructions (one per 16-row block).
//   B operand (lane & 15 = weight row): 32 signs of one group as f4.
//   D: lane holds tokens 4q .. 4q+3 of weight row lane & 15, so a group's scale is one value per lane.
// The digits of the next half tile travel to the other LDS buffer (lds_dma) while this one is
// multiplied; its signs go into the registers that the expansion has just read.  Two workgroups share a CU
// (2 x 72 KiB of LDS), so one's barrier and scale fmas hide behind the other's matrix instructions.
// Per group and wave 96 matrix instructions (16 cycles each) against 18 KiB of LDS reads (48 B per cycle and
// CU) and ~130 VALU operations.  Matrix cores busy at 1024 tokens (share of the launch, all SIMDs): 34816 x 5120 59%,
// 5120 x 17408 53%, 16480 x 5120 49%, 5120 x 6144 35%: the first is mostly waiting within a CU, the others lose whole
// rounds besides (1056 workgroups of 16480 rows over 512 places; 320 of 6144 columns, so most CUs hold one).
// Grid: 1-D, row groups x token groups x splits (wide_tile); a split writes its partial to y + z·zstride.
struct WideGrid {
  int nrg;  // row groups: ceil(nrb / kWideRb)
  int ntg;  // token groups: Np / kWideTok
  int tps;  // K tiles per split
};

// The row-block, counted from its row group's first, whose weights stand for row-block i of row group rg: i itself, or
// the matrix's last where i lies past it.
__host__ __device__ constexpr int wide_row_block(int rg, int i, int64_t nrb) {
  const int64_t left = nrb - (int64_t)rg * kWideRb;
  return i < left ? i : (int)left - 1;
}

// Workgroup index -> (row group, token group, split).  The hardware deals workgroups to the eight XCDs in turn, so
// XCD x takes a contiguous run of the tile order, and that order walks bands of eight row groups token group by token
// group: the workgroups an XCD runs together share eight row groups' weights and a few token groups' digits in its L2.
__device__ __forceinline__ void wide_tile(const WideGrid& g, int total, int& rg, int& tg, int& z) {
  const int b = (int)blockIdx.x, per = g.nrg * g.ntg;
  const int full = total / 8, rem = total % 8, x = b % 8;
  int T = x * full + min(x, rem) + b / 8;
  z = T / per;
  T %= per;
  const int band = T / (8 * g.ntg), r0 = 8 * band, w = min(8, g.nrg - r0), in = T - band * 8 * g.ntg;
  tg = in / w;
  rg = r0 + in % w;
}

__global__ __launch_bounds__(256, 2) void q1_wide_kernel(const uint8_t* __restrict__ W, int64_t rows, int64_t nrb, int ntiles,
                                                         const WideGrid wg, const DigitX x, int n_tok, float* __restrict__ y,
                                                         int64_t ldy, int64_t zstride, int accumulate) {
  constexpr int SB = 8, NB = kWideTokBlocks;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ float tok_inv[kWideTok];
  int rg, tg, z;
  wide_tile(wg, (int)gridDim.x, rg, tg, z);
  const unsigned tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, q = lane >> 4;
  const unsigned wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int t0 = z * wg.tps, t1 = min(ntiles, t0 + wg.tps);
  const int s_end = 2 * t1;
  y += (size_t)z * zstride;
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem);
  // stage s's digits of the workgroup's token blocks: 36 KiB, nine consecutive ones per wave (two waves
  // per token block)
  static_assert(kHalfBytes == 2 * 9216 && NB == 2, "nine KiB per wave");
  const uint8_t* dsrc = x.dig + ((size_t)(tg * NB + (int)(wave >> 1)) * ntiles * 2) * kHalfBytes + 9216 * (wave & 1u);
  auto stage = [&](int s, int b) {
    const uint8_t* src = dsrc + (size_t)s * kHalfBytes;
    const unsigned dst = lds0 + (unsigned)b * kWideStage + 9216u * wave;
    lds_dma<4>(src, 16 * lane, dst);
    lds_dma<4>(src, 16 * lane + 4096, dst + 4096);
    lds_dma<1>(src, 16 * lane + 8192, dst + 8192);
  };
  // the weights of the workgroup's row-blocks; a row-block past the matrix reads the last one's (its rows are not
  // stored): the buffer's bounds check does not cover the scalar offset
  const int64_t rb0 = (int64_t)rg * kWideRb + 2 * wave;
  const size_t wbytes = (size_t)(nrb - (int64_t)rg * kWideRb) * ntiles * kUnitBytes;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(W) + (size_t)rg * kWideRb * ntiles * kUnitBytes, 0, (int)(wbytes < 0x7FFFFFFFu ? wbytes : 0x7FFFFFFFu), 0x00027000);
  const int u0 = wide_row_block(rg, 2 * (int)wave, nrb) * ntiles * kUnitBytes;
  const int u1 = wide_row_block(rg, 2 * (int)wave + 1, nrb) * ntiles * kUnitBytes;
  const int woff = (int)(16u * r + 4u * (q ^ (r >> 2)));   // the lane's dword of a 16-row block's chunk
  const int soff = kUnitSignBytes + 8 * (int)r;
  const unsigned psel = 0x03020100u ^ (0x01010101u * (r & 3u));  // its bytes back to column order
  unsigned sg[2][SB];
  u32x2 sc[SB];
  auto load_signs = [&](int t, int h, int g) {
    const int uo = t * kUnitBytes;
#pragma unroll
    for (int sb = 0; sb < SB; ++sb)
      sg[g][sb] = __builtin_amdgcn_raw_buffer_load_b32(
          wr, woff, (sb < 4 ? u0 : u1) + uo + (int)(1024u * ((2u * h + g) ^ (sb & 3u)) + 256u * (sb & 3)), 0);
  };
  auto load_scales = [&](int t) {
#pragma unroll
    for (int sb = 0; sb < SB; ++sb)
      sc[sb] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(wr, soff, (sb < 4 ? u0 : u1) + t * kUnitBytes + 128 * (sb & 3), 0));
  };
  unsigned exv[NB], exn[NB];
  auto load_ex = [&](int t, unsigned (&o)[NB]) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) o[nb] = x.ex[((size_t)(tg * NB + nb) * ntiles + t) * 64 + lane];
  };
  f32x4 acc[NB][SB];
#pragma unroll
  for (int sb = 0; sb < SB; ++sb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb][sb] = f32x4{0.f, 0.f, 0.f, 0.f};
  stage(2 * t0, 0);
  load_signs(t0, 0, 0);
  load_signs(t0, 0, 1);
  load_ex(t0, exv);
  if (tid < kWideTok) {  // 1/rms of the tokens, from the tiles' sums of squares
    float inv = kSignUp;
    if (x.ssq) inv = kSignUp / sqrtf(ordered_sum(x.ssq + tg * kWideTok + tid, x.Np, ntiles) / (float)x.K + x.eps);
    tok_inv[tid] = inv;
  }
  lds_dma_wait();
  __syncthreads();
  for (int t = t0; t < t1; ++t) {
    const int tn = min(t + 1, t1 - 1);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int s = 2 * t + h;
      if (s + 1 < s_end) stage(s + 1, h ^ 1);  // the buffer's last reads ended before the previous barrier
      // the tile's scales, first used after the first group's matrix instructions
      if (h == 0) load_scales(t);
      if (h == 1) load_ex(tn, exn);
      // the 24 digit operands of the half tile in order (group, token block, digit 5 .. 0), each read one
      // ahead of the eight matrix instructions that use it
      const unsigned char* buf = smem + h * kWideStage;
      i32x8 a = read_frag(buf + (kDigits - 1) * kFragBytes, lane);
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        i32x8 b[SB];
        asm volatile("" : "+v"(sg[g][0]), "+v"(sg[g][1]), "+v"(sg[g][2]), "+v"(sg[g][3]), "+v"(sg[g][4]), "+v"(sg[g][5]),
                     "+v"(sg[g][6]), "+v"(sg[g][7]));  // this group's signs are expanded here, not earlier
#pragma unroll
        for (int sb = 0; sb < SB; ++sb) expand_f4(__builtin_amdgcn_perm(sg[g][sb], sg[g][sb], psel), b[sb]);
        load_signs(h == 0 ? t : tn, h ^ 1, g);  // half a tile ahead, into the registers just read
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          f32x4 d[SB];
          // digit k's block scales: 5k below digit 0's in every byte (no borrow: digit 0's are >= 25)
          unsigned sx = exv[nb] - 0x19191919u;
#pragma unroll
          for (int k = kDigits - 1; k >= 0; --k) {
            const int nx = k > 0 ? (nb * 2 + g) * kDigits + k - 1
                                 : nb + 1 < NB ? ((nb + 1) * 2 + g) * kDigits + kDigits - 1 : (g + 1) * kDigits + kDigits - 1;
            const i32x8 an = k > 0 || nb + 1 < NB || g == 0 ? read_frag(buf + nx * kFragBytes, lane) : a;
#pragma unroll
            for (int sb = 0; sb < SB; ++sb) {
              const f32x4 c = k == kDigits - 1 ? f32x4{0.f, 0.f, 0.f, 0.f} : d[sb];
              if (h == 0 && g == 0) d[sb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[sb], c, 2, 4, 0, (int)sx, 0, kSignScale);
              else if (h == 0) d[sb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[sb], c, 2, 4, 1, (int)sx, 0, kSignScale);
              else if (g == 0) d[sb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[sb], c, 2, 4, 2, (int)sx, 0, kSignScale);
              else d[sb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[sb], c, 2, 4, 3, (int)sx, 0, kSignScale);
            }
            a = an;
            asm("v_add_u32 %0, 0x5050505, %0" : "+v"(sx));  // (opaque: the six values would each take a register)
            step_fence(d);
          }
#pragma unroll
          for (int sb = 0; sb < SB; ++sb) {
            const unsigned slot = (2u * h + g) ^ (sb & 3u);  // the scale slot of this group
            const unsigned two = sc[sb][slot >> 1];
            const float sf = (float)__builtin_bit_cast(_Float16, (unsigned short)(slot & 1 ? two >> 16 : two & 0xFFFFu));
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[nb][sb][v] = __builtin_fmaf(sf, d[sb][v], acc[nb][sb][v]);
          }
          step_fence(acc[nb]);
        }
      }
      lds_dma_wait();
      __syncthreads();
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) exv[nb] = exn[nb];
  }
  // lane (r, q): weight row 16·sb + r, tokens 16·nb + 4q .. +3
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int tl = 16 * nb + 4 * (int)q + v, n = tg * kWideTok + tl;
      if (n >= n_tok) continue;
      const float inv = tok_inv[tl];
      float* yr = y + (size_t)n * ldy;
#pragma unroll
      for (int sb = 0; sb < SB; ++sb) {
        const int64_t row = (rb0 + (sb >> 2)) * kRowBlock + 16 * (sb & 3) + r;
        if (row < rows) {
          const float val = acc[nb][sb][v] * inv;
          yr[row] = accumulate ? yr[row] + val : val;
        }
      }
    }
}

// y[n][row] (=|+=) Σ_z part[z][n][row] for z < splits in order (the partials of a split product),
// times token n's 1/rms when ssq is given (a normed product: sums of squares [ssq_n][ssq_ld], K).
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(const float* __restrict__ part, int splits,
                                                                int64_t zstride, int64_t rows, int n_tok,
                                                                float* __restrict__ y, int64_t ldy, int accumulate,
                                                                const float* __restrict__ ssq, int ssq_n, int ssq_ld, int64_t K,
                                                                float eps) {
  const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int n = blockIdx.y;
  if (row >= rows || n >= n_tok) return;
  const size_t off = (size_t)n * rows + row;
  float v = ordered_sum(part + off, zstride, splits);
  if (ssq) v *= split_inv_rms(ssq, ssq_ld, ssq_n, n, K, eps);
  float* yr = y + (size_t)n * ldy + row;
  *yr = accumulate ? *yr + v : v;
}

}  // namespace dz
