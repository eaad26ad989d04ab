// batch_kernels.h — the n-token forward (forward_batch, Daiza-engine/src/model/forward.rs:394-1407)
// outside the projections, which run on the matrix cores (q1_digits.h, q1_wide.h).  Activations are token-major
// [n][width] f32.  Used for prefill (dz_forward_batch) and for speculative verify, where the
// DeltaNet scan records what a rollback needs instead of writing the state back.
#pragma once
#include "model_kernels.h"
#include "q1_digits.h"

namespace dz {

// The 8-lane sum of v within each aligned group of 8 lanes (quad xor 1, quad xor 2, half-row
// mirror); every lane of the group gets it.
__device__ __forceinline__ float lane8_sum(float v) {
  v = dpp_add<0xB1>(v);
  v = dpp_add<0x4E>(v);
  v = dpp_add<0x141>(v);
  return v;
}

// h[t] = embedding row of ids[t] (forward.rs:212): the f16 table through the reference's
// f16_to_f32 (tensor/tensor.rs:62-76), or a Q1_0 table through dequantize_q1_0_row_into
// (quant.rs:161-194).  Grid (n, ceil(H / 1024)), 256 threads of four columns each: with one workgroup per token
// the row's twenty dependent rounds took 13 us for eight tokens.
struct FewIds {  // up to 16 tokens as a kernel argument (ids keeps them for what follows the forward)
  int id[16];
  int n;  // 0: the ids are in memory
};
__global__ __launch_bounds__(256) void bt_embed_kernel(int* __restrict__ ids, const FewIds fi, int64_t H,
                                                       const uint16_t* __restrict__ emb_f16,
                                                       const uint8_t* __restrict__ emb_q1, int emb_ntiles,
                                                       float* __restrict__ h) {
  const int t = blockIdx.x;
  int tok;
  if (fi.n) {
    tok = fi.id[t];
    if (blockIdx.y == 0 && threadIdx.x == 0) ids[t] = tok;
  } else {
    tok = ids[t];
  }
  const int64_t k0 = ((int64_t)blockIdx.y * 256 + threadIdx.x) * 4;  // H is a multiple of 128
  if (k0 >= H) return;
  float o[4];
  if (emb_f16) {
    const ushort4 v = *reinterpret_cast<const ushort4*>(emb_f16 + (size_t)tok * H + k0);
    o[0] = ref_f16_to_f32_dev(v.x);
    o[1] = ref_f16_to_f32_dev(v.y);
    o[2] = ref_f16_to_f32_dev(v.z);
    o[3] = ref_f16_to_f32_dev(v.w);
  } else {
    const int64_t rb = tok / kRowBlock;
    const unsigned L = (unsigned)(tok % kRowBlock);
    const int tt = (int)(k0 / kTileCols);
    const unsigned p = (unsigned)((k0 % kTileCols) / 8), s = L ^ p;
    const uint8_t* u = emb_q1 + ((size_t)rb * emb_ntiles + tt) * kUnitBytes;
    const unsigned byte = u[((s >> 4) * 64 + L) * 16 + (s & 15)];
    const uint16_t* scp = reinterpret_cast<const uint16_t*>(u + kUnitSignBytes);
    const float scale = ref_f16_to_f32_dev(scp[L * 4 + ((p >> 4) ^ (L >> 4))]);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = ((float)((byte >> ((k0 & 7) + i)) & 1u) * 2.0f - 1.0f) * scale;
  }
  *reinterpret_cast<float4*>(h + (size_t)t * H + k0) = make_float4(o[0], o[1], o[2], o[3]);
}

// Causal conv over the chunk + SiLU (ssm.rs:467-518): out[t][ch] = silu(Σ_tap x[t-3+tap][ch]·w[tap][ch]),
// fma in tap order (oldest first), x[t'] = in-proj output of token t' for t' >= 0 and the conv
// ring's entry for the earlier tokens (the token at chunk offset t' < 0 sits in slot
// (head0 + t') & 3, head0 = slot of token 0).  Thread per (token, channel).  keep (verify, else null)
// receives the conv inputs themselves, keep[t][ch] = x[t][ch], from which the commit rebuilds the ring.
// The q and k channels (the first 2 nkh·128, whole heads per workgroup: 2 nkh·128 is a multiple of
// 256) also get their per-head L2 norm (l2norm_inplace, ssm.rs:76-135; q additionally times
// 1/sqrt(128), ssm.rs:532-533) into qk[t][0 .. 2 nkh·128): a head is two whole waves of the workgroup.
__global__ __launch_bounds__(256) void bt_conv_kernel(const float* __restrict__ yin, int64_t ldin, int n,
                                                      const float* __restrict__ ring, int head0,
                                                      const float* __restrict__ conv_w, int64_t qkvd,
                                                      float* __restrict__ cout, float* __restrict__ keep, int nkh,
                                                      float* __restrict__ qk) {
  __shared__ float red[4];
  const unsigned tid = threadIdx.x;
  const int64_t ch = (int64_t)blockIdx.x * 256 + tid;
  const int t = blockIdx.y;
  const bool live = ch < qkvd && t < n;
  float o = 0.f, xt = 0.f;
  if (live) {
    // every tap's input and weight requested before the sums (the address is selected, not the
    // load: a load under a branch waits for the loads before it)
    float xs[4], ws[4];
#pragma unroll
    for (int tap = 0; tap < 4; ++tap) {
      const int tt = t - 3 + tap;
      const float* src = tt >= 0 ? yin + (size_t)tt * ldin + ch : ring + (size_t)((head0 + tt) & 3) * qkvd + ch;
      xs[tap] = *src;
      ws[tap] = conv_w[(size_t)tap * qkvd + ch];
    }
    __builtin_amdgcn_sched_barrier(0);  // all eight loads issued before the first sum waits for one
#pragma unroll
    for (int tap = 0; tap < 4; ++tap) o = __builtin_fmaf(xs[tap], ws[tap], o);
    xt = xs[3];
  }
  const float v = siluf_(o);
  if (live) {
    cout[(size_t)t * qkvd + ch] = v;
    if (keep) keep[(size_t)t * qkvd + ch] = xt;
  }
  const int64_t kdim = (int64_t)nkh * 128;
  if ((int64_t)blockIdx.x * 256 >= 2 * kdim) return;  // a v-channel workgroup (uniform)
  const float sq = wave_sum(v * v);
  if ((tid & 63u) == 0) red[tid >> 6] = sq;
  __syncthreads();
  const int hw = (int)(tid >> 7) * 2;  // this head's first wave
  const float inv = 1.0f / sqrtf((red[hw] + red[hw + 1]) + 1e-6f);
  if (live) qk[(size_t)t * 2 * kdim + ch] = ch < kdim ? (v * inv) * (1.0f / sqrtf(128.0f)) : v * inv;
}

// Conv ring after tokens [0, t1) of a chunk: the inputs of tokens [t0, t1) (t0 = max(0, t1 - 4))
// go to their slots (head0 + t) & 3 (ssm.rs:467-470).
__global__ __launch_bounds__(256) void bt_ring_kernel(const float* __restrict__ yin, int64_t ldin, int t0, int t1,
                                                      float* __restrict__ ring, int head0, int64_t qkvd) {
  const int64_t ch = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (ch >= qkvd) return;
  for (int t = t0; t < t1; ++t) ring[(size_t)((head0 + t) & 3) * qkvd + ch] = yin[(size_t)t * ldin + ch];
}

// Rollback record of a verify chunk for one DeltaNet layer: the decay and the delta of every token
// (the rank-1 update S <- decay·S + d ⊗ k) and the token's key; replaying the first a of them
// reproduces the state after a tokens bit for bit.
struct DnRecord {
  float* decay;  // [n][nvh]
  float* d;      // [n][nvh * 128]
  float* k;      // [n][nkh * 128]
};

// Gated delta rule over the chunk's tokens in order (ssm_scan_vhead, ssm.rs:153-180; fused form
// 378-418).  Workgroup (v-head vh, quarter) holds state rows i = quarter·32 + (tid >> 3),
// columns j = 16·(tid & 7) .. +16 of S[vh][i][j] in registers (64 contiguous bytes per thread); the 8
// threads of a row sum with DPP.
// Per token: g = ssm_a·softplus(alpha + dt_bias), decay = exp(g), beta = sigmoid(b); s *= decay;
// kv = s·k; d = (v_i - kv)·beta; s += d·k; y_i = s·q.  The inputs of 16 tokens at a time (q and k
// of the k-head, v of the workgroup's rows, alpha, beta) are staged in LDS by the whole workgroup,
// the next 16 requested while these compute: one load latency per 16 tokens instead of one per
// token.  With rec == null the state is written back at the end; otherwise it is left as it was
// and every token's (decay, d, k) is recorded.
__global__ __launch_bounds__(256) void bt_scan_kernel(const float* __restrict__ yin, int64_t ldin,
                                                      const float* __restrict__ cout, int64_t qkvd,
                                                      const float* __restrict__ qk, int n, int nkh, int nvh,
                                                      int64_t off_a, int64_t off_b, const float* __restrict__ ssm_a,
                                                      const float* __restrict__ dt_bias, float* __restrict__ state,
                                                      float* __restrict__ y, DnRecord rec) {
  constexpr int HD = 128, G = 16;
  __shared__ __align__(16) float sqk[G][2 * HD];  // token's q then k of this k-head
  __shared__ float sv[G][32], sab[G][2];
  const unsigned tid = threadIdx.x;
  const int vh = blockIdx.x >> 2, quarter = blockIdx.x & 3, kh = vh % nkh;
  const int i = quarter * 32 + (int)(tid >> 3), js = (int)(tid & 7u);
  const int64_t kdim = (int64_t)nkh * HD;
  float* S = state + (size_t)vh * HD * HD + (size_t)i * HD + 16 * js;
  float s[16];
  state_row_load(S, s);
  const float A = ssm_a[vh], dtb = dt_bias[vh];
  // staging of tokens [g0, g0 + G): thread (tt = tid >> 4, part = tid & 15) takes 16 of token tt's
  // 256 q|k values, 2 of its v rows, and (tid < 32) one alpha or beta
  // (the staged values are returned by value and kept in named registers: held in an array
  // captured by a lambda, they went to scratch memory, one wait per load)
  const int st = (int)(tid >> 4), sp = (int)(tid & 15u);
  struct Stage {
    float4 q0, q1, q2, q3;
    float v0, v1, ab;
  };
  auto gload = [&](int g0) -> Stage {
    const int t = min(g0 + st, n - 1);
    const float* src = qk + (size_t)t * 2 * kdim + (sp < 8 ? (size_t)kh * HD + 16 * sp : kdim + (size_t)kh * HD + 16 * (sp - 8));
    const float* vr = cout + (size_t)t * qkvd + 2 * kdim + (int64_t)vh * HD + quarter * 32 + 2 * sp;
    // every thread loads alpha or beta (a valid address) and tid < 32 keep it: a load under a
    // branch waits for the loads before it
    const int ta = min(g0 + (int)(tid & 15u), n - 1);
    Stage r;
    r.q0 = *reinterpret_cast<const float4*>(src);
    r.q1 = *reinterpret_cast<const float4*>(src + 4);
    r.q2 = *reinterpret_cast<const float4*>(src + 8);
    r.q3 = *reinterpret_cast<const float4*>(src + 12);
    r.v0 = vr[0];
    r.v1 = vr[1];
    r.ab = yin[(size_t)ta * ldin + ((tid & 16u) ? off_b : off_a) + vh];
    return r;
  };
  auto gstore = [&](const Stage& r) {
    float4* dq = reinterpret_cast<float4*>(&sqk[st][16 * sp]);
    dq[0] = r.q0;
    dq[1] = r.q1;
    dq[2] = r.q2;
    dq[3] = r.q3;
    sv[st][2 * sp] = r.v0;
    sv[st][2 * sp + 1] = r.v1;
    if (tid < 32) sab[tid & 15u][tid >> 4] = r.ab;
  };
  Stage nx = gload(0);
  gstore(nx);
  __syncthreads();
  for (int g0 = 0; g0 < n; g0 += G) {
    const bool more = g0 + G < n;
    if (more) nx = gload(g0 + G);
    const int gn = min(G, n - g0);
    for (int tt = 0; tt < gn; ++tt) {
      const int t = g0 + tt;
      const float x = sab[tt][0] + dtb;
      const float spl = x > 20.0f ? x : logf(1.0f + expf(x));
      const float decay = expf(A * spl);
      const float beta = sigmoidf_(sab[tt][1]);
      float kf[16], qf[16];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float4 q4 = *reinterpret_cast<const float4*>(&sqk[tt][16 * js + 4 * c]);
        const float4 k4 = *reinterpret_cast<const float4*>(&sqk[tt][HD + 16 * js + 4 * c]);
        qf[4 * c] = q4.x; qf[4 * c + 1] = q4.y; qf[4 * c + 2] = q4.z; qf[4 * c + 3] = q4.w;
        kf[4 * c] = k4.x; kf[4 * c + 1] = k4.y; kf[4 * c + 2] = k4.z; kf[4 * c + 3] = k4.w;
      }
      float kvp = 0.f;
#pragma unroll
      for (int jj = 0; jj < 16; ++jj) {
        s[jj] *= decay;
        kvp = __builtin_fmaf(s[jj], kf[jj], kvp);
      }
      const float kv = lane8_sum(kvp);
      const float d = (sv[tt][i & 31] - kv) * beta;
      float yp = 0.f;
#pragma unroll
      for (int jj = 0; jj < 16; ++jj) {
        s[jj] = __builtin_fmaf(d, kf[jj], s[jj]);
        yp = __builtin_fmaf(s[jj], qf[jj], yp);
      }
      const float yy = lane8_sum(yp);
      if (js == 0) {
        y[(size_t)t * nvh * HD + (int64_t)vh * HD + i] = yy;
        if (rec.d) rec.d[(size_t)t * nvh * HD + (int64_t)vh * HD + i] = d;
      }
      if (rec.d && tid == 0) rec.decay[(size_t)t * nvh + vh] = decay;
      if (rec.d && vh < nkh && quarter == 0 && js == 0) {
        // the key of k-head vh, written once: rows i < 32 of quarter 0 cover 32 of its 128 columns x 4
#pragma unroll
        for (int c = 0; c < 4; ++c) rec.k[(size_t)t * kdim + (int64_t)vh * HD + 4 * (i & 31) + c] = sqk[tt][HD + 4 * (i & 31) + c];
      }
    }
    if (more) {
      __syncthreads();  // every thread is done with this group's inputs
      gstore(nx);
      __syncthreads();
    }
  }
  if (!rec.d) state_row_store(S, s);
}

// ---- the delta rule over many tokens, 32 at a time on the matrix cores ----
//
// With a_t the decay, β_t the gate, L_t = Σ_{s<=t} ln a_s within a chunk of 32 tokens and S the state before
// it, the recurrence of bt_scan_kernel is, for the chunk's tokens together:
//   N[t][s] = β_t e^(L_t - L_s) k_t·k_s (s < t),  T = (I + N)^-1
//   U = T diag(β) V,  W = T diag(β e^L) K          [32][128] each
//   D = U - W S^T                                    the tokens' deltas d_t
//   Y = diag(e^L) Q S^T + A D,  A[t][s] = e^(L_t - L_s) q_t·k_s (s <= t)
//   S <- e^(L_31) S + Σ_t e^(L_31 - L_t) d_t k_t^T
// bt_chunk_prep_kernel forms what does not depend on the state (-W, U, A, K^T and the decays) for every
// chunk at once; bt_chunk_scan_kernel walks the chunks.  All products are f32 matrix instructions; L is
// summed and subtracted in f64 (ln a is known directly, so e^(L_t - L_s) keeps an f32's precision), and
// every factor is at most 1.  The token-by-token kernel is one chain of about 1100 cycles per token (489 us
// for 1024 tokens of 48 heads, 161 for 333); the chunks take 37 + 145 us (prep + walk), 18 + 56 for 333.
constexpr int kScanC = 32;

// What bt_chunk_prep_kernel leaves for the walk, per chunk c and v-head (k-head for kt).
struct ChunkPrep {
  float* w;   // [c][nvh][32][128]  -W
  float* u;   // [c][nvh][32][128]
  float* a;   // [c][nvh][32][32]
  float* kt;  // [c][nkh][128][32]  K^T
  float* g;   // [c][nvh][2][32]    e^(L_t), e^(L_31 - L_t)
};
__host__ __device__ inline size_t chunk_prep_floats(int n, int nkh, int nvh) {
  const size_t c = (size_t)(n + kScanC - 1) / kScanC;
  return c * ((size_t)nvh * (2 * kScanC * 128 + kScanC * kScanC + 2 * kScanC) + (size_t)nkh * 128 * kScanC);
}
__host__ __device__ inline ChunkPrep chunk_prep_carve(float* p, int n, int nkh, int nvh) {
  const size_t c = (size_t)(n + kScanC - 1) / kScanC, hv = c * nvh;
  ChunkPrep r;
  r.w = p;
  r.u = r.w + hv * kScanC * 128;
  r.a = r.u + hv * kScanC * 128;
  r.kt = r.a + hv * kScanC * kScanC;
  r.g = r.kt + c * nkh * 128 * kScanC;
  return r;
}

// Causality for infinities and NaN.  T, N10 and A are 0 for a token's later ones, and 0 times a non-finite value is
// NaN.  x: NT tiles of B operands (tile t, register r: token 16t + 4·(lane >> 4) + r of the lane's column).  Non-finite
// values are set to 0; returns the first token that held one in the lane's column (16·NT: none), from which on the
// column's results are NaN: a value that entered the recurrence stays in it.
template <int NT>
__device__ __forceinline__ int take_non_finite(f32x4 (&x)[NT], int lk) {
  float nf = 0.f;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) nf = __builtin_fmaf(x[t][r], 0.f, nf);
  int first = 16 * NT;
  if (__builtin_amdgcn_ballot_w64(nf != 0.f)) {
#pragma unroll
    for (int t = NT - 1; t >= 0; --t)
#pragma unroll
      for (int r = 3; r >= 0; --r)
        if (x[t][r] - x[t][r] != 0.f) {
          x[t][r] = 0.f;
          first = 16 * t + 4 * lk + r;
        }
    first = min(first, __shfl_xor(first, 16));
    first = min(first, __shfl_xor(first, 32));
  }
  return first;
}

// Grid (nvh, chunks), 256 threads.  Tokens past n count as k = q = v = 0, β = 0, a = 1.
// 16x16x4 f32 products: A lane (row = lane & 15, slot = lane >> 4), B lane (column, slot), D lane column
// lane & 15, rows 4(lane >> 4) + i; step r of a 16-wide K block takes K index 4·slot + r, so that a lane's
// four A values are one float4 of a row and a D tile's registers are the B operand of the next product.
__global__ __launch_bounds__(256, 4) void bt_chunk_prep_kernel(const float* __restrict__ yin, int64_t ldin,
                                                            const float* __restrict__ cout, int64_t qkvd,
                                                            const float* __restrict__ qk, int n, int nkh, int nvh,
                                                            int64_t off_a, int64_t off_b, const float* __restrict__ ssm_a,
                                                            const float* __restrict__ dt_bias, ChunkPrep o) {
  constexpr int HD = 128, C = kScanC, LDT = 36;
  __shared__ double Ls[C];
  __shared__ float la[C], bet[C], be[C];  // ln a, β, β e^L
  __shared__ __align__(16) float N[C][LDT], T[C][LDT];
  const int vh = blockIdx.x, c = blockIdx.y, kh = vh % nkh, t0 = c * C;
  const unsigned tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
  const int ln = (int)(lane & 15u), lk = (int)(lane >> 4);
  const int64_t kdim = (int64_t)nkh * HD;
  if (tid < C) {
    const int t = t0 + (int)tid, tc = min(t, n - 1);
    const float x = yin[(size_t)tc * ldin + off_a + vh] + dt_bias[vh], b = yin[(size_t)tc * ldin + off_b + vh];
    const float spl = x > 20.0f ? x : logf(1.0f + expf(x));
    // e^-10000 is 0 already: held there, differences of L stay exact enough behind a token that clears the state
    // (an ln a of -inf would make them NaN)
    const float ga = ssm_a[vh] * spl, gc = ga < -1e4f ? -1e4f : ga;
    la[tid] = t < n ? gc : 0.f;
    bet[tid] = t < n ? sigmoidf_(b) : 0.f;
  }
  __syncthreads();
  if (tid < C) {
    double L = 0.0, last = 0.0;
    for (int s = 0; s < C; ++s) {
      last += (double)la[s];
      if (s <= (int)tid) L += (double)la[s];
    }
    Ls[tid] = L;
    const float eL = expf((float)L);
    be[tid] = bet[tid] * eL;
    float* g = o.g + ((size_t)c * nvh + vh) * 2 * C;
    g[tid] = eL;
    g[C + tid] = expf((float)(last - L));
  }
  __syncthreads();
  const size_t hv = (size_t)c * nvh + vh;
  // K·K^T and Q·K^T: wave w < 3 takes tile (t, s) = (0, 0), (1, 0), (1, 1); tile (0, 1) lies above the diagonal
  auto krow = [&](int t) { return qk + (size_t)min(t0 + t, n - 1) * 2 * kdim + kdim + (size_t)kh * HD; };
  if (w < 3) {
    const int tt = w > 0, ts = w > 1;
    const float* kr = krow(16 * tt + ln) + 4 * lk;
    const float* qr = qk + (size_t)min(t0 + 16 * tt + ln, n - 1) * 2 * kdim + (size_t)kh * HD + 4 * lk;
    const float* sr = krow(16 * ts + ln) + 4 * lk;
    f32x4 dk = {0.f, 0.f, 0.f, 0.f}, dq = dk;
#pragma unroll
    for (int J = 0; J < HD / 16; ++J) {
      const float4 ka = *reinterpret_cast<const float4*>(kr + 16 * J), qa = *reinterpret_cast<const float4*>(qr + 16 * J),
                   sb = *reinterpret_cast<const float4*>(sr + 16 * J);
      dk = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.x, sb.x, dk, 0, 0, 0);
      dq = __builtin_amdgcn_mfma_f32_16x16x4f32(qa.x, sb.x, dq, 0, 0, 0);
      dk = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.y, sb.y, dk, 0, 0, 0);
      dq = __builtin_amdgcn_mfma_f32_16x16x4f32(qa.y, sb.y, dq, 0, 0, 0);
      dk = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.z, sb.z, dk, 0, 0, 0);
      dq = __builtin_amdgcn_mfma_f32_16x16x4f32(qa.z, sb.z, dq, 0, 0, 0);
      dk = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.w, sb.w, dk, 0, 0, 0);
      dq = __builtin_amdgcn_mfma_f32_16x16x4f32(qa.w, sb.w, dq, 0, 0, 0);
    }
    const int s = 16 * ts + ln;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * tt + 4 * lk + i;
      const bool in = t0 + t < n;  // (a token past n has read the last one's rows)
      const bool sees = s <= t && in;
      const float e = sees ? expf((float)(Ls[t] - Ls[s])) : 0.f;
      N[t][s] = s < t ? bet[t] * e * dk[i] : 0.f;
      o.a[(hv * C + t) * C + s] = sees ? e * dq[i] : 0.f;
    }
  } else {  // the tile above the diagonal, and (once per k-head) K^T
#pragma unroll
    for (int i = 0; i < 4; ++i) o.a[(hv * C + 4 * lk + i) * C + 16 + ln] = 0.f;
    if (vh < nkh) {
      float* kt = o.kt + ((size_t)c * nkh + kh) * HD * C;
      // lane: token lane & 31, dims 64(lane >> 5) .. +63
      const int t = (int)(lane & 31u), j0 = 64 * (int)(lane >> 5);
      const float4* kr = reinterpret_cast<const float4*>(krow(t) + j0);
      const bool in = t0 + t < n;
      float4 f[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) f[j] = kr[j];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        float* d = kt + (size_t)(j0 + 4 * j) * C + t;
        d[0] = in ? f[j].x : 0.f;
        d[C] = in ? f[j].y : 0.f;
        d[2 * C] = in ? f[j].z : 0.f;
        d[3 * C] = in ? f[j].w : 0.f;
      }
    }
  }
  __syncthreads();
  // T = [[T0, 0], [-T1 N10 T0, T1]]: the 16x16 inverses T0 and T1 by forward substitution, a column per
  // lane (four partial sums break the chain), then the block below by two products
  if (w == 0) {
    if (lane < 32u) {
      const int b0 = 16 * lk;  // lanes 0..15: T0, 16..31: T1
      float col[16];
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        float p[4] = {t == ln ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < t; ++s) p[s & 3] = __builtin_fmaf(-N[b0 + t][b0 + s], col[s], p[s & 3]);
        col[t] = (p[0] + p[1]) + (p[2] + p[3]);
        T[b0 + t][b0 + ln] = col[t];
      }
    }
    __builtin_amdgcn_wave_barrier();  // LDS accesses of one wave complete in order
    f32x4 m[1] = {{0.f, 0.f, 0.f, 0.f}}, tl = m[0];
    const float4 na = *reinterpret_cast<const float4*>(&N[16 + ln][4 * lk]);
    const float4 t1 = *reinterpret_cast<const float4*>(&T[16 + ln][16 + 4 * lk]);
    const float nr[4] = {na.x, na.y, na.z, na.w}, tr[4] = {t1.x, t1.y, t1.z, t1.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) m[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(nr[r], T[4 * lk + r][ln], m[0], 0, 0, 0);
    const int nan0 = take_non_finite(m, lk);
#pragma unroll
    for (int r = 0; r < 4; ++r) tl = __builtin_amdgcn_mfma_f32_16x16x4f32(tr[r], m[0][r], tl, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) T[16 + 4 * lk + i][ln] = 4 * lk + i < nan0 ? -tl[i] : __builtin_nanf("");
  }
  __syncthreads();
  // -W and U: wave w takes columns 32w .. 32w + 31 of both
#pragma unroll
  for (int jt = 0; jt < 2; ++jt) {
    const int col = 32 * (int)w + 16 * jt + ln;
    f32x4 kx[2], vx[2];
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int s = 16 * st + 4 * lk + r;
        const float* vr = cout + (size_t)min(t0 + s, n - 1) * qkvd + 2 * kdim + (size_t)vh * HD;
        kx[st][r] = krow(s)[col];
        vx[st][r] = vr[col];
      }
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int s = 16 * st + 4 * lk + r;
        kx[st][r] *= -be[s];
        vx[st][r] *= bet[s];
      }
    const int nan_w = take_non_finite(kx, lk), nan_u = take_non_finite(vx, lk);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      f32x4 dw = {0.f, 0.f, 0.f, 0.f}, du = dw;
#pragma unroll
      for (int st = 0; st <= tt; ++st) {
        const float4 ta = *reinterpret_cast<const float4*>(&T[16 * tt + ln][16 * st + 4 * lk]);
        const float tr[4] = {ta.x, ta.y, ta.z, ta.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          dw = __builtin_amdgcn_mfma_f32_16x16x4f32(tr[r], kx[st][r], dw, 0, 0, 0);
          du = __builtin_amdgcn_mfma_f32_16x16x4f32(tr[r], vx[st][r], du, 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * tt + 4 * lk + i;
        const size_t off = (hv * C + t) * HD + col;
        o.w[off] = t < nan_w ? dw[i] : __builtin_nanf("");
        o.u[off] = t < nan_u ? du[i] : __builtin_nanf("");
      }
    }
  }
}

// The walk over the chunks: one wave per (v-head, 16 rows i of its state), no exchange between waves.  The
// state's S^T tiles (rows j, columns i) stay in the wave's accumulators and are the B operands of W S^T and
// Q S^T; D's tiles are the B operands of A D and K^T D.  W, U and Q are requested two chunks ahead, the
// rest when this chunk is done with it.  Bound by the f32 matrix instructions (208 of 32 cycles per chunk, one wave per
// SIMD on 384 of the 1024 SIMDs).  Workgroup b runs on XCD b % 8, which takes heads b % 8 + 8k: the eight
// waves of a head read the same operands in one L2.  Grid 8·8·ceil(nvh / 8), 64 threads.
__global__ __launch_bounds__(64) void bt_chunk_scan_kernel(const float* __restrict__ qk, int n, int nkh, int nvh,
                                                           const ChunkPrep o, float* __restrict__ state,
                                                           float* __restrict__ y) {
  constexpr int HD = 128, C = kScanC;
  const int b = (int)blockIdx.x, vh = (b >> 6) * 8 + (b & 7), ib = (b >> 3) & 7;
  if (vh >= nvh) return;
  const int lane = (int)threadIdx.x, ln = lane & 15, lk = lane >> 4, kh = vh % nkh;
  const int i = 16 * ib + ln;
  const int64_t kdim = (int64_t)nkh * HD;
  float* Sp = state + (size_t)vh * HD * HD + (size_t)i * HD + 4 * lk;
  f32x4 S[8];  // S^T tile J: rows j = 16J + 4lk + r, column i
#pragma unroll
  for (int J = 0; J < 8; ++J) S[J] = *reinterpret_cast<const f32x4*>(Sp + 16 * J);
  const int nc = (n + C - 1) / C;
  // W, Q rows t (of two chunks); K^T rows j; A tiles (0,0), (1,0), (1,1)
  struct WQ {
    f32x4 w[2][8], q[2][8];
    float u[2][4];
  } even, odd;
  f32x4 kv[8][2], av[3];
  f32x4 ge[2], gd[2];
  auto load_w = [&](int c, WQ& o_) {
    const float* p = o.w + (((size_t)c * nvh + vh) * C + ln) * HD + 4 * lk;
    const float* u = o.u + (((size_t)c * nvh + vh) * C + 4 * lk) * HD + i;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
      for (int J = 0; J < 8; ++J) o_.w[tt][J] = *reinterpret_cast<const f32x4*>(p + 16 * tt * HD + 16 * J);
#pragma unroll
      for (int r = 0; r < 4; ++r) o_.u[tt][r] = u[(16 * tt + r) * HD];
    }
  };
  auto load_q = [&](int c, WQ& o_) {
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const float* p = qk + (size_t)min(c * C + 16 * tt + ln, n - 1) * 2 * kdim + (size_t)kh * HD + 4 * lk;
#pragma unroll
      for (int J = 0; J < 8; ++J) o_.q[tt][J] = *reinterpret_cast<const f32x4*>(p + 16 * J);
    }
  };
  auto load_k = [&](int c) {
    const size_t hv = (size_t)c * nvh + vh;
    const float* p = o.kt + (((size_t)c * nkh + kh) * HD + ln) * C + 4 * lk;
#pragma unroll
    for (int J = 0; J < 8; ++J)
#pragma unroll
      for (int st = 0; st < 2; ++st) kv[J][st] = *reinterpret_cast<const f32x4*>(p + (size_t)16 * J * C + 16 * st);
    const float* a = o.a + (hv * C + ln) * C + 4 * lk;
    av[0] = *reinterpret_cast<const f32x4*>(a);
    av[1] = *reinterpret_cast<const f32x4*>(a + 16 * C);
    av[2] = *reinterpret_cast<const f32x4*>(a + 16 * C + 16);
    const float* g = o.g + hv * 2 * C + 4 * lk;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      ge[tt] = *reinterpret_cast<const f32x4*>(g + 16 * tt);
      gd[tt] = *reinterpret_cast<const f32x4*>(g + C + 16 * tt);
    }
  };
  load_w(0, even);
  load_q(0, even);
  load_k(0);
  load_w(min(1, nc - 1), odd);
  load_q(min(1, nc - 1), odd);
  auto chunk = [&](int c, WQ& x) {
    f32x4 d[2], yy[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      d[tt] = f32x4{x.u[tt][0], x.u[tt][1], x.u[tt][2], x.u[tt][3]};
      yy[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int J = 0; J < 8; ++J)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        d[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[0][J][r], S[J][r], d[0], 0, 0, 0);
        d[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[1][J][r], S[J][r], d[1], 0, 0, 0);
        yy[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[0][J][r], S[J][r], yy[0], 0, 0, 0);
        yy[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[1][J][r], S[J][r], yy[1], 0, 0, 0);
      }
    load_w(min(c + 2, nc - 1), x);
    load_q(min(c + 2, nc - 1), x);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int r = 0; r < 4; ++r) yy[tt][r] *= ge[tt][r];
    const int nan0 = take_non_finite(d, lk);
    if (__builtin_amdgcn_ballot_w64(nan0 < C)) {  // the column's tokens from nan0 on, and its state
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (16 * tt + 4 * lk + r >= nan0) yy[tt][r] = __builtin_nanf("");
      if (nan0 < C)
#pragma unroll
        for (int J = 0; J < 8; ++J) S[J] = f32x4{__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf("")};
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      yy[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[0][r], d[0][r], yy[0], 0, 0, 0);
      yy[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[1][r], d[0][r], yy[1], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) yy[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[2][r], d[1][r], yy[1], 0, 0, 0);
    // e^(L_31): the last token's e^(L_t), in lane group 3's fourth slot of the second tile
    const float gc = __shfl(ge[1][3], 48);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int r = 0; r < 4; ++r) d[tt][r] *= gd[tt][r];
#pragma unroll
    for (int J = 0; J < 8; ++J)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[J][r] *= gc;
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int J = 0; J < 8; ++J) S[J] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[J][st][r], d[st][r], S[J], 0, 0, 0);
    load_k(min(c + 1, nc - 1));
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = c * C + 16 * tt + 4 * lk + r;
        if (t < n) y[(size_t)t * nvh * HD + (size_t)vh * HD + i] = yy[tt][r];
      }
  };
  for (int c = 0; c < nc; c += 2) {
    chunk(c, even);
    if (c + 1 < nc) chunk(c + 1, odd);
  }
#pragma unroll
  for (int J = 0; J < 8; ++J) *reinterpret_cast<f32x4*>(Sp + 16 * J) = S[J];
}

// Rollback records and conv inputs of a verify chunk, every DeltaNet layer's one after another.
struct DnRecords {
  float* decay;  // [layer][cap][nvh]
  float* d;      // [layer][cap][nvh * 128]
  float* k;      // [layer][cap][nkh * 128]
  float* x;      // [layer][cap][qkvd]
  int cap;       // tokens per layer
  __host__ __device__ DnRecord layer(int si, int nkh, int nvh) const {
    const size_t c = (size_t)si * cap;
    return DnRecord{decay + c * nvh, d + c * nvh * 128, k + c * nkh * 128};
  }
  __host__ __device__ float* conv(int si, int64_t qkvd) const { return x + (size_t)si * cap * qkvd; }
};

// Keeps the first a recorded tokens of a verify chunk in every DeltaNet layer (blockIdx.y).  Workgroups
// [0, 4·nvh) apply them to the state: s = decay·s, s = fma(d, k, s) per token, the same operations in the same
// order as the scan (and its row mapping), so the result equals a scan over those a tokens; the others
// write the last four tokens' conv inputs to the ring (bt_ring_kernel; head0 = slot of the chunk's first token).
__global__ __launch_bounds__(256) void bt_commit_kernel(float* __restrict__ state, float* __restrict__ conv,
                                                        const int* __restrict__ ring_base, int p0, DnRecords recs, int a,
                                                        int nkh, int nvh, int64_t qkvd) {
  constexpr int HD = 128;
  const unsigned tid = threadIdx.x;
  const int si = blockIdx.y;
  if ((int)blockIdx.x >= 4 * nvh) {
    const int64_t ch = (int64_t)((int)blockIdx.x - 4 * nvh) * 256 + tid;
    if (ch >= qkvd) return;
    const int head0 = (ring_base[si] + p0) & 3;
    const float* xin = recs.conv(si, qkvd);
    for (int t = max(0, a - 4); t < a; ++t) conv[((size_t)si * 4 + ((head0 + t) & 3)) * qkvd + ch] = xin[(size_t)t * qkvd + ch];
    return;
  }
  const DnRecord rec = recs.layer(si, nkh, nvh);
  const int vh = blockIdx.x >> 2, quarter = blockIdx.x & 3, kh = vh % nkh;
  const int i = quarter * 32 + (int)(tid >> 3), js = (int)(tid & 7u);
  float* S = state + ((size_t)si * nvh + vh) * HD * HD + (size_t)i * HD + 16 * js;
  float s[16];
  state_row_load(S, s);
  for (int t = 0; t < a; ++t) {
    const float decay = rec.decay[(size_t)t * nvh + vh];
    const float d = rec.d[(size_t)t * nvh * HD + (int64_t)vh * HD + i];
    const float* kr = rec.k + (size_t)t * nkh * HD + (size_t)kh * HD + 16 * js;
#pragma unroll
    for (int jj = 0; jj < 16; ++jj) s[jj] *= decay;
#pragma unroll
    for (int jj = 0; jj < 16; ++jj) s[jj] = __builtin_fmaf(d, kr[jj], s[jj]);
  }
  state_row_store(S, s);
}

// After a forward of tokens [0, n) at position p0 that is kept: the token log, TokState and the context's logits
// (the last kept token's row), as forward_single_token leaves them.  Grid ceil(vocab / 1024), 256 threads.
__global__ __launch_bounds__(256) void bt_finish_kernel(const int* __restrict__ ids, int n, int p0, int* __restrict__ toklog,
                                                        TokState* __restrict__ st, const float* __restrict__ src,
                                                        float* __restrict__ logits, int vocab) {
  if (blockIdx.x == 0) {
    for (int t = (int)threadIdx.x; t < n; t += 256) toklog[p0 + t] = ids[t];
    if (threadIdx.x == 0) *st = TokState{p0 + n - 1, ids[n - 1], 0, 0, p0 + n, {0, 0, 0}};
  }
  const int c = (int)blockIdx.x * 1024 + (int)threadIdx.x;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (c + 256 * k < vocab) logits[c + 256 * k] = src[c + 256 * k];
}

// TokState's next position, and the ring bases shifted with it (ring heads are kept relative to the position).
__global__ __launch_bounds__(64) void set_pos_kernel(TokState* st, int pos, int* ring_base, int n, int shift) {
  if (threadIdx.x == 0) st->pos_next = pos;
  for (int i = (int)threadIdx.x; i < n; i += 64) ring_base[i] = (ring_base[i] + shift) & 3;
}

// Output gate per v-head (ssm_output_gate_avx2, ssm.rs:246-286):
// g[t][vh·128 + i] = ((y·(1/sqrt(Σy²/128 + eps)))·w_norm[i])·silu(z).  Grid (n, nvh), 128 threads.
__global__ __launch_bounds__(128) void bt_gate_y_kernel(const float* __restrict__ y, const float* __restrict__ yin,
                                                        int64_t ldin, int64_t off_z, const float* __restrict__ nw,
                                                        float eps, int nvh, float* __restrict__ g) {
  __shared__ float red[2];
  const int t = blockIdx.x, vh = blockIdx.y;
  const unsigned tid = threadIdx.x;
  const int64_t col = (int64_t)vh * 128 + tid;
  const float v = y[(size_t)t * nvh * 128 + col];
  const float z = yin[(size_t)t * ldin + off_z + col];  // requested with y: one memory round trip
  const float w = nw[tid];
  const float s = wave_sum(v * v);
  if ((tid & 63u) == 0) red[tid >> 6] = s;
  __syncthreads();
  const float inv = 1.0f / sqrtf((red[0] + red[1]) * (1.0f / 128.0f) + eps);
  g[(size_t)t * nvh * 128 + col] = ((v * inv) * w) * siluf_(z);
}

// Attention inputs of token t at position pos0 + t (attention.rs:87-123): per q-head RMSNorm
// (q_norm), the reference's partial RoPE (pairs (d, d + rope_dim/2) on d < rope_dim/2, both terms
// added: rope.rs:205-208), q·1/sqrt(256) -> qb[t][h]; the gate half -> gate[t][h]; per kv-head the
// same for k (k_norm, no scale) appended to the cache with v.  Grid (n, nq + nkv), 256 threads.
__global__ __launch_bounds__(256) void bt_attn_prep_kernel(const float* __restrict__ yin, int64_t ldin, int nq,
                                                           int nkv, const float* __restrict__ q_norm,
                                                           const float* __restrict__ k_norm, float eps,
                                                           const float* __restrict__ rope, int rope_dim, int pos0,
                                                           float* __restrict__ qb, float* __restrict__ gate,
                                                           float* __restrict__ kcache, float* __restrict__ vcache,
                                                           int max_ctx) {
  constexpr int HD = 256;
  __shared__ float xs[HD];
  __shared__ float red[4];
  const int t = blockIdx.x, hh = blockIdx.y;
  const unsigned tid = threadIdx.x;
  const float* row = yin + (size_t)t * ldin;
  const bool isq = hh < nq;
  const int kvh = hh - nq;
  const float raw = isq ? row[(size_t)hh * 2 * HD + tid] : row[(size_t)nq * 2 * HD + (size_t)kvh * HD + tid];
  // the gate (q-head) or v (kv-head) value of this dim, the norm weight and the RoPE factors,
  // requested with raw: one memory round trip
  const float other = isq ? row[(size_t)hh * 2 * HD + HD + tid] : row[(size_t)nq * 2 * HD + (size_t)nkv * HD + (size_t)kvh * HD + tid];
  const float nwt = isq ? q_norm[tid] : k_norm[tid];
  const int half = rope_dim / 2;
  const int pos = pos0 + t;
  const int dd = (int)tid < half ? (int)tid : (int)tid - half;
  const bool rot = (int)tid < rope_dim;
  const float* cs = rope + (size_t)pos * rope_dim;
  const float c = rot ? cs[dd] : 0.f, sn = rot ? cs[half + dd] : 0.f;
  const float s = wave_sum(raw * raw);
  if ((tid & 63u) == 0) red[tid >> 6] = s;
  __syncthreads();
  const float ssum = (red[0] + red[1]) + (red[2] + red[3]);
  const float in = 1.0f / sqrtf(ssum / (float)HD + eps);
  xs[tid] = (raw * in) * nwt;
  __syncthreads();
  float v = xs[tid];
  if (rot) {
    const float x1 = xs[dd], x2 = xs[dd + half];
    v = (int)tid < half ? __builtin_fmaf(x1, c, x2 * sn) : __builtin_fmaf(x2, c, x1 * sn);
  }
  if (isq) {
    qb[((size_t)t * nq + hh) * HD + tid] = v * (1.0f / sqrtf((float)HD));
    gate[((size_t)t * nq + hh) * HD + tid] = other;
  } else {
    kcache[((size_t)kvh * max_ctx + pos) * HD + tid] = v;
    vcache[((size_t)kvh * max_ctx + pos) * HD + tid] = other;
  }
}

// Causal GQA attention of a chunk's tokens on the matrix cores, f32 operands (v_mfma_f32_16x16x4_f32: the
// products and sums are f32, in another order than the reference's loop, attention.rs:149-203).
// The n·GRP (token, q-head) rows of kv-head kvh, row ρ = t·GRP + g, are one matrix; a workgroup takes 64
// of them (wave w rows 16w .. 16w+15), so each cache row it reads serves about 64/GRP tokens.
// Workgroup (row tile, kvh, z) takes the positions [z·csz, (z+1)·csz) that its rows see, in blocks of 16,
// and writes the record (m, l, o[256]) of each row to rec[t][h][z] for bt_attn_merge_kernel, or with one
// chunk (nch == 1) the gated output itself.  Per block:
//   S^T = K_blk · Q^T: A = K rows (lane = position p0 + (lane & 15), dims 16j + 4(lane >> 4) + c
//   in step 4j + c), B = the same dims of the wave's Q rows (registers); the result leaves lane
//   (r, k) the scores of row 16w + r at positions p0 + 4k + i, so the online softmax of a row runs
//   in the 4 lanes r, r+16, r+32, r+48, and those probabilities are already the A operand of
//   O += P · V_blk in position order 4k + s (step s): no transpose through LDS.
//   B of step s, tile (th, c): V[p0 + 4k + s][64th + 4r + c]; O tile (th, c) leaves lane (r, k)
//   rows 16w + 4k + i at dim 64th + 4r + c.
// Bound by the f32 matrix instructions (128 of 32 cycles per wave and block) once a workgroup walks many
// blocks.  Against the vector kernel that prefill used (one lane per position, a token per workgroup),
// whose cache rows were read once per token: 1024 tokens into an empty context 414 -> 194 us per layer,
// 333 tokens behind 7000 1821 -> 679 (and 27 for the merge).
// 1-D grid row tiles x (kv-head, chunk) pairs, 256 threads, no LDS: workgroup L runs on XCD L % 8
// (round-robin dispatch), so where the pairs are a multiple (or a divisor) of eight a pair's row tiles meet
// in one L2 (or a few); the last row tiles, which see the most positions, come first.
// AHEAD: the next block's scores are formed while this block's softmax runs (one wave per SIMD: nothing else
// would fill the matrix cores then), at the price of one block's scores for nothing per chunk; without
// it a chunk's last block is the only one.  The launch takes it for chunks of at least 32 blocks: at 112
// blocks 679 against 710 us, at nine 39.5 against 37.4.
template <int GRP, bool AHEAD>
__global__ __launch_bounds__(256) void bt_attn_mfma_kernel(const float* __restrict__ qb, const float* __restrict__ kcache,
                                                           const float* __restrict__ vcache, int max_ctx, int nq,
                                                           int pos0, int n, int csz, int nch, int nkv, float* __restrict__ rec,
                                                           const float* __restrict__ gate, float* __restrict__ ao) {
  constexpr int HD = 256;
  const int ntile = (n * GRP + 63) / 64;
  const int pairs = nkv * nch, pair = (int)blockIdx.x % pairs;
  const int tile = ntile - 1 - (int)blockIdx.x / pairs, kvh = pair % nkv, z = pair / nkv;
  const unsigned tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
  const int ln = (int)(lane & 15u), lk = (int)(lane >> 4);
  const int rows = n * GRP;
  // the chunk's positions seen by any row of the tile
  const int pbeg = z * csz, pend = min((z + 1) * csz, pos0 + (min(64 * tile + 64, rows) - 1) / GRP + 1);
  // the softmax row of this lane, visible positions [pbeg, ctx_r)
  const int rho = 64 * tile + 16 * (int)w + ln;
  const bool rv = rho < rows;
  const int ctx_r = rv ? min(pos0 + rho / GRP + 1, pend) : pbeg;
  float4 q[16];  // Q[ρ][16j + 4lk .. +3]
  {
    const float* qr = qb + ((size_t)(rv ? rho / GRP : 0) * nq + kvh * GRP + (rv ? rho % GRP : 0)) * HD + 4 * lk;
#pragma unroll
    for (int j = 0; j < 16; ++j) q[j] = rv ? *reinterpret_cast<const float4*>(qr + 16 * j) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  f32x4 o[16];  // tile 4th + c
#pragma unroll
  for (int t = 0; t < 16; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const float* kb = kcache + (size_t)kvh * max_ctx * HD;
  const float* vb = vcache + (size_t)kvh * max_ctx * HD;
  // A block's key and value rows are requested ahead (keys while the values of the block before the
  // previous one are multiplied, values while its scores are formed), so that no matrix instruction waits
  // for a load issued just before it.  Positions past the chunk are clamped to its last one
  // (written, finite) and masked.
  float4 kk[16], vv[16];  // kk[j]: K[p][16j + 4lk ..]; vv[4s + th]: V[p0 + 4lk + s][64th + 4ln ..]
  auto load_k = [&](int pb) {
    const float* kr = kb + (size_t)min(pb + ln, pend - 1) * HD + 4 * lk;
#pragma unroll
    for (int j = 0; j < 16; ++j) kk[j] = *reinterpret_cast<const float4*>(kr + 16 * j);
  };
  auto load_v = [&](int pb) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float* vr = vb + (size_t)min(pb + 4 * lk + s, pend - 1) * HD + 4 * ln;
#pragma unroll
      for (int th = 0; th < 4; ++th) vv[4 * s + th] = *reinterpret_cast<const float4*>(vr + 64 * th);
    }
  };
  // A block that some row of the wave does not see whole: the matrix instructions multiply the values of a masked
  // position by that row's probability 0, which must not make NaN of an infinity or a NaN.  A position with such a
  // value counts as zeros, and the rows that do see it get NaN.  (One fma per value; the rest is rare.)
  const int rho_0 = 64 * tile + 16 * (int)w;
  const int ctx_0 = rho_0 < rows ? min(pos0 + rho_0 / GRP + 1, pend) : pbeg;  // of the wave's first row: the smallest
  auto hide_non_finite = [&](int pb) {
    unsigned long long bad[4];  // positions pb + 4lk + s, as lanes
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      float nf = 0.f;
#pragma unroll
      for (int th = 0; th < 4; ++th) {
        const float4 v4 = vv[4 * s + th];
        nf = __builtin_fmaf(v4.x, 0.f, __builtin_fmaf(v4.y, 0.f, __builtin_fmaf(v4.z, 0.f, __builtin_fmaf(v4.w, 0.f, nf))));
      }
      bad[s] = __builtin_amdgcn_ballot_w64(nf != 0.f);
    }
    if ((bad[0] | bad[1] | bad[2] | bad[3]) == 0) return;
    int first = 0x7FFFFFFF;
#pragma unroll
    for (int s = 3; s >= 0; --s) {
      if (bad[s]) first = min(first, pb + 4 * (__builtin_ctzll(bad[s]) >> 4) + s);
      if ((bad[s] >> (16 * lk)) & 0xFFFFu)
#pragma unroll
        for (int th = 0; th < 4; ++th) vv[4 * s + th] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (first < __shfl(ctx_r, 4 * lk + i))
#pragma unroll
        for (int t = 0; t < 16; ++t) o[t][i] = __builtin_nanf("");
  };
  // scores of the block whose keys are in kk
  f32x4 s0, s1;
  auto scores = [&]() {
    s0 = f32x4{0.f, 0.f, 0.f, 0.f};
    s1 = s0;
#pragma unroll
    for (int j = 0; j < 16; j += 2) {
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[j].x, q[j].x, s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[j + 1].x, q[j + 1].x, s1, 0, 0, 0);
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[j].y, q[j].y, s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[j + 1].y, q[j + 1].y, s1, 0, 0, 0);
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[j].z, q[j].z, s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[j + 1].z, q[j + 1].z, s1, 0, 0, 0);
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[j].w, q[j].w, s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[j + 1].w, q[j + 1].w, s1, 0, 0, 0);
    }
  };
  if (pbeg < pend) {
    load_k(pbeg);
    load_v(pbeg);
    if constexpr (AHEAD) {
      scores();
      load_k(min(pbeg + 16, pend - 1));
    }
  }
  for (int p0 = pbeg; p0 < pend; p0 += 16) {
    f32x4 cur;
    if constexpr (AHEAD) {
      cur = s0 + s1;
      scores();  // of the next block (of nothing at the last one)
    } else {
      scores();
      load_k(min(p0 + 16, pend - 1));
      cur = s0 + s1;
    }
    float sc[4], bm = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sc[i] = p0 + 4 * lk + i < ctx_r ? cur[i] : -INFINITY;
      bm = fmaxf(bm, sc[i]);
    }
    bm = fmaxf(bm, __shfl_xor(bm, 16));
    bm = fmaxf(bm, __shfl_xor(bm, 32));
    const float mn = fmaxf(m, bm);
    // a row with no visible position yet keeps m = -inf: its factors are 0 and 1 by definition
    const float al = mn == -INFINITY ? 1.0f : expf(m - mn);
    float p[4], ps = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = sc[i] == -INFINITY ? 0.f : expf(sc[i] - mn);
      ps += p[i];
    }
    ps += __shfl_xor(ps, 16);
    ps += __shfl_xor(ps, 32);
    l = l * al + ps;
    m = mn;
    if constexpr (AHEAD) {
#pragma unroll
      for (int i = 0; i < 32; ++i) {  // the softmax among the next block's matrix instructions
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x006, 6, 0);
      }
      load_k(min(p0 + 32, pend - 1));
    }
    // the O rows of this lane are 16w + 4lk + i: their factors live in lanes 4lk + i (skipped when
    // no row of the wave has a new maximum: every factor is then exactly 1)
    if (__builtin_amdgcn_ballot_w64(al != 1.0f)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a = __shfl(al, 4 * lk + i);
#pragma unroll
        for (int t = 0; t < 16; ++t) o[t][i] *= a;
      }
    }
    if (p0 + 16 > ctx_0) hide_non_finite(p0);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int th = 0; th < 4; ++th) {
        const float4 v4 = vv[4 * s + th];
        o[4 * th + 0] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[s], v4.x, o[4 * th + 0], 0, 0, 0);
        o[4 * th + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[s], v4.y, o[4 * th + 1], 0, 0, 0);
        o[4 * th + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[s], v4.z, o[4 * th + 2], 0, 0, 0);
        o[4 * th + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[s], v4.w, o[4 * th + 3], 0, 0, 0);
      }
    load_v(min(p0 + 16, pend - 1));
  }
  const int ro0 = 64 * tile + 16 * (int)w + 4 * lk;  // the lane's first o row
  if (nch == 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float inv = 1.0f / __shfl(l, 4 * lk + i);
      const int ro = ro0 + i;
      if (ro >= rows) continue;
      const size_t off = ((size_t)(ro / GRP) * nq + kvh * GRP + ro % GRP) * HD + 4 * ln;
#pragma unroll
      for (int th = 0; th < 4; ++th) {
        const float4 gt = *reinterpret_cast<const float4*>(gate + off + 64 * th);
        *reinterpret_cast<float4*>(ao + off + 64 * th) =
            make_float4((o[4 * th][i] * inv) * sigmoidf_(gt.x), (o[4 * th + 1][i] * inv) * sigmoidf_(gt.y),
                        (o[4 * th + 2][i] * inv) * sigmoidf_(gt.z), (o[4 * th + 3][i] * inv) * sigmoidf_(gt.w));
      }
    }
    return;
  }
  // records: (m, l) of row ρ from lanes lk = 0; o rows ro0 + i, dims 64th + 4ln .. +3
  if (lk == 0 && rv) {
    float* rr = rec + (((size_t)(rho / GRP) * nq + kvh * GRP + rho % GRP) * nch + z) * (2 + HD);
    rr[0] = m;
    rr[1] = l;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int ro = ro0 + i;
    if (ro >= rows) continue;
    float* rr = rec + (((size_t)(ro / GRP) * nq + kvh * GRP + ro % GRP) * nch + z) * (2 + HD) + 2 + 4 * ln;
#pragma unroll
    for (int th = 0; th < 4; ++th)  // rr is 8-byte aligned
#pragma unroll
      for (int c = 0; c < 2; ++c)
        *reinterpret_cast<float2*>(rr + 64 * th + 2 * c) = make_float2(o[4 * th + 2 * c][i], o[4 * th + 2 * c + 1][i]);
  }
}

// Merge of the position chunks of bt_attn_mfma_kernel (records with l = 0 held no position), then
// o·sigmoid(gate).  Grid (n, nq), 256 threads (one output dim each); nch <= 256.  Thread z < nch
// brings chunk z's (m, l) to LDS, so that every chunk's weight exp(m_z - M) is formed once, and the
// dims are summed over the chunks in order, the first 64 requested with the statistics and the
// rest 16 at a time.
__global__ __launch_bounds__(256) void bt_attn_merge_kernel(const float* __restrict__ rec, int nch,
                                                            const float* __restrict__ gate, int nq,
                                                            float* __restrict__ ao) {
  constexpr int HD = 256;
  __shared__ float ml[2][256];  // m, then the chunk weight; l
  __shared__ float red[8];
  const int t = blockIdx.x, h = blockIdx.y;
  const unsigned tid = threadIdx.x;
  const float* rr = rec + ((size_t)t * nq + h) * nch * (2 + HD);
  const bool has = (int)tid < nch;
  // this dim of the first NO chunks, requested together with the chunk statistics (they do not
  // depend on the maximum): one memory round trip for up to NO chunks
  constexpr int NO = 64;
  const float gt = gate[((size_t)t * nq + h) * HD + tid];  // the output gate, with the rest
  float o0[NO];
#pragma unroll
  for (int k = 0; k < NO; ++k) o0[k] = k < nch ? rr[(size_t)k * (2 + HD) + 2 + tid] : 0.f;
  const float mz = has ? rr[(size_t)tid * (2 + HD)] : -INFINITY;
  const float lz = has ? rr[(size_t)tid * (2 + HD) + 1] : 0.f;
  // M = max of m over the chunks that held a position (in any order: max is exact)
  float m = lz > 0.f ? mz : -INFINITY;
  m = wave_max(m);
  if ((tid & 63u) == 0) red[tid >> 6] = m;
  __syncthreads();
  const float M = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  ml[0][tid] = lz > 0.f ? expf(mz - M) : 0.f;
  ml[1][tid] = lz;
  __syncthreads();
  float L = 0.f, O = 0.f;
#pragma unroll
  for (int k = 0; k < NO; ++k) {
    if (k < nch) {
      const float e = ml[0][k];
      L = __builtin_fmaf(ml[1][k], e, L);
      O = __builtin_fmaf(o0[k], e, O);
    }
  }
  for (int z0 = NO; z0 < nch; z0 += 16) {
    float o[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) o[k] = z0 + k < nch ? rr[(size_t)(z0 + k) * (2 + HD) + 2 + tid] : 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (z0 + k < nch) {
        const float e = ml[0][z0 + k];
        L = __builtin_fmaf(ml[1][z0 + k], e, L);
        O = __builtin_fmaf(o[k], e, O);
      }
    }
  }
  ao[((size_t)t * nq + h) * HD + tid] = (O * (1.0f / L)) * sigmoidf_(gt);
}

// ---- few tokens (n <= 16): the kernels that form a product's activations hand them over as digits ----
//
// One wave per (token, K tile of the next product), lane columns 4·lane .. +3 and 256 + 4·lane .. +3 of the tile; the
// digits go to dig[tile] (FewForm<T>), for a normed product with the next norm's weight nw multiplied in and the
// tile's sum of squares beside them (ssq[tile][n]).  Grid (tiles, n), 64 threads.
template <int T>
struct FewOut {
  uint8_t* dig;
  const float* nw;  // null: no norm follows
  float* ssq;
  int64_t K;
};
template <int T>
__device__ __forceinline__ void few_out(const FewOut<T>& o, float4 x0, float4 x1) {
  __shared__ __align__(16) float st[kFewStage / 4];
  const unsigned lane = threadIdx.x;
  const int t = blockIdx.x, tok = blockIdx.y;
  if (o.nw) {
    const float s = wave_sum(((x0.x * x0.x + x0.y * x0.y) + (x0.z * x0.z + x0.w * x0.w)) +
                             ((x1.x * x1.x + x1.y * x1.y) + (x1.z * x1.z + x1.w * x1.w)));
    if (lane == 0) o.ssq[(size_t)t * gridDim.y + tok] = s;
    const int64_t c0 = (int64_t)t * kTileCols + 4 * lane;  // columns past K hold zeros
    const float4 w0 = *reinterpret_cast<const float4*>(o.nw + (c0 < o.K ? c0 : 0));
    const float4 w1 = *reinterpret_cast<const float4*>(o.nw + (c0 + 256 < o.K ? c0 + 256 : 0));
    x0 = make_float4(x0.x * w0.x, x0.y * w0.y, x0.z * w0.z, x0.w * w0.w);
    x1 = make_float4(x1.x * w1.x, x1.y * w1.y, x1.z * w1.z, x1.w * w1.w);
  }
  few_stage(st, lane, x0, x1);
  few_pack<T>(o.dig + (size_t)t * FewForm<T>::kTile, st, lane, tok);
}

// out[m] = Σ_z p[m][z·stride] for z < n in split order (four consecutive columns each), N splits of all M sums in
// flight at a time (a split past n reloads the last one; its value is not added): one memory round trip per N.
template <int M, int N>
__device__ __forceinline__ void ordered_sums4(const float* const (&p)[M], int64_t stride, int n, float4 (&out)[M]) {
  for (int b = 0; b < n; b += N) {
    float4 v[N][M];
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int m = 0; m < M; ++m) v[k][m] = *reinterpret_cast<const float4*>(p[m] + (size_t)min(b + k, n - 1) * stride);
    __builtin_amdgcn_sched_barrier(0);  // every load issued before the first sum waits for one
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const float4 f = v[k][m];
        if (b + k == 0) out[m] = f;
        else if (b + k < n) out[m] = make_float4(out[m].x + f.x, out[m].y + f.y, out[m].z + f.z, out[m].w + f.w);
      }
  }
}

// h += Σ_z part[z] (a split product into the residual; part null: h as it is), and h's digits.
template <int T>
__global__ __launch_bounds__(64) void few_resid_kernel(float* __restrict__ h, int64_t H, const float* __restrict__ part,
                                                       int splits, int64_t zstride, FewOut<T> o) {
  const int64_t c0 = (int64_t)blockIdx.x * kTileCols + 4 * threadIdx.x, c1 = c0 + 256;
  const size_t row = (size_t)blockIdx.y * H;
  const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
  const int64_t cc[2] = {c0 < H ? c0 : 0, c1 < H ? c1 : 0};
  float4 x[2] = {*reinterpret_cast<const float4*>(h + row + cc[0]), *reinterpret_cast<const float4*>(h + row + cc[1])};
  if (part) {
    const float* const p[2] = {part + row + cc[0], part + row + cc[1]};
    float4 d[2];
    ordered_sums4<2, 18>(p, zstride, splits, d);
#pragma unroll
    for (int i = 0; i < 2; ++i) x[i] = make_float4(x[i].x + d[i].x, x[i].y + d[i].y, x[i].z + d[i].z, x[i].w + d[i].w);
    if (c0 < H) *reinterpret_cast<float4*>(h + row + c0) = x[0];
    if (c1 < H) *reinterpret_cast<float4*>(h + row + c1) = x[1];
  }
  if (c0 >= H) x[0] = z;
  if (c1 >= H) x[1] = z;
  few_out<T>(o, x[0], x[1]);
}

// silu(gate) · up from a split gate/up product's partials part[z][t][2F] (with its tokens' 1/rms), as digits.
template <int T>
__global__ __launch_bounds__(64) void few_swiglu_kernel(const float* __restrict__ part, int splits, int64_t zstride, int64_t F,
                                                        const float* __restrict__ ssq, int ssq_n, int ssq_ld, int64_t K,
                                                        float eps, FewOut<T> o) {
  const int64_t c0 = (int64_t)blockIdx.x * kTileCols + 4 * threadIdx.x;
  const size_t row = (size_t)blockIdx.y * 2 * F;
  const int64_t d0 = c0 < F ? c0 : 0, d1 = c0 + 256 < F ? c0 + 256 : 0;
  const float* const p[4] = {part + row + d0, part + row + d1, part + row + F + d0, part + row + F + d1};
  float4 gu[4], x[2];
  const float* sp = ssq + blockIdx.y;
  const float sq = threadIdx.x < (unsigned)ssq_n ? sp[(size_t)threadIdx.x * ssq_ld] : 0.f;  // ssq_n <= 16 tiles of H
  ordered_sums4<4, 5>(p, zstride, splits, gu);
  const float inv = 1.0f / sqrtf(wave_sum(sq) / (float)K + eps);
  const float4 g[2] = {gu[0], gu[1]}, u[2] = {gu[2], gu[3]};
#pragma unroll
  for (int i = 0; i < 2; ++i)
    x[i] = c0 + 256 * i < F ? make_float4(siluf_(g[i].x * inv) * (u[i].x * inv), siluf_(g[i].y * inv) * (u[i].y * inv),
                                          siluf_(g[i].z * inv) * (u[i].z * inv), siluf_(g[i].w * inv) * (u[i].w * inv))
                            : make_float4(0.f, 0.f, 0.f, 0.f);
  few_out<T>(o, x[0], x[1]);
}

// bt_gate_y_kernel's result as digits: a tile holds four v-heads, each 32 lanes' columns of one half.
template <int T>
__global__ __launch_bounds__(64) void few_gate_kernel(const float* __restrict__ y, const float* __restrict__ yin, int64_t ldin,
                                                      int64_t off_z, const float* __restrict__ nw, float eps, int nvh,
                                                      FewOut<T> o) {
  const unsigned lane = threadIdx.x;
  const int64_t inner = (int64_t)nvh * 128, c0 = (int64_t)blockIdx.x * kTileCols + 4 * lane;
  const int t = blockIdx.y;
  float4 v[2], zz[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t c = c0 + 256 * i, cc = c < inner ? c : 0;
    v[i] = *reinterpret_cast<const float4*>(y + (size_t)t * inner + cc);
    const float* zp = yin + (size_t)t * ldin + off_z + cc;  // rows of yin are not 16-byte aligned for every shape
    zz[i] = make_float4(zp[0], zp[1], zp[2], zp[3]);
  }
  const float4 w = *reinterpret_cast<const float4*>(nw + 4 * (lane & 31u));
  float4 x[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    float s = (v[i].x * v[i].x + v[i].y * v[i].y) + (v[i].z * v[i].z + v[i].w * v[i].w);
    s = dpp_add<0xB1>(s);  // the 16 lanes of a DPP row, then the head's two rows
    s = dpp_add<0x4E>(s);
    s = dpp_add<0x141>(s);
    s = dpp_add<0x140>(s);
    s += __shfl_xor(s, 16);
    const float inv = 1.0f / sqrtf(s * (1.0f / 128.0f) + eps);
    x[i] = c0 + 256 * i < inner ? make_float4(((v[i].x * inv) * w.x) * siluf_(zz[i].x), ((v[i].y * inv) * w.y) * siluf_(zz[i].y),
                                              ((v[i].z * inv) * w.z) * siluf_(zz[i].z), ((v[i].w * inv) * w.w) * siluf_(zz[i].w))
                                : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  few_out<T>(o, x[0], x[1]);
}

// SwiGLU (mlp.rs:28-47, swiglu_inplace_simd): s[t][i] = silu(gate[t][i]) · up[t][i], gate rows
// [0, F) and up rows [F, 2F) of the gate/up product.
__global__ __launch_bounds__(256) void bt_swiglu_kernel(const float* __restrict__ gu, int64_t F, int n,
                                                        float* __restrict__ s) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int t = blockIdx.y;
  if (i >= F || t >= n) return;
  const float* row = gu + (size_t)t * 2 * F;
  s[(size_t)t * F + i] = siluf_(row[i]) * row[F + i];
}

// The same from the partials of a split gate/up product of many tokens (part[z][t][2F], zstride apart, 1/rms
// applied): each sum in split order, as gemm_split_reduce_kernel forms it, then silu(gate) · up.
__global__ __launch_bounds__(256) void bt_split_swiglu_kernel(const float* __restrict__ part, int splits,
                                                              int64_t zstride, int64_t F, int n,
                                                              float* __restrict__ s) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int t = blockIdx.y;
  if (i >= F || t >= n) return;
  const size_t off = (size_t)t * 2 * F + i;
  const float g = ordered_sum(part + off, zstride, splits), u = ordered_sum(part + off + F, zstride, splits);
  s[(size_t)t * F + i] = siluf_(g) * u;
}

}  // namespace dz
