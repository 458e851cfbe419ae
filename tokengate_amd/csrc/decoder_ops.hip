// Per-token decoder work around the attention of the gated prefill, one HBM pass each:
//   * residual add + RMSNorm (the input / post-attention norms of a Qwen3 layer and the final norm),
//   * per-head q/k RMSNorm + rotary embedding at each token's own position, writing q in place
//     and k / v into the layer's KV cache rows,
//   * SiLU(gate) * up of the fused gate/up projection;
//   * for the few rows of a decode step: the projections on the matrix cores, streaming the weight
//     once, optionally with the RMSNorm or the SwiGLU product folded into their input, or the SwiGLU
//     product into their output; the counters and rotary table that its layers share; and the greedy
//     argmax over the logits.
// The prefill's projections (many rows) are plain GEMMs and stay on hipBLASLt.
#include <type_traits>

#include "tg_common.h"
#include "../../include/tokengate_hip.h"

namespace tg {
namespace {

// ---- residual add + RMSNorm: one wave per row, CPL chunks of 8 elements per lane ----------------
// s = residual ? bf16(x + residual) : x;  residual_out = s;  out = bf16(w * s / sqrt(mean(s^2) + eps))
template <int CPL>
__global__ __launch_bounds__(256) void rmsnorm_kernel(const bf16_t *x, int64_t x_rs,
                                                      const bf16_t *res, int64_t res_rs, bf16_t *res_out,
                                                      int64_t ro_rs, const bf16_t *__restrict__ w,
                                                      bf16_t *out, int64_t o_rs, int64_t rows, int d, float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave_id();
  if (row >= rows) return;
  const int nch = d >> 3;
  float v[CPL][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    const int ch = lane + 64 * c;
    if (ch < nch) {
      unpack8(ld16(x + row * x_rs + 8 * ch), v[c]);
      if (res) {
        float r[8];
        unpack8(ld16(res + row * res_rs + 8 * ch), r);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[c][e] = (float)(__bf16)(v[c][e] + r[e]);  // bf16 residual stream
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += v[c][e] * v[c][e];
    }
  }
  ss = wave_sum(ss);
  const float rinv = rsqrtf(ss / (float)d + eps);
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    const int ch = lane + 64 * c;
    if (ch < nch) {
      if (res_out) st16(res_out + row * ro_rs + 8 * ch, pack8(v[c]));
      float wf[8], y[8];
      unpack8(ld16(w + 8 * ch), wf);
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = wf[e] * (v[c][e] * rinv);
      st16(out + row * o_rs + 8 * ch, pack8(y));
    }
  }
}

// ---- q/k RMSNorm + RoPE + KV-cache write -----------------------------------------------------
// A workgroup handles kTok tokens.  Their (cos, sin) tables are computed once into LDS; then each
// 16-lane group takes one 128-element head row at a time (lane j holds elements 8j..8j+7, the
// rotate-half partner 8j+-64 sits in lane j^8).
constexpr int kRopeTok = 2;

__global__ __launch_bounds__(256) void qk_rope_kernel(const bf16_t *qkv, int64_t qkv_rs,
                                                      const int64_t *__restrict__ pos, int64_t T, int H,
                                                      int Hkv, const bf16_t *__restrict__ qw,
                                                      const bf16_t *__restrict__ kw, float eps,
                                                      const float *__restrict__ inv_freq,
                                                      const float *__restrict__ q_head_scale,
                                                      const float *__restrict__ q_row_scale, bf16_t *q_out,
                                                      int64_t q_rs, bf16_t *__restrict__ k_out, int64_t k_rs,
                                                      bf16_t *__restrict__ v_out, int64_t v_rs,
                                                      const int32_t *__restrict__ kv_rows) {
  __shared__ float cs[kRopeTok][kHeadDim / 2][2];
  const int tid = threadIdx.x;
  const int64_t tok0 = (int64_t)blockIdx.x * kRopeTok;
  if (tid < kRopeTok * 64) {
    const int tt = tid >> 6, i = tid & 63;
    const int64_t t = tok0 + tt;
    float s = 0.f, c = 1.f;
    if (t < T) {
      // angle = position * inv_freq, both fp32 (the rotary table's own arithmetic)
      const float ang = (float)pos[t] * inv_freq[i];
      sincosf(ang, &s, &c);
    }
    cs[tt][i][0] = c;
    cs[tt][i][1] = s;
  }
  __syncthreads();
  const int grp = tid >> 4, j = tid & 15;
  const int R = H + 2 * Hkv;
  for (int r = grp; r < kRopeTok * R; r += 16) {
    const int tt = r / R, rr = r - tt * R;
    const int64_t t = tok0 + tt;
    if (t >= T) continue;  // uniform over the 16-lane group
    const bf16_t *src = qkv + t * qkv_rs + (int64_t)rr * kHeadDim + 8 * j;
    const u32x4 raw = ld16(src);
    const int64_t crow = kv_rows ? (int64_t)kv_rows[t] : t;   // this token's KV-cache row
    if (rr >= H + Hkv) {  // value row: copied into the cache
      st16(v_out + crow * v_rs + (int64_t)(rr - H - Hkv) * kHeadDim + 8 * j, raw);
      continue;
    }
    const bool is_q = rr < H;
    float x[8], wf[8];
    unpack8(raw, x);
    unpack8(ld16((is_q ? qw : kw) + 8 * j), wf);
    // Query multiplier s = bf16(head * row), applied to the bf16-rounded rotated query with one
    // more bf16 rounding: the reference scales its bf16 query states in bf16 (q * s_eff,
    // qwen3_flex_attention.py:442-451, :400).  With no multiplier s = 1 and the second rounding
    // is exact.
    const float hs = is_q ? (float)(__bf16)((q_head_scale ? q_head_scale[rr] : 1.f) *
                                            (q_row_scale ? q_row_scale[t] : 1.f))
                          : 1.f;
    float y[8];
    norm_rope8(x, wf, eps, cs[tt] + 8 * (j & 7), j, hs, y);
    bf16_t *dst = is_q ? q_out + t * q_rs + (int64_t)rr * kHeadDim
                       : k_out + crow * k_rs + (int64_t)(rr - H) * kHeadDim;
    st16(dst + 8 * j, pack8(y));
  }
}

// ---- SiLU(gate) * up -----------------------------------------------------------------------
__global__ __launch_bounds__(256) void silu_mul_kernel(const bf16_t *__restrict__ gu, int64_t gu_rs,
                                                       int64_t rows, int inter, bf16_t *__restrict__ out,
                                                       int64_t o_rs) {
  const int nch = inter >> 3;
  const int64_t total = rows * nch;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / nch;
    const int ch = (int)(i - r * nch);
    float g[8], u[8], y[8];
    unpack8(ld16(gu + r * gu_rs + 8 * ch), g);
    unpack8(ld16(gu + r * gu_rs + inter + 8 * ch), u);
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = g[e] / (1.f + __expf(-g[e])) * u[e];
    st16(out + r * o_rs + 8 * ch, pack8(y));
  }
}

// ---- scoring-branch readout: one wave per row --------------------------------------------------
// score[r] = bf16(sum_i bf16(bf16(silu(g_ri)) * u_ri) * w_i) stored as fp32: the finalized gate's
// SwiGLU branch with its down projection absorbed into one (1, inter) row, evaluated with the
// bf16 roundings of an eager bf16 Qwen3MLP (silu output, gate * up product, the GEMM's output);
// the dot product accumulates in fp32.  silu uses the accurate expf, as torch's bf16 silu does.
__global__ __launch_bounds__(256) void branch_readout_kernel(const bf16_t *__restrict__ gu, int64_t gu_rs,
                                                             int64_t rows, int inter,
                                                             const bf16_t *__restrict__ w,
                                                             float *__restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave_id();
  if (row >= rows) return;
  const int nch = inter >> 3;
  const bf16_t *g = gu + row * gu_rs;
  const bf16_t *u = g + inter;
  float acc = 0.f;
#pragma unroll 4
  for (int ch = lane; ch < nch; ch += 64) {
    float gf[8], uf[8], wf[8];
    unpack8(ld16(g + 8 * ch), gf);
    unpack8(ld16(u + 8 * ch), uf);
    unpack8(ld16(w + 8 * ch), wf);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float sl = (float)(__bf16)(gf[e] / (1.f + expf(-gf[e])));
      acc = fmaf((float)(__bf16)(sl * uf[e]), wf[e], acc);
    }
  }
  acc = wave_sum(acc);
  if (lane == 0) out[row] = (float)(__bf16)acc;
}

// ---- Linear layer on a few rows: y[b, v] = bf16(sum_d x[b, d] * w[v, d]) ------------------------
// F.linear on bf16 tensors for the rows of a decode step (1..8): the vocab projection of the rows
// that produce the next token (written as fp32, .float() of the bf16 result) and the decoder
// layers' projections (written as bf16).  HBM-bound on the (n_out, dim) weight.
// The input x can be formed on the fly from the previous kernel's output, removing a launch:
//   kPreNorm:   x = bf16(w_n * s / sqrt(mean(s^2) + eps)) with s = bf16(h + res) (res optional),
//               exactly the RMSNorm kernel's arithmetic and summation order; block 0 writes
//               res_out = s (a buffer other than res: every block reads res);
//   kPreSwiGLU: x = bf16(silu(g) * u) of the gate/up rows [g | u], as the silu_mul kernel;
// and of a gate|up projection the SwiGLU product can be formed on the way out (ACT), each workgroup
// owning the gate and the up rows of its outputs.
constexpr int kLmMaxRows = 8;
constexpr int kPrePlain = 0, kPreNorm = 1, kPreSwiGLU = 2;
struct LinIn {
  const bf16_t *x;          // plain: input rows; norm: h; swiglu: [gate | up] rows
  int64_t x_rs;
  const bf16_t *res;        // norm: residual stream in (NULL: s = h)
  int64_t res_rs;
  bf16_t *res_out;          // norm: s out (NULL: not written)
  int64_t ro_rs;
  const bf16_t *nw;         // norm weight (dim)
  float eps;
  int inter;                // swiglu: offset of u within a row (= dim)
};
__device__ __forceinline__ u32x4 swiglu8(u32x4 gv, u32x4 uv) {
  float g[8], u[8], y[8];
  unpack8(gv, g);
  unpack8(uv, u);
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = g[e] / (1.f + __expf(-g[e])) * u[e];
  return pack8(y);
}
__device__ __forceinline__ u32x4 norm8(u32x4 sv, u32x4 nwv, float rinv) {
  float v[8], wf[8], y[8];
  unpack8(sv, v);
  unpack8(nwv, wf);
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = wf[e] * (v[e] * rinv);
  return pack8(y);
}
// Eight inputs of input row b from column c on (rinv: the row's normaliser, norm stage only)
template <int PRE>
__device__ __forceinline__ u32x4 lin_input(const LinIn &in, int b, int c, float rinv) {
  if constexpr (PRE == kPrePlain) {
    return ld16(in.x + b * in.x_rs + c);
  } else if constexpr (PRE == kPreSwiGLU) {
    return swiglu8(ld16(in.x + b * in.x_rs + c), ld16(in.x + b * in.x_rs + in.inter + c));
  } else {
    float v[8];
    unpack8(ld16(in.x + b * in.x_rs + c), v);
    if (in.res) {
      float r[8];
      unpack8(ld16(in.res + b * in.res_rs + c), r);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (float)(__bf16)(v[e] + r[e]);
    }
    return norm8(pack8(v), ld16(in.nw + c), rinv);   // (v is exact in bf16)
  }
}
// A workgroup (8 waves) owns RB blocks of 8 output rows; wave w takes the 64-column pieces w, w + 8,
// w + 16, ... of the inner dimension, so that every request of a wave is 8 whole 128-byte lines and,
// with all of a wave's pieces requested before the first product (NK of them, when dim = 512 NK), the
// workgroup's whole slice of the weight is in flight at once.  One MFMA (16x16x32) takes a piece of a
// block: rows 0..7 of its A operand are the block's weights at the piece's first 32 columns and rows
// 8..15 the same output rows at the other 32; the columns of B are the (up to 8) input rows in the
// same two halves.  The diagonal quarters of the result hold the two halves' sums, the other two are
// not used.  Each input element is read once per workgroup, by the one lane that feeds it to the
// matrix core.  The dot products used to run on the VALU, each wave reading all input rows for 4
// output rows: twice the weight's bytes at 8 rows.  Before -> now, weights from HBM, at 1 / 8 rows
// (us): 4096 x 2048 with the norm 6.9 / 14.5 -> 5.3 / 7.0, 2048 x 2048 4.3 / 8.3 -> 3.9 / 4.4,
// 12288 x 2048 with the norm 12.4 / 28.6 -> 11.8 / 13.4 (with the SwiGLU product on the way out 11.0 /
// 13.6), 2048 x 6144 6.3 / 12.1 -> 6.6 / 8.2, 151936 x 2048 with the norm 109 / 250 -> 104 / 112 (6.0 /
// 5.6 TB/s).  WALK: fewer workgroups than blocks, which walk them with the next blocks' weights in flight
// (only where a launch has that many: the second set of weight registers costs a 2048 x 6144 launch of
// one block per workgroup 6.6 -> 7.6 us).
template <int RB, int NK, typename OutT, int PRE, bool ACT, bool WALK>
__global__ __launch_bounds__(512) void linear_rows_mfma_kernel(LinIn in, const bf16_t *__restrict__ w, int64_t n_out,
                                                               int dim, int nr, OutT *__restrict__ out,
                                                               int64_t out_rs) {
  constexpr int kWaves = 8, NKR = NK > 0 ? NK : 1;
  constexpr bool kStage = PRE == kPreNorm && NK == 4;   // dim = 2048
  constexpr bool kStageAct = PRE == kPreSwiGLU && NK > 0;   // each wave forms its own pieces, in LDS
  constexpr int kXsRow = kStageAct ? 64 * NK + 8 : 2048 + 8;   // padded: 8 rows' 16-byte reads on different banks
  __shared__ __attribute__((aligned(16))) bf16_t xs[kStage ? 8 * kXsRow : kStageAct ? kWaves * 8 * kXsRow : 8];
  __shared__ __attribute__((aligned(16))) float part2[WALK ? 2 : 1][kWaves][RB][2][64];
  __shared__ float rinv_s[8];
  const int lane = threadIdx.x & 63, wv = wave_id();
  const int c = lane & 7, G = lane >> 4;
  const int xr = min(c, nr - 1);                         // input rows past nr repeat the last (not stored)
  const int kl = 64 * wv + 32 * ((lane >> 3) & 1) + 8 * G;
  constexpr int OB = ACT ? RB / 2 : RB;                  // blocks of stored rows
  const bf16_t *wr[RB];
  auto rows_from = [&](int64_t v0) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      // rows past the end read the last row (in bounds; not stored)
      const int64_t v = min(v0 + 8 * (rb % OB) + c, n_out - 1);
      wr[rb] = w + (v + (rb / OB) * n_out) * dim + kl;
    }
  };
  const int64_t step = (int64_t)gridDim.x * (8 * OB);
  int64_t v0 = (int64_t)blockIdx.x * (8 * OB);
  rows_from(v0);
  // inputs are requested before the weights: loads complete in issue order, so the input stage runs
  // while the weight bytes stream in
  u32x4 xin[NKR], rin[NKR], nwv[NKR], wf[NKR][RB];
  u32x4 sx[kStage ? 4 : 1], sr[kStage ? 4 : 1];
  if constexpr (NK > 0) {
    if constexpr (PRE == kPrePlain) {
#pragma unroll
      for (int s = 0; s < NK; ++s) xin[s] = ld16(in.x + xr * in.x_rs + kl + 512 * s);
    } else if constexpr (kStageAct) {
      // the wave's 8 NK chunks of every row, once each (NK rounds at 8 rows)
#pragma unroll
      for (int s = 0; s < NK; ++s) {
        const int idx = lane + 64 * s, b = idx / (8 * NK), j = idx % (8 * NK);
        if (b < nr) {
          const bf16_t *p = in.x + b * in.x_rs + 64 * wv + 512 * (j >> 3) + 8 * (j & 7);
          xin[s] = ld16(p);
          rin[s] = ld16(p + in.inter);
        }
      }
    } else if constexpr (kStage) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int idx = threadIdx.x + 512 * i, b = idx >> 8, ch = 8 * (idx & 255);
        if (b < nr) {
          sx[i] = ld16(in.x + b * in.x_rs + ch);
          if (in.res) sr[i] = ld16(in.res + b * in.res_rs + ch);
        }
      }
#pragma unroll
      for (int s = 0; s < NK; ++s) nwv[s] = ld16(in.nw + kl + 512 * s);
    }
#pragma unroll
    for (int s = 0; s < NK; ++s)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) wf[s][rb] = ld16(wr[rb] + 512 * s);
  }
  float rinv = 0.f;
  if constexpr (PRE == kPreNorm) {
    const bool writer = blockIdx.x == 0 && in.res_out != nullptr;
    if constexpr (kStage) {
      // s = bf16(h + res) to LDS (block 0 also writes res_out), then wave b sums row b's squares in
      // the RMSNorm kernel's order (lane l its chunks l, l + 64, ..., then the wave butterfly)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int idx = threadIdx.x + 512 * i, b = idx >> 8, ch = 8 * (idx & 255);
        if (b < nr) {
          float v[8];
          unpack8(sx[i], v);
          if (in.res) {
            float r[8];
            unpack8(sr[i], r);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = (float)(__bf16)(v[e] + r[e]);
          }
          const u32x4 pv = pack8(v);
          if (writer) st16(in.res_out + b * in.ro_rs + ch, pv);
          *reinterpret_cast<u32x4 *>(xs + b * kXsRow + ch) = pv;
        }
      }
      __syncthreads();
      if (wv < nr) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v[8];
          unpack8(*reinterpret_cast<const u32x4 *>(xs + wv * kXsRow + 8 * lane + 512 * i), v);
#pragma unroll
          for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
        }
        ss = wave_sum(ss);
        if (lane == 0) rinv_s[wv] = rsqrtf(ss / (float)dim + in.eps);
      }
    } else if (wv < nr) {
      float ss = 0.f;
      for (int ch = 8 * lane; ch < dim; ch += 512) {
        float v[8];
        unpack8(ld16(in.x + wv * in.x_rs + ch), v);
        if (in.res) {
          float r[8];
          unpack8(ld16(in.res + wv * in.res_rs + ch), r);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = (float)(__bf16)(v[e] + r[e]);
        }
        if (writer) st16(in.res_out + wv * in.ro_rs + ch, pack8(v));
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
      }
      ss = wave_sum(ss);
      if (lane == 0) rinv_s[wv] = rsqrtf(ss / (float)dim + in.eps);
    }
    __syncthreads();
    rinv = rinv_s[xr];
  }
  if constexpr (kStageAct) {
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      const int idx = lane + 64 * s, b = idx / (8 * NK), j = idx % (8 * NK);
      if (b < nr) *reinterpret_cast<u32x4 *>(xs + (8 * wv + b) * kXsRow + 8 * j) = swiglu8(xin[s], rin[s]);
    }
    // only this wave reads its part: its LDS operations complete in order
  }
  u32x4 xf[NKR];
  if constexpr (NK > 0) {
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      if constexpr (PRE == kPrePlain)
        xf[s] = xin[s];
      else if constexpr (kStageAct)
        xf[s] = *reinterpret_cast<const u32x4 *>(xs + (8 * wv + xr) * kXsRow + 64 * s + (kl - 64 * wv));
      else if constexpr (kStage)
        xf[s] = norm8(*reinterpret_cast<const u32x4 *>(xs + xr * kXsRow + kl + 512 * s), nwv[s], rinv);
      else
        xf[s] = lin_input<PRE>(in, xr, kl + 512 * s, rinv);
    }
  }
  int buf = 0;
  do {
    f32x4 acc[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) acc[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (NK > 0) {
      // the next blocks' weights are requested before these are used
      u32x4 wn[WALK ? NK : 1][RB];
      if (WALK && v0 + step < n_out) {
        rows_from(v0 + step);
#pragma unroll
        for (int s = 0; s < NK; ++s)
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) wn[s][rb] = ld16(wr[rb] + 512 * s);
      }
#pragma unroll
      for (int s = 0; s < NK; ++s)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          acc[rb] = mfma16(__builtin_bit_cast(bf16x8, wf[s][rb]), __builtin_bit_cast(bf16x8, xf[s]), acc[rb]);
      if constexpr (WALK)
#pragma unroll
        for (int s = 0; s < NK; ++s)
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) wf[s][rb] = wn[s][rb];
    } else {
      for (int k = 0; k < dim; k += 512) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) wf[0][rb] = ld16(wr[rb] + k);
        const u32x4 x = lin_input<PRE>(in, xr, kl + k, rinv);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          acc[rb] = mfma16(__builtin_bit_cast(bf16x8, wf[0][rb]), __builtin_bit_cast(bf16x8, x), acc[rb]);
      }
    }
    // lane l holds rows 4 (G % 2) .. + 3 of column half G / 2 for input row c where its own column is
    // of that half
    float (*part)[RB][2][64] = part2[WALK ? buf : 0];
    if (((lane >> 3) & 1) == (G >> 1)) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) *reinterpret_cast<f32x4 *>(&part[wv][rb][G >> 1][8 * c + 4 * (G & 1)]) = acc[rb];
    }
    // one barrier per round: the sums of a round are read while the next round writes the other buffer.
    // Not __syncthreads(), which would wait for the weights in flight.
    ring_barrier();
    const int t = threadIdx.x;
    if (t < 64 * OB) {
      const int ob = t >> 6, e = t & 63, b = e >> 3, r = e & 7;
      auto total = [&](int rb) {
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < kWaves; ++i) sum += part[i][rb][0][e] + part[i][rb][1][e];
        return sum;
      };
      const int64_t v = v0 + 8 * ob + r;
      if (b < nr && v < n_out) {
        if constexpr (ACT) {
          const float g = (float)(__bf16)total(ob), u = (float)(__bf16)total(OB + ob);
          out[b * out_rs + v] = __builtin_bit_cast(bf16_t, (__bf16)(g / (1.f + __expf(-g)) * u));
        } else {
          const __bf16 y = (__bf16)total(ob);
          if constexpr (std::is_same<OutT, float>::value)
            out[b * out_rs + v] = (float)y;
          else
            out[b * out_rs + v] = __builtin_bit_cast(bf16_t, y);
        }
      }
    }
    v0 += step;
    buf ^= 1;
  } while (WALK && v0 < n_out);
}

// ---- start of a decode step -----------------------------------------------------------------------
// What the layers of a step share, one workgroup per sequence: the position's rotary table (angle =
// position * inv_freq in fp32, accurate sincosf: tg_qk_norm_rope's, which forms it in every launch), the
// caches' used counts (+ 1, the new row), the new token's scaled-softmax ratio
// min(1, ln max(2, slots) / ln max(2, position + 1)), then position (+ 1).
__global__ __launch_bounds__(64) void decode_begin_kernel(int64_t *pos, const float *__restrict__ inv_freq, float2 *rope,
                                                          int32_t *used, int n_used, float *slots, float *ratio) {
  const int b = blockIdx.x, nseq = gridDim.x, t = threadIdx.x;
  const int64_t p = pos[b];   // one wave: read before lane 0 raises it
  float s, c;
  sincosf((float)p * inv_freq[t], &s, &c);
  rope[b * (kHeadDim / 2) + t] = float2{c, s};
  for (int i = t; i < n_used; i += 64) used[i * nseq + b] += 1;
  if (t == 0) {
    if (slots) {
      const float m = slots[b] + 1.f;
      slots[b] = m;
      ratio[b] = fminf(1.f, logf(fmaxf(m, 2.f)) / logf(fmaxf((float)p + 1.f, 2.f)));
    }
    pos[b] = p + 1;
  }
}

// ---- Greedy token: the index of each row's largest logit -----------------------------------------
// torch.argmax semantics: a NaN beats every number, and equal values go to the lower index.  One
// 1024-thread workgroup per row: each thread scans its strided 16-byte pieces, then the (value,
// index) pairs are folded across the wave and, through LDS, across the 16 waves.
__device__ __forceinline__ bool amax_better(float a, int64_t ia, float b, int64_t ib) {
  const bool na = a != a, nb = b != b;
  if (na) return nb ? ia < ib : true;
  if (nb) return false;
  return a == b ? ia < ib : a > b;
}
__global__ __launch_bounds__(1024) void argmax_rows_kernel(const float *__restrict__ x, int64_t rs, int64_t n,
                                                           int64_t *__restrict__ out) {
  const float *row = x + (int64_t)blockIdx.x * rs;
  float best = -INFINITY;
  int64_t bi = n;   // no element yet: loses every comparison with a real one
  const int64_t n4 = n / 4;
  int64_t j = threadIdx.x;
  for (; j + 3 * 1024 < n4; j += 4 * 1024) {   // four independent loads in flight per thread
    f32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const f32x4 *>(row + 4 * (j + u * 1024));
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = v[u][e];
        const int64_t ix = 4 * (j + u * 1024) + e;
        if (amax_better(x, ix, best, bi)) { best = x; bi = ix; }
      }
  }
  for (; j < n4; j += 1024) {
    const f32x4 v = *reinterpret_cast<const f32x4 *>(row + 4 * j);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = v[e];
      if (amax_better(x, 4 * j + e, best, bi)) { best = x; bi = 4 * j + e; }
    }
  }
  for (int64_t j = 4 * n4 + threadIdx.x; j < n; j += 1024)
    if (amax_better(row[j], j, best, bi)) { best = row[j]; bi = j; }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float ob = __shfl_xor(best, o);
    const int64_t oi = __shfl_xor(bi, o);
    if (amax_better(ob, oi, best, bi)) { best = ob; bi = oi; }
  }
  __shared__ float sb[16];
  __shared__ int64_t si[16];
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { sb[w] = best; si[w] = bi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < 16; ++k)
      if (amax_better(sb[k], si[k], best, bi)) { best = sb[k]; bi = si[k]; }
    out[blockIdx.x] = bi;
  }
}

}  // namespace
}  // namespace tg

using namespace tg;

extern "C" int tg_rmsnorm(const void *x, int64_t x_row_stride, const void *residual, int64_t residual_row_stride,
                          void *residual_out, int64_t residual_out_row_stride, const void *weight, void *out,
                          int64_t out_row_stride, int64_t n_rows, int32_t dim, float eps, hipStream_t stream) {
  clear_error();
  TG_CHECK(x && weight && out, "rmsnorm: null pointer");
  TG_CHECK(n_rows >= 0, "rmsnorm: negative row count");
  TG_CHECK(dim > 0 && dim % 8 == 0 && dim <= 64 * 8 * 8, "rmsnorm: dim must be a multiple of 8, at most 4096");
  TG_CHECK(x_row_stride >= dim && out_row_stride >= dim && (!residual || residual_row_stride >= dim) &&
               (!residual_out || residual_out_row_stride >= dim),
           "rmsnorm: row strides must be at least dim");
  TG_CHECK(x_row_stride % 8 == 0 && out_row_stride % 8 == 0 && (!residual || residual_row_stride % 8 == 0) &&
               (!residual_out || residual_out_row_stride % 8 == 0),
           "rmsnorm: row strides must be multiples of 8 elements");
  TG_CHECK(aligned16(x) && aligned16(weight) && aligned16(out) && aligned16(residual) && aligned16(residual_out),
           "rmsnorm: pointers must be 16-byte aligned");
  TG_CHECK(eps >= 0.f, "rmsnorm: eps must be non-negative");
  if (n_rows == 0) return 0;
  const int64_t blocks = (n_rows + 3) / 4;
  TG_CHECK(blocks < (1ll << 31), "rmsnorm: too many rows");
  const int cpl = (dim / 8 + 63) / 64;
  auto *xp = static_cast<const bf16_t *>(x);
  auto *rp = static_cast<const bf16_t *>(residual);
  auto *rop = static_cast<bf16_t *>(residual_out);
  auto *wp = static_cast<const bf16_t *>(weight);
  auto *op = static_cast<bf16_t *>(out);
#define TG_RMS(N)                                                                                  \
  case N:                                                                                          \
    hipLaunchKernelGGL(rmsnorm_kernel<N>, dim3((unsigned)blocks), dim3(256), 0, stream, xp, x_row_stride, rp, \
                       residual_row_stride, rop, residual_out_row_stride, wp, op, out_row_stride, n_rows, dim, eps); \
    break;
  switch (cpl) {
    TG_RMS(1) TG_RMS(2) TG_RMS(4) TG_RMS(8)
    case 3: hipLaunchKernelGGL(rmsnorm_kernel<4>, dim3((unsigned)blocks), dim3(256), 0, stream, xp, x_row_stride, rp,
                               residual_row_stride, rop, residual_out_row_stride, wp, op, out_row_stride, n_rows, dim,
                               eps); break;
    default: hipLaunchKernelGGL(rmsnorm_kernel<8>, dim3((unsigned)blocks), dim3(256), 0, stream, xp, x_row_stride, rp,
                                residual_row_stride, rop, residual_out_row_stride, wp, op, out_row_stride, n_rows,
                                dim, eps); break;
  }
#undef TG_RMS
  TG_HIP_CHECK(hipGetLastError());
  return 0;
}

extern "C" int tg_qk_norm_rope(const void *qkv, int64_t qkv_row_stride, const int64_t *positions, int64_t n_tokens,
                               int32_t num_heads, int32_t num_heads_k, int32_t head_dim, const void *q_norm_weight,
                               const void *k_norm_weight, float eps, const float *inv_freq, const float *q_head_scale,
                               const float *q_row_scale, void *q_out, int64_t q_row_stride, void *k_out,
                               int64_t k_row_stride, void *v_out, int64_t v_row_stride, const int32_t *kv_rows,
                               hipStream_t stream) {
  clear_error();
  TG_CHECK(qkv && positions && q_norm_weight && k_norm_weight && inv_freq && q_out && k_out && v_out,
           "qk_norm_rope: null pointer");
  TG_CHECK(head_dim == kHeadDim, "qk_norm_rope: head_dim must be 128");
  TG_CHECK(num_heads > 0 && num_heads_k > 0 && num_heads <= 256 && num_heads_k <= 256,
           "qk_norm_rope: head counts must be in 1..256");
  TG_CHECK(n_tokens >= 0, "qk_norm_rope: negative token count");
  TG_CHECK(qkv_row_stride % 8 == 0 && q_row_stride % 8 == 0 && k_row_stride % 8 == 0 && v_row_stride % 8 == 0,
           "qk_norm_rope: row strides must be multiples of 8 elements");
  TG_CHECK(qkv_row_stride >= (int64_t)(num_heads + 2 * num_heads_k) * kHeadDim,
           "qk_norm_rope: qkv rows must hold q, k and v of every head");
  TG_CHECK(q_row_stride >= (int64_t)num_heads * kHeadDim && k_row_stride >= (int64_t)num_heads_k * kHeadDim &&
               v_row_stride >= (int64_t)num_heads_k * kHeadDim,
           "qk_norm_rope: q/k/v output rows must hold every head");
  TG_CHECK(aligned16(qkv) && aligned16(q_out) && aligned16(k_out) && aligned16(v_out) &&
               aligned16(q_norm_weight) && aligned16(k_norm_weight),
           "qk_norm_rope: pointers must be 16-byte aligned");
  if (n_tokens == 0) return 0;
  const int64_t blocks = (n_tokens + kRopeTok - 1) / kRopeTok;
  TG_CHECK(blocks < (1ll << 31), "qk_norm_rope: too many tokens");
  hipLaunchKernelGGL(qk_rope_kernel, dim3((unsigned)blocks), dim3(256), 0, stream,
                     static_cast<const bf16_t *>(qkv), qkv_row_stride, positions, n_tokens, num_heads, num_heads_k,
                     static_cast<const bf16_t *>(q_norm_weight), static_cast<const bf16_t *>(k_norm_weight), eps,
                     inv_freq, q_head_scale, q_row_scale, static_cast<bf16_t *>(q_out), q_row_stride,
                     static_cast<bf16_t *>(k_out), k_row_stride, static_cast<bf16_t *>(v_out), v_row_stride,
                     kv_rows);
  TG_HIP_CHECK(hipGetLastError());
  return 0;
}

extern "C" int tg_silu_mul(const void *gate_up, int64_t gate_up_row_stride, int64_t n_rows, int32_t inter,
                           void *out, int64_t out_row_stride, hipStream_t stream) {
  clear_error();
  TG_CHECK(gate_up && out, "silu_mul: null pointer");
  TG_CHECK(n_rows >= 0 && inter > 0 && inter % 8 == 0, "silu_mul: inter must be a positive multiple of 8");
  TG_CHECK(gate_up_row_stride % 8 == 0 && out_row_stride % 8 == 0 && gate_up_row_stride >= 2 * (int64_t)inter &&
               out_row_stride >= inter,
           "silu_mul: row strides must be multiples of 8, gate_up rows must hold 2*inter and out rows inter "
           "elements");
  TG_CHECK(aligned16(gate_up) && aligned16(out), "silu_mul: pointers must be 16-byte aligned");
  if (n_rows == 0) return 0;
  const int64_t chunks = n_rows * (inter / 8);
  const int64_t blocks = std::min<int64_t>((chunks + 255) / 256, 256 * 64);
  hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)blocks), dim3(256), 0, stream,
                     static_cast<const bf16_t *>(gate_up), gate_up_row_stride, n_rows, inter,
                     static_cast<bf16_t *>(out), out_row_stride);
  TG_HIP_CHECK(hipGetLastError());
  return 0;
}

extern "C" int tg_gate_branch_readout(const void *gate_up, int64_t gate_up_row_stride, int64_t n_rows,
                                      int32_t inter, const void *w_row, float *scores, hipStream_t stream) {
  clear_error();
  TG_CHECK(gate_up && w_row && scores, "branch_readout: null pointer");
  TG_CHECK(n_rows >= 0 && inter > 0 && inter % 8 == 0, "branch_readout: inter must be a positive multiple of 8");
  TG_CHECK(gate_up_row_stride % 8 == 0 && gate_up_row_stride >= 2 * (int64_t)inter,
           "branch_readout: gate_up row stride must be a multiple of 8 holding 2*inter elements");
  TG_CHECK(aligned16(gate_up) && aligned16(w_row), "branch_readout: gate_up and w_row must be 16-byte aligned");
  if (n_rows == 0) return 0;
  const int64_t blocks = (n_rows + 3) / 4;
  TG_CHECK(blocks < (1ll << 31), "branch_readout: too many rows");
  hipLaunchKernelGGL(branch_readout_kernel, dim3((unsigned)blocks), dim3(256), 0, stream,
                     static_cast<const bf16_t *>(gate_up), gate_up_row_stride, n_rows, inter,
                     static_cast<const bf16_t *>(w_row), scores);
  TG_HIP_CHECK(hipGetLastError());
  return 0;
}

namespace tg {
namespace {

template <int RB, int NK, typename OutT, int PRE, bool ACT>
void launch_linear_rows_form(const LinIn &in, int32_t n_rows, const bf16_t *w, int64_t n_out, int32_t dim, OutT *out,
                             int64_t out_row_stride, int64_t max_grid, hipStream_t stream) {
  const int64_t rows = ACT ? 4 * RB : 8 * RB;
  const int64_t blocks = (n_out + rows - 1) / rows;
  if constexpr (NK == 4 && RB >= 2) {
    if (blocks > max_grid) {
      hipLaunchKernelGGL((linear_rows_mfma_kernel<RB, NK, OutT, PRE, ACT, true>), dim3((unsigned)max_grid), dim3(512), 0,
                         stream, in, w, n_out, dim, n_rows, out, out_row_stride);
      return;
    }
  }
  hipLaunchKernelGGL((linear_rows_mfma_kernel<RB, NK, OutT, PRE, ACT, false>), dim3((unsigned)blocks), dim3(512), 0,
                     stream, in, w, n_out, dim, n_rows, out, out_row_stride);
}
// n_out: stored outputs (ACT: weight holds 2 n_out rows, [gate; up]).
// Blocks of 8 weight rows per workgroup (RB) and workgroups, us at 1 / 8 input rows:
//   * 2048 rows fill the CUs with one block each (2048 x 2048: RB 1 / 2 / 4 3.9 / 4.7 / 6.3 and 4.4 / 5.4 / 6.9;
//     2048 x 6144: 6.6 / 9.0 / 16.1 and 8.2 / 10.8 / 17.6);
//   * up to 65536 rows two blocks spread the input stage over more weight bytes, except at 4096 rows and
//     up to two input rows (RB 1 / 2: 5.3 / 5.6 and 7.7 / 7.0); two workgroups per CU that walk the
//     blocks, the next block's weights in flight, beat one workgroup per block (12288 rows with the
//     SwiGLU product: 11.0 against 12.2, 13.6 against 14.5);
//   * beyond (the LM head) the blocks' own workgroups keep more bytes in flight: plain input RB 1 / 2 /
//     4 99.8 / 104.2 / 105.5 and 145 / 112 / 119; with the norm in every workgroup 143 / 104 / 114 and
//     172 / 133 / 126, four blocks walked by four workgroups per CU 108 and 112.
template <typename OutT, int PRE, bool ACT = false>
int launch_linear_rows(const LinIn &in, int32_t n_rows, const void *weight, int64_t n_out, int32_t dim, OutT *out,
                       int64_t out_row_stride, hipStream_t stream) {
  const bf16_t *w = static_cast<const bf16_t *>(weight);
  const int64_t w_rows = ACT ? 2 * n_out : n_out;
  const int64_t cus = device_cus();
  int rb = 1;
  int64_t max_grid = INT32_MAX;
  if (w_rows >= 65536) {
    rb = PRE == kPreNorm ? (n_rows == 1 ? 2 : 4) : (n_rows <= 2 ? 1 : 2);
    if (rb == 4) max_grid = 4 * cus;
  } else if (w_rows > 4096 || (w_rows == 4096 && n_rows > 2)) {
    rb = 2;
    max_grid = 2 * cus;
  }
  if (ACT) rb = std::max(rb, 2);
  if (dim > 2048) rb = ACT ? 2 : 1;
  auto form = [&](auto rb_c) {
    constexpr int RB = decltype(rb_c)::value;
    if (dim == 2048)
      launch_linear_rows_form<RB, 4, OutT, PRE, ACT>(in, n_rows, w, n_out, dim, out, out_row_stride, max_grid, stream);
    else if (RB == 1 && PRE != kPreNorm && dim == 6144)
      launch_linear_rows_form<RB, RB == 1 && PRE != kPreNorm ? 12 : 0, OutT, PRE, ACT>(
          in, n_rows, w, n_out, dim, out, out_row_stride, max_grid, stream);
    else
      launch_linear_rows_form<RB, 0, OutT, PRE, ACT>(in, n_rows, w, n_out, dim, out, out_row_stride, max_grid, stream);
  };
  if constexpr (!ACT)
    if (rb == 1) form(std::integral_constant<int, 1>());
  if (rb == 2) form(std::integral_constant<int, 2>());
  if (rb == 4) form(std::integral_constant<int, 4>());
  TG_HIP_CHECK(hipGetLastError());
  return 0;
}
int check_linear_rows(const char *what, const void *x, int64_t x_row_stride, int32_t n_rows, const void *weight,
                      int64_t n_out, int32_t dim, const void *out, int64_t out_row_stride) {
  TG_CHECK(x && weight && out, "%s: null pointer", what);
  TG_CHECK(n_rows >= 1 && n_rows <= kLmMaxRows, "%s: 1 to %d rows (got %d)", what, kLmMaxRows, n_rows);
  TG_CHECK(dim > 0 && dim % 512 == 0, "%s: dim must be a positive multiple of 512 (got %d)", what, dim);
  TG_CHECK(n_out > 0 && x_row_stride % 8 == 0 && x_row_stride >= dim && out_row_stride >= n_out,
           "%s: bad output size or row strides", what);
  TG_CHECK(aligned16(x) && aligned16(weight), "%s: x and weight must be 16-byte aligned", what);
  TG_CHECK((n_out + 3) / 4 < (1ll << 31), "%s: too many output features", what);
  return 0;
}

}  // namespace
}  // namespace tg

using namespace tg;

extern "C" int tg_lm_head(const void *x, int64_t x_row_stride, int32_t n_rows, const void *weight, int64_t vocab,
                          int32_t dim, float *out, int64_t out_row_stride, hipStream_t stream) {
  clear_error();
  if (int e = check_linear_rows("lm_head", x, x_row_stride, n_rows, weight, vocab, dim, out, out_row_stride)) return e;
  LinIn in{};
  in.x = static_cast<const bf16_t *>(x);
  in.x_rs = x_row_stride;
  return launch_linear_rows<float, kPrePlain>(in, n_rows, weight, vocab, dim, out, out_row_stride, stream);
}

extern "C" int tg_linear_rows(const void *x, int64_t x_row_stride, int32_t n_rows, const void *weight,
                              int64_t n_out, int32_t dim, void *out, int64_t out_row_stride, hipStream_t stream) {
  clear_error();
  if (int e = check_linear_rows("linear_rows", x, x_row_stride, n_rows, weight, n_out, dim, out, out_row_stride))
    return e;
  LinIn in{};
  in.x = static_cast<const bf16_t *>(x);
  in.x_rs = x_row_stride;
  return launch_linear_rows<bf16_t, kPrePlain>(in, n_rows, weight, n_out, dim, static_cast<bf16_t *>(out),
                                               out_row_stride, stream);
}

namespace tg {
namespace {
int norm_input(const char *what, const void *h, int64_t h_row_stride, const void *residual, int64_t residual_row_stride,
               void *residual_out, int64_t residual_out_row_stride, const void *norm_weight, float eps, int32_t dim,
               LinIn *in) {
  TG_CHECK(norm_weight && aligned16(norm_weight), "%s: norm weight must be non-null and 16-byte aligned", what);
  TG_CHECK(!residual || (aligned16(residual) && residual_row_stride % 8 == 0 && residual_row_stride >= dim),
           "%s: bad residual", what);
  TG_CHECK(!residual_out || (aligned16(residual_out) && residual_out_row_stride % 8 == 0 &&
                             residual_out_row_stride >= dim && residual_out != residual),
           "%s: bad residual_out (it must not be the residual input)", what);
  TG_CHECK(eps >= 0.f, "%s: eps must be non-negative", what);
  in->x = static_cast<const bf16_t *>(h);
  in->x_rs = h_row_stride;
  in->res = static_cast<const bf16_t *>(residual);
  in->res_rs = residual_row_stride;
  in->res_out = static_cast<bf16_t *>(residual_out);
  in->ro_rs = residual_out_row_stride;
  in->nw = static_cast<const bf16_t *>(norm_weight);
  in->eps = eps;
  return 0;
}
}  // namespace
}  // namespace tg

extern "C" int tg_linear_rows_norm(const void *h, int64_t h_row_stride, const void *residual,
                                   int64_t residual_row_stride, void *residual_out, int64_t residual_out_row_stride,
                                   const void *norm_weight, float eps, int32_t n_rows, const void *weight,
                                   int64_t n_out, int32_t dim, void *out, int64_t out_row_stride, int32_t out_fp32,
                                   hipStream_t stream) {
  clear_error();
  if (int e = check_linear_rows("linear_rows_norm", h, h_row_stride, n_rows, weight, n_out, dim, out, out_row_stride))
    return e;
  LinIn in{};
  if (int e = norm_input("linear_rows_norm", h, h_row_stride, residual, residual_row_stride, residual_out,
                         residual_out_row_stride, norm_weight, eps, dim, &in))
    return e;
  if (out_fp32)
    return launch_linear_rows<float, kPreNorm>(in, n_rows, weight, n_out, dim, static_cast<float *>(out),
                                               out_row_stride, stream);
  return launch_linear_rows<bf16_t, kPreNorm>(in, n_rows, weight, n_out, dim, static_cast<bf16_t *>(out),
                                              out_row_stride, stream);
}

extern "C" int tg_linear_rows_norm_act(const void *h, int64_t h_row_stride, const void *residual,
                                       int64_t residual_row_stride, void *residual_out,
                                       int64_t residual_out_row_stride, const void *norm_weight, float eps,
                                       int32_t n_rows, const void *weight, int64_t inter, int32_t dim, void *out,
                                       int64_t out_row_stride, hipStream_t stream) {
  clear_error();
  if (int e = check_linear_rows("linear_rows_norm_act", h, h_row_stride, n_rows, weight, inter, dim, out,
                                out_row_stride))
    return e;
  LinIn in{};
  if (int e = norm_input("linear_rows_norm_act", h, h_row_stride, residual, residual_row_stride, residual_out,
                         residual_out_row_stride, norm_weight, eps, dim, &in))
    return e;
  return launch_linear_rows<bf16_t, kPreNorm, true>(in, n_rows, weight, inter, dim, static_cast<bf16_t *>(out),
                                                    out_row_stride, stream);
}

extern "C" int tg_linear_rows_swiglu(const void *gate_up, int64_t gate_up_row_stride, int32_t n_rows, int32_t inter,
                                     const void *weight, int64_t n_out, void *out, int64_t out_row_stride,
                                     hipStream_t stream) {
  clear_error();
  if (int e = check_linear_rows("linear_rows_swiglu", gate_up, gate_up_row_stride, n_rows, weight, n_out, inter, out,
                                out_row_stride))
    return e;
  TG_CHECK(gate_up_row_stride >= 2 * (int64_t)inter, "linear_rows_swiglu: gate/up rows hold 2 * inter values");
  LinIn in{};
  in.x = static_cast<const bf16_t *>(gate_up);
  in.x_rs = gate_up_row_stride;
  in.inter = inter;
  return launch_linear_rows<bf16_t, kPreSwiGLU>(in, n_rows, weight, n_out, inter, static_cast<bf16_t *>(out),
                                                out_row_stride, stream);
}

extern "C" int tg_argmax_rows(const float *x, int64_t x_row_stride, int32_t n_rows, int64_t n_cols, int64_t *out,
                              hipStream_t stream) {
  clear_error();
  TG_CHECK(x && out, "argmax_rows: null pointer");
  TG_CHECK(n_rows >= 0 && n_cols > 0, "argmax_rows: need n_rows >= 0 and n_cols > 0");
  TG_CHECK(x_row_stride >= n_cols && x_row_stride % 4 == 0, "argmax_rows: row stride must be >= n_cols and a multiple of 4");
  TG_CHECK(aligned16(x), "argmax_rows: x must be 16-byte aligned");
  if (n_rows == 0) return 0;
  hipLaunchKernelGGL(argmax_rows_kernel, dim3((unsigned)n_rows), dim3(1024), 0, stream, x, x_row_stride, n_cols, out);
  TG_HIP_CHECK(hipGetLastError());
  return 0;
}

extern "C" int tg_decode_begin(int64_t *positions, int32_t num_seqs, const float *inv_freq, float *rope,
                               int32_t *kv_used, int32_t n_used, float *slots, float *ratio, hipStream_t stream) {
  clear_error();
  TG_CHECK(positions && inv_freq && rope && (kv_used || n_used == 0) && (ratio || !slots), "decode_begin: null pointer");
  TG_CHECK(num_seqs >= 0 && n_used >= 0, "decode_begin: negative size");
  TG_CHECK(aligned16(rope), "decode_begin: rope must be 16-byte aligned");
  if (num_seqs == 0) return 0;
  hipLaunchKernelGGL(decode_begin_kernel, dim3((unsigned)num_seqs), dim3(64), 0, stream, positions, inv_freq,
                     reinterpret_cast<float2 *>(rope), kv_used, n_used, slots, ratio);
  TG_HIP_CHECK(hipGetLastError());
  return 0;
}
