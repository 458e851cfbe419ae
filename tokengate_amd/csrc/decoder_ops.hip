// Per-token decoder work around the attention of the gated prefill, one HBM pass each:
//   * residual add + RMSNorm (the input / post-attention norms of a Qwen3 layer and the final norm),
//   * per-head q/k RMSNorm + rotary embedding at each token's own position, writing q in place
//     and k / v into the layer's KV cache rows,
//   * SiLU(gate) * up of the fused gate/up projection;
//   * for the few rows of a decode step: the projections, HBM-bound on the weight (a row form for rows of
//     up to 2048 inputs, a split-K form for longer ones), optionally with the RMSNorm or the SwiGLU
//     product folded into their input, or the SwiGLU product into their output; the counters and
//     rotary table that its layers share; and the greedy argmax over the logits.
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
__device__ __forceinline__ u32x4 norm8(const float (&v)[8], u32x4 nwv, float rinv) {
  float wf[8], y[8];
  unpack8(nwv, wf);
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = wf[e] * (v[e] * rinv);
  return pack8(y);
}
__device__ __forceinline__ u32x4 norm8(u32x4 sv, u32x4 nwv, float rinv) {
  float v[8];
  unpack8(sv, v);
  return norm8(v, nwv, rinv);
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
    return norm8(v, ld16(in.nw + c), rinv);
  }
}
// The order of every sum is fixed: lane l of a wave takes columns 8 l .. 8 l + 7 of each 512-column chunk,
// chunk by chunk, as bf16 pair dot products, and the 64 lanes are added as a butterfly.  (Other orders,
// the matrix cores' among them, flip about 1 in 5000 of the rounded outputs, which 28 layers of bf16 turn
// into 3 % of the logits.)
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
// Butterfly sum over the 16 lanes of a row (x += x[l ^ 1], ^ 2, ^ 4, ^ 8) without the LDS crossbar: pairs
// inside a quad, then mirrored halves of 8 and 16 lanes, whose quads / octets already agree.
__device__ __forceinline__ float row_sum_dpp(float x) {
  x += dpp<0xB1>(x);    // quad_perm 1 0 3 2
  x += dpp<0x4E>(x);    // quad_perm 2 3 0 1
  x += dpp<0x141>(x);   // row_half_mirror
  x += dpp<0x140>(x);   // row_mirror
  return x;
}
// a[l] + a[l ^ 16] in rows 0 and 2, b's in rows 1 and 3
__device__ __forceinline__ float swap16_add(float a, float b) {
  const auto sw = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                   false, false);
  const uint32_t lo = sw[0], hi = sw[1];
  return u32_as_f32(lo) + u32_as_f32(hi);
}
// a[l] + a[l ^ 32] in the lower half, b's in the upper
__device__ __forceinline__ float swap32_add(float a, float b) {
  const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                   false, false);
  const uint32_t lo = sw[0], hi = sw[1];
  return u32_as_f32(lo) + u32_as_f32(hi);
}
// The additions of wave_sum, so its bits
__device__ __forceinline__ float wave_sum_dpp(float x) {
  x = row_sum_dpp(x);
  x = swap16_add(x, x);
  return swap32_add(x, x);
}
// wave_sum of N values at once: the row swaps take two values each and leave value 4 k + r in row r of
// register k, so a value costs 4 + 1 + 1/2 additions instead of six and no select per value.  Lane l gets
// value wave_sums_index(l) (of N, if it is less).
template <int N>
__device__ __forceinline__ float wave_sums(const float (&v)[N], int lane) {
  constexpr int K = (N + 3) / 4;
  float y = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    float x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = 4 * k + i < N ? row_sum_dpp(v[4 * k + i < N ? 4 * k + i : 0]) : 0.f;
    const float t = swap32_add(swap16_add(x[0], x[1]), swap16_add(x[2], x[3]));
    y = (lane & 15) == k ? t : y;
  }
  return y;
}
__device__ __forceinline__ int wave_sums_index(int lane) { return 4 * (lane & 15) + (lane >> 4); }
// acc[r][b] += the 8 columns of weight row r times those of input row b
template <int RW>
__device__ __forceinline__ void lin_dot8(const u32x4 (&wv)[RW], u32x4 xv, float (&acc)[RW]) {
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t wd = wv[r][e], xd = xv[e];   // scalar copies: see u32_as_f32
      acc[r] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, wd), __builtin_bit_cast(bf16x2, xd), acc[r],
                                               false);
    }
}
template <typename OutT>
__device__ __forceinline__ void lin_store(OutT *p, float sum) {
  const __bf16 y = (__bf16)sum;
  if constexpr (std::is_same<OutT, float>::value) *p = (float)y;
  else *p = __builtin_bit_cast(bf16_t, y);
}
// Rows of at most 2048 inputs (512 NC; NC = 0: 512, 1024 or 1536).  A workgroup of 8 waves, each wave
// RW weight rows (ACT: RW / 2 outputs, their gate and up rows) per round.  The NR input rows are formed
// once per workgroup in LDS, requested before the weights (loads complete in issue order, so the stage
// runs while the weights stream in).  Before, workgroups of 16 rows formed them (or every wave read them
// for 4 rows: twice the weight's bytes at 8 input rows) and each of the 4 NR sums took six steps through
// the LDS crossbar.  Before -> now, weights from HBM, at 1 / 8 input rows (us): 4096 x 2048 with the norm
// 6.9 / 14.5 -> 4.8 / 7.5, 2048 x 2048 4.3 / 8.3 -> 3.3 / 4.3, 12288 x 2048 with the norm 12.4 / 28.6 ->
// 10.5 / 13.4 (and with the SwiGLU product 10.4 / 13.2), 151936 x 2048 with the norm 109 / 250 -> 105 /
// 117 (5.9 / 5.3 TB/s).  WALK: fewer workgroups than blocks, which walk them with the next round's weights
// in flight, so that the input stage is paid once for more of the weight.  NC = 0 requests its chunks one by
// one after the stage (more of them in flight cost eight rows up to 18 %, in registers), except for one input
// row (kAhead), whose chunks are requested before it: 4096 x 1024 4.0 -> 3.8 us, 4096 x 1536 4.95 -> 4.5 (with
// the norm and two weight rows the stage hides it: 6144 x 1024 5.1 against 5.2).
template <int NR, int RW, int NC, typename OutT, int PRE, bool ACT, bool WALK>
__global__ __launch_bounds__(512) void linear_rows_kernel(LinIn in, const bf16_t *__restrict__ w, int64_t n_out,
                                                          int dim, OutT *__restrict__ out, int64_t out_rs) {
  static_assert(!WALK || NC > 0, "the next round's weights are held in registers");
  constexpr int kXsRow = 2048, OW = ACT ? RW / 2 : RW;
  constexpr bool kAhead = NC > 0 || (NR == 1 && (RW != 2 || PRE != kPreNorm));
  constexpr int NCR = NC > 0 ? NC : kAhead ? 3 : 1;
  constexpr bool kRowWave = PRE == kPreNorm && NR >= 5 && RW <= 2;
  constexpr int kIn = kRowWave ? 4 : (NR + 1) / 2;   // rows of at most 2048
  __shared__ __attribute__((aligned(16))) bf16_t xs[NR * kXsRow];
  __shared__ float rinv_s[8];
  const int lane = threadIdx.x & 63, wv = wave_id();
  // The thread's 16-byte pieces of the input rows.  kRowWave: wave b forms row b, lane l its pieces l,
  // l + 64, ..., so that the norm needs neither LDS nor a barrier; with fewer rows, or four weight rows
  // per wave (whose registers leave no room), the pieces are dealt over all waves instead (4096 / 12288 x
  // 2048 with the norm, us, dealt and row per wave: 4.8 / 10.4 and 5.2 / 11.0 at one row, 6.5 / 11.3 and
  // 5.7 / 11.8 at four, 7.8 / 13.2 and 7.5 / 13.2 at eight; 151936 rows, eight rows: 115 and 131).
  u32x4 xin[kIn], rin[kIn], nwv[kIn];
  int row[kIn], col[kIn];
#pragma unroll
  for (int i = 0; i < kIn; ++i) {
    if constexpr (kRowWave) {
      col[i] = 8 * lane + 512 * i;
      row[i] = NC > 0 || col[i] < dim ? wv : NR;
    } else {
      const int groups = NC > 0 ? 64 * NC : dim / 8, idx = threadIdx.x + 512 * i;
      row[i] = idx / groups;
      col[i] = 8 * (idx - row[i] * groups);
    }
    if (row[i] < NR) {
      xin[i] = ld16(in.x + row[i] * in.x_rs + col[i]);
      if constexpr (PRE == kPreNorm) {
        if (in.res) rin[i] = ld16(in.res + row[i] * in.res_rs + col[i]);
        nwv[i] = ld16(in.nw + col[i]);
      } else if constexpr (PRE == kPreSwiGLU) {
        rin[i] = ld16(in.x + row[i] * in.x_rs + in.inter + col[i]);
      }
    }
  }
  const int64_t step = (int64_t)gridDim.x * (8 * OW);
  int64_t v0 = ((int64_t)blockIdx.x * 8 + wv) * OW;
  const bf16_t *wr[RW];
  auto rows_from = [&](int64_t v) {   // rows past the end read the last row (in bounds; not stored)
#pragma unroll
    for (int r = 0; r < RW; ++r)
      wr[r] = w + (min(v + r % OW, n_out - 1) + (r / OW) * n_out) * dim + 8 * lane;
  };
  auto load = [&](u32x4 (&wf)[RW], int ch) {
#pragma unroll
    for (int r = 0; r < RW; ++r) wf[r] = ld16(wr[r] + 512 * ch);
  };
  rows_from(v0);
  u32x4 wf[NCR][RW];
  if constexpr (kAhead)
#pragma unroll
    for (int ch = 0; ch < NCR; ++ch)
      if (NC > 0 || 512 * ch < dim) load(wf[ch], ch);
  // ---- input stage ----
  auto to_lds = [&](int i) { *reinterpret_cast<u32x4 *>(xs + row[i] * kXsRow + col[i]) = xin[i]; };
  if constexpr (PRE == kPreNorm) {
    // s = bf16(h + res) (block 0 also writes res_out); the sum of a row's squares is a lane's pieces element
    // by element, then the butterfly, as in the RMSNorm kernel
    const bool writer = blockIdx.x == 0 && in.res_out != nullptr;
#pragma unroll
    for (int i = 0; i < kIn; ++i)
      if (row[i] < NR) {
        if (in.res) {
          float v[8], r[8];
          unpack8(xin[i], v);
          unpack8(rin[i], r);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = (float)(__bf16)(v[e] + r[e]);
          xin[i] = pack8(v);
        }
        if (writer) st16(in.res_out + row[i] * in.ro_rs + col[i], xin[i]);
        if constexpr (!kRowWave) to_lds(i);
      }
    float ss = 0.f;
    auto squares = [&](u32x4 x) {
      float v[8];
      unpack8(x, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
    };
    if constexpr (kRowWave) {
#pragma unroll
      for (int i = 0; i < kIn; ++i)
        if (row[i] < NR) squares(xin[i]);
    } else {
      ring_barrier();
      if (wv < NR)
        for (int c = 8 * lane; c < dim; c += 512) squares(*reinterpret_cast<const u32x4 *>(xs + wv * kXsRow + c));
    }
    float rinv = rsqrtf(wave_sum_dpp(ss) / (float)dim + in.eps);
    if constexpr (!kRowWave) {
      if (wv < NR && lane == 0) rinv_s[wv] = rinv;
      ring_barrier();
    }
#pragma unroll
    for (int i = 0; i < kIn; ++i)
      if (row[i] < NR) {
        if constexpr (!kRowWave) rinv = rinv_s[row[i]];
        xin[i] = norm8(xin[i], nwv[i], rinv);
      }
  } else if constexpr (PRE == kPreSwiGLU) {
#pragma unroll
    for (int i = 0; i < kIn; ++i)
      if (row[i] < NR) xin[i] = swiglu8(xin[i], rin[i]);
  }
#pragma unroll
  for (int i = 0; i < kIn; ++i)
    if (row[i] < NR) to_lds(i);
  ring_barrier();
  // ---- rounds ----
  auto xrow = [&](int b, int ch) { return *reinterpret_cast<const u32x4 *>(xs + b * kXsRow + 512 * ch + 8 * lane); };
  do {
    if (!WALK && v0 >= n_out) return;   // (no barrier follows)
    float acc[NR][RW] = {};
    if constexpr (NC > 0) {
      u32x4 wn[WALK ? NC : 1][RW];
      if (WALK && v0 + step < n_out) {
        rows_from(v0 + step);
#pragma unroll
        for (int ch = 0; ch < NC; ++ch) load(wn[ch], ch);
      }
#pragma unroll
      for (int ch = 0; ch < NC; ++ch)
#pragma unroll
        for (int b = 0; b < NR; ++b) lin_dot8(wf[ch], xrow(b, ch), acc[b]);
      if constexpr (WALK)
#pragma unroll
        for (int ch = 0; ch < NC; ++ch)
#pragma unroll
          for (int r = 0; r < RW; ++r) wf[ch][r] = wn[ch][r];
    } else {
      if constexpr (kAhead) {
#pragma unroll
        for (int ch = 0; ch < NCR; ++ch)
          if (512 * ch < dim)
#pragma unroll
            for (int b = 0; b < NR; ++b) lin_dot8(wf[ch], xrow(b, ch), acc[b]);
      } else {
        for (int ch = 0; 512 * ch < dim; ++ch) {
          load(wf[0], ch);
#pragma unroll
          for (int b = 0; b < NR; ++b) lin_dot8(wf[0], xrow(b, ch), acc[b]);
        }
      }
    }
    // value b OW + o: output o of input row b
    float sums[NR * OW], ups[ACT ? NR * OW : 1];
#pragma unroll
    for (int b = 0; b < NR; ++b)
#pragma unroll
      for (int o = 0; o < OW; ++o) {
        sums[b * OW + o] = acc[b][o];
        if constexpr (ACT) ups[b * OW + o] = acc[b][OW + o];
      }
    float mine = wave_sums(sums, lane);
    if constexpr (ACT) {
      const float g = (float)(__bf16)mine, u = (float)(__bf16)wave_sums(ups, lane);
      mine = g / (1.f + __expf(-g)) * u;
    }
    const int vi = wave_sums_index(lane);
    const int64_t v = v0 + vi % OW;
    if (vi < NR * OW && v < n_out) lin_store(out + (vi / OW) * out_rs + v, mine);
    v0 += step;
  } while (WALK && v0 < n_out);
}

// Rows of more than 2048 inputs (the down projection, 6144): four waves per 4 weight rows, wave wv the
// 512-column chunks wv, wv + 4, wv + 8, ... of them, their partial sums added in wave order through LDS.
// When dim is 2048 * NJ (NJ = 3: 6144) a wave's inputs and then all its weights are requested at once;
// other multiples of 512 go chunk by chunk (NJ = 0).  2048 x 6144 at 1 / 8 input rows: 6.3 / 12.1 -> 6.0 /
// 8.8 us (the weights used to come first, so that the inputs' way was paid after theirs).
template <int NR, typename OutT, int PRE, int NJ>
__global__ __launch_bounds__(256) void linear_rows_splitk_kernel(LinIn in, const bf16_t *__restrict__ w, int64_t n_out,
                                                                 int dim, OutT *__restrict__ out, int64_t out_rs) {
  constexpr int R = 4, NJR = NJ > 0 ? NJ : 1;
  constexpr bool kAhead = NJ > 0 && (PRE == kPrePlain || (PRE == kPreSwiGLU && NR <= 2));
  __shared__ float part[4][NR][R];
  const int lane = threadIdx.x & 63, wv = wave_id();
  const int64_t v0 = (int64_t)blockIdx.x * R;
  // rows past the end read the last row (in bounds; not stored)
  const bf16_t *wr[R];
#pragma unroll
  for (int r = 0; r < R; ++r) wr[r] = w + min(v0 + r, n_out - 1) * dim + 512 * wv + 8 * lane;
  u32x4 xf[kAhead ? NJ : 1][NR], uf[kAhead && PRE == kPreSwiGLU ? NJ : 1][NR], wf[NJR][R];
  if constexpr (kAhead)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int b = 0; b < NR; ++b) {
        const bf16_t *p = in.x + b * in.x_rs + 512 * wv + 8 * lane + 2048 * j;
        xf[j][b] = ld16(p);
        if constexpr (PRE == kPreSwiGLU) uf[j][b] = ld16(p + in.inter);
      }
  if constexpr (NJ > 0)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < R; ++r) wf[j][r] = ld16(wr[r] + 2048 * j);
  float rinv[NR] = {};
  if constexpr (PRE == kPreNorm) {
    // sum of squares in the RMSNorm kernel's order
    const bool writer = blockIdx.x == 0 && wv == 0 && in.res_out != nullptr;
#pragma unroll
    for (int b = 0; b < NR; ++b) {
      float ss = 0.f;
      for (int c = 8 * lane; c < dim; c += 512) {
        float v[8];
        unpack8(ld16(in.x + b * in.x_rs + c), v);
        if (in.res) {
          float r[8];
          unpack8(ld16(in.res + b * in.res_rs + c), r);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = (float)(__bf16)(v[e] + r[e]);
        }
        if (writer) st16(in.res_out + b * in.ro_rs + c, pack8(v));
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
      }
      rinv[b] = rsqrtf(wave_sum_dpp(ss) / (float)dim + in.eps);
    }
  }
  float acc[NR][R] = {};
  if constexpr (NJ > 0) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int b = 0; b < NR; ++b) {
        u32x4 x;
        if constexpr (!kAhead) x = lin_input<PRE>(in, b, 512 * wv + 8 * lane + 2048 * j, rinv[b]);
        else if constexpr (PRE == kPreSwiGLU) x = swiglu8(xf[j][b], uf[j][b]);
        else x = xf[j][b];
        lin_dot8(wf[j], x, acc[b]);
      }
  } else {
    for (int c = 512 * wv; c < dim; c += 2048) {
#pragma unroll
      for (int r = 0; r < R; ++r) wf[0][r] = ld16(wr[r] + c - 512 * wv);
#pragma unroll
      for (int b = 0; b < NR; ++b) lin_dot8(wf[0], lin_input<PRE>(in, b, c + 8 * lane, rinv[b]), acc[b]);
    }
  }
  float sums[NR * R];
#pragma unroll
  for (int b = 0; b < NR; ++b)
#pragma unroll
    for (int r = 0; r < R; ++r) sums[b * R + r] = acc[b][r];
  const float mine = wave_sums(sums, lane);
  const int vi = wave_sums_index(lane);
  if (vi < NR * R) part[wv][vi / R][vi % R] = mine;
  __syncthreads();
  const int t = threadIdx.x;
  if (t < R * NR && v0 + t % R < n_out) {
    const int b = t / R, r = t % R;
    lin_store(out + b * out_rs + v0 + r, ((part[0][b][r] + part[1][b][r]) + part[2][b][r]) + part[3][b][r]);
  }
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
// index) pairs are folded across the wave and, through LDS, across the 16 waves.  The scan is bound by the
// VALU of the row's one CU, and in nearly every piece some lane of a wave finds a new best, so a piece only
// updates the best value and its piece's number (5.5 instructions; the element inside the piece is found
// afterwards, from one more read of it).  Its maxima propagate NaNs: a row with a NaN is scanned again for the
// first one.  151936 columns: value, NaN and index compared per element 25 us, now 9.5 (with a NaN 15).
__device__ __forceinline__ bool amax_better(float a, int64_t ia, float b, int64_t ib) {
  const bool na = a != a, nb = b != b;
  if (na) return nb ? ia < ib : true;
  if (nb) return false;
  return a == b ? ia < ib : a > b;
}
__global__ __launch_bounds__(1024) void argmax_rows_kernel(const float *__restrict__ x, int64_t rs, int64_t n,
                                                           int64_t *__restrict__ out) {
  constexpr int kAhead = 8;   // independent loads in flight per thread
  const float *row = x + (int64_t)blockIdx.x * rs;
  const int64_t n4 = n / 4;
  auto load = [&](int64_t i) { return *reinterpret_cast<const f32x4 *>(row + 4 * i); };
  // f(pieces j, j + 1024, ... of this thread, their number), kAhead at a time
  auto scan = [&](auto f) {
    int64_t j = threadIdx.x;
    int32_t k = 0;
    for (; j + (kAhead - 1) * 1024 < n4; j += kAhead * 1024, k += kAhead) {
      f32x4 v[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) v[u] = load(j + u * 1024);
#pragma unroll
      for (int u = 0; u < kAhead; u += 2) f(v[u], v[u + 1], k + u);
    }
    for (; j < n4; j += 1024, ++k) {
      const f32x4 v = load(j);
      f(v, v, k);
    }
  };
  auto max4 = [](f32x4 v) {
    float m;
    asm("v_maximum3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(v[0]), "v"(v[1]), "v"(v[2]));
    asm("v_maximum3_f32 %0, %1, %2, %2" : "=v"(m) : "v"(m), "v"(v[3]));
    return m;
  };
  float best = -INFINITY, any = -INFINITY;   // any: NaN once a value is one
  int32_t at = 0;                            // the best's piece; the first of equals stays
  scan([&](f32x4 v0, f32x4 v1, int32_t k) {
    const float m0 = max4(v0), m1 = max4(v1);
    asm("v_maximum3_f32 %0, %0, %1, %2" : "+v"(any) : "v"(m0), "v"(m1));
    at = m0 > best ? k : at;
    best = m0 > best ? m0 : best;
    at = m1 > best ? k + 1 : at;
    best = m1 > best ? m1 : best;
  });
  bool nan = any != any;
  int64_t bi = n;   // no element: loses every comparison with a real one
  if (threadIdx.x < n4) {
    const int64_t i = threadIdx.x + 1024 * (int64_t)at;
    const f32x4 v = load(i);
    bi = 4 * i + (v[0] == best ? 0 : v[1] == best ? 1 : v[2] == best ? 2 : 3);
  }
  if (const int64_t i = 4 * n4 + threadIdx.x; i < n) {
    const float v = row[i];
    nan |= v != v;
    if (v > best || bi == n) { best = v; bi = i; }
  }
  if (__syncthreads_or(nan)) {
    int32_t first = -1;
    scan([&](f32x4 v0, f32x4 v1, int32_t k) {
      first = first < 0 && max4(v0) != max4(v0) ? k : first;
      first = first < 0 && max4(v1) != max4(v1) ? k + 1 : first;
    });
    best = -INFINITY;
    bi = n;
    if (first >= 0) {
      const int64_t i = threadIdx.x + 1024 * (int64_t)first;
      const f32x4 v = load(i);
      best = NAN;
      bi = 4 * i + (v[0] != v[0] ? 0 : v[1] != v[1] ? 1 : v[2] != v[2] ? 2 : 3);
    } else if (const int64_t i = 4 * n4 + threadIdx.x; i < n && row[i] != row[i]) {
      best = NAN;
      bi = i;
    }
  }
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

// n_out: stored outputs (ACT: weight holds 2 n_out rows, [gate; up]).
// Weight rows per wave and round (RW) and workgroups, us at 1 / 8 input rows, weights from HBM (before the
// lane sums shared their swaps, which took 0.3 to 1 us off every eight-row figure):
//   * under 4096 weight rows one each, for enough workgroups (2048 x 2048: RW 1 / 2 / 4 3.3 / 3.6 / 4.7 and
//     4.6 / 5.7 / 8.2);
//   * from 65536 (the LM head) four, half as many workgroups that form the input (151936 rows with the
//     norm: RW 2 / 4 110 / 104 and 143 / 123; walked, RW 2, 112 and 123);
//     With one or two plain rows of 1024 or 1536 inputs two (151936 x 1024 56.7 -> 54.3);
//   * between them two (4096 rows with the norm: RW 1 / 2 / 4 5.0 / 4.9 / 5.5 and 8.9 / 8.4 / 10.8); with two
//     blocks per CU and more, one workgroup per CU walks them (12288 rows with norm and SwiGLU: 10.4
//     against 10.3 and 14.1 against 16.9; two workgroups per CU 10.5 and 17.5).
template <int NR, typename OutT, int PRE, bool ACT>
void launch_linear_rows_nr(const LinIn &in, const bf16_t *w, int64_t n_out, int32_t dim, OutT *out, int64_t out_row_stride,
                           hipStream_t stream) {
  if (!ACT && dim > 2048) {
    // (4 weight rows per workgroup; 2 / 8 took 5.9 / 6.3 us against 6.1 at one row, 10.5 / 11.8 against
    // 9.7 at eight)
    constexpr int NJ = PRE != kPreNorm ? 3 : 0;
    const dim3 grid((unsigned)((n_out + 3) / 4)), block(256);
    if (dim == 2048 * NJ)
      hipLaunchKernelGGL((linear_rows_splitk_kernel<NR, OutT, PRE, NJ>), grid, block, 0, stream, in, w, n_out, dim, out,
                         out_row_stride);
    else
      hipLaunchKernelGGL((linear_rows_splitk_kernel<NR, OutT, PRE, 0>), grid, block, 0, stream, in, w, n_out, dim, out,
                         out_row_stride);
    return;
  }
  auto launch = [&](auto rw_c, auto nc_c, auto walk_c, int64_t grid) {
    constexpr int RW = decltype(rw_c)::value, NC = decltype(nc_c)::value;
    hipLaunchKernelGGL((linear_rows_kernel<NR, RW, NC, OutT, PRE, ACT, decltype(walk_c)::value>), dim3((unsigned)grid),
                       dim3(512), 0, stream, in, w, n_out, dim, out, out_row_stride);
  };
  auto with_rows = [&](auto rw_c) {
    constexpr int RW = decltype(rw_c)::value, rows = ACT ? 4 * RW : 8 * RW;
    typedef std::integral_constant<int, 4> C4;
    typedef std::integral_constant<int, 0> C0;
    const int64_t blocks = (n_out + rows - 1) / rows, cus = device_cus();
    if (dim != 2048) return launch(rw_c, C0(), std::false_type(), blocks);
    if constexpr (RW == 2)
      if (blocks >= 2 * cus) return launch(rw_c, C4(), std::true_type(), cus);
    launch(rw_c, C4(), std::false_type(), blocks);
  };
  const int64_t w_rows = ACT ? 2 * n_out : n_out;
  if constexpr (!ACT)
    if (w_rows < 4096) return with_rows(std::integral_constant<int, 1>());
  if (w_rows < 65536 || (PRE == kPrePlain && NR <= 2 && dim > 512 && dim < 2048))
    return with_rows(std::integral_constant<int, 2>());
  with_rows(std::integral_constant<int, 4>());
}
template <typename OutT, int PRE, bool ACT = false>
int launch_linear_rows(const LinIn &in, int32_t n_rows, const void *weight, int64_t n_out, int32_t dim, OutT *out,
                       int64_t out_row_stride, hipStream_t stream) {
  const bf16_t *w = static_cast<const bf16_t *>(weight);
#define TG_LR(NR) \
  case NR: launch_linear_rows_nr<NR, OutT, PRE, ACT>(in, w, n_out, dim, out, out_row_stride, stream); break;
  switch (n_rows) { TG_LR(1) TG_LR(2) TG_LR(3) TG_LR(4) TG_LR(5) TG_LR(6) TG_LR(7) TG_LR(8) }
#undef TG_LR
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
  TG_CHECK(dim <= 2048, "linear_rows_norm_act: dim must be at most 2048 (got %d)", dim);
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
