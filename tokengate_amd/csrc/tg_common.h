// Shared device helpers for the gfx950 kernels: vector types, MFMA wrappers, LDS access,
// cross-lane reductions, and the thread-local error string behind tg_last_error().
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

namespace tg {

typedef uint16_t bf16_t;  // raw bf16 bits in global memory

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// ---- host-side error reporting -------------------------------------------------------------
int set_error(const char *fmt, ...);   // formats into the thread-local buffer, returns 1
void clear_error();
const char *last_error();

#define TG_CHECK(cond, ...)                 \
  do {                                      \
    if (!(cond)) return ::tg::set_error(__VA_ARGS__); \
  } while (0)

#define TG_HIP_CHECK(expr)                                                              \
  do {                                                                                  \
    hipError_t _e = (expr);                                                             \
    if (_e != hipSuccess)                                                               \
      return ::tg::set_error("%s failed: %s", #expr, hipGetErrorString(_e));            \
  } while (0)

// ---- device helpers -----------------------------------------------------------------------

// C = A(32x16) * B(16x32) + C on the bf16 matrix cores.  Lane l holds A[l%32][8*(l/32)+j] and
// B[8*(l/32)+j][l%32] for j=0..7; C value v sits at row 8*(v/4)+4*(l/32)+(v%4), column l%32.
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// 16-byte LDS load / store at a byte offset into a __shared__ buffer.
__device__ __forceinline__ bf16x8 lds_load16(const char *base, uint32_t byte_off) {
  return *reinterpret_cast<const bf16x8 *>(base + byte_off);
}
__device__ __forceinline__ void lds_store16(char *base, uint32_t byte_off, u32x4 v) {
  *reinterpret_cast<u32x4 *>(base + byte_off) = v;
}
__device__ __forceinline__ void lds_store8(char *base, uint32_t byte_off, u32x2 v) {
  *reinterpret_cast<u32x2 *>(base + byte_off) = v;
}

// 16-byte global load with a validity predicate (zero when invalid, no access made).
__device__ __forceinline__ u32x4 gload16(const bf16_t *p, bool valid) {
  u32x4 r = {0u, 0u, 0u, 0u};
  if (valid) r = *reinterpret_cast<const u32x4 *>(p);
  return r;
}

// Combine a value held by lane l and lane l^32 (the two halves of a wave64).
__device__ __forceinline__ float pair_max(float x) { return fmaxf(x, __shfl_xor(x, 32)); }
// Reinterpret a 32-bit value as float.  Use this (or a copy into a scalar) instead of applying
// __builtin_bit_cast to an element of a vector or of a builtin's result pair directly: this
// compiler lowers __builtin_bit_cast(float, v[i]) to element 0 whatever i is.
__device__ __forceinline__ float u32_as_f32(uint32_t u) { return __builtin_bit_cast(float, u); }
// max of the two values a permlane swap returns.  A bare v_max_f32: fmaxf would first
// canonicalise both operands (two more VALU instructions), which only matters for signalling
// NaNs, and the values reduced here are arithmetic results, never signalling NaNs.
template <typename Pair> __device__ __forceinline__ float swap_pair_max(const Pair &sw) {
  const uint32_t lo = sw[0], hi = sw[1];
  float d;
  asm("v_max_f32 %0, %1, %2" : "=v"(d) : "v"(u32_as_f32(lo)), "v"(u32_as_f32(hi)));
  return d;
}
// Same as pair_max without the LDS crossbar: v_permlane32_swap(x, x) returns (lower half in both
// halves, upper half in both halves), so the max of the two is max(x[l], x[l^32]) in every lane.
__device__ __forceinline__ float half_swap_max(float x) {
  return swap_pair_max(__builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x),
                                                        __builtin_bit_cast(uint32_t, x), false, false));
}
__device__ __forceinline__ float pair_sum(float x) { return x + __shfl_xor(x, 32); }
// Max over the four 16-lane groups (lanes l, l^16, l^32, l^48): v_permlane16_swap(x, x) returns
// (rows 0 and 2 in both rows of each pair, rows 1 and 3 likewise), whose max is max(x[l], x[l^16]);
// then the same across the two halves.
__device__ __forceinline__ float quad_swap_max(float x) {
  return half_swap_max(swap_pair_max(__builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x),
                                                                      __builtin_bit_cast(uint32_t, x), false, false)));
}
__device__ __forceinline__ float quad_sum(float x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}
// C = A(16x32) * B(32x16) + C on the bf16 matrix cores.  Lane l holds A[l%16][8*(l/16)+j] and
// B[8*(l/16)+j][l%16] for j=0..7; C value i sits at row 4*(l/16)+i, column l%16.
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ---- buffer resources and LDS DMA (gfx950) --------------------------------------------------
typedef __amdgpu_buffer_rsrc_t brsrc_t;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4_t;

// Raw buffer descriptor over [base, base + num_bytes): loads past num_bytes return zero and
// make no memory access.
__device__ __forceinline__ brsrc_t make_rsrc(const void *base, uint32_t num_bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)num_bytes, 0x00020000);
}
// Asynchronous 16-byte-per-lane copy global -> LDS: lane i's 16 bytes land at
// lds_wave_base + 16*i.  Completion is tracked by vmcnt.
__device__ __forceinline__ void dma16(brsrc_t rs, void *lds_wave_base, uint32_t voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t *)lds_wave_base, 16, voff, 0, 0, 0);
}
// Same, 4 bytes per lane (lds_wave_base + 4*i).
__device__ __forceinline__ void dma4(brsrc_t rs, void *lds_wave_base, uint32_t voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t *)lds_wave_base, 4, voff, 0, 0, 0);
}
// Transposing LDS read (ds_read_b64_tr_b16): within each group of 16 lanes, lane j receives
// element j%4 of the four 16-bit values addressed by lanes 4k + j/4, for k = 0..3.
__device__ __forceinline__ s16x4 lds_read_tr16(const void *lds_addr) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t *)lds_addr);
}
__device__ __forceinline__ void wait_all_mem() { __builtin_amdgcn_s_waitcnt(0); }
// Wait for this wave's outstanding vector-memory operations down to N (compile-time, 0..63).
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt is six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}
// Workgroup barrier for LDS ring buffers filled by LDS DMA: this wave's LDS reads are complete
// (lgkmcnt 0) and every wave has arrived.  Unlike __syncthreads() it does not make the wave wait
// for its own DMA still in flight into other ring slots (those are waited for by count, wait_vm);
// the empty asm statements keep the compiler from moving LDS accesses across the barrier.
__device__ __forceinline__ void ring_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0); vmcnt and expcnt unconstrained
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// Sum of 2 x 8 accumulators over the GR groups of CW waves of a workgroup, through LDS: group g adds up
// accumulators acc[.][DB g .. DB g + DB-1] (DB = 8 / GR) of all groups and is left with them in
// acc[.][0 .. DB-1].  d0 .. d3: GR LDS areas of merge_bytes() that no wave uses any more (the caller has
// synchronised the workgroup).
template <int GR, int CW> constexpr int merge_bytes() { return (GR - 1) * CW * 2 * (8 / GR) * 1024; }
template <int GR, int CW>
__device__ __forceinline__ void merge_groups(f32x4 (&acc)[2][8], int grp, int cw, int lane, char *d0, char *d1, char *d2,
                                             char *d3) {
  typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
  typedef __attribute__((address_space(3))) char lds_char;
  constexpr int DB = 8 / GR;
  // (selects of values: a branch on the group, or a conditional between two elements of acc, which is a
  // conditional between their addresses, leaves acc in scratch memory)
  auto piece = [&](int r, int d, int g) {
    f32x4 v = acc[r][d];
#pragma unroll
    for (int i = 1; i < GR; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = acc[r][i * DB + d][e], y = v[e];
        v[e] = g == i ? x : y;
      }
    return v;
  };
  auto area = [&](int g) { return (lds_char *)(g == 0 ? d0 : g == 1 ? d1 : g == 2 ? d2 : d3); };
  f32x4 own[2][DB];
#pragma unroll
  for (int j = 0; j < GR; ++j) {
    const int g = (grp + j) & (GR - 1);   // the pieces of group g; a group's area holds its peers in turn
    lds_char *p = area(g) + ((GR - 1 - j) * CW + cw) * 2 * DB * 1024 + lane * 16;
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        const f32x4 v = piece(r, d, g);
        if (j == 0) own[r][d] = v;
        else *reinterpret_cast<lds_f32x4 *>(p + (r * DB + d) * 1024) = v;
      }
  }
  __syncthreads();
  lds_char *src = area(grp);
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      f32x4 v = own[r][d];
#pragma unroll
      for (int i = 0; i < GR - 1; ++i)   // the groups after this one, in turn
        v += *reinterpret_cast<lds_f32x4 *>(src + ((i * CW + cw) * 2 * DB + r * DB + d) * 1024 + lane * 16);
      acc[r][d] = v;
    }
}

// Wait until at most n (0..63) vector-memory operations of this wave are outstanding (vmcnt: low
// four bits in [3:0], high two in [15:14]), leaving the LDS and export counters unconstrained.
__device__ __forceinline__ void wait_vm_outstanding(int n) {
#define TG_VMCNT(N) case N: __builtin_amdgcn_s_waitcnt(((N) & 15) | (((N) >> 4) << 14) | 0x0F70); break;
#define TG_VMCNT8(B) TG_VMCNT(B) TG_VMCNT(B + 1) TG_VMCNT(B + 2) TG_VMCNT(B + 3) TG_VMCNT(B + 4) TG_VMCNT(B + 5) \
  TG_VMCNT(B + 6) TG_VMCNT(B + 7)
  switch (n) {
    TG_VMCNT8(0) TG_VMCNT8(8) TG_VMCNT8(16) TG_VMCNT8(24) TG_VMCNT8(32) TG_VMCNT8(40) TG_VMCNT8(48)
    TG_VMCNT(56) TG_VMCNT(57) TG_VMCNT(58) TG_VMCNT(59) TG_VMCNT(60) TG_VMCNT(61) TG_VMCNT(62)
    default: __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | 0x0F70); break;
  }
#undef TG_VMCNT8
#undef TG_VMCNT
}

// Sum over the 64 lanes, in every lane, without the LDS crossbar.
__device__ __forceinline__ int wave_sum_int(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, true);    // quad_perm 1 0 3 2
  x += __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, true);    // quad_perm 2 3 0 1
  x += __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, true);   // row_half_mirror
  x += __builtin_amdgcn_update_dpp(0, x, 0x140, 0xf, 0xf, true);   // row_mirror
  const auto r = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)x, false, false);
  const uint32_t y = r[0] + r[1];
  const auto h = __builtin_amdgcn_permlane32_swap(y, y, false, false);
  return (int)(h[0] + h[1]);
}

// Level order of the tiles of n <= 64 packed sequences: the longest sequence's last tile first, then
// level by level down, at each level (tile index) one tile of every sequence that has it.  Only tiles that
// exist are counted: workgroups are handed to an XCD's shader engines in strict rotation, so workgroups
// that leave at once between those that stay would unbalance the engines (six packed sequences of 260 to
// 4021 tokens, forward, profiled: sequence-major 185 us, heaviest first with the shorter sequences'
// missing tiles in between 205, in level order 178).  Tile i of the order, for every lane of the wave
// alike; seq < 0 past the end.  Every workgroup pays for it before its first load.  Up to 16 sequences: each lane
// adds up the tiles from a level of its own on, by a walk over the sequences; more: bisection over the levels,
// a sum over the lanes per step.  64 sequences of 500 tokens, 16 / 8 heads, forward / backward: sequence-major
// 169 / 573 us, in level order with a walk over sequences and levels 232 / 672 (6 us per workgroup),
// bisection 148 / 482; 64 of 100 tokens, 8 / 8 heads, backward 55, 145, 60.  The six sequences above, forward +
// backward: bisection 683 us, with the longest first at a level (whose places in the order then do not move
// when others join) 681, lane by level 677.
struct LevelTile {
  int seq, level;
  int n_tiles, row0, len;   // of that sequence: the lanes hold them, a load by its index would wait once more
};
template <int ROWS>
__device__ __forceinline__ LevelTile level_tile(const int32_t *cu, int n, int max_len, int i, int lane) {
  const int row0 = lane < n ? cu[lane] : 0, len = lane < n ? max(0, min(cu[lane + 1] - row0, max_len)) : 0;
  const int nt = (len + ROWS - 1) / ROWS, levels = (int)(((uint32_t)max(1, max_len) + (ROWS - 1)) / ROWS);   // >= 1
  int level = 0, above = 0;   // the tile's level and the tiles above it
  int place = 0;              // of this lane's sequence among those that reach the level
  if (n <= 16) {
    int s = (levels + 63) >> 6;
    while (true) {
      const int l = level + s * lane;
      int t = 0;   // tiles at level l and above, falling from lane to lane
      for (int j = 0; j < n; ++j) t += max(0, __builtin_amdgcn_readlane(nt, j) - l);
      const int k = __builtin_popcountll(__builtin_amdgcn_ballot_w64(t > i));
      if (k == 0) return LevelTile{-1, 0, 0, 0, 0};
      level += s * (k - 1);
      above = k < 64 ? __builtin_amdgcn_readlane(t, k) : above;
      if (s == 1) break;
      s = (s + 63) >> 6;
    }
    for (int j = 0; j < n; ++j) {   // by tiles, ties by index
      const int tj = __builtin_amdgcn_readlane(nt, j);
      place += (tj > nt || (tj == nt && j < lane)) ? 1 : 0;
    }
  } else {
    auto from = [&](int l) { return __builtin_amdgcn_readfirstlane(wave_sum_int(max(0, nt - l))); };
    if (i >= from(0)) return LevelTile{-1, 0, 0, 0, 0};
    int hi = levels;   // from(level) > i >= above = from(hi)
    while (hi - level > 1) {
      const int mid = (level + hi) >> 1, t = from(mid);
      if (t > i) {
        level = mid;
      } else {
        hi = mid;
        above = t;
      }
    }
    const uint64_t m = __builtin_amdgcn_ballot_w64(nt > level);
    place = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
  }
  const int seq = (int)__builtin_ctzll(__builtin_amdgcn_ballot_w64(nt > level && place == i - above));
  return LevelTile{seq, level, __builtin_amdgcn_readlane(nt, seq), __builtin_amdgcn_readlane(row0, seq),
                   __builtin_amdgcn_readlane(len, seq)};
}

// Index of this wave in its workgroup, held in a scalar register.  The compiler cannot prove that
// threadIdx.x / 64 is the same in every lane of a wave, so without this every condition derived
// from the wave index (tile skips, mask checks) is compiled as exec-masked per-lane code that
// runs on every path instead of a scalar branch.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Two floats -> packed bf16 pair (round to nearest even, v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  bf16x2 p;
  p[0] = (__bf16)lo;
  p[1] = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, p);
}

// acc + lo + hi of a packed bf16 pair, in fp32 (v_dot2c_f32_bf16 against (1, 1)).
__device__ __forceinline__ float sum_bf16x2(uint32_t pair, float acc) {
  bf16x2 one;
  one[0] = (__bf16)1.0f;
  one[1] = (__bf16)1.0f;
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), one, acc, false);
}

__device__ __forceinline__ float bf16_to_f32(bf16_t x) {
  return __builtin_bit_cast(float, (uint32_t)x << 16);
}

// ---- rows of bf16 in 16-byte pieces -------------------------------------------------------------
__device__ __forceinline__ void unpack8(u32x4 v, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __builtin_bit_cast(float, v[i] << 16);
    f[2 * i + 1] = __builtin_bit_cast(float, v[i] & 0xffff0000u);
  }
}
__device__ __forceinline__ u32x4 pack8(const float (&f)[8]) {
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = pack_bf16x2(f[2 * i], f[2 * i + 1]);
  return v;
}
__device__ __forceinline__ u32x4 ld16(const bf16_t *p) { return *reinterpret_cast<const u32x4 *>(p); }
__device__ __forceinline__ void st16(bf16_t *p, u32x4 v) { *reinterpret_cast<u32x4 *>(p) = v; }

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) x += __shfl_xor(x, m);
  return x;
}


// RMSNorm and rotary embedding of one 128-element head row held by 16 lanes: lane j has elements 8j ..
// 8j+7 in x and their norm weights in wf, the rotate-half partner 8j+-64 sits in lane j^8; cs[e] is
// (cos, sin) of frequency (8j + e) % 64.  y = hs * bf16(rotated), rounded by the caller.  The fused
// multiply-adds are written out, so that every kernel that rotates a row gets the same bits.
constexpr int kHeadDim = 128;
__device__ __forceinline__ void norm_rope8(float (&x)[8], const float (&wf)[8], float eps,
                                           const float (*cs)[2], int j, float hs, float (&y)[8]) {
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss = fmaf(x[e], x[e], ss);
  ss += __shfl_xor(ss, 1);
  ss += __shfl_xor(ss, 2);
  ss += __shfl_xor(ss, 4);
  ss += __shfl_xor(ss, 8);
  const float rinv = rsqrtf(ss * (1.f / kHeadDim) + eps);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = wf[e] * (x[e] * rinv);
  const float sgn = j < 8 ? -1.f : 1.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float p = __shfl_xor(x[e], 8);
    y[e] = hs * (float)(__bf16)fmaf(x[e], cs[e][0], sgn * p * cs[e][1]);
  }
}

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Estimated time, in microseconds, of a launch of `units` times n workgroups issued heaviest first to
// `slots` places; steps(r) is the work of the r-th heaviest.  A workgroup takes `wg` plus `full` per step
// while the chip is full and `solo` while the longest run on alone, so the launch takes at least its
// heaviest workgroup, its work over the places plus one start per round, and k + 1 times the
// (k slots + 1)-th heaviest workgroup.
template <typename F>
float grid_cost(int n, int64_t units, int64_t slots, float wg, float solo, float full, F steps) {
  int64_t total = 0;
  for (int r = 0; r < n; ++r) total += steps(r);
  const int64_t rounds = (n * units + slots - 1) / slots;
  const float even = full * total * units / slots + rounds * wg;
  float cost = solo * steps(0) + wg;
  cost = cost < even ? even : cost;
  for (int64_t k = 1; k < rounds; ++k) {
    const float c = (k + 1) * (solo * steps((int)(k * slots / units)) + wg);
    cost = cost < c ? c : cost;
  }
  return cost;
}

// Whether a varlen attention launch is small: up to 64 sequences (as many as one wave orders) and K/V of at most
// half the 256 MB last-level cache.
inline bool varlen_small(int num_seqs, int64_t key_rows, int num_heads_k) {
  return num_seqs <= 64 && key_rows * num_heads_k * 512 <= (128ll << 20);
}
// Whether a varlen attention launch takes its tiles in level order, which packs the CUs best but streams
// every sequence's K/V at once: small causal launches (without the mask a tile's work does not depend on its
// level, and the short sequences' tiles only come between those that share a long one's K/V: 8192 and 4096
// tokens, 8 / 8 heads, forward 329 us sequence-major, 411 in level order; backward 1121 and 1245).  Six packed
// sequences of 260 to 4021 tokens (48 MB): forward + backward 761 -> 674 us against sequence-major, four of
// 2048 forward 106 -> 74; eight prompts of 16k to 128k (2.9 GB) ran at 682 TFLOP/s heaviest first and 996
// sequence-major.
inline bool varlen_level_order(bool causal, int num_seqs, int64_t key_rows, int num_heads_k) {
  return causal && num_seqs > 1 && varlen_small(num_seqs, key_rows, num_heads_k);
}
// At most this many tiles of `rows` rows exist among total_rows rows of num_seqs sequences.
inline int64_t level_tiles(int num_seqs, int64_t total_rows, int rows) { return total_rows / rows + num_seqs; }

// Compute units of the current device (cached per device id).
inline int device_cus() {
  static int cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cache[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cache[dev] = n;
  }
  return cache[dev];
}

}  // namespace tg
