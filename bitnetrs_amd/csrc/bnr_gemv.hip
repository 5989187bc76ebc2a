// bnr_gemv.hip -- W2A8 ternary GEMV for gfx950 (Backend::ternary_gemv_preq).
//
// out[i] = (float)(sum_j W[i][j] * a[j]) * scale, with W in {-1, 0, +1}
// stored 2 bits per weight (row-aligned, ceil(K/4) bytes per row; code
// 0b00 -> +1, 0b01 -> 0, 0b10 -> -1, 0b11 -> 0, weight 4b+p at bits 2p of
// byte b) and a[] int8.  The integer sum is exact, so the result is
// bit-identical to the reference's (bitnet-cpu/src/gemv.rs:251-310).
//
// Memory-bound: each packed weight byte is read once.  A workgroup owns 16
// rows, 16 lanes per row; a lane takes the row's 16-byte pieces j, j+16, ...
// (64 weights each).  The K activations are staged in LDS once per workgroup
// and pass (4096 per pass), transposed so that one v_dot4_i32_i8 pairs four
// decoded weights with their activations without unpacking the 2-bit codes
// into bytes.
#include "bnr_internal.h"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace bnr {
namespace {

// 16 bytes with the non-temporal hint (global_load_dwordx4 ... nt), for
// weights: a decode token streams every matrix once (524 MB of ternary
// weights and 328 MB of LM head per token, more than the 256 MB MALL).
// Measured on MI355X: the 2B decode token 1.112 -> 1.069 ms, the
// 128256 x 2560 LM head 62.7-64.2 -> 57.9-58.8 us.
__device__ __forceinline__ uint4 ld16_nt(const void *p) {
  typedef unsigned u4v __attribute__((ext_vector_type(4)));
  const u4v v = __builtin_nontemporal_load(reinterpret_cast<const u4v *>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}

constexpr int kRowsPerWg = 16;
constexpr int kPass = 4096;                 // activations per LDS pass
constexpr int kGroups = kPass / 16;         // 16-activation groups per pass
constexpr int kPieces = kPass / 64;         // 16-byte weight pieces per row and pass
constexpr int kPiecesPerLane = kPieces / 16;

// Decode tables for v_perm_b32, whose selector bytes 0 .. 3 take that byte of
// the table, 4 .. 7 a byte of a zero word, 8 the sign of the table's byte 1 and
// 12 zero.  For codes in bits 0 and 1 of a byte (selectors 0 .. 3) byte c of
// kCodeLow is the int8 value of code c (+1, 0, -1, 0); for codes left in bits 2
// and 3 (selectors 0, 4, 8, 12) kCodeHigh gives the same values.
constexpr unsigned kCodeLow = 0x00FF0001u, kCodeHigh = 0x00008001u;

// One packed dword w = weights 16g .. 16g+15 (weight 16g + 4k + p at bits
// 8k + 2p): the codes of weights 4k + p, k = 0..3, are masked out of its four
// bytes (p = 0 and 1 of w, 2 and 3 of w >> 4) and mapped to their values.
// act.{x,y,z,w} hold the activations of the same positions for p = 0, 1, 2, 3.
__device__ __forceinline__ int dot16(unsigned w, uint4 act, int acc) {
  const unsigned lo = 0x03030303u, hi = 0x0C0C0C0Cu, v = w >> 4;
  acc = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_perm(0u, kCodeLow, w & lo), (int)act.x, acc, false);
  acc = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_perm(0u, kCodeHigh, w & hi), (int)act.y, acc, false);
  acc = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_perm(0u, kCodeLow, v & lo), (int)act.z, acc, false);
  acc = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_perm(0u, kCodeHigh, v & hi), (int)act.w, acc, false);
  return acc;
}

// 16 activations x0..x3 (dword t = activations 4t .. 4t+3) -> the four
// dwords dot16 expects: dword p = activations p, 4+p, 8+p, 12+p (a 4x4 byte
// transpose).
__device__ __forceinline__ uint4 transpose_bytes(uint4 x) {
  const unsigned t0 = __builtin_amdgcn_perm(x.y, x.x, 0x05010400u);  // x0b0 x1b0 x0b1 x1b1
  const unsigned t1 = __builtin_amdgcn_perm(x.y, x.x, 0x07030602u);  // x0b2 x1b2 x0b3 x1b3
  const unsigned t2 = __builtin_amdgcn_perm(x.w, x.z, 0x05010400u);  // x2b0 x3b0 x2b1 x3b1
  const unsigned t3 = __builtin_amdgcn_perm(x.w, x.z, 0x07030602u);  // x2b2 x3b2 x2b3 x3b3
  return make_uint4(__builtin_amdgcn_perm(t2, t0, 0x05040100u), __builtin_amdgcn_perm(t2, t0, 0x07060302u),
                    __builtin_amdgcn_perm(t3, t1, 0x05040100u), __builtin_amdgcn_perm(t3, t1, 0x07060302u));
}

template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float lanef(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}

// Sum over the 16 lanes of a DPP row.
__device__ __forceinline__ int row_sum16_i(int v) {
  v += dpp_i<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_i<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_i<0x141>(v);  // row_half_mirror
  v += dpp_i<0x140>(v);  // row_mirror
  return v;
}
// Sum over aligned groups of L = 4, 8 or 16 lanes, in the group's first lane.
template <int L>
__device__ __forceinline__ int lane_group_sum_i(int v) {
  v += dpp_i<0xB1>(v);
  v += dpp_i<0x4E>(v);
  if (L >= 8) v += dpp_i<0x141>(v);
  if (L >= 16) v += dpp_i<0x140>(v);
  if (L >= 32) {
    const auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    v = (int)((unsigned)r[0] + (unsigned)r[1]);
  }
  if (L >= 64) {
    const auto r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    v = (int)((unsigned)r[0] + (unsigned)r[1]);
  }
  return v;
}

// Bytes [off, off+16) of p, the ones at or past `limit` read as zero.
__device__ __forceinline__ uint4 load16_bounded(const uint8_t *p, long long off, long long limit) {
  unsigned d[4] = {0u, 0u, 0u, 0u};
  for (int b = 0; b < 16; ++b)
    if (off + b < limit) d[b >> 2] |= (unsigned)p[off + b] << (8 * (b & 3));
  return make_uint4(d[0], d[1], d[2], d[3]);
}

// Rows [16*wg, 16*wg+16) of one matrix: out[row] = (float)dot * scale.
// VEC: rows start 16-byte aligned with a whole number of 16-byte pieces
// (ceil(K/4) % 16 == 0) and the activations are 16-byte aligned.
template <bool VEC>
__device__ __forceinline__ void gemv_rows(const uint8_t *w, const int8_t *act, float *out,
                                          int out_features, int in_features,
                                          long long packed_cols, float scale, int wg,
                                          uint4 *s_act) {
  const int tid = threadIdx.x, slot = tid >> 4, j = tid & 15;
  const int row = wg * kRowsPerWg + slot;
  const long long prow = (long long)min(row, out_features - 1) * packed_cols;
  int acc = 0;
  for (int k0 = 0; k0 < in_features; k0 += kPass) {
    const int kn = min(kPass, in_features - k0);     // activations of this pass
    const long long b0 = prow + k0 / 4;              // first packed byte of the pass
    const int nb = (kn + 3) / 4;                     // packed bytes of the pass
    // Activation groups first: loads return in order, so the small,
    // cache-resident activations arrive (and go to LDS) while the weights
    // are still in flight.
    uint4 xa[kGroups / 256];
#pragma unroll
    for (int t = 0; t < kGroups / 256; ++t) {
      const int a0 = 16 * (tid + 256 * t);
      if (VEC && a0 + 16 <= kn) {
        xa[t] = *reinterpret_cast<const uint4 *>(act + k0 + a0);
      } else {
        xa[t] = load16_bounded(reinterpret_cast<const uint8_t *>(act), (long long)k0 + a0,
                               (long long)k0 + kn);
      }
    }
    uint4 wv[kPiecesPerLane];
#pragma unroll
    for (int i = 0; i < kPiecesPerLane; ++i) {
      const int c = j + 16 * i;
      if (VEC) {
        wv[i] = 16 * c < nb ? ld16_nt(w + b0 + 16 * c) : make_uint4(0, 0, 0, 0);
      } else {
        wv[i] = 16 * c < nb ? load16_bounded(w, b0 + 16 * c, b0 + nb) : make_uint4(0, 0, 0, 0);
      }
    }
    __syncthreads();  // the previous pass has finished reading s_act
#pragma unroll
    for (int t = 0; t < kGroups / 256; ++t) {
      const int g = tid + 256 * t;
      s_act[(g & 3) * kPieces + (g >> 2)] = transpose_bytes(xa[t]);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPiecesPerLane; ++i) {
      const int c = j + 16 * i;
      if (16 * c < nb) {
        acc = dot16(wv[i].x, s_act[c], acc);
        acc = dot16(wv[i].y, s_act[kPieces + c], acc);
        acc = dot16(wv[i].z, s_act[2 * kPieces + c], acc);
        acc = dot16(wv[i].w, s_act[3 * kPieces + c], acc);
      }
    }
  }
  acc = row_sum16_i(acc);
  if (j == 0 && row < out_features) out[row] = (float)acc * scale;
}

template <bool VEC>
__global__ __launch_bounds__(256) void ternary_gemv_kernel(TernaryGemvArgs a) {
  // Activations of the pass, transposed: group g (activations 16g..16g+15)
  // at s_act[(g % 4) * kPieces + g / 4], so that the 16 lanes of a row read
  // consecutive 16-byte slots.
  __shared__ uint4 s_act[kGroups];
  gemv_rows<VEC>(a.weight, a.act, a.out, a.out_features, a.in_features, a.packed_cols, a.scale,
                 blockIdx.x, s_act);
}

template <bool VEC>
__global__ __launch_bounds__(256) void ternary_gemv_group_kernel(TernaryGemvGroupArgs a) {
  __shared__ uint4 s_act[kGroups];
  const int b = blockIdx.x;
  // Matrix of this workgroup, selected with constant indices so that the
  // argument arrays stay in scalar registers.
  const uint8_t *w = a.weight[0];
  float *out = a.out[0];
  float scale = a.scale[0], ws = a.weight_scale[0];
  int m = a.out_features[0], off = 0;
#pragma unroll
  for (int i = 1; i < kMaxGemvGroup; ++i) {
    if (i < a.n && b >= a.wg_off[i]) {
      w = a.weight[i];
      out = a.out[i];
      scale = a.scale[i];
      ws = a.weight_scale[i];
      m = a.out_features[i];
      off = a.wg_off[i];
    }
  }
  if (a.act_absmax_dev) {
    // combined_scale = weight_scale * act_scale / 127.0 (gemv.rs:297), f32, left to right
    const float t = ws * *a.act_absmax_dev;
    scale = t / 127.0f;
  }
  gemv_rows<VEC>(w, a.act, out, m, a.in_features, a.packed_cols, scale, b - off, s_act);
}

// ---------------------------------------------------------------------------
// Ternary GEMV with the activation's RMSNorm and int8 quantisation as its
// prologue (the glue launch folded into the projection).  Every workgroup
// forms x from f32 inputs (a | a + b | max(a,0)^2 * b) and reduces sum(x^2) and
// max|y| with one tree, so that a launch's workgroups agree on every int8
// activation and on the scale; the int8 vector never leaves LDS.  The order of
// the sum is not norm_quant_kernel's, and differs between the forms here (quads
// over 256 or 512 threads, 16 consecutive values per thread): y agrees to
// rounding, and an activation at a half-way case may differ by one.  The aligned kernel below issues the (cache-resident) activation loads
// first and its weight loads right after, so the prologue runs under the
// weights' latency; the one here takes unaligned rows and vectors and any K <=
// 4096 NG (NG = 1 or 2 16-activation groups per thread), element by element.
// Workgroup 0 writes h_out (mode residual), which must not alias a or b.
// A workgroup of T threads owns T / LPR rows, LPR lanes per row: every workgroup reads
// the whole of a (and b) and gamma, so a launch with many rows takes 32 or
// 64 rows per workgroup to read those vectors fewer times.
// ---------------------------------------------------------------------------
constexpr int kNormK = 8192;

// x from the glue inputs: a | a + b | max(a, 0)^2 * b (mode kGlue*).
__device__ __forceinline__ float norm_x_of(int mode, float u, float v) {
#pragma clang fp contract(off)
  if (mode == kGlueResidual) return u + v;
  if (mode == kGlueSqrelu) {
    const float r = fmaxf(u, 0.0f);
    return r * r * v;
  }
  return u;
}

__device__ __forceinline__ float norm_x(const GemvNormArgs &p, int i) {
  return norm_x_of(p.mode, p.a[i], p.mode == kGluePlain ? 0.f : p.b[i]);
}

// Sum / max over the 64 lanes of a wave: DPP inside each 16-lane row, then
// the four row results (the same order in every wave).
__device__ __forceinline__ float wave_sum_f(float v) {
  v += dppf<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dppf<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dppf<0x141>(v);  // row_half_mirror
  v += dppf<0x140>(v);  // row_mirror
  return (lanef(v, 0) + lanef(v, 16)) + (lanef(v, 32) + lanef(v, 48));
}
__device__ __forceinline__ float wave_max_f(float v) {
  v = fmaxf(v, dppf<0xB1>(v));
  v = fmaxf(v, dppf<0x4E>(v));
  v = fmaxf(v, dppf<0x141>(v));
  v = fmaxf(v, dppf<0x140>(v));
  return fmaxf(fmaxf(lanef(v, 0), lanef(v, 16)), fmaxf(lanef(v, 32), lanef(v, 48)));
}

__device__ __forceinline__ float norm_y(float x, float inv, float g) {
#pragma clang fp contract(off)
  return x * inv * g;
}

template <int NG, int LPR>
__global__ __launch_bounds__(256) void ternary_gemv_norm_kernel(TernaryGemvGroupArgs a,
                                                                GemvNormArgs p) {
  constexpr int kNormGroupsPerThread = NG;
  constexpr int kNormPieces = 64 * NG;  // 16-byte weight pieces per row (K <= 4096 NG)
  constexpr int kNormPiecesPerLane = kNormPieces / LPR;
  constexpr int kRows = 256 / LPR;
  __shared__ uint4 s_act[256 * NG];
  __shared__ float red[4];
  const int tid = threadIdx.x, slot = tid / LPR, j = tid % LPR, lane = tid & 63, wv_id = tid >> 6;
  const int b = blockIdx.x;
  const uint8_t *w = a.weight[0];
  float *out = a.out[0];
  float ws = a.weight_scale[0];
  int m = a.out_features[0], off = 0;
#pragma unroll
  for (int i = 1; i < kMaxGemvGroup; ++i) {
    if (i < a.n && b >= a.wg_off[i]) {
      w = a.weight[i];
      out = a.out[i];
      ws = a.weight_scale[i];
      m = a.out_features[i];
      off = a.wg_off[i];
    }
  }
  const int K = a.in_features, nb = (K + 3) / 4;
  const int row = (b - off) * kRows + slot;
  const long long b0 = (long long)min(row, m - 1) * a.packed_cols;
  float x[kNormGroupsPerThread][16], g[kNormGroupsPerThread][16];
  // 2. this lane's weight pieces (in flight during the prologue)
  uint4 wq[kNormPiecesPerLane];
#pragma unroll
  for (int i = 0; i < kNormPiecesPerLane; ++i) {
    const int c = j + LPR * i;
    wq[i] = 16 * c < nb ? load16_bounded(w, b0 + 16 * c, b0 + nb) : make_uint4(0, 0, 0, 0);
  }
#pragma unroll
  for (int q = 0; q < kNormGroupsPerThread; ++q) {
    const int e0 = 16 * (tid + 256 * q);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int i = e0 + e;
      x[q][e] = i < K ? norm_x(p, i) : 0.f;
      g[q][e] = i < K ? p.gamma[i] : 0.f;
    }
  }
  // 3. sum of squares
  float ss = 0.f;
#pragma unroll
  for (int q = 0; q < kNormGroupsPerThread; ++q)
#pragma unroll
    for (int e = 0; e < 16; ++e) ss = fmaf(x[q][e], x[q][e], ss);
  if (p.h_out && b == 0) {
#pragma unroll
    for (int q = 0; q < kNormGroupsPerThread; ++q) {
      const int e0 = 16 * (tid + 256 * q);
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (e0 + e < K) p.h_out[e0 + e] = x[q][e];
    }
  }
  // block sum (4 waves); the same tree in every workgroup
  ss = wave_sum_f(ss);
  if (lane == 0) red[wv_id] = ss;
  __syncthreads();
  const float sum_sq = (red[0] + red[1]) + (red[2] + red[3]);
  const float inv = 1.0f / sqrtf(sum_sq / (float)K + p.eps);
  float mx = 0.f;
#pragma unroll
  for (int q = 0; q < kNormGroupsPerThread; ++q)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      x[q][e] = norm_y(x[q][e], inv, g[q][e]);  // zero past K (x = 0)
      mx = fmaxf(mx, fabsf(x[q][e]));
    }
  mx = wave_max_f(mx);
  __syncthreads();  // everyone has read red[] as sums
  if (lane == 0) red[wv_id] = mx;
  __syncthreads();
  const float mm = fmaxf(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])), 1e-5f);
  const float scale = mm / 127.0f, inv_scale = 127.0f / mm;
  // 3. int8 activations into LDS, transposed as the GEMV reads them
#pragma unroll
  for (int q = 0; q < kNormGroupsPerThread; ++q) {
    unsigned d[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      d[t] = 0u;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int qv = (int)fminf(fmaxf(roundf(x[q][4 * t + e] * inv_scale), -128.0f), 127.0f);
        d[t] |= (unsigned)(qv & 0xFF) << (8 * e);
      }
    }
    const int gi = tid + 256 * q;
    s_act[(gi & 3) * kNormPieces + (gi >> 2)] = transpose_bytes(make_uint4(d[0], d[1], d[2], d[3]));
  }
  __syncthreads();
  // 4. the projection
  int acc = 0;
#pragma unroll
  for (int i = 0; i < kNormPiecesPerLane; ++i) {
    const int c = j + LPR * i;
    if (16 * c < nb) {
      acc = dot16(wq[i].x, s_act[c], acc);
      acc = dot16(wq[i].y, s_act[kNormPieces + c], acc);
      acc = dot16(wq[i].z, s_act[2 * kNormPieces + c], acc);
      acc = dot16(wq[i].w, s_act[3 * kNormPieces + c], acc);
    }
  }
  acc = lane_group_sum_i<LPR>(acc);
  // combined_scale = weight_scale * act_scale / 127.0 (gemv.rs:297), act_scale = scale * 127
  const float t = ws * (scale * 127.0f);
  const float cs = t / 127.0f;
  if (j == 0 && row < m) out[row] = (float)acc * cs;
}

// int8 of v: round half away from zero, clamped.  trunc(v + 0.5 - 2^-25 with
// v's sign) is roundf(v) for |v| < 2^22: the sum of a half-way value rounds up
// to the next integer, that of the float below it does not.
__device__ __forceinline__ unsigned quant_byte(float v) {
  const float r = v + copysignf(0x1.fffffep-2f, v);
  return (unsigned)((int)fminf(fmaxf(r, -128.0f), 127.0f)) & 0xFFu;
}

// The aligned form (K % 64 == 0, 16-byte aligned rows and vectors).  Thread t
// forms the quads t, t + 256, ... of the activations (NQ >= K / 1024 of them):
// a wave's load takes 1 KB in a row.  The four lanes that hold a group of 16
// exchange bytes (two quad permutes) so that each stores one of the group's
// four dwords for dot16.  Everything before the weights are there is latency:
// three vectors from the other side of a kernel boundary, two block
// reductions; everything after is the decode.  Per launch of the two in a 2B
// feed-forward layer: 7.46 us with 16 consecutive activations per thread (a
// load then took 16 bytes of 64 lines, and 96 of the threads had none at K =
// 2560) and the library's roundf, 6.33 us with quads and 256 threads, 6.1 us
// with the workgroups below.
//
// T threads, LPR lanes per row: 16 or 32 rows in 256 threads; 64 rows in 512,
// where the launch is that long (gate + up: 216 workgroups read the vectors
// instead of 432, 6.4 -> 6.2 us on the average of gate + up and down); 16 rows
// in 512 past K = 4096, where the vectors are most of the prologue (down: 30
// layers 3 us less; q/k/v and o, at K = 2560, lose 0.4 us each in 512).
template <int NQ, int LPR, int T>
__global__ __launch_bounds__(T) void ternary_gemv_norm_vec_kernel(TernaryGemvGroupArgs a,
                                                                    GemvNormArgs p) {
  constexpr int kPcs = NQ * T / 16;  // 16-byte weight pieces per row
  constexpr int kPcsPerLane = (kPcs + LPR - 1) / LPR;
  constexpr int kRows = T / LPR, kWaves = T / 64;
  __shared__ unsigned s_act[16 * kPcs];  // group g: 4 dwords at 4 ((g % 4) kPcs + g / 4)
  __shared__ float red[2][kWaves];
  const int tid = threadIdx.x, slot = tid / LPR, j = tid % LPR, lane = tid & 63, wave = tid >> 6;
  const int b = blockIdx.x;
  const uint8_t *w = a.weight[0];
  float *out = a.out[0];
  float ws = a.weight_scale[0];
  int m = a.out_features[0], off = 0;
#pragma unroll
  for (int i = 1; i < kMaxGemvGroup; ++i) {
    if (i < a.n && b >= a.wg_off[i]) {
      w = a.weight[i];
      out = a.out[i];
      ws = a.weight_scale[i];
      m = a.out_features[i];
      off = a.wg_off[i];
    }
  }
  const int K = a.in_features, quads = K / 4, pcs = K / 64;
  const int row = (b - off) * kRows + slot;
  // 1. the activations' loads, ahead of the weights: loads return in order.
  // No branches between them: the second operand is a itself when the mode
  // has none; quads past K read quad 0 (discarded).
  const float *pb = p.mode == kGluePlain ? p.a : p.b;
  float4 xa[NQ], xb[NQ], xg[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int q = tid + T * i, o = q < quads ? 4 * q : 0;
    xa[i] = *reinterpret_cast<const float4 *>(p.a + o);
    xb[i] = *reinterpret_cast<const float4 *>(pb + o);
    xg[i] = *reinterpret_cast<const float4 *>(p.gamma + o);
  }
  __builtin_amdgcn_sched_barrier(0);
  // 2. this lane's weight pieces (in flight during the prologue)
  const uint8_t *wrow = w + (long long)min(row, m - 1) * a.packed_cols;
  uint4 wq[kPcsPerLane];
#pragma unroll
  for (int i = 0; i < kPcsPerLane; ++i) {
    const int c = j + LPR * i;
    wq[i] = c < pcs ? ld16_nt(wrow + 16 * c) : make_uint4(0, 0, 0, 0);
  }
  // 3. x, its sum of squares; the same tree in every workgroup
  float x[NQ][4], ss = 0.f;
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const bool in = tid + T * i < quads;
    x[i][0] = in ? norm_x_of(p.mode, xa[i].x, xb[i].x) : 0.f;
    x[i][1] = in ? norm_x_of(p.mode, xa[i].y, xb[i].y) : 0.f;
    x[i][2] = in ? norm_x_of(p.mode, xa[i].z, xb[i].z) : 0.f;
    x[i][3] = in ? norm_x_of(p.mode, xa[i].w, xb[i].w) : 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) ss = fmaf(x[i][e], x[i][e], ss);
  }
  if (p.h_out && b == 0) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int q = tid + T * i;
      if (q < quads)
        *reinterpret_cast<float4 *>(p.h_out + 4 * q) = make_float4(x[i][0], x[i][1], x[i][2], x[i][3]);
    }
  }
  ss = wave_sum_f(ss);
  if (lane == 0) red[0][wave] = ss;
  __syncthreads();
  float sum_sq = 0.f;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) sum_sq += red[0][i];
  const float inv = 1.0f / sqrtf(sum_sq / (float)K + p.eps);
  float mx = 0.f;
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const float g[4] = {xg[i].x, xg[i].y, xg[i].z, xg[i].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[i][e] = tid + T * i < quads ? norm_y(x[i][e], inv, g[e]) : 0.f;
      mx = fmaxf(mx, fabsf(x[i][e]));
    }
  }
  mx = wave_max_f(mx);
  if (lane == 0) red[1][wave] = mx;
  __syncthreads();
  float mm = 1e-5f;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) mm = fmaxf(mm, red[1][i]);
  const float scale = mm / 127.0f, inv_scale = 127.0f / mm;
  // 4. int8 activations: lane 4g + t holds activations 4t .. 4t+3 of its
  // group, and stores dword t: activations t, 4+t, 8+t, 12+t.
  const unsigned sel1 = (lane & 1) ? 0x03070105u : 0x06020400u;
  const unsigned sel2 = (lane & 2) ? 0x03020706u : 0x05040100u;
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    unsigned d = quant_byte(x[i][0] * inv_scale) | quant_byte(x[i][1] * inv_scale) << 8 |
                 quant_byte(x[i][2] * inv_scale) << 16 | quant_byte(x[i][3] * inv_scale) << 24;
    d = __builtin_amdgcn_perm((unsigned)dpp_i<0xB1>((int)d), d, sel1);  // lane ^ 1
    d = __builtin_amdgcn_perm((unsigned)dpp_i<0x4E>((int)d), d, sel2);  // lane ^ 2
    const int q = tid + T * i, g = q >> 2;
    s_act[4 * ((g & 3) * kPcs + (g >> 2)) + (q & 3)] = d;
  }
  __syncthreads();
  // 5. the projection
  const uint4 *act = reinterpret_cast<const uint4 *>(s_act);
  int acc = 0;
#pragma unroll
  for (int i = 0; i < kPcsPerLane; ++i) {
    const int c = j + LPR * i;
    if (c < pcs) {
      acc = dot16(wq[i].x, act[c], acc);
      acc = dot16(wq[i].y, act[kPcs + c], acc);
      acc = dot16(wq[i].z, act[2 * kPcs + c], acc);
      acc = dot16(wq[i].w, act[3 * kPcs + c], acc);
    }
  }
  acc = lane_group_sum_i<LPR>(acc);
  // combined_scale = weight_scale * act_scale / 127.0 (gemv.rs:297), act_scale = scale * 127
  const float t = ws * (scale * 127.0f);
  const float cs = t / 127.0f;
  if (j == 0 && row < m) out[row] = (float)acc * cs;
}

template <int LPR, int T>
hipError_t launch_norm_vec(const TernaryGemvGroupArgs &a, const GemvNormArgs &p, int wgs, hipStream_t s) {
  const dim3 grid(wgs), block(T);
  const int nq = (a.in_features + 4 * T - 1) / (4 * T);
  if (nq * T <= 768) ternary_gemv_norm_vec_kernel<(768 + T - 1) / T, LPR, T><<<grid, block, 0, s>>>(a, p);
  else if (nq * T <= 1024) ternary_gemv_norm_vec_kernel<1024 / T, LPR, T><<<grid, block, 0, s>>>(a, p);
  else if (nq * T <= 1792) ternary_gemv_norm_vec_kernel<(1792 + T - 1) / T, LPR, T><<<grid, block, 0, s>>>(a, p);
  else ternary_gemv_norm_vec_kernel<2048 / T, LPR, T><<<grid, block, 0, s>>>(a, p);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_ternary_gemv_norm(const TernaryGemvGroupArgs &a, const GemvNormArgs &p, bool vec,
                                    hipStream_t s) {
  const int wgs = a.wg_off[a.n];
  if (wgs <= 0) return hipSuccess;
  if (a.in_features > kNormK) return hipErrorInvalidValue;
  if (vec) {
    switch (p.rows) {
      case 16:
        return a.in_features > 4096 ? launch_norm_vec<32, 512>(a, p, wgs, s)
                                    : launch_norm_vec<16, 256>(a, p, wgs, s);
      case 32: return launch_norm_vec<8, 256>(a, p, wgs, s);
      case 64: return launch_norm_vec<8, 512>(a, p, wgs, s);
      default: return hipErrorInvalidValue;
    }
  }
  const bool one = a.in_features <= kNormK / 2;
  auto go = [&](auto kern) { kern<<<dim3(wgs), dim3(256), 0, s>>>(a, p); };
  switch (p.rows) {
    case 16: one ? go(ternary_gemv_norm_kernel<1, 16>) : go(ternary_gemv_norm_kernel<2, 16>); break;
    case 32: one ? go(ternary_gemv_norm_kernel<1, 8>) : go(ternary_gemv_norm_kernel<2, 8>); break;
    case 64: one ? go(ternary_gemv_norm_kernel<1, 4>) : go(ternary_gemv_norm_kernel<2, 4>); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_ternary_gemv_group(const TernaryGemvGroupArgs &a, bool vec, hipStream_t s) {
  const int wgs = a.wg_off[a.n];
  if (wgs <= 0) return hipSuccess;
  if (vec)
    ternary_gemv_group_kernel<true><<<dim3(wgs), dim3(256), 0, s>>>(a);
  else
    ternary_gemv_group_kernel<false><<<dim3(wgs), dim3(256), 0, s>>>(a);
  return hipGetLastError();
}

hipError_t launch_ternary_gemv(const TernaryGemvArgs &a, bool vec, hipStream_t s) {
  if (a.out_features <= 0) return hipSuccess;
  const dim3 grid((a.out_features + kRowsPerWg - 1) / kRowsPerWg);
  if (vec)
    ternary_gemv_kernel<true><<<grid, dim3(256), 0, s>>>(a);
  else
    ternary_gemv_kernel<false><<<grid, dim3(256), 0, s>>>(a);
  return hipGetLastError();
}

}  // namespace bnr

// ---------------------------------------------------------------------------
// LM head with i8 weights (CpuBackend::lm_head_matmul_i8_into,
// bitnet-cpu/src/lib.rs:544-575): out[v] = (sum_k w[v][k] * h[k]) * scale[v],
// w int8 [vocab x K], h f32 [K].  One HBM stream of vocab*K bytes (328 MB at
// 128256 x 2560): a workgroup owns 128 rows (8 blocks of 16 rows, 16 lanes
// per row, 16-byte pieces j, j+16, ... per lane) so that the hidden vector,
// staged in LDS once per pass of 4096 values, is reused over 320 KB of
// weights; the next block's pieces are loaded while the current block is
// multiplied.  fp32 products and sums (any order; the reference's AVX2 lane
// order is not reproduced, results agree to rounding).  For unaligned weights
// and K > kLmMaxK; the aligned form is lm_head_mfma_kernel.
// ---------------------------------------------------------------------------
namespace bnr {
namespace {

constexpr int kLmBlocks = 8;                     // row blocks of 16 per workgroup
constexpr int kLmPass = 4096;                    // hidden values per LDS pass
constexpr int kLmPieces = kLmPass / 16;          // 16-weight pieces per row and pass
constexpr int kLmPiecesPerLane = kLmPieces / 16;

__device__ __forceinline__ float row_sum16_f(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, false));
  return v;
}

// acc += the 4 signed bytes of d times h.x .. h.w
__device__ __forceinline__ float fma4_i8(unsigned d, float4 h, float acc) {
  acc = fmaf((float)(int)(signed char)(d & 0xFF), h.x, acc);
  acc = fmaf((float)(int)(signed char)((d >> 8) & 0xFF), h.y, acc);
  acc = fmaf((float)(int)(signed char)((d >> 16) & 0xFF), h.z, acc);
  acc = fmaf((float)((int)d >> 24), h.w, acc);
  return acc;
}

// VEC: rows 16-byte aligned (K % 16 == 0, weights aligned).
template <bool VEC>
__global__ __launch_bounds__(256) void lm_head_i8_kernel(LmHeadArgs a) {
  // hidden values 16c + 4t .. 16c + 4t + 3 of the pass at s_h[t * kLmPieces + c]
  __shared__ float4 s_h[kLmPass / 4];
  const int tid = threadIdx.x, slot = tid >> 4, j = tid & 15;
  const long long row0 = (long long)blockIdx.x * (16 * kLmBlocks) + slot;
  float acc[kLmBlocks][2];
#pragma unroll
  for (int b = 0; b < kLmBlocks; ++b) acc[b][0] = acc[b][1] = 0.f;
  for (int k0 = 0; k0 < a.hidden_size; k0 += kLmPass) {
    const int kn = min(kLmPass, a.hidden_size - k0);
    const int np = (kn + 15) / 16;  // pieces of the pass
    __syncthreads();                // previous pass done with s_h
    for (int g = tid; g < kLmPass / 4; g += 256) {
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      const int e = 4 * g;
      if (e + 4 <= kn) {
        v = *reinterpret_cast<const float4 *>(a.hidden + k0 + e);
      } else if (e < kn) {
        v.x = a.hidden[k0 + e];
        if (e + 1 < kn) v.y = a.hidden[k0 + e + 1];
        if (e + 2 < kn) v.z = a.hidden[k0 + e + 2];
      }
      s_h[(g & 3) * kLmPieces + (g >> 2)] = v;
    }
    __syncthreads();
    auto load = [&](int b, uint4 *wv) {
      const long long row = min(row0 + 16 * b, (long long)a.vocab_size - 1);
      const int8_t *wr = a.weight + row * a.hidden_size + k0;
#pragma unroll
      for (int i = 0; i < kLmPiecesPerLane; ++i) {
        const int c = j + 16 * i;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (c < np) {
          if (VEC) {
            v = ld16_nt(wr + 16 * c);
          } else {
            unsigned d[4] = {0u, 0u, 0u, 0u};
            for (int q = 0; q < 16; ++q)
              if (16 * c + q < kn) d[q >> 2] |= (unsigned)(uint8_t)wr[16 * c + q] << (8 * (q & 3));
            v = make_uint4(d[0], d[1], d[2], d[3]);
          }
        }
        wv[i] = v;
      }
    };
    uint4 wa[kLmPiecesPerLane], wb[kLmPiecesPerLane];
    load(0, wa);
#pragma unroll
    for (int b = 0; b < kLmBlocks; ++b) {
      uint4 *cur = (b & 1) ? wb : wa;
      uint4 *nxt = (b & 1) ? wa : wb;
      if (b + 1 < kLmBlocks) load(b + 1, nxt);
#pragma unroll
      for (int i = 0; i < kLmPiecesPerLane; ++i) {
        const int c = j + 16 * i;
        if (c < np) {
          acc[b][0] = fma4_i8(cur[i].x, s_h[c], acc[b][0]);
          acc[b][1] = fma4_i8(cur[i].y, s_h[kLmPieces + c], acc[b][1]);
          acc[b][0] = fma4_i8(cur[i].z, s_h[2 * kLmPieces + c], acc[b][0]);
          acc[b][1] = fma4_i8(cur[i].w, s_h[3 * kLmPieces + c], acc[b][1]);
        }
      }
    }
  }
#pragma unroll
  for (int b = 0; b < kLmBlocks; ++b) {
    const float s = row_sum16_f(acc[b][0] + acc[b][1]);
    const long long row = row0 + 16 * b;
    if (j == 0 && row < a.vocab_size) a.out[row] = s * a.scales[row];
  }
}

// ---------------------------------------------------------------------------
// The aligned form on the i8 matrix cores (v_mfma_i32_16x16x64_i8).  The hidden
// vector becomes fixed point: X[k] = h[k] 2^s with |X| < 2^62, s from the
// largest |h| (every value down to 2^-38 of it keeps its 24 bits), and X = sum
// over n < 8 of d[n] 256^n with signed bytes d[n].  A product of 16 rows of
// weights, as they lie in memory, with the digits as columns sums w d[n]
// exactly in int32 (2^14 K < 2^31), so the only roundings are those of the eight
// sums to fp32 and of their scaled total: a few 2^-24 of sum |w h|, whatever K
// (normal data at K = 2560: 4.4e-8 of the result; fp32 sums 1.7e-7).
//
// Bound by the weights' stream.  The earlier kernel spent a conversion and an
// FMA on every weight and read the hidden vector from LDS beside them: 57.3 us
// = 5.7 TB/s at 128256 x 2560; here the vector unit has little to do in the
// loop.  A wave streams whole blocks of 16 rows, 512 bytes of each per set of
// loads, two sets in turn; the first is in flight while the workgroup forms the
// digits.  One load instruction takes 256 consecutive bytes of four rows: in
// the operand's own layout it would take 64 of 16 rows, half a cache line each,
// and with the non-temporal hint the stream then ran at 4.6 TB/s (5.5 without
// it).  The pieces change places through 4 KB of LDS per wave, chunk c of row r
// at slot c ^ r so that neither side has bank conflicts.
//
// A hidden vector that does not fit the fixed point -- an infinity, a NaN, or a
// nonzero value below 2^-38 of the largest, which would lose bits that count
// in rows whose weights are zero at the larger ones -- takes fp32 sums
// (lm_head_fp32_rows).
// ---------------------------------------------------------------------------
constexpr int kLmLoads = 8;     // loads of a set: steps of 64 weights of 16 rows
constexpr int kLmMaxK = 6144;   // digits, 8 bytes per value, beside 16 KB in 64 KB of LDS
constexpr int kLmWgsPerCu = 4;
constexpr int kLmRange = 38;    // bits of fixed point below the largest value's significand
typedef int int4_t __attribute__((ext_vector_type(4)));

// Every row by fp32 products and sums as lm_head_i8_kernel forms them, 16 lanes
// per row, the whole hidden vector in LDS (s_h: K floats).
__device__ __forceinline__ void lm_head_fp32_rows(const LmHeadArgs &a, float4 *s_h) {
  const int tid = threadIdx.x, slot = tid >> 4, j = tid & 15;
  const int K = a.hidden_size, np = K / 16;
  for (int g = tid; g < K / 4; g += 256)
    s_h[(g & 3) * np + (g >> 2)] = *reinterpret_cast<const float4 *>(a.hidden + 4 * g);
  __syncthreads();
  for (long long row = (long long)blockIdx.x * 16 + slot; row < a.vocab_size; row += (long long)gridDim.x * 16) {
    const int8_t *wr = a.weight + row * K;
    float acc[2] = {0.f, 0.f};
    constexpr int kAhead = 10;  // loads in flight: a row of 2560 weights
    for (int c0 = j; c0 < np; c0 += 16 * kAhead) {
      uint4 w[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        const int c = c0 + 16 * i;
        w[i] = c < np ? ld16_nt(wr + 16 * c) : make_uint4(0, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        const int c = c0 + 16 * i;
        if (c < np) {
          acc[0] = fma4_i8(w[i].x, s_h[c], acc[0]);
          acc[1] = fma4_i8(w[i].y, s_h[np + c], acc[1]);
          acc[0] = fma4_i8(w[i].z, s_h[2 * np + c], acc[0]);
          acc[1] = fma4_i8(w[i].w, s_h[3 * np + c], acc[1]);
        }
      }
    }
    const float v = row_sum16_f(acc[0] + acc[1]);
    if (j == 0) a.out[row] = v * a.scales[row];
  }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
void lm_head_mfma_kernel(LmHeadArgs a) {
  extern __shared__ uint4 s_digits[];  // step ks (64 values): digit n's 64 bytes at 512 ks + 64 n
  __shared__ uint4 s_swap[4][256];
  __shared__ unsigned s_max[4], s_min[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, u = lane >> 4;
  const int K = a.hidden_size, chunks = (K + 64 * kLmLoads - 1) / (64 * kLmLoads);
  const long long blocks = (a.vocab_size + 15) / 16;
  const long long stride = (long long)gridDim.x * 4;
  long long block = (long long)blockIdx.x * 4 + wave;

  // Load i: bytes 512 c + 256 (i / 4) + 16 n of row 4 (i % 4) + u.
  auto load = [&](int4_t (&x)[kLmLoads], long long b, int c) {
#pragma unroll
    for (int i = 0; i < kLmLoads; ++i) {
      const long long row = min(16 * b + 4 * (i & 3) + u, a.vocab_size - 1);
      // past the row: its last bytes (their digits are zero)
      const int k = min(512 * c + 256 * (i >> 2) + 16 * n, K - 16);
      x[i] = __builtin_nontemporal_load(reinterpret_cast<const int4_t *>(a.weight + row * K + k));
    }
  };
  int4_t wa[kLmLoads], wb[kLmLoads];
  load(wa, min(block, blocks - 1), 0);
  __builtin_amdgcn_sched_barrier(0);

  // Digits of the hidden vector, four values per thread and round.
  const int quads = chunks * kLmLoads * 16;
  // Largest magnitude and one less than the smallest nonzero one (zeros wrap).
  unsigned mx = 0, mn = ~0u;
  for (int q = tid; 4 * q < K; q += 256) {
    const uint4 h = *reinterpret_cast<const uint4 *>(a.hidden + 4 * q);
    const unsigned b[4] = {h.x & 0x7fffffffu, h.y & 0x7fffffffu, h.z & 0x7fffffffu, h.w & 0x7fffffffu};
    mx = max(mx, max(max(b[0], b[1]), max(b[2], b[3])));
    mn = min(mn, min(min(b[0] - 1, b[1] - 1), min(b[2] - 1, b[3] - 1)));
  }
  for (int m = 1; m < 64; m <<= 1) {
    mx = max(mx, (unsigned)__shfl_xor((int)mx, m));
    mn = min(mn, (unsigned)__shfl_xor((int)mn, m));
  }
  if (lane == 0) {
    s_max[wave] = mx;
    s_min[wave] = mn;
  }
  __syncthreads();
  mx = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3]));
  mn = min(min(s_min[0], s_min[1]), min(s_min[2], s_min[3]));
  const int e_max = max((int)(mx >> 23), 1);
  if (mx >= 0x7f800000u || max((int)(mn >> 23), 1) < e_max - kLmRange) {  // uniform over the grid
    lm_head_fp32_rows(a, reinterpret_cast<float4 *>(s_digits));
    return;
  }
  unsigned *digits = reinterpret_cast<unsigned *>(s_digits);
  for (int q = tid; q < quads; q += 256) {
    const uint4 h = 4 * q < K ? *reinterpret_cast<const uint4 *>(a.hidden + 4 * q) : make_uint4(0, 0, 0, 0);
    const unsigned hb[4] = {h.x, h.y, h.z, h.w};
    unsigned lo[4], hi[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ef = (int)(hb[i] >> 23 & 255u);
      const long long m = (long long)((hb[i] & 0x7fffffu) | (ef ? 0x800000u : 0u));
      const int sh = kLmRange - (e_max - max(ef, 1));  // >= 0
      long long x = m << max(sh, 0);  // zeros may lie below the range
      x = (hb[i] >> 31) ? -x : x;
      // signed bytes: add 128 to the lower seven with their carries, then take it off each
      const unsigned long long C = 0x0080808080808080ull;
      const unsigned long long d = ((unsigned long long)x + C) ^ C;
      lo[i] = (unsigned)d;
      hi[i] = (unsigned)(d >> 32);
    }
    const uint4 d0 = transpose_bytes(make_uint4(lo[0], lo[1], lo[2], lo[3]));
    const uint4 d4 = transpose_bytes(make_uint4(hi[0], hi[1], hi[2], hi[3]));
    unsigned *p = digits + (q >> 4) * 128 + (q & 15);
    p[0] = d0.x;
    p[16] = d0.y;
    p[32] = d0.z;
    p[48] = d0.w;
    p[64] = d4.x;
    p[80] = d4.y;
    p[96] = d4.z;
    p[112] = d4.w;
  }
  __syncthreads();

  // Column n and n + 8 both hold digit n % 8.
  const uint4 *op = s_digits + (n & 7) * 4 + u;
  const int ex = 8 * (n & 7) + e_max - 188;
  int4_t *swap = reinterpret_cast<int4_t *>(s_swap[wave]);
  int4_t *put = swap + 16 * u;  // row 4 j + u at 64 j + 16 u
  const int4_t *get = swap + 16 * n;
  int4_t acc = {0, 0, 0, 0};
  int c = 0;
  auto chunk = [&](int4_t (&cur)[kLmLoads], int4_t (&nxt)[kLmLoads]) {
    const int cn = c + 1 < chunks ? c + 1 : 0;
    const long long bn = cn ? block : block + stride;
    if (bn < blocks) load(nxt, bn, cn);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kLmLoads; i += 4) {
#pragma unroll
      for (int j = 0; j < 4; ++j) put[64 * j + (n ^ (4 * j + u))] = cur[i + j];
      __builtin_amdgcn_wave_barrier();  // the wave's own LDS operations keep their order
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int4_t w = get[(4 * j + u) ^ n];
        const int4_t d = __builtin_bit_cast(int4_t, op[(kLmLoads * c + i + j) * 32]);
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, d, acc, 0, 0, 0);
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (cn == 0) {
      // rows 16 block + 4 u + r: the eight digits' sums, scaled, added over the lanes
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = ldexpf((float)acc[r], ex);
        v += dppf<0xB1>(v);
        v += dppf<0x4E>(v);
        v += dppf<0x141>(v);
        const long long row = 16 * block + 4 * u + r;
        if (n == r && row < a.vocab_size) a.out[row] = v * a.scales[row];
      }
      acc = int4_t{0, 0, 0, 0};
    }
    c = cn;
    block = bn;
  };
  while (block < blocks) {
    chunk(wa, wb);
    if (block >= blocks) break;
    chunk(wb, wa);
  }
}

}  // namespace

hipError_t launch_lm_head_i8(const LmHeadArgs &a, bool vec, int n_cu, hipStream_t s) {
  if (a.vocab_size <= 0) return hipSuccess;
  if (vec && a.hidden_size >= 16 && a.hidden_size <= kLmMaxK) {
    const long long blocks = (a.vocab_size + 15) / 16;
    const int chunks = (a.hidden_size + 64 * kLmLoads - 1) / (64 * kLmLoads);
    const long long wgs = std::min<long long>((blocks + 3) / 4, (long long)kLmWgsPerCu * n_cu);
    lm_head_mfma_kernel<<<dim3((unsigned)wgs), dim3(256), (size_t)chunks * kLmLoads * 512, s>>>(a);
    return hipGetLastError();
  }
  const long long rows_per_wg = 16 * kLmBlocks;
  const dim3 grid((unsigned)((a.vocab_size + rows_per_wg - 1) / rows_per_wg));
  if (vec)
    lm_head_i8_kernel<true><<<grid, dim3(256), 0, s>>>(a);
  else
    lm_head_i8_kernel<false><<<grid, dim3(256), 0, s>>>(a);
  return hipGetLastError();
}

}  // namespace bnr
