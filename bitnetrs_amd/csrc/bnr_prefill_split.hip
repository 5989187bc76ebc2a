// bnr_prefill_split.hip -- gfx950 causal flash prefill with every fp32
// operand split into two fp16 halves (head_dim 128).
//
// x * 2^e = h + l, h = fp16(x * 2^e), l = fp16(x * 2^e - h): two 11-bit
// significands, so h + l holds x to 2^-23 of its value, and a product of two
// such pairs is h h' + h l' + l h' to 2^-22 (l l' is left out): three fp16
// matrix products with fp32 accumulation take the place of one fp32 product
// at 3/16 of its matrix-core time.  The sums are shorter as well: a 32 x 32 x
// 16 product adds 16 terms before it rounds, the fp32 one 2.  Measured
// against 64 bits the outputs are closer than the fp32 kernels' (relative
// 2-norm, fp32 products -> pairs: 1024 tokens 3.7 -> 2.0e-7, 2048 3.8 -> 2.4e-7,
// 333 after 1207 5.3 -> 2.8e-7).
//
// The scales 2^e are exact powers of two that put the largest magnitude of a
// 32-key tile of K, of V, or of a query row in [2^14, 2^15), and l is stored
// times 2^12 (kLowScale): values down to 2^-28 of that largest one keep their
// bits.  A K or V tile with a nonzero value below that, an infinity, a NaN, or
// (V) rows far apart is marked and takes fp32 products, which the attention
// kernel has beside the others; so does a query row, against the K tiles where
// what it lost counts.  One K or V tile in 20000 of normal data is marked.  With
// one K and one V dim 2^30 above the others in every row all are: 2048 tokens
// then take 311 us (K alone 202, V alone 184; the fp32 launches 186).
//
//   prefill_split_kv_kernel  K/V tiles -> fp16 pairs in MFMA operand order
//                            (with RoPE of q/k and the append fused in)
//   prefill_split_kernel     attention over those tiles
#include "bnr_device.h"
#include "bnr_internal.h"

#include <hip/hip_runtime.h>
#include <math.h>

namespace bnr {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// Timeline stamps of a measurement build (BNR_TIMELINE; PfStamp): wave 0's
// readings of the 100 MHz counter, for the run's first piece.
#if defined(BNR_TIMELINE)
#define SP_STAMP(k)                                    \
  do {                                                 \
    __builtin_amdgcn_sched_barrier(0);                 \
    if (!stamp[k]) stamp[k] = __builtin_amdgcn_s_memrealtime(); \
    __builtin_amdgcn_sched_barrier(0);                 \
  } while (0)
#else
#define SP_STAMP(k) ((void)0)
#endif

constexpr int kHalfTile = kSplitTileFloats / 2;  // floats of a tile's K (or V) part
// The low half of a pair is stored times 2^12, where it is as large as the high
// half at most.  Then fp16's subnormals cut off at 2^-37 of a scaled value: down
// to 2^-28 of the largest h + l holds a value to 2^-23 of it.
constexpr int kLowScale = 4096;
constexpr int kElemRange = 28;
// V rows: a weight's pair cuts off at 2^-36 of the tile's largest (typically;
// 2^-26 at worst), so a row of 2^-12 of the tile's largest value or less -- a
// zero row too -- under the largest weight could leave an output to weights
// that have lost bits.
constexpr int kVRowRange = 12;

// x0 .. x7 (already scaled) -> h and l times LOW: two conversions of a pair
// (v_cvt_pk) and one subtraction that reads h as it is (v_fma_mix) per value.
template <int LOW>
__device__ __forceinline__ void split8(const float (&x)[8], half8 &h, half8 &l) {
  typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
  typedef float float2_t __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const float2_t v = {x[i], x[i + 1]};
    const half2_t a = __builtin_convertvector(v, half2_t);
    float2_t r;
    const unsigned ab = __builtin_bit_cast(unsigned, a);
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r.x) : "v"(ab), "v"(x[i]));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r.y) : "v"(ab), "v"(x[i + 1]));
    if (LOW != 1) r *= (float)LOW;
    const half2_t b = __builtin_convertvector(r, half2_t);
    h[i] = a.x;
    h[i + 1] = a.y;
    l[i] = b.x;
    l[i + 1] = b.y;
  }
}

// p[r] .. p[r + 7] times f (a power of two) -> h and l: l is what h leaves of
// the product, formed and rounded in one instruction (v_fma_mixlo, _mixhi).
// The empty asm keeps the compiler from converting the products a second time.
__device__ __forceinline__ void split8f(const float (&p)[16], int r, float f, half8 &h, half8 &l) {
  typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
  typedef float float2_t __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const float x = p[r + i], y = p[r + i + 1];
    unsigned w = __builtin_bit_cast(unsigned, __builtin_convertvector((float2_t{x * f, y * f}), half2_t));
    asm("" : "+v"(w));
    const half2_t a = __builtin_bit_cast(half2_t, w);
    h[i] = a.x;
    h[i + 1] = a.y;
    l[i] = (_Float16)fmaf(x, f, -(float)a.x);
    l[i + 1] = (_Float16)fmaf(y, f, -(float)a.y);
  }
}

__device__ __forceinline__ unsigned abs_bits(float x) {
  return __builtin_bit_cast(unsigned, x) & 0x7fffffffu;
}
// The largest magnitude and one less than the smallest nonzero one (zeros wrap
// to ~0) of x and what came before.
__device__ __forceinline__ void mag4(float4 x, unsigned &mx, unsigned &elem_min) {
  const unsigned b[4] = {abs_bits(x.x), abs_bits(x.y), abs_bits(x.z), abs_bits(x.w)};
  mx = max(mx, max(max(b[0], b[1]), max(b[2], b[3])));
  elem_min = min(elem_min, min(min(b[0] - 1, b[1] - 1), min(b[2] - 1, b[3] - 1)));
}
__device__ __forceinline__ unsigned least4(float4 x) {
  return min(min(abs_bits(x.x), abs_bits(x.y)), min(abs_bits(x.z), abs_bits(x.w)));
}
__device__ __forceinline__ float exp2i(int e) {  // 2^e, -126 <= e <= 127
  return __builtin_bit_cast(float, (unsigned)(e + 127) << 23);
}
// The scale exponent that puts a magnitude of these bits in [2^14, 2^15);
// 0 and the smallest normals stop at 2^126.
__device__ __forceinline__ int scale_exp(unsigned bits) {
  return min(141 - (int)(bits >> 23), 126);
}

template <int CTRL>
__device__ __forceinline__ unsigned dpp_u(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}
template <bool MAX>
__device__ __forceinline__ unsigned pick(unsigned a, unsigned b) {
  return MAX ? max(a, b) : min(a, b);
}
// Maximum (or minimum) over the 32 lanes of a half wave, in all of them.
template <bool MAX>
__device__ __forceinline__ unsigned half_red(unsigned v) {
  v = pick<MAX>(v, dpp_u<0xB1>(v));
  v = pick<MAX>(v, dpp_u<0x4E>(v));
  v = pick<MAX>(v, dpp_u<0x141>(v));
  v = pick<MAX>(v, dpp_u<0x140>(v));
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return pick<MAX>((unsigned)r[0], (unsigned)r[1]);
}
template <bool MAX>
__device__ __forceinline__ unsigned wave_red(unsigned v) {
  v = half_red<MAX>(v);
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return pick<MAX>((unsigned)r[0], (unsigned)r[1]);
}

// Tile word: scale exponent + 128 in bits 0..7, kSplitFp32 and kSplitZero.
constexpr int kSplitFp32 = 0x100, kSplitZero = 0x200;
// Whether values whose largest magnitude has these bits, and whose smallest
// nonzero one has elem_min + 1 (~0: none), do not fit pairs: an infinity or a
// NaN, a scale past 2^126, a value below 2^-28 of the largest.
__device__ __forceinline__ bool no_pairs(unsigned mx, unsigned elem_min) {
  const int e = (int)(mx >> 23);
  return e == 255 || e < 15 || (int)(elem_min >> 23) < max(1, e - kElemRange);
}
// A V tile's word; row_min is its smallest row maximum.  A marked tile's
// exponent says how large its values are: O takes it for its own.
__device__ __forceinline__ int v_word(unsigned mx, unsigned row_min, unsigned elem_min) {
  if (mx == 0) return 128 | kSplitZero;
  const bool fp32 = no_pairs(mx, elem_min) || (int)(row_min >> 23) + kVRowRange < (int)(mx >> 23);
  return (scale_exp(mx) + 128) | (fp32 ? kSplitFp32 : 0);
}
// A K tile's.  Values past 2^54 are marked: the scales of K and q and their
// product then stay inside fp32 (a score may be small all the same, where K
// or q has zeros).  kSplitWide: a zero, or a value below 2^-24 of the largest
// (least: the smallest magnitude).  In a tile without, a key's values are within
// 2^24 of one another, and what a q pair cuts off, 2^-51 of the row's largest
// value, is 2^-27 at most of what that largest value adds to the score.
constexpr int kQkTop = 127 + 54, kWideRange = 24;
constexpr int kSplitWide = 0x400, kSplitAny = 0x800;  // kSplitAny: in every K word
__device__ __forceinline__ int k_word(unsigned mx, unsigned elem_min, unsigned least) {
  if (mx == 0) return 128 | kSplitZero | kSplitAny;
  const int e = (int)(mx >> 23);
  const bool fp32 = no_pairs(mx, elem_min) || e > kQkTop;
  const bool wide = (int)(least >> 23) < max(1, e - kWideRange);
  return (scale_exp(mx) + 128) | (fp32 ? kSplitFp32 : 0) | (wide ? kSplitWide : 0) | kSplitAny;
}
// The scale exponent that a V tile asks of O.  A marked tile's values are not
// scaled: the limits keep its weights, 2^(15 + exponent) at most, and their
// products with the values inside fp32.
__device__ __forceinline__ int v_exp(int word) {
  const int e = (word & 255) - 128;
  return (word & kSplitFp32) ? min(max(e, -50), 100) : e;
}

// One 32-key tile of one kv head per workgroup (blockIdx.x < n_kv * n_tiles,
// kv head fastest); with ROPE the workgroups after those rotate q, 512 quads
// each.  Tile layout: MFMA operands of v_mfma_f32_32x32x16_f16, 1 KB each,
// lane l's 16 bytes at 16 l, so that the attention kernel copies and reads
// them as they are.
//   K, step s (16 dims), part p (h, l): at 2 s + p; lane l holds key l % 32,
//     dims 16 s + 8 (l / 32) .. + 7.
//   V, step t (16 keys), dim block db, part p: at 16 + 8 t + 2 db + p; lane l
//     holds dim 4 (l % 32) + db of keys 16 t + 4 (l / 32) + {0..3} and 8 more:
//     the keys that lane's registers 8 t .. 8 t + 7 of S^T hold.
// A marked K part holds the fp32 values: dims + 0 .. 3 in place of h, + 4 .. 7 in
// place of l.  A marked V part holds zeros.
// Waves 0, 1 take V (step t = wave), waves 2, 3 take K (steps 2w', 2w'+1 and
// the four dims blocks 64 further, so that a rotation pair sits in one lane).
// Rows past the last cached one are zero.
//
// Bound by memory: every cached row is read once and its tile written once
// (5 KB + 5 KB a row at 5 kv heads).
template <bool ROPE>
__global__ __launch_bounds__(256) void prefill_split_kv_kernel(PrefillSplitArgs p) {
  const RopeAppendArgs &a = p.rope;
  const int tid = threadIdx.x;
  const int kv_wgs = a.n_kv * p.n_tiles;
  if (ROPE && (int)blockIdx.x >= kv_wgs) {
    const long long quads = (long long)a.n_tokens * a.n_heads * 16;
    const long long i0 = ((long long)blockIdx.x - kv_wgs) * 512 + tid;
    const int qpt = a.n_heads * 16;
    float4 lo[2], hi[2], c[2], s[2];
    float *x[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const long long idx = min(i0 + 256 * u, quads - 1);
      const int tok = (int)(idx / qpt), r = (int)(idx - (long long)tok * qpt);
      const int i = 4 * (r & 15);
      x[u] = a.q + ((long long)tok * a.n_heads + (r >> 4)) * kHeadDim + i;
      const long long pos = (long long)(a.start_pos + tok) * 64 + i;
      lo[u] = ld4_nt(x[u]);
      hi[u] = ld4_nt(x[u] + 64);
      c[u] = ld4(a.cos_tab + pos);
      s[u] = ld4(a.sin_tab + pos);
    }
    __builtin_amdgcn_sched_barrier(0);  // all loads before the first store
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (i0 + 256 * u >= quads) break;
      float4 rl, rh;
      rot4(lo[u], hi[u], c[u], s[u], rl, rh);
      st4(x[u], rl);
      st4(x[u] + 64, rh);
    }
    return;
  }
  __shared__ unsigned s_vmax[2], s_vmin[2], s_velem[2], s_kmax[2], s_kelem[2], s_kleast[2];
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int hl = lane >> 5, col = lane & 31;
  const int h = (int)blockIdx.x % a.n_kv, kt = (int)blockIdx.x / a.n_kv;
  const int rows = a.start_pos + a.n_tokens;
  float *tile = p.tiles + ((long long)h * p.tiles_per_head + kt) * kSplitTileFloats;
  int2 *info = p.info + (long long)h * p.tiles_per_head + kt;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  if (wave < 2) {
    const int t = wave;
    float4 x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = 32 * kt + 16 * t + 8 * (i >> 2) + 4 * hl + (i & 3);
      const bool fresh = ROPE && row >= a.start_pos;
      const float *src = fresh ? a.v + ((long long)(row - a.start_pos) * a.n_kv + h) * kHeadDim
                               : a.v_cache + h * a.kv_stride + (long long)row * kHeadDim;
      x[i] = row < rows ? ld4(src + 4 * col) : zero;
    }
    unsigned mx = 0, mn = ~0u, en = ~0u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = 32 * kt + 16 * t + 8 * (i >> 2) + 4 * hl + (i & 3);
      unsigned r = 0;
      mag4(x[i], r, en);
      r = half_red<true>(r);
      mx = max(mx, r);
      mn = min(mn, row < rows ? r : ~0u);
    }
    mx = wave_red<true>(mx);
    mn = wave_red<false>(mn);
    en = wave_red<false>(en);
    if (lane == 0) {
      s_vmax[t] = mx;
      s_vmin[t] = mn;
      s_velem[t] = en;
    }
    if (ROPE) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int row = 32 * kt + 16 * t + 8 * (i >> 2) + 4 * hl + (i & 3);
        if (row >= a.start_pos && row < rows)
          st4(a.v_cache + h * a.kv_stride + (long long)row * kHeadDim + 4 * col, x[i]);
      }
    }
    __syncthreads();
    const int word = v_word(max(s_vmax[0], s_vmax[1]), min(s_vmin[0], s_vmin[1]), min(s_velem[0], s_velem[1]));
    const bool marked = (word & kSplitFp32) != 0;
    const float sc = exp2i((word & 255) - 128);
    float *dst = tile + kHalfTile + t * 8 * 256 + 4 * lane;
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      float y[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        y[i] = marked ? 0.f : (db == 0 ? x[i].x : db == 1 ? x[i].y : db == 2 ? x[i].z : x[i].w) * sc;
      half8 hv, lv;
      split8<kLowScale>(y, hv, lv);
      *reinterpret_cast<half8 *>(dst + 512 * db) = hv;
      *reinterpret_cast<half8 *>(dst + 512 * db + 256) = lv;
    }
    if (tid == 0) info->y = word;
    return;
  }
  const int w = wave - 2;
  const int row = 32 * kt + col;
  const bool valid = row < rows, fresh = ROPE && row >= a.start_pos;
  float *src = fresh ? a.k + ((long long)(row - a.start_pos) * a.n_kv + h) * kHeadDim
                     : a.k_cache + h * a.kv_stride + (long long)row * kHeadDim;
  float4 lo[2][2], hi[2][2];  // dims d .. d+7 and 64 + d .. of step s = 2 w + u, d = 16 s + 8 hl
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int d = 16 * (2 * w + u) + 8 * hl;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      lo[u][e] = valid ? ld4(src + d + 4 * e) : zero;
      hi[u][e] = valid ? ld4(src + 64 + d + 4 * e) : zero;
    }
  }
  if (ROPE && valid && fresh) {
    float4 c[2][2], s[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const long long o = (long long)row * 64 + 16 * (2 * w + u) + 8 * hl + 4 * e;
        c[u][e] = ld4(a.cos_tab + o);
        s[u][e] = ld4(a.sin_tab + o);
      }
    float *dst = a.k_cache + h * a.kv_stride + (long long)row * kHeadDim;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int d = 16 * (2 * w + u) + 8 * hl;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        rot4(lo[u][e], hi[u][e], c[u][e], s[u][e], lo[u][e], hi[u][e]);
        st4(src + d + 4 * e, lo[u][e]);
        st4(src + 64 + d + 4 * e, hi[u][e]);
        st4(dst + d + 4 * e, lo[u][e]);
        st4(dst + 64 + d + 4 * e, hi[u][e]);
      }
    }
  }
  unsigned mx = 0, en = ~0u, least = ~0u;
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      mag4(lo[u][e], mx, en);
      mag4(hi[u][e], mx, en);
      least = min(least, min(least4(lo[u][e]), least4(hi[u][e])));
    }
  mx = wave_red<true>(mx);
  en = wave_red<false>(en);
  least = wave_red<false>(valid ? least : ~0u);
  if (lane == 0) {
    s_kmax[w] = mx;
    s_kelem[w] = en;
    s_kleast[w] = least;
  }
  __syncthreads();
  const int word = k_word(max(s_kmax[0], s_kmax[1]), min(s_kelem[0], s_kelem[1]), min(s_kleast[0], s_kleast[1]));
  const bool marked = (word & kSplitFp32) != 0;
  const float sc = exp2i((word & 255) - 128);
  if (tid == 128) info->x = word;
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const float4 e0 = half ? hi[u][0] : lo[u][0], e1 = half ? hi[u][1] : lo[u][1];
      float *dst = tile + (2 * w + u + 4 * half) * 512 + 4 * lane;
      if (marked) {
        st4(dst, e0);
        st4(dst + 256, e1);
        continue;
      }
      const float y[8] = {e0.x * sc, e0.y * sc, e0.z * sc, e0.w * sc,
                          e1.x * sc, e1.y * sc, e1.z * sc, e1.w * sc};
      half8 hv, lv;
      split8<kLowScale>(y, hv, lv);
      *reinterpret_cast<half8 *>(dst) = hv;
      *reinterpret_cast<half8 *>(dst + 256) = lv;
    }
}

// ---------------------------------------------------------------------------
// Attention.  Workgroup = W waves: one kv head's G query heads x W / G blocks
// of 32 queries, over one run of key tiles (PrefillRunsArgs).  S^T = K Q^T and
// O^T = V^T P^T: S^T's accumulator layout is P^T's operand layout (the order of
// the keys in a V operand is chosen for that), so P stays in registers.
// Register r of a 32 x 32 accumulator holds row 8 (r / 4) + 4 (lane / 32) +
// r % 4; row i of O^T's dim block db is head dim 4 i + db.
//
// Two workgroups share a CU (218 registers, 64 KB of LDS): one's softmax,
// starts and ends run under the other's products.  A workgroup's waves share a
// tile's operands; the next tile's go to the other LDS buffer while this one
// is multiplied, one barrier per tile.  One round: every CU gets two runs of
// about equal cost, and no item list is decoded.
//
// A tile of 32 queries x 4 heads takes 1536 cycles of a SIMD's matrix core (0.7
// us at the 2.2 GHz that the counters read) and 1.15 us per CU as measured with
// two workgroups (each 2.3): the younger one's products wait for the older's,
// and what is left of it then runs alone.  At 2048 tokens the matrix cores are
// busy 38 % of the cycles, at 1024 (5 tiles a run) 18 %: starts 5 us, a piece's
// end 4 to 6.  No LDS bank conflicts.  With RoPE and append (20/5 heads,
// MI355X): 1024 tokens 60 -> 40 us, 2048 199 -> 89, 333 after 1207 53 -> 42
// against the fp32 products.  One 8-wave workgroup of 64 queries per CU (half
// the operand traffic, one barrier per 64 keys) took 47, 93 and 48 us (before
// low halves were scaled).
//
// p = exp2(S c - m): c undoes the scales of K and q and applies log2(e) /
// sqrt(d); m is a lazily moved whole number above or near the query's largest
// S c.  (The power of two below is a factor, not part of the exponential's
// argument: that would be rounded near 11 where it is rounded near 0.)
//
// O holds sum(p V) 2^g, g a whole number per query, and the operand is p
// 2^(g - ev) for a V tile of scale exponent ev.  g stays while the tile's
// largest operand lies between 2^1 (what fp16's subnormals cut off is then 2^-26
// of it) and 2^15, else it is moved to 2^8, and O with it (scores of 4 times the
// spread of normal data move it in most tiles: 2048 tokens 97 us for 91).
// Weights and V so far below what O holds that it would overflow (kScaleSpan), and weights
// near fp32's end, take fp32 products for that tile.  The output is (O / l)
// 2^-g in that order: O alone, with the sum of the weights and a power of two in
// it, would pass fp32's largest value where the output does not.
// ---------------------------------------------------------------------------
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wpass-failed"

constexpr float kLazy = 4.0f, kNoRef = -3.4028234e38f, kLeastP = -126.0f, kPHalf = 7.0f;
constexpr int kPMid = 8;            // operands: the tile's largest is 2^8, in 2^(8 -+ 7)
constexpr int kScaleSpan = 72;      // sum(p V) 2^g <= 2^23 times the keys, and 2^72 more once g follows V down
constexpr int kNoScale = 1 << 28;   // O holds nothing yet
constexpr int kMaxFactor = 112;     // of 2^(g - ev), a float
constexpr int kMaxShift = 4096;     // more than any O keeps

// Maximum and sum over lanes l, l ^ 32.
__device__ __forceinline__ float max_half_swap(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
}

__device__ __forceinline__ float sum_half_swap(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}

// The lane, formed where it is used and not kept.
__device__ __forceinline__ int lane_here() {
  int lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(lane));
  return lane;
}

__device__ __forceinline__ half8 ld_op(const float *lds, int op) {
  return *reinterpret_cast<const half8 *>(lds + op * 256 + 4 * (threadIdx.x & 63));
}

// Value i of a pair operand, or of the fp32 values that take its place (x, y:
// the two 16-byte words of the lane).
__device__ __forceinline__ float op_value(half8 x, half8 y, int i, bool fp32, float unscale) {
  const float pair = fmaf((float)y[i], 1.0f / kLowScale, (float)x[i]) * unscale;
  const floatx4 v = __builtin_bit_cast(floatx4, i < 4 ? x : y);
  return fp32 ? v[i & 3] : pair;
}

// S^T of a tile with fp32 products (v_mfma_f32_32x32x2_f32): step 8 s + i takes
// dim 16 s + 8 (lane / 32) + i.  K as pairs (unscale_k undoes their scale) or
// fp32 values; q as pairs or, where they have lost bits, read from memory (qp:
// the lane's values of step 0, or null).  The caller's scale is log2(e) /
// sqrt(d) alone.
__device__ __forceinline__ floatx16 sp_fp32_s(const float *dk, bool fp32_k, float unscale_k, const half8 (&qh)[8],
                                              const half8 (&ql)[8], float unscale_q, bool q_lost, const float *qp) {
  floatx16 S = floatx16{};
  // hidden from the compiler, which would otherwise form q's 64 values ahead of
  // the tile loop and keep them in registers
  asm volatile("" : "+v"(unscale_q));
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    __builtin_amdgcn_sched_barrier(0);
    const half8 x = ld_op(dk, 2 * s), y = ld_op(dk, 2 * s + 1);
    half8 u = qh[s], v = ql[s];
    if (q_lost) {
      u = *reinterpret_cast<const half8 *>(qp + 16 * s);
      v = *reinterpret_cast<const half8 *>(qp + 16 * s + 4);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      S = __builtin_amdgcn_mfma_f32_32x32x2f32(op_value(x, y, i, fp32_k, unscale_k),
                                               op_value(u, v, i, q_lost, unscale_q), S, 0, 0, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
  return S;
}

// O^T += V^T P^T with fp32 products, V read from the cache: step s takes key
// 8 (s / 4) + 4 (lane / 32) + s % 4.  Rows past the last repeat it (masked).
__device__ __forceinline__ void sp_fp32_pv(const PrefillRunsArgs &a, int h, int kt,
                                           const float (&p)[16], floatx16 (&O)[4]) {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));  // addresses are formed here, not ahead of the tile loop
  const int hl = lane >> 5, col = lane & 31;
  const float *vp = a.v_cache + h * a.kv_stride + (long long)kt * 32 * kHeadDim;  // uniform
  const int last = a.start_pos + a.n_tokens - 1 - kt * 32;
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    if ((s & 3) == 0) __builtin_amdgcn_sched_barrier(0);  // the loads of four steps at a time
    const int row = min(8 * (s >> 2) + 4 * hl + (s & 3), last);
    const float4 vv = ld4(vp + (unsigned)(row * kHeadDim + 4 * col));
    O[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.x, p[s], O[0], 0, 0, 0);
    O[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.y, p[s], O[1], 0, 0, 0);
    O[2] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.z, p[s], O[2], 0, 0, 0);
    O[3] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv.w, p[s], O[3], 0, 0, 0);
  }
}

// 4 KB per wave from memory straight into LDS (16 bytes per lane and
// instruction): bytes 1024 j + 16 i of src + 16 * lane i go to `lds`, j < 4;
// src and lds are uniform.  Written as assembly so that the compiler, which
// would take every later LDS read of the array for a read of the bytes in
// flight, does not wait for them there: prefill_split_kernel waits for its
// copies itself, before the barrier that opens the buffer.  The copies have no
// register results, and a wait the compiler places for its own loads only
// becomes stricter by them.  m0, which the
// compiler does not let an asm declare as changed, is put back.
__device__ __forceinline__ void dma4k(const char *src, unsigned lane16, unsigned lds) {
  unsigned m0;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %2, %3\n\t"
      "global_load_lds_dwordx4 %2, %3 offset:1024\n\t"
      "global_load_lds_dwordx4 %2, %3 offset:2048\n\t"
      "global_load_lds_dwordx4 %2, %3 offset:3072\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(m0)
      : "s"(lds), "v"(lane16), "s"(src)
      : "memory");
}

template <int G>
__global__ __launch_bounds__(64 * split_waves(G)) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_split_kernel(PrefillRunsArgs a) {
  constexpr int W = split_waves(G), UQ = split_unit(G);
  __shared__ __attribute__((aligned(16))) float s_tile[2][kSplitTileFloats];
  __shared__ int s_last;
#if defined(BNR_TIMELINE)
  unsigned long long stamp[kTimelineStamps] = {};
#endif
  SP_STAMP(kPfEntry);
  // Workgroup i runs on XCD i % 8 and, of two that share a CU, the first half
  // of the grid holds the one with issue priority.  Runs are numbered XCD by
  // XCD, two to a CU, a kv head's consecutive: an XCD's L2 holds the tiles of
  // few heads, and even runs have the priority.
  const int per_xcd = a.grid >> 3, j8 = (int)blockIdx.x >> 3;
  const int half = W == 4 ? per_xcd >> 1 : per_xcd;
  const int id = ((int)blockIdx.x & 7) * per_xcd + (W == 4 ? (j8 % half) * 2 + j8 / half : j8);
  const int h = id / a.n_runs, run = id - h * a.n_runs;
  if (h >= a.n_kv) return;
  const unsigned w0 = a.run[run][0], w1 = a.run[run][1], w2 = a.run[run][2];
  const int tid = threadIdx.x, lane = tid & 63, hl = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int head = h * G + wave % G;
  const int rows = a.start_pos + a.n_tokens;
  const float *tiles = a.tiles + (long long)h * a.tiles_per_head * kSplitTileFloats;
  const int2 *infos = a.info + (long long)h * a.tiles_per_head;
  auto unit_tiles = [&](int u) { return (min(a.start_pos + (u + 1) * UQ, rows) + 31) >> 5; };

  // The next tile to fetch (tile pk of unit pu).
  int left = (int)(w1 & 0xffffu);
  int u = (int)(w0 & 0xffffu), kt = (int)(w0 >> 16), nk = unit_tiles(u);
  int pu = u, pk = kt, pn = nk;
  // Tile words come as vector loads (a scalar load in flight would hold every
  // wait for LDS reads to lgkmcnt(0)); the offset is zero.
  int vzero;
  asm volatile("v_mov_b32 %0, 0" : "=v"(vzero));
  int2 word;
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) void *)&s_tile[0][0];
  // Copies of the tile's operands, 32 / W KB per wave, straight into LDS.
  auto fetch = [&](int buf) {
    word = infos[pk + vzero];
    constexpr int NF = kSplitTileFloats / W;
    const char *src = (const char *)(tiles + (long long)pk * kSplitTileFloats + wave * NF);
    const unsigned dst = lds0 + (unsigned)(buf * kSplitTileFloats + wave * NF) * 4u;
#pragma unroll
    for (int j = 0; j < 8 / W; ++j) dma4k(src + 4096 * j, lane * 16u, dst + 4096 * j);
    if (++pk == pn) {
      pk = 0;
      pn = unit_tiles(++pu);
    }
  };

  half8 qh[8], ql[8];
  floatx16 O[4];
  float unscale_q, m, l;
  int g, g_cap, qrow, q0;
  int q_words;  // bits of the K words whose tiles take fp32 scores (uniform): kSplitFp32, and more where
                // a query of the wave's has lost bits as a pair

  // Four operands read ahead of the products that use them (two sets of
  // registers in turn): a wave's LDS reads run under its own products.
  auto rd = [&](half8 (&x)[4], const float *lds, int op) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = ld_op(lds, op + i);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mm = [](half8 x, half8 y, floatx16 &acc) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, y, acc, 0, 0, 0);
  };
  // Steps s, s + 1; L: products with a low half, times its scale.
  auto mm_s = [&](floatx16 &S, floatx16 &L, const half8 (&x)[4], int s) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      mm(x[2 * i + 1], qh[s + i], L);
      mm(x[2 * i], ql[s + i], L);
      mm(x[2 * i], qh[s + i], S);
    }
  };
  // Dim blocks db, db + 1; pq: ph over the scale of V's low half.
  auto mm_o = [&](const half8 (&x)[4], int db, half8 ph, half8 pl, half8 pq) {
    mm(x[1], pq, O[db]);
    mm(x[3], pq, O[db + 1]);
    mm(x[0], pl, O[db]);
    mm(x[2], pl, O[db + 1]);
    mm(x[0], ph, O[db]);
    mm(x[2], ph, O[db + 1]);
  };

  // The products of one tile (operands at dk, words wk and wv).
  auto step = [&](const float *dk, int kt, int wk, int wv) {
    const float *dv = dk + kHalfTile;
    floatx16 S = floatx16{}, L = floatx16{};
    half8 A[4], B[4];
    rd(A, dk, 0);
    rd(B, dk, 4);
    mm_s(S, L, A, 0);
    rd(A, dk, 8);
    mm_s(S, L, B, 2);
    rd(B, dk, 12);
    mm_s(S, L, A, 4);
    rd(A, dv, 0);
    mm_s(S, L, B, 6);
#pragma unroll
    for (int r = 0; r < 16; ++r) S[r] = fmaf(L[r], 1.0f / kLowScale, S[r]);
    const float unscale_k = exp2i(128 - (wk & 255));
    float c = fmaxf(unscale_q * (a.scale_log2 * unscale_k), 1e-37f);  // > 0: a masked -inf stays -inf
    if (__builtin_expect((wk & q_words) != 0, 0)) {
      const int lane = lane_here(), row = min(q0 + (lane & 31), a.n_tokens - 1);
      const float *qp = a.q + ((long long)row * a.n_heads + head) * kHeadDim + 8 * (lane >> 5);
      S = sp_fp32_s(dk, (wk & kSplitFp32) != 0, unscale_k, qh, ql, unscale_q, q_words != kSplitFp32, qp);
      c = a.scale_log2;
    }
    if (kt * 32 + 31 > a.start_pos + q0) {  // the tile reaches the causal diagonal
      const int pq = a.start_pos + qrow;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (kt * 32 + 8 * (r >> 2) + 4 * hl + (r & 3) > pq) S[r] = -INFINITY;
    }
    float mb = S[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mb = fmaxf(mb, S[r]);
    mb = max_half_swap(mb);
    // m or g moves for some query (uniform over the wave): rare.
    const int ev = v_exp(wv);
    const bool zero_v = (wv & kSplitZero) != 0;
    bool fp32_v = (wv & kSplitFp32) != 0;
    // t: log2 of the tile's largest weight; off: of its largest operand, past
    // the middle of the range.  One comparison for "t > kLazy, |off| > kPHalf, a
    // factor too large or a score of 2^22 and more".
    float t = fmaf(mb, c, -m);
    auto off = [&] { return t + (float)(g - ev - kPMid); };
    const float worst = fmaxf(fmaxf(fmaxf(fabsf(off()), t + (kPHalf - kLazy)), (float)(g - ev - kMaxFactor) + kPHalf),
                              fabsf(mb * c) * (kPHalf * 0x1p-22f));
    if (__builtin_expect(zero_v || __ballot(worst > kPHalf) != 0, 0)) {
      if (__ballot(fabsf(mb * c) > 0x1p22f && mb > -INFINITY) != 0) {
        // S c rounded once, in m and in the weights alike: what a fused product
        // keeps of it could be more than the weights' range here
#pragma unroll
        for (int r = 0; r < 16; ++r) S[r] *= c;
        mb *= c;
        c = 1.0f;
        t = mb - m;
      }
      if (t > kLazy) {
        const float mn = ceilf(mb * c);
        const int up = (int)fminf(mn - m, (float)kMaxShift);
        l *= fast_exp2(m - mn);
        g += up;
        g_cap += up;
        m = mn;
        t = fmaf(mb, c, -m);
      }
      if (!zero_v) {
        // queries that see no key of the tile, or none with a weight, stay
        const bool has = t >= kLeastP;
        const int want = kPMid - (int)ceilf(fmaxf(t, kLeastP));
        if (has) g_cap = min(g_cap, want + (wv & 255) - 128 + kScaleSpan);
        const bool move = has && (fabsf(off()) > kPHalf || g - ev > kMaxFactor);
        const int gn = move ? min(min(want, kMaxFactor) + ev, g_cap) : g;
        if (__ballot(gn != g) != 0) {
#pragma unroll
          for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) O[db][r] = ldexpf(O[db][r], gn - g);
          g = gn;
        }
        fp32_v = fp32_v || __ballot(has && off() < -kPHalf) != 0;
      }
    }
    float p[16], ls = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      p[r] = fast_exp2(fmaf(S[r], c, -m));
      ls += p[r];
    }
    l += ls;
    if (zero_v) return;
    // fp32 products come after these, whose factor is then 0 (a marked part's
    // operands are zeros; with a branch around them the compiler keeps O twice)
    const float f = fp32_v ? 0.f : ldexpf(1.0f, min(g - ev, kMaxFactor));
    const _Float16 down = (_Float16)(1.0f / kLowScale);
    half8 ph, pl, pq;
    split8f(p, 0, f, ph, pl);
    pq = ph * down;
    rd(B, dv, 4);
    mm_o(A, 0, ph, pl, pq);
    rd(A, dv, 8);
    mm_o(B, 2, ph, pl, pq);
    rd(B, dv, 12);
    split8f(p, 8, f, ph, pl);
    pq = ph * down;
    mm_o(A, 0, ph, pl, pq);
    mm_o(B, 2, ph, pl, pq);
    if (__builtin_expect(fp32_v, 0)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) p[r] = ldexpf(p[r], g);
      sp_fp32_pv(a, h, kt, p, O);
    }
  };

  // Queries of the unit's block: lane's dims 16 s + 8 hl + i of query q0 + col
  // (rows past the end repeat the last and are not stored), as fp16 pairs.
  auto begin = [&] {
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));
    const int hl = lane >> 5, col = lane & 31;
    q0 = u * UQ + 32 * (wave / G);
    qrow = min(q0 + col, a.n_tokens - 1);
    const float *qp = a.q + ((long long)qrow * a.n_heads + head) * kHeadDim;
    float4 x[16];
    unsigned mx = 0, en = ~0u;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      x[2 * s] = ld4(qp + 16 * s + 8 * hl);
      x[2 * s + 1] = ld4(qp + 16 * s + 8 * hl + 4);
    }
#pragma unroll
    for (int s = 0; s < 16; ++s) mag4(x[s], mx, en);
    const auto r = __builtin_amdgcn_permlane32_swap(mx, mx, false, false);
    mx = max((unsigned)r[0], (unsigned)r[1]);
    const auto re = __builtin_amdgcn_permlane32_swap(en, en, false, false);
    en = min((unsigned)re[0], (unsigned)re[1]);
    // Values below 2^-28 of the row's largest have lost bits, which counts with
    // some K tiles; an infinity, a NaN or a value past 2^54 with all.  (A small
    // row has nothing to lose: its scores with K up to 2^54 are.)
    const int e_mx = (int)(mx >> 23);
    q_words = kSplitFp32;
    if (__ballot((int)(en >> 23) < max(1, e_mx - kElemRange)) != 0) q_words |= kSplitWide;
    if (__ballot(e_mx > kQkTop) != 0) q_words |= kSplitAny;
    const int e = scale_exp(mx);
    const float sc = exp2i(e);
    unscale_q = ldexpf(1.0f, -e);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const float4 v = x[2 * s], w = x[2 * s + 1];
      const float y[8] = {v.x * sc, v.y * sc, v.z * sc, v.w * sc, w.x * sc, w.y * sc, w.z * sc, w.w * sc};
      split8<kLowScale>(y, qh[s], ql[s]);
    }
#pragma unroll
    for (int db = 0; db < 4; ++db) O[db] = floatx16{};
    // m starts finite: in a piece that is not the first, a query may see no
    // key at all (p = 0 for it throughout, and no -inf - -inf).
    m = kNoRef;
    l = 0.f;
    g = 0;
    g_cap = kNoScale;
  };

  // End of a piece: one of several stores its state and takes a ticket; the
  // unit's last to finish adds the others to its registers and, like a whole
  // unit, writes the output.  State of a wave: float4 k (components 4k ..
  // 4k+3 of O, 16 db + r) of lane l at float (k * 64 + l) * 4, then (m, l, g)
  // at 64 * 64 + 4 l.
  auto finish = [&](int nch, int ch, int base) {
    // lane values hidden from the compiler, which would otherwise form the
    // addresses below ahead of the tile loop and keep them in registers
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));
    const int hl = lane >> 5, col = lane & 31;
    auto state = [&](int c) {
      return agent_buf(a.ws + (((long long)h * a.n_slots + base + c) * W + wave) * kSplitStateFloats);
    };
    if (g_cap >= kNoScale / 2) g = kMaxShift;  // an empty O asks for no scale in a merge
    if (nch > 1) {
      const __amdgpu_buffer_rsrc_t mine = state(ch);
#pragma unroll
      for (int k = 0; k < 16; ++k)
        st4_agent(mine, lane * 16, 1024 * k,
                  make_float4(O[k >> 2][4 * (k & 3)], O[k >> 2][4 * (k & 3) + 1],
                              O[k >> 2][4 * (k & 3) + 2], O[k >> 2][4 * (k & 3) + 3]));
      st4_agent(mine, 64 * 64 * 4 + 16 * lane, make_float4(m, l, __builtin_bit_cast(float, g), 0.f));
      __builtin_amdgcn_s_waitcnt(0);  // this wave's state has been stored
      __syncthreads();
      unsigned *ctr = a.counters + ((long long)h * a.n_units + u) * kCounterStride;
      if (tid == 0) {
        const unsigned ticket =
            __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = ticket == (unsigned)(nch - 1);
      }
      __syncthreads();
      const bool last = s_last;
      SP_STAMP(kPfTicket);
      if (!last) return;  // s_last is written again only past the next tile's barrier
      if (tid == 0) __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      struct State {
        float4 o[16], mlg;
      };
      auto load = [&](State &x, int c) {
        const __amdgpu_buffer_rsrc_t src = state(c);
#pragma unroll
        for (int k = 0; k < 16; ++k) x.o[k] = ld4_agent(src, lane * 16, 1024 * k);
        x.mlg = ld4_agent(src, 64 * 64 * 4 + 16 * lane);
      };
      auto add = [&](const State &x) {
        // whole-number exponents: every factor is a power of two, 1 at most
        const float mn = fmaxf(m, x.mlg.x);
        const int da = (int)fminf(mn - m, (float)kMaxShift), db = (int)fminf(mn - x.mlg.x, (float)kMaxShift);
        const int ga = g + da, gb = __builtin_bit_cast(int, x.mlg.z) + db;
        l = ldexpf(l, -da) + ldexpf(x.mlg.y, -db);
        m = mn;
        g = min(ga, gb);
        const float wa = ldexpf(1.0f, g - ga), wb = ldexpf(1.0f, g - gb);
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          floatx16 &o = O[k >> 2];
          const int r = 4 * (k & 3);
          o[r] = o[r] * wa + x.o[k].x * wb;
          o[r + 1] = o[r + 1] * wa + x.o[k].y * wb;
          o[r + 2] = o[r + 2] * wa + x.o[k].z * wb;
          o[r + 3] = o[r + 3] * wa + x.o[k].w * wb;
        }
      };
      for (int c = 0; c < nch; ++c) {
        if (c == ch) continue;
        State x;
        load(x, c);
        add(x);
      }
      SP_STAMP(kPfMerged);
    }
    // Lane (col, hl) holds, for r = 4 rq + r3, dims 32 rq + 16 hl + 4 r3 + db.
    const float inv = 1.0f / sum_half_swap(l);
    if (q0 + col < a.n_tokens) {
      float *op = a.out + ((long long)(q0 + col) * a.n_heads + head) * kHeadDim + 16 * hl;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        st4(op + 32 * (r >> 2) + 4 * (r & 3),
            make_float4(ldexpf(O[0][r] * inv, -g), ldexpf(O[1][r] * inv, -g),
                        ldexpf(O[2][r] * inv, -g), ldexpf(O[3][r] * inv, -g)));
    }
    SP_STAMP(kPfStored);
  };

  int buf = 0;
  fetch(0);
  bool first = true;  // the run's first piece
  while (true) {
    begin();
    SP_STAMP(kPfReady);
    do {
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's copies have landed
      const int wk = __builtin_amdgcn_readfirstlane(word.x), wv = __builtin_amdgcn_readfirstlane(word.y);
      __syncthreads();  // every wave's have, and every wave is done with the other buffer
      if (left > 1) fetch(buf ^ 1);
      // a block without queries, or with none that sees the tile, only copies
      if (UQ == 32 || (q0 < a.n_tokens && kt * 32 <= a.start_pos + q0 + 31)) step(s_tile[buf], kt, wk, wv);
      buf ^= 1;
      ++kt;
      --left;
    } while (left > 0 && kt < nk);
    SP_STAMP(kPfTiles);
    const bool whole_run = first, last_piece = left == 0;
    finish(whole_run ? (int)(w1 >> 16 & 255u) : last_piece ? (int)(w2 >> 20) : 1,
           whole_run ? (int)(w1 >> 24) : 0,
           whole_run ? (int)(w2 & 1023u) : (int)(w2 >> 10 & 1023u));
    if (last_piece) break;
    first = false;
    kt = 0;
    nk = unit_tiles(++u);
  }
#if defined(BNR_TIMELINE)
  if (a.timeline && tid == 0) {
    constexpr int kHwId = 4 | (31 << 11), kXccId = 20 | (15 << 11);  // HW_REG_HW_ID, HW_REG_XCC_ID
    if ((w1 >> 16 & 255u) == 1) stamp[kPfTicket] = stamp[kPfTiles];
    stamp[kPfHwId] = ((unsigned long long)(unsigned)__builtin_amdgcn_s_getreg(kXccId) << 32) |
                     (unsigned)__builtin_amdgcn_s_getreg(kHwId);
    stamp[kPfItem] = (unsigned long long)(w1 & 0xffffu) | (unsigned long long)(w1 >> 16 & 255u) << 16 |
                     (unsigned long long)(w0 & 0xffffu) << 32;
    for (int k = 0; k < kTimelineStamps; ++k) a.timeline[(long long)blockIdx.x * kTimelineStamps + k] = stamp[k];
  }
#endif
}
#pragma clang diagnostic pop

}  // namespace

hipError_t launch_prefill_split_kv(const PrefillSplitArgs &p, hipStream_t s) {
  const RopeAppendArgs &a = p.rope;
  const long long kv_wgs = (long long)a.n_kv * p.n_tiles;
  if (a.cos_tab) {
    const long long q_wgs = ((long long)a.n_tokens * a.n_heads * 16 + 511) / 512;
    prefill_split_kv_kernel<true><<<dim3((unsigned)(kv_wgs + q_wgs)), dim3(256), 0, s>>>(p);
  } else {
    prefill_split_kv_kernel<false><<<dim3((unsigned)kv_wgs), dim3(256), 0, s>>>(p);
  }
  return hipGetLastError();
}

hipError_t launch_prefill_split(const PrefillRunsArgs &a, int group, hipStream_t s) {
  switch (group) {
    case 2: prefill_split_kernel<2><<<dim3(a.grid), dim3(64 * split_waves(2)), 0, s>>>(a); break;
    case 4: prefill_split_kernel<4><<<dim3(a.grid), dim3(64 * split_waves(4)), 0, s>>>(a); break;
    case 8: prefill_split_kernel<8><<<dim3(a.grid), dim3(64 * split_waves(8)), 0, s>>>(a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace bnr
