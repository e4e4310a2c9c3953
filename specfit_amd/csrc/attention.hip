// K5: tree-verification attention (grouped-query) on gfx950.
//
// Replaces the attention the target model runs in the verification forward
// (src/specfit/runtime/eagle3_tree.py:1202-1240 calls the HF target with the
// draft tree's mask; Qwen3MoeAttention then runs sdpa_attention_forward of
// transformers/integrations/sdpa_attention.py with that 4-D bool mask).
// For query token qi, query head qh = h*G + j of key/value head h:
//   out[qi, qh] = sum_s softmax_s(scale * q[qi, qh] . k[h, s]) * v[h, s]
// over keys s the mask admits (mask[qi, s] != 0; with no mask, s <= S - Q + qi,
// i.e. causal aligned to the end of the keys).  A query with no admitted key
// gets 0.
//
// Head dims 64 and 128 with 2..16 query heads per KV head run the tiled MFMA
// form below; device time on MI355X at 32 query / 4 KV heads of 128, against
// the 16-row MFMA form it replaced: a 4096-token prompt 1565 -> 187 us (735
// TFLOP/s of the causal half), one token over 4097 keys 49 -> 9.3 us, a 61-node
// tree over 1085 keys 26 -> 17 us; at 16 / 4 heads of 64: 2048 tokens 106 ->
// 36 us, 35 -> 8 and 18 -> 9 us.  What bounds it: prompts, the softmax's vector
// work next to the matrix work (each SIMD has two wavefronts, which overlap
// only in part); decoding and trees, latency (the K/V of 1085 keys is 2 MB).
// The loop form covers every other shape: one workgroup per (query, KV head)
// keeps the G query heads of the group together so each K/V row is read once
// per query.  Its 8 wavefronts take interleaved 64-key chunks: scores with one
// key per lane (the key row in registers, the query rows broadcast from
// LDS), an online softmax per head across the wavefront, then P.V with the
// head-dim elements spread over the lanes and the value rows of 16 keys
// loaded together.  The eight partial (max, sum, accumulator) states are
// merged in wavefront order, so the fp32 summation order is fixed and
// results are run-to-run identical.
#include "sf_common.h"

namespace {

constexpr int kChunk = SF_WAVE;  // keys per wavefront chunk

struct AttnArgs {
  const uint16_t* q;
  int64_t q_tok, q_head;
  const uint16_t* k;
  int64_t k_head, k_tok;
  const uint16_t* v;
  int64_t v_head, v_tok;
  const uint8_t* mask;  // nullptr: causal aligned to the end
  int64_t mask_q;
  int Q, S, Hkv, D;
  float scale;
  uint16_t* out;  // [Q, Hkv * G, D]
};

__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o, SF_WAVE));
  return x;
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, SF_WAVE);
  return x;
}

// x plus the value of lane `CTRL`-permuted lane (a DPP move: no LDS).
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
  const int moved = __builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false);
  return x + __int_as_float(moved);
}

// Sum over aligned groups of N lanes (N = 8 or 16), every lane gets it:
// quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror, row_mirror.
template <int N>
__device__ __forceinline__ float group_sum(float x) {
  x = dpp_add<0xB1>(x);
  x = dpp_add<0x4E>(x);
  x = dpp_add<0x141>(x);
  if (N == 16) x = dpp_add<0x140>(x);
  return x;
}

__device__ __forceinline__ void unpack8(const uint4 v, float (&f)[8]) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[2 * e] = __uint_as_float(w[e] << 16);
    f[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
  }
}

// G query heads per KV head.  DC > 0: head dim 8*DC known at compile time
// (every loop unrolled, a chunk's key and value loads issued together);
// DC == 0: any head dim (multiple of 8, <= 256) read from the arguments.
// DPL head-dim elements per lane in P.V.  NW wavefronts per workgroup.
template <int G, int DC, int DPL, int NW>
__global__ __launch_bounds__(NW * SF_WAVE) void tree_attention_kernel(const AttnArgs a) {
  constexpr int kWaves = NW;
  constexpr int kThreads = NW * SF_WAVE;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int D = DC > 0 ? 8 * DC : a.D;
  float* sq = smem;                                 // [G][D] scaled query rows
  float* sm = sq + G * D;                           // [kWaves][G] running max
  float* sl = sm + kWaves * G;                      // [kWaves][G] running sum
  float* sp = sl + kWaves * G;                      // [kWaves][G][kChunk] probabilities
  float* sacc = sp;                                 // [kWaves][G][D] accumulators (after
                                                    // the key loop, over sp)
  const int qi = blockIdx.x / a.Hkv;
  const int h = blockIdx.x - qi * a.Hkv;
  const int lane = threadIdx.x & (SF_WAVE - 1);
  const int wave = threadIdx.x / SF_WAVE;

  for (int i = threadIdx.x; i < G * D; i += kThreads) {
    const int j = i / D;
    const int d = i - j * D;
    sq[i] = sf_bf16_to_f32(a.q[qi * a.q_tok + static_cast<int64_t>(h * G + j) * a.q_head + d]) *
            a.scale;
  }
  __syncthreads();

  const uint16_t* kh = a.k + h * a.k_head;
  const uint16_t* vh = a.v + h * a.v_head;
  const int causal_last = a.S - a.Q + qi;  // last admitted key without a mask
  float m[G], l[G], acc[G][DPL];
#pragma unroll
  for (int j = 0; j < G; ++j) {
    m[j] = -INFINITY;
    l[j] = 0.f;
#pragma unroll
    for (int e = 0; e < DPL; ++e) acc[j][e] = 0.f;
  }
  float* pw = sp + wave * G * kChunk;
  const int d0 = lane * DPL;
  // Compile-time head dim: this lane's 8 query elements of every head.
  float qreg[DC > 0 ? G : 1][8];
  if (DC > 0) {
    const int dc = lane % (DC > 0 ? DC : 1);
#pragma unroll
    for (int j = 0; j < (DC > 0 ? G : 1); ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) qreg[j][e] = sq[j * D + 8 * dc + e];
  }
  const bool has_d = d0 < D;

  for (int kb = wave * kChunk; kb < a.S; kb += kWaves * kChunk) {
    const int nkeys = min(kChunk, a.S - kb);
    // Scores.  With the head dim known (DC > 0), DC lanes share one key: lane
    // l holds query elements 8*(l%DC) .. +7 of every head in registers,
    // multiplies them with its 16 B of the key row and the DC partial sums
    // are added by a butterfly; the chunk's scores go through LDS to the
    // one-key-per-lane layout of the softmax.  Otherwise lane -> key.
    const int key = kb + lane;
    bool ok = key < a.S;
    if (ok) ok = a.mask ? a.mask[qi * a.mask_q + key] != 0 : key <= causal_last;
    float s[G];
    if (DC > 0) {
      constexpr int kKeysPer = DC > 0 ? SF_WAVE / DC : 1;  // keys per instruction
      constexpr int kIters = kChunk / kKeysPer;
      const int kq = lane / (DC > 0 ? DC : 1);
      const int dc = lane % (DC > 0 ? DC : 1);
      uint4 kv[kIters];
#pragma unroll
      for (int i = 0; i < kIters; ++i) {
        const int kk = min(kb + i * kKeysPer + kq, a.S - 1);
        kv[i] = *reinterpret_cast<const uint4*>(kh + kk * a.k_tok + 8 * dc);
      }
#pragma unroll
      for (int i = 0; i < kIters; ++i) {
        float kf[8];
        unpack8(kv[i], kf);
#pragma unroll
        for (int j = 0; j < G; ++j) {
          float part = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) part = __builtin_fmaf(qreg[j][e], kf[e], part);
          part = group_sum<(DC == 16 ? 16 : 8)>(part);
          if (dc == 0) pw[j * kChunk + i * kKeysPer + kq] = part;
        }
      }
#pragma unroll
      for (int j = 0; j < G; ++j) s[j] = pw[j * kChunk + lane];
    } else {
#pragma unroll
      for (int j = 0; j < G; ++j) s[j] = 0.f;
      const uint16_t* kr = kh + min(key, a.S - 1) * a.k_tok;
      for (int d = 0; d < D; d += 8) {
        float kf[8];
        unpack8(*reinterpret_cast<const uint4*>(kr + d), kf);
#pragma unroll
        for (int j = 0; j < G; ++j) {
          const float* qr = sq + j * D + d;
#pragma unroll
          for (int e = 0; e < 8; ++e) s[j] = __builtin_fmaf(qr[e], kf[e], s[j]);
        }
      }
    }
    // Online softmax per head over this chunk.
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const float cmax = wave_max(ok ? s[j] : -INFINITY);
      const float mnew = fmaxf(m[j], cmax);
      float p = 0.f;
      float alpha = 1.f;
      if (mnew != -INFINITY) {
        alpha = m[j] == -INFINITY ? 0.f : __expf(m[j] - mnew);
        if (ok) p = __expf(s[j] - mnew);
      }
      l[j] = l[j] * alpha + wave_sum(p);
      m[j] = mnew;
#pragma unroll
      for (int e = 0; e < DPL; ++e) acc[j][e] *= alpha;
      pw[j * kChunk + lane] = p;
    }
    // P.V: head-dim elements d0 .. d0+DPL-1 per lane; the value rows of a
    // group of 16 keys are loaded together, then accumulated.
    if (has_d) {
      const uint16_t* vc = vh + kb * a.v_tok + d0;
      for (int t0 = 0; t0 < nkeys; t0 += 16) {
        float vf[16][DPL];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          const uint16_t* vr = vc + min(t0 + t, nkeys - 1) * a.v_tok;
#pragma unroll
          for (int e = 0; e < DPL; ++e) vf[t][e] = sf_bf16_to_f32(vr[e]);
        }
        // Keys past the end carry p = 0 (and a finite repeated row).
#pragma unroll
        for (int j = 0; j < G; ++j) {
          const float4* p4 = reinterpret_cast<const float4*>(pw + j * kChunk + t0);
#pragma unroll
          for (int t4 = 0; t4 < 4; ++t4) {
            const float4 p = p4[t4];
            const float pp[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
              for (int e = 0; e < DPL; ++e)
                acc[j][e] = __builtin_fmaf(pp[u], vf[4 * t4 + u][e], acc[j][e]);
          }
        }
      }
    }
  }

  // Merge the wavefront states in wavefront order.
  __syncthreads();  // every wavefront is done with sp, which sacc overlays
  if (lane == 0) {
#pragma unroll
    for (int j = 0; j < G; ++j) {
      sm[wave * G + j] = m[j];
      sl[wave * G + j] = l[j];
    }
  }
  if (has_d) {
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int e = 0; e < DPL; ++e) sacc[(wave * G + j) * D + d0 + e] = acc[j][e];
  }
  __syncthreads();
  const int Hq = a.Hkv * G;
  for (int i = threadIdx.x; i < G * D; i += kThreads) {
    const int j = i / D;
    const int d = i - j * D;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) M = fmaxf(M, sm[w * G + j]);
    float L = 0.f, O = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float mw = sm[w * G + j];
        if (mw == -INFINITY) continue;
        const float f = __expf(mw - M);
        L = __builtin_fmaf(sl[w * G + j], f, L);
        O = __builtin_fmaf(sacc[(w * G + j) * D + d], f, O);
      }
    }
    const float o = L > 0.f ? O / L : 0.f;
    a.out[(static_cast<int64_t>(qi) * Hq + h * G + j) * D + d] = sf_f32_to_bf16(o);
  }
}

// ------------------------------------------------------ tiled MFMA form --
// For head dims 64 / 128 and 2..16 query heads per KV head, with 16-byte
// aligned rows.  The Q tokens x G heads of one KV head form R = Q G query
// rows that share its keys and values.  A wavefront owns 32 of these rows
// and walks the keys in tiles of 64; the four wavefronts of a workgroup are
// WR row groups x 4 / WR key groups:
//   WR = 4: 128 rows; each K/V tile is staged once for the four wavefronts
//           (two LDS buffers, one barrier per tile; registers hold the next
//           tile's loads).  The form of prompts.
//   WR = 1: 32 rows; each wavefront takes every fourth tile into LDS of its
//           own (no barrier until the states are merged).  The form of
//           decoding and of small draft trees.
// The keys are also split over workgroups when the row tiles alone would
// leave the chip idle: each split writes its (max, sum, accumulator) in fp32
// to the caller's workspace and combine_kernel merges them in split order.
//
// Scores are computed transposed, S^T = K Q^T (v_mfma_f32_32x32x16_bf16, A =
// key rows, B = query rows): lane l then holds 32 of the tile's 64 scores of
// query row l % 32 and lane l ^ 32 the other 32, so the softmax state is one
// register per lane and its reductions are in-lane but for one half swap.
// O^T += V^T P^T takes the probabilities (bf16) as the B operand straight
// from those registers: the 16 keys of a k-step are {8 g + 4 (l / 32) ..+3},
// g = 0, 1, on both sides, and the V^T fragments in that order come from
// ds_read_b64_tr_b16 on the row-major value tile.
typedef float sf_f32x16 __attribute__((ext_vector_type(16)));
typedef short sf_i16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 sf_bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int sf_u32x4 __attribute__((ext_vector_type(4)));

constexpr int kTileKeys = 64;
constexpr int kTileWaves = 4;
constexpr int kTileThreads = kTileWaves * SF_WAVE;
constexpr int kMaxSplits = 64;

struct TiledArgs {
  AttnArgs a;
  int log_g;         // G = 1 << log_g
  int rows;          // Q * G
  int row_tiles;     // of 32 WR rows
  int splits;
  int split_keys;    // keys of one split, a multiple of 64 * 4 / WR
  float c;           // |scale| log2(e): scores to log2 units
  float* part_acc;   // [splits][Hkv][rows][D], splits > 1 only
  float2* part_ml;   // [splits][Hkv][rows] (max of the unscaled scores, sum)
};

// p = exp2(s c - m c) is one fused multiply-add per score, but it subtracts
// the rounded m c from the exact s c.  Up to this |m c| the difference at the
// row's maximum is at most 2^-13, far below the rounding of P to bf16 (2^-9);
// at 2^31 it would be 128, and the row's sum 0 or infinite.  Rows past it
// subtract before they scale (a wavefront with such a row runs the subtraction,
// of 0 for its other rows).
constexpr float kFusedMax = 4096.f;

// A wavefront multiplies V by what the bf16 rounding of P left in the first
// and then every fourth of its tiles.  One running maximum per row makes fewer
// probabilities exact (1) than eight per row (keys dealt to 8 wavefronts) do,
// so without it the error against 64 bits is larger than that form's.  Error
// of N(0, 1) inputs in 1e-3 (1.6 of them the rounding of the result): eight
// maxima / one / one with the rest of every 4th tile / of every 2nd, and
// device time of the last three: 4096-token prompt 1.97 / 2.05 / 1.84 / 1.77,
// 174 / 189 / 204 us; 512 tokens after 3000: 2.17 / 2.23 / 2.09 / 1.95, 55 /
// 57 / 60 us; 61-node tree, 1085 keys: 2.09 / 2.11 / 1.91 / 1.91, 16 us each.
// (Every 6th: 2.17 for 2000 tokens after 2096, where eight maxima have 2.16
// and every 4th 2.12.)  A tile with an infinite value or NaN goes without, as the
// rest may be 0 or negative where its key has a weight (the check: 189 -> 192 us
// for the prompt, 16.7 -> 16.9 for the tree).
constexpr int kRestTurns = 4;

// Rows padded so the fragment reads spread over the banks: 16 B for the
// 16-byte reads of K (16 consecutive rows), 32 B for the transposed reads of
// V (32 B of each of 4 rows).
template <int D>
struct TileLds {
  static constexpr int krow = 2 * D + 16;
  static constexpr int vrow = 2 * D + 32;
  static constexpr int bytes = kTileKeys * (krow + vrow);
  static constexpr int orow = D + 4;  // floats, merge of the key groups
};

template <int D, int WR>
constexpr int tiled_lds_bytes() {
  constexpr int loop = (WR == 4 ? 2 : 4 / WR) * TileLds<D>::bytes;
  constexpr int merge = WR == 4 ? 0 : (4 / WR) * 32 * WR * (TileLds<D>::orow + 2) * 4;
  return loop > merge ? loop : merge;
}

__device__ __forceinline__ sf_f32x16 mfma_32(sf_bf16x8 a, sf_bf16x8 b, sf_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Whether any of a thread's pieces of a value tile holds infinity or NaN: then
// their sum is not finite (nor is that of finite values past fp32's range,
// which may go without the rest too).
template <int N>
__device__ __forceinline__ bool has_nonfinite(const sf_u32x4 (&v)[N]) {
  const sf_bf16x2 one = __builtin_bit_cast(sf_bf16x2, 0x3f803f80u);
  float sum[2] = {0.f, 0.f};
#pragma unroll
  for (int j = 0; j < N; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = v[j][i];
      sum[i & 1] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(sf_bf16x2, w), one,
                                                   sum[i & 1], false);
    }
  return !(fabsf(sum[0]) < INFINITY && fabsf(sum[1]) < INFINITY);
}

// 16-byte load, explicitly from global memory (a flat load would also hold
// up the LDS waits).  With a byte offset: uniform address + 32-bit offset.
__device__ __forceinline__ sf_u32x4 ld16(const uint16_t* p) {
  return *(const __attribute__((address_space(1))) sf_u32x4*)(p);
}

__device__ __forceinline__ sf_u32x4 ld16(const uint16_t* p, uint32_t byte_offset) {
  return *(const __attribute__((address_space(1))) sf_u32x4*)(reinterpret_cast<const char*>(p) +
                                                             byte_offset);
}

// max(x, y) as one instruction: fmaxf first canonicalises operands that come
// from a matrix instruction.  A NaN operand gives the other one, as fmaxf.
__device__ __forceinline__ float max_raw(float x, float y) {
  return __builtin_amdgcn_fmed3f(x, y, INFINITY);
}

// Four values of a column of a row-major bf16 tile: the 16 lanes of a group
// pass the addresses of 4 rows x 4 eight-byte pieces, lane i gets column i.
__device__ __forceinline__ sf_i16x4 read_tr4(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) sf_i16x4*)(p));
}

// Value of the lane 32 away combined with the own one.
__device__ __forceinline__ float half_max(float x) {
  const int v = __float_as_int(x);
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
}

__device__ __forceinline__ float half_sum(float x) {
  const int v = __float_as_int(x);
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return __int_as_float(r[0]) + __int_as_float(r[1]);
}

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const sf_bf16x2 v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
  return __builtin_bit_cast(uint32_t, v);
}

// Registers 4 g .. 4 g + 3 of an accumulator: four consecutive head-dim elements.
__device__ __forceinline__ float4 quad(const sf_f32x16& a, int g) {
  return make_float4(a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]);
}

// Mask bytes of keys key .. key + 3 of one row (0 past the last key).
__device__ __forceinline__ uint32_t mask_word(const uint8_t* row, int key, int S) {
  uint32_t w = 0;
  if (key + 4 <= S) {
    __builtin_memcpy(&w, row + key, 4);
  } else {
    for (int i = 0; key + i < S; ++i) w |= static_cast<uint32_t>(row[key + i]) << (8 * i);
  }
  return w;
}

// One more (max, sum, accumulator) state, weighted against the maximum M of
// the unscaled scores (subtracted before scaling, see kFusedMax).
__device__ __forceinline__ void add_state(float m, float l, const float4& v, float M, float c,
                                          float& sum, float (&o)[4]) {
  const float f = __builtin_amdgcn_exp2f((m - M) * c);
  sum = __builtin_fmaf(l, f, sum);
  o[0] = __builtin_fmaf(v.x, f, o[0]);
  o[1] = __builtin_fmaf(v.y, f, o[1]);
  o[2] = __builtin_fmaf(v.z, f, o[2]);
  o[3] = __builtin_fmaf(v.w, f, o[3]);
}

// Elements d .. d + 3 of query row r (token r / G) of KV head h, divided by
// the row's sum (0 where the row admits no key).
__device__ __forceinline__ void store_row4(const TiledArgs& t, int h, int r, int D, int d,
                                           const float (&o)[4], float sum) {
  const int64_t hq = static_cast<int64_t>(t.a.Hkv) << t.log_g;
  const int64_t head = (static_cast<int64_t>(h) << t.log_g) + (r & ((1 << t.log_g) - 1));
  const float inv = 1.f / sum;
  float y[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) y[i] = sum > 0.f ? o[i] * inv : 0.f;
  *reinterpret_cast<uint2*>(t.a.out + ((r >> t.log_g) * hq + head) * D + d) =
      make_uint2(pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3]));
}

// acc += V^T P^T of a tile, P (fp32) as bf16, or with REST what that rounding
// leaves of it, as bf16.
template <int D, bool REST>
__device__ __forceinline__ void add_values(const sf_f32x16 (&p)[2], const char* vlane,
                                           sf_f32x16 (&acc)[D / 32]) {
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    sf_u32x4 w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float p0 = p[ks >> 1][8 * (ks & 1) + 2 * j];
      const float p1 = p[ks >> 1][8 * (ks & 1) + 2 * j + 1];
      w[j] = pack_bf16(p0, p1);
      if (REST)
        w[j] = pack_bf16(p0 - __uint_as_float(w[j] << 16),
                         p1 - __uint_as_float(w[j] & 0xffff0000u));
    }
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) {
      struct { sf_i16x4 lo, hi; } vf;
      vf.lo = read_tr4(vlane + 16 * ks * TileLds<D>::vrow + 64 * dt);
      vf.hi = read_tr4(vlane + (16 * ks + 8) * TileLds<D>::vrow + 64 * dt);
      acc[dt] = mfma_32(__builtin_bit_cast(sf_bf16x8, vf), __builtin_bit_cast(sf_bf16x8, w),
                        acc[dt]);
    }
  }
}

template <int D, int WR, bool MASK>
__global__ __launch_bounds__(kTileThreads, WR == 4 ? 2 : 1) void tree_attention_tiled_kernel(
    const TiledArgs t) {
  const AttnArgs& a = t.a;
  constexpr int kWk = kTileWaves / WR;      // key groups
  constexpr int kSteps = D / 16;            // MFMA k-steps of a score tile
  constexpr int kDt = D / 32;               // 32-wide head-dim tiles of the output
  constexpr int kRowLanes = D / 8;          // 16-byte pieces of a row
  constexpr int kLoads = kRowLanes / WR;    // pieces of a 64-row tile per thread
  using L = TileLds<D>;
  __shared__ __attribute__((aligned(16))) char lds[tiled_lds_bytes<D, WR>()];
  // WR = 4: what each wavefront found in its part of the value tile.
  __shared__ __attribute__((aligned(16))) int nonfinite[2][kTileWaves];
  const int lane = threadIdx.x & (SF_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SF_WAVE);
  const int kg = wave / WR;
  const int hf = lane >> 5;
  const int col = lane & 31;
  // Consecutive workgroups take different KV heads (an XCD then keeps one or
  // few heads' K/V in its L2); the last row tiles, which see the most keys
  // under the causal rule, go first.
  const int h = blockIdx.x % a.Hkv;
  const int rest = blockIdx.x / a.Hkv;
  const int split = rest % t.splits;
  const int block_row = (t.row_tiles - 1 - rest / t.splits) * 32 * WR;
  const int wave_row = block_row + 32 * (wave % WR);
  const bool active = wave_row < t.rows;
  const int row = wave_row + col;
  const int row_c = min(row, t.rows - 1);
  const int tok = row_c >> t.log_g;
  const int head = (h << t.log_g) + (row_c & ((1 << t.log_g) - 1));

  // B operand of the scores: this lane's query row.  A negative scale flips
  // the signs here (exact), so the row maximum is that of the scaled scores.
  sf_bf16x8 qf[kSteps];
  {
    const uint16_t* qr = a.q + tok * a.q_tok + head * a.q_head + 8 * hf;
    const uint32_t flip = a.scale < 0.f ? 0x80008000u : 0u;
#pragma unroll
    for (int s = 0; s < kSteps; ++s)
      qf[s] = __builtin_bit_cast(sf_bf16x8, ld16(qr + 16 * s) ^ flip);
  }
  const float c = t.c;

  // Keys: [begin, end) for the workgroup; the wavefront's rows see none from
  // wave_end on, and all of them see the keys below wave_full.
  const int last_row = min(block_row + 32 * WR, t.rows) - 1;
  const int diag = a.S - a.Q + 1;
  const int begin = split * t.split_keys;
  int end = min(a.S, begin + t.split_keys);
  int wave_end = end, wave_full = 0;
  if (!MASK) {
    end = min(end, diag + (last_row >> t.log_g));
    wave_end = min(end, diag + (min(wave_row + 31, t.rows - 1) >> t.log_g));
    wave_full = diag + (min(wave_row, t.rows - 1) >> t.log_g);
  }
  const int lane_end = MASK ? a.S : diag + tok;  // keys this lane's row sees (no mask)
  const uint16_t* kh = a.k + h * a.k_head;
  const uint16_t* vh = a.v + h * a.v_head;
  const uint8_t* mrow = MASK ? a.mask + tok * a.mask_q : nullptr;

  float m = -INFINITY, l = 0.f;  // row maximum (unscaled), this half's sum
  sf_f32x16 acc[kDt];
#pragma unroll
  for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;

  // Piece gt + j * 64 WR of a tile: row piece / kRowLanes.
  const int gt = threadIdx.x % (SF_WAVE * WR);
  const int ld_row = gt / kRowLanes;
  const int ld_col = gt % kRowLanes;
  constexpr int kRowsPerLoad = SF_WAVE * WR / kRowLanes;
  sf_u32x4 kr[kLoads], vr[kLoads];
  uint32_t mw[8];
  const uint32_t k_off = 2 * (ld_row * static_cast<uint32_t>(a.k_tok) + 8 * ld_col);
  const uint32_t v_off = 2 * (ld_row * static_cast<uint32_t>(a.v_tok) + 8 * ld_col);
  auto load_tile = [&](int kb) {
    if (kb + kTileKeys <= a.S) {
      const uint16_t* kp = kh + kb * a.k_tok;
      const uint16_t* vp = vh + kb * a.v_tok;
#pragma unroll
      for (int j = 0; j < kLoads; ++j) kr[j] = ld16(kp + j * kRowsPerLoad * a.k_tok, k_off);
#pragma unroll
      for (int j = 0; j < kLoads; ++j) vr[j] = ld16(vp + j * kRowsPerLoad * a.v_tok, v_off);
    } else {
      // Rows past the end: the last key's score, masked, and values of 0 (an
      // infinite last value would meet p = 0).
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const int at = kb + j * kRowsPerLoad + ld_row;
        const int64_t key = min(at, a.S - 1);
        kr[j] = ld16(kh + key * a.k_tok + 8 * ld_col);
        vr[j] = sf_u32x4(0u);
        if (at < a.S) vr[j] = ld16(vh + key * a.v_tok + 8 * ld_col);
      }
    }
    if (MASK) {
#pragma unroll
      for (int g = 0; g < 8; ++g) mw[g] = mask_word(mrow, kb + 8 * g + 4 * hf, a.S);
    }
  };

  int kb = begin + kg * kTileKeys;
  if (kb < end) load_tile(kb);
  char* tile = lds + kg * L::bytes;
  int buf = 0;
  for (int turn = 0; kb < end; kb += kTileKeys * kWk, ++turn) {
    if (WR == 4) tile = lds + (buf ^= 1) * L::bytes;
    char* ktile = tile;
    char* vtile = tile + kTileKeys * L::krow;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int r = j * kRowsPerLoad + ld_row;
      *reinterpret_cast<sf_u32x4*>(ktile + r * L::krow + 16 * ld_col) = kr[j];
      *reinterpret_cast<sf_u32x4*>(vtile + r * L::vrow + 16 * ld_col) = vr[j];
    }
    bool rest = turn % kRestTurns == 0;
    if (rest) {
      rest = !__any(has_nonfinite(vr));
      if (WR == 4 && lane == 0) nonfinite[buf][wave] = !rest;
    }
    uint32_t mc[8];
    if (MASK) {
#pragma unroll
      for (int g = 0; g < 8; ++g) mc[g] = mw[g];
    }
    if (kb + kTileKeys * kWk < end) load_tile(kb + kTileKeys * kWk);
    if (WR == 4)
      __syncthreads();  // the tile is complete; the other buffer's reads are done
    else
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (active && kb < wave_end) {
      sf_f32x16 s[2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[kt][i] = 0.f;
#pragma unroll
        for (int st = 0; st < kSteps; ++st) {
          const sf_bf16x8 kf = *reinterpret_cast<const sf_bf16x8*>(
              ktile + (32 * kt + col) * L::krow + 32 * st + 16 * hf);
          s[kt] = mfma_32(kf, qf[st], s[kt]);
        }
      }
      // Keys the row does not admit: -inf (their p is 0).
      if (MASK) {
        bool all = true;
#pragma unroll
        for (int g = 0; g < 8; ++g) all = all && mc[g] == 0x01010101u;
        if (!__all(all)) {
#pragma unroll
          for (int g = 0; g < 8; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (!((mc[g] >> (8 * i)) & 0xffu)) s[g >> 2][4 * (g & 3) + i] = -INFINITY;
        }
      } else if (kb + kTileKeys > wave_full) {
#pragma unroll
        for (int g = 0; g < 8; ++g)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (kb + 8 * g + 4 * hf + i >= lane_end) s[g >> 2][4 * (g & 3) + i] = -INFINITY;
      }
      float mx[2] = {s[0][0], s[1][0]};
#pragma unroll
      for (int i = 1; i < 16; ++i)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) mx[kt] = max_raw(mx[kt], s[kt][i]);
      const float mnew = fmaxf(m, half_max(max_raw(mx[0], mx[1])));
      if (__any(mnew > m)) {
        const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - mnew) * c);
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[dt][i] *= alpha;
        m = mnew;
      }
      float base = m == -INFINITY ? 0.f : -(m * c);
      const bool large = fabsf(base) > kFusedMax;
      if (__any(large)) {
        const float top = large ? m : 0.f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[kt][i] -= top;
        if (large) base = 0.f;
      }
      float sum[2] = {0.f, 0.f};
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[kt][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][i], c, base));
          sum[i & 1] += s[kt][i];
        }
      l += sum[0] + sum[1];
      const char* vlane = vtile + (4 * hf + ((lane & 15) >> 2)) * L::vrow +
                          32 * ((lane >> 4) & 1) + 8 * (lane & 3);
      add_values<D, false>(s, vlane, acc);
      if (turn % kRestTurns == 0) {
        if (WR == 4) {
          const int4 bad = *reinterpret_cast<const int4*>(nonfinite[buf]);
          rest = !__builtin_amdgcn_readfirstlane(bad.x | bad.y | bad.z | bad.w);
        }
        if (rest) add_values<D, true>(s, vlane, acc);
      }
    }
    if (WR != 4) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // tile reused
  }
  l = half_sum(l);

  const int64_t part_row = (static_cast<int64_t>(split) * a.Hkv + h) * t.rows;
  if (WR == 4) {
    if (row >= t.rows) return;
    if (t.splits > 1) {
      if (hf == 0) t.part_ml[part_row + row] = make_float2(m, l);
      if (m == -INFINITY) return;  // never read
      float* o = t.part_acc + (part_row + row) * D + 4 * hf;
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<float4*>(o + 32 * dt + 8 * g) = quad(acc[dt], g);
      return;
    }
#pragma unroll
    for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 v = quad(acc[dt], g);
        const float o[4] = {v.x, v.y, v.z, v.w};
        store_row4(t, h, row, D, 32 * dt + 8 * g + 4 * hf, o, l);
      }
  } else {
    // Merge the key groups in order.  Their state overlays every tile.
    __syncthreads();
    constexpr int kRows = 32 * WR;
    float* sacc = reinterpret_cast<float*>(lds);                 // [kWk][kRows][orow]
    float* sml = sacc + kWk * kRows * L::orow;                   // [kWk][kRows][2]
    const int lrow = kg * kRows + 32 * (wave % WR) + col;
    if (hf == 0) {
      sml[2 * lrow] = m;
      sml[2 * lrow + 1] = l;
    }
#pragma unroll
    for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(sacc + lrow * L::orow + 32 * dt + 8 * g + 4 * hf) =
            quad(acc[dt], g);
    __syncthreads();
    for (int i = threadIdx.x; i < kRows * (D / 4); i += kTileThreads) {
      const int lr = i / (D / 4);
      const int d = 4 * (i % (D / 4));
      const int r = block_row + lr;
      if (r >= t.rows) break;
      float M = -INFINITY, sum = 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < kWk; ++w) M = fmaxf(M, sml[2 * (w * kRows + lr)]);
#pragma unroll
      for (int w = 0; w < kWk; ++w) {
        const float wm = sml[2 * (w * kRows + lr)];
        if (wm == -INFINITY) continue;
        add_state(wm, sml[2 * (w * kRows + lr) + 1],
                  *reinterpret_cast<const float4*>(sacc + (w * kRows + lr) * L::orow + d), M, c,
                  sum, o);
      }
      if (t.splits > 1) {
        if (d == 0) t.part_ml[part_row + r] = make_float2(M, sum);
        *reinterpret_cast<float4*>(t.part_acc + (part_row + r) * D + d) =
            make_float4(o[0], o[1], o[2], o[3]);
      } else {
        store_row4(t, h, r, D, d, o, sum);
      }
    }
  }
}

// Merges the key splits of every query row in split order.  A row's D / 4
// threads read its splits' accumulators with all loads in flight at once: one
// group of threads for up to 8 splits, eight groups (merged through LDS, in
// group order) above.
constexpr int kMergeDepth = 8;  // splits per group

template <int D, int GROUPS>
__global__ __launch_bounds__(kTileThreads) void tree_attention_merge_kernel(const TiledArgs t) {
  constexpr int kLanes = D / 4;
  constexpr int kSubs = kTileThreads / kLanes;
  constexpr int kRows = kSubs / GROUPS;
  static_assert(GROUPS * kMergeDepth <= kMaxSplits, "splits per row");
  __shared__ float sml[kSubs][2];
  __shared__ float4 sacc[GROUPS > 1 ? kSubs : 1][kLanes];
  const AttnArgs& a = t.a;
  const int sub = threadIdx.x / kLanes;
  const int dl = threadIdx.x % kLanes;
  const int g = sub % GROUPS;
  const int64_t total = static_cast<int64_t>(a.Hkv) * t.rows;
  const int64_t hr = static_cast<int64_t>(blockIdx.x) * kRows + sub / GROUPS;
  const bool valid = hr < total;
  const int64_t base = valid ? hr : 0;
  float2 ml[kMergeDepth];
  float4 v[kMergeDepth];
#pragma unroll
  for (int j = 0; j < kMergeDepth; ++j) {
    const int s = g + GROUPS * j;
    ml[j] = make_float2(-INFINITY, 0.f);
    v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (s < t.splits) {
      ml[j] = t.part_ml[s * total + base];
      // Not written (and not used) where the split admits no key of the row.
      v[j] = *reinterpret_cast<const float4*>(t.part_acc + (s * total + base) * D + 4 * dl);
    }
  }
  float M = -INFINITY, sum = 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < kMergeDepth; ++j) M = fmaxf(M, ml[j].x);
#pragma unroll
  for (int j = 0; j < kMergeDepth; ++j) {
    if (ml[j].x == -INFINITY) continue;
    add_state(ml[j].x, ml[j].y, v[j], M, t.c, sum, o);
  }
  if (GROUPS > 1) {
    if (dl == 0) {
      sml[sub][0] = M;
      sml[sub][1] = sum;
    }
    sacc[sub][dl] = make_float4(o[0], o[1], o[2], o[3]);
    __syncthreads();
    if (g != 0) return;
    M = -INFINITY;
#pragma unroll
    for (int w = 0; w < GROUPS; ++w) M = fmaxf(M, sml[sub + w][0]);
    sum = o[0] = o[1] = o[2] = o[3] = 0.f;
#pragma unroll
    for (int w = 0; w < GROUPS; ++w) {
      if (sml[sub + w][0] == -INFINITY) continue;
      add_state(sml[sub + w][0], sml[sub + w][1], sacc[sub + w][dl], M, t.c, sum, o);
    }
  }
  if (valid)
    store_row4(t, static_cast<int>(hr / t.rows), static_cast<int>(hr % t.rows), D, 4 * dl, o, sum);
}

bool aligned(const void* p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

// |scale| log2(e), the factor that takes scores to log2 units.  It must be a
// normal finite number: a masked score of -inf times 0 would be NaN.
float log2_scale(float scale) { return __builtin_fabsf(scale) * 1.44269504088896341f; }

bool scale_ok(float scale) {
  const float c = log2_scale(scale);
  return c >= 1.17549435e-38f && c <= 3.0e38f;
}

// Shapes of the tiled form: head dim 64 or 128, 2..16 query heads per KV head
// (powers of two), row and key numbers that stay in 32 bits (a plan's splits
// reach up to kMaxSplits steps past the last key).
bool tiled_shape(int queries, int keys, int G, int head_dim) {
  return (head_dim == 64 || head_dim == 128) && G >= 2 && G <= 16 && (G & (G - 1)) == 0 &&
         static_cast<int64_t>(queries) * G <= 0x3fffffff &&
         keys <= 0x7fffffff - 4 * kMaxSplits * kTileKeys * kTileWaves;
}

// Row groups (WR) and key splits of a call.
struct TiledPlan {
  int wr, row_tiles, splits, split_keys;
};

// The form and split with the least estimated time.  A workgroup's step (one
// 64-key tile at WR = 4, four at WR = 1) takes about 1.2 / 2.4 us on MI355X,
// 1.6 / 2.9 us with a mask; splitting adds the merge launch (2.5 us on the
// device, and 3 us of the caller's time with the scratch allocation, which
// short calls wait for) and the partial states' way through memory (0.28 ns
// per row and split, 1 KiB each); a CU runs one WR = 1 workgroup at a time,
// and WR = 4 workgroups above 1.5 per CU wait for each other.  Measured at 32
// query / 4 KV heads of 128 (us; all but the first line before the rest of P,
// which lengthens every form by 2 - 10%):
//   1 query, 4097 keys:     82.6 unsplit, 9.0 in 33 splits (WR = 4); 43.7 unsplit (WR = 1)
//   32 queries, 1056 keys:  21.8 unsplit, 12.2 in 5 (WR = 1); 13.4 WR = 4
//   61 queries, 1085 keys:  22.0 unsplit, 15.9 in 3, 20.2 in 5 (WR = 1)
//   129 queries, 8129 keys: 227 unsplit, 46.8 in 11, 54.3 in 32 (WR = 4)
//   256 queries and keys:   8.8 unsplit (WR = 1), 10.9 (WR = 4), 13.9 in 2
// Head dim 64 shares these numbers; its steps are shorter, and its plans were
// only checked against the form before the key splits (16 / 4 heads: 64
// queries, 4096 keys: 35.7 -> 10.6; 256, 3000: 30.3 -> 16.5; 129, 8129 with a
// mask: 96.7 -> 27.4).
// may_split: the caller has scratch for the partial states.
TiledPlan tiled_plan(int queries, int keys, int kv_heads, int G, bool mask, bool may_split) {
  const int64_t rows = static_cast<int64_t>(queries) * G;
  TiledPlan best{};
  double best_cost = 0.0;
  for (int wr = 4; wr >= 1; wr -= 3) {
    const int unit = kTileKeys * (kTileWaves / wr);
    const int units = (keys + unit - 1) / unit;
    const int64_t row_tiles = (rows + 32 * wr - 1) / (32 * wr);
    const int64_t blocks = row_tiles * kv_heads;
    const double step = wr == 4 ? (mask ? 1.6 : 1.2) : (mask ? 2.9 : 2.4);
    const int most = !may_split ? 1 : units < kMaxSplits ? units : kMaxSplits;
    int last = 0;
    for (int want = 1; want <= most; ++want) {
      const int per = (units + want - 1) / want;
      const int splits = (units + per - 1) / per;
      if (splits == last) continue;
      last = splits;
      const double total = static_cast<double>(blocks) * splits;
      double turns = wr == 4 ? total / 384.0 : __builtin_ceil(total / 256.0);
      if (turns < 1.0) turns = 1.0;
      double cost = per * step * turns + (wr == 4 ? 0.0 : 0.4);
      if (splits > 1) cost += 5.5 + 0.28e-3 * static_cast<double>(rows) * kv_heads * splits;
      if (best.wr && cost >= best_cost) continue;
      best_cost = cost;
      best = TiledPlan{wr, static_cast<int>(row_tiles), splits, per * unit};
      if (total > 2048) break;  // the chip is full: more splits only add to the merge
    }
  }
  return best;
}

int64_t tiled_workspace(const TiledPlan& p, int queries, int q_heads, int head_dim) {
  if (p.splits == 1) return 0;
  return static_cast<int64_t>(p.splits) * queries * q_heads * (head_dim + 2) * 4;
}

template <int D>
int launch_tiled(const AttnArgs& a, int G, void* workspace, int64_t workspace_bytes,
                 hipStream_t s) {
  // Without the scratch of the best split, the best unsplit form: its row
  // groups may be others (one token over 4097 keys: 43.7 us, where the split
  // plan's row groups in one split take 82.6).
  TiledPlan p = tiled_plan(a.Q, a.S, a.Hkv, G, a.mask != nullptr, true);
  const int64_t need = tiled_workspace(p, a.Q, a.Hkv * G, D);
  if (need > workspace_bytes || (need && (!workspace || !aligned(workspace, 16))))
    p = tiled_plan(a.Q, a.S, a.Hkv, G, a.mask != nullptr, false);
  TiledArgs t{};
  t.a = a;
  t.log_g = __builtin_ctz(G);
  t.rows = a.Q * G;
  t.row_tiles = p.row_tiles;
  t.splits = p.splits;
  t.split_keys = p.split_keys;
  t.c = log2_scale(a.scale);
  if (p.splits > 1) {
    t.part_acc = static_cast<float*>(workspace);
    t.part_ml = reinterpret_cast<float2*>(
        t.part_acc + static_cast<int64_t>(p.splits) * a.Hkv * t.rows * D);
  }
  const dim3 grid(static_cast<unsigned>(static_cast<int64_t>(p.row_tiles) * a.Hkv * p.splits));
  const dim3 block(kTileThreads);
  if (p.wr == 4) {
    if (a.mask) tree_attention_tiled_kernel<D, 4, true><<<grid, block, 0, s>>>(t);
    else tree_attention_tiled_kernel<D, 4, false><<<grid, block, 0, s>>>(t);
  } else {
    if (a.mask) tree_attention_tiled_kernel<D, 1, true><<<grid, block, 0, s>>>(t);
    else tree_attention_tiled_kernel<D, 1, false><<<grid, block, 0, s>>>(t);
  }
  SF_LAUNCH_CHECK();
  if (p.splits > 1) {
    constexpr int kSubs = kTileThreads / (D / 4);
    const int64_t total = static_cast<int64_t>(a.Hkv) * t.rows;
    const int64_t rows = p.splits <= kMergeDepth ? kSubs : kSubs / 8;  // of a workgroup
    const dim3 merge_grid(static_cast<unsigned>((total + rows - 1) / rows));
    if (p.splits <= kMergeDepth) tree_attention_merge_kernel<D, 1><<<merge_grid, block, 0, s>>>(t);
    else tree_attention_merge_kernel<D, 8><<<merge_grid, block, 0, s>>>(t);
    SF_LAUNCH_CHECK();
  }
  return SF_OK;
}

// Wavefronts per workgroup: 8 up to 8 heads per group, 4 for 16 (LDS).
constexpr int waves_for(int G) { return G <= 8 ? 8 : 4; }

// LDS bytes of one workgroup: query rows, merge state, and the larger of
// the chunk probabilities and the merge accumulators.
size_t lds_bytes(int G, int D) {
  const size_t w = waves_for(G);
  const size_t shared = w * G * (D > kChunk ? D : kChunk);
  return sizeof(float) * (static_cast<size_t>(G) * D + 2 * w * G + shared);
}

constexpr size_t kMaxLds = 64 * 1024;

template <int G>
int launch_g(const AttnArgs& a, hipStream_t s) {
  constexpr int NW = waves_for(G);
  const size_t lds = lds_bytes(G, a.D);
  const dim3 grid(static_cast<unsigned>(a.Q) * a.Hkv);
  const dim3 block(NW * SF_WAVE);
  // Fixed head dims 64 / 128 up to 8 heads per group (more would spill).
  if (G <= 8 && a.D == 128)
    tree_attention_kernel<G, (G <= 8 ? 16 : 0), 2, NW><<<grid, block, lds, s>>>(a);
  else if (G <= 8 && a.D == 64)
    tree_attention_kernel<G, (G <= 8 ? 8 : 0), 1, NW><<<grid, block, lds, s>>>(a);
  else if (a.D <= SF_WAVE)
    tree_attention_kernel<G, 0, 1, NW><<<grid, block, lds, s>>>(a);
  else if (a.D <= 2 * SF_WAVE)
    tree_attention_kernel<G, 0, 2, NW><<<grid, block, lds, s>>>(a);
  else
    tree_attention_kernel<G, 0, 4, NW><<<grid, block, lds, s>>>(a);
  SF_LAUNCH_CHECK();
  return SF_OK;
}

}  // namespace

namespace {

int attention_call(const void* q, int64_t q_stride_token, int64_t q_stride_head, const void* k,
                   int64_t k_stride_head, int64_t k_stride_token, const void* v,
                   int64_t v_stride_head, int64_t v_stride_token, const uint8_t* mask,
                   int64_t mask_stride_query, int queries, int keys, int q_heads, int kv_heads,
                   int head_dim, float scale, void* out, void* workspace, int64_t workspace_bytes,
                   hipStream_t s) {
  if (queries < 1 || keys < 1 || q_heads < 1 || kv_heads < 1 || head_dim < 1)
    return SF_ERR_INVALID_ARGUMENT;
  if (!q || !k || !v || !out) return SF_ERR_INVALID_ARGUMENT;
  if (q_heads % kv_heads) return SF_ERR_UNSUPPORTED_SHAPE;
  const int G = q_heads / kv_heads;
  if (head_dim % 8 || head_dim > 4 * SF_WAVE) return SF_ERR_UNSUPPORTED_SHAPE;
  if (lds_bytes(G, head_dim) > kMaxLds) return SF_ERR_UNSUPPORTED_SHAPE;
  if (static_cast<long long>(queries) * kv_heads > 0x7fffffffLL) return SF_ERR_UNSUPPORTED_SHAPE;
  if (q_stride_token < 0 || q_stride_head < 0 || k_stride_head < 0 || v_stride_head < 0 ||
      k_stride_token < head_dim || v_stride_token < head_dim ||
      (mask && mask_stride_query < keys))
    return SF_ERR_INVALID_ARGUMENT;
  // Key rows are read 16 B at a time; value rows DPL elements per lane.
  const int dpl = (head_dim + SF_WAVE - 1) / SF_WAVE;
  if (!aligned(k, 16) || k_stride_token % 8 || k_stride_head % 8) return SF_ERR_MISALIGNED;
  const int dpl_bytes = dpl * 2;
  if (!aligned(v, dpl_bytes) || (v_stride_token * 2) % dpl_bytes || (v_stride_head * 2) % dpl_bytes)
    return SF_ERR_MISALIGNED;
  AttnArgs a{};
  a.q = static_cast<const uint16_t*>(q);
  a.q_tok = q_stride_token;
  a.q_head = q_stride_head;
  a.k = static_cast<const uint16_t*>(k);
  a.k_head = k_stride_head;
  a.k_tok = k_stride_token;
  a.v = static_cast<const uint16_t*>(v);
  a.v_head = v_stride_head;
  a.v_tok = v_stride_token;
  a.mask = mask;
  a.mask_q = mask_stride_query;
  a.Q = queries;
  a.S = keys;
  a.Hkv = kv_heads;
  a.D = head_dim;
  a.scale = scale;
  a.out = static_cast<uint16_t*>(out);
  // The tiled form: 16-byte aligned query / key / value rows (8-element
  // strides) and a scale its log2 units can hold.
  const bool tiled = tiled_shape(queries, keys, G, head_dim) && aligned(q, 16) && aligned(v, 16) &&
                     aligned(out, 8) && q_stride_token % 8 == 0 && q_stride_head % 8 == 0 &&
                     v_stride_token % 8 == 0 && v_stride_head % 8 == 0 &&
                     k_stride_token < (1 << 24) && v_stride_token < (1 << 24) &&
                     scale_ok(scale);
  if (tiled && head_dim == 128) return launch_tiled<128>(a, G, workspace, workspace_bytes, s);
  if (tiled && head_dim == 64) return launch_tiled<64>(a, G, workspace, workspace_bytes, s);
  switch (G) {
    case 1: return launch_g<1>(a, s);
    case 2: return launch_g<2>(a, s);
    case 4: return launch_g<4>(a, s);
    case 8: return launch_g<8>(a, s);
    case 16: return launch_g<16>(a, s);
    default: return SF_ERR_UNSUPPORTED_SHAPE;
  }
}

}  // namespace

extern "C" int sf_tree_attention(const void* q, int64_t q_stride_token, int64_t q_stride_head,
                                 const void* k, int64_t k_stride_head, int64_t k_stride_token,
                                 const void* v, int64_t v_stride_head, int64_t v_stride_token,
                                 const uint8_t* mask, int64_t mask_stride_query, int queries,
                                 int keys, int q_heads, int kv_heads, int head_dim, float scale,
                                 void* out, sf_stream_t stream) {
  return attention_call(q, q_stride_token, q_stride_head, k, k_stride_head, k_stride_token, v,
                        v_stride_head, v_stride_token, mask, mask_stride_query, queries, keys,
                        q_heads, kv_heads, head_dim, scale, out, nullptr, 0,
                        reinterpret_cast<hipStream_t>(stream));
}

extern "C" int64_t sf_tree_attention_workspace(int queries, int keys, int q_heads, int kv_heads,
                                               int head_dim, int masked) {
  if (queries < 1 || keys < 1 || kv_heads < 1 || q_heads < kv_heads || q_heads % kv_heads) return 0;
  const int G = q_heads / kv_heads;
  if (!tiled_shape(queries, keys, G, head_dim)) return 0;
  return tiled_workspace(tiled_plan(queries, keys, kv_heads, G, masked != 0, true), queries,
                         q_heads, head_dim);
}

extern "C" int sf_tree_attention_split(const void* q, int64_t q_stride_token,
                                       int64_t q_stride_head, const void* k,
                                       int64_t k_stride_head, int64_t k_stride_token,
                                       const void* v, int64_t v_stride_head,
                                       int64_t v_stride_token, const uint8_t* mask,
                                       int64_t mask_stride_query, int queries, int keys,
                                       int q_heads, int kv_heads, int head_dim, float scale,
                                       void* out, void* workspace, int64_t workspace_bytes,
                                       sf_stream_t stream) {
  return attention_call(q, q_stride_token, q_stride_head, k, k_stride_head, k_stride_token, v,
                        v_stride_head, v_stride_token, mask, mask_stride_query, queries, keys,
                        q_heads, kv_heads, head_dim, scale, out, workspace, workspace_bytes,
                        reinterpret_cast<hipStream_t>(stream));
}
