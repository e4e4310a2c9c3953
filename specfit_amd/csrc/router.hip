// K1: fused router -- bf16 logits, fp32 softmax, top-k with wavefront-shuffle
// argmax, optional renormalisation.  Restates Qwen3MoeTopKRouter.forward
// (transformers qwen3_moe modeling file, tf:258-267) for gfx950.
//
// Arithmetic contract (the CPU oracle evaluates exactly this):
//  * logit[t,e]: lane l of a 64-wide wavefront owns the 8-element chunks
//    c = l, l+64, l+128, ... of the hidden dimension and accumulates
//    hidden[k]*W[e,k] for its k in ascending order into an fp32 partial that
//    starts at +0 (bf16*bf16 products are exact in fp32, so fused and unfused
//    accumulation agree).  The 64 partials are combined by an xor butterfly
//    with distances 1,2,4,8,16,32 (v[l] += v[l^d]); the result is rounded to
//    bf16 (nearest even).
//  * softmax: m = max logit; x_e = exp(logit_e - m) with sf_exp_nonpos; lane l
//    owns experts l, l+64, l+128, l+192 and sums its x_e in that order from
//    +0, then the same butterfly combines lanes; p_e = x_e / sum (IEEE
//    division).
//  * top-k: k rounds of argmax over unselected experts with key
//    (p descending, expert id ascending).
//  * weights: v_j / (((v_0 + v_1) + v_2) + ...) when renormalising, else v_j,
//    rounded to bf16.
// Wavefront reductions are DPP moves and lane reads (sf_wave_sum /
// sf_wave_max), which give exactly these butterfly sums.
#include "sf_common.h"

namespace {

constexpr int kRouterThreads = 256;
constexpr int kRouterWaves = kRouterThreads / SF_WAVE;

__device__ __forceinline__ float dot8_acc(uint4 hv, uint4 wv, float acc) {
  const uint32_t hw[4] = {hv.x, hv.y, hv.z, hv.w};
  const uint32_t ww[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float h0 = __uint_as_float(hw[q] << 16);
    float w0 = __uint_as_float(ww[q] << 16);
    float h1 = __uint_as_float(hw[q] & 0xffff0000u);
    float w1 = __uint_as_float(ww[q] & 0xffff0000u);
    acc = __builtin_fmaf(h0, w0, acc);
    acc = __builtin_fmaf(h1, w1, acc);
  }
  return acc;
}

typedef unsigned int router_u32x4 __attribute__((ext_vector_type(4)));

// 16 bytes at a uniform address plus a 32-bit byte offset.
__device__ __forceinline__ router_u32x4 router_ld16(const uint16_t* p, uint32_t byte_offset) {
  return *(const __attribute__((address_space(1))) router_u32x4*)(
      reinterpret_cast<const char*>(p) + byte_offset);
}

// Softmax + top-k + renorm over s_logit[0..E) by one wavefront.  Lane l
// reads only experts l, l+64, ... of s_logit.  Each top-k round takes the
// wave maximum of the unselected probabilities and the lowest expert id
// holding it (ballots per 64-expert slice, lowest lane first).  The rounds
// compare the probabilities' bit patterns as integers: p is in [0, 1] for
// finite logits, so integer order is float order and equal bits are equal
// values; -1 marks a slot past E or an expert already taken.  Lane r keeps
// round r's value and id, so the renormalisation divides in K lanes at once
// and the stores are contiguous.
template <int J>  // experts per lane: E <= 64 * J
__device__ void softmax_topk_wave(const float* s_logit, int E, int K, int renorm,
                                  uint16_t* topw, int64_t* topi) {
  const int lane = threadIdx.x & (SF_WAVE - 1);
  float m = -__builtin_inff();
#pragma unroll
  for (int j = 0; j < J; ++j) {
    int e = lane + SF_WAVE * j;
    if (e < E) m = fmaxf(m, s_logit[e]);
  }
  m = sf_wave_max(m);
  float x[J];
  float part = 0.0f;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    int e = lane + SF_WAVE * j;
    if (e < E) {
      x[j] = sf_exp_nonpos(s_logit[e] - m);
      part += x[j];
    } else {
      x[j] = 0.0f;
    }
  }
  const float total = sf_wave_sum(part);
  int key[J];
#pragma unroll
  for (int j = 0; j < J; ++j) key[j] = lane + SF_WAVE * j < E ? __float_as_int(x[j] / total) : -1;
  float mine = 0.0f;
  int mine_id = 0;
  for (int r = 0; r < K; ++r) {
    int lk = key[0];
#pragma unroll
    for (int j = 1; j < J; ++j) lk = max(lk, key[j]);
    const int bk = sf_wave_max_int(lk);
    int be = -1;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const unsigned long long hit = __ballot(key[j] == bk);
      if (be < 0 && hit) be = SF_WAVE * j + __ffsll(hit) - 1;
    }
#pragma unroll
    for (int j = 0; j < J; ++j)
      if (be == lane + SF_WAVE * j) key[j] = -1;
    if (lane == r) {
      mine = __int_as_float(bk);
      mine_id = be;
    }
  }
  float sum = 0.0f;
  if (renorm)
    for (int r = 0; r < K; ++r) sum += sf_readlane(mine, r);
  if (lane < K) {
    const float v = renorm ? mine / sum : mine;
    topw[lane] = sf_f32_to_bf16(v);
    topi[lane] = static_cast<int64_t>(mine_id);
  }
}

// Vector path: hidden_size % 8 == 0, 16-byte aligned rows and at most NCH
// chunks of 8 elements per lane.  Two kernels, so the dot products spread
// over the whole chip: the logits kernel gives each wavefront a tile of TT
// tokens x EPW experts (all loads of the tile issued before any use, each
// logit summed per lane and butterflied exactly as above), the select
// kernel runs softmax / top-k / renormalisation with one wavefront per
// token.
constexpr int kLogitWaves = 4;
template <int NCH>
struct LogitTile {
  static constexpr int experts = NCH <= 4 ? 4 : (NCH <= 8 ? 2 : 1);  // per wavefront
  static constexpr int tokens = NCH <= 4 ? 2 : 1;
};

template <int NCH>
__global__ __launch_bounds__(kLogitWaves * SF_WAVE) void router_logits_kernel(
    const uint16_t* __restrict__ hidden, const uint16_t* __restrict__ wr, int T, int H,
    int E, uint16_t* __restrict__ logits) {
  constexpr int EPW = LogitTile<NCH>::experts;
  constexpr int TT = LogitTile<NCH>::tokens;
  const int lane = threadIdx.x & (SF_WAVE - 1);
  const int wave = threadIdx.x / SF_WAVE;
  const int t0 = blockIdx.x * TT;
  const int e0 = (blockIdx.y * kLogitWaves + wave) * EPW;
  if (e0 >= E) return;  // wave-uniform; the kernel has no block barrier
  const int nchunks = H / 8;
  uint4 hreg[TT][NCH];
  uint4 wv[EPW][NCH];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) {
    const uint4* h4 =
        reinterpret_cast<const uint4*>(hidden + static_cast<size_t>(min(t0 + tt, T - 1)) * H);
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = lane + SF_WAVE * i;
      hreg[tt][i] = c < nchunks ? h4[c] : make_uint4(0, 0, 0, 0);
    }
  }
#pragma unroll
  for (int g = 0; g < EPW; ++g) {
    const uint4* w4 = reinterpret_cast<const uint4*>(wr + static_cast<size_t>(min(e0 + g, E - 1)) * H);
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = lane + SF_WAVE * i;
      wv[g][i] = c < nchunks ? w4[c] : make_uint4(0, 0, 0, 0);
    }
  }
  float acc[TT][EPW];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int g = 0; g < EPW; ++g) {
      acc[tt][g] = 0.0f;
#pragma unroll
      for (int i = 0; i < NCH; ++i)
        if (lane + SF_WAVE * i < nchunks) acc[tt][g] = dot8_acc(hreg[tt][i], wv[g][i], acc[tt][g]);
    }
  // Lane tt*EPW + g stores logit (t0+tt, e0+g).
  float a = 0.0f;
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int g = 0; g < EPW; ++g) {
      const float total = sf_wave_sum(acc[tt][g]);
      if (lane == tt * EPW + g) a = total;
    }
  const int t = t0 + lane / EPW;
  const int e = e0 + lane % EPW;
  if (lane < TT * EPW && t < T && e < E)
    logits[static_cast<size_t>(t) * E + e] = sf_f32_to_bf16(a);
}

// Many tokens: a wavefront takes 8 tokens x 8 experts, so a chunk's 16 loads
// and 128 unpacking instructions serve 512 multiply-adds (the 2 x 4 tile
// above: 6 loads and 48 for 64), and the 64 sums of the tile go through one
// transposed butterfly: at distance d a lane keeps the half of its sums whose
// index has the lane's bit d and adds the partner's copy of those (about 3
// instructions a logit instead of 11), ending with logit l of the tile in
// lane l.  Every addition has the same two operands as in sf_wave_sum, so the
// bits are the same.  Bound by the vector ALU (2048 of its 2754 instructions
// per tile are the multiply-adds of H = 2048).  Any H of whole chunk rounds
// (512 elements).
// Taken where its tiles fill the chip, from 40960 logits on up to H = 4096 and
// from 32768 above.  Both kernels of the call, small / large tile, us: E = 128,
// H = 1024, T = 256: 9.2 / 9.7, 384: 10.7 / 9.8, 2048: 26.2 / 16.7; H = 2048, T =
// 256: 13.1 / 12.9, 512: 19.6 / 13.1, 2048: 53.3 / 24.4; H = 4096, T = 256: 19.1
// / 19.1, 384: 25.5 / 19.4, 2048: 94.9 / 40.6; H = 6144, T = 256: 33.8 / 25.2.
// E = 256, T = 128: H = 1024: 10.8 / 11.3, 4096: 19.9 / 20.4, 8192: 40.7 / 36.3;
// E = 8 (three of a workgroup's four wavefronts idle), T = 4096: H = 1024: 9.8 /
// 9.9, 4096: 21.2 / 20.7, T = 16384: 24.3 / 20.6, 64.6 / 44.4.
constexpr int kManyTile = 8;  // tokens and experts of a wavefront

long long many_logits(int hidden_size) { return hidden_size <= 4096 ? 40960 : 32768; }

template <int CTRL>
__device__ __forceinline__ float butterfly_pair(float even, float odd, bool bit) {
  const float keep = bit ? odd : even;
  const float send = bit ? even : odd;
  return keep + sf_dpp<CTRL>(send);
}

__device__ __forceinline__ float unpack_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float unpack_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

__global__ __launch_bounds__(kLogitWaves * SF_WAVE, 2) void router_logits_many_kernel(
    const uint16_t* __restrict__ hidden, const uint16_t* __restrict__ wr, int T, int H, int E,
    uint16_t* __restrict__ logits) {
  const int lane = threadIdx.x & (SF_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / SF_WAVE);
  const int t0 = blockIdx.x * kManyTile;
  const int e0 = (blockIdx.y * kLogitWaves + wave) * kManyTile;
  if (e0 >= E) return;  // wave-uniform; the kernel has no block barrier
  uint32_t ho[kManyTile], wo[kManyTile];  // byte offsets: T H and E H stay below 2^31
#pragma unroll
  for (int i = 0; i < kManyTile; ++i) {
    ho[i] = 2u * min(t0 + i, T - 1) * H + 16 * lane;
    wo[i] = 2u * min(e0 + i, E - 1) * H + 16 * lane;
  }
  router_u32x4 h[kManyTile], w[kManyTile];
  auto load = [&](int k) {  // the lane's chunk at element k + 8 lane of every row
#pragma unroll
    for (int i = 0; i < kManyTile; ++i) {
      h[i] = router_ld16(hidden + k, ho[i]);
      w[i] = router_ld16(wr + k, wo[i]);
    }
  };
  float acc[kManyTile * kManyTile];
#pragma unroll
  for (int v = 0; v < kManyTile * kManyTile; ++v) acc[v] = 0.0f;
  constexpr int kStep = 8 * SF_WAVE;
  load(0);
  for (int k = 0; k < H; k += kStep) {
    router_u32x4 hc[kManyTile], wc[kManyTile];
#pragma unroll
    for (int i = 0; i < kManyTile; ++i) {
      hc[i] = h[i];
      wc[i] = w[i];
    }
    load(min(k + kStep, H - kStep));
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        float hf[kManyTile], wf[kManyTile];
#pragma unroll
        for (int i = 0; i < kManyTile; ++i) {
          hf[i] = half ? unpack_hi(hc[i][q]) : unpack_lo(hc[i][q]);
          wf[i] = half ? unpack_hi(wc[i][q]) : unpack_lo(wc[i][q]);
        }
#pragma unroll
        for (int t = 0; t < kManyTile; ++t)
#pragma unroll
          for (int e = 0; e < kManyTile; ++e)
            acc[kManyTile * t + e] = __builtin_fmaf(hf[t], wf[e], acc[kManyTile * t + e]);
      }
    }
  }
  // Distances 1, 2, 4, 8, 16, 32 over sum-index bits 0 .. 5.
#pragma unroll
  for (int p = 0; p < 32; ++p) acc[p] = butterfly_pair<0xB1>(acc[2 * p], acc[2 * p + 1], lane & 1);
#pragma unroll
  for (int p = 0; p < 16; ++p) acc[p] = butterfly_pair<0x4E>(acc[2 * p], acc[2 * p + 1], lane & 2);
#pragma unroll
  for (int p = 0; p < 8; ++p) {  // lane ^ 4 = the half-row mirror (^ 7) of ^ 3
    const bool bit = lane & 4;
    const float keep = bit ? acc[2 * p + 1] : acc[2 * p];
    const float send = bit ? acc[2 * p] : acc[2 * p + 1];
    acc[p] = keep + sf_dpp<0x141>(sf_dpp<0x1B>(send));
  }
#pragma unroll
  for (int p = 0; p < 4; ++p) acc[p] = butterfly_pair<0x128>(acc[2 * p], acc[2 * p + 1], lane & 8);
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const auto r = __builtin_amdgcn_permlane16_swap(
        __float_as_int(acc[2 * p]), __float_as_int(acc[2 * p + 1]), false, false);
    acc[p] = __int_as_float(r[0]) + __int_as_float(r[1]);
  }
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(acc[0]), __float_as_int(acc[1]),
                                                  false, false);
  const float total = __int_as_float(r[0]) + __int_as_float(r[1]);
  const int t = t0 + lane / kManyTile;
  const int e = e0 + lane % kManyTile;
  if (t < T && e < E) logits[static_cast<size_t>(t) * E + e] = sf_f32_to_bf16(total);
}

constexpr int kSelectWaves = 4;

template <int J>  // experts per lane: E <= 64 * J
__global__ __launch_bounds__(kSelectWaves * SF_WAVE) void router_select_kernel(
    const uint16_t* __restrict__ logits, int T, int E, int K, int renorm,
    uint16_t* __restrict__ topw, int64_t* __restrict__ topi) {
  __shared__ float s_logit[kSelectWaves][SF_MAX_EXPERTS];
  const int lane = threadIdx.x & (SF_WAVE - 1);
  const int wave = threadIdx.x / SF_WAVE;
  const int t = blockIdx.x * kSelectWaves + wave;
  if (t >= T) return;  // wave-uniform; the kernel has no block barrier
  // Lane l writes and later reads only experts l, l+64, ...: no barrier.
  for (int e = lane; e < E; e += SF_WAVE)
    s_logit[wave][e] = sf_bf16_to_f32(logits[static_cast<size_t>(t) * E + e]);
  softmax_topk_wave<J>(s_logit[wave], E, K, renorm, topw + static_cast<size_t>(t) * K,
                       topi + static_cast<size_t>(t) * K);
}

// Scalar path for any hidden_size / alignment: same summation order.
__global__ __launch_bounds__(kRouterThreads) void router_topk_scalar_kernel(
    const uint16_t* __restrict__ hidden, const uint16_t* __restrict__ wr, int H,
    int E, int K, int renorm, uint16_t* __restrict__ logits,
    uint16_t* __restrict__ topw, int64_t* __restrict__ topi) {
  __shared__ float s_logit[SF_MAX_EXPERTS];
  const int t = blockIdx.x;
  const int lane = threadIdx.x & (SF_WAVE - 1);
  const int wave = threadIdx.x / SF_WAVE;
  const int nchunks = (H + 7) / 8;
  const uint16_t* h = hidden + static_cast<size_t>(t) * H;
  for (int e = wave; e < E; e += kRouterWaves) {
    const uint16_t* w = wr + static_cast<size_t>(e) * H;
    float acc = 0.0f;
    for (int c = lane; c < nchunks; c += SF_WAVE) {
      for (int j = 0; j < 8; ++j) {
        int k = c * 8 + j;
        if (k < H) acc = __builtin_fmaf(sf_bf16_to_f32(h[k]), sf_bf16_to_f32(w[k]), acc);
      }
    }
    acc = sf_wave_sum(acc);
    if (lane == 0) {
      uint16_t b = sf_f32_to_bf16(acc);
      logits[static_cast<size_t>(t) * E + e] = b;
      s_logit[e] = sf_bf16_to_f32(b);
    }
  }
  __syncthreads();
  if (wave == 0)
    softmax_topk_wave<SF_MAX_EXPERTS / SF_WAVE>(s_logit, E, K, renorm,
                                                topw + static_cast<size_t>(t) * K,
                                                topi + static_cast<size_t>(t) * K);
}

}  // namespace

extern "C" int sf_router_topk(const void* hidden, const void* router_weight,
                              int tokens, int hidden_size, int num_experts,
                              int top_k, int norm_topk_prob, void* logits,
                              void* topk_weights, int64_t* topk_index,
                              sf_stream_t stream) {
  if (tokens < 0 || hidden_size < 1 || num_experts < 1 ||
      num_experts > SF_MAX_EXPERTS || top_k < 1 || top_k > num_experts ||
      top_k > SF_MAX_TOPK)
    return SF_ERR_INVALID_ARGUMENT;
  if (tokens == 0) return SF_OK;
  if (!hidden || !router_weight || !logits || !topk_weights || !topk_index)
    return SF_ERR_INVALID_ARGUMENT;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const uint16_t* h = static_cast<const uint16_t*>(hidden);
  const uint16_t* w = static_cast<const uint16_t*>(router_weight);
  uint16_t* lg = static_cast<uint16_t*>(logits);
  uint16_t* tw = static_cast<uint16_t*>(topk_weights);
  const bool aligned = (reinterpret_cast<uintptr_t>(hidden) % 16 == 0) &&
                       (reinterpret_cast<uintptr_t>(router_weight) % 16 == 0) &&
                       (hidden_size % 8 == 0);
  const int nchunks = (hidden_size + 7) / 8;
  const int per_lane = (nchunks + SF_WAVE - 1) / SF_WAVE;
  const bool many = aligned && hidden_size % (8 * SF_WAVE) == 0 &&
                    static_cast<long long>(tokens) * num_experts >= many_logits(hidden_size) &&
                    static_cast<long long>(tokens) * hidden_size < (1ll << 31) &&
                    static_cast<long long>(num_experts) * hidden_size < (1ll << 31);
  if (aligned && (many || per_lane <= 16)) {
    int tt = 1, epw = 1;
    auto logits_launch = [&](auto kernel, int tile_tokens, int tile_experts) {
      tt = tile_tokens;
      epw = tile_experts;
      const int per_block = kLogitWaves * epw;
      dim3 grid((tokens + tt - 1) / tt, (num_experts + per_block - 1) / per_block);
      kernel<<<grid, dim3(kLogitWaves * SF_WAVE), 0, s>>>(h, w, tokens, hidden_size, num_experts, lg);
    };
    if (many)
      logits_launch(router_logits_many_kernel, kManyTile, kManyTile);
    else if (per_lane <= 1)
      logits_launch(router_logits_kernel<1>, LogitTile<1>::tokens, LogitTile<1>::experts);
    else if (per_lane <= 2)
      logits_launch(router_logits_kernel<2>, LogitTile<2>::tokens, LogitTile<2>::experts);
    else if (per_lane <= 4)
      logits_launch(router_logits_kernel<4>, LogitTile<4>::tokens, LogitTile<4>::experts);
    else if (per_lane <= 8)
      logits_launch(router_logits_kernel<8>, LogitTile<8>::tokens, LogitTile<8>::experts);
    else
      logits_launch(router_logits_kernel<16>, LogitTile<16>::tokens, LogitTile<16>::experts);
    SF_LAUNCH_CHECK();
    // Experts per lane of the select wavefront: dead slots (e >= E) add +0
    // to the lane sums and are never selected, so J only trims the loops.
    const dim3 sgrid((tokens + kSelectWaves - 1) / kSelectWaves), sblock(kSelectWaves * SF_WAVE);
    if (num_experts <= SF_WAVE)
      router_select_kernel<1><<<sgrid, sblock, 0, s>>>(lg, tokens, num_experts, top_k,
                                                       norm_topk_prob, tw, topk_index);
    else if (num_experts <= 2 * SF_WAVE)
      router_select_kernel<2><<<sgrid, sblock, 0, s>>>(lg, tokens, num_experts, top_k,
                                                       norm_topk_prob, tw, topk_index);
    else
      router_select_kernel<SF_MAX_EXPERTS / SF_WAVE><<<sgrid, sblock, 0, s>>>(
          lg, tokens, num_experts, top_k, norm_topk_prob, tw, topk_index);
  } else {
    router_topk_scalar_kernel<<<dim3(tokens), dim3(kRouterThreads), 0, s>>>(
        h, w, hidden_size, num_experts, top_k, norm_topk_prob, lg, tw, topk_index);
  }
  SF_LAUNCH_CHECK();
  return SF_OK;
}
