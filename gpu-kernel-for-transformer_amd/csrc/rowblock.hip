// Everything of a layer except its attention, in one kernel, for narrow models
// (d_model 32, 64 or 128, ffn_dim a small multiple of it, any length):
//
//   a = ctx Wo^T + bo; x += a; n2 = LN2(x); x += gelu_erf(n2 W1^T + b1) W2^T + b2;
//   n1 = LN1 of the next layer (x); q, k, v = n1 Wqkv^T + b of the next layer
//
// (torch_transformer_benchmark.py:1112-1148 from one attention to the next).
// The first launch of a forward does only LN1 + QKV, the last one ends with the
// final LayerNorm instead.  At these widths each of the five kernels this
// replaces reads and writes whole activations around a few microseconds of
// matrix work, so it is bound by memory traffic and, on small batches, by the
// number of launches; here a token's row stays in registers from the context
// to the next projection and HBM sees ctx, x (in and out) and q, k, v only:
// 16 D bytes per token instead of 44 D.  65536 tokens of width 128: 93 -> 34 us
// per layer (4.0 TB/s; the reads come first and the writes last in every block,
// and one round of blocks fills the chip, so they overlap little); the 32-wide
// model's 29 launches become 9.
//
// Layout.  A wave owns NBT blocks of 16 tokens and all features; products are
// out^T = W . act^T, whose C layout (lane: token l % 16, features 16 fb + 4 (l
// / 16) + i) is read back as the next product's operand with the reduction
// index 32 ks + 4 (l / 16) + (m & 3) + 16 (m >> 2), so nothing but the weights
// (fragment-major, xb_pack_linear_fragments in that order) goes through LDS.
// A token's result does not depend on the block, wave or lane that holds it.
//
// Weights, in groups of one D x D matrix (Wo, then W1 and W2 in D-wide pieces
// of ffn_dim, then Wq, Wk, Wv), arrive by direct global -> LDS loads.  Below
// width 128 all groups fit: they are requested at once and waited for once.
// At 128 (32 KB a group) they go through a ring of four stages, three groups
// ahead; the waits count the loads and stores issued since (memory operations
// of a wave retire in order), so no group waits for the output stores before it.
#include <type_traits>

#include "common.h"
#include "../../include/xblock.h"

namespace xb {
namespace rowblock {

enum Mode { kFirst, kMid, kLast };
constexpr int kRing = 4;          // stages at D = 128
constexpr int kMaxChunksNarrow = 4;  // ffn_dim / D below 128
constexpr int kMaxChunksWide = 8;    // at 128

struct Args {
  const float* res_in;          // residual stream before this layer's attention update (kFirst: x)
  const half_t* ctx;            // attention context
  float* res_out;               // kMid; never res_in
  half_t* qkv;                  // [rows, 3D] (kFirst, kMid)
  float* y;                     // kLast
  const uint8_t* row_valid;     // kLast, may be NULL
  const half_t *w, *w_next;     // packed Wq Wk Wv Wo W1 W2 of this and of the next layer
  const float *bo, *b1, *b2, *g2, *be2;
  const float *g1, *be1, *bqkv; // the next layer's norm1 and QKV bias (kLast: the final LayerNorm)
  float eps2, eps1;
  int64_t rows;
  int chunks;                   // ffn_dim / D
};

// Mean and 1 / sqrt(var + eps) of each token block's rows (lanes l, l ^ 16, l ^ 32, l ^ 48 share a row).
template <int D, int NBT>
__device__ __forceinline__ void stats(const float4_t (&r)[NBT][D / 16], float eps, float (&mean)[NBT], float (&rstd)[NBT]) {
#pragma unroll
  for (int b = 0; b < NBT; ++b) {
    float s = 0.f;
#pragma unroll
    for (int fb = 0; fb < D / 16; ++fb) s += (r[b][fb][0] + r[b][fb][1]) + (r[b][fb][2] + r[b][fb][3]);
    mean[b] = quad_group_sum(s) * (1.0f / D);
    float q = 0.f;
#pragma unroll
    for (int fb = 0; fb < D / 16; ++fb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float c = r[b][fb][i] - mean[b];
        q += c * c;
      }
    rstd[b] = rsqrtf(quad_group_sum(q) * (1.0f / D) + eps);
  }
}

__device__ __forceinline__ float4_t lds4(const float* p) { return *reinterpret_cast<const float4_t*>(p); }

// LayerNorm of each token block -> operands.
template <int D, int NBT>
__device__ __forceinline__ void norm_operands(const float4_t (&r)[NBT][D / 16], float eps, const float* gamma,
                                              const float* beta, int g, half8_t (&xn)[NBT][D / 32]) {
  float mean[NBT], rstd[NBT];
  stats<D, NBT>(r, eps, mean, rstd);
#pragma unroll
  for (int fb = 0; fb < D / 16; ++fb) {
    const float4_t gg = lds4(gamma + 16 * fb + 4 * g), bb = lds4(beta + 16 * fb + 4 * g);
#pragma unroll
    for (int b = 0; b < NBT; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        xn[b][fb / 2][4 * (fb & 1) + i] = (half_t)((r[b][fb][i] - mean[b]) * rstd[b] * gg[i] + bb[i]);
  }
}

// a[b][ob] += W . act^T over the staged D x D matrix.
template <int D, int NBT>
__device__ __forceinline__ void product(const char* st, const half8_t (&act)[NBT][D / 32], float4_t (&a)[NBT][D / 16],
                                        int lane) {
  constexpr int FB = D / 16, KS = D / 32;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    half8_t f[FB];
#pragma unroll
    for (int ob = 0; ob < FB; ++ob) f[ob] = *reinterpret_cast<const half8_t*>(st + (ob * KS + ks) * 1024 + lane * 16);
#pragma unroll
    for (int b = 0; b < NBT; ++b)
#pragma unroll
      for (int ob = 0; ob < FB; ++ob) a[b][ob] = mfma16x16x32(f[ob], act[b][ks], a[b][ob]);
  }
}

template <int N>
__device__ __forceinline__ void wait_vm() {  // vmcnt(N), other counters untouched
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Workgroup barrier after this wave's LDS accesses; memory operations stay in flight.
__device__ __forceinline__ void barrier() {
  __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int D, int NBT, int NW, int MODE, int MAXC>
__global__ __launch_bounds__(64 * NW, 1) void row_block_kernel(const Args p) {
  constexpr int FB = D / 16, KS = D / 32, FRAGS = FB * KS, GB = FRAGS * 1024;
  constexpr bool kRinged = D == 128;
  constexpr int kGroups = (MODE == kFirst ? 0 : 1 + 2 * MAXC) + (MODE == kLast ? 0 : 3);
  constexpr int kStages = kRinged ? kRing : kGroups;
  constexpr int FPW = kRinged ? FRAGS / NW : 0;         // ring: fragments each wave copies per group
  constexpr int CPR = D / 8, SPB = CPR / 4;             // 16-byte chunks per row; store instructions per token block
  constexpr int PRM = 9 * D + MAXC * D;
  static_assert(!kRinged || FRAGS % NW == 0, "whole fragments per wave");
  static_assert(kRing * FPW + 2 * NBT * SPB < 64, "countable");
  __shared__ __attribute__((aligned(1024))) char wst[kStages][GB];
  __shared__ __attribute__((aligned(16))) float prm[PRM];
  __shared__ __attribute__((aligned(16))) char stage_out[kRinged ? 16 : NW * 16 * D * 2];
  float* const s_bo = prm, *const s_b2 = prm + D, *const s_g2 = prm + 2 * D, *const s_be2 = prm + 3 * D;
  float* const s_g1 = prm + 4 * D, *const s_be1 = prm + 5 * D, *const s_bqkv = prm + 6 * D, *const s_b1 = prm + 9 * D;

  const int lane = threadIdx.x % kWave, g = lane / 16, r16 = lane % 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int chunks = p.chunks, ffn = chunks * D;
  const int g_qkv = MODE == kFirst ? 0 : 1 + 2 * chunks;
  const int groups = g_qkv + (MODE == kLast ? 0 : 3);

  // Tokens past the end repeat the last one (same values written twice), so
  // every wave issues the same memory operations.
  int64_t tok[NBT];
#pragma unroll
  for (int b = 0; b < NBT; ++b) {
    const int64_t t = ((int64_t)blockIdx.x * NW + wave) * (16 * NBT) + 16 * b + r16;
    tok[b] = t < p.rows ? t : p.rows - 1;
  }

  // Inputs first, then the per-layer vectors, then the weights.
  float4_t res[NBT][FB];
  half8_t act[NBT][KS];
#pragma unroll
  for (int b = 0; b < NBT; ++b)
#pragma unroll
    for (int fb = 0; fb < FB; ++fb) res[b][fb] = *reinterpret_cast<const float4_t*>(p.res_in + tok[b] * D + 16 * fb + 4 * g);
  if constexpr (MODE != kFirst) {
#pragma unroll
    for (int b = 0; b < NBT; ++b)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const half_t* c = p.ctx + tok[b] * D + 32 * ks + 4 * g;
        const half4_t lo = *reinterpret_cast<const half4_t*>(c), hi = *reinterpret_cast<const half4_t*>(c + 16);
        act[b][ks] = half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
  }
  {
    auto put = [&](float* dst, const float* src, int n) {
      for (int i = threadIdx.x; i < n; i += 64 * NW) dst[i] = src[i];
    };
    if constexpr (MODE != kFirst) {
      put(s_bo, p.bo, D);
      put(s_b2, p.b2, D);
      put(s_g2, p.g2, D);
      put(s_be2, p.be2, D);
      put(s_b1, p.b1, ffn);
    }
    put(s_g1, p.g1, D);
    put(s_be1, p.be1, D);
    if constexpr (MODE != kLast) put(s_bqkv, p.bqkv, 3 * D);
  }

  // Fragment f of group gi in the packed buffers.
  auto source = [&](int gi, int f) -> const half_t* {
    if (gi >= g_qkv) return p.w_next + ((int64_t)(gi - g_qkv) * FRAGS + f) * 512;
    const half_t* w = p.w + (int64_t)3 * FRAGS * 512;  // past Wq Wk Wv
    if (gi == 0) return w + (int64_t)f * 512;
    w += (int64_t)FRAGS * 512;
    const int c = (gi - 1) / 2;
    if (gi & 1) return w + ((int64_t)c * FRAGS + f) * 512;                    // W1: D rows from cD
    w += (int64_t)chunks * FRAGS * 512;
    return w + ((int64_t)(f / KS) * (ffn / 32) + c * KS + f % KS) * 512;      // W2: D columns from cD
  };
  auto issue = [&](int gi) {  // ring: this wave's share of group gi
#pragma unroll
    for (int j = 0; j < FPW; ++j) {
      const int f = wave + NW * j;
      dma16_untracked(source(gi, f) + lane * 8, wst[gi % kRing] + f * 1024);
    }
  };
  if constexpr (kRinged) {
#pragma unroll
    for (int i = 0; i < kRing; ++i)
      if (i < groups) issue(i);
  } else {
    for (int f = wave; f < groups * FRAGS; f += NW)
      dma16_untracked(source(f / FRAGS, f % FRAGS) + lane * 8, &wst[0][0] + f * 1024);
    wait_vm<0>();
    barrier();
  }
  // Start of group gi: its fragments are in LDS for every wave.  `stores`
  // output stores were issued after every load still awaited.
  auto begin = [&](int gi, auto stores) -> const char* {
    if constexpr (kRinged) {
      constexpr int S = decltype(stores)::value;
      const int newer = min(groups, gi < 1 ? kRing : gi + kRing - 1) - 1 - gi;  // groups requested after gi
      switch (newer) {
        case 0: wait_vm<S>(); break;
        case 1: wait_vm<S + FPW>(); break;
        case 2: wait_vm<S + 2 * FPW>(); break;
        default: wait_vm<S + 3 * FPW>(); break;
      }
      barrier();
      if (gi > 0 && gi + kRing - 1 < groups) issue(gi + kRing - 1);  // into group gi - 1's stage
      return wst[gi % kRing];
    } else {
      return wst[gi];
    }
  };
  constexpr std::integral_constant<int, 0> kNoStores{};
  auto start_at = [&](float4_t (&a)[NBT][FB], const float* bias) {
#pragma unroll
    for (int ob = 0; ob < FB; ++ob) {
      const float4_t v = lds4(bias + 16 * ob + 4 * g);
#pragma unroll
      for (int b = 0; b < NBT; ++b) a[b][ob] = v;
    }
  };

  if constexpr (MODE != kFirst) {
    {
      const char* st = begin(0, kNoStores);
      float4_t a[NBT][FB];
      start_at(a, s_bo);
      product<D, NBT>(st, act, a, lane);
#pragma unroll
      for (int b = 0; b < NBT; ++b)
#pragma unroll
        for (int ob = 0; ob < FB; ++ob) res[b][ob] += a[b][ob];
    }
    half8_t xn[NBT][KS];
    norm_operands<D, NBT>(res, p.eps2, s_g2, s_be2, g, xn);
#pragma unroll
    for (int ob = 0; ob < FB; ++ob) {  // the FFN's output bias; its products accumulate onto the residual
      const float4_t v = lds4(s_b2 + 16 * ob + 4 * g);
#pragma unroll
      for (int b = 0; b < NBT; ++b) res[b][ob] += v;
    }
    for (int c = 0; c < chunks; ++c) {
      half8_t hf[NBT][KS];
      {
        const char* st = begin(1 + 2 * c, kNoStores);
        float4_t a[NBT][FB];
        start_at(a, s_b1 + c * D);
        product<D, NBT>(st, xn, a, lane);
#pragma unroll
        for (int b = 0; b < NBT; ++b)
#pragma unroll
          for (int ob = 0; ob < FB; ++ob)
#pragma unroll
            for (int i = 0; i < 4; ++i) hf[b][ob / 2][4 * (ob & 1) + i] = (half_t)gelu_erf(a[b][ob][i]);
      }
      const char* st = begin(2 + 2 * c, kNoStores);
      product<D, NBT>(st, hf, res, lane);
    }
  }

  if constexpr (MODE == kLast) {
    float mean[NBT], rstd[NBT];
    stats<D, NBT>(res, p.eps1, mean, rstd);
#pragma unroll
    for (int b = 0; b < NBT; ++b) {
      const bool zero = p.row_valid != nullptr && p.row_valid[tok[b]] == 0;  // padded tokens leave as zero rows
#pragma unroll
      for (int fb = 0; fb < FB; ++fb) {
        const float4_t gg = lds4(s_g1 + 16 * fb + 4 * g), bb = lds4(s_be1 + 16 * fb + 4 * g);
        float4_t o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = zero ? 0.f : (res[b][fb][i] - mean[b]) * rstd[b] * gg[i] + bb[i];
        *reinterpret_cast<float4_t*>(p.y + tok[b] * D + 16 * fb + 4 * g) = o;
      }
    }
    return;
  } else {
    half8_t xn[NBT][KS];
    if constexpr (kRinged && MODE == kFirst) barrier();  // the vectors, stored by every wave, are in LDS
    norm_operands<D, NBT>(res, p.eps1, s_g1, s_be1, g, xn);
    // A projection's rows leave through this wave's own piece of LDS (ring:
    // of the stage before Q's, free by then) as whole-row 16-byte chunks;
    // chunk k of row r sits at k ^ (r mod CPR).
    char* const own = (kRinged ? wst[(g_qkv + kRing - 1) % kRing] : stage_out) + wave * (16 * D * 2);
    auto project = [&](auto which, auto stores) {
      constexpr int W = decltype(which)::value;
      const char* st = begin(g_qkv + W, stores);
      float4_t a[NBT][FB];
      start_at(a, s_bqkv + W * D);
      product<D, NBT>(st, xn, a, lane);
#pragma unroll
      for (int b = 0; b < NBT; ++b) {
#pragma unroll
        for (int ob = 0; ob < FB; ++ob) {
          half4_t h;
#pragma unroll
          for (int i = 0; i < 4; ++i) h[i] = (half_t)a[b][ob][i];
          *reinterpret_cast<half4_t*>(own + r16 * (D * 2) + 16 * ((2 * ob + g / 2) ^ (r16 % CPR)) + 8 * (g & 1)) = h;
        }
        const int64_t t0 = ((int64_t)blockIdx.x * NW + wave) * (16 * NBT) + 16 * b;
#pragma unroll
        for (int j = 0; j < SPB; ++j) {
          const int row = (j * kWave + lane) / CPR, k = lane % CPR;
          const int64_t t = t0 + row < p.rows ? t0 + row : p.rows - 1;
          *reinterpret_cast<half8_t*>(p.qkv + t * (3 * D) + W * D + 8 * k) =
              *reinterpret_cast<const half8_t*>(own + row * (D * 2) + 16 * (k ^ (row % CPR)));
        }
      }
    };
    project(std::integral_constant<int, 0>(), kNoStores);
    project(std::integral_constant<int, 1>(), std::integral_constant<int, NBT * SPB>());
    project(std::integral_constant<int, 2>(), std::integral_constant<int, 2 * NBT * SPB>());
    if constexpr (MODE == kMid) {
#pragma unroll
      for (int b = 0; b < NBT; ++b)
#pragma unroll
        for (int fb = 0; fb < FB; ++fb)
          *reinterpret_cast<float4_t*>(p.res_out + tok[b] * D + 16 * fb + 4 * g) = res[b][fb];
    }
  }
}

template <int D, int MAXC, int NBT, int NW>
static hipError_t launch(int mode, const Args& a, hipStream_t s) {
  const int64_t per = 16 * NBT * NW;
  const int64_t blocks = (a.rows + per - 1) / per;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)blocks), block(64 * NW);
  switch (mode) {
    case kFirst: hipLaunchKernelGGL((row_block_kernel<D, NBT, NW, kFirst, MAXC>), grid, block, 0, s, a); break;
    case kMid: hipLaunchKernelGGL((row_block_kernel<D, NBT, NW, kMid, MAXC>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((row_block_kernel<D, NBT, NW, kLast, MAXC>), grid, block, 0, s, a); break;
  }
  return hipGetLastError();
}

// Tokens per block: two blocks of 16 per wave halve the weight reads from LDS
// per product but need 32768 tokens to leave no CU idle, eight waves share the
// weight copies but need 16384.
template <int D, int MAXC>
static hipError_t launch_rows(int mode, const Args& a, hipStream_t s) {
  if (a.rows > 32768) return launch<D, MAXC, 2, 8>(mode, a, s);
  if (a.rows > 16384) return launch<D, MAXC, 1, 8>(mode, a, s);
  return launch<D, MAXC, 1, 4>(mode, a, s);
}

static bool supported(int d, int ffn) {
  if (ffn <= 0 || (d != 32 && d != 64 && d != 128) || ffn % d != 0) return false;
  return ffn / d <= (d == 128 ? kMaxChunksWide : kMaxChunksNarrow);
}

}  // namespace rowblock
}  // namespace xb

using namespace xb;

extern "C" int xb_select_row_block(int32_t d_model, int32_t ffn_dim) {
  if (d_model <= 0 || ffn_dim <= 0) return XB_ERR_BAD_SIZE;
  return rowblock::supported(d_model, ffn_dim) ? XB_OK : XB_ERR_UNSUPPORTED_SHAPE;
}

extern "C" int xb_row_block(const xb_stack* st, int32_t layer, const float* residual, const void* ctx,
                            float* residual_out, void* qkv, float* y, const uint8_t* row_valid, int64_t rows,
                            void* stream) {
  if (!st || rows < 0 || layer < -1 || layer >= st->layers || st->heads <= 0 || st->head_dim <= 0) return XB_ERR_BAD_SIZE;
  if (rows > 0x7fffffffLL) return XB_ERR_BAD_SIZE;
  const int d = st->heads * st->head_dim;
  if (!rowblock::supported(d, st->ffn_dim)) return XB_ERR_UNSUPPORTED_SHAPE;
  if (rows == 0) return XB_OK;
  const bool first = layer < 0, last = layer + 1 == st->layers;
  if (!st->blocks || !residual || (!first && !ctx)) return XB_ERR_NULL_POINTER;
  if (last ? !y : (!qkv || (!first && !residual_out))) return XB_ERR_NULL_POINTER;
  if (!last && !first && residual_out == residual) return XB_ERR_BAD_SIZE;  // rows are read again while others are written
  rowblock::Args a = {};
  a.res_in = residual;
  a.ctx = static_cast<const half_t*>(ctx);
  a.res_out = residual_out;
  a.qkv = static_cast<half_t*>(qkv);
  a.y = y;
  a.row_valid = row_valid;
  a.rows = rows;
  a.chunks = st->ffn_dim / d;
  uintptr_t all = (uintptr_t)residual | (uintptr_t)ctx | (uintptr_t)residual_out | (uintptr_t)qkv | (uintptr_t)y;
  if (!first) {
    const xb_block& b = st->blocks[layer];
    a.w = static_cast<const half_t*>(b.packed);
    a.bo = b.out_b;
    a.b1 = b.ffn_in_b;
    a.b2 = b.ffn_out_b;
    a.g2 = b.norm2_g;
    a.be2 = b.norm2_b;
    a.eps2 = b.norm2_eps;
    if (!a.w || !a.bo || !a.b1 || !a.b2 || !a.g2 || !a.be2) return XB_ERR_NULL_POINTER;
    all |= (uintptr_t)a.w;
  }
  if (last) {
    a.g1 = st->final_g;
    a.be1 = st->final_b;
    a.eps1 = st->final_eps;
  } else {
    const xb_block& n = st->blocks[layer + 1];
    a.w_next = static_cast<const half_t*>(n.packed);
    a.g1 = n.norm1_g;
    a.be1 = n.norm1_b;
    a.eps1 = n.norm1_eps;
    a.bqkv = n.qkv_b;
    if (!a.w_next || !a.bqkv) return XB_ERR_NULL_POINTER;
    all |= (uintptr_t)a.w_next;
  }
  if (!a.g1 || !a.be1) return XB_ERR_NULL_POINTER;
  if (all & 15u) return XB_ERR_MISALIGNED;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int mode = first ? rowblock::kFirst : last ? rowblock::kLast : rowblock::kMid;
  const bool one = a.chunks == 1;
  switch (d) {
    case 32: return (int)(one ? rowblock::launch_rows<32, 1>(mode, a, s)
                              : rowblock::launch_rows<32, rowblock::kMaxChunksNarrow>(mode, a, s));
    case 64: return (int)(one ? rowblock::launch_rows<64, 1>(mode, a, s)
                              : rowblock::launch_rows<64, rowblock::kMaxChunksNarrow>(mode, a, s));
    default: return (int)rowblock::launch_rows<128, rowblock::kMaxChunksWide>(mode, a, s);
  }
}
