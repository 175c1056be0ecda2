// FP16 MFMA GEMM with fused bias / exact-erf GELU epilogue for gfx950.
//
//   C[M, N] = epi(A[M, K] . W[N, K]^T + bias[N])
//
// W is nn.Linear's [out_features, in_features] layout, so both operands are
// K-contiguous: every lane feeds v_mfma_f32_16x16x32_f16 with one 16-byte
// LDS read per operand fragment.  The reference instead transposes weights to
// [K, N] for Triton's tl.dot (torch_transformer_benchmark.py:540-566) and
// computes GELU with tanh (triton_fused_ffn.py:198-213); the baseline it must
// match uses exact erf (torch_transformer_benchmark.py:286), as done here.
//
// Three kernels:
//  * gemm_dma_kernel (K % 64 == 0, K >= 256): 64 x 64 up to 256 x 256 tiles,
//    direct global -> LDS loads; used for the D >= 256 projections and FFN.
//  * gemm_rows_kernel (M <= 32, K % 32 == 0, N % 16 == 0): decode steps.
//  * gemm_nt_kernel (any K % 8 == 0): 4 waves in a 2 x 2 grid, tiles of A and
//    W go global -> registers -> padded LDS, double buffered; the epilogue
//    stages the FP16 tile through LDS so the stores to C are full 16-byte row
//    segments.
// Accumulators stay in VGPRs (the library builds this file with
// -amdgpu-mfma-vgpr-form): with AGPR accumulators the register allocator
// rotates accumulator tuples through copies on every loop iteration.
#include <cstdint>

#include "common.h"
#include "../../include/xblock.h"

namespace xb {

constexpr int kGemmBK = 64;
constexpr int kGemmLDK = kGemmBK + 8;  // padded LDS row (halves): 144 bytes

// Tile coordinates of the direct-to-LDS kernel: tiles are ordered in bands of
// 1024 rows (four row blocks of 256), column by column inside a band, and
// each XCD takes a contiguous range of that order (xcd_contiguous_tile).  One
// round of 32 256 x 256 tiles on an XCD then covers 4 row blocks x 8 column
// blocks instead of 2 x 16 (row-major), which for the QKV projection (N =
// 3072) reads 5 MB of distinct operands per round instead of 7 MB through
// that XCD's 4 MB L2, and the next round keeps the same A rows.  Measured,
// outputs bitwise equal: 3.2M x 3072 x 1024 (256 x 256) 20.9 -> 19.6 ms, 3.2M
// x 1024 x 1024 7.23 -> 7.08 ms; lower tiles with the same band height
// instead of four row blocks: 65536 x 3072 x 1024 (128 x 192) 438 -> 419 us,
// 65536 x 2304 x 768 (64 x 64) 405 -> 368 us.
template <int BM>
__device__ __forceinline__ void banded_tile(int tile, int tiles_m, int tiles_n, int& tm, int& tn) {
  constexpr int kBandRows = 1024 / BM;
  const int band = tile / (kBandRows * tiles_n);
  const int l = tile - band * kBandRows * tiles_n;
  const int rows = min(kBandRows, tiles_m - band * kBandRows);  // the last band may be shorter
  tm = band * kBandRows + l % rows;
  tn = l / rows;
}

// FP32 -> FP16 of an epilogue value, rounded once from the FP32 value.  The
// empty asm pins the FP32 result: otherwise the backend may fold the last
// multiply or add into a singly-rounded v_fma_mix conversion in some tile
// instantiations and not others, and the FP16 output would then depend on
// the tile (hence on the batch size that selected it).
__device__ __forceinline__ half_t to_half_pinned(float v) {
  asm volatile("" : "+v"(v));
  return (half_t)v;
}

template <int BM, int BN, int WGM, int WGN, int EPI>
__global__ __launch_bounds__(64 * WGM * WGN, 1) void gemm_nt_kernel(
    const half_t* __restrict__ A, const half_t* __restrict__ W,
    const float* __restrict__ bias, half_t* __restrict__ C, int M, int N,
    int K, int tiles_n) {
  constexpr int NT = 64 * WGM * WGN;  // threads
  constexpr int BK = kGemmBK, LDK = kGemmLDK;
  constexpr int WM = BM / WGM, WN = BN / WGN;  // wave tile
  constexpr int FM = WM / 16, FN = WN / 16;
  constexpr int CPR = BK / 8;  // 16-byte chunks per tile row
  constexpr int A_CH = BM * CPR / NT, B_CH = BN * CPR / NT;
  static_assert(A_CH * NT == BM * CPR && B_CH * NT == BN * CPR, "tile/thread mismatch");
  constexpr int LDC = BN + 8;
  static_assert(BM * LDC <= 2 * (BM + BN) * LDK, "epilogue staging must fit");
  __shared__ __attribute__((aligned(16))) half_t smem[2 * (BM + BN) * LDK];

  const int tile = xcd_contiguous_tile(blockIdx.x, gridDim.x);
  const int m0 = (tile / tiles_n) * BM, n0 = (tile % tiles_n) * BN;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;

  half8_t ra[A_CH], rb[B_CH];
  const half8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  auto gload = [&](int k0) {
#pragma unroll
    for (int j = 0; j < A_CH; ++j) {
      const int id = tid + NT * j, r = id / CPR, c = id % CPR;
      const int gm = m0 + r, gk = k0 + c * 8;
      ra[j] = (gm < M && gk < K) ? *reinterpret_cast<const half8_t*>(A + (int64_t)gm * K + gk) : zero8;
    }
#pragma unroll
    for (int j = 0; j < B_CH; ++j) {
      const int id = tid + NT * j, r = id / CPR, c = id % CPR;
      const int gn = n0 + r, gk = k0 + c * 8;
      rb[j] = (gn < N && gk < K) ? *reinterpret_cast<const half8_t*>(W + (int64_t)gn * K + gk) : zero8;
    }
  };
  auto sstore = [&](int buf) {
    half_t* as = smem + buf * (BM + BN) * LDK;
    half_t* bs = as + BM * LDK;
#pragma unroll
    for (int j = 0; j < A_CH; ++j) {
      const int id = tid + NT * j;
      *reinterpret_cast<half8_t*>(as + (id / CPR) * LDK + (id % CPR) * 8) = ra[j];
    }
#pragma unroll
    for (int j = 0; j < B_CH; ++j) {
      const int id = tid + NT * j;
      *reinterpret_cast<half8_t*>(bs + (id / CPR) * LDK + (id % CPR) * 8) = rb[j];
    }
  };

  float4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  const int KT = (K + BK - 1) / BK;
  gload(0);
  sstore(0);
  __syncthreads();
  for (int kt = 0; kt < KT; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < KT) gload((kt + 1) * BK);
    const half_t* as = smem + cur * (BM + BN) * LDK;
    const half_t* bs = as + BM * LDK;
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      half8_t af[FM], bf[FN];
      const int koff = ks * 32 + (lane / 16) * 8;
#pragma unroll
      for (int i = 0; i < FM; ++i)
        af[i] = *reinterpret_cast<const half8_t*>(as + (wm + 16 * i + lane % 16) * LDK + koff);
#pragma unroll
      for (int j = 0; j < FN; ++j)
        bf[j] = *reinterpret_cast<const half8_t*>(bs + (wn + 16 * j + lane % 16) * LDK + koff);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = mfma16x16x32(af[i], bf[j], acc[i][j]);
    }
    if (kt + 1 < KT) sstore(cur ^ 1);
    __syncthreads();
  }

  // Epilogue: bias (+ GELU) in FP32, FP16 tile staged in LDS, 16-byte stores.
  half_t* cs = smem;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int c = wn + 16 * j + lane % 16;
    const float bv = (bias != nullptr && n0 + c < N) ? bias[n0 + c] : 0.f;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = acc[i][j][e] + bv;
        if constexpr (EPI == XB_EPI_BIAS_GELU) v = gelu_erf(v);
        cs[(wm + 16 * i + (lane / 16) * 4 + e) * LDC + c] = to_half_pinned(v);
      }
  }
  __syncthreads();
  constexpr int CCH = BM * (BN / 8) / NT;
#pragma unroll
  for (int j = 0; j < CCH; ++j) {
    const int id = tid + NT * j, r = id / (BN / 8), c = (id % (BN / 8)) * 8;
    const int gm = m0 + r, gn = n0 + c;
    if (gm < M && gn < N)
      *reinterpret_cast<half8_t*>(C + (int64_t)gm * N + gn) = *reinterpret_cast<const half8_t*>(cs + r * LDC + c);
  }
}

// ---------------------------------------------------------------------------
// Large-tile kernel for K % 64 == 0.  Up to 8 waves share a BM x BN
// tile; each wave owns a (BM/WGM) x (BN/WGN) sub-tile with its FP32
// accumulators in VGPRs.  Operands reach LDS by direct global -> LDS loads
// (global_load_lds_dwordx4), one 64-wide K slab at a time, in a ring of ST
// slab stages: slab kt+ST is requested as soon as every wave has read slab
// kt, so ST-1 slabs are in flight while one is consumed.
//
// What is left over is each tile's start (the first slab's latency) and end
// (the output stores), which nothing hides while a CU holds one tile: for
// 8192 x 3072 x 1024 time against K put 17 of 55 us there.  So the library
// chooses, below 256 x 256, tiles of which a CU runs two and more, one
// starting or storing while another multiplies: 128 x 192 and 128 x 128 by
// eight waves (123 and 98 registers, 80 and 64 KB of LDS; two blocks) and 64 x
// 64 (by eight waves with three stages, 43 registers and 48 KB: three blocks;
// by four waves with two stages, 64 registers: five).  8192 x 3072 x 1024 54.5
// -> 50.2 us (256 x 192 by one block -> two of 128 x 192), 3001 x 3072 x 1024
// 26.1 -> 23.2 us, 8192 x 1024 x 1024 21.0 -> 19.4 us (128 x 128 by four waves
// -> by eight).  128 x 256 (151 registers, 96 KB: one block) runs only when a
// caller asks for it.
//
// LDS slab layout: the A rows (BM) and then the W rows (BN), 128 bytes each
// (64 halves = eight 16-byte chunks).  Chunk c of row r lives at slot
// c ^ (r & 7), so the 8 rows one 8-lane phase of ds_read_b128 touches land in
// 8 distinct 16-byte bank groups.  A DMA load writes lane i's 16 bytes to
// consecutive LDS addresses, so the swizzle is applied on the global side:
// lane i of a 1 KB segment (8 rows) fetches the chunk that belongs in its slot.


// s_waitcnt with vmcnt <= N and lgkmcnt == 0 (gfx9 field layout:
// vmcnt[3:0], expcnt[6:4], lgkmcnt[11:8], vmcnt_hi[15:14]).
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | ((N >> 4) << 14));
}

// Workgroup barrier that orders this wave's memory operations in the compiler
// without the vmcnt(0) a release fence would add.
__device__ __forceinline__ void slab_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The same with this wave's LDS writes completed first: the barrier alone does
// not wait for them (nor does the compiler, for this target), so a wave could
// read what another wave's write in flight has not yet put there.
__device__ __forceinline__ void lds_slab_barrier() {
  __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));  // vmcnt(63) expcnt(7) lgkmcnt(0)
  slab_barrier();
}

__device__ __forceinline__ int row128_offset(int r, int c) { return r * 128 + ((c ^ (r & 7)) << 4); }

// V of a packed QKV projection written transposed per head for the long-
// sequence attention: vt[b][h][d][p] with rows of `row` = seq_len rounded up
// to 64 elements, the positions p of each 32-token group in the attention's
// key order (token 32t + 4g + i at 32t + 8g + i, token 32t + 16 + 4g + i at
// 32t + 8g + 4 + i), so one 16-byte LDS read there is one operand fragment.
// Positions seq_len .. row-1 hold zeros.  Columns from v_col0 on are V.
struct VtOut {
  half_t* vt;
  int64_t row;
  int seq_len, head_dim, heads, v_col0;
};

template <int BM, int BN, int WGM, int WGN, int EPI, int ST, bool VT = false>
__global__ __launch_bounds__(64 * WGM * WGN, 1) void gemm_dma_kernel(
    const half_t* __restrict__ A, const half_t* __restrict__ W,
    const float* __restrict__ bias, half_t* __restrict__ C, int M, int N,
    int K, int tiles_n, VtOut vo) {
  constexpr int NW = WGM * WGN;
  constexpr int WM = BM / WGM, WN = BN / WGN, FM = WM / 16, FN = WN / 16;
  constexpr int SLAB = (BM + BN) * 128;        // 64-wide K slab, 128-byte rows
  constexpr int SEGS = (BM + BN) / 8;          // 1 KB wave-loads per slab (8 rows)
  constexpr int SPW = SEGS / NW;
  static_assert(SEGS % NW == 0 && WM % 16 == 0 && WN % 16 == 0, "tile shape");
  static_assert(ST >= 2 && ST * SLAB <= 160 * 1024 && (ST - 1) * SPW < 64, "slab ring");
  __shared__ __attribute__((aligned(1024))) char smem[ST * SLAB];
  int tile_m, tile_n;
  banded_tile<BM>(xcd_contiguous_tile(blockIdx.x, gridDim.x), gridDim.x / tiles_n, tiles_n, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;
  const half_t* src[SPW];
#pragma unroll
  for (int j = 0; j < SPW; ++j) {
    const int r = (wave + NW * j) * 8 + lane / 8;
    const int c = (lane % 8) ^ (r & 7);
    src[j] = r < BM ? A + (int64_t)min(m0 + r, M - 1) * K + 8 * c
                    : W + (int64_t)min(n0 + r - BM, N - 1) * K + 8 * c;
  }
  auto issue = [&](int kt, int stage) {
#pragma unroll
    for (int j = 0; j < SPW; ++j)
      __builtin_amdgcn_global_load_lds((global_void_t*)(src[j] + kt * 64),
                                       (lds_void_t*)(smem + stage * SLAB + (wave + NW * j) * 1024), 16, 0, 0);
  };
  float4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  const int KT = K / 64;
  auto read_frags = [&](int stage, int ks, half8_t (&af)[FM], half8_t (&bf)[FN]) {
    const char* st = smem + stage * SLAB;
    const int q = ks * 4 + lane / 16;
#pragma unroll
    for (int j = 0; j < FN; ++j)
      bf[j] = *reinterpret_cast<const half8_t*>(st + row128_offset(BM + wn + 16 * j + lane % 16, q));
#pragma unroll
    for (int i = 0; i < FM; ++i)
      af[i] = *reinterpret_cast<const half8_t*>(st + row128_offset(wm + 16 * i + lane % 16, q));
  };
  auto mma = [&](const half8_t (&af)[FM], const half8_t (&bf)[FN]) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = mfma16x16x32(bf[j], af[i], acc[i][j]);
  };
  // Slab kt: sub-step 0 reads sub-step 1's fragments of the same slab while
  // its own MFMAs run; sub-step 1 waits for slab kt+1 (leaving the ST-2 slabs
  // after it in flight), refills slab kt's stage with slab kt+ST and reads
  // slab kt+1's first fragments.  vmcnt retires loads in issue order, so
  // "at most (ST-2)*SPW outstanding" means slab kt+1 has landed.
  half8_t a0[FM], b0[FN], a1[FM], b1[FN];
#pragma unroll
  for (int s = 0; s < ST; ++s)
    if (s < KT) issue(s, s);
  if (KT >= ST) wait_vm_lgkm0<(ST - 1) * SPW>(); else wait_vm_lgkm0<0>();
  slab_barrier();
  read_frags(0, 0, a0, b0);
  int stage = 0;  // stage of slab kt
  for (int kt = 0; kt < KT; ++kt) {
    const int next = stage + 1 == ST ? 0 : stage + 1;
    __builtin_amdgcn_sched_barrier(0);
    read_frags(stage, 1, a1, b1);
    __builtin_amdgcn_sched_barrier(0);
    mma(a0, b0);
    __builtin_amdgcn_sched_barrier(0);
    if (kt + 1 < KT) {
      if (kt + ST - 1 < KT) wait_vm_lgkm0<(ST - 2) * SPW>(); else wait_vm_lgkm0<0>();
      slab_barrier();
      if (kt + ST < KT) issue(kt + ST, stage);
      read_frags(next, 0, a0, b0);
    } else {
      wait_vm_lgkm0<0>();
    }
    __builtin_amdgcn_sched_barrier(0);
    mma(a1, b1);
    stage = next;
  }

  // Epilogue: bias (+ GELU) in FP32, the FP16 tile staged in LDS (free once
  // every wave has read the last slab), then written out in 16-byte row
  // chunks, a wave covering whole rows: lane-sized row pieces of 8 bytes
  // scattered over 16 rows per store made the stores a fifth of the time.
  // Chunk k of tile row r sits at chunk k ^ (r & SW) of its LDS row, which
  // keeps both the 8-byte fragment writes and the 16-byte reads spread over
  // the banks.
  constexpr int CPR = BN / 8;                       // 16-byte chunks per tile row
  constexpr int SW = CPR % 16 == 0 ? 15 : 7;
  static_assert(BM * BN * 2 <= ST * SLAB, "the C tile fits in the slab stages");
  slab_barrier();
  if constexpr (VT) {
    if (n0 >= vo.v_col0) {  // a V tile (the host checked v_col0 % BN == 0, seq_len % 32 == 0)
      static_assert(BM % 32 == 0, "whole 32-token groups per tile");
      // Staged feature-major, [BN][BM], positions in key order, then written
      // as whole 16-byte chunks of the transposed rows.
      half_t* vs = reinterpret_cast<half_t*>(smem);
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = wn + 16 * j + (lane / 16) * 4;
        float b[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = bias != nullptr ? bias[n0 + col + e] : 0.f;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const int r = wm + 16 * i + lane % 16;
          const int p = (r & ~31) | (((r & 15) >> 2) << 3) | (((r >> 4) & 1) << 2) | (r & 3);
#pragma unroll
          for (int e = 0; e < 4; ++e) vs[(col + e) * BM + p] = to_half_pinned(acc[i][j][e] + b[e]);
        }
      }
      lds_slab_barrier();
      constexpr int NT = 64 * NW, CPF = BM / 8;  // 16-byte chunks per staged feature row
      static_assert((BN * CPF) % NT == 0, "whole rounds of chunks");
#pragma unroll
      for (int id0 = 0; id0 < BN * CPF; id0 += NT) {
        const int id = id0 + (int)threadIdx.x;
        const int f = id / CPF, c = id % CPF;
        const int m = m0 + 32 * (c / 4);  // first token of the chunk's 32-token group
        if (m < M) {
          const int bq = m / vo.seq_len, sq = m - bq * vo.seq_len;
          const int n = n0 + f - vo.v_col0;
          const int h = n / vo.head_dim, d = n - h * vo.head_dim;
          half_t* dst = vo.vt + ((int64_t)(bq * vo.heads + h) * vo.head_dim + d) * vo.row + sq + 8 * (c % 4);
          *reinterpret_cast<half8_t*>(dst) = *reinterpret_cast<const half8_t*>(vs + f * BM + 8 * c);
          if (sq + 32 == vo.seq_len && c % 4 == 0) {  // the sequence's last group: zero the row's padding
            for (int64_t z = vo.seq_len; z < vo.row; z += 8)
              *reinterpret_cast<half8_t*>(dst - sq + z) = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
          }
        }
      }
      return;
    }
  }
  half_t* cs = reinterpret_cast<half_t*>(smem);
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int col = wn + 16 * j + (lane / 16) * 4;  // tile column of this lane's 4 values
    float b[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias != nullptr && n0 + col < N) {
#pragma unroll
      for (int e = 0; e < 4; ++e) b[e] = bias[n0 + col + e];
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int row = wm + 16 * i + lane % 16;
      half4_t h;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = acc[i][j][e] + b[e];
        if constexpr (EPI == XB_EPI_BIAS_GELU) v = gelu_erf(v);
        h[e] = to_half_pinned(v);
      }
      *reinterpret_cast<half4_t*>(cs + row * BN + 8 * ((col / 8) ^ (row & SW)) + (col & 7)) = h;
    }
  }
  lds_slab_barrier();
  constexpr int NT = 64 * NW;
  static_assert((BM * CPR) % NT == 0, "whole rounds of 16-byte chunks");
#pragma unroll
  for (int id0 = 0; id0 < BM * CPR; id0 += NT) {
    const int id = id0 + (int)threadIdx.x;
    const int row = id / CPR, k = id % CPR;
    const int gm = m0 + row, gn = n0 + 8 * k;
    if (gm < M && gn < N)
      *reinterpret_cast<half8_t*>(C + (int64_t)gm * N + gn) =
          *reinterpret_cast<const half8_t*>(cs + row * BN + 8 * (k ^ (row & SW)));
  }
}

// ---------------------------------------------------------------------------
// Few-row kernel (M <= 32: decode steps, short prompts).  The product is then
// a single pass over the weights, so what counts is how many CUs pull them
// and how much each has in flight: a 128 x 128 tile at M = 4 put N = 1024 on
// 8 CUs, each waiting on one slab at a time (13 us).  Here a block owns 16
// output columns and its waves split K, 256 of it each, so the block's whole
// weight slab (and the activations) is requested in the first instructions,
// straight into registers.  The partial sums are not added up: wave w starts
// its products from wave w - 1's accumulator (handed over in LDS), which
// keeps one chain over K per output, the same products in the same order and
// so the same bits as every other tile; a row's result does not depend on how
// many rows are in the call.  Row groups of 16 follow each other down the
// chain.
constexpr int kRowsMax = 32, kRowsSteps = 8, kRowsMaxK = 16 * kRowsSteps * 32;

//
// CH > 0 (xb_norm_linear, M <= 8, K = 256 CH): the activations are LN(x +
// upd), computed here by every block, a row per wave at a time in
// ln_rows_kernel's order (the same bits), while the weights are on their way;
// block 0 also writes x + upd.  A decode step's LayerNorms were launches of
// 4.4 us for a few KB.  KV columns also go to the caches, which saves the
// append's launch.
struct RowsExtra {
  const float* x;          // [M, K] residual stream; not res_out (every block reads it)
  const half_t* upd;       // [M, K] or NULL
  const float *gamma, *beta;
  float* res_out;          // x + upd, or NULL
  float eps;
  int affine;
  half_t *k_cache, *v_cache;  // NULL: none; N = 3D then
  int heads, head_dim, chunk; // M = batch * chunk
  int64_t start, capacity;
};
constexpr int kNormRowsMax = 8;

template <int RG, int EPI, int CH>
__global__ __launch_bounds__(1024) void gemm_rows_kernel(
    const half_t* __restrict__ A, const half_t* __restrict__ W,
    const float* __restrict__ bias, half_t* __restrict__ C, int M, int N, int K, RowsExtra ex) {
  __shared__ float4_t hand[16][RG][kWave];
  constexpr int LDN = CH * 256 + 8;
  __shared__ __attribute__((aligned(16))) half_t normed[CH > 0 ? kNormRowsMax * LDN : 8];
  const int lane = threadIdx.x % kWave, g = lane / 16, r16 = lane % 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int waves = blockDim.x / kWave;
  const int n0 = blockIdx.x * 16;
  const int steps = min(kRowsSteps, K / 32 - wave * kRowsSteps);  // >= 1: waves = ceil(K / 256)
  const half_t* wrow = W + (int64_t)(n0 + r16) * K + wave * (kRowsSteps * 32) + 8 * g;
  const half_t* arow = A + wave * (kRowsSteps * 32) + 8 * g;
  half8_t wf[kRowsSteps], af[RG][kRowsSteps];
  // Steps past the end repeat the last one's loads and are not multiplied.
  auto load_a = [&](int rg) {
    const half_t* p = arow + (int64_t)min(16 * rg + r16, M - 1) * K;
#pragma unroll
    for (int s = 0; s < kRowsSteps; ++s) af[rg][s] = *reinterpret_cast<const half8_t*>(p + 32 * min(s, steps - 1));
  };
#pragma unroll
  for (int s = 0; s < kRowsSteps; ++s) wf[s] = *reinterpret_cast<const half8_t*>(wrow + 32 * min(s, steps - 1));
  if constexpr (CH == 0) {
    load_a(0);
    if constexpr (RG > 1) load_a(1);
  } else {
    constexpr int D = CH * 256;
    for (int row = wave; row < M; row += waves) {
      float v[CH][4];
      float4_t gm[CH], bt[CH];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int col = (c * kWave + lane) * 4;
        const float4_t x4 = *reinterpret_cast<const float4_t*>(ex.x + (int64_t)row * D + col);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[c][i] = x4[i];
        if (ex.upd != nullptr) {
          const half4_t u = *reinterpret_cast<const half4_t*>(ex.upd + (int64_t)row * D + col);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[c][i] += (float)u[i];
        }
        if (ex.affine) {
          gm[c] = *reinterpret_cast<const float4_t*>(ex.gamma + col);
          bt[c] = *reinterpret_cast<const float4_t*>(ex.beta + col);
        }
      }
      if (ex.res_out != nullptr && blockIdx.x == 0) {
#pragma unroll
        for (int c = 0; c < CH; ++c)
          *reinterpret_cast<float4_t*>(ex.res_out + (int64_t)row * D + (c * kWave + lane) * 4) =
              float4_t{v[c][0], v[c][1], v[c][2], v[c][3]};
      }
      float s = 0.f;
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) s += v[c][i];
      const float mean = group_sum<kWave>(s) * (1.0f / D);
      float q = 0.f;
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[c][i] -= mean;
          q += v[c][i] * v[c][i];
        }
      const float rstd = rsqrtf(group_sum<kWave>(q) * (1.0f / D) + ex.eps);
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        half4_t h;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          h[i] = (half_t)(ex.affine ? v[c][i] * rstd * gm[c][i] + bt[c][i] : v[c][i] * rstd);
        *reinterpret_cast<half4_t*>(normed + row * LDN + (c * kWave + lane) * 4) = h;
      }
    }
    lds_slab_barrier();
    const half_t* p = normed + min(r16, M - 1) * LDN + wave * (kRowsSteps * 32) + 8 * g;
#pragma unroll
    for (int st = 0; st < kRowsSteps; ++st) af[0][st] = *reinterpret_cast<const half8_t*>(p + 32 * st);
  }
  float b[4] = {0.f, 0.f, 0.f, 0.f};
  if (wave == waves - 1 && bias != nullptr) {
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = bias[n0 + 4 * g + e];
  }
  // Every wave passes waves + RG - 1 barriers; row group rg is at wave w
  // between the barriers w + rg and w + rg + 1.
  for (int i = 0; i < wave; ++i) lds_slab_barrier();
#pragma unroll
  for (int rg = 0; rg < RG; ++rg) {
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    if (wave > 0) acc = hand[wave - 1][rg][lane];
#pragma unroll
    for (int s = 0; s < kRowsSteps; ++s)
      if (s < steps) acc = mfma16x16x32(wf[s], af[rg][s], acc);
    if (wave + 1 < waves) {
      hand[wave][rg][lane] = acc;
    } else if (16 * rg + r16 < M) {  // lane: row r16, columns 4g .. 4g + 3
      half4_t h;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = acc[e] + b[e];
        if constexpr (EPI == XB_EPI_BIAS_GELU) v = gelu_erf(v);
        h[e] = to_half_pinned(v);
      }
      *reinterpret_cast<half4_t*>(C + (int64_t)(16 * rg + r16) * N + n0 + 4 * g) = h;
      if constexpr (CH > 0) {
        if (ex.k_cache != nullptr && n0 >= K) {  // K = D here: a block is all Q, all K or all V
          const int col = (n0 - K) % K + 4 * g;
          const int64_t row = 16 * rg + r16, bt = row / ex.chunk, t = row - bt * ex.chunk;
          const int head = col / ex.head_dim, d = col - head * ex.head_dim;
          half_t* cache = n0 < 2 * K ? ex.k_cache : ex.v_cache;
          *reinterpret_cast<half4_t*>(cache + ((bt * ex.heads + head) * ex.capacity + ex.start + t) * ex.head_dim + d) = h;
        }
      }
    }
    lds_slab_barrier();
  }
  for (int i = wave + 1; i < waves; ++i) lds_slab_barrier();
}

template <int EPI>
static hipError_t launch_gemm_rows(const half_t* a, const half_t* w, const float* bias, half_t* c,
                                   int64_t m, int n, int k, hipStream_t s) {
  const dim3 grid((unsigned)(n / 16)), block((unsigned)(kWave * ((k + 255) / 256)));
  const int rows = (int)m;
  if (m <= 16) hipLaunchKernelGGL((gemm_rows_kernel<1, EPI, 0>), grid, block, 0, s, a, w, bias, c, rows, n, k, RowsExtra{});
  else hipLaunchKernelGGL((gemm_rows_kernel<2, EPI, 0>), grid, block, 0, s, a, w, bias, c, rows, n, k, RowsExtra{});
  return hipGetLastError();
}

template <int EPI>
static hipError_t launch_norm_rows(const RowsExtra& ex, const half_t* w, const float* bias, half_t* c, int m, int n,
                                   int k, hipStream_t s) {
  const dim3 grid((unsigned)(n / 16)), block((unsigned)(kWave * (k / 256)));
  switch (k / 256) {
    case 2: hipLaunchKernelGGL((gemm_rows_kernel<1, EPI, 2>), grid, block, 0, s, nullptr, w, bias, c, m, n, k, ex); break;
    case 3: hipLaunchKernelGGL((gemm_rows_kernel<1, EPI, 3>), grid, block, 0, s, nullptr, w, bias, c, m, n, k, ex); break;
    case 4: hipLaunchKernelGGL((gemm_rows_kernel<1, EPI, 4>), grid, block, 0, s, nullptr, w, bias, c, m, n, k, ex); break;
    default: hipLaunchKernelGGL((gemm_rows_kernel<1, EPI, 8>), grid, block, 0, s, nullptr, w, bias, c, m, n, k, ex); break;
  }
  return hipGetLastError();
}

// Widths whose LayerNorm ln_rows_kernel reduces over 64 lanes of 4 columns.
static bool norm_rows_fit(int64_t m, int n, int k) {
  return m <= kNormRowsMax && n % 16 == 0 && (k == 512 || k == 768 || k == 1024 || k == 2048);
}

template <int BM, int BN, int WGM, int WGN, int EPI, int ST, bool VT = false>
static hipError_t launch_gemm_dma(const half_t* a, const half_t* w, const float* bias, half_t* c,
                                  int64_t m, int n, int k, hipStream_t s, VtOut vo = {}) {
  const int64_t tm = (m + BM - 1) / BM, tn = (n + BN - 1) / BN;
  if (tm * tn > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((gemm_dma_kernel<BM, BN, WGM, WGN, EPI, ST, VT>), dim3((unsigned)(tm * tn)),
                     dim3(64 * WGM * WGN), 0, s, a, w, bias, c, (int)m, n, k, (int)tn, vo);
  return hipGetLastError();
}

template <int BM, int BN, int WGM, int WGN, int EPI>
static hipError_t launch_gemm(const half_t* a, const half_t* w, const float* bias, half_t* c,
                              int64_t m, int n, int k, hipStream_t s) {
  const int64_t tm = (m + BM - 1) / BM, tn = (n + BN - 1) / BN;
  if (tm * tn > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((gemm_nt_kernel<BM, BN, WGM, WGN, EPI>), dim3((unsigned)(tm * tn)),
                     dim3(64 * WGM * WGN), 0, s, a, w, bias, c, (int)m, n, k, (int)tn);
  return hipGetLastError();
}

// Variants (XB_LINEAR_*): the gemm_dma_kernel tiles need K % 64 == 0 and K >=
// 256 (256 x 192, a pair of 128 x 192 blocks on a CU, also N % 192 == 0); the
// gemm_nt_kernel tiles take any K % 8 == 0; gemm_rows_kernel a few rows.
static bool linear_variant_fits(int variant, int64_t m, int n, int k) {
  const bool dma = k % 64 == 0 && k >= 256;
  switch (variant) {
    case XB_LINEAR_DMA_256x256: case XB_LINEAR_DMA_128x256: case XB_LINEAR_DMA_128x128:
    case XB_LINEAR_DMA_64x64: return dma;
    case XB_LINEAR_DMA_256x192: return dma && n % 192 == 0;
    case XB_LINEAR_NT_128x128: case XB_LINEAR_NT_64x64: return true;
    case XB_LINEAR_ROWS: return m <= kRowsMax && n % 16 == 0 && k % 32 == 0 && k <= kRowsMaxK;
    default: return false;
  }
}

// The library's choice for a shape.  Up to kRowsMax rows the few-row kernel is
// the faster one at every N and K it takes.  A DMA tile costs rounds of one
// tile per CU, r = ceil(tiles / 256), times what a tile costs a busy CU; the
// microseconds below are at K = 1024 (all of them grow with K alike) and
// reproduce a sweep over 777 to 65536 rows, N 512 to 4096, K 512 to 4096 to
// within 10 %, or pick a tile within 10 % of its best.  64 x 64 tiles read the
// most operand bytes per output but start and end in the least time and are
// the only ones with a block for every CU at a few hundred rows (1500 x 1024:
// 8.2 us against 13.1 with 128 x 128); 128 x 192 pairs (XB_LINEAR_DMA_256x192)
// are the cheapest per output up to 16384 rows, 256 x 256 beyond.
static int select_linear(int64_t m, int n, int k) {
  if (linear_variant_fits(XB_LINEAR_ROWS, m, n, k)) return XB_LINEAR_ROWS;
  auto tiles = [&](int64_t bm, int64_t bn) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); };
  auto rounds = [&](int64_t bm, int64_t bn) { return (double)((tiles(bm, bn) + 255) / 256); };
  if (k % 64 == 0 && k >= 256) {
    const double big = 32.0 * rounds(256, 256) - 1.0;
    const double wide = n % 192 == 0 ? 12.0 * rounds(128, 192) : 1e30;
    const double mid = 8.6 * rounds(128, 128) + 2.5;
    const double small = 3.1 * rounds(64, 64) + 1.5;
    if (big <= wide && big <= mid && big <= small) return XB_LINEAR_DMA_256x256;
    if (wide <= mid && wide <= small) return XB_LINEAR_DMA_256x192;
    return mid <= small ? XB_LINEAR_DMA_128x128 : XB_LINEAR_DMA_64x64;
  }
  return tiles(128, 128) >= 512 ? XB_LINEAR_NT_128x128 : XB_LINEAR_NT_64x64;
}

// 64 x 64 tiles: two slabs ahead (a ring of three) where the grid is at most a
// round, or two with a long K -- the operands of such a product are too much
// for the L2s and its blocks too few to hide each other's misses (1500 x 768 x
// 3072 24.2 -> 20.3 us, 777 x 1024 x 4096 30.4 -> 19.6) -- else a ring of two,
// which lets five blocks share a CU (8192 x 1024 x 1024 28.1 against 25.8 us).
template <int EPI>
static hipError_t launch_gemm_64(const half_t* a, const half_t* w, const float* bias, half_t* c,
                                 int64_t m, int n, int k, hipStream_t s) {
  const int64_t tiles = ((m + 63) / 64) * ((n + 63) / 64);
  if (tiles <= 256 || (tiles <= 512 && k >= 2048)) return launch_gemm_dma<64, 64, 4, 2, EPI, 3>(a, w, bias, c, m, n, k, s);
  return launch_gemm_dma<64, 64, 2, 2, EPI, 2>(a, w, bias, c, m, n, k, s);
}

template <int EPI>
static hipError_t run_gemm(int variant, const half_t* a, const half_t* w, const float* bias, half_t* c,
                           int64_t m, int n, int k, hipStream_t s) {
  switch (variant) {
    case XB_LINEAR_DMA_256x256: return launch_gemm_dma<256, 256, 2, 4, EPI, 2>(a, w, bias, c, m, n, k, s);
    case XB_LINEAR_DMA_256x192: return launch_gemm_dma<128, 192, 2, 4, EPI, 2>(a, w, bias, c, m, n, k, s);  // two per CU
    case XB_LINEAR_DMA_128x256: return launch_gemm_dma<128, 256, 2, 4, EPI, 2>(a, w, bias, c, m, n, k, s);
    case XB_LINEAR_DMA_128x128: return launch_gemm_dma<128, 128, 2, 4, EPI, 2>(a, w, bias, c, m, n, k, s);
    case XB_LINEAR_DMA_64x64: return launch_gemm_64<EPI>(a, w, bias, c, m, n, k, s);
    case XB_LINEAR_NT_128x128: return launch_gemm<128, 128, 2, 2, EPI>(a, w, bias, c, m, n, k, s);
    case XB_LINEAR_ROWS: return launch_gemm_rows<EPI>(a, w, bias, c, m, n, k, s);
    default: return launch_gemm<64, 64, 2, 2, EPI>(a, w, bias, c, m, n, k, s);
  }
}

}  // namespace xb

using namespace xb;

static int check_linear(int64_t m, int32_t n, int32_t k, int epilogue) {
  if (m < 0 || n <= 0 || k <= 0 || m > 0x7fffffffLL) return XB_ERR_BAD_SIZE;
  if (n % 8 != 0 || k % 8 != 0) return XB_ERR_UNSUPPORTED_SHAPE;
  if (epilogue != XB_EPI_BIAS && epilogue != XB_EPI_BIAS_GELU) return XB_ERR_BAD_EPILOGUE;
  return XB_OK;
}

extern "C" int xb_select_linear(int64_t m, int32_t n, int32_t k, int epilogue) {
  const int bad = check_linear(m, n, k, epilogue);
  return bad ? bad : select_linear(m, n, k);
}

extern "C" int xb_linear_v(const void* a, const void* w, const float* bias, void* c, int64_t m, int32_t n,
                           int32_t k, int epilogue, int variant, void* stream) {
  const int bad = check_linear(m, n, k, epilogue);
  if (bad) return bad;
  if (variant == XB_VARIANT_AUTO) variant = select_linear(m, n, k);
  if (!linear_variant_fits(variant, m, n, k)) return XB_ERR_BAD_VARIANT;
  if (m == 0) return XB_OK;  // empty tensors may carry NULL data pointers
  if (!a || !w || !c) return XB_ERR_NULL_POINTER;
  if (((uintptr_t)a | (uintptr_t)w | (uintptr_t)c) & 15u) return XB_ERR_MISALIGNED;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const half_t* A = static_cast<const half_t*>(a);
  const half_t* Wt = static_cast<const half_t*>(w);
  half_t* Cc = static_cast<half_t*>(c);
  hipError_t e = epilogue == XB_EPI_BIAS_GELU
      ? run_gemm<XB_EPI_BIAS_GELU>(variant, A, Wt, bias, Cc, m, n, k, s)
      : run_gemm<XB_EPI_BIAS>(variant, A, Wt, bias, Cc, m, n, k, s);
  return (int)e;
}

extern "C" int xb_linear(const void* a, const void* w, const float* bias, void* c,
                         int64_t m, int32_t n, int32_t k, int epilogue, void* stream) {
  return xb_linear_v(a, w, bias, c, m, n, k, epilogue, XB_VARIANT_AUTO, stream);
}

extern "C" int64_t xb_vt_row_stride(int64_t seq_len) { return seq_len <= 0 ? 0 : (seq_len + 63) / 64 * 64; }

extern "C" int xb_linear_qkv_vt(const void* a, const void* w, const float* bias, void* qkv, void* vt,
                                int32_t batch, int64_t seq_len, int32_t heads, int32_t head_dim, int32_t k,
                                int variant, void* stream) {
  if (batch < 0 || seq_len < 0 || heads <= 0 || head_dim <= 0 || k <= 0) return XB_ERR_BAD_SIZE;
  const int64_t m = (int64_t)batch * seq_len;
  const int64_t d = (int64_t)heads * head_dim;
  if (m > 0x7fffffffLL || 3 * d > 0x7fffffffLL) return XB_ERR_BAD_SIZE;
  const int n = (int)(3 * d);
  if (seq_len % 32 != 0 || head_dim % 8 != 0 || k % 64 != 0 || k < 256) return XB_ERR_UNSUPPORTED_SHAPE;
  if (variant == XB_VARIANT_AUTO) {
    variant = select_linear(m, n, k);
    if (variant == XB_LINEAR_DMA_256x192) variant = XB_LINEAR_DMA_256x256;
    if (variant != XB_LINEAR_DMA_256x256 || d % 256 != 0) variant = XB_LINEAR_DMA_128x128;
  }
  int bn = 0;
  switch (variant) {
    case XB_LINEAR_DMA_256x256: case XB_LINEAR_DMA_128x256: bn = 256; break;
    case XB_LINEAR_DMA_128x128: bn = 128; break;
    default: return XB_ERR_BAD_VARIANT;  // the V boundary must fall between DMA tiles
  }
  if (d % bn != 0) return XB_ERR_BAD_VARIANT;  // every tile is all Q/K or all V
  if (m == 0) return XB_OK;
  if (!a || !w || !qkv || !vt) return XB_ERR_NULL_POINTER;
  if (((uintptr_t)a | (uintptr_t)w | (uintptr_t)qkv | (uintptr_t)vt) & 15u) return XB_ERR_MISALIGNED;
  const VtOut vo{static_cast<half_t*>(vt), xb_vt_row_stride(seq_len), (int)seq_len, head_dim, heads, (int)(2 * d)};
  const half_t* A = static_cast<const half_t*>(a);
  const half_t* Wt = static_cast<const half_t*>(w);
  half_t* Cc = static_cast<half_t*>(qkv);
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipError_t e;
  switch (variant) {
    case XB_LINEAR_DMA_256x256:
      e = launch_gemm_dma<256, 256, 2, 4, XB_EPI_BIAS, 2, true>(A, Wt, bias, Cc, m, n, k, s, vo); break;
    case XB_LINEAR_DMA_128x256:
      e = launch_gemm_dma<128, 256, 2, 4, XB_EPI_BIAS, 2, true>(A, Wt, bias, Cc, m, n, k, s, vo); break;
    default:
      e = launch_gemm_dma<128, 128, 2, 4, XB_EPI_BIAS, 2, true>(A, Wt, bias, Cc, m, n, k, s, vo); break;
  }
  return (int)e;
}

extern "C" int xb_select_norm_linear(int64_t rows, int32_t n, int32_t k) {
  if (rows < 0 || n <= 0 || k <= 0) return XB_ERR_BAD_SIZE;
  return norm_rows_fit(rows, n, k) ? XB_OK : XB_ERR_UNSUPPORTED_SHAPE;
}

extern "C" int xb_norm_linear(const float* residual, const void* update, const float* gamma, const float* beta,
                              float eps, int apply_affine, float* residual_out, const void* w, const float* bias,
                              void* c, int64_t rows, int32_t n, int32_t k, int epilogue, void* k_cache, void* v_cache,
                              int32_t heads, int64_t chunk, int64_t start, int64_t capacity, void* stream) {
  if (rows < 0 || n <= 0 || k <= 0) return XB_ERR_BAD_SIZE;
  if (epilogue != XB_EPI_BIAS && epilogue != XB_EPI_BIAS_GELU) return XB_ERR_BAD_EPILOGUE;
  if (!norm_rows_fit(rows, n, k)) return XB_ERR_UNSUPPORTED_SHAPE;
  const bool caches = k_cache != nullptr || v_cache != nullptr;
  if (caches) {
    if (n != 3 * k || heads <= 0 || k % heads != 0 || (k / heads) % 8 != 0) return XB_ERR_UNSUPPORTED_SHAPE;
    if (chunk <= 0 || rows % chunk != 0 || start < 0 || start + chunk > capacity) return XB_ERR_BAD_SIZE;
  }
  if (rows == 0) return XB_OK;
  if (!residual || !w || !c || (apply_affine && (!gamma || !beta))) return XB_ERR_NULL_POINTER;
  if (caches && (!k_cache || !v_cache)) return XB_ERR_NULL_POINTER;
  if (residual_out == residual) return XB_ERR_BAD_SIZE;  // other blocks still read it
  uintptr_t all = (uintptr_t)residual | (uintptr_t)update | (uintptr_t)residual_out | (uintptr_t)w | (uintptr_t)c |
                  (uintptr_t)k_cache | (uintptr_t)v_cache;
  if (apply_affine) all |= (uintptr_t)gamma | (uintptr_t)beta;
  if (all & 15u) return XB_ERR_MISALIGNED;
  const RowsExtra ex{residual, static_cast<const half_t*>(update), gamma, beta, residual_out, eps, apply_affine,
                     static_cast<half_t*>(k_cache), static_cast<half_t*>(v_cache), heads,
                     caches ? k / heads : 0, caches ? (int)chunk : 1, start, capacity};
  const half_t* Wt = static_cast<const half_t*>(w);
  half_t* Cc = static_cast<half_t*>(c);
  hipStream_t s = static_cast<hipStream_t>(stream);
  return (int)(epilogue == XB_EPI_BIAS_GELU
      ? launch_norm_rows<XB_EPI_BIAS_GELU>(ex, Wt, bias, Cc, (int)rows, n, k, s)
      : launch_norm_rows<XB_EPI_BIAS>(ex, Wt, bias, Cc, (int)rows, n, k, s));
}
