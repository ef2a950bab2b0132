// Dense bf16 GEMM  C = A . B^T  (A [M,K], B [N,K], fp32 accumulate).
//
// Three shapes of work:
//  * M <= 8 ("GEMV", decode; to 16 where the next kernels do not apply):
//    HBM-bound on B.  The M activation rows are
//    staged once in LDS; each wave streams R rows of B with 16-byte
//    non-temporal loads (K/512 loads per row per lane, all in flight), and
//    reduces the per-lane partial dots with cross-lane shuffles.
//  * 9 <= M <= 64 (batched decode, from 2 rows at vocabulary-size N): the
//    weights stream through LDS past the rows, where that is ahead
//    (gemm_skinny_kernel: skinny_cols, gemm_slice_kernel: slice_ok,
//    gemm_vocab_kernel: vocab_ok).
//  * larger M: the direct-to-LDS MFMA pipelines (mfma_pipe.hpp; from 224
//    tiles of 256 x 256 on, the deep-staged 8-wave one of mfma_wide.hpp).
#include "decode_util.hpp"
#include "gemm.hpp"
#include "mfma_pipe.hpp"
#include "mfma_wide.hpp"
#include "norm_impl.hpp"

#include <hipblaslt/hipblaslt.h>

#include <map>
#include <mutex>
#include <tuple>

namespace qmoe {

template <int MODE>
__device__ __forceinline__ void store_out(void* C, int64_t idx, float v) {
  if constexpr (MODE == QMOE_GEMM_STORE_BF16) {
    reinterpret_cast<uint16_t*>(C)[idx] = f32_to_bf16(v);
  } else if constexpr (MODE == QMOE_GEMM_STORE_F32) {
    reinterpret_cast<float*>(C)[idx] = v;
  } else {
    reinterpret_cast<float*>(C)[idx] += v;
  }
}

// ------------------------------------------------------------------ GEMV
template <int MT, int R, int MODE>
__global__ __launch_bounds__(256) void gemv_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                   const uint16_t* __restrict__ B, int M, int N,
                                                   int K, void* __restrict__ C, int64_t ldc) {
  extern __shared__ __attribute__((aligned(16))) uint16_t xs[];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  // stage the M activation rows (16-byte chunks)
  const int kchunks = K / 8;
  stage16<256, 16>(reinterpret_cast<u32x4*>(xs), M * kchunks, [&](int c) {
    const int m = c / kchunks;
    return A + m * lda + (c - m * kchunks) * 8;
  });
  __syncthreads();

  const int n0 = (blockIdx.x * 4 + wave) * R;
  float acc[MT][R];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < R; ++r) acc[m][r] = 0.0f;

  const uint16_t* brow[R];
#pragma unroll
  for (int r = 0; r < R; ++r) brow[r] = B + int64_t(min(n0 + r, N - 1)) * K;

#pragma unroll 4
  for (int k = lane * 8; k < K; k += 512) {
    u32x4 w[R];
#pragma unroll
    for (int r = 0; r < R; ++r) w[r] = ld_stream(brow[r] + k);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (m < M) {
        const u32x4 xv = *reinterpret_cast<const u32x4*>(xs + m * K + k);
        float x8[8] = {bf16_lo(xv.x), bf16_hi(xv.x), bf16_lo(xv.y), bf16_hi(xv.y),
                       bf16_lo(xv.z), bf16_hi(xv.z), bf16_lo(xv.w), bf16_hi(xv.w)};
#pragma unroll
        for (int r = 0; r < R; ++r) acc[m][r] += dot8(w[r], x8);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (m < M) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float v = wave_sum(acc[m][r]);
        if (lane == 0 && n0 + r < N) store_out<MODE>(C, int64_t(m) * ldc + n0 + r, v);
      }
    }
  }
}

// GEMV for K = 512 * KC <= 4096: every weight load of a wave (R rows x KC
// 16-byte chunks per lane) is issued before the activation rows are staged,
// so the weight stream starts with the workgroup and all of it is in flight
// at once (R * KC <= 16 loads per lane).
template <int MT, int R, int KC, int MODE>
__global__ __launch_bounds__(256) void gemv_reg_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                       const uint16_t* __restrict__ B, int M, int N,
                                                       int K, void* __restrict__ C, int64_t ldc) {
  extern __shared__ __attribute__((aligned(16))) uint16_t xs[];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int n0 = (blockIdx.x * 4 + wave) * R;
  u32x4 w[R][KC];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint16_t* brow = B + int64_t(min(n0 + r, N - 1)) * K + lane * 8;
#pragma unroll
    for (int c = 0; c < KC; ++c) w[r][c] = ld_stream(brow + c * 512);
  }
  const int kchunks = K / 8;
  stage16<256, 16>(reinterpret_cast<u32x4*>(xs), M * kchunks, [&](int c) {
    const int m = c / kchunks;
    return A + m * lda + (c - m * kchunks) * 8;
  });
  __syncthreads();
  float acc[MT][R];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < R; ++r) acc[m][r] = 0.0f;
#pragma unroll
  for (int c = 0; c < KC; ++c) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (m < M) {
        const u32x4 xv = *reinterpret_cast<const u32x4*>(xs + m * K + c * 512 + lane * 8);
#pragma unroll
        for (int r = 0; r < R; ++r) acc[m][r] = dot8_bf16(w[r][c], xv, acc[m][r]);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (m < M) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float v = wave_sum(acc[m][r]);
        if (lane == 0 && n0 + r < N) store_out<MODE>(C, int64_t(m) * ldc + n0 + r, v);
      }
    }
  }
}

// Single-row GEMV with the input RMSNorm fused into the activation staging:
// x = bf16(w_rms * h * rsqrt(mean(h^2) + eps)) from the fp32 residual row h,
// with the same chunking, summation order and rounding as
// rmsnorm_residual_kernel (so x has the same bits), then the one-row-per-wave
// dot of gemv_reg_kernel.  Weight loads are issued first, so the norm's
// reduction overlaps the weight stream.
template <int KC, int MODE>
__global__ __launch_bounds__(256) void gemv_rms_kernel(const float* __restrict__ h,
                                                       const uint16_t* __restrict__ rms_w, float eps,
                                                       const uint16_t* __restrict__ B, int N,
                                                       void* __restrict__ C) {
  constexpr int K = KC * 512, NCH = K / 4 / 256 > 0 ? K / 4 / 256 : 1;  // float4 chunks per thread
  __shared__ __attribute__((aligned(16))) uint16_t xs[K];
  __shared__ float red[4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int n0 = blockIdx.x * 4 + wave;
  u32x4 w[KC];
  {
    const uint16_t* brow = B + int64_t(min(n0, N - 1)) * K + lane * 8;
#pragma unroll
    for (int c = 0; c < KC; ++c) w[c] = ld_stream(brow + c * 512);
  }
  float4 v[NCH];
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int c = t + j * 256;
    if (c < K / 4) {
      const float4 a = reinterpret_cast<const float4*>(h)[c];
      v[j] = a;
      ss += a.x * a.x + a.y * a.y + a.z * a.z + a.w * a.w;
    }
  }
  ss = wave_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  float tot = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) tot += red[i];
  const float r = rsqrtf(tot / float(K) + eps);
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int c = t + j * 256;
    if (c < K / 4) {
      const float4 a = v[j];
      const uint2 wv = reinterpret_cast<const uint2*>(rms_w)[c];
      uint2 o;
      o.x = pack_bf16x2(bf16_lo(wv.x) * (a.x * r), bf16_hi(wv.x) * (a.y * r));
      o.y = pack_bf16x2(bf16_lo(wv.y) * (a.z * r), bf16_hi(wv.y) * (a.w * r));
      reinterpret_cast<uint2*>(xs)[c] = o;
    }
  }
  __syncthreads();
  float acc = 0.0f;
#pragma unroll
  for (int c = 0; c < KC; ++c)
    acc = dot8_bf16(w[c], *reinterpret_cast<const u32x4*>(xs + c * 512 + lane * 8), acc);
  const float out = wave_sum(acc);
  if (lane == 0 && n0 < N) store_out<MODE>(C, n0, out);
}

// Skinny GEMM for 2 <= M <= 16 rows of A (batched decode), K = 128 * KS:
// v_mfma_f32_16x16x32_bf16 with the A rows padded to 16 (zeros past M).  A
// workgroup owns NB (8 or 16) output columns; wave w owns the K range
// [w*K/4, (w+1)*K/4): its KS B operands (16 bytes of a weight row each, lane
// l -> column l % 16, k offset (l / 16) * 8) are all loaded before A is
// staged (plain loads: a load touches half of each 128-byte line and the next
// one the other half, which the nontemporal form does not keep in L1; 3-4%
// faster), the KS MFMAs accumulate, and the four waves' 16x16 partials are
// added in wave order through LDS.  HBM-bound like the M = 1 GEMV: the
// arithmetic that makes dot-product GEMVs slow at M = 8 costs KS MFMAs here.
template <int NB, int KS, int MODE>
__global__ __launch_bounds__(256) void gemv_mfma_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                        const uint16_t* __restrict__ B, int M, int N,
                                                        int K, void* __restrict__ C, int64_t ldc) {
  extern __shared__ __attribute__((aligned(16))) uint16_t xs[];  // [M][K] bf16
  __shared__ float red[4][16][17];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int n0 = blockIdx.x * NB;
  const int col = lane & 15, kq = lane >> 4;
  const int kw = wave * (K / 4);
  u32x4 bw[KS];
  {
    const bool live = col < NB && n0 + col < N;
    const uint16_t* bp = B + int64_t(min(n0 + col, N - 1)) * K + kw + kq * 8;
#pragma unroll
    for (int s = 0; s < KS; ++s) bw[s] = live ? ld16(bp + s * 32) : u32x4{0u, 0u, 0u, 0u};
  }
  const int kchunks = K / 8;
  stage16<256, 16>(reinterpret_cast<u32x4*>(xs), M * kchunks, [&](int c) {
    const int m = c / kchunks;
    return A + m * lda + (c - m * kchunks) * 8;
  });
  __syncthreads();
  f32x4 acc = f32x4{};
  const uint16_t* ap = xs + min(col, M - 1) * K + kw + kq * 8;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const u32x4 a = col < M ? *reinterpret_cast<const u32x4*>(ap + s * 32) : u32x4{0u, 0u, 0u, 0u};
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                  __builtin_bit_cast(bf16x8, bw[s]), acc, 0, 0, 0);
  }
  // lane l holds column l % 16, rows (l / 16) * 4 + 0..3
#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][kq * 4 + i][col] = acc[i];
  __syncthreads();
  const int m = t >> 4, n = t & 15;
  if (m < M && n < NB && n0 + n < N) {
    const float v = ((red[0][m][n] + red[1][m][n]) + red[2][m][n]) + red[3][m][n];
    store_out<MODE>(C, int64_t(m) * ldc + n0 + n, v);
  }
}

// Skinny GEMM for 2 <= M <= 8 rows of A (batched decode) with the weights
// streamed through LDS: K = 512 * WAVES, wave w owns k in [512 w, 512 w +
// 512), a workgroup owns NB output columns (one workgroup per CU at the
// decode shapes: 20 for N = 5120, 8 for N = 2048).  Each wave copies its NB
// weight rows (1 KB each) into LDS with one non-temporal LDS-DMA per row (64
// lanes x 16 contiguous bytes: whole 128-byte lines, the access the one-row
// GEMV streams at), rows GV_ROWB = 1040 bytes apart so the 16 rows of an MFMA
// B fragment fall on distinct LDS banks.
// The A fragments come straight from global memory (the activation rows are
// L2-resident) and are loaded packed: the 16x16x32 MFMA has 16 A rows and
// only rows 0-7 are live, so lane (c, g) loads 8 k-values of row c % 8 at
// step 2p + c / 8 and a DPP rotation by 8 within each row of 16 lanes hands
// step 2p + 1 to lanes 0-7 (rows 8-15 of the product are never read).  Every
// lane's load is live: half the A load instructions of a zero-padded
// fragment, which is what an 8-row GEMV pays for (the A bytes per workgroup
// equal the weight bytes at 8 columns).  The waves' 8 x NB partials are added
// in k order through LDS.
constexpr int GV_ROWB = 1040;
template <int WAVES, int NB, int MODE>
__global__ __launch_bounds__(64 * WAVES) void gemv_pk_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                             const uint16_t* __restrict__ B, int M, int N,
                                                             int K, void* __restrict__ C, int64_t ldc) {
  constexpr int NT = (NB + 15) / 16;  // 16-column MFMA tiles
  __shared__ __attribute__((aligned(1024))) uint8_t wl[WAVES][NB * GV_ROWB];
  __shared__ float red[WAVES][8][NB + 1];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int n0 = blockIdx.x * NB;
  const int kw = wave * 512;
  const int col = lane & 15, kg = lane >> 4;
  u32x4 ap[8];  // ap[p]: row col % 8, k = kw + (2p + col / 8) * 32 + 8 kg .. + 8
  {
    const uint16_t* p = A + min(col & 7, M - 1) * lda + kw + (col >> 3) * 32 + kg * 8;
#pragma unroll
    for (int s = 0; s < 8; ++s) ap[s] = ld16(p + s * 64);
  }
  {
    const pipe::i32x4 rb = pipe::make_rsrc(B, uint32_t(int64_t(N) * K * 2));
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(&wl[wave][0]));
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      const uint32_t off = n0 + r < N ? uint32_t((int64_t(n0 + r) * K + kw) * 2) + lane * 16u : pipe::PAD;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
                   :
                   : "s"(lds0 + uint32_t(r * GV_ROWB)), "v"(off), "s"(rb)
                   : "memory");
    }
  }
  pipe::wait_vm<0>();  // this wave's weight rows are in LDS (and its A fragments in registers)
  f32x4 acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = f32x4{};
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    u32x4 a = ap[s >> 1];
    if (s & 1) {
#pragma unroll
      for (int d = 0; d < 4; ++d) a[d] = __builtin_amdgcn_update_dpp(0u, a[d], 0x128, 0xf, 0xf, false);  // row_ror:8
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const u32x4 b = *reinterpret_cast<const u32x4*>(&wl[wave][0] + min(j * 16 + col, NB - 1) * GV_ROWB +
                                                      kg * 16 + s * 64);
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                       acc[j], 0, 0, 0);
    }
  }
  // lane l holds column l % 16 of tile j, rows (l / 16) * 4 + 0..3; rows 8-15 are not used
  if (kg < 2) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
      if (j * 16 + col < NB)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][kg * 4 + i][j * 16 + col] = acc[j][i];
  }
  __syncthreads();
  for (int i = t; i < 8 * NB; i += 64 * WAVES) {
    const int m = i / NB, n = i % NB;
    if (m < M && n0 + n < N) {
      float v = red[0][m][n];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) v += red[w][m][n];
      store_out<MODE>(C, int64_t(m) * ldc + n0 + n, v);
    }
  }
}

// Skinny GEMM for 9 <= M <= 64 rows of A (larger decode batches, short
// prompts): gemv_pk_kernel's weight stream (K = 512 * WAVES, one 1 KB LDS-DMA
// per weight row and wave, NB columns per workgroup) with whole 16-row A
// fragments.  The weights stay in LDS while the MT = ceil(M / 16) row tiles
// pass over them; a tile's 16 fragments (8 k-values of 16 rows each) come
// straight from global memory, the next tile's in flight behind this one's
// MFMAs.  Bound by the weight stream plus the A rows that every workgroup
// re-reads from L2 (M * K * 2 bytes, 1-4 us of a CU's L2 port).
// Up to 16 rows K is summed in at least the four chains of gemv_mfma_kernel,
// quarter by quarter and added in order: the same bits, where one chain per
// wave was further from the exact sum at K = 512 (1.25e-7 against 0.72e-7 of
// its norm) and 1024 (1.27e-7 against 0.95e-7), at the same time (N = 4096 at
// 16 rows: 3.4 and 3.9 us).
template <int WAVES, int MT>
struct Skinny {
  static constexpr int CHAINS = MT == 1 && WAVES < 4 ? 4 / WAVES : 1;  // of each wave
};
template <int WAVES, int NB, int MT, int MODE>
__global__ __launch_bounds__(64 * WAVES) void gemm_skinny_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                                 const uint16_t* __restrict__ B, int M, int N,
                                                                 int K, void* __restrict__ C, int64_t ldc) {
  constexpr int NT = (NB + 15) / 16;  // 16-column MFMA tiles
  constexpr int RLD = NB + 1;
  constexpr int CH = Skinny<WAVES, MT>::CHAINS, PARTS = WAVES * CH;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];  // weights; then the partials
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int n0 = blockIdx.x * NB;
  const int kw = wave * 512;
  const int col = lane & 15, kg = lane >> 4;
  uint8_t* wl = smem + wave * (NB * GV_ROWB);
  u32x4 af[2][16];
  auto load_a = [&](u32x4 (&dst)[16], int mt) {  // rows past M repeat the last one; their products are not stored
    const uint16_t* p = A + int64_t(min(mt * 16 + col, M - 1)) * lda + kw + kg * 8;
#pragma unroll
    for (int s = 0; s < 16; ++s) dst[s] = ld16(p + s * 32);
  };
  load_a(af[0], 0);
  {
    const pipe::i32x4 rb = pipe::make_rsrc(B, uint32_t(int64_t(N) * K * 2));
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(wl));
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      const uint32_t off = n0 + r < N ? uint32_t((int64_t(n0 + r) * K + kw) * 2) + lane * 16u : pipe::PAD;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
                   :
                   : "s"(lds0 + uint32_t(r * GV_ROWB)), "v"(off), "s"(rb)
                   : "memory");
    }
  }
  pipe::wait_vm<0>();  // this wave's weight rows are in LDS (and its first A tile in registers)
  f32x4 acc[MT][NT][CH];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int c = 0; c < CH; ++c) acc[i][j][c] = f32x4{};
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    if (i + 1 < MT) load_a(af[(i + 1) & 1], i + 1);
#pragma unroll
    for (int s = 0; s < 16; ++s)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const u32x4 b = *reinterpret_cast<const u32x4*>(wl + min(j * 16 + col, NB - 1) * GV_ROWB + kg * 16 + s * 64);
        f32x4& a = acc[i][j][s * CH / 16];
        a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, af[i & 1][s]),
                                                    __builtin_bit_cast(bf16x8, b), a, 0, 0, 0);
      }
  }
  // lane l holds column l % 16 of tile j, rows 16 i + (l / 16) * 4 + 0..3
  __syncthreads();  // the weights are used up: their LDS takes the partials
  float* red = reinterpret_cast<float*>(smem);  // [PARTS][MT * 16][RLD]
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      if (j * 16 + col < NB)
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            red[((wave * CH + c) * MT * 16 + i * 16 + kg * 4 + e) * RLD + j * 16 + col] = acc[i][j][c][e];
  __syncthreads();
  for (int i = t; i < min(M, MT * 16) * NB; i += 64 * WAVES) {
    const int m = i / NB, n = i % NB;
    if (n0 + n < N) {
      float v = red[m * RLD + n];
#pragma unroll
      for (int p = 1; p < PARTS; ++p) v += red[(p * MT * 16 + m) * RLD + n];
      store_out<MODE>(C, int64_t(m) * ldc + n0 + n, v);
    }
  }
}

// Vocabulary-size projections of 2 <= M <= 64 rows (batched lm_head): N
// columns in tiles of 16, persistent workgroups taking every gridDim-th tile.
// Wave w of the K / 256 owns k in [256 w, 256 w + 256): its A fragments stay
// in registers for the whole launch (re-reading them per workgroup is what
// the column-owning kernels above spend their time on here), and its slice of
// a tile's weight rows (16 x 512 bytes: whole lines, non-temporal) streams
// through a private LDS ring of VO_S tiles without workgroup barriers.  The
// waves' partial tiles are added in k order through LDS, one barrier a tile.
// Bound by the weight stream: 622 MB (N = 151936, K = 2048).
constexpr int VO_S = 2, VO_TILE = 16 * 512;
// Row m of a partial tile sits at vo_row(m): the four lane groups' rows (4
// apart) are neighbours, so their stores and the sums' reads hit all banks.
__device__ __forceinline__ int vo_row(int m) { return (m & ~15) | ((m & 3) << 2) | ((m >> 2) & 3); }
// 8 waves fill a CU: two workgroups of 4 waves (K = 1024) share it, so the
// second set of partial tiles (one barrier less per tile) is taken only where
// both still fit.  With it, 33 rows and more of K = 1024 left one workgroup per
// CU and half of the launch waiting (N = 40000, 33 / 64 rows 21.3 / 26.4 us,
// 18.9 / 23.8 on one set).
template <int WAVES, int MT>
struct Vocab {
  static constexpr int PER_CU = 8 / WAVES, LDS = 160 * 1024 / PER_CU;  // workgroups of a CU, LDS of each
  static constexpr int RED = WAVES * MT * 256 * 4;  // bytes of one set of partial tiles
  static constexpr int NRED = WAVES * VO_S * VO_TILE + 2 * RED <= LDS ? 2 : 1;
  static constexpr int SMEM = WAVES * VO_S * VO_TILE + NRED * RED;
  static_assert(SMEM <= LDS, "LDS");
};
template <int WAVES, int MT, int MODE>
__global__ __launch_bounds__(64 * WAVES) void gemm_vocab_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                                const uint16_t* __restrict__ B, int M, int N,
                                                                int K, void* __restrict__ C, int64_t ldc) {
  using V = Vocab<WAVES, MT>;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];  // rings, then partial tiles
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int col = lane & 15, kg = lane >> 4, kw = wave * 256;
  const int tiles = (N + 15) / 16;
  uint8_t* ring = smem + wave * (VO_S * VO_TILE);
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(ring));
  const pipe::i32x4 rb = pipe::make_rsrc(B, uint32_t(int64_t(N) * K * 2));
  // DMA instruction i: rows 2i, 2i + 1 of the tile; chunk c of row r at slot c ^ r (32 chunks of 16 bytes a row)
  uint32_t vo[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = 2 * i + (lane >> 5);
    vo[i] = uint32_t(r) * uint32_t(K * 2) + uint32_t(kw * 2 + ((lane & 31) ^ r) * 16);
  }
  auto copy = [&](int tile, int slot) {
    const uint32_t base = uint32_t(tile) * 16u * uint32_t(K * 2);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 2 * i + (lane >> 5);
      pipe::dma16_nt(lds0 + uint32_t(slot * VO_TILE + i * 1024), tile * 16 + r < N ? vo[i] + base : pipe::PAD, rb, 0);
    }
  };
  bf16x8 af[MT][8];
#pragma unroll
  for (int i = 0; i < MT; ++i) {  // rows past M repeat the last one; their products are not stored
    const uint16_t* p = A + int64_t(min(i * 16 + col, M - 1)) * lda + kw + kg * 8;
#pragma unroll
    for (int s = 0; s < 8; ++s) af[i][s] = *reinterpret_cast<const bf16x8*>(p + s * 32);
  }
  int tile = blockIdx.x;
#pragma unroll
  for (int s = 0; s < VO_S; ++s)
    if (tile + s * int(gridDim.x) < tiles) copy(tile + s * gridDim.x, s);
  for (int it = 0; tile < tiles; tile += gridDim.x, ++it) {
    const int slot = it % VO_S;
    const bool more = tile + VO_S * int(gridDim.x) < tiles;
    // the tile has landed when only the copies issued after it are pending
    // (the stores in between make this wait for a little more than that)
    if (tile + int(gridDim.x) < tiles)
      pipe::wait_vm<8 * (VO_S - 1)>();
    else
      pipe::wait_vm<0>();
    const uint8_t* wt = ring + slot * VO_TILE + col * 512;
    bf16x8 bf[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) bf[s] = *reinterpret_cast<const bf16x8*>(wt + ((s * 4 + kg) ^ col) * 16);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot is read: its next copy may land
    if (more) copy(tile + VO_S * gridDim.x, slot);
    f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = f32x4{};
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][s], bf[s], acc[i], 0, 0, 0);
    // lane l holds column l % 16, rows 16 i + (l / 16) * 4 + 0..3
    float* red = reinterpret_cast<float*>(smem + WAVES * VO_S * VO_TILE + (it % V::NRED) * V::RED);
    if (V::NRED == 1) lds_barrier();  // the previous tile's sums are read
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) red[(wave * MT * 16 + i * 16 + e * 4 + kg) * 16 + col] = acc[i][e];
    lds_barrier();
    for (int i = threadIdx.x; i < MT * 256; i += 64 * WAVES) {
      const int m = vo_row(i >> 4), n = i & 15;  // vo_row is its own inverse
      if (m < M && tile * 16 + n < N) {
        float v = red[i];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) v += red[w * MT * 256 + i];
        store_out<MODE>(C, int64_t(m) * ldc + tile * 16 + n, v);
      }
    }
  }
}

// ------------------------------------------------------------------ MFMA tile
// Grid = every (row tile, column tile) pair, renumbered XCD-contiguously and
// then walked in groups of 8 row tiles per column sweep, so the workgroups
// one XCD runs together share A row panels and B column panels in its L2.
template <class P, int OCC, int MODE>
__global__ __launch_bounds__(256, OCC) void gemm_pipe_kernel(const uint16_t* __restrict__ A,
                                                             int64_t lda,
                                                             const uint16_t* __restrict__ B,
                                                             int M, int N, int K,
                                                             void* __restrict__ C, int64_t ldc) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int gx = (N + P::BN - 1) / P::BN, gy = (M + P::BM - 1) / P::BM;
  const int item = pipe::xcd_contiguous(int(blockIdx.x), gx * gy);
  constexpr int GM = 8;
  const int group = item / (GM * gx), first = group * GM, gm = min(gy - first, GM);
  const int r = item - group * GM * gx;
  const int m0 = (first + r % gm) * P::BM, n0 = (r / gm) * P::BN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const pipe::i32x4 ra = pipe::make_rsrc(A, uint32_t((int64_t(M) - 1) * lda * 2 + int64_t(K) * 2));
  const pipe::i32x4 rb = pipe::make_rsrc(B, uint32_t(int64_t(N) * K * 2));
  uint32_t vo[P::NDMA];
#pragma unroll
  for (int j = 0; j < P::NDMA; ++j) {
    const int rr = P::dma_row(j, wave, lane);
    const uint32_t c = P::dma_chunk(rr, lane);
    if (j < P::AI)
      vo[j] = m0 + rr < M ? uint32_t(int64_t(m0 + rr) * lda * 2) + c : pipe::PAD;
    else
      vo[j] = n0 + rr < N ? uint32_t(int64_t(n0 + rr) * K * 2) + c : pipe::PAD;
  }
  typename P::Acc acc;
  P::run(ra, rb, vo, K / P::BK, smem, acc);
#pragma unroll
  for (int i = 0; i < P::FM; ++i)
#pragma unroll
    for (int j = 0; j < P::FN; ++j) {
      const int col = n0 + P::acc_col(wave, j, lane);
      if (col < N) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = m0 + P::acc_row(wave, i, e, lane);
          if (row < M) store_out<MODE>(C, int64_t(row) * ldc + col, acc[i][j][e]);
        }
      }
    }
}

template <class P, int OCC, int MODE>
static int launch_pipe(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K,
                       void* C, int64_t ldc, hipStream_t s) {
  static const bool attr = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_pipe_kernel<P, OCC, MODE>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, P::SMEM);
    return true;
  }();
  (void)attr;
  const int64_t tiles = int64_t((M + P::BM - 1) / P::BM) * ((N + P::BN - 1) / P::BN);
  hipLaunchKernelGGL((gemm_pipe_kernel<P, OCC, MODE>), dim3(unsigned(tiles)), dim3(256), P::SMEM, s,
                     A, lda, B, M, N, K, C, ldc);
  return hip_status("qmoe_gemm(tile)");
}

// ------------------------------------------------------------------ large GEMMs
// Problems of at least 224 tiles of 256 x 256 run the grouped expert GEMMs'
// mainloop (mfma_wide.hpp: 8 waves, four 32-column stages, three in flight).
// Its A operand is B (weight rows n, 256 per tile) and its B operand is A
// (rows m), so each lane holds one output row m and, per 32 x 32 block, runs
// of 4 consecutive columns n: the epilogue stores them as one 16-byte fp32
// (8-byte bf16) piece straight from the accumulators (N % 4 == 0, ldc % 4 ==
// 0, C 16-byte aligned).  Tiles are walked as in gemm_pipe_kernel: XCD-
// contiguous, in groups of 8 row tiles per column sweep.
using WideDense = pipe::Wide<4, 2, 32, 4, 256>;

template <int MODE>
__device__ __forceinline__ void store_out4(void* C, int64_t idx, float a, float b, float c, float d) {
  if constexpr (MODE == QMOE_GEMM_STORE_BF16) {
    *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(C) + idx) = make_uint2(pack_bf16x2(a, b), pack_bf16x2(c, d));
  } else if constexpr (MODE == QMOE_GEMM_STORE_F32) {
    *reinterpret_cast<float4*>(reinterpret_cast<float*>(C) + idx) = make_float4(a, b, c, d);
  } else {
    float4* p = reinterpret_cast<float4*>(reinterpret_cast<float*>(C) + idx);
    const float4 v = *p;
    *p = make_float4(v.x + a, v.y + b, v.z + c, v.w + d);
  }
}

template <int MODE>
__global__ __launch_bounds__(WideDense::THREADS, 1) void gemm_wide_kernel(const uint16_t* __restrict__ A,
                                                                        int64_t lda,
                                                                        const uint16_t* __restrict__ B, int M,
                                                                        int N, int K, void* __restrict__ C,
                                                                        int64_t ldc) {
  using P = WideDense;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int gx = (N + P::BM - 1) / P::BM, gy = (M + P::BN - 1) / P::BN;
  const int item = pipe::xcd_contiguous(int(blockIdx.x), gx * gy);
  constexpr int GM = 8;
  const int group = item / (GM * gx), first = group * GM, gm = min(gy - first, GM);
  const int r = item - group * GM * gx;
  const int m0 = (first + r % gm) * P::BN, n0 = (r / gm) * P::BM;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const pipe::i32x4 ra = pipe::make_rsrc(B, uint32_t(int64_t(N) * K * 2));
  const pipe::i32x4 rb = pipe::make_rsrc(A, uint32_t((int64_t(M) - 1) * lda * 2 + int64_t(K) * 2));
  uint32_t vo[P::NDMA];
#pragma unroll
  for (int j = 0; j < P::NDMA; ++j) {
    const int rr = P::dma_row(j, wave, lane);
    const uint32_t c = P::dma_chunk(rr, lane);
    if (j < P::AI)
      vo[j] = n0 + rr < N ? uint32_t(int64_t(n0 + rr) * K * 2) + c : pipe::PAD;
    else
      vo[j] = m0 + rr < M ? uint32_t(int64_t(m0 + rr) * lda * 2) + c : pipe::PAD;
  }
  // this wave's live 32-row blocks of A rows (none when its weight rows lie past N)
  const int nb = n0 + P::wave_arow(wave) < N ? P::wave_blocks(wave, (min(M - m0, P::BN) + 31) / 32) : 0;
  typename P::Acc acc;
  P::run_dyn(nb, ra, rb, vo, K / P::BK, smem, acc, uint32_t(P::BK * 2), uint32_t(P::BK * 2));
#pragma unroll
  for (int j = 0; j < P::FN; ++j) {
    if (j >= nb) break;
    const int row = m0 + P::acc_brow(wave, j, lane);
    if (row >= M) continue;
#pragma unroll
    for (int i = 0; i < P::FM; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = n0 + P::wave_arow(wave) + i * 32 + q * 8 + (lane >> 5) * 4;
        if (col < N)
          store_out4<MODE>(C, int64_t(row) * ldc + col, acc[i][j][4 * q], acc[i][j][4 * q + 1],
                           acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
      }
  }
}

template <int MODE>
static int launch_wide(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K, void* C,
                       int64_t ldc, hipStream_t s) {
  using P = WideDense;
  static const bool attr = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_wide_kernel<MODE>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, P::SMEM);
    return true;
  }();
  (void)attr;
  const int64_t tiles = int64_t((M + P::BN - 1) / P::BN) * ((N + P::BM - 1) / P::BM);
  hipLaunchKernelGGL((gemm_wide_kernel<MODE>), dim3(unsigned(tiles)), dim3(P::THREADS), P::SMEM, s, A, lda, B,
                     M, N, K, C, ldc);
  return hip_status("qmoe_gemm(wide)");
}

// Tile shape by how many tiles the problem has: 256x256 (one workgroup per
// CU, least L2 traffic per flop) once it fills the GPU, else smaller tiles
// with two workgroups per CU; problems that would still leave most CUs idle
// (the prefill router: 4096 x 128 x 2048) take 64x64 tiles with four stages
// in flight, since each of their few workgroups walks a long K.
// Large fp32-output GEMMs (the 8-wave pipeline's sizes, K >= 2048: the
// batch-8 prompt's o_proj, 8192 x 2048 x 4096) go to hipBLASLt, a plain
// library GEMM: C (fp32, ldc) = A . B^T (+ C with ADD_F32).  It keeps the
// long-K tiles' MFMA rate and overlaps the fp32 C read-modify-write that the
// one-tile-per-CU pipeline leaves to the end (8192 x 2048 x 4096: 103 us
// against 145-155 us).  One handle per device, one plan per shape (the
// heuristic's first algorithm, no workspace); a shape the library has no
// algorithm for stays on the pipeline.
namespace {
struct BltPlan {
  hipblasLtMatmulDesc_t op = nullptr;
  hipblasLtMatrixLayout_t la = nullptr, lb = nullptr, lc = nullptr;
  hipblasLtMatmulAlgo_t algo{};
  bool ok = false;
};
std::mutex blt_mu;
std::map<int, hipblasLtHandle_t> blt_handles;
std::map<std::tuple<int, int64_t, int64_t, int64_t, int64_t, int64_t>, BltPlan> blt_plans;

const BltPlan* blt_plan(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldc, hipblasLtHandle_t* h) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> g(blt_mu);
  auto hi = blt_handles.find(dev);
  if (hi == blt_handles.end()) {
    hipblasLtHandle_t nh = nullptr;
    if (hipblasLtCreate(&nh) != HIPBLAS_STATUS_SUCCESS) nh = nullptr;
    hi = blt_handles.emplace(dev, nh).first;
  }
  if (!hi->second) return nullptr;
  *h = hi->second;
  auto key = std::make_tuple(dev, M, N, K, lda, ldc);
  auto pi = blt_plans.find(key);
  if (pi != blt_plans.end()) return pi->second.ok ? &pi->second : nullptr;
  BltPlan p;
  // column-major view: C^T (N x M, ld ldc) = B (N x K row-major = K x N, op T) . A^T (K x M, ld lda)
  const hipblasOperation_t ta = HIPBLAS_OP_T, tb = HIPBLAS_OP_N;
  bool ok = hipblasLtMatmulDescCreate(&p.op, HIPBLAS_COMPUTE_32F, HIP_R_32F) == HIPBLAS_STATUS_SUCCESS &&
            hipblasLtMatmulDescSetAttribute(p.op, HIPBLASLT_MATMUL_DESC_TRANSA, &ta, sizeof(ta)) ==
                HIPBLAS_STATUS_SUCCESS &&
            hipblasLtMatmulDescSetAttribute(p.op, HIPBLASLT_MATMUL_DESC_TRANSB, &tb, sizeof(tb)) ==
                HIPBLAS_STATUS_SUCCESS &&
            hipblasLtMatrixLayoutCreate(&p.la, HIP_R_16BF, uint64_t(K), uint64_t(N), K) == HIPBLAS_STATUS_SUCCESS &&
            hipblasLtMatrixLayoutCreate(&p.lb, HIP_R_16BF, uint64_t(K), uint64_t(M), lda) == HIPBLAS_STATUS_SUCCESS &&
            hipblasLtMatrixLayoutCreate(&p.lc, HIP_R_32F, uint64_t(N), uint64_t(M), ldc) == HIPBLAS_STATUS_SUCCESS;
  if (ok) {
    hipblasLtMatmulPreference_t pref = nullptr;
    uint64_t wsb = 0;
    hipblasLtMatmulHeuristicResult_t res{};
    int n = 0;
    ok = hipblasLtMatmulPreferenceCreate(&pref) == HIPBLAS_STATUS_SUCCESS &&
         hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &wsb,
                                               sizeof(wsb)) == HIPBLAS_STATUS_SUCCESS &&
         hipblasLtMatmulAlgoGetHeuristic(*h, p.op, p.la, p.lb, p.lc, p.lc, pref, 1, &res, &n) ==
             HIPBLAS_STATUS_SUCCESS &&
         n > 0 && res.workspaceSize == 0;
    if (pref) hipblasLtMatmulPreferenceDestroy(pref);
    if (ok) p.algo = res.algo;
  }
  p.ok = ok;
  auto& slot = blt_plans[key] = p;
  return ok ? &slot : nullptr;
}
}  // namespace

// true when the call went to hipBLASLt (rc holds its status)
static bool blt_gemm(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t M, int64_t N, int64_t K, float* C,
                     int64_t ldc, bool add, hipStream_t s, int* rc) {
  hipblasLtHandle_t h = nullptr;
  const BltPlan* p = blt_plan(M, N, K, lda, ldc, &h);
  if (!p) return false;
  const float alpha = 1.0f, beta = add ? 1.0f : 0.0f;
  const hipblasStatus_t st = hipblasLtMatmul(h, p->op, &alpha, B, p->la, A, p->lb, &beta, C, p->lc, C, p->lc,
                                             &p->algo, nullptr, 0, s);
  *rc = st == HIPBLAS_STATUS_SUCCESS ? hip_status("qmoe_gemm(hipblaslt)")
                                     : fail(QMOE_ERR_HIP, "qmoe_gemm: hipblasLtMatmul failed (%d)", int(st));
  return true;
}

template <int MODE>
static int launch_tile(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K,
                       void* C, int64_t ldc, hipStream_t s) {
  using Big = pipe::Pipe<256, 256, 64, 2>;
  using Mid = pipe::Pipe<128, 256, 32, 3>;
  using Small = pipe::Pipe<128, 128, 64, 2>;
  using Tiny = pipe::Pipe<64, 64, 64, 4>;
  auto count = [&](int bm, int bn) { return int64_t((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  if (MODE != QMOE_GEMM_STORE_BF16 && count(256, 256) >= 224 && K >= 2048) {
    int rc = QMOE_OK;
    if (blt_gemm(A, lda, B, M, N, K, static_cast<float*>(C), ldc, MODE == QMOE_GEMM_ADD_F32, s, &rc)) return rc;
  }
  if (count(256, 256) >= 224 && N % 4 == 0 && ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0)
    return launch_wide<MODE>(A, lda, B, M, N, K, C, ldc, s);
  if (count(256, 256) >= 224) return launch_pipe<Big, 1, MODE>(A, lda, B, M, N, K, C, ldc, s);
  if (count(128, 256) >= 224) return launch_pipe<Mid, 2, MODE>(A, lda, B, M, N, K, C, ldc, s);
  if (count(128, 128) >= 96) return launch_pipe<Small, 2, MODE>(A, lda, B, M, N, K, C, ldc, s);
  return launch_pipe<Tiny, 2, MODE>(A, lda, B, M, N, K, C, ldc, s);
}

// ------------------------------------------------------------------ split-K
// For problems with too few output tiles to occupy the GPU (prefill-size
// o_proj: 640 x 2048 with K = 4096 is 80 tiles of 128 x 128; the router
// logits: 640 x 128 with K = 2048 is 20 tiles of 64 x 64), K is split into
// `splits` slices: workgroup (tile, slice) writes its fp32 partial tile to a
// caller-owned workspace part[slice][M][N], and splitk_reduce_kernel adds the
// slices in slice order (fixed order: repeat calls are bit-identical) and
// applies the epilogue mode.
template <class P, int OCC>
__global__ __launch_bounds__(256, OCC) void gemm_splitk_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                               const uint16_t* __restrict__ B, int M, int N,
                                                               int K, int splits, float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tiles_n = (N + P::BN - 1) / P::BN;
  const int slice = int(blockIdx.x) % splits, tile = int(blockIdx.x) / splits;
  const int m0 = (tile / tiles_n) * P::BM, n0 = (tile % tiles_n) * P::BN;
  const int ks = K / splits;
  const uint32_t k0b = uint32_t(slice) * uint32_t(ks) * 2u;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const pipe::i32x4 ra = pipe::make_rsrc(A, uint32_t((int64_t(M) - 1) * lda * 2 + int64_t(K) * 2));
  const pipe::i32x4 rb = pipe::make_rsrc(B, uint32_t(int64_t(N) * K * 2));
  uint32_t vo[P::NDMA];
#pragma unroll
  for (int j = 0; j < P::NDMA; ++j) {
    const int rr = P::dma_row(j, wave, lane);
    const uint32_t c = P::dma_chunk(rr, lane);
    if (j < P::AI)
      vo[j] = m0 + rr < M ? uint32_t(int64_t(m0 + rr) * lda * 2) + k0b + c : pipe::PAD;
    else
      vo[j] = n0 + rr < N ? uint32_t(int64_t(n0 + rr) * K * 2) + k0b + c : pipe::PAD;
  }
  typename P::Acc acc;
  P::run(ra, rb, vo, ks / P::BK, smem, acc);
  float* dst = part + int64_t(slice) * M * N;
#pragma unroll
  for (int i = 0; i < P::FM; ++i)
#pragma unroll
    for (int j = 0; j < P::FN; ++j) {
      const int col = n0 + P::acc_col(wave, j, lane);
      if (col < N) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = m0 + P::acc_row(wave, i, e, lane);
          if (row < M) dst[int64_t(row) * N + col] = acc[i][j][e];
        }
      }
    }
}

// The slices of a 17 <= M <= 64 row problem (decode-batch o_proj): workgroup
// (64 columns, 512 k-values) copies its weight rows and the A rows' slice
// into LDS in one go (1 KB LDS-DMA per row: whole lines, everything requested
// at once), then 8 waves run the 16 x 16 tiles.  One memory round trip long:
// splitting K keeps the A bytes per workgroup at M KB, where a workgroup that
// owns whole columns re-reads all of A (M * K * 2 bytes at the 16-row fragment
// loads' 16 B per clock: 2048 x 4096 takes 10.9 us at 32 rows, 18.2 at 64).
constexpr int SL_K = 512, SL_N = 64;
template <int MT>
__global__ __launch_bounds__(512) void gemm_slice_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                         const uint16_t* __restrict__ B, int M, int N, int K,
                                                         float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];  // SL_N weight rows, then 16 MT A rows
  const int splits = K / SL_K, slice = int(blockIdx.x) % splits, n0 = int(blockIdx.x) / splits * SL_N;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const pipe::i32x4 ra = pipe::make_rsrc(A, uint32_t((int64_t(M) - 1) * lda * 2 + int64_t(K) * 2));
  const pipe::i32x4 rb = pipe::make_rsrc(B, uint32_t(int64_t(N) * K * 2));
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(smem));
  const uint32_t kb = uint32_t(slice) * SL_K * 2 + lane * 16u;
#pragma unroll
  for (int i = 0; i < SL_N / 8; ++i) {
    const int r = wave * (SL_N / 8) + i;
    const uint32_t off = n0 + r < N ? uint32_t(int64_t(n0 + r) * K * 2) + kb : pipe::PAD;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
                 :
                 : "s"(lds0 + uint32_t(r * GV_ROWB)), "v"(off), "s"(rb)
                 : "memory");
  }
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) {
    const int r = wave * 2 * MT + i;
    pipe::dma16(lds0 + uint32_t((SL_N + r) * GV_ROWB), r < M ? uint32_t(int64_t(r) * lda * 2) + kb : pipe::PAD, ra, 0);
  }
  pipe::wait_vm<0>();
  __syncthreads();
  const int col = lane & 15, kg = lane >> 4, ct = wave & 3;
  const uint8_t* bp = smem + (ct * 16 + col) * GV_ROWB + kg * 16;
  float* dst = part + int64_t(slice) * M * N;
  for (int mt = wave >> 2; mt < MT; mt += 2) {
    const uint8_t* ap = smem + (SL_N + mt * 16 + col) * GV_ROWB + kg * 16;
    f32x4 acc[2] = {f32x4{}, f32x4{}};
#pragma unroll
    for (int s = 0; s < SL_K / 32; ++s)
      acc[s & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(ap + s * 64),
                                                           *reinterpret_cast<const bf16x8*>(bp + s * 64), acc[s & 1],
                                                           0, 0, 0);
    const int n = n0 + ct * 16 + col;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = mt * 16 + kg * 4 + e;
      if (m < M && n < N) dst[int64_t(m) * N + n] = acc[0][e] + acc[1][e];
    }
  }
}

// Sum of the slices' float4 at float offset o, in slice order; with S known
// every load is in flight at once (S = 0: any count).
template <int S>
__device__ __forceinline__ float4 sum_slices(const float* __restrict__ part, int splits, int64_t slab, int64_t o) {
  const int n = S ? S : splits;
  float4 v[S ? S : 1];
  if constexpr (S > 0) {
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = *reinterpret_cast<const float4*>(part + s * slab + o);
  } else {
    v[0] = *reinterpret_cast<const float4*>(part + o);
  }
  float4 a = v[0];
#pragma unroll
  for (int s = 1; s < n; ++s) {
    const float4 w = S ? v[S ? s : 0] : *reinterpret_cast<const float4*>(part + s * slab + o);
    a.x += w.x;
    a.y += w.y;
    a.z += w.z;
    a.w += w.w;
  }
  return a;
}

// C (mode) = sum over slices in order; 4 consecutive columns per thread.
template <int MODE, int S>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, int splits, int M,
                                                           int N, void* C, int64_t ldc) {
  const int64_t q = int64_t(blockIdx.x) * 256 + threadIdx.x;  // float4 index
  const int64_t per_row = N / 4;
  if (q >= int64_t(M) * per_row) return;
  const int64_t row = q / per_row, col = (q - row * per_row) * 4;
  const int64_t slab = int64_t(M) * N;
  const float4 v = sum_slices<S>(part, splits, slab, row * N + col);
  store_out<MODE>(C, row * ldc + col, v.x);
  store_out<MODE>(C, row * ldc + col + 1, v.y);
  store_out<MODE>(C, row * ldc + col + 2, v.z);
  store_out<MODE>(C, row * ldc + col + 3, v.w);
}

// The ADD_F32 reduction of whole rows (one workgroup per row, the chunks of
// norm_impl.hpp) followed by the row's RMSNorm: C[row] += sum of the slices
// (splitk_reduce_kernel's order), x_out[row] = bf16(rms_w * C[row] * r).
template <int S>
__global__ __launch_bounds__(NORM_THREADS) void splitk_reduce_norm_kernel(
    const float* __restrict__ part, int splits, int M, int N, float* C, const uint16_t* __restrict__ rms_w,
    float eps, uint16_t* __restrict__ x_out) {
  const int64_t row = blockIdx.x;
  const int64_t slab = int64_t(M) * N;
  float4 v[NORM_MAX_CHUNKS];
  float ss = 0.0f;
  const int nchunk = N / 4;
#pragma unroll
  for (int j = 0; j < NORM_MAX_CHUNKS; ++j) {
    const int c = int(threadIdx.x) + j * NORM_THREADS;
    if (c < nchunk) {
      const int64_t o = row * N + 4 * c;
      float4 h = *reinterpret_cast<const float4*>(C + o);
      const float4 a = sum_slices<S>(part, splits, slab, o);
      h.x += a.x;
      h.y += a.y;
      h.z += a.z;
      h.w += a.w;
      *reinterpret_cast<float4*>(C + o) = h;
      v[j] = h;
      ss += norm_sq4(h);
    }
  }
  __shared__ float red[NORM_THREADS / 64];
  const float r = norm_rsqrt(ss, N, eps, red);
  uint16_t* xr = x_out + row * N;
#pragma unroll
  for (int j = 0; j < NORM_MAX_CHUNKS; ++j) {
    const int c = int(threadIdx.x) + j * NORM_THREADS;
    if (c < nchunk) reinterpret_cast<uint2*>(xr)[c] = norm_out4(v[j], r, rms_w, c);
  }
}

using SplitSmall = pipe::Pipe<128, 128, 64, 2>;
using SplitMid = pipe::Pipe<64, 128, 64, 3>;
using SplitTiny = pipe::Pipe<64, 64, 64, 4>;

// Tile shape of a split-K plan.
enum SplitTile { SPLIT_TINY = 0, SPLIT_SMALL = 1, SPLIT_MID = 2 };

// Split-K plan for an M > 16 problem: 0 slices = do not split (the problem
// already has at least 256 tiles, or K is too short to split).  Tiles: 128 x
// 128 when there are at least 16 of them, but 64 x 128 when there are 40-127
// (twice the tiles at half the slices: the o_proj of a 640-token prompt,
// 640 x 2048 x 4096, runs 29.8 us as 80 tiles x 4 slices and 26.8 us as 160
// x 2; 384 x 2048 x 4096: 21.7 -> 20.5 us), else 64 x 64.  Slices double
// while the grid stays within 512 workgroups and each slice keeps >= 512
// (128-column tiles) or >= 256 (64 x 64) columns of K, a multiple of the
// 64-column stage.
static int splitk_plan(int64_t M, int64_t N, int64_t K, SplitTile* tile) {
  if (M <= 16 || N % 4 != 0 || K % 64 != 0) return 0;
  const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
  *tile = t128 >= 40 && t128 < 128 ? SPLIT_MID : t128 >= 16 ? SPLIT_SMALL : SPLIT_TINY;
  const int64_t tiles = *tile == SPLIT_SMALL ? t128
                        : *tile == SPLIT_MID ? ((M + 63) / 64) * ((N + 127) / 128)
                                             : ((M + 63) / 64) * ((N + 63) / 64);
  const int64_t kmin = *tile == SPLIT_TINY ? 256 : 512;
  if (t128 >= 256) return 0;
  int splits = 1;
  while (tiles * splits * 2 <= 512 && K % (int64_t(splits) * 2 * 64) == 0 && K / (splits * 2) >= kmin) splits *= 2;
  return splits > 1 ? splits : 0;
}

// The sum of the slices into C (mode), with x_out (ADD_F32, rows of N floats)
// followed by the rows' RMSNorm.
template <int MODE, int S>
static int launch_reduce_s(const float* part, int splits, int M, int N, void* C, int64_t ldc, hipStream_t s,
                           const uint16_t* rms_w, float eps, uint16_t* x_out) {
  if (x_out) {
    hipLaunchKernelGGL(splitk_reduce_norm_kernel<S>, dim3(unsigned(M)), dim3(NORM_THREADS), 0, s, part, splits, M, N,
                       static_cast<float*>(C), rms_w, eps, x_out);
    return hip_status("qmoe_gemm_ws(reduce + norm)");
  }
  const int64_t n4 = int64_t(M) * (N / 4);
  hipLaunchKernelGGL((splitk_reduce_kernel<MODE, S>), dim3(unsigned((n4 + 255) / 256)), dim3(256), 0, s, part, splits,
                     M, N, C, ldc);
  return hip_status("qmoe_gemm_ws(reduce)");
}

template <int MODE>
static int launch_reduce(const float* part, int splits, int M, int N, void* C, int64_t ldc, hipStream_t s,
                         const uint16_t* rms_w, float eps, uint16_t* x_out) {
  switch (splits) {
    case 2: return launch_reduce_s<MODE, 2>(part, splits, M, N, C, ldc, s, rms_w, eps, x_out);
    case 4: return launch_reduce_s<MODE, 4>(part, splits, M, N, C, ldc, s, rms_w, eps, x_out);
    case 8: return launch_reduce_s<MODE, 8>(part, splits, M, N, C, ldc, s, rms_w, eps, x_out);
    default: return launch_reduce_s<MODE, 0>(part, splits, M, N, C, ldc, s, rms_w, eps, x_out);
  }
}

// gemm_slice_kernel takes a split-K plan whose slices are its 512 columns,
// while its workgroups fit the CUs in one round.  o_proj into the residual
// with the norm (N = 2048, K = 4096; 17 / 32 / 64 rows, reduction included):
// 18.1 / 18.2 / 19.2 us on 128 x 128 tiles, 10.2 / 10.6 / 12.9 us here; with
// 1.25 rounds (N = 5120, K = 2048) 13.4 us against 10.9.
static bool slice_ok(int64_t M, int64_t N, int64_t K, int splits) {
  return M >= 17 && M <= 64 && splits * SL_K == K && (N + SL_N - 1) / SL_N * splits <= current_device_cus();
}

template <int MT>
static void launch_slices(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K, float* part,
                          hipStream_t s) {
  constexpr int SMEM = (SL_N + 16 * MT) * GV_ROWB;
  static const bool attr = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_slice_kernel<MT>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
    return true;
  }();
  (void)attr;
  hipLaunchKernelGGL(gemm_slice_kernel<MT>, dim3(unsigned((N + SL_N - 1) / SL_N * (K / SL_K))), dim3(512), SMEM, s, A,
                     lda, B, M, N, K, part);
}

template <class P, int MODE>
static int launch_splitk(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K, int splits,
                         float* part, void* C, int64_t ldc, hipStream_t s, const uint16_t* rms_w = nullptr,
                         float eps = 0.0f, uint16_t* x_out = nullptr) {
  static const bool attr = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_splitk_kernel<P, 2>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, P::SMEM);
    return true;
  }();
  (void)attr;
  if (slice_ok(M, N, K, splits)) {
    if (M <= 32)
      launch_slices<2>(A, lda, B, M, N, K, part, s);
    else if (M <= 48)
      launch_slices<3>(A, lda, B, M, N, K, part, s);
    else
      launch_slices<4>(A, lda, B, M, N, K, part, s);
  } else {
    const int64_t tiles = int64_t((M + P::BM - 1) / P::BM) * ((N + P::BN - 1) / P::BN);
    hipLaunchKernelGGL((gemm_splitk_kernel<P, 2>), dim3(unsigned(tiles * splits)), dim3(256), P::SMEM, s, A, lda,
                       B, M, N, K, splits, part);
  }
  if (int rc = hip_status("qmoe_gemm_ws(slices)")) return rc;
  return launch_reduce<MODE>(part, splits, M, N, C, ldc, s, rms_w, eps, x_out);
}

int64_t gemm_splitk_bytes(int64_t M, int64_t N, int64_t K) {
  SplitTile tile = SPLIT_TINY;
  const int splits = (M >= 0 && N >= 0 && K >= 0) ? splitk_plan(M, N, K, &tile) : 0;
  return splits ? int64_t(splits) * M * N * int64_t(sizeof(float)) : 0;
}

int gemm_splitk_slices(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t M, int64_t N, int64_t K,
                       float* part, int64_t part_bytes, int* splits, hipStream_t s) {
  SplitTile tile = SPLIT_TINY;
  const int n = splitk_plan(M, N, K, &tile);
  *splits = 0;
  if (n == 0 || part == nullptr || part_bytes < int64_t(n) * M * N * int64_t(sizeof(float)) ||
      M >= (1ll << 31) || N >= (1ll << 31) || lda < K || lda % 8 != 0 ||
      (M - 1) * lda * 2 + K * 2 >= (1ll << 31) || N * K * 2 >= (1ll << 31))
    return QMOE_OK;
  QMOE_REQUIRE(A && B, "gemm_splitk_slices: null pointer");
  auto go = [&](auto tile) {
    using P = decltype(tile);
    static const bool attr = [] {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_splitk_kernel<P, 2>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, P::SMEM);
      return true;
    }();
    (void)attr;
    const int64_t tiles = ((M + P::BM - 1) / P::BM) * ((N + P::BN - 1) / P::BN);
    hipLaunchKernelGGL((gemm_splitk_kernel<P, 2>), dim3(unsigned(tiles * n)), dim3(256), P::SMEM, s, A, lda, B,
                       int(M), int(N), int(K), n, part);
  };
  if (tile == SPLIT_SMALL)
    go(SplitSmall{});
  else if (tile == SPLIT_MID)
    go(SplitMid{});
  else
    go(SplitTiny{});
  *splits = n;
  return hip_status("gemm_splitk_slices");
}

// ------------------------------------------------------------------ launcher
template <int MT, int MODE>
static int launch_gemv_reg(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K,
                           void* C, int64_t ldc, hipStream_t s) {
  // One weight row per wave for a single activation row (the most waves, each
  // with its whole row in flight); more rows per wave amortise the staging
  // of several activation rows.
  constexpr int R = MT == 1 ? 1 : 4;
  const size_t shm = size_t(M) * K * 2;
  static const bool attr = [] {
    for (const void* f : {reinterpret_cast<const void*>(gemv_reg_kernel<MT, R, 1, MODE>),
                          reinterpret_cast<const void*>(gemv_reg_kernel<MT, R, 2, MODE>),
                          reinterpret_cast<const void*>(gemv_reg_kernel<MT, R, 4, MODE>),
                          reinterpret_cast<const void*>(gemv_reg_kernel<MT, (R > 2 ? 2 : R), 8, MODE>)})
      (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 64 * 1024);
    return true;
  }();
  (void)attr;
  switch (K / 512) {
#define QMOE_GR(RR, KC)                                                                            \
  case KC:                                                                                         \
    hipLaunchKernelGGL((gemv_reg_kernel<MT, RR, KC, MODE>), dim3(unsigned((N + 4 * RR - 1) / (4 * RR))), \
                       dim3(256), shm, s, A, lda, B, M, N, K, C, ldc);                             \
    return hip_status("qmoe_gemm(gemv)");
    QMOE_GR(R, 1)
    QMOE_GR(R, 2)
    QMOE_GR(R, 4)
    QMOE_GR((R > 2 ? 2 : R), 8)
#undef QMOE_GR
    default:
      return fail(QMOE_ERR_INVALID, "qmoe_gemm: gemv register path needs K in {512, 1024, 2048, 4096}");
  }
}

template <int MODE>
static int launch_gemv_mfma(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K,
                            void* C, int64_t ldc, hipStream_t s) {
  const size_t shm = size_t(M) * K * 2;
  // 8 columns per workgroup unless that makes very many workgroups: at 8 rows
  // the QKV (N = 5120, K = 2048) and o_proj (N = 2048, K = 4096) shapes run
  // 8.7 -> 8.4 and 8.8 -> 7.9 us against 16 columns
  const bool narrow = (N + 15) / 16 < 1024;
  static const bool attr = [] {
    for (const void* f : {reinterpret_cast<const void*>(gemv_mfma_kernel<8, 4, MODE>),
                          reinterpret_cast<const void*>(gemv_mfma_kernel<16, 4, MODE>),
                          reinterpret_cast<const void*>(gemv_mfma_kernel<8, 8, MODE>),
                          reinterpret_cast<const void*>(gemv_mfma_kernel<16, 8, MODE>),
                          reinterpret_cast<const void*>(gemv_mfma_kernel<8, 16, MODE>),
                          reinterpret_cast<const void*>(gemv_mfma_kernel<16, 16, MODE>),
                          reinterpret_cast<const void*>(gemv_mfma_kernel<8, 32, MODE>),
                          reinterpret_cast<const void*>(gemv_mfma_kernel<16, 32, MODE>)})
      (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 64 * 1024);
    return true;
  }();
  (void)attr;
  switch (K / 128) {
#define QMOE_GM(KS)                                                                                \
  case KS:                                                                                         \
    if (narrow)                                                                                    \
      hipLaunchKernelGGL((gemv_mfma_kernel<8, KS, MODE>), dim3(unsigned((N + 7) / 8)), dim3(256), shm, \
                         s, A, lda, B, M, N, K, C, ldc);                                           \
    else                                                                                           \
      hipLaunchKernelGGL((gemv_mfma_kernel<16, KS, MODE>), dim3(unsigned((N + 15) / 16)), dim3(256),  \
                         shm, s, A, lda, B, M, N, K, C, ldc);                                      \
    return hip_status("qmoe_gemm(gemv mfma)");
    QMOE_GM(4)
    QMOE_GM(8)
    QMOE_GM(16)
    QMOE_GM(32)
#undef QMOE_GM
    default:
      return fail(QMOE_ERR_INVALID, "qmoe_gemm: skinny MFMA path needs K in {512, 1024, 2048, 4096}");
  }
}

template <int MODE>
static int launch_gemv_pk(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K,
                          void* C, int64_t ldc, hipStream_t s) {
  // the most columns per workgroup that still leaves one workgroup per CU
  // (fewer workgroups load the A rows fewer times: at 8 rows the QKV shape N
  // = 5120, K = 2048 runs 7.3 / 6.5 / 6.0 us at 8 / 10 / 20 columns, and
  // o_proj N = 2048, K = 4096 5.7 us at 8 columns against 7.2 at 4)
  const int cus = current_device_cus();
  const int nb = N >= 20 * cus && K <= 2048 ? 20 : N >= 16 * cus ? 16 : N >= 8 * cus ? 8 : 4;
#define QMOE_PK(W, NB_)                                                                            \
  if (K == 512 * W && nb == NB_) {                                                                 \
    hipLaunchKernelGGL((gemv_pk_kernel<W, NB_, MODE>), dim3(unsigned((N + NB_ - 1) / NB_)), dim3(64 * W), 0, \
                       s, A, lda, B, M, N, K, C, ldc);                                             \
    return hip_status("qmoe_gemm(gemv pk)");                                                       \
  }
#define QMOE_PK_W(W) QMOE_PK(W, 4) QMOE_PK(W, 8) QMOE_PK(W, 16)
  QMOE_PK_W(1)
  QMOE_PK_W(2)
  QMOE_PK_W(4)
  QMOE_PK_W(8)
  QMOE_PK(1, 20)
  QMOE_PK(2, 20)
  QMOE_PK(4, 20)
#undef QMOE_PK_W
#undef QMOE_PK
  return fail(QMOE_ERR_INVALID, "qmoe_gemm: packed GEMV needs K in {512, 1024, 2048, 4096}");
}

// The skinny and vocabulary kernels copy B by LDS-DMA, 16 bytes a lane; a B
// that is not 16-byte aligned stays on the kernels of the general order: the
// 9 to 16 rows of those load it into registers, the others (packed GEMV, MFMA
// tiles) copy it by LDS-DMA too.
static bool dma_aligned(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// Columns per workgroup of gemm_skinny_kernel, 0 where another kernel takes
// the shape.  Every workgroup reads all of A from L2 and runs every row tile,
// so the fewest columns that give each CU at most one workgroup are taken
// (N = 1536, K = 2048 at 16 / 48 rows on 8 columns 4.6 / 8.1 us, on 4 and
// twice the workgroups 6.6 / 13.0).  us against the kernels that had these
// shapes before (16-row GEMV up to 16 rows of K <= 2048, 64 x 64 tiles), at 9 /
// 16 / 32 / 64 rows:
//   N = 5120, K = 2048   8.9 / 11.5 / 12.1 / 12.8 -> 6.2 / 6.9 / 9.1 / 12.4
//   N = 2048, K = 4096   20.1 / 20.1 / 20.4 / 21.5 -> 6.1 / 7.3 / 10.5 / 17.6
// A short K leaves a wave so little to do that the columns of 20 (two MFMA
// column tiles) and the last row tile lose: N = 5120, K = 1024 at 40 rows 7.2 ->
// 8.3, K = 512 at 17 rows 4.8 -> 5.3; N = 4096, K = 512 at 64 rows 5.0 -> 5.4.
// A second round of workgroups wins up to 16 rows once it is about half full
// (N = 7168, K = 2048, 9 / 16 rows 10.4 / 14.1 -> 9.9 / 11.4; N = 6144 at 9
// rows 9.1 -> 9.7) and loses above (N = 8192, 17 / 64 rows 12.2 / 13.4 -> 14.4
// / 22.6); where the others are slow, at K = 4096, it wins from its start and
// up to 24 rows (N = 8192 at 24 / 32 rows 23.1 / 23.4 -> 21.5 / 24.1; N =
// 10240, two and a half rounds, at 12 / 17 rows 25.2 / 25.4 -> 22.9 / 26.8).
static int skinny_cols(const void* B, int64_t M, int64_t N, int64_t K) {
  if (!dma_aligned(B) || M < 9 || M > 64 || (K != 512 && K != 1024 && K != 2048 && K != 4096) ||
      N * K * 2 >= (1ll << 31))
    return 0;
  const int64_t cus = current_device_cus();
  for (int nb : {4, 8, 16, 20}) {
    if (N > nb * cus || (nb == 20 && K == 4096)) continue;  // 20 columns of 4096 do not fit in LDS
    const int64_t rows = nb == 20 ? (K == 512 ? 16 : K == 1024 ? 32 : 64) : (K == 512 ? 48 : 64);
    return M <= rows ? nb : 0;
  }
  if (K == 4096) return M <= (N <= 32 * cus ? 24 : N <= 40 * cus ? 16 : 0) ? 16 : 0;
  return K >= 1024 && M <= 16 && N >= 28 * cus && N <= 40 * cus ? 20 : 0;
}

// Rows and shapes of gemm_vocab_kernel: more than the skinny kernel's columns.
// N = 151936, K = 2048 at 2 / 8 / 16 / 32 / 64 rows, against the packed GEMV,
// the 16-row GEMV and the 256 x 256 tiles: 118 / 131 / 149 / 159 / 174 -> 102 /
// 109 / 116 / 122 / 132 us (6.1 to 4.7 TB/s, of which the fp32 output takes 1
// to 39 MB); N = 20000, K = 1024, 32 rows 19.4 -> 11.7 us.  The others stay
// ahead, and have the shape,
//   - above 24 rows while the 64 x 64 tiles are used (fewer than 96 column
//     tiles of 128; at 24 / 32 / 64 rows N = 12160 runs 14.3 / 14.7 / 15.2 us
//     there and 14.2 / 14.9 / 19.8 here at K = 2048, 7.9 / 8.2 / 8.7 and 7.7 /
//     8.6 / 12.8 at K = 1024);
//   - at K = 1024, above 48 rows while the 256 x 256 tiles make one full round
//     (N = 65536 at 64 rows 32.3 against 33.9 us), and up to 4 rows past 400
//     columns per CU (packed GEMV; N = 151936 at 2 rows 49.1 against 50.1);
//   - at K = 512, where a tile is too short for its barrier (N = 10243, 33
//     rows: 5.1 against 6.8 us).
// At K = 4096 the 16-wave form does not fit a CU's LDS: its ring alone is 256 KB.
static bool vocab_ok(const void* B, int64_t M, int64_t N, int64_t K) {
  const int64_t cus = current_device_cus(), wide = (N + 255) / 256;
  if (!dma_aligned(B) || M < 2 || M > 64 || (K != 1024 && K != 2048) || N * K * 2 >= (1ll << 31) || N <= 40 * cus)
    return false;
  if ((N + 127) / 128 < 96) return M <= 24;
  if (K == 1024) return !(M > 48 && wide >= 224 && wide <= cus) && !(M <= 4 && N > 400 * cus);
  return true;
}

template <int WAVES, int MT, int MODE>
static int launch_vocab_t(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K, void* C,
                          int64_t ldc, hipStream_t s) {
  constexpr int SMEM = Vocab<WAVES, MT>::SMEM;
  static const bool attr = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_vocab_kernel<WAVES, MT, MODE>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
    return true;
  }();
  (void)attr;
  const int64_t groups = int64_t(std::max(current_device_cus(), 1)) * Vocab<WAVES, MT>::PER_CU;
  hipLaunchKernelGGL((gemm_vocab_kernel<WAVES, MT, MODE>), dim3(unsigned(std::min<int64_t>((N + 15) / 16, groups))),
                     dim3(64 * WAVES), SMEM, s, A, lda, B, M, N, K, C, ldc);
  return hip_status("qmoe_gemm(vocab)");
}

template <int WAVES, int MODE>
static int launch_vocab_w(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K, void* C,
                          int64_t ldc, hipStream_t s) {
  return M <= 16   ? launch_vocab_t<WAVES, 1, MODE>(A, lda, B, M, N, K, C, ldc, s)
         : M <= 32 ? launch_vocab_t<WAVES, 2, MODE>(A, lda, B, M, N, K, C, ldc, s)
         : M <= 48 ? launch_vocab_t<WAVES, 3, MODE>(A, lda, B, M, N, K, C, ldc, s)
                   : launch_vocab_t<WAVES, 4, MODE>(A, lda, B, M, N, K, C, ldc, s);
}

template <int MODE>
static int launch_vocab(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K, void* C,
                        int64_t ldc, hipStream_t s) {
  return K == 1024 ? launch_vocab_w<4, MODE>(A, lda, B, M, N, K, C, ldc, s)
                   : launch_vocab_w<8, MODE>(A, lda, B, M, N, K, C, ldc, s);
}

template <int WAVES, int NB, int MT, int MODE>
static int launch_skinny_t(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K, void* C,
                           int64_t ldc, hipStream_t s) {
  constexpr int W_BYTES = WAVES * NB * GV_ROWB, R_BYTES = WAVES * Skinny<WAVES, MT>::CHAINS * MT * 16 * (NB + 1) * 4;
  constexpr int SMEM = W_BYTES > R_BYTES ? W_BYTES : R_BYTES;
  static_assert(SMEM <= 160 * 1024, "LDS");
  static const bool attr = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_skinny_kernel<WAVES, NB, MT, MODE>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
    return true;
  }();
  (void)attr;
  hipLaunchKernelGGL((gemm_skinny_kernel<WAVES, NB, MT, MODE>), dim3(unsigned((N + NB - 1) / NB)), dim3(64 * WAVES),
                     SMEM, s, A, lda, B, M, N, K, C, ldc);
  return hip_status("qmoe_gemm(skinny)");
}

template <int MODE>
static int launch_skinny(int nb, const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K, void* C,
                         int64_t ldc, hipStream_t s) {
#define QMOE_SK(W, NB_)                                                                            \
  if (K == 512 * W && nb == NB_)                                                                   \
    return M <= 16   ? launch_skinny_t<W, NB_, 1, MODE>(A, lda, B, M, N, K, C, ldc, s)              \
           : M <= 32 ? launch_skinny_t<W, NB_, 2, MODE>(A, lda, B, M, N, K, C, ldc, s)              \
           : M <= 48 ? launch_skinny_t<W, NB_, 3, MODE>(A, lda, B, M, N, K, C, ldc, s)              \
                     : launch_skinny_t<W, NB_, 4, MODE>(A, lda, B, M, N, K, C, ldc, s);
#define QMOE_SK_W(W) QMOE_SK(W, 4) QMOE_SK(W, 8) QMOE_SK(W, 16)
  QMOE_SK_W(1)
  QMOE_SK_W(2)
  QMOE_SK_W(4)
  QMOE_SK_W(8)
  QMOE_SK(1, 20)
  QMOE_SK(2, 20)
  QMOE_SK(4, 20)
#undef QMOE_SK_W
#undef QMOE_SK
  return fail(QMOE_ERR_INVALID, "qmoe_gemm: skinny GEMM needs K in {512, 1024, 2048, 4096}");
}

template <int MODE>
static int launch_gemv(const uint16_t* A, int64_t lda, const uint16_t* B, int M, int N, int K,
                       void* C, int64_t ldc, hipStream_t s) {
  const size_t shm = size_t(M) * K * 2;
  const int kc = K / 512;
  if (M >= 2 && M <= 8 && (kc == 1 || kc == 2 || kc == 4 || kc == 8) && int64_t(N) * K * 2 < (1ll << 31))
    return launch_gemv_pk<MODE>(A, lda, B, M, N, K, C, ldc, s);
  if (M >= 2 && (kc == 1 || kc == 2 || kc == 4 || kc == 8))
    return launch_gemv_mfma<MODE>(A, lda, B, M, N, K, C, ldc, s);
  if (kc == 1 || kc == 2 || kc == 4 || kc == 8) {
    if (M <= 1) return launch_gemv_reg<1, MODE>(A, lda, B, M, N, K, C, ldc, s);
    if (M <= 4) return launch_gemv_reg<4, MODE>(A, lda, B, M, N, K, C, ldc, s);
    if (M <= 8) return launch_gemv_reg<8, MODE>(A, lda, B, M, N, K, C, ldc, s);
    return launch_gemv_reg<16, MODE>(A, lda, B, M, N, K, C, ldc, s);
  }
  // 16 rows per workgroup (4 per wave) for wide outputs, and whenever the
  // staged activations are large (fewer workgroups re-staging them)
  const bool wide = N >= 4096 || shm > 16384;
  const int rows_per_block = wide ? 16 : 4;
  dim3 grid((N + rows_per_block - 1) / rows_per_block);
#define QMOE_GEMV(MT)                                                                        \
  if (M <= MT) {                                                                             \
    if (wide)                                                                                \
      hipLaunchKernelGGL((gemv_kernel<MT, 4, MODE>), grid, dim3(256), shm, s, A, lda, B, M, N, \
                         K, C, ldc);                                                         \
    else                                                                                     \
      hipLaunchKernelGGL((gemv_kernel<MT, 1, MODE>), grid, dim3(256), shm, s, A, lda, B, M, N, \
                         K, C, ldc);                                                         \
    return hip_status("qmoe_gemm(gemv)");                                                    \
  }
  QMOE_GEMV(1)
  QMOE_GEMV(2)
  QMOE_GEMV(4)
  QMOE_GEMV(8)
  QMOE_GEMV(16)
#undef QMOE_GEMV
  return fail(QMOE_ERR_INVALID, "qmoe_gemm: gemv path needs M <= 16");
}

int gemm_launch(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t M, int64_t N,
                int64_t K, int mode, void* C, int64_t ldc, hipStream_t s) {
  QMOE_REQUIRE(B && (M == 0 || (A && C)), "qmoe_gemm: null pointer");
  QMOE_REQUIRE(M >= 0 && N > 0 && K > 0, "qmoe_gemm: empty shape M=%lld N=%lld K=%lld",
               (long long)M, (long long)N, (long long)K);
  QMOE_REQUIRE(mode >= 0 && mode <= 2, "qmoe_gemm: bad mode %d", mode);
  QMOE_REQUIRE(lda >= K && ldc >= N, "qmoe_gemm: lda/ldc smaller than the row length");
  QMOE_REQUIRE(lda % 8 == 0, "qmoe_gemm: lda must be a multiple of 8");
  QMOE_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), "qmoe_gemm: dims overflow");
  if (M == 0) return QMOE_OK;
  if (vocab_ok(B, M, N, K)) {
    switch (mode) {
      case QMOE_GEMM_STORE_BF16:
        return launch_vocab<QMOE_GEMM_STORE_BF16>(A, lda, B, int(M), int(N), int(K), C, ldc, s);
      case QMOE_GEMM_STORE_F32:
        return launch_vocab<QMOE_GEMM_STORE_F32>(A, lda, B, int(M), int(N), int(K), C, ldc, s);
      default:
        return launch_vocab<QMOE_GEMM_ADD_F32>(A, lda, B, int(M), int(N), int(K), C, ldc, s);
    }
  }
  if (const int nb = skinny_cols(B, M, N, K); nb && (M - 1) * lda * 2 + K * 2 < (1ll << 31)) {
    switch (mode) {
      case QMOE_GEMM_STORE_BF16:
        return launch_skinny<QMOE_GEMM_STORE_BF16>(nb, A, lda, B, int(M), int(N), int(K), C, ldc, s);
      case QMOE_GEMM_STORE_F32:
        return launch_skinny<QMOE_GEMM_STORE_F32>(nb, A, lda, B, int(M), int(N), int(K), C, ldc, s);
      default:
        return launch_skinny<QMOE_GEMM_ADD_F32>(nb, A, lda, B, int(M), int(N), int(K), C, ldc, s);
    }
  }
  if (M <= 16 && M * K <= 32768) {
    QMOE_REQUIRE(K % 512 == 0, "qmoe_gemm: gemv path needs K %% 512 == 0 (K=%lld)", (long long)K);
    switch (mode) {
      case QMOE_GEMM_STORE_BF16:
        return launch_gemv<QMOE_GEMM_STORE_BF16>(A, lda, B, int(M), int(N), int(K), C, ldc, s);
      case QMOE_GEMM_STORE_F32:
        return launch_gemv<QMOE_GEMM_STORE_F32>(A, lda, B, int(M), int(N), int(K), C, ldc, s);
      default:
        return launch_gemv<QMOE_GEMM_ADD_F32>(A, lda, B, int(M), int(N), int(K), C, ldc, s);
    }
  }
  QMOE_REQUIRE(K % 64 == 0, "qmoe_gemm: K %% 64 != 0 (K=%lld)", (long long)K);
  // DMA offsets are 32-bit with the zero-row marker at 2^31
  QMOE_REQUIRE((M - 1) * lda * 2 + K * 2 < (1ll << 31) && N * K * 2 < (1ll << 31),
               "qmoe_gemm: A or B larger than 2 GiB");
  switch (mode) {
    case QMOE_GEMM_STORE_BF16:
      return launch_tile<QMOE_GEMM_STORE_BF16>(A, lda, B, int(M), int(N), int(K), C, ldc, s);
    case QMOE_GEMM_STORE_F32:
      return launch_tile<QMOE_GEMM_STORE_F32>(A, lda, B, int(M), int(N), int(K), C, ldc, s);
    default:
      return launch_tile<QMOE_GEMM_ADD_F32>(A, lda, B, int(M), int(N), int(K), C, ldc, s);
  }
}

}  // namespace qmoe

namespace qmoe {
template <int MODE>
static int launch_gemv_rms(const float* h, const uint16_t* rms_w, float eps, const uint16_t* B, int N, int K,
                           void* C, hipStream_t s) {
  const dim3 grid(unsigned((N + 3) / 4));
  switch (K / 512) {
#define QMOE_GRMS(KC)                                                                                \
  case KC:                                                                                           \
    hipLaunchKernelGGL((gemv_rms_kernel<KC, MODE>), grid, dim3(256), 0, s, h, rms_w, eps, B, N, C); \
    return hip_status("qmoe_gemv_rmsnorm");
    QMOE_GRMS(1)
    QMOE_GRMS(2)
    QMOE_GRMS(4)
    QMOE_GRMS(8)
#undef QMOE_GRMS
    default:
      return fail(QMOE_ERR_INVALID, "qmoe_gemv_rmsnorm: K must be 512, 1024, 2048 or 4096");
  }
}

int gemv_rmsnorm_launch(const float* h, const uint16_t* rms_w, float eps, const uint16_t* B, int64_t N,
                        int64_t K, int mode, void* C, hipStream_t s) {
  QMOE_REQUIRE(h && rms_w && B && C, "qmoe_gemv_rmsnorm: null pointer");
  QMOE_REQUIRE(N > 0 && N < (1ll << 31), "qmoe_gemv_rmsnorm: bad N");
  QMOE_REQUIRE(K == 512 || K == 1024 || K == 2048 || K == 4096, "qmoe_gemv_rmsnorm: K must be 512, 1024, 2048 or 4096");
  QMOE_REQUIRE(mode >= 0 && mode <= 2, "qmoe_gemv_rmsnorm: bad mode %d", mode);
  QMOE_REQUIRE(eps >= 0.0f, "qmoe_gemv_rmsnorm: eps < 0");
  switch (mode) {
    case QMOE_GEMM_STORE_BF16:
      return launch_gemv_rms<QMOE_GEMM_STORE_BF16>(h, rms_w, eps, B, int(N), int(K), C, s);
    case QMOE_GEMM_STORE_F32:
      return launch_gemv_rms<QMOE_GEMM_STORE_F32>(h, rms_w, eps, B, int(N), int(K), C, s);
    default:
      return launch_gemv_rms<QMOE_GEMM_ADD_F32>(h, rms_w, eps, B, int(N), int(K), C, s);
  }
}
}  // namespace qmoe

extern "C" int qmoe_gemv_rmsnorm(const float* h, const qmoe_bf16* rms_w, float eps, const qmoe_bf16* B,
                                 int64_t N, int64_t K, int mode, void* C, qmoe_stream_t stream) {
  return qmoe::gemv_rmsnorm_launch(h, rms_w, eps, B, N, K, mode, C, qmoe::as_stream(stream));
}

extern "C" int qmoe_gemm(const qmoe_bf16* A, int64_t lda, const qmoe_bf16* B, int64_t M, int64_t N,
                         int64_t K, int mode, void* C, int64_t ldc, qmoe_stream_t stream) {
  return qmoe::gemm_launch(A, lda, B, M, N, K, mode, C, ldc, qmoe::as_stream(stream));
}

extern "C" int64_t qmoe_gemm_ws_workspace(int64_t M, int64_t N, int64_t K) {
  if (M < 0 || N < 0 || K < 0) return -1;
  qmoe::SplitTile tile = qmoe::SPLIT_TINY;
  const int splits = qmoe::splitk_plan(M, N, K, &tile);
  return splits ? int64_t(splits) * M * N * int64_t(sizeof(float)) : 0;
}

extern "C" int qmoe_gemm_ws(const qmoe_bf16* A, int64_t lda, const qmoe_bf16* B, int64_t M, int64_t N,
                            int64_t K, int mode, void* C, int64_t ldc, void* workspace, int64_t workspace_bytes,
                            qmoe_stream_t stream) {
  using namespace qmoe;
  SplitTile tile = SPLIT_TINY;
  const int splits = splitk_plan(M, N, K, &tile);
  const int64_t need = splits ? int64_t(splits) * M * N * int64_t(sizeof(float)) : 0;
  if (splits == 0 || workspace == nullptr || workspace_bytes < need || M >= (1ll << 31) || N >= (1ll << 31))
    return gemm_launch(A, lda, B, M, N, K, mode, C, ldc, as_stream(stream));
  QMOE_REQUIRE(A && B && C, "qmoe_gemm_ws: null pointer");
  QMOE_REQUIRE(mode >= 0 && mode <= 2, "qmoe_gemm_ws: bad mode %d", mode);
  QMOE_REQUIRE(lda >= K && ldc >= N && lda % 8 == 0, "qmoe_gemm_ws: bad lda/ldc");
  QMOE_REQUIRE((M - 1) * lda * 2 + K * 2 < (1ll << 31) && N * K * 2 < (1ll << 31),
               "qmoe_gemm_ws: A or B larger than 2 GiB");
  hipStream_t s = as_stream(stream);
  float* part = static_cast<float*>(workspace);
#define QMOE_SPLIT(MODE)                                                                                    \
  return tile == SPLIT_SMALL ? launch_splitk<SplitSmall, MODE>(A, lda, B, int(M), int(N), int(K), splits, part, C, \
                                                               ldc, s)                                            \
         : tile == SPLIT_MID ? launch_splitk<SplitMid, MODE>(A, lda, B, int(M), int(N), int(K), splits, part, C,   \
                                                             ldc, s)                                              \
                             : launch_splitk<SplitTiny, MODE>(A, lda, B, int(M), int(N), int(K), splits, part, C,  \
                                                              ldc, s);
  switch (mode) {
    case QMOE_GEMM_STORE_BF16:
      QMOE_SPLIT(QMOE_GEMM_STORE_BF16)
    case QMOE_GEMM_STORE_F32:
      QMOE_SPLIT(QMOE_GEMM_STORE_F32)
    default:
      QMOE_SPLIT(QMOE_GEMM_ADD_F32)
  }
#undef QMOE_SPLIT
}

extern "C" int qmoe_gemm_ws_add_rmsnorm(const qmoe_bf16* A, int64_t lda, const qmoe_bf16* B, int64_t M, int64_t N,
                                       int64_t K, float* C, const qmoe_bf16* rms_w, float eps, qmoe_bf16* x_out,
                                       void* workspace, int64_t workspace_bytes, qmoe_stream_t stream) {
  using namespace qmoe;
  QMOE_REQUIRE(B && rms_w && (M == 0 || (A && C && x_out)), "qmoe_gemm_ws_add_rmsnorm: null pointer");
  QMOE_REQUIRE(M >= 0 && M < (1ll << 31) && N > 0 && K > 0, "qmoe_gemm_ws_add_rmsnorm: bad shape");
  QMOE_REQUIRE(N % 4 == 0 && N <= NORM_THREADS * 4 * NORM_MAX_CHUNKS,
               "qmoe_gemm_ws_add_rmsnorm: N must be a multiple of 4 and <= 8192 (N=%lld)", (long long)N);
  QMOE_REQUIRE(eps >= 0.0f, "qmoe_gemm_ws_add_rmsnorm: eps < 0");
  QMOE_REQUIRE(lda >= K && lda % 8 == 0, "qmoe_gemm_ws_add_rmsnorm: bad lda");
  if (M == 0) return QMOE_OK;
  SplitTile tile = SPLIT_TINY;
  const int splits = splitk_plan(M, N, K, &tile);
  const int64_t need = splits ? int64_t(splits) * M * N * int64_t(sizeof(float)) : 0;
  hipStream_t s = as_stream(stream);
  if (splits == 0 || workspace == nullptr || workspace_bytes < need) {
    // no split: the GEMM's own epilogue adds into C, then the norm reads it back
    if (int rc = gemm_launch(A, lda, B, M, N, K, QMOE_GEMM_ADD_F32, C, N, s)) return rc;
    return qmoe_rmsnorm_residual(C, nullptr, rms_w, M, N, eps, nullptr, x_out, stream);
  }
  QMOE_REQUIRE((M - 1) * lda * 2 + K * 2 < (1ll << 31) && N * K * 2 < (1ll << 31),
               "qmoe_gemm_ws_add_rmsnorm: A or B larger than 2 GiB");
  float* part = static_cast<float*>(workspace);
  const uint16_t* w = reinterpret_cast<const uint16_t*>(rms_w);
  uint16_t* xo = reinterpret_cast<uint16_t*>(x_out);
  return tile == SPLIT_SMALL ? launch_splitk<SplitSmall, QMOE_GEMM_ADD_F32>(A, lda, B, int(M), int(N), int(K), splits,
                                                                           part, C, N, s, w, eps, xo)
         : tile == SPLIT_MID ? launch_splitk<SplitMid, QMOE_GEMM_ADD_F32>(A, lda, B, int(M), int(N), int(K), splits,
                                                                         part, C, N, s, w, eps, xo)
                             : launch_splitk<SplitTiny, QMOE_GEMM_ADD_F32>(A, lda, B, int(M), int(N), int(K),
                                                                          splits, part, C, N, s, w, eps, xo);
}
