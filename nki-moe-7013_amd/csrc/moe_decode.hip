// Decode-shape expert MLPs driven by dispatch metadata (T <= 64 tokens):
// HBM-bound GEMVs, each touched expert's weights streamed from HBM once.
//
//   moe_gateup_gemv_kernel   act[s,i] = silu(x.Wg[e,i]) * (x.Wu[e,i]) (fp32).
//                            The expert's gate/up rows go into registers and are
//                            applied to the expert's (few) token rows staged in LDS.
//   moe_down_mfma_kernel     y_slot[s,h] = bf16(act[s]).W2[e,h] (fp32 accumulation)
//                            on MFMA, from the blocked w2 layout [E][I/8][H][8].
//
// Grid: (row group, active-expert slot); slots beyond the number of touched
// experts (meta[1]) exit at once, so the host sizes the grid as min(E, T*k)
// without knowing the routing.  Row groups are the fastest index: an expert's
// workgroups then go round the 8 XCDs (with 128 slots fastest, each expert
// had its XCD and a crowded one kept it busy alone: 48 tokens, 46 of them in
// one expert, 237 -> 139 us; equally popular experts 177 -> 172 us at 32).
// (The T <= 8 fused block is moe_block_decode.hip.)
#include "decode_util.hpp"
#include "mfma_pipe.hpp"

namespace qmoe {

// ================================================================== gate/up
// Workgroup: 8 intermediate units (i0 = 8*blockIdx.x); wave w: units i0+2w,
// i0+2w+1 = 2 gate rows + the 2 matching up rows of the packed w13, all in
// registers (whole 1 KB row pieces per load, requested at once).  The
// expert's tokens pass over them GU_TOK_CHUNK at a time: wave w copies token
// c0 + w by LDS-DMA, the next chunk's copy in flight behind this chunk's dots
// (v_dot2 on packed bf16 pairs, a wave reduction per row).  Bound by HBM
// where experts hold a few tokens (16 tokens, 83 experts: 86 us for 522 MB).
// A crowded expert's chunks used to wait for one copy after another: 32
// tokens with 93 experts touched, 18 tokens in the largest, took 162 us for
// 585 MB; 48 tokens with 46 in the largest 300 us.
// Two chunks of 4 tokens (32 KB at H = 2048) leave room for five workgroups
// per CU, so each new workgroup's dependent first loads (routing metadata,
// then its expert's rows) overlap the others' weight streams.
// (The rows as MFMA operands straight from global memory ran 5.2 TB/s
// whatever the tile: 16 rows x 64 bytes per load are half lines.)
constexpr int GU_TOK_CHUNK = 4;

// DMA = false (x not 16-byte aligned): the copies go through registers.
template <int HC, bool DMA>
__global__ __launch_bounds__(256) void moe_gateup_gemv_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w13,
    const int32_t* __restrict__ offsets, const int32_t* __restrict__ slot_token,
    const int32_t* __restrict__ active, const int32_t* __restrict__ meta, int T, int I,
    float* __restrict__ act) {
  constexpr int H = HC * 512, TC = GU_TOK_CHUNK;
  __shared__ __attribute__((aligned(1024))) uint16_t xs[2][TC][H];
  // both requested before the branch (active has E >= gridDim.x entries)
  const int n_active = meta[1], e = active[blockIdx.y];
  if (int(blockIdx.y) >= n_active) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int i_base = blockIdx.x * 8 + wave * 2;
  const int grp = i_base / 32, off = i_base % 32;
  const uint16_t* we = w13 + int64_t(e) * 2 * I * H;
  u32x4 w[4][HC];  // rows: gate i_base, gate i_base+1, up i_base, up i_base+1
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int prow = grp * 64 + (r < 2 ? 0 : 32) + off + (r & 1);
    const uint16_t* p = we + int64_t(prow) * H + lane * 8;
#pragma unroll
    for (int c = 0; c < HC; ++c) w[r][c] = ld_stream(p + c * 512);
  }
  const int s0 = offsets[e], s1 = offsets[e + 1];
  const pipe::i32x4 rx = pipe::make_rsrc(x, uint32_t(T) * uint32_t(H) * 2u);
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(&xs[0][wave][0]));
  int tok = slot_token[min(s0 + wave, s1 - 1)];  // this wave's token of the next chunk to copy
  auto copy = [&](int c0, int buf) {
    if (c0 + wave < s1) {  // wave-uniform
#pragma unroll
      for (int c = 0; c < HC; ++c)
        if constexpr (DMA)
          pipe::dma16(lds0 + uint32_t(buf * TC * H * 2 + c * 1024), uint32_t(lane * 16),
                      rx, uint32_t(tok) * uint32_t(H * 2) + uint32_t(c * 1024));
        else
          *reinterpret_cast<u32x4*>(&xs[buf][wave][c * 512 + lane * 8]) = ld16(x + int64_t(tok) * H + c * 512 + lane * 8);
    }
    tok = slot_token[min(c0 + TC + wave, s1 - 1)];
  };
  copy(s0, 0);
  int buf = 0;
  for (int c0 = s0; c0 < s1; c0 += TC, buf ^= 1) {
    const int n = min(TC, s1 - c0);
    pipe::wait_vm<0>();  // this wave's part of the chunk (and its weights) has landed
    lds_barrier();       // everyone's; and the other buffer's readers are done
    if (c0 + TC < s1) copy(c0 + TC, buf ^ 1);
    for (int j = 0; j < n; ++j) {
      float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int c = 0; c < HC; ++c) {
        const u32x4 xv = *reinterpret_cast<const u32x4*>(&xs[buf][j][c * 512 + lane * 8]);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = dot8_bf16(w[r][c], xv, acc[r]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = wave_sum(acc[r]);
      if (lane < 2) {
        const float g = lane ? acc[1] : acc[0];
        const float u = lane ? acc[3] : acc[2];
        act[int64_t(c0 + j) * I + i_base + lane] = silu(g) * u;
      }
    }
  }
}

// ================================================================== down
// Workgroup: (active-expert slot, 64 output columns); wave w owns the 16
// columns h = 64*blockIdx.x + 16*w + l%16 and computes, on
// v_mfma_f32_16x16x32_bf16, y[token][h] for up to 16 of the expert's tokens
// at a time:
//   A (16 x 32): the tokens' fp32 SwiGLU activations as two bf16 parts,
//       hi = bf16(a) and lo = bf16(a - hi), one MFMA each (rows past the
//       expert's count are zeros), staged in LDS; lane l -> token l % 16, k
//       offset (l / 16) * 8.  hi + lo carries 16 significant bits, so the
//       product keeps the fp32-activation accuracy of this path;
//   B (16 x 32): the weights, lane l -> column l % 16 and the 8 units of
//       blocked-w2 block 4*ks + l/16 ([I/8][H][8]: 16 contiguous bytes, so
//       the 16 columns of one block are 256 contiguous bytes).
// The weights stream in batches of DN_KB k-steps, two of them requested before
// the activations are staged (32 tokens 170.7 -> 169.2 us with gate/up, 48 187.0 -> 185.2).
constexpr int DN_KB = 6;                // k-steps of 32 per weight batch (two in flight from the start; 12: 5% slower, fewer waves)
constexpr int DN_COLS = 64;             // output columns per workgroup
constexpr int DN_ROWS = 16;             // tokens per MFMA pass

__global__ __launch_bounds__(256) void moe_down_mfma_kernel(
    const float* __restrict__ act, const uint16_t* __restrict__ w2b,
    const int32_t* __restrict__ offsets, const int32_t* __restrict__ active,
    const int32_t* __restrict__ meta, int H, int I, float* __restrict__ y_slot) {
  extern __shared__ __attribute__((aligned(16))) uint16_t as[];  // hi, lo: [2][DN_ROWS][I + 8] bf16
  const int n_active = meta[1], e = active[blockIdx.y];  // both requested before the branch
  if (int(blockIdx.y) >= n_active) return;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, col = lane & 15, kq = lane >> 4;
  const int h = blockIdx.x * DN_COLS + wave * 16 + col;
  const int NS = I / QMOE_W2_BLOCK, KS = I / 32, ald = I + 8;
  const int nkb = (KS + DN_KB - 1) / DN_KB;
  // block kb = 4*ks + kq of column h: w2b[((e*NS + kb)*H + h)*8 .. +8]
  const uint16_t* wp = w2b + ((int64_t(e) * NS + kq) * H + h) * QMOE_W2_BLOCK;
  const int64_t ks_stride = int64_t(4) * H * QMOE_W2_BLOCK;
  u32x4 wa[2][DN_KB];
  auto load = [&](u32x4 (&dst)[DN_KB], int kb) {
#pragma unroll
    for (int u = 0; u < DN_KB; ++u) {
      const int ks = kb * DN_KB + u;
      dst[u] = ks < KS ? ld_stream(wp + ks * ks_stride) : u32x4{0u, 0u, 0u, 0u};
    }
  };
  const int s0 = offsets[e], s1 = offsets[e + 1];
  for (int c0 = s0; c0 < s1; c0 += DN_ROWS) {
    const int n = min(DN_ROWS, s1 - c0);
    load(wa[0], 0);
    if (nkb > 1) load(wa[1], 1);
    lds_barrier();  // the previous pass's fragment reads are done
    // act rows -> bf16 hi / lo parts in LDS; 4 floats per chunk, all loads
    // before the stores
    const int i4 = I / 4, total = DN_ROWS * i4;
    constexpr int SI = 6;
    for (int q0 = t; q0 < total; q0 += 256 * SI) {
      float4 v[SI];
#pragma unroll
      for (int u = 0; u < SI; ++u) {
        const int q = q0 + u * 256, j = q / i4, c = q - j * i4;
        v[u] = (q < total && j < n) ? reinterpret_cast<const float4*>(act + int64_t(c0 + j) * I)[c]
                                    : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      }
#pragma unroll
      for (int u = 0; u < SI; ++u) {
        const int q = q0 + u * 256, j = q / i4, c = q - j * i4;
        if (q < total) {
          const uint32_t h01 = pack_bf16x2(v[u].x, v[u].y), h23 = pack_bf16x2(v[u].z, v[u].w);
          *reinterpret_cast<uint2*>(as + j * ald + c * 4) = make_uint2(h01, h23);
          *reinterpret_cast<uint2*>(as + (DN_ROWS + j) * ald + c * 4) =
              make_uint2(pack_bf16x2(v[u].x - bf16_lo(h01), v[u].y - bf16_hi(h01)),
                         pack_bf16x2(v[u].z - bf16_lo(h23), v[u].w - bf16_hi(h23)));
        }
      }
    }
    lds_barrier();
    f32x4 acc = f32x4{};
    const uint16_t* ap = as + col * ald + kq * 8;
    auto step = [&](const u32x4 (&src)[DN_KB], int kb) {
#pragma unroll
      for (int u = 0; u < DN_KB; ++u) {
        const int ks = kb * DN_KB + u;
        if (ks < KS) {
          const u32x4 ahi = *reinterpret_cast<const u32x4*>(ap + ks * 32);
          const u32x4 alo = *reinterpret_cast<const u32x4*>(ap + DN_ROWS * ald + ks * 32);
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ahi),
                                                        __builtin_bit_cast(bf16x8, src[u]), acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, alo),
                                                        __builtin_bit_cast(bf16x8, src[u]), acc, 0, 0, 0);
        }
      }
    };
    for (int kb = 0; kb < nkb; kb += 2) {
      step(wa[0], kb);
      if (kb + 2 < nkb) load(wa[0], kb + 2);
      if (kb + 1 < nkb) {
        step(wa[1], kb + 1);
        if (kb + 3 < nkb) load(wa[1], kb + 3);
      }
    }
    // lane l holds column h and tokens kq*4 + 0..3
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = kq * 4 + r;
      if (j < n) y_slot[int64_t(c0 + j) * H + h] = acc[r];
    }
  }
}

// ================================================================== launchers
static int check_dec_shapes(const char* fn, int64_t T, int64_t H, int64_t I, int64_t E, int64_t k) {
  QMOE_REQUIRE(T >= 0 && T <= DEC_MAX_T, "%s: T must be <= 64 (T=%lld)", fn, (long long)T);
  QMOE_REQUIRE(E > 0 && E <= 256 && k > 0 && k <= E, "%s: bad E/k", fn);
  QMOE_REQUIRE(H % 512 == 0 && H >= 512 && H <= 4096 && (H / 512 & (H / 512 - 1)) == 0,
               "%s: H must be 512, 1024, 2048 or 4096 (H=%lld)", fn, (long long)H);
  QMOE_REQUIRE(I % 32 == 0 && I > 0 && I <= 1536, "%s: I must be a multiple of 32, <= 1536", fn);
  return QMOE_OK;
}

static int launch_experts(const uint16_t* x, const uint16_t* w13, const uint16_t* w2,
                          const int32_t* offsets, const int32_t* slot_token, const int32_t* active,
                          const int32_t* meta, int64_t T, int64_t H, int64_t I, int64_t E, int64_t k,
                          float* act, float* y_slot, hipStream_t s) {
  const unsigned nact = unsigned(std::min<int64_t>(E, T * k));
  dim3 g1(unsigned(I / 8), nact);
  switch (H / 512) {
#define QMOE_GU(HC)                                                                                  \
  case HC:                                                                                           \
    if (reinterpret_cast<uintptr_t>(x) % 16 == 0)                                                    \
      hipLaunchKernelGGL((moe_gateup_gemv_kernel<HC, true>), g1, dim3(256), 0, s, x, w13, offsets,   \
                         slot_token, active, meta, int(T), int(I), act);                             \
    else                                                                                             \
      hipLaunchKernelGGL((moe_gateup_gemv_kernel<HC, false>), g1, dim3(256), 0, s, x, w13, offsets,  \
                         slot_token, active, meta, int(T), int(I), act);                             \
    break;
    QMOE_GU(1)
    QMOE_GU(2)
    QMOE_GU(4)
    QMOE_GU(8)
#undef QMOE_GU
  }
  int rc = hip_status("moe experts (gate_up)");
  if (rc) return rc;
  const size_t shm2 = size_t(2 * DN_ROWS) * (I + 8) * 2;
  dim3 g2(unsigned(H / DN_COLS), nact);
  hipLaunchKernelGGL(moe_down_mfma_kernel, g2, dim3(256), shm2, s, act, w2, offsets, active, meta, int(H),
                     int(I), y_slot);
  return hip_status("moe experts (down)");
}

}  // namespace qmoe

using namespace qmoe;

extern "C" int qmoe_moe_experts_gemv(const qmoe_bf16* x, const qmoe_bf16* w13,
                                     const qmoe_bf16* w2, const int32_t* offsets,
                                     const int32_t* slot_token, const int32_t* active,
                                     const int32_t* meta, int64_t T, int64_t H, int64_t I,
                                     int64_t E, int64_t k, float* act, float* y_slot,
                                     qmoe_stream_t stream) {
  QMOE_REQUIRE(w13 && w2 && offsets && active && meta && (T == 0 || (x && slot_token && act && y_slot)),
               "qmoe_moe_experts_gemv: null pointer");
  int rc = check_dec_shapes("qmoe_moe_experts_gemv", T, H, I, E, k);
  if (rc) return rc;
  if (T == 0) return QMOE_OK;
  return launch_experts(x, w13, w2, offsets, slot_token, active, meta, T, H, I, E, k, act, y_slot,
                        as_stream(stream));
}

