// Everything of a transformer block after its attention, in one launch, for d_model 128 and
// ffn_dim 128 (the loop body of the reference's _run_fused after the attention,
// torch_transformer_benchmark.py:1255-1290: _tl_linear_ln, _tl_linear(gelu), _tl_linear_ln):
//
//   r1  = resid + mask_branch(ctx W_o^T + b_o)        (fp32)
//   h2  = LN2(r1)                                     (fp16)
//   f   = gelu(h2 W1^T + b1)                          (fp16, exact erf GELU)
//   r2  = (r1 + f W2^T + b2) * row_valid              (fp32 -> r_out, optional)
//   out = LNn(r2) [* row_valid]                       (fp16 or fp32)
//
// Bound by memory: a row costs 256 B of ctx and 512 B of resid in, 512 B of r and 256 B of
// out back.  As three launches it also wrote and read h2 and f (1 KB a row) and the
// residual twice more (1 KB).  65536 rows: 57 us as three launches, 31 us as this one; 262144
// rows: 240 and 108 us (3.7 TB/s: past a fixed cost of ~5 us for the weights, the first tiles
// and the launch, 26 us for each 65536 rows, 14 of them vector arithmetic); 1024 rows, where
// launches count: 30 and 14 us.
//
// Persistent workgroups of four waves walk 32-row blocks.  Wave w owns output features
// 32w .. 32w+31 of all three products and keeps those rows of W_o, W1 and W2 in registers
// (96 VGPRs) as A operands, so weights are read once per workgroup; activations pass between
// the waves through LDS.  Accumulators hold products transposed: lane (li, g) owns token li
// and, per quad q, features 32w + 8q + 4g .. + 3; r1 and r2 never leave those registers but
// for the final store.  LayerNorm statistics: each wave reduces its 32 features of a token
// to (mean, M2), the four pairs meet in LDS and combine exactly (Chan et al.).
//
// LDS (62 KB; with 230 VGPRs two workgroups per CU, which overlap one another's transfers,
// barriers and arithmetic; three per CU at 168 VGPRs spilled 36 to 64 of them): the ctx and
// resid tiles arrive by LDS-DMA with 16-byte chunks XOR-swizzled by row (conflict-free for
// both the operand reads and the per-lane residual reads); r2 is staged in the resid tile's
// place and out in h2's, and both leave as whole rows.  The next block's resid goes to a
// second tile from the block's start (one tile, fetched after r2 had left it, cost 6% at
// 262144 rows) and its ctx follows once this block's has been read.
#include "common.hpp"
#include "kernels.hpp"
#include "lds_dma.hpp"

namespace cobra {

namespace {

constexpr int kBtD = 128;               // d_model and ffn_dim
constexpr int kBtRows = 32;             // rows per block
constexpr int kBtCtx = 0;               // [32][128] fp16
constexpr int kBtH = 8192;              // [32][128] fp16: h2, then out
constexpr int kBtF = 2 * 8192;          // [32][128] fp16: f
constexpr int kBtRes = 3 * 8192;        // two of [32][128]: resid dtype, then r2 (or out) in fp32
constexpr int kBtStat = kBtRes + 32768; // [2][4 waves][32 tokens] (mean, M2)
constexpr int kBtPar = kBtStat + 2048;  // [7][128] fp32 parameters
constexpr int kBtLds = kBtPar + 7 * kBtD * 4;
enum { kParBo, kParG2, kParB2n, kParB1, kParB2, kParGn, kParBn };

// Byte offset of 16-byte chunk c of row r: rows of 16 chunks (fp16), rows of 32 (fp32).
__device__ __forceinline__ int row16(int r, int c) { return r * 256 + 16 * (c ^ (r & 15)); }
__device__ __forceinline__ int row32(int r, int c) { return r * 512 + 16 * (c ^ (r & 7)); }

}  // namespace

template <typename TR, typename TY, bool MASKED>
__global__ __launch_bounds__(256, 2) void block_tail_kernel(BlockTailArgs a) {
  __shared__ __attribute__((aligned(1024))) char smem[kBtLds];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 31, g = lane >> 5;
  const int64_t nblk = (a.M + kBtRows - 1) / kBtRows;
  const uint32_t lds0 = lds_addr(smem);
  const f16* ctx = static_cast<const f16*>(a.ctx);
  const TR* resid = static_cast<const TR*>(a.resid);
  TY* out = static_cast<TY*>(a.out);

  // Transfers: 1 KB bands, lane-contiguous in LDS; rows past M read row M - 1.
  auto fetch_ctx = [&](int64_t m0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int band = 2 * w + i, row = 4 * band + (lane >> 4), c = (lane & 15) ^ (row & 15);
      dma16_untracked(ctx + min(m0 + row, a.M - 1) * kBtD + 8 * c, lds0 + kBtCtx + band * 1024);
    }
  };
  auto fetch_res = [&](int64_t m0, int tile) {
    if constexpr (sizeof(TR) == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int band = 4 * w + i, row = 2 * band + (lane >> 5), c = (lane & 31) ^ (row & 7);
        dma16_untracked(resid + min(m0 + row, a.M - 1) * kBtD + 4 * c, lds0 + tile + band * 1024);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int band = 2 * w + i, row = 4 * band + (lane >> 4), c = (lane & 15) ^ (row & 15);
        dma16_untracked(resid + min(m0 + row, a.M - 1) * kBtD + 8 * c, lds0 + tile + band * 1024);
      }
    }
  };

  int64_t blk = blockIdx.x;
  uint8_t mask_byte = 0;
  auto fetch_mask = [&](int64_t m0) {
    if constexpr (MASKED) mask_byte = a.row_mask[min(m0 + li, a.M - 1)];
  };
  // The first tiles go out ahead of the weights: one latency, not two.
  fetch_mask(blk * kBtRows);
  fetch_ctx(blk * kBtRows);
  fetch_res(blk * kBtRows, kBtRes);

  // Weight rows 32w + li as A operands, and the parameters into LDS.
  f16x8 wo[8], w1[8], w2[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    const int64_t at = (int64_t)(32 * w + li) * kBtD + 16 * ks + 8 * g;
    wo[ks] = *reinterpret_cast<const f16x8*>(static_cast<const f16*>(a.w_o) + at);
    w1[ks] = *reinterpret_cast<const f16x8*>(static_cast<const f16*>(a.w1) + at);
    w2[ks] = *reinterpret_cast<const f16x8*>(static_cast<const f16*>(a.w2) + at);
  }
  float* par = reinterpret_cast<float*>(smem + kBtPar);
  {
    const float* src[7] = {a.b_o, a.ln2_w, a.ln2_b, a.b1, a.b2, a.lnn_w, a.lnn_b};
#pragma unroll
    for (int p = 0; p < 7; ++p)
      if (threadIdx.x < kBtD) par[p * kBtD + threadIdx.x] = src[p][threadIdx.x];
  }
  auto param = [&](int p, int q) { return *reinterpret_cast<const f32x4*>(par + p * kBtD + 32 * w + 8 * q + 4 * g); };
  // The product of this wave's rows of a weight matrix with an activation tile in LDS.
  auto product = [&](const f16x8(&wt)[8], int tile) {
    f32x16 acc = zero16();
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
      acc = mfma32x32x16(wt[ks], *reinterpret_cast<const f16x8*>(smem + tile + row16(li, 2 * ks + g)), acc);
    return acc;
  };
  // (mean, M2) of this wave's 32 features of token li, published; then, past a barrier, the
  // row's mean and 1 / sigma.
  f32x2* stat = reinterpret_cast<f32x2*>(smem + kBtStat);
  auto publish = [&](const f32x16& r, int slot) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) s += r[i];
    const float mean = sum_xor32(s) * (1.0f / 32);
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) q += (r[i] - mean) * (r[i] - mean);
    q = sum_xor32(q);
    if (g == 0) stat[(slot * 4 + w) * 32 + li] = f32x2{mean, q};
  };
  auto combine = [&](int slot, float& mean, float& rstd) {
    f32x2 p[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) p[j] = stat[(slot * 4 + j) * 32 + li];
    mean = (p[0].x + p[1].x + p[2].x + p[3].x) * 0.25f;
    float m2 = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) m2 += p[j].y + 32.f * (p[j].x - mean) * (p[j].x - mean);
    rstd = rsqrtf(m2 * (1.0f / kBtD) + a.eps);
  };

  wait_vmcnt<0>();
  int res = kBtRes;
  for (; blk < nblk; blk += gridDim.x, res = 2 * kBtRes + 16384 - res) {
    const int64_t m0 = blk * kBtRows, next = (blk + gridDim.x) * kBtRows;
    const bool more = blk + gridDim.x < nblk;
    const float mv = !MASKED || mask_byte != 0 ? 1.f : 0.f;
    lds_barrier();  // every wave's part of the tiles has landed (and the parameters)
    if (more) {
      fetch_mask(next);
      fetch_res(next, 2 * kBtRes + 16384 - res);
    }

    // r1 = resid + branch
    const f32x16 o = product(wo, kBtCtx);
    f32x16 r;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f32x4 x;
      if constexpr (sizeof(TR) == 4) {
        x = *reinterpret_cast<const f32x4*>(smem + res + row32(li, 8 * w + 2 * q + g));
      } else {
        const f16x4 h = *reinterpret_cast<const f16x4*>(smem + res + row16(li, 4 * w + q) + 8 * g);
        x = f32x4{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
      }
      const f32x4 b = param(kParBo, q);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = o[4 * q + e] + b[e];
        if constexpr (MASKED) v = mv == 0.f ? 0.f : v;
        r[4 * q + e] = v + x[e];
      }
    }
    publish(r, 0);
    lds_barrier();
    if (more) fetch_ctx(next);
    float mean, rstd;
    combine(0, mean, rstd);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 gm = param(kParG2, q), bt = param(kParB2n, q);
      f16x4 h;
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = (f16)((r[4 * q + e] - mean) * rstd * gm[e] + bt[e]);
      *reinterpret_cast<f16x4*>(smem + kBtH + row16(li, 4 * w + q) + 8 * g) = h;
    }
    lds_barrier();
    const f32x16 u = product(w1, kBtH);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 b = param(kParB1, q);
      f16x4 h;
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = (f16)gelu_erf(u[4 * q + e] + b[e]);
      *reinterpret_cast<f16x4*>(smem + kBtF + row16(li, 4 * w + q) + 8 * g) = h;
    }
    lds_barrier();
    const f32x16 y = product(w2, kBtF);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 b = param(kParB2, q);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = y[4 * q + e] + b[e] + r[4 * q + e];
        if constexpr (MASKED) v *= mv;
        r[4 * q + e] = v;
      }
      if (a.r_out)
        *reinterpret_cast<f32x4*>(smem + res + row32(li, 8 * w + 2 * q + g)) =
            f32x4{r[4 * q], r[4 * q + 1], r[4 * q + 2], r[4 * q + 3]};
    }
    publish(r, 1);
    lds_barrier();
    combine(1, mean, rstd);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 gm = param(kParGn, q), bt = param(kParBn, q);
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = (r[4 * q + e] - mean) * rstd * gm[e] + bt[e];
        if constexpr (MASKED) v[e] = a.mask_out ? v[e] * mv : v[e];
      }
      if constexpr (sizeof(TY) == 4) {  // r_out is null: its place is free
        *reinterpret_cast<f32x4*>(smem + res + row32(li, 8 * w + 2 * q + g)) = v;
      } else {
        *reinterpret_cast<f16x4*>(smem + kBtH + row16(li, 4 * w + q) + 8 * g) =
            f16x4{(f16)v[0], (f16)v[1], (f16)v[2], (f16)v[3]};
      }
    }
    lds_barrier();
    // Whole rows out: a pass of the workgroup is 8 fp32 rows or 16 fp16 rows.
    const int t = threadIdx.x;
    f32x4 rv[4], hv[2];
    if (a.r_out || sizeof(TY) == 4)
#pragma unroll
      for (int p = 0; p < 4; ++p) rv[p] = *reinterpret_cast<const f32x4*>(smem + res + row32(8 * p + t / 32, t % 32));
    if constexpr (sizeof(TY) == 2)
#pragma unroll
      for (int p = 0; p < 2; ++p) hv[p] = *reinterpret_cast<const f32x4*>(smem + kBtH + row16(16 * p + t / 16, t % 16));
    // Only the very last block is ragged, and no block follows it in its workgroup, so the
    // count of stores behind the transfers is the same whenever it is waited for.
    float* const r_dst = sizeof(TY) == 4 ? reinterpret_cast<float*>(out) : a.r_out;
    if (m0 + kBtRows <= a.M) {
      if (r_dst)
#pragma unroll
        for (int p = 0; p < 4; ++p) *reinterpret_cast<f32x4*>(r_dst + (m0 + 8 * p + t / 32) * kBtD + 4 * (t % 32)) = rv[p];
      if constexpr (sizeof(TY) == 2)
#pragma unroll
        for (int p = 0; p < 2; ++p) *reinterpret_cast<f32x4*>(out + (m0 + 16 * p + t / 16) * kBtD + 8 * (t % 16)) = hv[p];
    } else {
      if (r_dst)
#pragma unroll
        for (int p = 0; p < 4; ++p)
          if (m0 + 8 * p + t / 32 < a.M)
            *reinterpret_cast<f32x4*>(r_dst + (m0 + 8 * p + t / 32) * kBtD + 4 * (t % 32)) = rv[p];
      if constexpr (sizeof(TY) == 2)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          if (m0 + 16 * p + t / 16 < a.M)
            *reinterpret_cast<f32x4*>(out + (m0 + 16 * p + t / 16) * kBtD + 8 * (t % 16)) = hv[p];
    }
    // Everything older than this block's stores, the next block's transfers among it.
    if constexpr (sizeof(TY) == 4) {
      wait_vmcnt<4>();
    } else if (a.r_out) {
      wait_vmcnt<6>();
    } else {
      wait_vmcnt<2>();
    }
  }
}

template <typename TR, typename TY>
static hipError_t launch_block_tail(const BlockTailArgs& a, unsigned grid) {
  if (a.row_mask)
    hipLaunchKernelGGL((block_tail_kernel<TR, TY, true>), dim3(grid), dim3(256), 0, a.stream, a);
  else
    hipLaunchKernelGGL((block_tail_kernel<TR, TY, false>), dim3(grid), dim3(256), 0, a.stream, a);
  return hipGetLastError();
}

// 128 is where a wave's rows of all three weights fit its registers and 32 whole rows of
// every intermediate fit LDS; wider blocks take the separate GEMM and LayerNorm launches.
bool block_tail_ok(int64_t d_model, int64_t ffn_dim) { return d_model == kBtD && ffn_dim == kBtD; }

hipError_t run_block_tail(const BlockTailArgs& a) {
  if (a.M < 0 || (a.out_dtype == kF32 && a.r_out) || (a.mask_out && !a.row_mask)) return hipErrorInvalidValue;
  if (a.M == 0) return hipSuccess;
  // Two workgroups per CU (registers and LDS), each walking an equal share of the blocks.
  const int64_t nblk = (a.M + kBtRows - 1) / kBtRows, slots = 2 * (int64_t)compute_units();
  const int64_t rounds = (nblk + slots - 1) / slots;
  const unsigned grid = (unsigned)((nblk + rounds - 1) / rounds);
  const bool r16 = a.resid_dtype == kF16, y16 = a.out_dtype == kF16;
  if (r16) return y16 ? launch_block_tail<f16, f16>(a, grid) : launch_block_tail<f16, float>(a, grid);
  return y16 ? launch_block_tail<float, f16>(a, grid) : launch_block_tail<float, float>(a, grid);
}

}  // namespace cobra
