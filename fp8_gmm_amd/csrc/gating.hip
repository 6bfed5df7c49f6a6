// The backward pass of a router's gating linear, for gfx950: logits = x W^T with a few experts (the gating_network of
// the reference's example layers, fp8_gmm/example.py:38,47,76,84,109,112; there torch's linear and its autograd).
//
//   grad_W[e, :] = sum_t g[t, e] * x[t, :]                 a contraction over the tokens with at most 128 rows
//   grad_x[t, :] = grad_in[t, :] + sum_e g[t, e] * W[e, :]  the other gradient of x added on the way
//
// Both are bound by the rows of x and of its gradient, which pass once; the products are v_mfma_f32_16x16x32_bf16 and
// hide behind the loads.  A row of a fragment may be any expert and a column any token or column of x, as long as
// both operands agree, so the assignment below is the one that makes a lane's accumulators consecutive in memory.
// Measured, microseconds, operands from HBM, against the library's products and torch's addition behind the one of x
// (some 22 of which per product are its host path, where it is the longer one):
//   tokens, hidden, experts   grad_x + grad_in        with grad_W as well
//   16384, 4096, 16           65    (library 108)     99    (185)        134 MB read, 134 MB written; 134 MB more read
//   16384, 4096, 64           78    (95)              130   (227)
//   16384, 4096, 72, 104      79    (111, 116)        165   (242, 249)
//   16384, 4096, 66, 100      119, 131 (112, 116)     201, 211 (243, 249)
//   16384, 4096, 65, 127      143, 152 (115, 125)     228, 238 (254, 270)
//   4096, 4096, 64, 72, 100   24, 30, 40 (32, 37, 37) 44, 65, 76 (61, 65, 66)
//   8192, 4096, 65, 100       81, 70 (65, 65)         134, 120 (137, 135)
//   4096, 2048, 65, 100       30, 24 (28, 29)         57, 52 (64, 59)
//   4096, 8192, 64, 72, 100   39, 45, 67 (55, 63, 65) 68, 96, 117 (84, 92, 95)
//   1024, 16384, 63, 104      33, 28 (36, 36)         52, 64 (53, 52)
//   16384, 1024, 63, 65       33, 50 (38, 39)         54, 86 (181, 172)
//   1531, 1024, 16, 65        5, 12 (22)              11, 25 (42)
//   64, 4096, 16, 127         4, 7 (22)               7, 16 (42)
#include <algorithm>

#include "device_utils.h"

namespace fp8gmm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kGateMaxExperts = 128;
constexpr int kGateWaves = 4;      // wavefronts per workgroup
constexpr int kGateCols = 64;      // columns of x per wavefront
constexpr int kGateStep = 32;      // tokens per product of the weight gradient
constexpr int kGateBlocks = 1024;  // workgroups wanted: four per compute unit
// More experts than this: two workgroups per compute unit fit, and the sums of a slice of tokens weigh more.  Half the
// slices: 4096 x 4096, 128 experts 56 -> 38 us; 16384 x 4096, 64 and 128 experts 56 -> 51 and 100 -> 82 us.
constexpr int kGateManyExperts = 32;
constexpr int kGateRows = 16;      // tokens per product of the input gradient

__device__ __forceinline__ uint32_t load_u16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0);
}
__device__ __forceinline__ f32x4 product(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// One workgroup: 64 columns of x, `steps` * 128 tokens from blockIdx.y * that, a quarter of them per wavefront.  Lane
// (q, c) = (lane / 16, lane % 16) loads four columns of eight tokens; two of its dwords of neighbouring tokens make one
// of each fragment, so that nothing passes through LDS before the sum over the four wavefronts.  One slice of tokens:
// the result itself, otherwise fp32 sums for gating_sum_kernel, in [slice][expert][hidden].
template <int TILES>  // 16 experts each
__global__ __launch_bounds__(kGateWaves * 64) void gating_wgrad_kernel(const uint16_t* __restrict__ grad,
                                                                       const uint16_t* __restrict__ x, int tokens,
                                                                       int hidden, int experts, int steps,
                                                                       float* __restrict__ sums,
                                                                       uint16_t* __restrict__ out) {
  __shared__ f32x4 part[kGateWaves][4][64];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int q = lane / 16, c = lane % 16;
  const int block_tokens = steps * kGateStep * kGateWaves;
  const int t0 = blockIdx.y * block_tokens;
  const int rows = min(block_tokens, tokens - t0);
  const int col = blockIdx.x * kGateCols + c * 4;
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(x + (size_t)t0 * hidden, (uint32_t)rows * hidden * 2u);
  const __amdgpu_buffer_rsrc_t rg = make_rsrc(grad + (size_t)t0 * experts, (uint32_t)rows * experts * 2u);
  f32x4 acc[TILES][4];
#pragma unroll
  for (int m = 0; m < TILES; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[m][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x2 v[8];
  uint32_t g[TILES][8];
  // the loads of a step are issued before the products of the step before; past the last step there are none
  const auto load = [&](int s) {
    const int t = (wave * steps + s) * kGateStep + q * 8;  // of the workgroup's rows; past them both operands are zero
    const bool any = s < steps;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = buf_load8_stream(rx, any && col < hidden ? ((uint32_t)(t + j) * hidden + col) * 2u : kOobOffset);
#pragma unroll
    for (int m = 0; m < TILES; ++m)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        g[m][j] = load_u16(rg, any && m * 16 + c < experts ? ((uint32_t)(t + j) * experts + m * 16 + c) * 2u : kOobOffset);
  };
  load(0);
  for (int s = 0; s < steps; ++s) {
    u32x4 a[TILES], b[4];
#pragma unroll
    for (int m = 0; m < TILES; ++m)
      a[m] = u32x4{g[m][0] | g[m][1] << 16, g[m][2] | g[m][3] << 16, g[m][4] | g[m][5] << 16, g[m][6] | g[m][7] << 16};
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const u32x2 lo = v[2 * p], hi = v[2 * p + 1];
      b[0][p] = __builtin_amdgcn_perm(hi.x, lo.x, 0x05040100u);
      b[1][p] = __builtin_amdgcn_perm(hi.x, lo.x, 0x07060302u);
      b[2][p] = __builtin_amdgcn_perm(hi.y, lo.y, 0x05040100u);
      b[3][p] = __builtin_amdgcn_perm(hi.y, lo.y, 0x07060302u);
    }
    load(s + 1);
#pragma unroll
    for (int m = 0; m < TILES; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[m][i] = product(a[m], b[i], acc[m][i]);  // columns col + i
  }
#pragma unroll
  for (int m = 0; m < TILES; ++m) {
    if (m > 0) __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) part[wave][r][lane] = f32x4{acc[m][0][r], acc[m][1][r], acc[m][2][r], acc[m][3][r]};
    __syncthreads();
    // thread (wave, lane) sums accumulator row r = wave: expert m * 16 + 4 q + r, columns col .. col + 3
    f32x4 sum = part[0][wave][lane];
#pragma unroll
    for (int w = 1; w < kGateWaves; ++w) {
      const f32x4 o = part[w][wave][lane];
      sum.x += o.x;
      sum.y += o.y;
      sum.z += o.z;
      sum.w += o.w;
    }
    const int e = m * 16 + q * 4 + wave;
    if (e < experts && col < hidden) {
      const size_t at = (size_t)e * hidden + col;
      if (out != nullptr) *reinterpret_cast<u32x2*>(out + at) = u32x2{pack_bf16x2(sum.x, sum.y), pack_bf16x2(sum.z, sum.w)};
      else *reinterpret_cast<f32x4*>(sums + (size_t)blockIdx.y * experts * hidden + at) = sum;
    }
  }
}

// out[i] = bf16(sum over the slices, in their order): four values per thread, `count` a multiple of four
__global__ __launch_bounds__(256) void gating_sum_kernel(const float* __restrict__ sums, int slices, int count,
                                                         uint16_t* __restrict__ out) {
  const int i = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= count) return;
  f32x4 sum = *reinterpret_cast<const f32x4*>(sums + i);
#pragma unroll 8
  for (int s = 1; s < slices; ++s) {
    const f32x4 o = *reinterpret_cast<const f32x4*>(sums + (size_t)s * count + i);
    sum.x += o.x;
    sum.y += o.y;
    sum.z += o.z;
    sum.w += o.w;
  }
  *reinterpret_cast<u32x2*>(out + i) = u32x2{pack_bf16x2(sum.x, sum.y), pack_bf16x2(sum.z, sum.w)};
}

// One workgroup: `groups` * 16 tokens, 64 columns per wavefront.  The weights are the first operand and stay in
// registers; fragment (p, j) holds the columns 32 p + 8 (m / 4) + 4 j + m % 4 in its rows m, so that lane (q, c) gets
// the eight columns 32 p + 8 q .. of token c out of two products: one 16-byte load of grad_in, which is what the
// accumulators start from, and one 16-byte store.
enum { kOddExperts = 1, kEvenExperts = 2, kWholeExperts = 8 };  // what the number of experts is a multiple of
template <int STEPS, int OF>  // 32 experts each; what the loads of a token's gradients may take at once
__global__ __launch_bounds__(kGateWaves * 64) void gating_dgrad_kernel(const uint16_t* __restrict__ grad,
                                                                       const uint16_t* __restrict__ weight,
                                                                       const uint16_t* __restrict__ grad_in,
                                                                       uint16_t* __restrict__ out, int tokens,
                                                                       int hidden, int experts, int groups) {
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int q = lane / 16, c = lane % 16;
  const int t0 = blockIdx.y * groups * kGateRows;
  const int rows = min(groups * kGateRows, tokens - t0);
  const int h0 = (blockIdx.x * kGateWaves + wave) * kGateCols;
  if (h0 >= hidden) return;
  const uint32_t bytes = (uint32_t)rows * hidden * 2u;
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(weight, (uint32_t)experts * hidden * 2u);
  const __amdgpu_buffer_rsrc_t rg = make_rsrc(grad + (size_t)t0 * experts, (uint32_t)rows * experts * 2u);
  const __amdgpu_buffer_rsrc_t ri =
      make_rsrc(grad_in != nullptr ? grad_in + (size_t)t0 * hidden : weight, grad_in != nullptr ? bytes : 0u);  // none: zeros
  const __amdgpu_buffer_rsrc_t ro = make_rsrc(out + (size_t)t0 * hidden, bytes);
  u32x4 w[2][2][STEPS];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        const int h = h0 + 32 * p + 8 * (c / 4) + 4 * j + c % 4;
        uint32_t v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int e = 32 * s + 8 * q + k;
          v[k] = load_u16(rw, e < experts && h < hidden ? ((uint32_t)e * hidden + h) * 2u : kOobOffset);
        }
        w[p][j][s] = u32x4{v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16};
      }
  u32x4 b[STEPS], in[2];
  // the loads of a group are issued before the products of the group before; past the rows they deliver zeros
  const auto load = [&](int g) {
    const uint32_t t = g * kGateRows + c;
    const bool any = g < groups;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int e = 32 * s + 8 * q;
      if constexpr (OF == kWholeExperts) {
        b[s] = buf_load16(rg, any && e < experts ? (t * experts + e) * 2u : kOobOffset);
      } else if constexpr (OF == kEvenExperts) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          b[s][k] = __builtin_amdgcn_raw_buffer_load_b32(
              rg, (int)(any && e + 2 * k < experts ? (t * experts + e + 2 * k) * 2u : kOobOffset), 0, 0);
      } else {
        uint32_t v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = load_u16(rg, any && e + k < experts ? (t * experts + e + k) * 2u : kOobOffset);
        b[s] = u32x4{v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16};
      }
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int h = h0 + 32 * p + 8 * q;
      in[p] = buf_load16(ri, any && h < hidden ? (t * hidden + h) * 2u : kOobOffset);
    }
  };
  load(0);
  for (int g = 0; g < groups; ++g) {
    u32x4 bb[STEPS];
    f32x4 sum[2][2];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) bb[s] = b[s];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      sum[p][0] = f32x4{bf16_lo_to_f32(in[p].x), bf16_hi_to_f32(in[p].x), bf16_lo_to_f32(in[p].y), bf16_hi_to_f32(in[p].y)};
      sum[p][1] = f32x4{bf16_lo_to_f32(in[p].z), bf16_hi_to_f32(in[p].z), bf16_lo_to_f32(in[p].w), bf16_hi_to_f32(in[p].w)};
    }
    load(g + 1);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int s = 0; s < STEPS; ++s)
#pragma unroll
        for (int j = 0; j < 2; ++j) sum[p][j] = product(w[p][j][s], bb[s], sum[p][j]);
      const int h = h0 + 32 * p + 8 * q;
      buf_store16(u32x4{pack_bf16x2(sum[p][0].x, sum[p][0].y), pack_bf16x2(sum[p][0].z, sum[p][0].w),
                        pack_bf16x2(sum[p][1].x, sum[p][1].y), pack_bf16x2(sum[p][1].z, sum[p][1].w)},
                  ro, h < hidden ? ((uint32_t)(g * kGateRows + c) * hidden + h) * 2u : kOobOffset);
    }
  }
}

int ceil_div(int a, int b) { return (a + b - 1) / b; }

// steps of 32 tokens per wavefront of the weight gradient: kGateBlocks workgroups over the columns and the tokens, the
// rows of one within 1 GB (32-bit offsets)
int gate_steps(int tokens, int hidden, int experts) {
  const int most = ceil_div(tokens, kGateStep * kGateWaves);              // slices of one step per wavefront
  const int blocks = experts > kGateManyExperts ? kGateBlocks / 2 : kGateBlocks;
  const int slices = ceil_div(blocks, ceil_div(hidden, kGateCols));       // that fill the chip
  const int64_t fit = (1 << 30) / ((int64_t)kGateStep * kGateWaves * std::max(hidden, kGateMaxExperts) * 2);
  return (int)std::max<int64_t>(1, std::min<int64_t>(slices >= most ? 1 : ceil_div(most, slices), fit));
}
int gate_slices(int tokens, int hidden, int experts) {
  return ceil_div(tokens, gate_steps(tokens, hidden, experts) * kGateStep * kGateWaves);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace fp8gmm

extern "C" {

size_t fp8gmm_gating_workspace_bytes(int tokens, int hidden, int experts) {
  using namespace fp8gmm;
  if (tokens <= 0 || hidden <= 0 || experts <= 0) return 0;
  const int slices = gate_slices(tokens, hidden, experts);
  return slices > 1 ? (size_t)slices * experts * hidden * sizeof(float) : 0;
}

int fp8gmm_gating_backward(const void* grad, const void* x, const void* weight, const void* grad_in, void* grad_x,
                           void* grad_weight, int tokens, int hidden, int experts, void* workspace, void* stream) {
  using namespace fp8gmm;
  if (tokens < 1 || hidden < 8 || hidden % 8 != 0 || experts < 1 || experts > kGateMaxExperts)
    return FP8GMM_ERR_BAD_ARGUMENT;
  // 32-bit offsets: the weights, and the rows of one workgroup
  const int groups = std::max(1, std::min(16, (int)((int64_t)ceil_div(tokens, kGateRows) *
                                                    ceil_div(hidden, kGateCols * kGateWaves) / kGateBlocks)));
  const int steps = gate_steps(tokens, hidden, experts);
  const int64_t rows = std::max<int64_t>(groups * kGateRows, (int64_t)steps * kGateStep * kGateWaves);
  if ((int64_t)experts * hidden * 2 > 0x7fffffff || rows * std::max(hidden, experts) * 2 > 0x7fffffff ||
      ceil_div(tokens, groups * kGateRows) > 65535)
    return FP8GMM_ERR_BAD_SHAPE;
  if (grad == nullptr) return FP8GMM_ERR_NULL_POINTER;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint16_t* g = static_cast<const uint16_t*>(grad);
  if (grad_weight != nullptr) {
    const int slices = gate_slices(tokens, hidden, experts);
    if (x == nullptr || (slices > 1 && workspace == nullptr)) return FP8GMM_ERR_NULL_POINTER;
    if (!aligned16(x) || !aligned16(grad_weight) || !aligned16(workspace)) return FP8GMM_ERR_BAD_ARGUMENT;
    float* sums = static_cast<float*>(workspace);
    uint16_t* out = slices > 1 ? nullptr : static_cast<uint16_t*>(grad_weight);
    const dim3 grid(ceil_div(hidden, kGateCols), slices), block(kGateWaves * 64);
    auto* kernel = experts <= 16   ? &gating_wgrad_kernel<1>
                         : experts <= 32 ? &gating_wgrad_kernel<2>
                         : experts <= 64 ? &gating_wgrad_kernel<4>
                                         : &gating_wgrad_kernel<8>;
    hipLaunchKernelGGL(kernel, grid, block, 0, s, g, static_cast<const uint16_t*>(x), tokens, hidden, experts, steps,
                       sums, out);
    if (slices > 1) {
      const int count = experts * hidden;
      hipLaunchKernelGGL(gating_sum_kernel, dim3(ceil_div(count, 1024)), dim3(256), 0, s, sums, slices, count,
                         static_cast<uint16_t*>(grad_weight));
    }
  }
  if (grad_x != nullptr) {
    if (weight == nullptr) return FP8GMM_ERR_NULL_POINTER;
    if (!aligned16(grad_x) || !aligned16(grad_in) || !aligned16(grad)) return FP8GMM_ERR_BAD_ARGUMENT;
    const dim3 grid(ceil_div(hidden, kGateCols * kGateWaves), ceil_div(tokens, groups * kGateRows));
    const auto pick = [&](auto* odd, auto* even, auto* whole) {
      return experts % 8 == 0 ? whole : experts % 2 == 0 ? even : odd;
    };
    auto* kernel = experts <= 32   ? pick(&gating_dgrad_kernel<1, kOddExperts>, &gating_dgrad_kernel<1, kEvenExperts>,
                                          &gating_dgrad_kernel<1, kWholeExperts>)
                   : experts <= 64 ? pick(&gating_dgrad_kernel<2, kOddExperts>, &gating_dgrad_kernel<2, kEvenExperts>,
                                          &gating_dgrad_kernel<2, kWholeExperts>)
                                   : pick(&gating_dgrad_kernel<4, kOddExperts>, &gating_dgrad_kernel<4, kEvenExperts>,
                                          &gating_dgrad_kernel<4, kWholeExperts>);
    hipLaunchKernelGGL(kernel, grid, dim3(kGateWaves * 64), 0, s, g, static_cast<const uint16_t*>(weight),
                       static_cast<const uint16_t*>(grad_in), static_cast<uint16_t*>(grad_x), tokens, hidden, experts,
                       groups);
  }
  return hipGetLastError() == hipSuccess ? FP8GMM_OK : FP8GMM_ERR_LAUNCH;
}

}  // extern "C"
