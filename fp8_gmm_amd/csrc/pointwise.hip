// Multi-tensor element-wise kernels for gfx950: quantize (bf16 -> fp8 + amax) and
// scale_mul (in-place bf16 *= s1 * s2).  One launch covers every tensor of the call;
// each workgroup finds its tensor by a binary search over a device-side table.
//
// Replaces csrc/multi_pointwise.cu of the reference (multi_quantize_kernel :34-97,
// multi_scale_mul_kernel :99-151).  HBM-bound: 2 B read + 1 B written per element
// (quantize), 2 B + 2 B (scale_mul); a wavefront reads 1 KB of contiguous bf16 per step
// (one 128-bit load per lane, all steps issued before the first conversion), the wave reduces amax with cross-lane shuffles and the
// workgroup issues a single integer atomic max.
#include <type_traits>

#include "device_utils.h"
#include "internal.h"
#include "scaling_update.h"
#include "tiling.h"

namespace fp8gmm {
namespace {

// NaNs are looked for once per lane, behind its 64 values (amax_or_nan), and the values taken one by one only where there is
// one: in the step of 128 experts (65536 rows, 2048 -> 768 -> 2048) cast + dGELU 58 -> 54 us, forward cast 249 -> 245, against a look
// at every value and a branch for every four.  A step gains no more than its runs differ by (1209 -> 1199; 16 experts of 4096 x 6400,
// 4096 rows: 1053, 1054).
// DGELU: the value cast is x = in * dgelu(in2) (in = gradient of the GELU output, in2 = pre-GELU activation),
// the same product, in the same order, as the transposing kernel forms.
template <int FMT, bool DGELU>
__global__ __launch_bounds__(kPwThreads) void multi_quantize_kernel(fp8gmm_tensor_desc* __restrict__ descs, int n) {
  __shared__ float stage[kPwThreads / kWaveSize];
  const int bid = blockIdx.x;
  const int t = upper_slot(n, bid, [&](int i) { return descs[i].block_begin; });
  const fp8gmm_tensor_desc d = descs[t];
  const int64_t numel = (int64_t)d.rows * d.cols;
  const int64_t base = (int64_t)(bid - d.block_begin) * kPwBlockElems;
  const uint16_t* __restrict__ in = static_cast<const uint16_t*>(d.in);
  const uint16_t* __restrict__ pre = static_cast<const uint16_t*>(d.in2);
  uint8_t* __restrict__ out = static_cast<uint8_t*>(d.out);
  const float scale = d.scale ? *d.scale : 1.f;
  const bool vec = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out) |
                     (DGELU ? reinterpret_cast<uintptr_t>(pre) : 0)) & 15) == 0 &&
                   numel * 2 < (int64_t)0xffffffff;
  float mx = 0.f;
  auto value = [&](int64_t j) {
    float x = bf16_to_f32(in[j]);
    if constexpr (DGELU) x *= dgelu(bf16_to_f32(pre[j]));
    return x;
  };

  if (vec) {
    // fast path: all loads of the workgroup's 16384 elements are issued before the first conversion
    const __amdgpu_buffer_rsrc_t rin = make_rsrc(in, (uint32_t)(numel * 2));
    const __amdgpu_buffer_rsrc_t rout = make_rsrc(out, (uint32_t)numel);
    const __amdgpu_buffer_rsrc_t rpre = make_rsrc(DGELU ? pre : in, (uint32_t)(numel * 2));
    u32x4 a[kPwSteps];
    u32x4 g[DGELU ? kPwSteps : 1] = {};
    bool full[kPwSteps];
#pragma unroll
    for (int it = 0; it < kPwSteps; ++it) {
      const int64_t off = base + (int64_t)(it * kPwThreads + threadIdx.x) * kPwVec;
      full[it] = off + kPwVec <= numel;
      a[it] = buf_load16_stream(rin, full[it] ? (uint32_t)(off * 2) : kOobOffset);
      if constexpr (DGELU) g[it] = buf_load16_stream(rpre, full[it] ? (uint32_t)(off * 2) : kOobOffset);
    }
    auto take = [&](auto numbers, const u32x4& in8, const u32x4& pre8, uint32_t off) {
      const uint32_t w[4] = {in8.x, in8.y, in8.z, in8.w};
      [[maybe_unused]] const uint32_t p[4] = {pre8.x, pre8.y, pre8.z, pre8.w};
      uint32_t o[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        float x0 = bf16_lo_to_f32(w[2 * q]), x1 = bf16_hi_to_f32(w[2 * q]);
        float x2 = bf16_lo_to_f32(w[2 * q + 1]), x3 = bf16_hi_to_f32(w[2 * q + 1]);
        if constexpr (DGELU) {
          x0 *= dgelu(bf16_lo_to_f32(p[2 * q]));
          x1 *= dgelu(bf16_hi_to_f32(p[2 * q]));
          x2 *= dgelu(bf16_lo_to_f32(p[2 * q + 1]));
          x3 *= dgelu(bf16_hi_to_f32(p[2 * q + 1]));
        }
        if constexpr (decltype(numbers)::value) {
          mx = amax_or_nan(amax_or_nan(mx, x0, x1), x2, x3);
          o[q] = cvt4_fp8_numbers<FMT>(x0 * scale, x1 * scale, x2 * scale, x3 * scale);
        } else {
          mx = amax_step(amax_step(mx, x0), x1);
          mx = amax_step(amax_step(mx, x2), x3);
          o[q] = cvt4_fp8<FMT>(x0 * scale, x1 * scale, x2 * scale, x3 * scale);
        }
      }
      buf_store8(u32x2{o[0], o[1]}, rout, off);
    };
#pragma unroll
    for (int it = 0; it < kPwSteps; ++it) {
      const int64_t off = base + (int64_t)(it * kPwThreads + threadIdx.x) * kPwVec;
      take(std::true_type{}, a[it], g[DGELU ? it : 0], full[it] ? (uint32_t)off : kOobOffset);
      __builtin_amdgcn_sched_barrier(0);   // steps side by side would take the registers of half the wavefronts
    }
    if (__builtin_expect(!keeps_numbers(scale) || mx != mx, 0)) {
      mx = 0.f;
#pragma unroll 1
      for (int it = 0; it < kPwSteps; ++it) {
        const int64_t off = base + (int64_t)(it * kPwThreads + threadIdx.x) * kPwVec;
        const bool whole = off + kPwVec <= numel;
        const u32x4 in8 = buf_load16(rin, whole ? (uint32_t)(off * 2) : kOobOffset);
        const u32x4 pre8 = DGELU ? buf_load16(rpre, whole ? (uint32_t)(off * 2) : kOobOffset) : in8;
        take(std::false_type{}, in8, pre8, whole ? (uint32_t)off : kOobOffset);
      }
    }
#pragma unroll
    for (int it = 0; it < kPwSteps; ++it) {
      const int64_t off = base + (int64_t)(it * kPwThreads + threadIdx.x) * kPwVec;
      if (!full[it] && off < numel) {  // the one partial group at the end of the tensor
        for (int64_t j = off; j < numel; ++j) {
          const float x = value(j);
          mx = amax_step(mx, x);
          out[j] = cvt1_fp8<FMT>(x * scale);
        }
      }
    }
  } else {
#pragma unroll 1
    for (int it = 0; it < kPwSteps; ++it) {
      const int64_t off = base + (int64_t)(it * kPwThreads + threadIdx.x) * kPwVec;
      if (off < numel) {
        const int cnt = (numel - off < kPwVec) ? (int)(numel - off) : kPwVec;
        for (int j = 0; j < cnt; ++j) {
          const float x = value(off + j);
          mx = amax_step(mx, x);
          out[off + j] = cvt1_fp8<FMT>(x * scale);
        }
      }
    }
  }
  block_amax_merge<kPwThreads / kWaveSize>(mx, d.amax != nullptr ? &descs[t].amax_partial : nullptr, stage);
}

__global__ __launch_bounds__(kPwThreads) void multi_scale_mul_kernel(const fp8gmm_tensor_desc* __restrict__ descs,
                                                                     int n) {
  const int bid = blockIdx.x;
  const int t = upper_slot(n, bid, [&](int i) { return descs[i].block_begin; });
  const fp8gmm_tensor_desc d = descs[t];
  const int64_t numel = (int64_t)d.rows * d.cols;
  const int64_t base = (int64_t)(bid - d.block_begin) * kPwBlockElems;
  // in-place: `in` is the tensor being scaled
  uint16_t* __restrict__ x = const_cast<uint16_t*>(static_cast<const uint16_t*>(d.in));
  const float s1 = d.scale ? *d.scale : 1.f;
  const float* s2p = static_cast<const float*>(d.in2);
  const float s2 = s2p ? *s2p : 1.f;
  const bool vec = (reinterpret_cast<uintptr_t>(x) & 15) == 0 && numel * 2 < (int64_t)0xffffffff;

  if (vec) {
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(x, (uint32_t)(numel * 2));
    u32x4 a[kPwSteps];
    bool full[kPwSteps];
#pragma unroll
    for (int it = 0; it < kPwSteps; ++it) {
      const int64_t off = base + (int64_t)(it * kPwThreads + threadIdx.x) * kPwVec;
      full[it] = off + kPwVec <= numel;
      a[it] = buf_load16_stream(rx, full[it] ? (uint32_t)(off * 2) : kOobOffset);
    }
#pragma unroll
    for (int it = 0; it < kPwSteps; ++it) {
      const int64_t off = base + (int64_t)(it * kPwThreads + threadIdx.x) * kPwVec;
      uint32_t w[4] = {a[it].x, a[it].y, a[it].z, a[it].w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        // left to right, as the reference: (x * s1) * s2
        const float lo = bf16_lo_to_f32(w[q]) * s1 * s2;
        const float hi = bf16_hi_to_f32(w[q]) * s1 * s2;
        w[q] = pack_bf16x2(lo, hi);
      }
      buf_store16(u32x4{w[0], w[1], w[2], w[3]}, rx, full[it] ? (uint32_t)(off * 2) : kOobOffset);
      if (!full[it] && off < numel) {
        for (int64_t j = off; j < numel; ++j) x[j] = (uint16_t)f32_to_bf16_bits(bf16_to_f32(x[j]) * s1 * s2);
      }
    }
  } else {
#pragma unroll 1
    for (int it = 0; it < kPwSteps; ++it) {
      const int64_t off = base + (int64_t)(it * kPwThreads + threadIdx.x) * kPwVec;
      if (off < numel) {
        const int cnt = (numel - off < kPwVec) ? (int)(numel - off) : kPwVec;
        for (int j = 0; j < cnt; ++j) x[off + j] = (uint16_t)f32_to_bf16_bits(bf16_to_f32(x[off + j]) * s1 * s2);
      }
    }
  }
}

__global__ __launch_bounds__(kScalingThreads) void delayed_scaling_update_kernel(
    float* __restrict__ history, float* __restrict__ scale, float* __restrict__ scale_inv, int history_len, int slots,
    float fp8_max, float margin_factor, int most_recent, int keep_period, int keep_phase) {
  delayed_scaling_update_columns(history, scale, scale_inv, history_len, slots, fp8_max, margin_factor, most_recent,
                                 keep_period, keep_phase, nullptr, (int)blockIdx.x * kScalingCols);
}

// Several directions in one launch
__global__ __launch_bounds__(kScalingThreads) void delayed_scaling_updates_kernel(const ScalingUpdates all) {
  run_scaling_update(all, (int)blockIdx.x);
}

}  // namespace
}  // namespace fp8gmm

namespace {
// Very large plain casts claim this much LDS per workgroup, so that four share a compute unit where the registers would let eight
// (with the 16 bytes of `stage` 26 of its 128 granules of 1280 bytes; at 31744 bytes, which leave five, nothing is gained: 522 / 509 us
// for the first of these): bound by HBM, they have more loads in flight than it takes, and fewer workgroups at a time keep fewer of its
// rows open.  Eight against four, kernel alone: the forward cast of an MLP's step, 8 experts of 4096 x 14336, 16384 rows 511 / 491 us
// (61 thousand workgroups), both weight stacks of 16 experts of 4096 x 6400 399 / 391 (51 thousand); tensors of 49 - 66
// thousand 417 / 411, 426 / 413, 484 / 477, 537 / 525, 550 / 544.  Smaller launches gain as little as they lose inside a step
// (33 thousand 247 / 248, 14 thousand 115 / 115); the dGELU form needs the wavefronts for its arithmetic (200 / 204).
constexpr int kApartBlocks = 40000;
constexpr size_t kApartLds = 32000;

template <bool DGELU>
int launch_quantize(fp8gmm_tensor_desc* descs_dev, int n, int total_blocks, int out_fmt, void* stream, bool merge = true) {
  if (n < 0 || total_blocks < 0) return FP8GMM_ERR_BAD_ARGUMENT;
  if (out_fmt != FP8GMM_E4M3 && out_fmt != FP8GMM_E5M2) return FP8GMM_ERR_BAD_FORMAT;
  if (n == 0 || total_blocks == 0) return FP8GMM_OK;
  if (descs_dev == nullptr) return FP8GMM_ERR_NULL_POINTER;
  const size_t apart = !DGELU && total_blocks >= kApartBlocks ? kApartLds : 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (out_fmt == FP8GMM_E4M3)
    hipLaunchKernelGGL((fp8gmm::multi_quantize_kernel<FP8GMM_E4M3, DGELU>), dim3(total_blocks),
                       dim3(fp8gmm::kPwThreads), apart, s, descs_dev, n);
  else
    hipLaunchKernelGGL((fp8gmm::multi_quantize_kernel<FP8GMM_E5M2, DGELU>), dim3(total_blocks),
                       dim3(fp8gmm::kPwThreads), apart, s, descs_dev, n);
  if (merge) hipLaunchKernelGGL(fp8gmm::amax_merge_kernel, dim3((n + 255) / 256), dim3(256), 0, s, descs_dev, n);
  return hipGetLastError() == hipSuccess ? FP8GMM_OK : FP8GMM_ERR_LAUNCH;
}
}  // namespace

namespace fp8gmm {
int launch_cast_unmerged(fp8gmm_tensor_desc* descs_dev, int n, int total_blocks, int out_fmt, bool dgelu, void* stream) {
  return dgelu ? launch_quantize<true>(descs_dev, n, total_blocks, out_fmt, stream, false)
               : launch_quantize<false>(descs_dev, n, total_blocks, out_fmt, stream, false);
}
}  // namespace fp8gmm

namespace fp8gmm {
// Tables travel host -> device through this kernel: it reads page-locked host memory that is mapped into the
// device's address space, 16 bytes per thread, and writes device memory.  A copy enqueued with hipMemcpyAsync runs
// as a transfer of its own whose hand-over to the next kernel of the stream took 25 - 30 us on this machine; a
// kernel of the stream hands over like any other kernel.
__global__ void __launch_bounds__(256) upload_kernel(uint4* __restrict__ dst, const uint4* __restrict__ src,
                                                     unsigned pieces) {
  const unsigned i = blockIdx.x * 256u + threadIdx.x;
  if (i < pieces) dst[i] = src[i];
}
}  // namespace fp8gmm

extern "C" {

int fp8gmm_delayed_scaling_update(float* amax_history, float* scale, float* scale_inv, int history_len, int slots,
                                  float fp8_max, int margin, int most_recent, int keep_period, int keep_phase,
                                  void* stream) {
  if (history_len < 1 || slots < 0 || slots > INT32_MAX - fp8gmm::kScalingCols || margin < -126 || margin > 126)
    return FP8GMM_ERR_BAD_ARGUMENT;
  if (keep_period < 0 || (keep_period > 0 && (keep_phase < 0 || keep_phase >= keep_period)))
    return FP8GMM_ERR_BAD_ARGUMENT;
  if (slots == 0) return FP8GMM_OK;
  if (amax_history == nullptr || scale == nullptr || scale_inv == nullptr) return FP8GMM_ERR_NULL_POINTER;
  const float margin_factor = __builtin_ldexpf(1.0f, -margin);
  hipLaunchKernelGGL(fp8gmm::delayed_scaling_update_kernel, dim3((slots + fp8gmm::kScalingCols - 1) / fp8gmm::kScalingCols),
                     dim3(fp8gmm::kScalingThreads), 0, static_cast<hipStream_t>(stream), amax_history, scale, scale_inv, history_len, slots, fp8_max,
                     margin_factor, most_recent != 0, keep_period, keep_phase);
  return hipGetLastError() == hipSuccess ? FP8GMM_OK : FP8GMM_ERR_LAUNCH;
}

int fp8gmm_delayed_scaling_updates(const fp8gmm_scaling_update* updates, int n, void* stream) {
  fp8gmm::ScalingUpdates all;
  const int rc = fp8gmm::collect_scaling_updates(updates, n, &all);
  if (rc != FP8GMM_OK || all.first_block[all.n] == 0) return rc;
  hipLaunchKernelGGL(fp8gmm::delayed_scaling_updates_kernel, dim3(all.first_block[all.n]), dim3(fp8gmm::kScalingThreads), 0,
                     static_cast<hipStream_t>(stream), all);
  return hipGetLastError() == hipSuccess ? FP8GMM_OK : FP8GMM_ERR_LAUNCH;
}

int fp8gmm_multi_quantize(fp8gmm_tensor_desc* descs_dev, int n, int total_blocks, int out_fmt, void* stream) {
  return launch_quantize<false>(descs_dev, n, total_blocks, out_fmt, stream);
}

int fp8gmm_multi_cast_dgelu(fp8gmm_tensor_desc* descs_dev, int n, int total_blocks, int out_fmt, void* stream) {
  return launch_quantize<true>(descs_dev, n, total_blocks, out_fmt, stream);
}

int fp8gmm_multi_scale_mul(const fp8gmm_tensor_desc* descs_dev, int n, int total_blocks, void* stream) {
  if (n < 0 || total_blocks < 0) return FP8GMM_ERR_BAD_ARGUMENT;
  if (n == 0 || total_blocks == 0) return FP8GMM_OK;
  if (descs_dev == nullptr) return FP8GMM_ERR_NULL_POINTER;
  hipLaunchKernelGGL(fp8gmm::multi_scale_mul_kernel, dim3(total_blocks), dim3(fp8gmm::kPwThreads), 0,
                     static_cast<hipStream_t>(stream), descs_dev, n);
  return hipGetLastError() == hipSuccess ? FP8GMM_OK : FP8GMM_ERR_LAUNCH;
}

void* fp8gmm_host_alloc(size_t bytes) {
  if (bytes == 0) return nullptr;
  // while a stream is being captured the runtime refuses allocations from any thread; this one is safe there (it
  // touches no stream), so the calling thread's capture mode is relaxed for its duration
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  const bool exchanged = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
  void* p = nullptr;
  const hipError_t e = hipHostMalloc(&p, bytes, hipHostMallocDefault);
  if (exchanged) (void)hipThreadExchangeStreamCaptureMode(&mode);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  return p;
}

void fp8gmm_host_free(void* p) {
  if (p == nullptr) return;
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  const bool exchanged = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
  (void)hipHostFree(p);
  if (exchanged) (void)hipThreadExchangeStreamCaptureMode(&mode);
}

int fp8gmm_upload(void* dst_dev, const void* src_host, size_t bytes, void* stream) {
  if (bytes == 0) return FP8GMM_OK;
  if (dst_dev == nullptr || src_host == nullptr) return FP8GMM_ERR_NULL_POINTER;
  if (((reinterpret_cast<uintptr_t>(dst_dev) | reinterpret_cast<uintptr_t>(src_host) | bytes) & 15) != 0)
    return FP8GMM_ERR_ALIGNMENT;
  if (bytes > (size_t(1) << 30)) return FP8GMM_ERR_BAD_ARGUMENT;
  const unsigned pieces = (unsigned)(bytes / 16);
  hipLaunchKernelGGL(fp8gmm::upload_kernel, dim3((pieces + 255) / 256), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<uint4*>(dst_dev),
                     static_cast<const uint4*>(src_host), pieces);
  return hipGetLastError() == hipSuccess ? FP8GMM_OK : FP8GMM_ERR_LAUNCH;
}

}  // extern "C"
