// Delayed-scaling update of TransformerEngine's recipe, which the reference's modules run through
// `self.prepare_forward(...)` (fp8_gmm/grouped_linear.py:206, fp8_gmm/grouped_mlp.py:349): the device function, and the
// launch arguments of several updates.  Run by launches of its own (pointwise.hip) and by the workgroups of a pass's
// table kernel (pass_tables.hip), which it has nothing in common with but the moment: both come first in a forward pass.
#pragma once

#include "device_utils.h"

namespace fp8gmm {

// Delayed-scaling update of one direction.  Columns of the [history, slots] amax matrix are independent:
//   amax      = max over the history column (or its row 0)
//   scale     = (1 / amax) * fp8_max * 2^-margin   where amax is finite and > 0, else unchanged
//   scale_inv = 1 / scale, except in slots with slot % keep_period == keep_phase (keep_period > 0): those
//               keep their value, for tensors whose fp8 copy from an earlier pass is still in use
//   history   : row i <- row i + 1, last row <- old row 0, then row 0 <- 0 (a history of one row is just cleared)
// The factor is formed as reciprocal times fp8_max, which is what `fp8_max / amax` on a torch tensor
// evaluates to; the two differ in the last bit for some inputs.
//
// Bound: latency.  The default recipe keeps 1024 rows; a module of 128 expert MLPs then has 1280 columns, 5 MB to
// read and to write, a few microseconds of memory traffic.  With one lane per column the rows are a chain of dependent
// round trips (61 us for 20 columns, 111 us for 1280 with the rows read eight at a time).  Here a workgroup owns
// kScalingCols neighbouring columns (one 64-byte piece of every row) and moves kScalingRows rows at once: every lane
// has its 64 rows in flight together, all of them are read before the barrier and written one place up behind it, so the
// shift can be done in place; longer histories take the next rows in turn.  A workgroup per column piece and not per
// row range: the row that one range writes is the row its neighbour still has to read.
constexpr int kScalingCols = 16;
constexpr int kScalingThreads = 256;
constexpr int kScalingLanes = kScalingThreads / kScalingCols;   // rows side by side: 16
constexpr int kScalingPerLane = 64;
constexpr int kScalingRows = kScalingLanes * kScalingPerLane;   // 1024
constexpr int kScalingChunkSlots = 0xffffffffu / 4 / kScalingRows;   // columns of a chunk that 32-bit offsets reach: 2^20 - 1

// torch.max semantics: a NaN anywhere in the column wins
__device__ __forceinline__ float history_max(float a, float b) { return (b > a || b != b) ? b : a; }

__device__ __forceinline__ void delayed_scaling_update_columns(float* __restrict__ history, float* __restrict__ scale,
                                                                float* __restrict__ scale_inv, int history_len, int slots,
                                                                float fp8_max, float margin_factor, int most_recent,
                                                                int keep_period, int keep_phase, float* __restrict__ snapshot, int c0) {
  __shared__ float stage[kScalingThreads / kWaveSize][kScalingCols];
  const int lane_col = threadIdx.x % kScalingCols, lane_row = threadIdx.x / kScalingCols;
  const int c = c0 + lane_col;
  const bool live = c < slots;
  float* col = history + c;
  const float first = live ? col[0] : 0.f;
  float amax = first;
  if (slots > kScalingChunkSlots) {
    // a chunk of so wide a table is out of a buffer descriptor's reach: a lane per column, row by row
    if (threadIdx.x >= kScalingCols || !live) return;
    for (int r = 1; r < history_len; ++r) {
      const float v = col[(size_t)r * slots];
      amax = history_max(amax, v);
      col[(size_t)(r - 1) * slots] = v;
    }
  } else {
    const uint32_t pitch = (uint32_t)slots * 4;
    const uint32_t lane_off = live ? (uint32_t)lane_row * pitch + (uint32_t)c * 4 : kOobOffset;
    for (int base = 0; base < history_len; base += kScalingRows) {
      // rows past the history read as zeros, which never raise a maximum of magnitudes, and are not stored; the
      // descriptor of the stores begins one row above that of the loads
      const int rows = history_len - base < kScalingRows ? history_len - base : kScalingRows;
      float* const chunk = history + (int64_t)base * slots;
      const __amdgpu_buffer_rsrc_t from = make_rsrc(chunk, (uint32_t)rows * pitch);
      const __amdgpu_buffer_rsrc_t to = make_rsrc(chunk - slots, (uint32_t)rows * pitch);
      uint32_t v[kScalingPerLane];
      uint32_t off = lane_off;
#pragma unroll
      for (int j = 0; j < kScalingPerLane; ++j) {
        v[j] = __builtin_amdgcn_raw_buffer_load_b32(from, (int)off, 0, 0);
        off = live ? off + kScalingLanes * pitch : kOobOffset;
      }
#pragma unroll
      for (int j = 0; j < kScalingPerLane; ++j) amax = history_max(amax, __uint_as_float(v[j]));
      __syncthreads();
      off = base == 0 && lane_row < 2 ? kOobOffset : lane_off;   // row 1 falls on row 0, which is cleared below
#pragma unroll
      for (int j = 0; j < kScalingPerLane; ++j) {
        __builtin_amdgcn_raw_buffer_store_b32(v[j], to, (int)off, 0, 0);
        off = live ? lane_off + (uint32_t)(j + 1) * (kScalingLanes * pitch) : kOobOffset;
      }
    }
    // lanes 16 apart hold the same column
    for (int off = kScalingCols; off < kWaveSize; off <<= 1) amax = history_max(amax, __shfl_xor(amax, off));
    if (threadIdx.x % kWaveSize < kScalingCols) stage[threadIdx.x / kWaveSize][lane_col] = amax;
    __syncthreads();   // (the last rows have been read by now, too: the row written below is one of them)
    if (threadIdx.x >= kScalingCols || !live) return;
    for (int w = 1; w < kScalingThreads / kWaveSize; ++w) amax = history_max(amax, stage[w][lane_col]);
  }
  if (most_recent) amax = first;
  float sc = scale[c];
  if (amax > 0.f && amax <= 3.4028234663852886e38f) sc = ((1.0f / amax) * fp8_max) * margin_factor;
  scale[c] = sc;
  const bool keep = keep_period > 0 && c % keep_period == keep_phase;
  if (!keep) scale_inv[c] = 1.0f / sc;
  if (snapshot != nullptr) snapshot[c] = keep ? scale_inv[c] : 1.0f / sc;
  if (history_len > 1) col[(size_t)(history_len - 1) * slots] = first;
  col[0] = 0.f;
}

// Several directions (a module's forward and backward scaling state) in one launch: the workgroups of update u
// follow those of update u - 1.  The updates travel as a kernel argument.
template <int N>
struct ScalingUpdatesOf {
  fp8gmm_scaling_update u[N];
  float* snapshot[N];      // a second place that receives the scale_inv of update i (null: none)
  float margin_factor[N];
  int first_block[N + 1];
  int n;
};
using ScalingUpdates = ScalingUpdatesOf<FP8GMM_MAX_SCALING_UPDATES>;

template <int N>
__device__ __forceinline__ void run_scaling_update(const ScalingUpdatesOf<N>& all, int block) {
  int i = 0;
  while (i + 1 < all.n && block >= all.first_block[i + 1]) ++i;
  const fp8gmm_scaling_update& u = all.u[i];
  delayed_scaling_update_columns(u.amax_history, u.scale, u.scale_inv, u.history_len, u.slots, u.fp8_max,
                                 all.margin_factor[i], u.most_recent, u.keep_period, u.keep_phase, all.snapshot[i],
                                 (block - all.first_block[i]) * kScalingCols);
}

template <int N>
int collect_scaling_updates(const fp8gmm_scaling_update* updates, int n, ScalingUpdatesOf<N>* all) {
  *all = ScalingUpdatesOf<N>{};
  if (n < 0 || n > N) return FP8GMM_ERR_BAD_ARGUMENT;
  if (n == 0) return FP8GMM_OK;
  if (updates == nullptr) return FP8GMM_ERR_NULL_POINTER;
  int blocks = 0;
  for (int i = 0; i < n; ++i) {
    const fp8gmm_scaling_update& u = updates[i];
    if (u.history_len < 1 || u.slots < 0 || u.slots > INT32_MAX - kScalingCols || u.margin < -126 || u.margin > 126) return FP8GMM_ERR_BAD_ARGUMENT;
    if (u.keep_period < 0 || (u.keep_period > 0 && (u.keep_phase < 0 || u.keep_phase >= u.keep_period)))
      return FP8GMM_ERR_BAD_ARGUMENT;
    if (u.slots > 0 && (u.amax_history == nullptr || u.scale == nullptr || u.scale_inv == nullptr))
      return FP8GMM_ERR_NULL_POINTER;
    all->u[i] = u;
    all->margin_factor[i] = __builtin_ldexpf(1.0f, -u.margin);
    all->first_block[i] = blocks;
    blocks += (u.slots + kScalingCols - 1) / kScalingCols;
  }
  all->first_block[n] = blocks;
  all->n = n;
  return FP8GMM_OK;
}

}  // namespace fp8gmm
