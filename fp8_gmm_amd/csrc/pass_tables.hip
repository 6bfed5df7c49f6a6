// The tables of a pass of a grouped linear layer or MLP, written by the device: cast descriptors, problem tables, work
// lists and shared-tile records, byte for byte what the host planners (pass_plan.cpp) write for the same pass.
//
// The reference packs the same tables into launch arguments or copies them one by one (csrc/multi_pad_fusion.cu:495-501,
// csrc/fp8_gmm.cu:116-135).
//
// Bound: latency of one small launch.  Written on the host and read over the host link, the tables of a step (64 bytes
// per tile, up to 0.9 MB) took 3 - 52 us of copy kernel in front of every pass and as much host time to plan.  Here they
// follow from 4 KB of kernel argument: the group sizes, a description of every launch (pass_spec.h) and the tile ranges
// of its XCDs, which the host works out in a few microseconds.  Every record of a work list is independent of the others
// - its tile is a closed form of (round, workgroup), its problem a binary search over the experts in LDS - so a lane
// writes a record, and the whole chip writes the lists of a pass at once.
// What such a launch waits for is memory that nothing has touched before: its argument (host memory, read over the link:
// copied to LDS with one load per lane at the start, not line by line as the code meets it) and its own instructions
// (fetched line by line: one copy of every computation, 32-bit arithmetic - 64-bit divisions inlined from the host's
// functions made it 34 KB and 12 - 16 us).
// Then come steps that wait for each other: the prefix sums.  One round of them, several lists side by side and without LDS
// inside a wavefront, against up to four rounds of shuffles, us a launch under a kernel trace: 8 experts 9.0 -> 6.0, 64 experts
// 10.9 -> 7.3, 128 experts 10.0 -> 7.5, with tiles shared along K 14.7 -> 12.0 (the rest is numbering their slots); with the
// update of 1280 columns on the side 13.2 -> 11.3, which is that update's time.
#include "device_utils.h"
#include "internal.h"
#include "pass_spec.h"
#include "scaling_update.h"

namespace fp8gmm {
namespace {

constexpr int kThreads = 256;
constexpr int kExperts = kPassMaxExperts;
static_assert(kPassRecordsPerBlock == kThreads, "a lane per record");

// Inclusive sums over a wavefront, all of whose lanes are here: four shifts inside rows of 16 lanes, then the last lane of
// rows 0 and 2 to the row behind and that of the lower half to the upper one.  Data-parallel primitives: a shuffle through
// LDS is ten times as far away, and six of them follow each other.
__device__ __forceinline__ int wave_inclusive(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31
  return v;
}

constexpr int kScans = 3;   // lists that are summed side by side
struct Scan {
  int v[kScans];
};

// Exclusive prefix sums of `kScans` lists at once: `value(i)` are the entries i of [0, n), n >= 1; `take(i, sums)` gets the
// sums in front of entry i, in the thread that gave its values; the totals are returned.  All threads of the workgroup; what
// `value` and `take` have stored is visible to all of them behind it.
template <typename Value, typename Take>
__device__ __forceinline__ Scan exclusive_scan(int n, int (*wave_sums)[kThreads / kWaveSize], Value value, Take take) {
  const int lane = threadIdx.x % kWaveSize, wave = threadIdx.x / kWaveSize;
  Scan carry = {};
#pragma unroll 1
  for (int base = 0; base < n; base += kThreads) {
    const int i = base + (int)threadIdx.x;
    Scan own = {}, sum;
    if (i < n) own = value(i);
#pragma unroll
    for (int q = 0; q < kScans; ++q) {
      sum.v[q] = wave_inclusive(own.v[q]);
      if (lane == kWaveSize - 1) wave_sums[q][wave] = sum.v[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kScans; ++q) {
      sum.v[q] += carry.v[q] - own.v[q];
#pragma unroll
      for (int w = 0; w < kThreads / kWaveSize; ++w) {
        const int of = wave_sums[q][w];
        sum.v[q] += w < wave ? of : 0;
        carry.v[q] += of;
      }
    }
    if (i < n) take(i, sum);
    __syncthreads();
  }
  return carry;
}

// `sums`: room for the sums of every run
__device__ void write_cast(const PassTables& t, const CastSpec& spec, uint8_t* blob, const int* row_begin,
                           int* const (&sums)[kScans], int (*wave_sums)[kThreads / kWaveSize]) {
  static_assert(sizeof(spec.run) / sizeof(spec.run[0]) == kScans, "the runs of a cast side by side");
  fp8gmm_tensor_desc* out = reinterpret_cast<fp8gmm_tensor_desc*>(blob + spec.table_offset);
  const Scan total = exclusive_scan(
      t.experts, wave_sums,
      [&](int i) {
        Scan own = {};
#pragma unroll
        for (int s = 0; s < kScans; ++s)
          if (s < spec.n_runs) own.v[s] = cast_blocks(cast_desc(spec.run[s], i, row_begin[i], row_begin[i + 1] - row_begin[i]));
        return own;
      },
      [&](int i, const Scan& before) {
#pragma unroll
        for (int s = 0; s < kScans; ++s) sums[s][i] = before.v[s];
      });
  int block = 0;
#pragma unroll
  for (int s = 0; s < kScans; ++s) {
    if (s < spec.n_runs)
      for (int i = threadIdx.x; i < t.experts; i += kThreads) {
        fp8gmm_tensor_desc d = cast_desc(spec.run[s], i, row_begin[i], row_begin[i + 1] - row_begin[i]);
        d.block_begin = block + sums[s][i];
        out[s * t.experts + i] = d;
      }
    block += total.v[s];
  }
}

// last i of [0, n) with begin[i] <= x, begin[0] = 0
__device__ __forceinline__ int last_at_or_below(const int* begin, int n, int x) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (begin[mid] <= x) lo = mid; else hi = mid - 1;
  }
  return lo;
}

struct Gemm {   // one GEMM's view inside a workgroup; the arrays are in LDS
  const GemmSpec& spec;
  const GemmRanges& ranges;
  const fp8gmm_gemm_problem* probs;
  const int* begin;    // first tile of every problem in the launch's tile size
  const int* cost;     // K = 128 steps in front of every problem (large tiles)
  int n, wgs;
  bool large;

  // The shared remainder of an XCD (gemm_schedule.h): piece j covers the steps [bound(j), bound(j + 1)) of its region.
  __device__ __forceinline__ int bound(const GemmRanges::Xcd& r, int j) const {   // sk_cost * j / sk_wgs
    const unsigned w = (unsigned)r.sk_wgs, q = (unsigned)r.sk_cost / w;
    return (int)(q * (unsigned)j + ((unsigned)r.sk_cost - q * w) * (unsigned)j / w);
  }
  __device__ __forceinline__ int steps_of(int p) const {
    const int s = (probs[p].k + 127) / 128;
    return s > 0 ? s : 1;
  }
  // tile that holds step `c` of an XCD's region: its problem, and the step (of the region) it begins with
  __device__ __forceinline__ int tile_at(const GemmRanges::Xcd& r, int c, int* prob, int* first_step) const {
    const int p = last_at_or_below(cost, n, r.sk_c0 + c);
    const int steps = steps_of(p), local = (r.sk_c0 + c - cost[p]) / steps;
    *prob = p;
    *first_step = cost[p] + local * steps - r.sk_c0;
    return begin[p] + local;
  }
  // The tile that boundary j completes, as fixup_tile: pieces in *pieces (0: none)
  __device__ __forceinline__ int completed_by(int x, int j, int* prob, int* pieces) const {
    const GemmRanges::Xcd& r = ranges.xcd[x];
    *pieces = 0;
    if (j < 1 || j >= r.sk_wgs) return -1;
    int first = 0;
    const int tile = tile_at(r, bound(r, j), prob, &first);
    if (bound(r, j) == first || bound(r, j - 1) > first) return -1;
    int q = j;
    while (q < r.sk_wgs && bound(r, q) < first + steps_of(*prob)) ++q;
    *pieces = q - j + 1;
    return tile;
  }
};

__device__ void write_gemm(const PassTables& t, int g, int block, uint8_t* blob, const int* row_begin,
                           fp8gmm_gemm_problem* probs, int* begin, int* cost, int* slots,
                           int (*wave_sums)[kThreads / kWaveSize]) {
  const GemmSpec& spec = t.gemm[g];
  const GemmRanges& ranges = t.ranges[g];
  const int n = t.experts;
  const Gemm gm{spec, ranges, probs, begin, cost, n, ranges.grid / kNumXcd, spec.tile_m == BM && spec.tile_n == BN};
  // problems, the tiles and K steps in front of each (in 256 x 256 tiles: what the problem table records), and the tiles of
  // the launch's own size
  exclusive_scan(
      n, wave_sums,
      [&](int i) {
        const fp8gmm_gemm_problem p = gemm_problem(spec, i, row_begin[i], row_begin[i + 1] - row_begin[i]);
        probs[i] = p;
        const int tiles = ((p.m + BM - 1) / BM) * ((p.n + BN - 1) / BN), steps = (p.k + 127) / 128;
        const int own = ((p.m + spec.tile_m - 1) / spec.tile_m) * ((p.n + spec.tile_n - 1) / spec.tile_n);
        return Scan{{tiles, tiles * (steps > 0 ? steps : 1), own}};
      },
      [&](int i, const Scan& before) {
        probs[i].tile_begin = before.v[0];
        probs[i].cost_begin = cost[i] = before.v[1];
        begin[i] = before.v[2];
      });
  if (block == 0) {
    static_assert(sizeof(fp8gmm_gemm_problem) % 16 == 0, "copied in words of 16 bytes");
    u32x4* dst = reinterpret_cast<u32x4*>(blob + spec.table_offset);
    const u32x4* src = reinterpret_cast<const u32x4*>(probs);
#pragma unroll 1
    for (int i = threadIdx.x; i < n * (int)(sizeof(fp8gmm_gemm_problem) / 16); i += kThreads) dst[i] = src[i];
  }
  if (ranges.total_tiles == 0) return;
  // Tiles shared along K: their workspace slots, numbered in the order (XCD, piece boundary); slots[i] becomes the first
  // slot of the tile that boundary i = (XCD, j) completes and, 16 bits up, the number of that tile.
  if (ranges.n_fixups > 0) {
    exclusive_scan(
        ranges.grid, wave_sums,
        [&](int i) {
          int p = 0, pieces = 0;
          return Scan{{gm.completed_by(i / gm.wgs, i % gm.wgs, &p, &pieces) >= 0 ? pieces + (1 << 16) : 0}};
        },
        [&](int i, const Scan& before) { slots[i] = before.v[0]; });
    if (block == 0) {
      fp8gmm_gemm_fixup_desc* fix = reinterpret_cast<fp8gmm_gemm_fixup_desc*>(blob + spec.fixups_offset);
#pragma unroll 1
      for (int i = threadIdx.x; i < ranges.grid; i += kThreads) {
        int p = 0, pieces = 0;
        const int tile = gm.completed_by(i / gm.wgs, i % gm.wgs, &p, &pieces);
        if (tile < 0) continue;
        fp8gmm_gemm_fixup_desc o{};
        o.prob = p;
        tile_origin(probs[p].m, probs[p].n, tile - begin[p], &o.m0, &o.n0);
        o.first_slot = slots[i] & 0xffff;
        o.n_pieces = pieces;
        fix[slots[i] >> 16] = o;
      }
    }
  }
  const int index = block * kPassRecordsPerBlock + (int)threadIdx.x;
  if (index >= ranges.rounds * ranges.grid) return;
  const int wg = index % ranges.grid, x = wg % kNumXcd, j = wg / kNumXcd;
  const GemmRanges::Xcd& xc = ranges.xcd[x];
  fp8gmm_gemm_item o = gemm_end_item();
  // Usually one turn: the record itself.  A large-tile record without K steps looks on, for the height of the
  // workgroup's next record that has some, which it repeats one bit up.
  const int own = index / ranges.grid;
#pragma unroll 1
  for (int round = own;; ++round) {
    int tile = -1, p = 0, k_begin = 0, nk = -1, slot = -1, half = -1;
    if (!gm.large) {
      const int whole = xc.begin + whole_tile_of(gm.wgs, j, round);
      if (whole < xc.end) tile = whole;
    } else if (round < xc.dp_rounds) {   // only the last strided round can be partial, and then nothing is shared
      const int whole = xc.begin + gm.wgs * round + (j + kRoundRotation * round) % gm.wgs;
      if (whole < xc.sk_begin) tile = whole;
    } else if (xc.sk_wgs < 0) {
      // a last round of half tiles: two positions per tile; a tile of at most half height takes the first one
      const int position = half_position(gm.wgs, j, round), pair = xc.sk_begin + position / 2;
      if (round == xc.dp_rounds && pair < xc.end) {
        tile = pair;
        half = position % 2;
      }
    } else if (j < xc.sk_wgs) {
      // the tiles under piece j of the shared remainder
      const int lo = gm.bound(xc, j), hi = gm.bound(xc, j + 1);
      int first = 0;
      const int opening = gm.tile_at(xc, lo, &p, &first) + (round - xc.dp_rounds);
      if (lo < hi && opening < xc.end) {
        p = last_at_or_below(begin, n, opening);
        const int steps = gm.steps_of(p);
        first = cost[p] + (opening - begin[p]) * steps - xc.sk_c0;
        if (first < hi) {
          tile = opening;
          const int from = lo > first ? lo - first : 0, to = hi < first + steps ? hi - first : steps;
          if (to - from < steps) {
            // a piece: the one from the tile's first step belongs to the boundary behind it, a later one to the first
            // boundary inside the tile, `piece` boundaries back
            k_begin = from;
            nk = to - from;
            int q = j + 1, piece = 0;
            if (from > 0)
              for (q = j, piece = 1; q > 1 && gm.bound(xc, q - 1) > first; --q) ++piece;
            slot = (slots[x * gm.wgs + q] & 0xffff) + piece;
          }
        }
      }
    }
    if (tile < 0) break;
    if (slot < 0) {
      p = last_at_or_below(begin, n, tile);
      nk = (probs[p].k + 127) / 128;
    }
    int m0 = 0, n0 = 0;
    tile_origin(probs[p].m, probs[p].n, tile - begin[p], spec.tile_m, spec.tile_n, &m0, &n0);
    if (half > 0) m0 += BM / 2;
    if (m0 >= probs[p].m) break;
    const int flags = gm.large && slot < 0 && (half >= 0 || probs[p].m - m0 <= BM / 2) ? FP8GMM_ITEM_HALF_HEIGHT : 0;
    if (round == own) {
      o = gemm_item(probs[p], p, m0, n0, half >= 0 ? BM / 2 : spec.tile_m, spec.tile_n, (spec.layout & FP8GMM_GEMM_A_KMAJOR) != 0,
                    (spec.layout & FP8GMM_GEMM_B_KMAJOR) != 0, k_begin, nk, slot);
      o.flags = flags;
      if (nk > 0 || !gm.large) break;
    } else if (nk > 0) {
      o.flags |= flags << 1;
      break;
    }
  }
  reinterpret_cast<fp8gmm_gemm_item*>(blob + spec.items_offset)[index] = o;
}

constexpr int kUpdates = 2;   // a module's two directions
static_assert(sizeof(PassTables) + sizeof(ScalingUpdatesOf<kUpdates>) + 64 <= 4096, "kernel arguments");
static_assert(kScalingThreads == kThreads, "one launch");

// Workgroups: the tables', one for the copy on the side if there is one, then the scaling updates'.
__global__ __launch_bounds__(kThreads) void pass_tables_kernel(const PassTables argument, uint8_t* __restrict__ blob,
                                                               const float* __restrict__ copy_src,
                                                               float* __restrict__ copy_dst, int copy_n,
                                                               const ScalingUpdatesOf<kUpdates> updates, int update_block) {
  if ((int)blockIdx.x >= update_block) {
    run_scaling_update(updates, (int)blockIdx.x - update_block);
    return;
  }
  __shared__ __attribute__((aligned(16))) fp8gmm_gemm_problem probs[kExperts];
  __shared__ int begin[kExperts], cost[kExperts];
  __shared__ int slots[FP8GMM_PASS_MAX_GRID];
  static_assert(FP8GMM_PASS_MAX_GRID >= kExperts, "the third run of a cast");
  __shared__ int wave_sums[kScans][kThreads / kWaveSize];
  static_assert(sizeof(PassTables) <= kThreads * 16, "four words per lane");
  __shared__ __attribute__((aligned(16))) uint32_t copy[kThreads * 4];
  const PassTables& t = *reinterpret_cast<const PassTables*>(copy);
  const int block = (int)blockIdx.x;
  {
    const uint32_t* words = reinterpret_cast<const uint32_t*>(&argument);
    uint32_t v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = q * kThreads + (int)threadIdx.x;
      v[q] = words[i < (int)(sizeof(PassTables) / 4) ? i : 0];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) copy[q * kThreads + (int)threadIdx.x] = v[q];
  }
  __syncthreads();
  if (block == t.blocks) {   // the last workgroup: the copy on the side
    for (int i = threadIdx.x; i < copy_n; i += kThreads) copy_dst[i] = copy_src[i];
    return;
  }
  if (block < t.n_casts) {
    write_cast(t, t.cast[block], blob, t.row_begin, {begin, cost, slots}, wave_sums);
    return;
  }
  int g = 0;
  while (g + 1 < t.n_gemms && block >= t.first_block[t.n_casts + g + 1]) ++g;
  write_gemm(t, g, block - t.first_block[t.n_casts + g], blob, t.row_begin, probs, begin, cost, slots, wave_sums);
}

}  // namespace

int launch_pass_tables(const PassTables& tables, void* blob_dev, const fp8gmm_scaling_update* updates, int n_updates,
                       const float* copy_src, float* copy_dst, int copy_n, void* stream) {
  ScalingUpdatesOf<kUpdates> all;
  const int rc = collect_scaling_updates(updates, n_updates, &all);
  if (rc != FP8GMM_OK) return rc;
  // a copy of what an update is about to write is made by that update
  for (int i = 0; i < all.n && copy_n > 0; ++i)
    if (all.u[i].scale_inv == copy_src) {
      if (copy_n != all.u[i].slots) return FP8GMM_ERR_BAD_ARGUMENT;
      all.snapshot[i] = copy_dst;
      copy_n = 0;
    }
  const int update_block = tables.blocks + (copy_n > 0 ? 1 : 0);
  const int blocks = update_block + all.first_block[all.n];
  if (blocks == 0) return FP8GMM_OK;
  hipLaunchKernelGGL(pass_tables_kernel, dim3(blocks), dim3(kThreads), 0, static_cast<hipStream_t>(stream), tables,
                     static_cast<uint8_t*>(blob_dev), copy_src, copy_dst, copy_n, all, update_block);
  return hipGetLastError() == hipSuccess ? FP8GMM_OK : FP8GMM_ERR_LAUNCH;
}

}  // namespace fp8gmm
