// What a pass of a grouped linear layer or of a grouped MLP launches, described in a few numbers per launch instead of
// a record per expert: every table of a pass follows from (group sizes, base addresses, strides).  The host planners
// (pass_plan.cpp) write the tables from such a description into host memory, the table kernel (pass_tables.hip) writes
// the same bytes into device memory from a copy of it that travels as a kernel argument.
#pragma once

#include <stdint.h>

#include "fp8gmm.h"
#include "gemm_schedule.h"
#include "tiling.h"

namespace fp8gmm {

// One run of cast descriptors, one per expert: slices of a token-major tensor (`cols` > 0: rows_i * cols elements) or
// the members of a weight stack (`numel` elements each).
struct CastRun {
  const void* in;
  const void* in2;        // dGELU: the pre-GELU activation, laid out like `in`
  void* out;
  const float* scale;     // of expert 0; expert i's lies i * slot_stride further, like its amax
  float* amax;
  int64_t cols;
  int64_t numel;
  int32_t slot_stride;
  int32_t routed;         // FP8GMM_OP_ROUTED_*: `in` are tokens, an expert's rows begin with rows_padded
};

struct CastSpec {
  CastRun run[3];
  int32_t n_runs;
  int32_t op, out_fmt;
  int32_t reserved;
  int64_t table_offset;
};

// One grouped GEMM.  An operand's address for expert i is base + row_begin_i * row + i * expert (bytes); m or k is the
// expert's row count where the spec says 0.
struct GemmSpec {
  const void* a;
  const void* b;
  void* c;
  void* aux;
  const float* a_scale_inv;
  const float* b_scale_inv;
  const float* c_scale;      // null: none; slots of expert i are i * 3 further
  float* c_amax;
  int64_t a_expert, b_expert, c_expert;
  int32_t a_row, b_row, c_row, aux_row;
  int32_t m, n, k;           // m, k: 0 = the expert's rows
  int32_t lda, ldb, ldc;
  int32_t a_slot, b_slot;    // strides of the scaling slots
  int32_t layout;            // FP8GMM_GEMM_*_KMAJOR
  int32_t tile_m, tile_n;    // tile of the launch
  int32_t reserved;
  int64_t table_offset, items_offset, fixups_offset;
};

// The schedule of one grouped GEMM as the host has worked it out (gemm_schedule.h): what is left to the table kernel
// is one independent computation per record.
struct GemmRanges {
  int32_t grid, rounds;      // records of the work list: rounds * grid, end records included
  int32_t total_tiles;
  int32_t total_cost;
  int32_t n_fixups;
  int32_t reserved;
  struct Xcd {
    int32_t begin, end;      // tiles of the XCD's range
    int32_t dp_rounds;
    int32_t sk_begin, sk_wgs, sk_c0, sk_cost;   // sk_wgs -1: the tiles from sk_begin on as two items of half height each
  } xcd[kNumXcd];
};

constexpr int kPassMaxExperts = FP8GMM_PASS_MAX_EXPERTS;
constexpr int kPassMaxCasts = 2, kPassMaxGemms = 4;
constexpr int kPassRecordsPerBlock = 256;   // records of a work list that a workgroup of the table kernel writes

// The table kernel's argument (and the opaque `tables` of the C ABI).  A kernel's arguments may take 4 KB.
struct PassTables {
  int32_t experts;
  int32_t n_casts, n_gemms;
  int32_t blocks;                               // workgroups of the table kernel
  int32_t first_block[kPassMaxCasts + kPassMaxGemms];   // of each cast, then of each GEMM
  CastSpec cast[kPassMaxCasts];
  GemmSpec gemm[kPassMaxGemms];
  GemmRanges ranges[kPassMaxGemms];
  int32_t row_begin[kPassMaxExperts + 1];               // rows in front of every expert, of all of them behind the last
};
static_assert(sizeof(PassTables) <= FP8GMM_PASS_TABLES_BYTES, "the opaque buffer of the C ABI");

FP8GMM_HD const void* offset_ptr(const void* base, int64_t bytes) {
  return base != nullptr ? static_cast<const uint8_t*>(base) + bytes : nullptr;
}
FP8GMM_HD void* offset_ptr(void* base, int64_t bytes) {
  return base != nullptr ? static_cast<uint8_t*>(base) + bytes : nullptr;
}

// descriptor of expert i of a run (block_begin is the caller's)
FP8GMM_HD fp8gmm_tensor_desc cast_desc(const CastRun& s, int i, int64_t row_begin, int64_t rows) {
  fp8gmm_tensor_desc d{};
  d.scale = s.scale + (int64_t)i * s.slot_stride;
  d.amax = s.amax + (int64_t)i * s.slot_stride;
  if (s.routed) {
    d.in = s.in;
    d.out = offset_ptr(s.out, row_begin * s.cols);
    d.rows = (int32_t)rows;
    d.cols = (int32_t)s.cols;
    d.rows_padded = (int32_t)row_begin;
    return d;
  }
  const int64_t numel = s.cols > 0 ? rows * s.cols : s.numel;
  const int64_t first = s.cols > 0 ? row_begin * s.cols : (int64_t)i * s.numel;
  d.in = offset_ptr(s.in, first * 2);
  d.in2 = offset_ptr(s.in2, first * 2);
  d.out = offset_ptr(s.out, first);
  d.rows = numel > 0;
  d.cols = (int32_t)numel;
  return d;
}
FP8GMM_HD int cast_blocks(const fp8gmm_tensor_desc& d) {
  return (int)(((int64_t)d.rows * d.cols + kPwBlockElems - 1) / kPwBlockElems);
}

// problem of expert i (tile_begin and cost_begin are the caller's)
FP8GMM_HD fp8gmm_gemm_problem gemm_problem(const GemmSpec& s, int i, int64_t row_begin, int32_t rows) {
  fp8gmm_gemm_problem p{};
  p.a = offset_ptr(s.a, row_begin * s.a_row + i * s.a_expert);
  p.b = offset_ptr(s.b, row_begin * s.b_row + i * s.b_expert);
  p.c = offset_ptr(s.c, row_begin * s.c_row + i * s.c_expert);
  p.aux = offset_ptr(s.aux, row_begin * s.aux_row);
  p.a_scale_inv = s.a_scale_inv + (int64_t)i * s.a_slot;
  p.b_scale_inv = s.b_scale_inv + (int64_t)i * s.b_slot;
  if (s.c_scale != nullptr) {
    p.c_scale = s.c_scale + (int64_t)i * 3;
    p.c_amax = s.c_amax + (int64_t)i * 3;
  }
  p.m = s.m > 0 ? s.m : rows;
  p.n = s.n;
  p.k = s.k > 0 ? s.k : rows;
  p.lda = s.lda;
  p.ldb = s.ldb;
  p.ldc = s.ldc;
  return p;
}

// The record of a tile (or of a piece of one): operand addresses of its first row / column and the extents of the
// load descriptors - up to the last byte of the tile's last row (row-major operand) or of the operand's last
// contraction row.  A row-major a whose k is not a multiple of 16 (allowed next to a contraction-major b) ends inside a
// 16-byte piece; the bound includes the whole piece, which lies inside the row's pitch: the hardware checks the range
// per dword, and a dword that straddled the bound would lose its valid bytes too.
FP8GMM_HD fp8gmm_gemm_item gemm_item(const fp8gmm_gemm_problem& p, int prob, int m0, int n0, int tile_m, int tile_n,
                                     bool a_kmajor, bool b_kmajor, int k_begin, int nk, int slot) {
  fp8gmm_gemm_item o{};
  const int64_t rows = p.m - m0 < tile_m ? p.m - m0 : tile_m;
  const int64_t cols = p.n - n0 < tile_n ? p.n - n0 : tile_n;
  if (p.k > 0) {
    if (!a_kmajor) {
      o.a = (uint64_t)reinterpret_cast<uintptr_t>(p.a) + (uint64_t)m0 * (uint64_t)p.lda;
      o.a_bytes = (uint32_t)((rows - 1) * p.lda + ((p.k + 15) & ~15));
    } else {
      o.a = (uint64_t)reinterpret_cast<uintptr_t>(p.a) + (uint64_t)m0;
      o.a_bytes = (uint32_t)((int64_t)(p.k - 1) * p.lda + (p.m - m0));
    }
    if (!b_kmajor) {
      o.b = (uint64_t)reinterpret_cast<uintptr_t>(p.b) + (uint64_t)n0 * (uint64_t)p.ldb;
      o.b_bytes = (uint32_t)((cols - 1) * p.ldb + p.k);
    } else {
      o.b = (uint64_t)reinterpret_cast<uintptr_t>(p.b) + (uint64_t)n0;
      o.b_bytes = (uint32_t)((int64_t)(p.k - 1) * p.ldb + (p.n - n0));
    }
  }
  o.lda = p.lda;
  o.ldb = p.ldb;
  o.k = p.k;
  o.k_begin = k_begin;
  o.nk = nk;
  o.m0 = m0;
  o.n0 = n0;
  o.prob = prob;
  o.slot = slot;
  return o;
}
FP8GMM_HD fp8gmm_gemm_item gemm_end_item() {
  fp8gmm_gemm_item o{};
  o.prob = -1;
  o.slot = -1;
  return o;
}

// Position of a workgroup in a round of the strided part of a whole-tile launch (plan.cpp, plan_whole_tiles): tile
// `local` = wgs * round + l of the XCD's range goes to workgroup (l + kRoundRotation * round) % wgs.
FP8GMM_HD int whole_tile_of(int wgs, int j, int round) {
  const int back = (int)(((int64_t)kRoundRotation * round) % wgs);
  return wgs * round + (j >= back ? j - back : j - back + wgs);
}

}  // namespace fp8gmm
