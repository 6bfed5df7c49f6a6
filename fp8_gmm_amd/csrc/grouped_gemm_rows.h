// Grouped GEMM of few rows per problem: the weights pass by once, and the launch is a stream of them.
//
// Bound: HBM, the fp8 weights (decoding: 64 tokens over 8 experts of 4096 x 14336 read 470 MB for 7.5 GFLOP).  The tiles of
// the other forms (grouped_gemm_kernel.h) keep half of their ring for token rows that do not exist here, 40 - 64 KB of
// weights under way per compute unit, and fetch weights like lines that somebody will ask for again.
//
// A tile is 64 rows x 128 columns here.  A step (K = 128: 16 KB of weights, 8 KB of tokens) is a stage of a ring of
// three; two workgroups share a compute unit, 64 KB of weights under way between them, and one's barriers, fragment reads
// and result stores hide behind the other's loads.  A wavefront has 32 columns, in two blocks of 32 rows, accumulated in
// ordinary registers; blocks without rows are skipped.  The weights are loaded with the streaming hint: they pass by once
// (plain loads of rows of 4096 / 14336 bytes reach 5.4 / 6.0 TB/s on this chip, with the hint 6.1 / 6.9).  The load stream
// runs on across tile boundaries.  Unit layout, K order and products are those of the other forms: the same bits.
//
// Back to back, other forms -> this one (us, table upload of 3 - 4 included): 8 experts, 8 rows each, K = 14336 to 4096
// columns 104 -> 73, K = 4096 to 14336 columns 108 -> 90 (with the GELU and an fp8 result 128 -> 94); 128 experts, 8 rows each, K = 2048 to 768 columns 45 -> 39.
// Tiles of 64 columns (ring of five) move the tokens twice as often: 85 against 73, 84 against 89 at 896 tiles, where
// their balance is better; one workgroup per compute unit with a ring of six: 74, 96.
#pragma once

#include "grouped_gemm_kernel.h"

namespace fp8gmm {

constexpr int kRowsTileM = FP8GMM_GEMM_ROWS_TILE_M, kRowsTileN = FP8GMM_GEMM_ROWS_TILE_N;
constexpr int kRowsUnitA = kRowsTileM * BK, kRowsUnitB = kRowsTileN * BK;   // a step's tokens and weights
constexpr int kRowsStage = kRowsUnitA + kRowsUnitB;
constexpr int kRowsStages = 3;
constexpr int kRowsLds = kRowsStages * kRowsStage;
static_assert(kRowsTileN == 32 * NWAVES && 2 * kRowsLds <= 160 * 1024, "32 columns per wavefront, two workgroups per compute unit");
// global -> LDS with the streaming hint
#define FP8GMM_DMA_STREAM(lds_addr, voff, rsrc) \
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds" ::"s"(lds_addr), "v"(voff), "s"(rsrc))

// One 32 x 32 block of a result: a lane holds rows m, columns n + 8 g + 0..3 (g = 0..3) of it.
__device__ __forceinline__ float store_rows_block(const fp8gmm_gemm_problem& pr, int m, int n, const f32x16& t, int out_kind,
                                                  int epilogue, float sa, float sb, float cs) {
  const bool gelu = (epilogue & FP8GMM_EPI_GELU) != 0, two = (epilogue & FP8GMM_EPI_TWO_ROUNDINGS) != 0;
  const int N = pr.n;
  const int64_t row = (int64_t)m * pr.ldc;
  uint16_t* const AUX = gelu ? static_cast<uint16_t*>(pr.aux) : nullptr;
  const int c_size = out_kind == FP8GMM_OUT_BF16 ? 2 : 1;
  const bool vec = ((pr.ldc & 3) == 0) && ((reinterpret_cast<uintptr_t>(pr.c) & (4 * c_size - 1)) == 0) &&
                   (AUX == nullptr || (reinterpret_cast<uintptr_t>(AUX) & 7) == 0);
  const float s = sa * sb;
  float amax = 0.f;
  if (m >= pr.m) return amax;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int col = n + 8 * g;
    if (col >= N) continue;
    float v[4], r[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[q] = two ? scaled_twice(t[4 * g + q], sa, sb) : t[4 * g + q] * s;
      r[q] = gelu ? gelu_tanh_fast(v[q]) : v[q];
      if (out_kind != FP8GMM_OUT_BF16 && col + q < N) amax = amax_step(amax, r[q]);
    }
    const bool whole = vec && col + 3 < N;
    if (out_kind == FP8GMM_OUT_BF16) {
      uint16_t* const C = static_cast<uint16_t*>(pr.c) + row + col;
      if (whole) {
        const u32x2 o = {pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3])};
        global_store(C, o);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (col + q < N) global_store(C + q, (uint16_t)f32_to_bf16_bits(r[q]));
      }
    } else {
      uint8_t* const C = static_cast<uint8_t*>(pr.c) + row + col;
      const uint32_t w = out_kind == FP8GMM_E4M3 ? cvt4_fp8<FP8GMM_E4M3>(r[0] * cs, r[1] * cs, r[2] * cs, r[3] * cs)
                                                 : cvt4_fp8<FP8GMM_E5M2>(r[0] * cs, r[1] * cs, r[2] * cs, r[3] * cs);
      if (whole) {
        global_store(C, w);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (col + q < N) global_store(C + q, (uint8_t)(w >> (8 * q)));
      }
    }
    if (AUX != nullptr) {
      uint16_t* const X = AUX + row + col;
      if (whole) {
        const u32x2 a = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        global_store(X, a);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (col + q < N) global_store(X + q, (uint16_t)f32_to_bf16_bits(v[q]));
      }
    }
  }
  return amax;
}

template <int A_FMT, int B_FMT>
__global__ __launch_bounds__(NTHREADS, 2) void grouped_gemm_rows_kernel(
    const fp8gmm_gemm_problem* __restrict__ probs, const fp8gmm_gemm_item* __restrict__ items, int out_kind, int epilogue,
    const fp8gmm_tensor_desc* __restrict__ merge_descs, int merge_n) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  if (merge_n > 0 && blockIdx.x == 0) merge_amax_partials(merge_descs, merge_n, threadIdx.x, NTHREADS);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int MB = kRowsTileM / 32;   // 32 x 32 blocks of a wavefront, one above the other
  const int l32 = lane & 31, khalf = lane >> 5;
  const uint32_t lds_base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);
  // loads: one instruction fills 8 rows x 128 B; wavefront w takes the groups w and w + 4 of each operand.  Chunk c of row
  // r is kept at chunk c ^ ((r >> 1) & 7).
  constexpr int kPartsA = kRowsUnitA / 1024 / NWAVES, kPartsB = kRowsUnitB / 1024 / NWAVES;
  const int drow = lane >> 3;
  const int dchunk = (lane & 7) ^ ((((wave & 1) << 2) + (lane >> 4)) & 7);
  // fragments: rows 32 * block + l32, K half hh, chunks 4 hh + 2 khalf + {0, 1}
  const int fsw = (l32 >> 1) & 7;
  int fc[2][2];
#pragma unroll
  for (int hh = 0; hh < 2; ++hh)
#pragma unroll
    for (int q = 0; q < 2; ++q) fc[hh][q] = ((4 * hh + 2 * khalf + q) ^ fsw) << 4;
  const int fa_off = l32 * BK, fb_off = kRowsUnitA + (wave * 32 + l32) * BK;

  const uint8_t* const my_items = reinterpret_cast<const uint8_t*>(items + blockIdx.x);
  const size_t item_stride = (size_t)gridDim.x * sizeof(fp8gmm_gemm_item);
  auto item_load = [&](int r) { return *reinterpret_cast<const ItemLoad*>(my_items + r * item_stride); };
  auto item_tile = [&](int r) { return *reinterpret_cast<const ItemTile*>(my_items + r * item_stride + 32); };
  int r_ld = 0;
  ItemLoad ld_next_l = item_load(0);
  ItemTile ld_next_t = item_tile(0);
  if (ld_next_t.prob < 0) return;

  // ---- the load cursor, kRowsStages - 1 steps ahead of the products, possibly in a later tile
  bool ld_live = true;
  int ld_kt = 0, ld_nk = 0, ld_kmax = 0;
  i32x4 rsrc_a = {0, 0, 0, 0x00020000}, rsrc_b = {0, 0, 0, 0x00020000};
  uint32_t a_base = 0, b_base = 0, a_step = 0, b_step = 0;
  auto load_setup = [&]() {   // the record after this one is fetched last, as in grouped_gemm_kernel
    for (;;) {
      const ItemLoad& gl = ld_next_l;
      const ItemTile& gt = ld_next_t;
      ld_live = gt.prob >= 0;
      if (!ld_live) break;
      const bool take = gt.nk > 0;   // an item without K work needs no loads
      if (take) {
        rsrc_a[0] = (int)(uint32_t)gl.a;
        rsrc_a[1] = (int)(uint32_t)(gl.a >> 32);
        rsrc_a[2] = (int)gl.a_bytes;
        rsrc_b[0] = (int)(uint32_t)gl.b;
        rsrc_b[1] = (int)(uint32_t)(gl.b >> 32);
        rsrc_b[2] = (int)gl.b_bytes;
        a_base = (uint32_t)(wave * 8 + drow) * (uint32_t)gl.lda + dchunk * 16;
        a_step = NWAVES * 8 * (uint32_t)gl.lda;
        b_base = (uint32_t)(wave * 8 + drow) * (uint32_t)gl.ldb + dchunk * 16;
        b_step = NWAVES * 8 * (uint32_t)gl.ldb;
        ld_kmax = gt.k - dchunk * 16;
        ld_kt = gt.k_begin;
        ld_nk = gt.k_begin + gt.nk;
      }
      FP8GMM_RECORD_USED(gt);
      ++r_ld;   // every list ends with an end record
      ld_next_l = item_load(r_ld);
      ld_next_t = item_tile(r_ld);
      if (take) return;
    }
    // past the end of the stream: zero fill from empty descriptors, which keeps the vmcnt arithmetic uniform
    rsrc_a[2] = 0;
    rsrc_b[2] = 0;
  };
  // the step under the cursor into a stage; rows past m / n and the K tail read as zeros
  auto load_step = [&](int stage) {
    const uint32_t k0 = (uint32_t)ld_kt * BK;
    const bool k_ok = (int)k0 < ld_kmax;
    const uint32_t dst = lds_base + stage * kRowsStage + wave * 1024;
#pragma unroll
    for (int j = 0; j < kPartsB; ++j) {
      const uint32_t v = k_ok ? b_base + k0 + j * b_step : 0xffffffffu;
      FP8GMM_DMA_STREAM(dst + kRowsUnitA + NWAVES * j * 1024, v, rsrc_b);
    }
#pragma unroll
    for (int j = 0; j < kPartsA; ++j) {
      const uint32_t v = k_ok ? a_base + k0 + j * a_step : 0xffffffffu;
      FP8GMM_DMA(dst + NWAVES * j * 1024, 0, v, rsrc_a);
    }
    if (ld_live && ++ld_kt == ld_nk) load_setup();
  };
  auto read_frag = [&](const uint8_t* base, int hh) {
    const u32x4 lo = *reinterpret_cast<const u32x4*>(base + fc[hh][0]);
    const u32x4 hi = *reinterpret_cast<const u32x4*>(base + fc[hh][1]);
    return i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
  };

  load_setup();
#pragma unroll 1
  for (int s = 0; s < kRowsStages - 1; ++s) load_step(s);
  int cur = 0;
  ItemTile cp_next = item_tile(0);
  // The running maximum of an fp8 result goes to its slot once per workgroup and run of tiles of one problem.  The slots of
  // a pass share a cache line or two, and 512 workgroups that look at one line are served one after the other: with a look
  // per wavefront and tile, 8 experts of 4096 -> 14336 columns took 137 us where slots of their own lines take 84.
  __shared__ float wave_amax[2][NWAVES];   // in turn: two runs may end without a K step's barrier in between
  int turn = 0;
  float amax = 0.f;
#pragma unroll 1
  for (int r_cp = 0;;) {
    const ItemTile g = cp_next;
    if (g.prob < 0) break;
    cp_next = item_tile(++r_cp);
    const fp8gmm_gemm_problem pr = probs[g.prob];
    const float sa = load_scale(pr.a_scale_inv), sb = load_scale(pr.b_scale_inv), cs = load_scale(pr.c_scale);
    const int blocks = (pr.m - g.m0 + 31) / 32;   // with rows, at least one
    f32x16 acc[MB] = {};
#pragma unroll 1
    for (int kt = 0; kt < g.nk; ++kt) {
      // The step's loads are older than those of the kRowsStages - 2 steps behind it.  (Result stores in between only
      // make the wait stricter.)  The barrier also says that every wavefront has read the stage of the step before -
      // lgkmcnt(0): those reads are complete, not only issued - which is the one to be filled next.
      FP8GMM_WAIT_VM_LGKM((kRowsStages - 2) * (kPartsA + kPartsB));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      load_step(cur == 0 ? kRowsStages - 1 : cur - 1);
      const uint8_t* const unit = lds + cur * kRowsStage;
      const i32x8 b0 = read_frag(unit + fb_off, 0), b1 = read_frag(unit + fb_off, 1);
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        if (i > 0 && blocks <= i) break;
        const i32x8 a0 = read_frag(unit + fa_off + i * 32 * BK, 0), a1 = read_frag(unit + fa_off + i * 32 * BK, 1);
        // source 0: weights, source 1: tokens; scales of zero select the form without them
        acc[i] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(b0, a0, acc[i], B_FMT, A_FMT, 0, 0, 0, 0);
        acc[i] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(b1, a1, acc[i], B_FMT, A_FMT, 0, 0, 0, 0);
      }
      cur = cur + 1 == kRowsStages ? 0 : cur + 1;
    }
#pragma unroll
    for (int i = 0; i < MB; ++i)
      if (i < blocks)
        amax = fmaxf(amax, store_rows_block(pr, g.m0 + i * 32 + l32, g.n0 + wave * 32 + khalf * 4, acc[i], out_kind,
                                            epilogue, sa, sb, cs));
    if (out_kind != FP8GMM_OUT_BF16 && cp_next.prob != g.prob) {
      const float own = wave_max(amax);
      if (lane == 0) wave_amax[turn][wave] = own;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (wave == 0) {
        float most = wave_amax[turn][0];
#pragma unroll
        for (int w = 1; w < NWAVES; ++w) most = fmaxf(most, wave_amax[turn][w]);
        merge_amax(pr.c_amax, most, lane);
      }
      turn ^= 1;
      amax = 0.f;
    }
  }
  // zero-fill loads issued past the end of the stream still target this workgroup's LDS
  FP8GMM_WAIT_VM(0);
}

}  // namespace fp8gmm
