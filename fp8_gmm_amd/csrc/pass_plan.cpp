// Plans a whole pass of a grouped linear layer or of a grouped MLP in one call: the tensor descriptors of its cast launches,
// the problem tables of its grouped GEMMs and their work lists.  A pass is described launch by launch (pass_spec.h); the
// planning calls write its tables into host memory (fp8gmm_plan_*: staging memory, a kernel copies it), or the description
// itself becomes the argument of the kernel that writes them on the device (fp8gmm_lay_out_pass, fp8gmm_build_pass;
// pass_tables.hip).  fp8gmm_run_planned runs one planned launch.  Host code; the kernels are elsewhere.
//
// The reference does the equivalent host work per call in C++: CutlassFp8GroupedGemm builds the problem sizes,
// pointers and strides of every expert (csrc/fp8_gmm.cu:115-135) and MultiPadCastTranspose packs the tensor list
// into its kernel arguments (csrc/multi_pad_fusion.cu:455-502), driven by a Python loop over the experts
// (fp8_gmm/grouped_linear.py:109-188, fp8_gmm/grouped_mlp.py:60-318).  With 64 experts that loop (here: the array
// arithmetic that replaced it) costs more host time than the kernels run; from (group_sizes, base pointers, scaling-metadata bases) the whole
// pass is a few microseconds of C.
#include <stdint.h>
#include <string.h>

#include <initializer_list>
#include <vector>

#include "../../include/fp8gmm.h"
#include "internal.h"
#include "pass_spec.h"
#include "tiling.h"

namespace {

using fp8gmm::CastRun;
using fp8gmm::CastSpec;
using fp8gmm::GemmSpec;
using fp8gmm::PassTables;

constexpr int64_t kLine = 128;
inline int64_t align_up(int64_t x) { return (x + kLine - 1) / kLine * kLine; }
inline uint8_t* at(void* base, int64_t bytes) { return static_cast<uint8_t*>(base) + bytes; }

// The launches of a pass, in their order, as descriptions (pass_spec.h).
struct Pass {
  int experts;
  const int64_t* group_sizes;
  int grid, stream_k, tile_policy;
  struct Launch {
    bool is_cast;
    CastSpec cast;
    GemmSpec gemm;
    int a_fmt, b_fmt, out_kind, epi;
    bool two_roundings;   // a flag of the launch that its plan does not see
  };
  Launch launch[8];
  int n_launches = 0;

  Launch& add(bool is_cast) {
    Launch& l = launch[n_launches++];
    l = Launch{};
    l.is_cast = is_cast;
    return l;
  }
  CastSpec& add_cast(int op, int out_fmt) {
    CastSpec& c = add(true).cast;
    c.op = op;
    c.out_fmt = out_fmt;
    return c;
  }
  // The rows of the pass: slices of `in` [rows, cols], or what `routed` says of tokens.
  CastSpec& add_rows_cast(int fmt, const fp8gmm_routed_rows* routed, int routed_op, const void* in, void* out, int64_t cols,
                          const float* scale, float* amax, int stride) {
    CastSpec& c = add_cast(routed != nullptr ? routed_op : FP8GMM_OP_QUANTIZE, fmt);
    slices(c, in, nullptr, out, cols, scale, amax, stride);
    c.run[0].routed = routed != nullptr;
    return c;
  }
  // slices of a token-major tensor [tokens, cols]
  static void slices(CastSpec& c, const void* in, const void* in2, void* out, int64_t cols, const float* scale, float* amax,
                     int stride) {
    CastRun& r = c.run[c.n_runs++];
    r.in = in;
    r.in2 = in2;
    r.out = out;
    r.cols = cols;
    r.scale = scale;
    r.amax = amax;
    r.slot_stride = stride;
  }
  // a weight stack [experts, numel]
  static void stack(CastSpec& c, const void* in, void* out, int64_t numel, const float* scale, float* amax) {
    CastRun& r = c.run[c.n_runs++];
    r.in = in;
    r.out = out;
    r.numel = numel;
    r.scale = scale;
    r.amax = amax;
    r.slot_stride = 3;
  }
  // c[rows_i][:n] = a[rows_i][:k] . b[i]: `b` a weight stack whose expert i is n x k (kmajor: k x n, read as it lies)
  Launch& row_gemm(const void* a, const void* b, void* c, int c_bytes, void* aux, int n, int k, bool b_kmajor, int a_fmt,
                   int b_fmt, const float* a_si, int a_slot, const float* b_si) {
    Launch& l = add(false);
    GemmSpec& g = l.gemm;
    g.a = a; g.b = b; g.c = c; g.aux = aux;
    g.a_row = k;
    g.b_expert = (int64_t)n * k;
    g.c_row = n * c_bytes;
    g.aux_row = n * 2;
    g.n = n; g.k = k;
    g.lda = k; g.ldb = b_kmajor ? n : k; g.ldc = n;
    g.a_scale_inv = a_si; g.a_slot = a_slot;
    g.b_scale_inv = b_si; g.b_slot = 3;
    g.layout = b_kmajor ? FP8GMM_GEMM_B_KMAJOR : 0;
    l.a_fmt = a_fmt; l.b_fmt = b_fmt; l.out_kind = FP8GMM_OUT_BF16;
    return l;
  }
  // c[i] (m x n) = a[rows_i]^T . b[rows_i]: both operands [tokens, m] / [tokens, n], contraction over the expert's rows
  Launch& weight_gradient(const void* a, const void* b, void* c, int m, int n, int a_fmt, int b_fmt, const float* a_si,
                          const float* b_si) {
    Launch& l = add(false);
    GemmSpec& g = l.gemm;
    g.a = a; g.b = b; g.c = c;
    g.a_row = m; g.b_row = n;
    g.c_expert = (int64_t)m * n * 2;
    g.m = m; g.n = n;
    g.lda = m; g.ldb = n; g.ldc = n;
    g.a_scale_inv = a_si; g.a_slot = 2;
    g.b_scale_inv = b_si; g.b_slot = 3;
    g.layout = FP8GMM_GEMM_A_KMAJOR | FP8GMM_GEMM_B_KMAJOR;
    l.a_fmt = a_fmt; l.b_fmt = b_fmt; l.out_kind = FP8GMM_OUT_BF16;
    return l;
  }
};

// Which tile a launch takes when the caller leaves the choice to the library: the 128 x 128 tile where the
// 256 x 256 tiles would be fewer than about half the compute units or mostly padding (see FP8GMM_GEMM_TILE_128), and
// where the launch is short for other reasons: two workgroups per compute unit hide each other's starts, results and tile
// switches, which are most of a short launch, and a range's end is spread over tiles a quarter of the size.  What the form
// pays, twice the operand bytes from L2 per flop, grows with the K = 128 steps of the large tiles ("steps" below).
// Weight gradients, traced inside a layer's step, large tiles -> this form in us (profiles/tile_rules.md has all of 462):
//   * Up to 9000 steps, 8.5 a tile, whatever the number of tiles: 2048 tiles of 3.5 steps 82 -> 85, of 6.2 (12800 steps) 113 ->
//     121; 4096 of 2.0 128 -> 117, of 2.7 (10880) 144 -> 145, of 3.5 (14208) 160 -> 176; 8330 of one step 169 -> 133; 448 of 27
//     (12012) 93 -> 150.  Not results of up to 144 columns in many tiles: their second column of tiles stores pieces of 32
//     bytes (144 columns, 1988, 3478 and 4750 tiles of 1.3 - 2.3 steps 93 -> 90, 125 -> 141, 149 -> 168; 160 columns, 2444 59 -> 56).
//   * Under a skewed split large tiles wait for the longest contraction, the more the larger it is against a compute unit's
//     share of the launch, at any number of steps: at 0.75 of a share and more 64 of 1408 x 2048 with 10464 / 13632 / 16560 /
//     19872 steps 148 / 187 / 199 / 228 -> 128 / 156 / 184 / 209, 8 of 2048 x 1024 with 2400 steps 46 -> 32, 16 of 2048 x 2048 with
//     12.6 / 16.5 / 20 / 24.4 steps a tile 150 / 182 / 174 / 250 -> 121 / 159 / 197 / 257; at half a share 32 of 4096 x 2048 186 ->
//     204 and 261 -> 353.  At 2.25 shares and more also with 16 to 24 steps a tile, where five launches took 15 % less; past 24 it
//     depends on how the long contraction falls into the XCDs' ranges (0.69 - 1.53 x).
// The 385 launches that the rule takes take 15 % less time in the mean.  16 lose more than a twentieth, eleven of them skewed and
// with 6 to 16 steps a tile; the most: 7 of 5408 x 1232, 8841 rows 79 -> 104; 28 of 11376 x 192, 12965 59 -> 73; 19 of 1360 x
// 1392, 26955 87 -> 104.  Steps a tile, share and tiles do not tell them from launches that gain as much.
bool small_tiles_pay(const fp8gmm_gemm_problem* p, int n, int layout) {
  int64_t large = 0, small = 0, steps = 0, longest = 0, widest = 0;
  for (int i = 0; i < n; ++i) {
    const int64_t m = p[i].m, nn = p[i].n;
    const int64_t tiles = ((m + 255) / 256) * ((nn + 255) / 256);
    const int64_t own = p[i].k > 128 ? (p[i].k + 127) / 128 : 1;
    large += tiles;
    small += ((m + 127) / 128) * ((nn + 127) / 128);
    steps += tiles * own;
    if (tiles > 0 && own > longest) longest = own;
    if (nn > widest) widest = nn;
  }
  if (large == 0) return false;
  if (large <= 160 || 2 * small <= 5 * large) return true;
  if (!(layout & FP8GMM_GEMM_A_KMAJOR)) return false;
  if (steps <= 9000 && 2 * steps <= 17 * large) return large <= 1800 || widest > 144;
  // one expert's contraction takes three quarters of a compute unit's share of the launch, or more than twice that
  return (1024 * longest >= 3 * steps && steps <= 16 * large) || (1024 * longest >= 9 * steps && steps <= 24 * large);
}

// ... and the form with two sets of accumulators (FP8GMM_GEMM_TILE_DUAL): a contraction of up to 2048 whose
// operands and result the 256 MB memory-side cache can largely hold, operand a row-major; what the tile boundaries
// cost such a launch is more than the form's extra operand traffic.
bool dual_tiles_pay(const fp8gmm_gemm_problem* p, int n, int layout) {
  if ((layout & FP8GMM_GEMM_A_KMAJOR) || n == 0) return false;
  int64_t bytes = 0;
  int32_t k_max = 0;
  for (int i = 0; i < n; ++i) {
    const int64_t m = p[i].m, nn = p[i].n, k = p[i].k;
    bytes += (m + nn) * k + 2 * m * nn;
    if (p[i].k > k_max) k_max = p[i].k;
  }
  return k_max <= 2048 && bytes <= ((int64_t)320 << 20);
}

// Which of those launches the 128 x 128 tile is the better one for all the same: the short ones, up to two rounds of large
// tiles; at more than nine K steps, up to one round and where the last round of 128 x 256 tiles is half empty: up to 77 % of
// whole rounds; not results of a column or two of tiles, whose operand a it reads twice as often.  Traced as above, two sets ->
// this form: K = 1024, 8 experts of 2048 columns, 6000 rows 20.9 -> 18.2, 12000 34.9 -> 30.1, 18000 (592 large tiles) 41.0 ->
// 40.7, 24576 (808) 55.5 -> 55.9; 96 of 1024, K = 512, 24576 26.7 -> 24.4; 8 of 256, K = 2048, 6000 rows each 34 -> 35.  By the
// share of whole rounds, K > 1152: 0.59 - 0.77 27 launches, 1.00 - 1.20 x, 1.12 in the mean (K = 1584, 10 of 6048, 0.66 31.9 ->
// 27.6; K = 2048, 16 of 2048, 0.69 41.9 -> 38.1); 0.77 - 0.95 25 launches, 1.01 in the mean, six lose more than a twentieth (K =
// 1824, 8 of 960, 0.79 31.8 -> 34.6; K = 2000, 7 of 816, 0.88 36.6 -> 39.7).  The 109 launches that the rule takes take 14 % less
// time in the mean; one loses a twentieth (K = 1104, 33 of 960, 576 large tiles 50.0 -> 52.8).
bool small_tiles_beat_dual(const fp8gmm_gemm_problem* p, int n) {
  int64_t large = 0, dual = 0;
  int32_t k = 0, narrowest = INT32_MAX;
  for (int i = 0; i < n; ++i) {
    const int64_t columns = ((int64_t)p[i].n + 255) / 256;
    large += (((int64_t)p[i].m + 255) / 256) * columns;
    dual += (((int64_t)p[i].m + 127) / 128) * columns;
    if (p[i].k > k) k = p[i].k;
    if (p[i].n < narrowest) narrowest = p[i].n;
  }
  if (narrowest < 512) return false;
  return k <= 1152 ? large <= 600 : large <= 300 && 100 * dual <= 77 * ((dual + 255) / 256 * 256);
}

// ... and the form for few rows (FP8GMM_GEMM_TILE_ROWS): row-major weights of 64 MB or more that (nearly) every problem
// reads for one tile of up to 64 rows.  The shorter the contraction, the more of a tile is its start and its result, and
// the fewer rows it takes for the other forms to be as fast.  Measured, other forms -> this one in us, at 8 / 32 / 64 rows
// per expert: K = 14336 (8 experts, 4096 columns) 104 / 105 / 106 -> 73 / 74 / 80; K = 4096 (16, 6400) 94 / 96 / 100 ->
// 83 / 86 / 99; K = 2048 (64, 1024) 32 / 32 / 32 -> 27 / 28 / 33; K = 768 (128, 2048) 46 / 49 / 53 -> 41 / 49 / 60; K = 256
// (64, 4096) 25 -> 25 and worse; with 34 MB of weights (16, K = 1024, 2048) 12.7 -> 13.5.  With the GELU and an fp8 result,
// which the 128 x 128 form does not have, every set of weights from HBM (1.2 GB in turn): 8 / 32 / 64 rows, K = 14336 (8, 4096)
// 153 -> 84 at 8, 146 -> 86 at 64; K = 4096 (8, 14336) 128 -> 94, 126 -> 113 at 64, (32, 2048) 81 / 81 / 82 -> 64 / 65 / 68;
// K = 2048 (32, 2048) 42 / 43 -> 32 / 33, (128, 768) 62 / 62 -> 42 / 46; K = 1024 (64, 1024) 29 / 29 -> 21 / 22; K = 768
// (128, 2048) 74 -> 46 at 8, 75 -> 50 at 16; under a skewed split of 64 rows (8, K = 4096, 14336) 138 -> 147, which is more
// tiles than the rule takes.
bool rows_pay(const fp8gmm_gemm_problem* p, int n, int layout) {
  if (layout != 0) return false;
  int64_t weights = 0, rows = 0, tiles = 0, problems = 0;
  int32_t k = 0;
  for (int i = 0; i < n; ++i) {
    if (p[i].m == 0) continue;
    ++problems;
    rows += p[i].m;
    tiles += (p[i].m + FP8GMM_GEMM_ROWS_TILE_M - 1) / FP8GMM_GEMM_ROWS_TILE_M;
    weights += (int64_t)p[i].n * p[i].k;
    if (p[i].k > k) k = p[i].k;
  }
  const int64_t most = k >= 4096 ? 64 : k >= 1024 ? 32 : k >= 512 ? 16 : 0;   // rows per problem
  return weights >= ((int64_t)64 << 20) && 8 * tiles <= 9 * problems && rows <= most * problems;
}

// what the forms with two workgroups per compute unit multiply the grid by
int grid_of(int flag, int grid) { return flag == FP8GMM_GEMM_TILE_128 || flag == FP8GMM_GEMM_TILE_ROWS ? 2 * grid : grid; }

int tile_flag(const fp8gmm_gemm_problem* probs, int n, const Pass& pass, const Pass::Launch& l) {
  // (a pass's fused GELU stores e4m3 and its argument: what the form for few rows takes)
  if ((l.epi & FP8GMM_EPI_DGELU) == 0 &&
      (pass.tile_policy == FP8GMM_GEMM_TILE_ROWS ? l.gemm.layout == 0 : pass.tile_policy == 0 && rows_pay(probs, n, l.gemm.layout)))
    return FP8GMM_GEMM_TILE_ROWS;
  bool small = l.epi == 0 && (pass.tile_policy == 128 || (pass.tile_policy == 0 && small_tiles_pay(probs, n, l.gemm.layout)));
  bool dual = !small && l.epi == 0 && l.out_kind == FP8GMM_OUT_BF16 &&
              (pass.tile_policy == FP8GMM_GEMM_TILE_DUAL ||
               (pass.tile_policy == 0 && dual_tiles_pay(probs, n, l.gemm.layout)));
  if (dual && pass.tile_policy == 0 && small_tiles_beat_dual(probs, n)) {
    small = true;
    dual = false;
  }
  return small ? FP8GMM_GEMM_TILE_128 : dual ? FP8GMM_GEMM_TILE_DUAL : 0;
}

// the fields of a launch's record that do not depend on where its tables lie
int describe_cast(const Pass& pass, const Pass::Launch& l, fp8gmm_pass_launch* rec) {
  int64_t blocks = 0, work = 0;
  // quantize: 2 B read + 1 B written per element; with the GELU's derivative a second bf16 input
  const int64_t per_element = l.cast.op == FP8GMM_OP_CAST_DGELU ? 5 : 3;
  for (int r = 0; r < l.cast.n_runs; ++r)
    for (int i = 0; i < pass.experts; ++i) {
      const int64_t numel = l.cast.run[r].cols > 0 ? pass.group_sizes[i] * l.cast.run[r].cols : l.cast.run[r].numel;
      if (numel >= ((int64_t)1 << 31)) return FP8GMM_ERR_BAD_SHAPE;
      blocks += (numel + fp8gmm::kPwBlockElems - 1) / fp8gmm::kPwBlockElems;   // routed rows: whether there are any
      work += numel * per_element;
    }
  if (blocks > INT32_MAX / 2) return FP8GMM_ERR_BAD_SHAPE;
  rec->kind = blocks > 0 ? FP8GMM_PASS_CAST : FP8GMM_PASS_NOTHING;
  rec->op = l.cast.op;
  rec->n = l.cast.n_runs * pass.experts;
  rec->total_blocks = (int32_t)blocks;
  rec->out_fmt = l.cast.out_fmt;
  rec->work = (double)work;
  rec->bytes = (double)work;
  return FP8GMM_OK;
}

void describe_gemm(const Pass& pass, const Pass::Launch& l, const fp8gmm_gemm_problem* probs, fp8gmm_pass_launch* rec) {
  rec->op = 0;
  rec->n = pass.experts;
  rec->a_fmt = l.a_fmt;
  rec->b_fmt = l.b_fmt;
  rec->out_kind = l.out_kind;
  rec->epilogue = l.gemm.layout | l.epi | (l.two_roundings ? FP8GMM_EPI_TWO_ROUNDINGS : 0);
  rec->kind = rec->plan.total_tiles > 0 ? FP8GMM_PASS_GEMM : FP8GMM_PASS_NOTHING;
  double flops = 0, bytes = 0;
  for (int i = 0; i < pass.experts; ++i) {
    const double m = probs[i].m, nn = probs[i].n, k = probs[i].k;
    flops += 2.0 * m * nn * k;
    bytes += (m + nn) * k + m * nn * ((l.out_kind == FP8GMM_OUT_BF16 ? 2.0 : 1.0) + (probs[i].aux != nullptr ? 2.0 : 0.0));
  }
  rec->work = flops;
  rec->bytes = bytes;
}

void fill_problems(const Pass& pass, const GemmSpec& spec, fp8gmm_gemm_problem* probs) {
  int64_t row = 0;
  for (int i = 0; i < pass.experts; ++i) {
    probs[i] = fp8gmm::gemm_problem(spec, i, row, (int32_t)pass.group_sizes[i]);
    row += pass.group_sizes[i];
  }
}

// A cast that is directly followed by a GEMM launch leaves the merge of its tensors' running maxima into the amax
// slots to that launch's first workgroup: the small launch that would do it, and the gap around it, cost a pass of
// config 3 or 4 as much as 1.5 % each.
void defer_amax_merges(fp8gmm_pass_plan* out) {
  for (int i = 0; i + 1 < out->n_launches; ++i) {
    fp8gmm_pass_launch& cast = out->launch[i];
    fp8gmm_pass_launch& next = out->launch[i + 1];
    if (cast.kind != FP8GMM_PASS_CAST || next.kind != FP8GMM_PASS_GEMM) continue;
    cast.merge_n = cast.n;
    next.merge_n = cast.n;
    next.merge_offset = cast.table_offset;
  }
}

// ---- the tables in host memory -----------------------------------------------------------------------------------
struct Writer {
  void* blob;
  int64_t capacity;
  int64_t used = 0;        // bytes laid out so far (may exceed capacity: the pass is then only sized)
  bool fits = true;
  std::vector<std::vector<uint8_t>> aside;   // tables of a pass that does not fit: needed to size its work lists
  // `bytes` of the blob on their own cache lines; once the blob is full, memory on the side that is thrown away
  void* take(int64_t bytes, int64_t* offset) {
    *offset = used;
    used += align_up(bytes);
    if (blob == nullptr || used > capacity) {
      fits = false;
      aside.emplace_back((size_t)bytes + 1);
      return aside.back().data();
    }
    return at(blob, *offset);
  }
};

int write_pass(Pass& pass, void* blob, size_t blob_bytes, fp8gmm_pass_plan* out) {
  Writer w{blob, (int64_t)blob_bytes};
  const int e = pass.experts;
  for (int q = 0; q < pass.n_launches; ++q) {
    Pass::Launch& l = pass.launch[q];
    fp8gmm_pass_launch* rec = &out->launch[q];
    if (l.is_cast) {
      int rc = describe_cast(pass, l, rec);
      if (rc != FP8GMM_OK) return rc;
      const int n = rec->n;
      fp8gmm_tensor_desc* d = static_cast<fp8gmm_tensor_desc*>(
          w.take((int64_t)n * (int64_t)sizeof(fp8gmm_tensor_desc), &rec->table_offset));
      for (int r = 0; r < l.cast.n_runs; ++r) {
        int64_t row = 0;
        for (int i = 0; i < e; ++i) {
          d[r * e + i] = fp8gmm::cast_desc(l.cast.run[r], i, row, pass.group_sizes[i]);
          row += pass.group_sizes[i];
        }
      }
      int total = 0;
      rc = fp8gmm_plan_multi_tensor(d, n, l.cast.op, &total);
      if (rc != FP8GMM_OK) return rc;
      continue;
    }
    fp8gmm_gemm_problem* probs = static_cast<fp8gmm_gemm_problem*>(
        w.take((int64_t)e * (int64_t)sizeof(fp8gmm_gemm_problem), &rec->table_offset));
    fill_problems(pass, l.gemm, probs);
    const int flag = tile_flag(probs, e, pass, l);
    // room for the work list: whatever is left of the blob
    int64_t room = w.fits ? (w.capacity - w.used) / (int64_t)sizeof(fp8gmm_gemm_item) : 0;
    if (room > INT32_MAX) room = INT32_MAX;
    if (room < 0) room = 0;
    fp8gmm_gemm_item* items = room > 0 ? reinterpret_cast<fp8gmm_gemm_item*>(at(w.blob, w.used)) : nullptr;
    // shared-tile records are few (at most one per workgroup): planned into a local array, appended afterwards
    static thread_local fp8gmm_gemm_fixup_desc fix[4096];
    const int rc = fp8gmm_plan_grouped_gemm_launch(
        probs, e, l.gemm.layout | l.epi | (flag != 0 ? flag : FP8GMM_GEMM_BALANCED), grid_of(flag, pass.grid),
        flag != 0 ? 0 : pass.stream_k, items, (int)room, fix, 4096, &rec->plan);
    if (rc != FP8GMM_OK && rc != FP8GMM_ERR_BUFFER_TOO_SMALL) return rc;
    if (rc == FP8GMM_ERR_BUFFER_TOO_SMALL) w.fits = false;
    // the work list lies where it was planned (w.used has not moved since); when it did not fit it is only counted
    rec->items_offset = w.used;
    w.used += align_up((int64_t)rec->plan.rounds * rec->plan.grid * (int64_t)sizeof(fp8gmm_gemm_item));
    if (w.used > w.capacity) w.fits = false;
    void* fix_dst = w.take((int64_t)rec->plan.n_fixups * (int64_t)sizeof(fp8gmm_gemm_fixup_desc), &rec->fixups_offset);
    if (rec->plan.n_fixups > 0) memcpy(fix_dst, fix, (size_t)rec->plan.n_fixups * sizeof(fp8gmm_gemm_fixup_desc));
    describe_gemm(pass, l, probs, rec);
  }
  out->n_launches = pass.n_launches;
  out->blob_bytes = w.used;
  defer_amax_merges(out);
  return w.fits ? FP8GMM_OK : FP8GMM_ERR_BUFFER_TOO_SMALL;
}

// ---- the tables in device memory: the same layout, described for the table kernel ---------------------------------
int lay_out_pass(Pass& pass, fp8gmm_pass_plan* out, PassTables* t) {
  const int e = pass.experts;
  if (e > fp8gmm::kPassMaxExperts || 2 * pass.grid > FP8GMM_PASS_MAX_GRID || pass.grid > fp8gmm::kPassMaxExperts)
    return FP8GMM_ERR_BAD_ARGUMENT;
  t->experts = e;
  t->n_casts = t->n_gemms = 0;
  int64_t rows = 0;
  t->row_begin[0] = 0;
  for (int i = 0; i < e; ++i) {
    rows += pass.group_sizes[i];
    if (pass.group_sizes[i] > INT32_MAX / 2 || rows > FP8GMM_PASS_MAX_ROWS) return FP8GMM_ERR_BAD_SHAPE;
    t->row_begin[i + 1] = (int32_t)rows;
  }
  static thread_local std::vector<fp8gmm_gemm_problem> scratch;
  scratch.resize((size_t)e + 1);
  fp8gmm_gemm_problem* probs = scratch.data();
  int64_t used = 0;
  auto take = [&](int64_t bytes) {
    const int64_t offset = used;
    used += align_up(bytes);
    return offset;
  };
  for (int q = 0; q < pass.n_launches; ++q) {
    Pass::Launch& l = pass.launch[q];
    fp8gmm_pass_launch* rec = &out->launch[q];
    if (l.is_cast) {
      const int rc = describe_cast(pass, l, rec);
      if (rc != FP8GMM_OK) return rc;
      rec->table_offset = l.cast.table_offset = take((int64_t)rec->n * (int64_t)sizeof(fp8gmm_tensor_desc));
      t->cast[t->n_casts++] = l.cast;
      continue;
    }
    fill_problems(pass, l.gemm, probs);
    const int flag = tile_flag(probs, e, pass, l);
    fp8gmm::GemmRanges* ranges = &t->ranges[t->n_gemms];
    const int rc = fp8gmm::plan_gemm_ranges(probs, e, l.gemm.layout | l.epi | (flag != 0 ? flag : FP8GMM_GEMM_BALANCED),
                                            grid_of(flag, pass.grid),
                                            flag != 0 ? 0 : pass.stream_k, &rec->plan, ranges);
    if (rc != FP8GMM_OK) return rc;
    l.gemm.tile_n = rec->plan.tile != 0 ? rec->plan.tile : fp8gmm::kGemmTileN;
    l.gemm.tile_m = rec->plan.tile_m != 0 ? rec->plan.tile_m : l.gemm.tile_n;
    rec->table_offset = l.gemm.table_offset = take((int64_t)e * (int64_t)sizeof(fp8gmm_gemm_problem));
    rec->items_offset = l.gemm.items_offset = take((int64_t)ranges->rounds * ranges->grid * (int64_t)sizeof(fp8gmm_gemm_item));
    rec->fixups_offset = l.gemm.fixups_offset = take((int64_t)ranges->n_fixups * (int64_t)sizeof(fp8gmm_gemm_fixup_desc));
    describe_gemm(pass, l, probs, rec);
    t->gemm[t->n_gemms++] = l.gemm;
  }
  // the table kernel's workgroups: one per cast, one per kPassRecordsPerBlock records of a work list
  int blocks = 0;
  for (int c = 0; c < t->n_casts; ++c) t->first_block[c] = blocks++;
  for (int g = 0; g < t->n_gemms; ++g) {
    t->first_block[t->n_casts + g] = blocks;
    const int records = t->ranges[g].rounds * t->ranges[g].grid;
    blocks += records > 0 ? (records + fp8gmm::kPassRecordsPerBlock - 1) / fp8gmm::kPassRecordsPerBlock : 1;
  }
  t->blocks = e > 0 ? blocks : 0;
  out->n_launches = pass.n_launches;
  out->blob_bytes = used;
  defer_amax_merges(out);
  return FP8GMM_OK;
}

int check_sizes(int experts, const int64_t* group_sizes, int64_t tokens) {
  if (experts > 0 && group_sizes == nullptr) return FP8GMM_ERR_NULL_POINTER;
  int64_t rows = 0;
  for (int i = 0; i < experts; ++i) {
    if (group_sizes[i] < 0) return FP8GMM_ERR_BAD_SHAPE;
    rows += group_sizes[i];
  }
  return rows == tokens ? FP8GMM_OK : FP8GMM_ERR_BAD_SHAPE;
}
// Token-major tensors of a pass: one without rows has no memory, and none of it is touched.
template <class Desc>
bool rows_missing(const Desc* s, std::initializer_list<const void*> tensors) {
  if (s->tokens == 0) return false;
  for (const void* t : tensors)
    if (t == nullptr) return true;
  return false;
}
// What the kernels of routed rows follow: `tensors` are the token-major tensors of the pass that they read or write.
int check_routed(const fp8gmm_routed_rows* r, int64_t tokens, bool backward, std::initializer_list<const void*> tensors) {
  if (r == nullptr) return FP8GMM_OK;
  if (r->top_k < 1 || r->top_k > FP8GMM_ROUTED_MAX_TOP_K || tokens % r->top_k != 0 || tokens > INT32_MAX)
    return FP8GMM_ERR_BAD_ARGUMENT;
  if (tokens == 0) return FP8GMM_OK;
  if (r->inverse == nullptr || (backward && r->weights == nullptr)) return FP8GMM_ERR_NULL_POINTER;
  if (backward && r->grad_weights != nullptr && r->y == nullptr) return FP8GMM_ERR_NULL_POINTER;
  uintptr_t low = backward ? reinterpret_cast<uintptr_t>(r->y) : 0;
  for (const void* t : tensors) low |= reinterpret_cast<uintptr_t>(t);
  return (low & 15) == 0 ? FP8GMM_OK : FP8GMM_ERR_ALIGNMENT;
}
bool tile_policy_ok(int p) { return p == 0 || p == 128 || p == 256 || p == FP8GMM_GEMM_TILE_DUAL || p == FP8GMM_GEMM_TILE_ROWS; }

void begin_pass(Pass& p, int experts, const int64_t* sizes, int grid, int stream_k, int tile_policy) {
  p.experts = experts;
  p.group_sizes = sizes;
  p.grid = grid;
  p.stream_k = stream_k;
  p.tile_policy = tile_policy;
}

int check_common(const fp8gmm_linear_pass* s) {
  if (s == nullptr) return FP8GMM_ERR_NULL_POINTER;
  if (s->experts < 0 || s->in_features <= 0 || s->out_features <= 0 || s->grid <= 0) return FP8GMM_ERR_BAD_ARGUMENT;
  if (s->experts > 0 && s->group_sizes == nullptr) return FP8GMM_ERR_NULL_POINTER;
  if ((s->in_features % 16) != 0 || (s->out_features % 16) != 0) return FP8GMM_ERR_ALIGNMENT;
  if (!tile_policy_ok(s->tile_policy)) return FP8GMM_ERR_BAD_ARGUMENT;
  const int rc = check_sizes(s->experts, s->group_sizes, s->tokens);
  if (rc != FP8GMM_OK) return rc;
  const int64_t widest = s->in_features > s->out_features ? s->in_features : s->out_features;
  if (s->tokens * widest >= ((int64_t)1 << 31) * 64) return FP8GMM_ERR_BAD_SHAPE;
  return FP8GMM_OK;
}

int linear_forward(const fp8gmm_linear_pass* s, const fp8gmm_routed_rows* routed, Pass& p) {
  const int rc = check_common(s);
  if (rc != FP8GMM_OK) return rc;
  if (rows_missing(s, {s->x, s->x_fp8, s->y}) || s->w_fp8 == nullptr || s->fwd_scale == nullptr ||
      s->fwd_scale_inv == nullptr || s->fwd_amax == nullptr || (s->cast_weights && s->w == nullptr))
    return FP8GMM_ERR_NULL_POINTER;
  const int K = s->in_features, N = s->out_features;
  if ((int64_t)N * K >= ((int64_t)1 << 31)) return FP8GMM_ERR_BAD_SHAPE;
  const int routed_rc = check_routed(routed, s->tokens, false, {s->x, s->x_fp8});
  if (routed_rc != FP8GMM_OK) return routed_rc;
  begin_pass(p, s->experts, s->group_sizes, s->grid, s->stream_k, s->tile_policy);
  // cast: the experts' activation slices, then (unless cached copies are reused) their weights; routed rows have a launch of
  // their own, right in front of the GEMM that reads them
  if (routed != nullptr && s->cast_weights)
    Pass::stack(p.add_cast(FP8GMM_OP_QUANTIZE, s->fwd_fmt), s->w, s->w_fp8, (int64_t)N * K, s->fwd_scale + 1, s->fwd_amax + 1);
  CastSpec& cast = p.add_rows_cast(s->fwd_fmt, routed, FP8GMM_OP_ROUTED_CAST, s->x, s->x_fp8, K, s->fwd_scale, s->fwd_amax, 3);
  if (routed == nullptr && s->cast_weights)
    Pass::stack(cast, s->w, s->w_fp8, (int64_t)N * K, s->fwd_scale + 1, s->fwd_amax + 1);
  // y[rows of expert i] = x_fp8[rows] . w_fp8[i]^T
  p.row_gemm(s->x_fp8, s->w_fp8, s->y, 2, nullptr, N, K, false, s->fwd_fmt, s->fwd_fmt, s->fwd_scale_inv, 3,
             s->fwd_scale_inv + 1).two_roundings = s->two_roundings != 0;
  return FP8GMM_OK;
}

int linear_backward(const fp8gmm_linear_pass* s, const fp8gmm_routed_rows* routed, Pass& p) {
  const int rc = check_common(s);
  if (rc != FP8GMM_OK) return rc;
  if (rows_missing(s, {s->dy, s->dy_fp8}) || s->bwd_scale == nullptr || s->bwd_scale_inv == nullptr ||
      s->bwd_amax == nullptr || s->fwd_scale_inv == nullptr)
    return FP8GMM_ERR_NULL_POINTER;
  if ((s->dgrad && (rows_missing(s, {s->dx}) || s->w_fp8 == nullptr)) ||
      (s->wgrad && (s->dw == nullptr || rows_missing(s, {s->x_fp8}))))
    return FP8GMM_ERR_NULL_POINTER;
  const int K = s->in_features, N = s->out_features;
  const int routed_rc = check_routed(routed, s->tokens, true, {s->dy, s->dy_fp8});
  if (routed_rc != FP8GMM_OK) return routed_rc;
  begin_pass(p, s->experts, s->group_sizes, s->grid, s->stream_k, s->tile_policy);
  p.add_rows_cast(s->bwd_fmt, routed, FP8GMM_OP_ROUTED_GRADIENT, s->dy, s->dy_fp8, N, s->bwd_scale, s->bwd_amax, 2);
  // dw[i] = dy_fp8[rows]^T . x_fp8[rows]: both read in place, contraction over the expert's rows.  Ahead of the data
  // gradient: its operands are the tensors the casts have just written, and a launch that reads them later, behind
  // the data gradient's pass over all the weights, finds less of them in the memory-side cache (config 3: 139 -> 126 us)
  if (s->wgrad)
    p.weight_gradient(s->dy_fp8, s->x_fp8, s->dw, N, K, s->bwd_fmt, s->fwd_fmt, s->bwd_scale_inv, s->fwd_scale_inv);
  // dx[rows] = dy_fp8[rows] . w_fp8[i]: the forward weight [N, K] read in place as b[k = N][n = K]
  if (s->dgrad)
    p.row_gemm(s->dy_fp8, s->w_fp8, s->dx, 2, nullptr, K, N, true, s->bwd_fmt, s->fwd_fmt, s->bwd_scale_inv, 2,
               s->fwd_scale_inv + 1).two_roundings = s->two_roundings != 0;
  return FP8GMM_OK;
}

int check_mlp(const fp8gmm_mlp_pass* s) {
  if (s == nullptr) return FP8GMM_ERR_NULL_POINTER;
  if (s->experts < 0 || s->hidden <= 0 || s->ffn <= 0 || s->grid <= 0) return FP8GMM_ERR_BAD_ARGUMENT;
  if (s->experts > 0 && s->group_sizes == nullptr) return FP8GMM_ERR_NULL_POINTER;
  if ((s->hidden % 16) != 0 || (s->ffn % 16) != 0) return FP8GMM_ERR_ALIGNMENT;
  if (!tile_policy_ok(s->tile_policy)) return FP8GMM_ERR_BAD_ARGUMENT;
  const int64_t widest = s->hidden > s->ffn ? s->hidden : s->ffn;
  for (int i = 0; i < s->experts; ++i)
    if (s->group_sizes[i] < 0 || s->group_sizes[i] * widest >= ((int64_t)1 << 31)) return FP8GMM_ERR_BAD_SHAPE;
  const int rc = check_sizes(s->experts, s->group_sizes, s->tokens);
  if (rc != FP8GMM_OK) return rc;
  if (s->tokens * widest >= ((int64_t)1 << 31) * 64 || (int64_t)s->hidden * s->ffn >= ((int64_t)1 << 31))
    return FP8GMM_ERR_BAD_SHAPE;
  return FP8GMM_OK;
}

int mlp_forward(const fp8gmm_mlp_pass* s, const fp8gmm_routed_rows* routed, Pass& p) {
  const int rc = check_mlp(s);
  if (rc != FP8GMM_OK) return rc;
  if (rows_missing(s, {s->x, s->x_fp8, s->pre, s->act_fp8, s->y}) || s->w1_fp8 == nullptr || s->w2_fp8 == nullptr ||
      s->fwd_scale == nullptr || s->fwd_scale_inv == nullptr || s->fwd_amax == nullptr ||
      (s->cast_weights && (s->w1 == nullptr || s->w2 == nullptr)))
    return FP8GMM_ERR_NULL_POINTER;
  const int H = s->hidden, F = s->ffn;
  const int64_t g2 = 3 * (int64_t)s->experts;   // first forward slot of the fc2 GEMMs
  const int routed_rc = check_routed(routed, s->tokens, false, {s->x, s->x_fp8});
  if (routed_rc != FP8GMM_OK) return routed_rc;
  begin_pass(p, s->experts, s->group_sizes, s->grid, s->stream_k, s->tile_policy);
  // cast.  fc2's weights first and the input last: the launch walks its table in order, and what it wrote last is
  // what the memory-side cache still holds when fc1's GEMM starts reading
  if (s->cast_weights) {
    CastSpec& cast = p.add_cast(FP8GMM_OP_QUANTIZE, s->fwd_fmt);
    Pass::stack(cast, s->w2, s->w2_fp8, (int64_t)H * F, s->fwd_scale + g2 + 1, s->fwd_amax + g2 + 1);
    Pass::stack(cast, s->w1, s->w1_fp8, (int64_t)H * F, s->fwd_scale + 1, s->fwd_amax + 1);
    if (routed == nullptr) Pass::slices(cast, s->x, nullptr, s->x_fp8, H, s->fwd_scale, s->fwd_amax, 3);
  }
  if (routed != nullptr || !s->cast_weights)
    p.add_rows_cast(s->fwd_fmt, routed, FP8GMM_OP_ROUTED_CAST, s->x, s->x_fp8, H, s->fwd_scale, s->fwd_amax, 3);
  // fc1 with the GELU in its epilogue: pre (bf16) and act_fp8 = fp8(gelu(pre) * scale of fc2's input)
  Pass::Launch& fc1 = p.row_gemm(s->x_fp8, s->w1_fp8, s->act_fp8, 1, s->pre, F, H, false, s->fwd_fmt, s->fwd_fmt,
                                 s->fwd_scale_inv, 3, s->fwd_scale_inv + 1);
  fc1.gemm.c_scale = s->fwd_scale + g2;
  fc1.gemm.c_amax = s->fwd_amax + g2;
  fc1.out_kind = s->fwd_fmt;   // an fp8 result's out_kind is its format
  fc1.epi = FP8GMM_EPI_GELU;
  p.row_gemm(s->act_fp8, s->w2_fp8, s->y, 2, nullptr, H, F, false, s->fwd_fmt, s->fwd_fmt, s->fwd_scale_inv + g2, 3,
             s->fwd_scale_inv + g2 + 1);
  return FP8GMM_OK;
}

int mlp_backward(const fp8gmm_mlp_pass* s, const fp8gmm_routed_rows* routed, Pass& p) {
  const int rc = check_mlp(s);
  if (rc != FP8GMM_OK) return rc;
  if (rows_missing(s, {s->dy, s->dy_fp8, s->pre, s->dact, s->dpre_fp8}) || s->w2_fp8 == nullptr ||
      s->bwd_scale == nullptr || s->bwd_scale_inv == nullptr || s->bwd_amax == nullptr || s->fwd_scale_inv == nullptr)
    return FP8GMM_ERR_NULL_POINTER;
  if ((s->dgrad && (rows_missing(s, {s->dx}) || s->w1_fp8 == nullptr)) ||
      (s->wgrad && (s->dw1 == nullptr || s->dw2 == nullptr || rows_missing(s, {s->x_fp8, s->act_fp8}))))
    return FP8GMM_ERR_NULL_POINTER;
  const int H = s->hidden, F = s->ffn;
  const int64_t f2 = 3 * (int64_t)s->experts, b2 = 2 * (int64_t)s->experts;   // first slots of the fc2 GEMMs
  const int routed_rc = check_routed(routed, s->tokens, true, {s->dy, s->dy_fp8});
  if (routed_rc != FP8GMM_OK) return routed_rc;
  begin_pass(p, s->experts, s->group_sizes, s->grid, s->stream_k, s->tile_policy);
  // cast of the gradient.  It takes the first group of backward slots although it belongs to fc2, and the
  // gradient of pre the second (fp8_gmm/grouped_mlp.py:183-184,278-279): the groups follow the order of the pass
  p.add_rows_cast(s->bwd_fmt, routed, FP8GMM_OP_ROUTED_GRADIENT, s->dy, s->dy_fp8, H, s->bwd_scale, s->bwd_amax, 2);
  // dw2[i] (H x F) = dy_fp8[rows_i]^T . act_fp8[rows_i]
  if (s->wgrad)
    p.weight_gradient(s->dy_fp8, s->act_fp8, s->dw2, H, F, s->bwd_fmt, s->fwd_fmt, s->bwd_scale_inv, s->fwd_scale_inv + f2);
  // dact[rows_i] = dy_fp8[rows_i] . w2_fp8[i]   (w2[i] is H x F: read in place as b[k = H][n = F])
  p.row_gemm(s->dy_fp8, s->w2_fp8, s->dact, 2, nullptr, F, H, true, s->bwd_fmt, s->fwd_fmt, s->bwd_scale_inv, 2,
             s->fwd_scale_inv + f2 + 1);
  // dpre_fp8 = fp8(dact * dgelu(pre))
  CastSpec& dgelu = p.add_cast(FP8GMM_OP_CAST_DGELU, s->bwd_fmt);
  Pass::slices(dgelu, s->dact, s->pre, s->dpre_fp8, F, s->bwd_scale + b2, s->bwd_amax + b2, 2);
  // dx[rows_i] = dpre_fp8[rows_i] . w1_fp8[i]   (w1[i] is F x H: b[k = F][n = H])
  if (s->dgrad)
    p.row_gemm(s->dpre_fp8, s->w1_fp8, s->dx, 2, nullptr, H, F, true, s->bwd_fmt, s->fwd_fmt, s->bwd_scale_inv + b2, 2,
               s->fwd_scale_inv + 1);
  // dw1[i] (F x H) = dpre_fp8[rows_i]^T . x_fp8[rows_i]
  if (s->wgrad)
    p.weight_gradient(s->dpre_fp8, s->x_fp8, s->dw1, F, H, s->bwd_fmt, s->fwd_fmt, s->bwd_scale_inv + b2, s->fwd_scale_inv);
  return FP8GMM_OK;
}

template <class Desc>
int plan_pass(int (*describe)(const Desc*, const fp8gmm_routed_rows*, Pass&), const Desc* desc, void* blob, size_t blob_bytes, fp8gmm_pass_plan* out) {
  if (out == nullptr) return FP8GMM_ERR_NULL_POINTER;
  Pass pass;
  const int rc = describe(desc, nullptr, pass);
  if (rc != FP8GMM_OK) return rc;
  memset(out, 0, sizeof(*out));
  return write_pass(pass, blob, blob_bytes, out);
}

}  // namespace

extern "C" {

int fp8gmm_plan_linear_forward(const fp8gmm_linear_pass* s, void* blob, size_t blob_bytes, fp8gmm_pass_plan* out) {
  return plan_pass(linear_forward, s, blob, blob_bytes, out);
}
int fp8gmm_plan_linear_backward(const fp8gmm_linear_pass* s, void* blob, size_t blob_bytes, fp8gmm_pass_plan* out) {
  return plan_pass(linear_backward, s, blob, blob_bytes, out);
}
int fp8gmm_plan_mlp_forward(const fp8gmm_mlp_pass* s, void* blob, size_t blob_bytes, fp8gmm_pass_plan* out) {
  return plan_pass(mlp_forward, s, blob, blob_bytes, out);
}
int fp8gmm_plan_mlp_backward(const fp8gmm_mlp_pass* s, void* blob, size_t blob_bytes, fp8gmm_pass_plan* out) {
  return plan_pass(mlp_backward, s, blob, blob_bytes, out);
}

int fp8gmm_lay_out_routed_pass(int which, const void* desc, const fp8gmm_routed_rows* routed, fp8gmm_pass_plan* out,
                               void* tables) {
  if (out == nullptr || desc == nullptr || tables == nullptr) return FP8GMM_ERR_NULL_POINTER;
  Pass pass;
  int rc = FP8GMM_ERR_BAD_ARGUMENT;
  switch (which) {
    case FP8GMM_LINEAR_FORWARD: rc = linear_forward(static_cast<const fp8gmm_linear_pass*>(desc), routed, pass); break;
    case FP8GMM_LINEAR_BACKWARD: rc = linear_backward(static_cast<const fp8gmm_linear_pass*>(desc), routed, pass); break;
    case FP8GMM_MLP_FORWARD: rc = mlp_forward(static_cast<const fp8gmm_mlp_pass*>(desc), routed, pass); break;
    case FP8GMM_MLP_BACKWARD: rc = mlp_backward(static_cast<const fp8gmm_mlp_pass*>(desc), routed, pass); break;
    default: break;
  }
  if (rc != FP8GMM_OK) return rc;
  memset(out, 0, sizeof(*out));
  rc = lay_out_pass(pass, out, static_cast<PassTables*>(tables));
  if (rc != FP8GMM_OK || routed == nullptr) return rc;
  for (int i = 0; i < out->n_launches; ++i) {
    fp8gmm_pass_launch& l = out->launch[i];
    if (l.op != FP8GMM_OP_ROUTED_CAST && l.op != FP8GMM_OP_ROUTED_GRADIENT) continue;
    // described as a cast of its rows: 2 B read + 1 B written per element.  A token is read once, a row of y once.
    const bool reads_y = l.op == FP8GMM_OP_ROUTED_GRADIENT && routed->grad_weights != nullptr;
    l.work = l.bytes = l.work / 3 * (1 + 2.0 / routed->top_k + (reads_y ? 2 : 0));
  }
  return FP8GMM_OK;
}

int fp8gmm_lay_out_pass(int which, const void* desc, fp8gmm_pass_plan* out, void* tables) {
  return fp8gmm_lay_out_routed_pass(which, desc, nullptr, out, tables);
}

int fp8gmm_build_pass(const void* tables, void* blob_dev, const fp8gmm_scaling_update* updates, int n_updates,
                      const float* copy_src, float* copy_dst, int copy_n, void* stream) {
  if (tables == nullptr || copy_n < 0 || (copy_n > 0 && (copy_src == nullptr || copy_dst == nullptr)))
    return FP8GMM_ERR_NULL_POINTER;
  const PassTables* t = static_cast<const PassTables*>(tables);
  if (t->blocks > 0 && blob_dev == nullptr) return FP8GMM_ERR_NULL_POINTER;
  return fp8gmm::launch_pass_tables(*t, blob_dev, updates, n_updates, copy_src, copy_dst, copy_n, stream);
}

int fp8gmm_run_planned(const void* blob_dev, const fp8gmm_pass_launch* rec, void* workspace, size_t workspace_bytes,
                       void* stream) {
  return fp8gmm_run_routed(blob_dev, rec, nullptr, 0, workspace, workspace_bytes, stream);
}

int fp8gmm_run_routed(const void* blob_dev, const fp8gmm_pass_launch* rec, const fp8gmm_routed_rows* routed, int64_t rows,
                      void* workspace, size_t workspace_bytes, void* stream) {
  if (rec == nullptr) return FP8GMM_ERR_NULL_POINTER;
  if (rec->kind == FP8GMM_PASS_NOTHING) return FP8GMM_OK;
  if (blob_dev == nullptr) return FP8GMM_ERR_NULL_POINTER;
  uint8_t* base = const_cast<uint8_t*>(static_cast<const uint8_t*>(blob_dev));
  if (rec->kind == FP8GMM_PASS_CAST) {
    fp8gmm_tensor_desc* descs = reinterpret_cast<fp8gmm_tensor_desc*>(base + rec->table_offset);
    switch (rec->op) {
      case FP8GMM_OP_QUANTIZE:
        if (rec->merge_n != 0)
          return fp8gmm::launch_cast_unmerged(descs, rec->n, rec->total_blocks, rec->out_fmt, false, stream);
        return fp8gmm_multi_quantize(descs, rec->n, rec->total_blocks, rec->out_fmt, stream);
      case FP8GMM_OP_CAST_DGELU:
        if (rec->merge_n != 0)
          return fp8gmm::launch_cast_unmerged(descs, rec->n, rec->total_blocks, rec->out_fmt, true, stream);
        return fp8gmm_multi_cast_dgelu(descs, rec->n, rec->total_blocks, rec->out_fmt, stream);
      case FP8GMM_OP_ROUTED_CAST:
      case FP8GMM_OP_ROUTED_GRADIENT:
        if (routed == nullptr) return FP8GMM_ERR_NULL_POINTER;
        return fp8gmm::launch_routed_cast(descs, rec->n, rec->op, rec->out_fmt, *routed, rows, rec->merge_n == 0, stream);
      default: return FP8GMM_ERR_BAD_ARGUMENT;
    }
  }
  if (rec->kind == FP8GMM_PASS_GEMM) {
    const fp8gmm_gemm_fixup_desc* fix =
        rec->plan.n_fixups > 0 ? reinterpret_cast<const fp8gmm_gemm_fixup_desc*>(base + rec->fixups_offset) : nullptr;
    return fp8gmm::launch_gemm_merging(
        reinterpret_cast<const fp8gmm_gemm_problem*>(base + rec->table_offset), rec->n,
        reinterpret_cast<const fp8gmm_gemm_item*>(base + rec->items_offset), fix, &rec->plan, rec->a_fmt, rec->b_fmt,
        rec->out_kind, rec->epilogue, workspace, workspace_bytes,
        rec->merge_n > 0 ? reinterpret_cast<const fp8gmm_tensor_desc*>(base + rec->merge_offset) : nullptr, rec->merge_n,
        stream);
  }
  return FP8GMM_ERR_BAD_ARGUMENT;
}

size_t fp8gmm_sizeof_linear_pass(void) { return sizeof(fp8gmm_linear_pass); }
size_t fp8gmm_sizeof_mlp_pass(void) { return sizeof(fp8gmm_mlp_pass); }
size_t fp8gmm_sizeof_pass_plan(void) { return sizeof(fp8gmm_pass_plan); }

}  // extern "C"
