// Entry points that one source file of the library offers another; not part of the C ABI.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "../../include/fp8gmm.h"

namespace fp8gmm {

// fp8gmm_multi_quantize / fp8gmm_multi_cast_dgelu without their second launch, the one that merges the tensors'
// running maxima into the callers' amax slots: the caller hands the table to the GEMM launch that follows
// (launch_gemm_merging), whose first workgroup does the merge before it starts on its tiles.  Two small launches
// fewer per pass of a module.
int launch_cast_unmerged(fp8gmm_tensor_desc* descs_dev, int n, int total_blocks, int out_fmt, bool dgelu, void* stream);

// fp8gmm_grouped_gemm, with the amax merge of the `merge_n` cast descriptors at `merge_descs` in front.
int launch_gemm_merging(const fp8gmm_gemm_problem* probs_dev, int n, const fp8gmm_gemm_item* items_dev,
                        const fp8gmm_gemm_fixup_desc* fixups_dev, const fp8gmm_gemm_plan* plan, int a_fmt, int b_fmt,
                        int out_kind, int epilogue, void* workspace, size_t workspace_bytes,
                        const fp8gmm_tensor_desc* merge_descs, int merge_n, void* stream);

// The casts of routed rows (FP8GMM_OP_ROUTED_*, fp8gmm_routed_rows), `rows` of them in all; without `merge` the merge of the
// experts' maxima is left to the GEMM launch that follows, as above.
int launch_routed_cast(fp8gmm_tensor_desc* descs_dev, int n, int op, int out_fmt, const fp8gmm_routed_rows& routed, int64_t rows,
                       bool merge, void* stream);

struct GemmRanges;
struct PassTables;

// fp8gmm_plan_grouped_gemm_launch without the records: the sizes of the launch and, per XCD, the ranges that the records
// follow from (pass_spec.h).  The same decisions from the same code.
int plan_gemm_ranges(fp8gmm_gemm_problem* probs, int n, int layout, int grid, int stream_k, fp8gmm_gemm_plan* plan,
                     GemmRanges* out);

// Writes the tables of a pass into device memory, runs up to two scaling updates and copies `copy_n` floats on the
// side, in one launch (pass_tables.hip).
int launch_pass_tables(const PassTables& tables, void* blob_dev, const fp8gmm_scaling_update* updates, int n_updates,
                       const float* copy_src, float* copy_dst, int copy_n, void* stream);

}  // namespace fp8gmm
