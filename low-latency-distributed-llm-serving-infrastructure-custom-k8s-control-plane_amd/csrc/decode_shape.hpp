// Which decode kernel serves a shape, and how its query heads split over
// workgroups (decode.hip, decode_mfma.hip); no HIP types, for the planner.
#pragma once

namespace pa {

// Workgroups sharing one KV head's query heads: the fewest equal sub-groups
// of at most 8 heads.
int decode_sub_groups(int group);
// Workgroups one KV head's query heads take in the decode launch: the
// sub-groups, or fewer where the matrix-core kernel serves up to 16 heads a
// workgroup (the unit count stays that of the sub-groups).
int decode_workgroups_per_head(int dtype, int head_dim, int group);
// Adjacent KV heads that run as one workgroup: 2 for 16-bit heads of 64 and
// 128 in groups of up to 4 with an even KV head count, else 1.  Such units are
// what pa_decode_workgroups_per_item counts (times the sub-groups) and what
// merge records are kept for.
int decode_unit_heads(int dtype, int head_dim, int num_kv_heads, int group);
// Whether the matrix-core kernel serves the shape.
bool decode_uses_mfma(int dtype, int head_dim);

}  // namespace pa
