// Launcher of the fused Q/K/V preparation (kernels and their order: prep_fused_kernels.hpp).
#include "prep_fused_kernels.hpp"

namespace risa {

bool can_prepare_fused(const QkArgs& qk, const ValueArgs& v) {
  return qk.k_len == v.length &&
         qk.batch == v.batch && qk.kv_heads == v.heads && qk.head_dim == v.head_dim &&
         qk.cta_k == v.cta_k && qk.dtype == v.dtype;
}

int launch_prepare_fused(const QkArgs& qk, const ValueArgs& v, hipStream_t stream) {
  if (!can_prepare_fused(qk, v)) return fail("risa_sdpa: operands do not qualify for the fused preparation");
  if (v.workspace_bytes < value_workspace_bytes(v.batch, v.heads, v.length, v.head_dim, v.midpoint_affine))
    return fail("risa_quantize_v: workspace is too small");
  const Workspace w = carve(v.workspace, v.batch, v.heads, v.length, v.head_dim, v.midpoint_affine);
  FusedArgs a{};
  a.qk = qk;
  a.v = v;
  a.part_max = w.part_max;
  a.part_min = w.part_min;
  a.inverse = w.inverse;
  a.midpoint = w.midpoint;
  a.partial = w.partial;
  const int slice_rows = qk.head_dim == 256 ? 16 : 32;
  a.q_slices = (qk.q_len + 127) / 128 * (128 / slice_rows);
  a.q_blocks = a.q_slices * qk.q_heads * qk.batch;
  a.kv = qk.batch * qk.kv_heads;
  a.anchor_blocks = a.kv;
  a.chunks = range_chunks(v.length);
  // Long absmax sequences whose Q work covers the longer V range walks: fewer, longer chunks,
  // so that the code blocks reduce the partial ranges themselves (no parameter launch).  Half as much
  // Q as V does: 24 heads x 4096 x 8000 x 64 33.8 -> 30.4 us, 40 x 8192 x 16000 x 128 156.7 -> 151.4,
  // 16/4 x 2048 x 16000 x 128 23.9 -> 23.4 (less was not measured).  The
  // long midpoint_affine path keeps the stored parameters its residual blocks read.
  if (!v.midpoint_affine && 2 * static_cast<int64_t>(qk.q_len) * qk.q_heads >= static_cast<int64_t>(v.length) * v.heads)
    a.chunks = capped_range_chunks(v.length);
  a.range_groups = (a.chunks + 3) / 4;
  a.key_tiles = (qk.k_len + qk.cta_k - 1) / qk.cta_k;
  a.key_blocks = 2 * a.key_tiles * a.kv;  // half a tile per workgroup
  a.code_blocks_x = (v.padded + kCodeBlockPositions - 1) / kCodeBlockPositions;
  a.q_wide = rows_are_16_byte_aligned(qk.q, qk.q_stride_b, qk.q_stride_h, qk.q_stride_n, qk.dtype);
  a.k_wide = rows_are_16_byte_aligned(qk.k, qk.k_stride_b, qk.k_stride_h, qk.k_stride_n, qk.dtype);
  if (qk.channels != qk.head_dim)
    launch_prepare_padded(a, stream);
  else
    launch_by_type<false>(a, stream);
  return check_launch("risa_sdpa preparation");
}

}  // namespace risa
