// Launcher of the fused Q/K/V preparation (kernels and their order: prep_fused_kernels.hpp).
#include "prep_fused_kernels.hpp"

namespace risa {

bool can_prepare_fused(const QkArgs& qk, const ValueArgs& v) {
  return qk.k_len == v.length &&
         qk.batch == v.batch && qk.kv_heads == v.heads && qk.head_dim == v.head_dim &&
         qk.cta_k == v.cta_k && qk.dtype == v.dtype;
}

int launch_prepare_fused(const QkArgs& qk, const ValueArgs& v, const PrepareRiders& riders, hipStream_t stream) {
  if (!can_prepare_fused(qk, v)) return fail("risa_sdpa: operands do not qualify for the fused preparation");
  if (v.workspace_bytes < value_workspace_bytes(v.batch, v.heads, v.length, v.head_dim, v.midpoint_affine))
    return fail("risa_quantize_v: workspace is too small");
  const Workspace w = carve(v.workspace, v.batch, v.heads, v.length, v.head_dim, v.midpoint_affine);
  FusedRiders a{};
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
  // Riders.  (The flags of a key list are LDS of every workgroup of the launch, so long rows get a
  // launch of their own: 4 KB, 262144 keys, take no workgroup from a compute unit.)
  const bool key_mask_rides = riders.key_mask != nullptr && key_mask_flag_bytes(*riders.key_mask) <= 4096;
  if (key_mask_rides) {
    a.key_mask = *riders.key_mask;
    a.key_mask_dtype = riders.key_mask_dtype;
    a.key_mask_blocks = key_mask_blocks(a.key_mask);
    a.key_mask_flag_bytes = static_cast<int>(key_mask_flag_bytes(a.key_mask));
  }
  const bool second_launch = !one_launch(a);
  // (lane words where the mask is read sixteen bytes at a time; the tile lists need the words first)
  const bool lanes_ride = riders.lanes != nullptr && second_launch && riders.lanes->aligned;
  if (lanes_ride) {
    a.lanes = *riders.lanes;
    a.lane_groups = mask_lane_groups(a.lanes);
    a.lane_blocks = a.lane_groups * a.lanes.query_waves * a.lanes.planes;
    a.list_blocks = (a.lanes.query_waves / 4 * a.lanes.planes + 3) / 4;
  }
  const bool masked = a.key_mask_blocks != 0 || a.lane_blocks != 0;
  const bool shift_rides = riders.shift != nullptr && second_launch && masked;
  if (shift_rides) {
    a.shift = *riders.shift;
    a.shift_rows = lse_shift_rows(a.shift);
    a.shift_blocks_x = lse_shift_blocks(a.shift, a.shift_rows);
    a.shift_blocks = a.shift_blocks_x * a.shift.q_heads * a.shift.batch;
  }
  if (qk.channels != qk.head_dim)
    (masked ? launch_prepare_padded_masked : launch_prepare_padded)(a, stream);
  else
    (masked ? launch_prepare_masked : launch_by_type<false, false>)(a, stream);
  int status = check_launch("risa_sdpa preparation");
  if (status == 0 && riders.key_mask != nullptr && !key_mask_rides)
    status = launch_key_mask(*riders.key_mask, riders.key_mask_dtype, stream);
  if (status == 0 && riders.lanes != nullptr && !lanes_ride) status = launch_mask_lanes(*riders.lanes, stream);
  if (status == 0 && riders.shift != nullptr && !shift_rides) status = launch_lse_shift(*riders.shift, stream);
  return status;
}

}  // namespace risa
