// Launcher of the sixteen-queries-per-wavefront attention kernel used for launches that
// leave compute units with at most one workgroup.
#include "attention_narrow_kernel.hpp"

#include <algorithm>

namespace risa {


namespace {

// Queries per workgroup: 128, or 64 / 32 when that still leaves compute units without
// a workgroup (every SIMD then runs one wavefront with a quarter of the usual work).
// Those smaller workgroups also split four or more key tiles over two sets of wavefronts:
// the launch is short of work, not of hardware.
template <int D, int CTA_K> int launch_narrow(const KernelParams& p, hipStream_t stream) {
  const int64_t workgroups = static_cast<int64_t>(p.n_qb) * p.q_heads * p.batch;
  const int compute_units = narrow_attention_limit();
  // two sets of stages must fit the 160 KB of LDS of a compute unit
  constexpr bool kSplitFits = 2 * TileShape<D, CTA_K>::kLdsBytes <= 160 * 1024;
  const bool split = kSplitFits && p.n_kb >= 4;
  // (a launch split over the key tiles has its workgroups: the largest ones, which share a tile's copy most)
  if (p.key_parts > 1) return launch_narrow_block<D, CTA_K, 8, 1>(p, stream);
  if (p.index_mode == 1) {
    // sparse reuse: the tile lists stay whole
    if (workgroups * 4 <= compute_units) return launch_narrow_block<D, CTA_K, 2, 1, true>(p, stream);
    if (workgroups * 2 <= compute_units) return launch_narrow_block<D, CTA_K, 4, 1, true>(p, stream);
    return launch_narrow_block<D, CTA_K, 8, 1, true>(p, stream);
  }
  if (workgroups * 4 <= compute_units) {
    if constexpr (kSplitFits) {
      if (split) return launch_narrow_block<D, CTA_K, 2, 2>(p, stream);
    }
    return launch_narrow_block<D, CTA_K, 2, 1>(p, stream);
  }
  if (workgroups * 2 <= compute_units) {
    if constexpr (kSplitFits) {
      if (split) return launch_narrow_block<D, CTA_K, 4, 2>(p, stream);
    }
    return launch_narrow_block<D, CTA_K, 4, 1>(p, stream);
  }
  return launch_narrow_block<D, CTA_K, 8, 1>(p, stream);
}

}  // namespace

// Number of workgroups up to which the narrow kernel is the faster one: the number of
// compute units, below which the wide kernel runs one wavefront per SIMD.  Where no device can
// be queried (size queries made on a host without a GPU) it is the MI355X's 256.
int narrow_attention_limit() {
  constexpr int kMi355xComputeUnits = 256;
  static thread_local int cached_device = -1;
  static thread_local int compute_units = 0;
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess) return kMi355xComputeUnits;
  if (device != cached_device) {
    int count = 0;
    if (hipDeviceGetAttribute(&count, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || count <= 0)
      return kMi355xComputeUnits;
    compute_units = count;
    cached_device = device;
  }
  return compute_units;
}

// How many ranges of the key tiles the workgroups of a launch of few query blocks walk.
//
// A workgroup takes its key tiles one after the other, 1 to 2.5 us per 64 keys however few workgroups
// there are, so a launch that leaves compute units idle is split until they have work: the fewest
// microseconds of a model of both sides.  Walking takes the longest chain of tiles (under the causal
// rule, where workgroups of all lengths follow each other, the work of all of them where that is
// more); a split adds 6 us and a write and read of the partial results.  Whole call, one range -> the best of
// 2 to 24 (which one in brackets), 128 channels unless said otherwise, heads x queries x keys:
//   plain       16 x 128 x 2048 35.0 -> 28.6 us (8), x 8192 91.4 -> 54.6 (16), 16 x 512 x 4096 55.1 -> 47.4 (4),
//               256 channels 16 x 128 x 2048 62.9 -> 39.5 (8), 16 x 1024 x 4096 118 -> 99.6 (2)
//   causal      1 x 8192 117 -> 50.9 us (4), 4 x 8192 133 -> 104 (2), 2 x 4096 66.2 -> 39.5 (4)
//   padding     16 x 128 x 2048 49.5 -> 31.3 us (8), 16 x 512 x 4096 80.7 -> 52.6 (4), 64 channels 80.7 -> 44.0 (8)
//   boolean     16 x 128 x 8192 269 -> 64.6 us (16), 16 x 512 x 1024 48.9 -> 34.1 (4), 16 x 1024 x 4096 141 -> 95.3 (2)
// and where the model does not split: plain 16 x 512 x 1024 29.1 -> 30.4 us (4), 16 x 1024 x 4096 59.0 -> 61.4 (2),
// 8 x 128 x 512 16.0 -> 16.9 (4); padding, 64 channels 16 x 1024 x 1024 32.7 -> 30.7 (4).
int attention_key_parts(const AttentionExtents& e, SplitKind kind, bool causal) {
  const int64_t blocks = (e.q_len + kQueryBlock - 1) / kQueryBlock;
  const int64_t workgroups = blocks * e.batch * e.q_heads;
  if (e.k_len <= 2 * e.cta_k) return 1;
  const int units = narrow_attention_limit();
  if (workgroups > units) return 1;
  const int wide = e.head_dim == 64 ? 0 : e.head_dim == 128 ? 1 : 2;
  constexpr float kPer64Keys[3][3] = {{0.85f, 1.05f, 1.5f}, {1.1f, 1.1f, 1.6f}, {1.7f, 2.0f, 2.5f}};
  const float per_tile = kPer64Keys[static_cast<int>(kind)][wide] * (e.cta_k / 64);
  const int tiles = ((causal ? std::min(e.k_len, e.q_len) : e.k_len) + e.cta_k - 1) / e.cta_k;
  // (without a split, plain launches of at most half a workgroup per unit split four or more tiles in two
  // inside their workgroups)
  const bool halves = kind == SplitKind::kPlain && !causal && workgroups * 2 <= units && tiles >= 4 &&
                      !(e.head_dim == 256 && e.cta_k == 128);
  const float all = causal ? 0.5f * workgroups * (tiles + 1) / units : 0.0f;  // tiles per unit
  float best = per_tile * std::max<float>(halves ? (tiles + 1) / 2 : tiles, all);
  int best_parts = 1;
  for (int parts = 2; parts <= 16 && parts <= tiles && workgroups * parts <= (causal ? 2 : 1) * units; ++parts) {
    const float megabytes = workgroups * parts * key_part_bytes(e.head_dim) * 1e-6f;
    const float time = per_tile * std::max<float>((tiles + parts - 1) / parts, all) + 6.0f + megabytes / 3.0f;
    if (time < best) best = time, best_parts = parts;
  }
  return best_parts;
}

size_t attention_split_bytes(const AttentionExtents& e, int mask_dtype, int64_t mask_stride_q) {
  const bool tensor = mask_dtype >= 0 && mask_stride_q != 0;
  int parts = 1;
  for (const bool causal : {false, true}) {
    parts = std::max(parts, attention_key_parts(e, tensor ? SplitKind::kMaskTensor : SplitKind::kScaled, causal));
    if (mask_dtype < 0) parts = std::max(parts, attention_key_parts(e, SplitKind::kPlain, causal));
    // (a key-only mask without its additive row is read like a mask tensor)
    if (mask_dtype >= 0) parts = std::max(parts, attention_key_parts(e, SplitKind::kMaskTensor, causal));
  }
  if (parts <= 1) return 0;
  const size_t blocks = static_cast<size_t>(e.batch) * e.q_heads * ((e.q_len + kQueryBlock - 1) / kQueryBlock);
  return parts * blocks * key_part_bytes(e.head_dim);
}

int launch_attention_narrow(const KernelParams& p, int head_dim, int cta_k, hipStream_t stream) {
  if (head_dim == 64) return launch_narrow<64, 64>(p, stream);
  if (head_dim == 128) return cta_k == 128 ? launch_narrow<128, 128>(p, stream) : launch_narrow<128, 64>(p, stream);
  if (head_dim == 256) return cta_k == 128 ? launch_narrow<256, 128>(p, stream) : launch_narrow<256, 64>(p, stream);
  return fail("risa_attention: unsupported head_dim");
}

}  // namespace risa
