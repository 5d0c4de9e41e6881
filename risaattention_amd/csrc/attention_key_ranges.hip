// Launches of few query blocks: ranges of the key tiles go to workgroups of their own (variants of the
// sixteen-query kernel, 128 queries a workgroup), and a second kernel puts their results together.  The
// variants are apart from those that walk all tiles: as run-time tests in the same kernels the ranges cost
// the launches that are not split 0.5 to 2 % (16/4 heads x 2048, whole call, one machine: midpoint_affine
// 48.7 us with the tests, 48.4 without; 48.5 before there were ranges).
#include "attention_narrow_kernel.hpp"

#include <algorithm>

namespace risa {
namespace {

// Puts the ranges of the key tiles together (p.key_parts partial results per query): the online-softmax
// update once more, so only the order of FP32 additions differs from a walk over all tiles.  A wavefront
// takes sixteen queries of an attention_narrow_kernel<D, CTA_K, 8> workgroup and 64 channels, so that
// few query blocks still fill the machine.
template <int D> __global__ __launch_bounds__(256) void merge_key_parts_kernel(const KernelParams p) {
  constexpr int CB = D / 16, VALUES = CB * 4 + 2, WAVES = 8, QUERIES = 16 * WAVES;
  const int lane = threadIdx.x & 63, ql = lane & 15, grp = lane >> 4;
  const int query_blocks = (p.q_len + QUERIES - 1) / QUERIES;
  const int blocks = query_blocks * p.q_heads * p.batch;
  const int index = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int first_cb = index % (D / 64) * 4, walked = index / (D / 64);  // wavefront of the walking launch
  if (walked >= blocks * WAVES) return;
  const int wave = walked % WAVES, block = walked / WAVES;
  int bx, head, batch;
  if (p.causal) {
    const int heads = p.q_heads * p.batch;
    const int rest = block % heads;
    bx = query_blocks - 1 - block / heads;
    head = rest % p.q_heads;
    batch = rest / p.q_heads;
  } else {
    bx = block % query_blocks;
    const int rest = block / query_blocks;
    head = rest % p.q_heads;
    batch = rest / p.q_heads;
  }
  const int64_t bhk = static_cast<int64_t>(batch) * p.kv_heads + head / (p.q_heads / p.kv_heads);
  const int64_t bhq = static_cast<int64_t>(batch) * p.q_heads + head;
  const int query = bx * QUERIES + wave * 16 + ql;
  const int64_t part_stride = static_cast<int64_t>(blocks) * WAVES * (VALUES * 64);
  const float* at = p.partial + static_cast<int64_t>(walked) * (VALUES * 64) + lane;
  // Four ranges at a time, their loads in flight together (one by one, a range costs its round trip:
  // 16 of them 23 us for 16 query blocks of 128 channels).  Past the last range the last one is read again
  // and counts nothing.
  constexpr int BATCH = 4;
  float m = kRowFloor, d = 0.0f, o_acc[4][4] = {};
  for (int first = 0; first < p.key_parts; first += BATCH) {
    float value[BATCH][4][4], its_m[BATCH], its_d[BATCH];
#pragma unroll
    for (int j = 0; j < BATCH; ++j) {
      const float* source = at + min(first + j, p.key_parts - 1) * part_stride;
      its_m[j] = source[CB * 4 * 64];
      its_d[j] = source[(CB * 4 + 1) * 64];
#pragma unroll
      for (int cb = 0; cb < 4; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i) value[j][cb][i] = source[((first_cb + cb) * 4 + i) * 64];
    }
    float top = m;
#pragma unroll
    for (int j = 0; j < BATCH; ++j) top = __builtin_fmaxf(top, its_m[j]);
    const float scale = __builtin_amdgcn_exp2f(m - top);
    m = top;
    d *= scale;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int i = 0; i < 4; ++i) o_acc[cb][i] *= scale;
#pragma unroll
    for (int j = 0; j < BATCH; ++j) {
      const float weight = first + j < p.key_parts ? __builtin_amdgcn_exp2f(its_m[j] - m) : 0.0f;
      d = __builtin_fmaf(its_d[j], weight, d);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i) o_acc[cb][i] = __builtin_fmaf(value[j][cb][i], weight, o_acc[cb][i]);
    }
  }
  float d_total = d + __shfl_xor(d, 16);
  d_total += __shfl_xor(d_total, 32);
  if (query < p.q_len) {
    store_narrow_rows<D, 4>(p, bhk, batch, head, query, grp, first_cb, o_acc, d_total, p.mask_dtype >= 0 || p.causal);
    if (p.lse != 0 && grp == 0 && first_cb == 0) store_narrow_lse(p, bhq, query, m, d_total);
  }
}

template <int D, int CTA_K, bool INDEXED, bool GENERAL, int MASK_DT = -1, bool MASK_VEC = false>
int launch_variant(const KernelParams& p, hipStream_t stream) {
  const int status = launch_narrow_block<D, CTA_K, 8, 1, INDEXED, GENERAL, false, MASK_DT, MASK_VEC, true>(p, stream);
  if (status != 0) return status;
  const unsigned wavefronts = static_cast<unsigned>(p.n_qb) * p.q_heads * p.batch * 8 * (D / 64);
  merge_key_parts_kernel<D><<<dim3((wavefronts + 3) / 4), 256, 0, stream>>>(p);
  return 0;
}

template <int D, int CTA_K, int MASK_DT>
int launch_mask(const KernelParams& p, bool vector_loads, hipStream_t stream) {
  if (vector_loads) return launch_variant<D, CTA_K, false, true, MASK_DT, true>(p, stream);
  return launch_variant<D, CTA_K, false, true, MASK_DT>(p, stream);
}

template <int D, int CTA_K> int launch_tile(const KernelParams& p, bool fast, int mask_mode, hipStream_t stream) {
  if (fast) return launch_variant<D, CTA_K, false, false>(p, stream);
  const bool vector_loads = mask_mode != kMaskScalar;
  switch (p.mask_dtype) {
    case kBool: return launch_mask<D, CTA_K, kBool>(p, vector_loads, stream);
    case kF32: return launch_mask<D, CTA_K, kF32>(p, vector_loads, stream);
    case kF16: return launch_mask<D, CTA_K, kF16>(p, vector_loads, stream);
    case kBF16: return launch_mask<D, CTA_K, kBF16>(p, vector_loads, stream);
    case kKeyBias:
      if (p.index_mode == 2) return launch_variant<D, CTA_K, true, true, kKeyBias>(p, stream);
      return launch_variant<D, CTA_K, false, true, kKeyBias>(p, stream);
    default: return launch_variant<D, CTA_K, false, true>(p, stream);
  }
}

}  // namespace

// How many ranges of the key tiles the workgroups of a launch of few query blocks walk.
//
// A workgroup takes its key tiles one after the other, 0.8 to 2.5 us per 64 keys however few workgroups
// there are, so a launch that leaves compute units idle is split until they have work: the fewest
// microseconds of a model of both sides.  Walking takes the longest chain of tiles (under the causal
// rule, where workgroups of all lengths follow each other, the work of all of them where that is
// more, 0.75 tiles per workgroup of a range included); a split adds a launch, its ranges' epilogues and a
// write and read of the partial results.
//
// The constants are those of 1647 launches of 1 to 256 workgroups and 300 to 16384 keys, attention from packed
// operands with one range and with up to nine numbers of them each.  Over 737 others, what the model picks
// takes 1.015 times the best number on the average (one range everywhere about 1.8), and 3 launches more than
// 1 % longer than with one range, up to 1.16 times.  (With one row for causal launches and those with pre-scaled
// scores, and none for plain launches that split in two inside their workgroups: 1.024, 18 launches, up to
// 1.20 times.)  One range -> the number picked (in brackets), us, heads x queries x keys x channels:
//   plain    16 x 96 x 11630 x 64 67.3 -> 25.7 (14), 2 x 1316 x 3494 x 256 64.8 -> 25.3 (10), 48 x 128 x 3072 x 128
//            27.8 -> 22.3 (5); not split: 2 x 1024 x 1792 x 64 13.8 (14.4 with 4)
//   causal   4 x 2688 x 64 43.2 -> 27.8 (4); not split: 16 x 1664 x 64 29.0 (31.4 with 2), 12 x 1664 x 128 28.0 (29.1 with 2)
//   boolean  2 x 1152 x 893 x 64 51.4 -> 19.6 (7); not split: 64 x 99 x 464 x 128 17.9 (19.3 with 2)
//   float    16 x 144 x 393 x 128 29.8 -> 18.9 (4)
struct RangeCosts {
  float per_64_keys[3];  // of head dims 64, 128 and 256
  float fixed, per_range, per_megabyte;
};

int attention_key_parts(const AttentionExtents& e, SplitKind kind, bool causal) {
  const int64_t blocks = (e.q_len + kQueryBlock - 1) / kQueryBlock;
  const int64_t workgroups = blocks * e.batch * e.q_heads;
  if (e.k_len <= 2 * e.cta_k) return 1;
  const int units = narrow_attention_limit();
  if (workgroups > units) return 1;
  const int tiles = ((causal ? std::min(e.k_len, e.q_len) : e.k_len) + e.cta_k - 1) / e.cta_k;
  // (without a split, plain launches of at most half a workgroup per unit split four or more tiles in two
  // inside their workgroups)
  const bool halves = kind == SplitKind::kPlain && !causal && workgroups * 2 <= units && tiles >= 4 &&
                      !(e.head_dim == 256 && e.cta_k == 128);
  const bool short_halves = halves && e.head_dim != 256;
  const bool causal_row = causal && kind == SplitKind::kScaled;
  constexpr RangeCosts kHalves{{0.75f, 1.05f, 1.5f}, 5.0f, 0.2f, 1.0f / 3.0f};
  constexpr RangeCosts kCausal{{0.8f, 1.1f, 2.1f}, 3.0f, 0.3f, 0.45f};
  constexpr RangeCosts kKinds[] = {{{0.85f, 1.05f, 1.5f}, 6.0f, 0.0f, 1.0f / 3.0f},   // plain
                                   {{1.1f, 1.1f, 1.6f}, 6.0f, 0.0f, 1.0f / 3.0f},     // scaled
                                   {{1.4f, 1.7f, 2.3f}, 5.0f, 0.0f, 1.0f / 3.0f},     // boolean masks
                                   {{1.7f, 2.0f, 2.5f}, 6.0f, 0.0f, 1.0f / 3.0f}};    // float masks
  const RangeCosts& costs = short_halves ? kHalves : causal_row ? kCausal : kKinds[static_cast<int>(kind)];
  const float per_tile = costs.per_64_keys[e.head_dim == 64 ? 0 : e.head_dim == 128 ? 1 : 2] * (e.cta_k / 64);
  const float all = causal ? 0.5f * workgroups * (tiles + 1) / units : 0.0f;  // tiles per unit
  float best = per_tile * std::max<float>(halves ? (tiles + 1) / 2 : tiles, all) * (short_halves ? 0.95f : 1.0f);
  int best_parts = 1;
  for (int parts = 2; parts <= 16 && parts <= tiles && workgroups * parts <= (causal ? 2 : 1) * units; ++parts) {
    const float megabytes = workgroups * parts * key_part_bytes(e.head_dim) * 1e-6f;
    const float walk = std::max<float>((tiles + parts - 1) / parts, causal_row ? all + 0.75f * workgroups * parts / units : all);
    const float time = per_tile * walk + costs.fixed + costs.per_range * parts + costs.per_megabyte * megabytes;
    if (time < best) best = time, best_parts = parts;
  }
  return best_parts;
}

size_t attention_split_bytes(const AttentionExtents& e, SplitKind kind, bool causal) {
  const size_t parts = attention_key_parts(e, kind, causal);
  const size_t blocks = static_cast<size_t>(e.batch) * e.q_heads * ((e.q_len + kQueryBlock - 1) / kQueryBlock);
  return parts > 1 ? parts * blocks * key_part_bytes(e.head_dim) : 0;
}

size_t attention_split_bytes(const AttentionExtents& e, int mask_dtype, int64_t mask_stride_q) {
  size_t bytes = 0;
  for (const bool causal : {false, true}) {
    // (unmasked calls: raw and pre-scaled scores; a key-only mask without its additive row is read like a mask tensor)
    for (const float sm_scale : {1.0f, -1.0f})
      bytes = std::max(bytes, attention_split_bytes(e, split_kind(mask_dtype, mask_stride_q == 0, causal, sm_scale), causal));
    if (mask_dtype >= 0) bytes = std::max(bytes, attention_split_bytes(e, split_kind(mask_dtype, false, causal, 1.0f), causal));
  }
  return bytes;
}

int launch_attention_key_ranges(const KernelParams& p, int head_dim, int cta_k, bool fast, int mask_mode,
                                hipStream_t stream) {
  if (head_dim == 64) return launch_tile<64, 64>(p, fast, mask_mode, stream);
  if (head_dim == 128) {
    if (cta_k == 128) return launch_tile<128, 128>(p, fast, mask_mode, stream);
    return launch_tile<128, 64>(p, fast, mask_mode, stream);
  }
  if (head_dim == 256) {
    if (cta_k == 128) return launch_tile<256, 128>(p, fast, mask_mode, stream);
    return launch_tile<256, 64>(p, fast, mask_mode, stream);
  }
  return fail("risa_attention: unsupported head_dim");
}

}  // namespace risa
