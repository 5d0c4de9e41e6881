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

size_t attention_split_bytes(const AttentionExtents& e, SplitKind kind, bool causal) {
  const size_t parts = attention_key_parts(e, kind, causal);
  const size_t blocks = static_cast<size_t>(e.batch) * e.q_heads * ((e.q_len + kQueryBlock - 1) / kQueryBlock);
  return parts > 1 ? parts * blocks * key_part_bytes(e.head_dim) : 0;
}

size_t attention_split_bytes(const AttentionExtents& e, int mask_dtype, int64_t mask_stride_q) {
  const bool tensor = mask_dtype >= 0 && mask_stride_q != 0;
  size_t bytes = 0;
  for (const bool causal : {false, true}) {
    bytes = std::max(bytes, attention_split_bytes(e, tensor ? SplitKind::kMaskTensor : SplitKind::kScaled, causal));
    // (a key-only mask without its additive row is read like a mask tensor)
    bytes = std::max(bytes, attention_split_bytes(e, mask_dtype < 0 ? SplitKind::kPlain : SplitKind::kMaskTensor, causal));
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
