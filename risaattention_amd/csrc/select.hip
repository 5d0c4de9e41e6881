// Retained-mass tile selection and broadcast key-mask tile metadata for gfx950.
//
// Contract: reference csrc/kernels/sparse_selection.cu:9-159 (FP64 total and
// prefix over masses already sorted in descending order, shortest prefix whose
// mass reaches theta * total, CSR compaction in ascending tile order, summary)
// and csrc/kernels/key_mask_tiles.cu:10-43.

#include "common.hpp"
#include "launchers.hpp"
#include "mask_kernels.hpp"

namespace risa {
namespace {

// One 32-lane half of a wavefront per row, so that lane-strided sums and the
// 32-wide inclusive scans associate exactly as in the contract.
__global__ __launch_bounds__(64) void select_rows_kernel(const float* __restrict__ sorted_mass,
                                                         const int64_t* __restrict__ order,
                                                         int32_t* __restrict__ counts,
                                                         uint8_t* __restrict__ support,
                                                         double* __restrict__ row_totals, int rows,
                                                         int tiles, double theta) {
  const int sub = threadIdx.x & 31;
  const int row = blockIdx.x * 2 + (threadIdx.x >> 5);
  if (row >= rows) return;
  const int64_t base = static_cast<int64_t>(row) * tiles;
  double lane_total = 0.0;
  for (int rank = sub; rank < tiles; rank += 32) {
    lane_total += static_cast<double>(sorted_mass[base + rank]);
    support[base + rank] = 0;
  }
  double total = lane_total;
#pragma unroll
  for (int offset = 16; offset > 0; offset >>= 1) total += __shfl_down(total, offset, 32);
  total = __shfl(total, 0, 32);

  const double target = theta * total;
  double cumulative = 0.0;
  double selected = total;
  int count = tiles;
  for (int chunk = 0; chunk < tiles; chunk += 32) {
    const int rank = chunk + sub;
    double prefix = rank < tiles ? static_cast<double>(sorted_mass[base + rank]) : 0.0;
#pragma unroll
    for (int offset = 1; offset < 32; offset <<= 1) {
      const double previous = __shfl_up(prefix, offset, 32);
      if (sub >= offset) prefix += previous;
    }
    const bool reaches = rank < tiles && cumulative + prefix >= target;
    const uint64_t ballot = __ballot(reaches);
    const uint32_t votes = static_cast<uint32_t>(ballot >> (threadIdx.x & 32));
    if (votes != 0) {
      const int first = __builtin_ctz(votes);
      count = chunk + first + 1;
      selected = cumulative + __shfl(prefix, first, 32);
      break;
    }
    cumulative += __shfl(prefix, 31, 32);
  }
  // The support bytes of this row were cleared by these same 32 lanes above.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  for (int rank = sub; rank < count; rank += 32) {
    support[base + static_cast<int>(order[base + rank])] = 1;
  }
  if (sub == 0) {
    counts[row] = count;
    row_totals[row * 2] = selected;
    row_totals[row * 2 + 1] = total;
  }
}

// Descending order of every row's masses with ties by ascending tile id (what a stable
// descending sort gives; the contract sorts with torch.sort in Python, reference
// src/risa_attention/sparse.py:24, and documents ties as free): one workgroup per row, a bitonic
// network over the row padded to a power of two in LDS.  Padding entries (-inf, ids past the row)
// end up last and are not written.
// THREADS: 64 for rows of up to 1024 entries (a single wavefront's barriers cost next to nothing
// and sixteen such workgroups share a compute unit), 256 beyond.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void sort_rows_kernel(const float* __restrict__ masses,
                                                            float* __restrict__ sorted_mass,
                                                            int64_t* __restrict__ order, int tiles, int padded) {
  extern __shared__ unsigned char sort_lds[];
  float* key = reinterpret_cast<float*>(sort_lds);
  int* id = reinterpret_cast<int*>(key + padded);
  const int tid = threadIdx.x;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * tiles;
  for (int i = tid; i < padded; i += THREADS) {
    key[i] = i < tiles ? masses[base + i] : -__builtin_inff();
    id[i] = i;
  }
  __syncthreads();
  for (int k = 2; k <= padded; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = tid; t < padded / 2; t += THREADS) {
        const int low = (t / j) * 2 * j + (t % j), high = low + j;
        const float a = key[low], b = key[high];
        const int ia = id[low], ib = id[high];
        const bool b_first = b > a || (b == a && ib < ia);  // b belongs in front of a
        const bool a_first = a > b || (a == b && ia < ib);
        // the first half of every 2k block ends up in order, the second half reversed
        if (((low & k) == 0) ? b_first : a_first) {
          key[low] = b, key[high] = a;
          id[low] = ib, id[high] = ia;
        }
      }
      __syncthreads();
    }
  }
  for (int i = tid; i < tiles; i += THREADS) {
    sorted_mass[base + i] = key[i];
    order[base + i] = id[i];
  }
}

// The same order for rows of up to 128 entries, one wavefront each: an entry's place is the number of
// entries in front of it, counted against all of them read from LDS (the network's 28 steps wait for LDS
// and each other: 14.9 us for 2048 rows of 128).  Entries are compared as (value, ~id) in
// one unsigned word, floats mapped to their order and -0 to 0, so every place is taken once whatever the
// masses hold.
constexpr int kRankedTiles = 128;
__global__ __launch_bounds__(64) void rank_rows_kernel(const float* __restrict__ masses, float* __restrict__ sorted_mass,
                                                       int64_t* __restrict__ order, int tiles) {
  __shared__ uint64_t entries[kRankedTiles];
  const int lane = threadIdx.x;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * tiles;
  float mass[2];
  uint64_t mine[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int id = lane + 64 * j;
    mass[j] = masses[base + min(id, tiles - 1)];
    const uint32_t bits = __float_as_uint(mass[j] + 0.0f);
    const uint32_t ordered = id < tiles ? ((bits >> 31) != 0 ? ~bits : bits | 0x80000000u) : 0u;
    mine[j] = static_cast<uint64_t>(ordered) << 32 | static_cast<uint32_t>(~id);
    entries[id] = mine[j];
  }
  __syncthreads();
  int place[2] = {0, 0};
#pragma unroll 16
  for (int i = 0; i < kRankedTiles; ++i) {
    const uint64_t entry = entries[i];
#pragma unroll
    for (int j = 0; j < 2; ++j) place[j] += entry > mine[j] ? 1 : 0;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int id = lane + 64 * j;
    if (id < tiles) {
      sorted_mass[base + place[j]] = mass[j];
      order[base + place[j]] = id;
    }
  }
}

// Single workgroup: exclusive scan of the per-row counts and the FP64 summary
// (pairwise tree over 256 partial sums, as in the contract).
__global__ __launch_bounds__(256) void offsets_summary_kernel(const int32_t* __restrict__ counts,
                                                              const double* __restrict__ row_totals,
                                                              int32_t* __restrict__ row_offsets,
                                                              double* __restrict__ summary, int rows) {
  __shared__ double selected_sums[256];
  __shared__ double total_sums[256];
  __shared__ int scan[256];
  __shared__ int carry;
  const int tid = threadIdx.x;
  double selected = 0.0, total = 0.0;
  // (eight loads in flight here and below: one after the other they were most of this launch's time)
  constexpr int IN_FLIGHT = 8;
  for (int first = tid; first < rows; first += 256 * IN_FLIGHT) {
    double value[IN_FLIGHT][2];
#pragma unroll
    for (int j = 0; j < IN_FLIGHT; ++j) {
      const int row = min(first + 256 * j, rows - 1);
      value[j][0] = row_totals[row * 2];
      value[j][1] = row_totals[row * 2 + 1];
    }
#pragma unroll
    for (int j = 0; j < IN_FLIGHT; ++j) {
      if (first + 256 * j < rows) {
        selected += value[j][0];
        total += value[j][1];
      }
    }
  }
  selected_sums[tid] = selected;
  total_sums[tid] = total;
  if (tid == 0) carry = 0;
  __syncthreads();
  for (int stride = 128; stride > 0; stride >>= 1) {
    if (tid < stride) {
      selected_sums[tid] += selected_sums[tid + stride];
      total_sums[tid] += total_sums[tid + stride];
    }
    __syncthreads();
  }
  // Exclusive scan of the counts: every thread owns a run of consecutive rows, the 256 run
  // totals are scanned through LDS once, and every thread then writes its run (integer sums:
  // any order gives the same offsets).
  const int run = (rows + 255) / 256;
  const int first = tid * run, last = min(first + run, rows);
  int mine = 0;
  for (int row = first; row < last; row += IN_FLIGHT) {
    int count[IN_FLIGHT];
#pragma unroll
    for (int j = 0; j < IN_FLIGHT; ++j) count[j] = counts[min(row + j, last - 1)];
#pragma unroll
    for (int j = 0; j < IN_FLIGHT; ++j) mine += row + j < last ? count[j] : 0;
  }
  scan[tid] = mine;
  __syncthreads();
  for (int offset = 1; offset < 256; offset <<= 1) {
    const int add = tid >= offset ? scan[tid - offset] : 0;
    __syncthreads();
    scan[tid] += add;
    __syncthreads();
  }
  int running = scan[tid] - mine;
  for (int row = first; row < last; row += IN_FLIGHT) {
    int count[IN_FLIGHT];
#pragma unroll
    for (int j = 0; j < IN_FLIGHT; ++j) count[j] = counts[min(row + j, last - 1)];
#pragma unroll
    for (int j = 0; j < IN_FLIGHT; ++j) {
      if (row + j < last) row_offsets[row + j] = running;
      running += row + j < last ? count[j] : 0;
    }
  }
  if (tid == 255) carry = scan[255];
  __syncthreads();
  if (tid == 0) {
    row_offsets[rows] = carry;
    summary[0] = selected_sums[0];
    summary[1] = total_sums[0];
    summary[2] = static_cast<double>(carry);
  }
}

// One wavefront per row: ordered compaction of the support bytes.
__global__ __launch_bounds__(256) void compact_rows_kernel(const uint8_t* __restrict__ support,
                                                           const int32_t* __restrict__ row_offsets,
                                                           int32_t* __restrict__ block_indices,
                                                           int rows, int tiles) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int64_t base = static_cast<int64_t>(row) * tiles;
  int written = row_offsets[row];
  for (int chunk = 0; chunk < tiles; chunk += 64) {
    const int tile = chunk + lane;
    const bool keep = tile < tiles && support[base + tile] != 0;
    const uint64_t votes = __ballot(keep);
    if (keep) {
      const uint64_t lower = lane == 0 ? 0ull : (votes & ((1ull << lane) - 1ull));
      block_indices[written + __builtin_popcountll(lower)] = tile;
    }
    written += __builtin_popcountll(votes);
  }
}

template <int DT> __global__ __launch_bounds__(256) void key_mask_kernel(const KeyMaskArgs a) {
  extern __shared__ unsigned char run_flags[];
  key_mask_block<DT>(a, blockIdx.x, run_flags);
}

void launch_key_mask_kernel(const KeyMaskArgs& a, int dtype, hipStream_t stream) {
  const int blocks = key_mask_blocks(a);
  const size_t flags = key_mask_flag_bytes(a);
  if (dtype == kBool)
    key_mask_kernel<kBool><<<blocks, 256, flags, stream>>>(a);
  else if (dtype == kF32)
    key_mask_kernel<kF32><<<blocks, 256, flags, stream>>>(a);
  else if (dtype == kF16)
    key_mask_kernel<kF16><<<blocks, 256, flags, stream>>>(a);
  else
    key_mask_kernel<kBF16><<<blocks, 256, flags, stream>>>(a);
}

template <bool ALIGNED> __global__ __launch_bounds__(256) void mask_lanes_kernel(const MaskLaneArgs a) {
  mask_lanes_block<ALIGNED>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

// grid (query blocks, planes)
__global__ __launch_bounds__(64) void mask_tile_lists_kernel(const MaskLaneArgs a) {
  mask_tile_list(a, blockIdx.x, blockIdx.y, threadIdx.x);
}

}  // namespace

size_t mask_lane_words(int batch, int heads, int q_len, int k_len) {
  const size_t query_waves = (static_cast<size_t>(q_len) + 127) / 128 * 4;
  const size_t key_tiles = (static_cast<size_t>(k_len) + 63) / 64;
  return static_cast<size_t>(batch) * heads * query_waves * key_tiles * 32;
}

// The buffer of one mask: the lane words, then one 32-bit class per 32 words (kLaneTile...),
// then per mask plane and block of 128 queries the list of tiles with a visible key.
size_t mask_lane_class_offset(int batch, int heads, int q_len, int k_len) {
  return mask_lane_words(batch, heads, q_len, k_len) * sizeof(uint64_t);
}
size_t mask_tile_list_offset(int batch, int heads, int q_len, int k_len) {
  const size_t classes = mask_lane_words(batch, heads, q_len, k_len) / 32;
  return mask_lane_class_offset(batch, heads, q_len, k_len) + (classes * sizeof(int32_t) + 7) / 8 * 8;
}
size_t mask_lane_bytes(int batch, int heads, int q_len, int k_len) {
  const size_t query_blocks = (static_cast<size_t>(q_len) + 127) / 128;
  const size_t key_tiles = (static_cast<size_t>(k_len) + 63) / 64;
  const size_t lists = static_cast<size_t>(batch) * heads * query_blocks * (key_tiles + 1);
  return mask_tile_list_offset(batch, heads, q_len, k_len) + (lists * sizeof(int32_t) + 7) / 8 * 8;
}

MaskLaneArgs mask_lane_args(const void* mask, uint64_t* lanes, int batch, int heads, int q_len, int k_len,
                            int64_t stride_b, int64_t stride_h, int64_t stride_q) {
  unsigned char* bytes = reinterpret_cast<unsigned char*>(lanes);
  MaskLaneArgs a{};
  a.mask = static_cast<const uint8_t*>(mask);
  a.lanes = lanes;
  a.classes = reinterpret_cast<int32_t*>(bytes + mask_lane_class_offset(batch, heads, q_len, k_len));
  a.lists = reinterpret_cast<int32_t*>(bytes + mask_tile_list_offset(batch, heads, q_len, k_len));
  a.heads = heads;
  a.planes = batch * heads;
  a.q_len = q_len;
  a.k_len = k_len;
  a.key_tiles = (k_len + 63) / 64;
  a.query_waves = (q_len + 127) / 128 * 4;
  a.stride_b = stride_b;
  a.stride_h = stride_h;
  a.stride_q = stride_q;
  a.aligned = reinterpret_cast<uintptr_t>(mask) % 16 == 0 && ((stride_b | stride_h | stride_q) & 15) == 0;
  return a;
}

int launch_mask_lanes(const MaskLaneArgs& a, hipStream_t stream) {
  const dim3 grid(mask_lane_groups(a), a.query_waves, a.planes);
  if (a.aligned)
    mask_lanes_kernel<true><<<grid, 256, 0, stream>>>(a);
  else
    mask_lanes_kernel<false><<<grid, 256, 0, stream>>>(a);
  mask_tile_lists_kernel<<<dim3(a.query_waves / 4, a.planes), 64, 0, stream>>>(a);
  return check_launch("risa_prepare_mask_lanes");
}

int launch_key_bias(const void* mask, float* bias, int batch, int heads, int length, int padded,
                    int64_t stride_b, int64_t stride_h, int64_t stride_k, int dtype,
                    hipStream_t stream) {
  KeyMaskArgs a{};
  a.mask = mask;
  a.bias = bias;
  a.bias_heads = heads;
  a.bias_planes = batch * heads;
  a.length = length;
  a.padded = padded;
  a.stride_k = stride_k;
  a.bias_stride_b = stride_b;
  a.bias_stride_h = stride_h;
  launch_key_mask_kernel(a, dtype, stream);
  return check_launch("risa_prepare_key_bias");
}

int launch_sort_rows(const float* masses, float* sorted_mass, int64_t* order, int rows, int tiles,
                     hipStream_t stream) {
  int padded = 2;
  while (padded < tiles) padded <<= 1;
  if (padded > kSortableTiles) return fail("risa_sort_select_retained_mass: more key tiles than one workgroup sorts");
  if (tiles <= kRankedTiles) {
    rank_rows_kernel<<<rows, 64, 0, stream>>>(masses, sorted_mass, order, tiles);
  } else if (padded <= 1024) {
    sort_rows_kernel<64><<<rows, 64, static_cast<size_t>(padded) * 8, stream>>>(masses, sorted_mass, order, tiles, padded);
  } else {
    sort_rows_kernel<256><<<rows, 256, static_cast<size_t>(padded) * 8, stream>>>(masses, sorted_mass, order, tiles, padded);
  }
  return check_launch("risa_sort_select_retained_mass");
}

int launch_select_retained_mass(const SelectArgs& a, hipStream_t stream) {
  select_rows_kernel<<<(a.rows + 1) / 2, 64, 0, stream>>>(a.sorted_mass, a.descending_indices,
                                                          a.counts, a.support, a.row_totals, a.rows,
                                                          a.tiles, a.theta);
  offsets_summary_kernel<<<1, 256, 0, stream>>>(a.counts, a.row_totals, a.row_offsets, a.summary,
                                                a.rows);
  compact_rows_kernel<<<(a.rows + 3) / 4, 256, 0, stream>>>(a.support, a.row_offsets,
                                                            a.block_indices, a.rows, a.tiles);
  return check_launch("risa_select_retained_mass");
}

int launch_key_mask_tiles(const void* mask, int32_t* tiles, int batch, int heads, int length,
                          int tile_size, int64_t stride_b, int64_t stride_h, int64_t stride_k,
                          int dtype, hipStream_t stream) {
  KeyMaskArgs a{};
  a.mask = mask;
  a.tiles = tiles;
  a.batch = batch;
  a.heads = heads;
  a.length = length;
  a.tile_size = tile_size;
  a.stride_b = stride_b;
  a.stride_h = stride_h;
  a.stride_k = stride_k;
  launch_key_mask_kernel(a, dtype, stream);
  return check_launch("risa_prepare_key_mask_tiles");
}

KeyMaskArgs key_mask_args(const void* mask, int32_t* tiles, float* bias, int batch, int heads, int mask_batch,
                          int mask_heads, int length, int padded, int tile_size, int64_t stride_b,
                          int64_t stride_h, int64_t stride_k) {
  KeyMaskArgs a{};
  a.mask = mask;
  a.tiles = tiles;
  a.bias = bias;
  a.batch = batch;
  a.heads = heads;
  a.bias_heads = mask_heads;
  a.bias_planes = mask_batch * mask_heads;
  a.length = length;
  a.tile_size = tile_size;
  a.padded = padded;
  a.stride_b = stride_b;
  a.stride_h = stride_h;
  a.stride_k = stride_k;
  a.bias_stride_b = mask_batch > 1 ? stride_b : 0;
  a.bias_stride_h = mask_heads > 1 ? stride_h : 0;
  return a;
}

int launch_key_mask(const KeyMaskArgs& a, int dtype, hipStream_t stream) {
  launch_key_mask_kernel(a, dtype, stream);
  return check_launch("risa_sdpa key mask");
}

}  // namespace risa
