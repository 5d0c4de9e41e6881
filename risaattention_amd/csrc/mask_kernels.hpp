// Device code that turns attention masks into the forms the attention kernels read: the tile lists and
// additive rows of key-only masks, the lane words and tile lists of boolean masks.  Workgroups of the
// launches of select.hip, or of the preparation's own launches (prep_fused_kernels.hpp).
#pragma once

#include "common.hpp"
#include "launchers.hpp"

namespace risa {

template <int DT> __device__ __forceinline__ float key_term(const void* mask, int64_t index) {
  if constexpr (DT == kBool) {
    return static_cast<const uint8_t*>(mask)[index] != 0 ? 0.0f : -__builtin_inff();
  } else {
    return load1<DT>(mask, index);
  }
}

// The first batch * heads workgroups (when lists are asked for): flags of 64-key runs, eight loads
// in flight per thread (one load per tile and wavefront, each waited for, took 10 us for 72
// tiles), then one wavefront compacts the active tile ids in ascending order and appends the
// count.  The others: 256 keys of a bias plane each.
template <int DT> __device__ __forceinline__ void key_mask_block(const KeyMaskArgs& a, int block, unsigned char* run_flags) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int rows = a.tiles != nullptr ? a.batch * a.heads : 0;
  if (block >= rows) {
    const int per_plane = (a.padded + 255) / 256;
    const int part = block - rows;
    const int plane = part / per_plane, key = part % per_plane * 256 + tid;
    if (key >= a.padded) return;
    float value = -__builtin_inff();
    if (key < a.length) {
      const float term = key_term<DT>(a.mask, plane / a.bias_heads * a.bias_stride_b + plane % a.bias_heads * a.bias_stride_h +
                                                  key * a.stride_k);
      if (__builtin_isfinite(term)) value = term * 1.44269504088896340736f;
    }
    a.bias[static_cast<int64_t>(plane) * a.padded + key] = value;
    return;
  }
  const int64_t row = block;
  const int64_t mask_row = row / a.heads * a.stride_b + row % a.heads * a.stride_h;
  constexpr int IN_FLIGHT = 8;
  for (int first = 0; first < a.length; first += 256 * IN_FLIGHT) {
    float term[IN_FLIGHT];
#pragma unroll
    for (int j = 0; j < IN_FLIGHT; ++j)
      term[j] = key_term<DT>(a.mask, mask_row + min(first + j * 256 + tid, a.length - 1) * a.stride_k);
#pragma unroll
    for (int j = 0; j < IN_FLIGHT; ++j) {
      const int run = first + j * 256 + wave * 64;  // first key of the wavefront's run
      const bool any = __ballot(run + lane < a.length && __builtin_isfinite(term[j])) != 0;
      if (lane == 0 && run < a.length) run_flags[run / 64] = any;
    }
  }
  __syncthreads();
  if (wave != 0) return;
  const int tiles = (a.length + a.tile_size - 1) / a.tile_size;
  const int runs = (a.length + 63) / 64, runs_per_tile = a.tile_size / 64;
  int32_t* out = a.tiles + row * (tiles + 1);
  int count = 0;
  for (int base = 0; base < tiles; base += 64) {
    const int tile = base + lane;
    bool active = false;
    for (int r = 0; r < runs_per_tile; ++r) {
      const int run = tile * runs_per_tile + r;
      active |= run < runs && run_flags[run] != 0;
    }
    const uint64_t votes = __ballot(active);
    if (active) {
      const uint64_t lower = lane == 0 ? 0ull : (votes & ((1ull << lane) - 1ull));
      out[count + __builtin_popcountll(lower)] = tile;
    }
    count += __builtin_popcountll(votes);
  }
  // Slots behind the active ids are never read by the attention kernel.
  for (int slot = count + lane; slot < tiles; slot += 64) out[slot] = -1;
  if (lane == 0) out[tiles] = count;
}

// Workgroups of both outputs, and the bytes of LDS that their flags take.
inline int key_mask_blocks(const KeyMaskArgs& a) {
  const int rows = a.tiles != nullptr ? a.batch * a.heads : 0;
  return rows + (a.bias != nullptr ? a.bias_planes * ((a.padded + 255) / 256) : 0);
}
inline size_t key_mask_flag_bytes(const KeyMaskArgs& a) { return a.tiles != nullptr ? (a.length + 63) / 64 : 0; }

__device__ __forceinline__ void key_mask_block_of(const KeyMaskArgs& a, int dtype, int block, unsigned char* run_flags) {
  if (dtype == kBool)
    key_mask_block<kBool>(a, block, run_flags);
  else if (dtype == kF32)
    key_mask_block<kF32>(a, block, run_flags);
  else if (dtype == kF16)
    key_mask_block<kF16>(a, block, run_flags);
  else
    key_mask_block<kBF16>(a, block, run_flags);
}

// Lane words of a boolean mask (the form kMaskLanes of the attention kernel reads): for
// every block of 32 queries and 64-key tile, 32 words; bit l of word 16*rb + i is the mask
// element of query 32*block + l % 32 and key 64*tile + 32*rb + 8*(i / 4) + 4*(l / 32) + i % 4,
// which is score (rb, i) of lane l in the attention kernel.  Rows past the last query and
// keys past the last key have no bit set.
//
// One workgroup per (group of 16 tiles, block of 32 queries, plane of the mask), 256 threads: a
// wavefront takes four consecutive key tiles of one query block (256 mask bytes per row, all
// requested before the first is used).  Lane (row, half) reads, per tile and 32-key block,
// the sixteen elements at keys 16*half .. 16*half+15 of the block (one 16-byte load when
// ALIGNED): the eight-key groups b4 = 2*half and 2*half+1, both four-key halves of each.
// A vote over element (b', h', r) of every lane therefore holds, in its low 32 bits, the
// rows' decisions for group b' and, in its high 32 bits, those for group 2+b', four-key
// half h' each; a lane word wants the two halves h' of one group side by side, which is a
// regrouping of 32-bit scalar registers.  Lane s keeps word s, so the 32 words of a tile
// leave in one 256-byte store.
constexpr int kLaneTilesPerWave = 4;
// The four votes of two eight-key groups (elements r of both four-key halves) into lanes slot + r of the words'
// halves: low halves of the votes at low_slot, high halves at high_slot.  The votes come from vector
// comparisons, and a vector instruction may read such a scalar register two wait states later: the compiler
// counts them for its own instructions only, so they stand in front of these, once for all sixteen (in front of
// every single one they took 0.4 to 0.9 us of 17 to 41 us whole call, boolean masks of odd rows).
__device__ __forceinline__ void write_lanes(uint32_t& words_low, uint32_t& words_high, const uint64_t (&first)[4],
                                            const uint64_t (&second)[4], int low_slot, int high_slot) {
  const auto low = [](uint64_t vote) { return static_cast<uint32_t>(vote); };
  const auto high = [](uint64_t vote) { return static_cast<uint32_t>(vote >> 32); };
#define RISA_WRITE_LANES(TARGET, VOTE, SLOT)                                          \
  "v_writelane_b32 %[" TARGET "], %[" VOTE "0], %[" SLOT "]\n\t"                      \
  "v_writelane_b32 %[" TARGET "], %[" VOTE "1], %[" SLOT "]+1\n\t"                    \
  "v_writelane_b32 %[" TARGET "], %[" VOTE "2], %[" SLOT "]+2\n\t"                    \
  "v_writelane_b32 %[" TARGET "], %[" VOTE "3], %[" SLOT "]+3\n\t"
  asm("s_nop 1\n\t"
      RISA_WRITE_LANES("words_low", "fl", "low_slot") RISA_WRITE_LANES("words_high", "sl", "low_slot")
      RISA_WRITE_LANES("words_low", "fh", "high_slot") RISA_WRITE_LANES("words_high", "sh", "high_slot")
      : [words_low] "+v"(words_low), [words_high] "+v"(words_high)
      : [fl0] "s"(low(first[0])), [fl1] "s"(low(first[1])), [fl2] "s"(low(first[2])), [fl3] "s"(low(first[3])),
        [fh0] "s"(high(first[0])), [fh1] "s"(high(first[1])), [fh2] "s"(high(first[2])), [fh3] "s"(high(first[3])),
        [sl0] "s"(low(second[0])), [sl1] "s"(low(second[1])), [sl2] "s"(low(second[2])), [sl3] "s"(low(second[3])),
        [sh0] "s"(high(second[0])), [sh1] "s"(high(second[1])), [sh2] "s"(high(second[2])), [sh3] "s"(high(second[3])),
        [low_slot] "n"(low_slot), [high_slot] "n"(high_slot));
#undef RISA_WRITE_LANES
}
template <bool ALIGNED>
__device__ __forceinline__ void mask_lanes_block(const MaskLaneArgs& a, int tile_group, int query_wave, int plane) {
  const int q_len = a.q_len, k_len = a.k_len, key_tiles = a.key_tiles, query_waves = a.query_waves;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = query_wave * 32 + (lane & 31), half = lane >> 5;
  const bool row_ok = row < q_len;
  const uint8_t* row_mask = a.mask + (plane / a.heads) * a.stride_b + (plane % a.heads) * a.stride_h +
                            static_cast<int64_t>(row_ok ? row : q_len - 1) * a.stride_q;
  uint64_t* out = a.lanes + (static_cast<int64_t>(plane) * query_waves + query_wave) * key_tiles * 32;
  const int first_tile = (tile_group * 4 + wave) * kLaneTilesPerWave;
  typedef uint32_t v4u __attribute__((ext_vector_type(4)));
  v4u chunk[kLaneTilesPerWave][2];
#pragma unroll
  for (int t = 0; t < kLaneTilesPerWave; ++t) {
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int key = (first_tile + t) * 64 + rb * 32 + half * 16;
      v4u words = {0u, 0u, 0u, 0u};
      if (ALIGNED && key + 15 < k_len) {
        words = *reinterpret_cast<const v4u*>(row_mask + key);
      } else {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          if (key + j < k_len && row_mask[key + j] != 0) words[j >> 2] |= 1u << (8 * (j & 3));
        }
      }
      if (!row_ok) words = v4u{0u, 0u, 0u, 0u};
      chunk[t][rb] = words;
    }
  }
#pragma unroll
  for (int t = 0; t < kLaneTilesPerWave; ++t) {
    if (first_tile + t >= key_tiles) break;  // wave-uniform
    // word s of the tile goes to lane s, 32 bits at a time, straight from the scalar registers
    uint32_t mine_low = 0, mine_high = 0;
    uint64_t every = ~uint64_t{0}, any = 0;  // what all words of the tile / at least one of them hold
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
      for (int group = 0; group < 2; ++group) {  // b'
        uint64_t first[4], second[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          first[r] = __ballot(((chunk[t][rb][group * 2] >> (8 * r)) & 0xffu) != 0);
          second[r] = __ballot(((chunk[t][rb][group * 2 + 1] >> (8 * r)) & 0xffu) != 0);
          every &= first[r] & second[r];
          any |= first[r] | second[r];
        }
        // b4 = b' and b4 = 2 + b'
        write_lanes(mine_low, mine_high, first, second, rb * 16 + group * 4, rb * 16 + (2 + group) * 4);
      }
    }
    const uint64_t mine = mine_low | (static_cast<uint64_t>(mine_high) << 32);
    if (lane < 32) out[static_cast<int64_t>(first_tile + t) * 32 + lane] = mine;
    if (lane == 0) {
      a.classes[(static_cast<int64_t>(plane) * query_waves + query_wave) * key_tiles + first_tile + t] =
          every == ~uint64_t{0} ? kLaneTileVisible : any == 0 ? kLaneTileHidden : kLaneTileMixed;
    }
  }
}

// (group of 16 tiles, block of 32 queries, plane) of a workgroup's number, groups first, for aligned masks.
inline int mask_lane_groups(const MaskLaneArgs& a) { return (a.key_tiles + 4 * kLaneTilesPerWave - 1) / (4 * kLaneTilesPerWave); }
__device__ __forceinline__ void mask_lanes_block_of(const MaskLaneArgs& a, int groups, int block) {
  const int rest = block / groups;
  mask_lanes_block<true>(a, block % groups, rest % a.query_waves, rest / a.query_waves);
}

// Tile lists of the mask: one wavefront per (query block, plane).  A tile is listed for a
// block of 128 queries unless all four of its 32-query classes say "no visible key"; entry
// [tiles] of a list holds its length (the layout the attention kernel reads for key-mask
// tiles).  A block that sees nothing keeps an empty list: its rows come out as zeros.
__device__ __forceinline__ void mask_tile_list(const MaskLaneArgs& a, int block, int plane, int lane) {
  const int key_tiles = a.key_tiles, query_blocks = a.query_waves / 4;
  const int32_t* wave_classes = a.classes + (static_cast<int64_t>(plane) * query_blocks + block) * 4 * key_tiles;
  int32_t* list = a.lists + (static_cast<int64_t>(plane) * query_blocks + block) * (key_tiles + 1);
  int count = 0;
  for (int first = 0; first < key_tiles; first += 64) {
    const int tile = first + lane;
    bool listed = false;
    if (tile < key_tiles) {
#pragma unroll
      for (int w = 0; w < 4; ++w) listed = listed || wave_classes[w * key_tiles + tile] != kLaneTileHidden;
    }
    const uint64_t ballot = __ballot(listed);
    if (listed) list[count + __popcll(ballot & ((uint64_t{1} << lane) - 1))] = tile;
    count += __popcll(ballot);
  }
  if (lane == 0) list[key_tiles] = count;
}

}  // namespace risa
