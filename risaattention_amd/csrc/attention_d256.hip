// Head dim 256 with thirty-two queries per wavefront: 128-key tiles, two 128-query workgroups per
// compute unit, every tile in a hand-scheduled walk (gen_d256_loops.py, which says how the operands
// are staged and why the compiler cannot schedule it).
//
// The sixteen-query kernel reads every K and V fragment twice as often from LDS and leaves its vector
// and matrix cycles (59 and 33 % of its time) one behind the other: one barrier holds all eight
// wavefronts of a compute unit in the same phase.  Here the two wavefronts of a SIMD belong to different
// workgroups and drift apart (77 and 50 %).  16/4 heads x 8192: 1.61 -> 1.04 million cycles, at 1.71 instead
// of 1.99 GHz (the power the part is allowed bounds it: on all-zero operands 2.11 GHz and 480 us), 810 -> 611 us
// with counters, whole call 740 -> 617 us = 1.78e15 operations a second.  Arithmetic per score as in
// attention_kernel.hpp.
#include "attention_kernel.hpp"

namespace risa {
namespace {

constexpr int kDim = 256, kKeys = 128;
// LDS (gen_d256_loops.py): accumulator seeds and additive row of the tile, V scale and centre, K tile, V tile
constexpr int kChannelOffset = 2048, kKeyOffset = 4096, kValueOffset = kKeyOffset + kDim * kKeys;
constexpr int kLdsBytes = kValueOffset + kDim * kKeys;

template <bool SCALED, bool BIAS, bool LISTED>
__global__ __launch_bounds__(256, 2) void attention_d256_kernel(const KernelParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int lane = tid & 63;
  // Query blocks of one head next to each other; under the causal rule longest first, across all heads.
  int bx, head, batch;
  if (SCALED && p.causal) {
    const int heads = p.q_heads * p.batch;
    const int rest = blockIdx.x % heads;
    bx = p.n_qb - 1 - blockIdx.x / heads;
    head = rest % p.q_heads;
    batch = rest / p.q_heads;
  } else {
    bx = blockIdx.x % p.n_qb;
    const int rest = blockIdx.x / p.n_qb;
    head = rest % p.q_heads;
    batch = rest / p.q_heads;
  }
  const int64_t bhk = static_cast<int64_t>(batch) * p.kv_heads + head / (p.q_heads / p.kv_heads);
  const int64_t bhq = static_cast<int64_t>(batch) * p.q_heads + head;
  const int8_t* k_base = p.k + bhk * p.k_len * kDim;
  const int8_t* v_base = p.v + bhk * kDim * p.padded;
  const int32_t* sum_base = p.v_tile_sum + bhk * p.n_kb * kDim;
  const float* ks_base = p.k_scale + bhk * p.n_kb * 4;
  [[maybe_unused]] const float* bias_base = nullptr;
  if constexpr (BIAS) bias_base = p.key_bias + batch * p.key_bias_stride_b + head * p.key_bias_stride_h;

  const int first_query = bx * kQueryBlock + wave * 32;
  v4i qreg[8];
  float q_scale = 1.0f;
  {
    const int l32 = lane & 31, half = lane >> 5, query = first_query + l32;
    const bool query_ok = query < p.q_len;
    const int8_t* q_row = p.q + (bhq * p.q_len + query) * kDim;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk)
      qreg[kk] = query_ok ? *reinterpret_cast<const v4i*>(q_row + kk * 32 + half * 16) : v4i{0, 0, 0, 0};
    const int q_groups = p.n_qb * 64;  // groups of the four tokens n, n + 8, ... of sixteen
    if (query_ok) q_scale = p.q_scale[bhq * q_groups + (query / 16) * 8 + (query & 7)];
  }
  if (wave >= 2) {  // V scale by the third wavefront, centre by the fourth
    copy16_to_lds_uniform(reinterpret_cast<const int8_t*>((wave == 2 ? p.v_scale : p.v_center) + bhk * kDim),
                          static_cast<uint32_t>(lane) * 16, lds + kChannelOffset + (wave - 2) * (kDim * 4));
  }

  int n_it = p.n_kb;
  [[maybe_unused]] const int32_t* indices = nullptr;
  if constexpr (LISTED) {
    indices = p.tile_indices + bhq * (p.n_kb + 1);
    n_it = indices[p.n_kb];
  } else if (SCALED && p.causal) {
    n_it = (min(p.k_len, (bx + 1) * kQueryBlock) + kKeys - 1) / kKeys;
  }
  n_it = __builtin_amdgcn_readfirstlane(n_it);

  v16i out[8];
#pragma unroll
  for (int cb = 0; cb < 8; ++cb)
#pragma unroll
    for (int i = 0; i < 16; ++i) out[cb][i] = 0;
  float m_run = kRowFloor;
  float d_part = 0.0f;  // this lane's half of the row denominator
  if (n_it > 0) {
    typedef __attribute__((address_space(3))) unsigned char* LdsBytes;
    const uint32_t lds_address = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((LdsBytes)lds));
    const int l32 = lane & 31, half = lane >> 5;
    // this lane's fragment addresses in row l32 of a 32-row block, and its shares of the copy sources
    const uint32_t k_address = lds_address + kKeyOffset + swizzled<kDim>(l32, half);
    const uint32_t v_address = lds_address + kValueOffset + swizzled<kKeys>(l32, half);
    uint32_t k_share = (lane >> 4) * kDim + (((lane & 15) ^ (lane >> 4)) << 4);
    uint32_t v_share = static_cast<uint32_t>(lane >> 3) * static_cast<uint32_t>(p.padded) + (((lane & 7) ^ (lane >> 4)) << 4);
    const int count = n_it - 1;
    // Keys of the last tile that its wavefront's first query sees: those in range, and under the
    // causal rule one more per query.  (An additive row hides the keys past the end by itself.)
    constexpr int kAll = 1 << 30;
    const int keys_left = BIAS ? kAll : p.k_len - count * kKeys;
    const int keys_to_query = SCALED && !LISTED && p.causal ? first_query + 1 - count * kKeys : kAll;
    if constexpr (LISTED) {
#include "d256_loop_bias_listed.inc"
    } else if constexpr (BIAS) {
#include "d256_loop_bias.inc"
    } else if constexpr (SCALED) {
#include "d256_loop_scaled.inc"
    } else {
#include "d256_loop_raw.inc"
    }
  }

  // ---- epilogue: as in attention_kernel.hpp, rows through LDS and out as whole rows ----
  lane = fresh_lane();
  const int l32 = lane & 31, half = lane >> 5, query = first_query + l32;
  __builtin_amdgcn_s_waitcnt(0x0f70);  // (without a listed tile nothing has waited for the channel parameters)
  __syncthreads();                     // no wavefront reads a tile any more
  constexpr int ROW_BYTES = kDim * 2;
  const float d_total = d_part + __shfl_xor(d_part, 32);
  const bool row_valid = d_total > 0.0f;
  const float inv_d = 1.0f / d_total;
  const bool zero_row = SCALED && (BIAS || p.causal) && !row_valid;
  unsigned char* mine = lds + kKeyOffset + wave * (32 * ROW_BYTES);
  unsigned char* out_block = static_cast<unsigned char*>(p.out) +
                             2 * (batch * p.out_stride_b + head * p.out_stride_h +
                                  static_cast<int64_t>(first_query) * p.out_stride_n);
#pragma unroll
  for (int cb = 0; cb < 8; ++cb)
#pragma unroll
    for (int b4 = 0; b4 < 4; ++b4) {
      const int c = cb * 32 + b4 * 8 + half * 4;
      const v4f scale4 = *reinterpret_cast<const v4f*>(lds + kChannelOffset + c * 4);
      const v4f center4 = *reinterpret_cast<const v4f*>(lds + kChannelOffset + kDim * 4 + c * 4);
      float value[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        value[r] = __builtin_fmaf(__int_as_float(out[cb][b4 * 4 + r]) * inv_d, scale4[r], center4[r]);
        value[r] = zero_row ? 0.0f : value[r];
      }
      typedef uint32_t v2u __attribute__((ext_vector_type(2)));
      v2u word;
      word.x = to_output_pair(value[0], value[1], p.out_dtype);
      word.y = to_output_pair(value[2], value[3], p.out_dtype);
      *reinterpret_cast<v2u*>(mine + l32 * ROW_BYTES + (((cb * 4 + b4) ^ (l32 & 31)) << 4) + half * 8) = word;
    }
  asm volatile("" ::: "memory");  // the pieces below are read from other lanes' writes
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int row = i * 2 + half, chunk = l32;
    const v4i piece = *reinterpret_cast<const v4i*>(mine + row * ROW_BYTES + ((chunk ^ row) << 4));
    if (first_query + row < p.q_len) {
      *reinterpret_cast<v4i*>(out_block + 2 * static_cast<int64_t>(row) * p.out_stride_n + chunk * 16) = piece;
    }
  }
  if (p.lse != 0 && half == 0 && query < p.q_len) {
    store_lse(p, bhq * p.q_len + query,
              row_valid ? (__builtin_amdgcn_logf(d_total) + m_run) / kLog2e : -__builtin_inff());
  }
}

template <bool SCALED, bool BIAS, bool LISTED> int launch(const KernelParams& p, hipStream_t stream) {
  auto kernel = attention_d256_kernel<SCALED, BIAS, LISTED>;
  static thread_local int configured_device = -1;
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess) return fail("risa_attention: hipGetDevice failed");
  if (device != configured_device) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                            kLdsBytes) != hipSuccess) {
      return fail("risa_attention: cannot reserve " + std::to_string(kLdsBytes) + " bytes of LDS");
    }
    configured_device = device;
  }
  const dim3 grid(static_cast<unsigned>(p.n_qb) * p.q_heads * p.batch);
  kernel<<<grid, 256, kLdsBytes, stream>>>(p);
  return 0;
}

}  // namespace

int launch_attention_d256(const KernelParams& p, bool fast, hipStream_t stream) {
  if (fast) return launch<false, false, false>(p, stream);
  if (p.mask_dtype != kKeyBias) return launch<true, false, false>(p, stream);
  return p.index_mode == 2 ? launch<true, true, true>(p, stream) : launch<true, true, false>(p, stream);
}

}  // namespace risa
