// The step before append, fused into one launch: optional head-wise RMS
// norm of q and k, optional RMS norm of v, RoPE of q and k, and the append
// of k and v into the paged pool (f16 or q8_0).  Restates the part of
// compute_layer_attention_residual between the Q/K/V projections and
// store_attention_kv_cache (text/generator/detail.hpp:3806-3825) and the same
// steps of the chunked-prefill row loop (detail.hpp:4335-4360).
//
// Every product and sum is evaluated unfused in the reference's order
// (floating-point contraction is off for this whole file), and division and
// square root are the correctly rounded IEEE ones (hipcc's default
// -fhip-fp32-correctly-rounded-divide-sqrt; __fsqrt_rn would be the native,
// 1-ulp v_sqrt_f32), so the results are bit-exact against that arithmetic.  cos/sin come from a
// table built on the host with the reference's recurrence.
//
// Launch: a wave takes up to RW rows of one token, where the rows of a token
// are its n_head q heads, n_head_kv k heads and n_head_kv v heads.  A row lies
// over D / 4 lanes, four dims each, in registers; the position, page and table
// reads are per wave (scalar), the (cos, sin) and weights are read once for
// all of its rows, and no step synchronises across waves.
#include <hip/hip_runtime.h>

#include <cmath>
#include <new>
#include <vector>

#include "device_common.hpp"
#include "emelk.h"
#include "pool_layout.hpp"

#pragma clang fp contract(off)

struct emelk_rope_table {
  emelk_rope_params params;
  int32_t head_dim = 0;
  int32_t pair_count = 0;
  int32_t x1_base = 0;
  int32_t max_positions = 0;
  float2 *dev = nullptr;  // [max_positions][pair_count] (cos, sin)
};

namespace emelk {
namespace {

using namespace emelk::dev;

constexpr int k_waves = 4;  // waves per workgroup
constexpr int k_max_dim = 512;

struct rope_append_args {
  pool_layout L;
  uint8_t *k_pool;
  uint8_t *v_pool;
  int32_t layer;
  const float *q_in;
  float *q_out;
  const float *k_rows;
  const float *v_rows;
  int32_t n_seq;
  int32_t n_tokens;
  const int32_t *positions;
  const uint16_t *tables;
  int32_t table_stride;
  const float2 *rope;
  int32_t rope_positions;
  int32_t pair_count;
  int32_t x0_stride;
  int32_t x1_stride;
  int32_t x1_base;
  const float *q_norm;
  const float *k_norm;
  int32_t v_rms;
  float eps;
  int32_t pairing;  // rope_pairs
};

// Which dims a pair has: neighbours, the two halves of the head, or any other
// pairing (rotated through LDS).
enum rope_pairs : int32_t { k_pairs_none, k_pairs_adjacent, k_pairs_halves, k_pairs_general };

// fp32 rows and weights may lie at any 4-byte address.
typedef float float4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef float float2_u __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t uint2_u __attribute__((ext_vector_type(2), aligned(4)));

// apply_rms_norm_in_place's scale (detail.hpp:1098-1106) of one token's whole
// v, summed in its order: the wave loads 64 values per coalesced load (8 chunks
// ahead) and every lane adds the squares one by one, each taken from its lane
// with readlane.
__device__ __forceinline__ float v_scale(const float *__restrict__ v, int32_t n, int32_t lane,
                                         float eps) {
  constexpr int kC = 8;
  double ss = 0.0;
  for (int32_t c0 = 0; c0 < n; c0 += kC * k_wave) {
    float sq[kC];
#pragma unroll
    for (int u = 0; u < kC; ++u) {
      const int32_t i = c0 + u * k_wave + lane;
      const float x = i < n ? v[i] : 0.0f;
      sq[u] = x * x;
    }
#pragma unroll
    for (int u = 0; u < kC; ++u) {
      const int32_t left = n - (c0 + u * k_wave);
      if (left <= 0) break;  // uniform
      const double dq = static_cast<double>(sq[u]);
      if (left >= k_wave) {  // a full chunk: lane indices known at compile time
#pragma unroll
        for (int j = 0; j < k_wave; ++j) {
          const int lo = __builtin_amdgcn_readlane(static_cast<int>(__builtin_bit_cast(uint64_t, dq)), j);
          const int hi = __builtin_amdgcn_readlane(static_cast<int>(__builtin_bit_cast(uint64_t, dq) >> 32), j);
          ss += __builtin_bit_cast(double, (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) |
                                               static_cast<uint32_t>(lo));
        }
      } else {
        for (int32_t j = 0; j < left; ++j) {
          ss += static_cast<double>(__builtin_bit_cast(
              float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sq[u]), j)));
        }
      }
    }
  }
  const float mean = static_cast<float>(ss / static_cast<double>(n));
  return 1.0f / sqrtf(mean + eps);
}

// NI row slots per lane: RW = NI * RPI rows per wave, RPI of them per load
// instruction.  What bounds it: memory for a prompt chunk, latency for a
// decode step.  The norm's sum must add a row's squares one after another
// (the reference's order), so the squares go through LDS to one lane per row:
// RW rows are summed at once, where one lane per wave summing row after row
// had made it the whole cost.
//
// NORMS: some norm is asked for; Q8: a q8_0 pool.  Launches without either are
// kernels of their own, with a third to a half of the registers (31 against 92
// at head_dim 512, one slot): with the norms in it, 8 x 512 rows of 8/1 heads
// of 512 took 28.0 us and 11 x 276 22.6, 26.2 and 20.9 without; 64/8 heads of
// 128 72 and 62.
template <int D, int NI, bool NORMS, bool Q8>
__global__ __launch_bounds__(k_waves *k_wave) void rope_append_kernel(rope_append_args A) {
  constexpr int LPR = D / 4 < k_wave ? D / 4 : k_wave;  // lanes of a row
  constexpr int RPI = k_wave / LPR;                     // rows per load instruction
  constexpr int NC = D / 4 / LPR;                       // 4-dim chunks of a row per lane
  constexpr int RW = NI * RPI;
  constexpr int LROW = D + 4;   // padded LDS row: one lane per row reads without bank conflicts
  constexpr int NPL = 4;        // (cos, sin) pairs held per lane
  static_assert(RW <= k_wave, "one lane per row in the norm's sum");
  extern __shared__ __align__(16) float s_rows[];  // [k_waves][RW][LROW], where a launch needs it

  const pool_layout &L = A.L;
  const int32_t wave = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(threadIdx.x / k_wave));
  const int32_t lane = threadIdx.x % k_wave;
  const uint32_t n_tok = static_cast<uint32_t>(A.n_tokens);
  const uint32_t tok = blockIdx.x * k_waves + static_cast<uint32_t>(wave);  // < 2^31 (host check)
  if (tok >= static_cast<uint32_t>(A.n_seq) * n_tok) return;
  const uint32_t s = tok / n_tok;
  const int32_t n_qk = L.n_head + L.n_head_kv;
  const int32_t n_rows = n_qk + L.n_head_kv;
  const int32_t row0 = static_cast<int32_t>(blockIdx.y) * RW;
  const int32_t sub = lane / LPR;
  const int32_t l = lane % LPR;

  // The rows are requested together with the position, before the token's
  // validity is known.
  const float *q_src = A.q_in + static_cast<uint64_t>(tok) * L.n_head * D;
  const float *k_src = A.k_rows + static_cast<uint64_t>(tok) * L.n_head_kv * D;
  const float *v_src = A.v_rows + static_cast<uint64_t>(tok) * L.n_head_kv * D;
  float4_t x[NI][NC];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int32_t row = row0 + i * RPI + sub;
    const float *src = row < L.n_head ? q_src + row * D
                       : row < n_qk   ? k_src + (row - L.n_head) * D
                                      : v_src + (row - n_qk) * D;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      x[i][c] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
      if (row < n_rows) x[i][c] = *reinterpret_cast<const float4_u *>(src + 4 * (l + c * LPR));
    }
  }
  const int32_t pos = A.positions[s] + static_cast<int32_t>(tok - s * n_tok);
  // An invalid token (no position, outside the rope table, past the table
  // row or on an invalid page) writes nothing, q included.
  if (pos < 0) return;
  if (A.pair_count > 0 && pos >= A.rope_positions) return;
  const bool rotates = row0 < n_qk && A.pairing != k_pairs_none;  // uniform
  // adjacent pairs: those of the lane's dims; halves: the four of the lane's
  // dims, which both halves share; general: pairs lane, lane + 64, ...
  float2 cs[NPL];
  if (rotates) {
    const float2 *table = A.rope + static_cast<uint64_t>(pos) * A.pair_count;
#pragma unroll
    for (int e = 0; e < NPL; ++e) {
      const int32_t pr = A.pairing == k_pairs_adjacent ? 2 * (l + e / 2 * LPR) + e % 2
                         : A.pairing == k_pairs_halves ? 4 * l % (D / 2) + e
                                                       : lane + e * k_wave;
      cs[e] = float2{1.0f, 0.0f};
      if (pr < A.pair_count) cs[e] = table[pr];
    }
  }
  const int32_t lb = pos / L.block_tokens;
  if (lb >= A.table_stride) return;
  const uint32_t page = A.tables[static_cast<uint64_t>(s) * A.table_stride + lb];
  if (page >= static_cast<uint32_t>(L.max_blocks)) return;
  const int32_t slot = pos % L.block_tokens;

  float *buf = s_rows + wave * (RW * LROW);
  // Each wave stages only its own rows, so ordering its own LDS operations is
  // all the synchronisation needed.
  auto wave_sync = []() {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
  };
  if (NORMS && row0 < n_qk && (A.q_norm != nullptr || A.k_norm != nullptr)) {  // uniform
    // apply_headwise_rms_norm (detail.hpp:1073-1082)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        *reinterpret_cast<float4_t *>(buf + (i * RPI + sub) * LROW + 4 * (l + c * LPR)) =
            x[i][c] * x[i][c];
      }
    }
    wave_sync();
    float sc = 1.0f;
    if (lane < RW) {
      float ss = 0.0f;
#pragma unroll 16
      for (int d = 0; d < D; d += 4) {
        const float4_t sq = *reinterpret_cast<const float4_t *>(buf + lane * LROW + d);
        ss += sq.x;
        ss += sq.y;
        ss += sq.z;
        ss += sq.w;
      }
      sc = 1.0f / sqrtf(ss / static_cast<float>(D) + A.eps);
    }
    float4_t wq[NC], wk[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (A.q_norm != nullptr) wq[c] = *reinterpret_cast<const float4_u *>(A.q_norm + 4 * (l + c * LPR));
      if (A.k_norm != nullptr) wk[c] = *reinterpret_cast<const float4_u *>(A.k_norm + 4 * (l + c * LPR));
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int32_t row = row0 + i * RPI + sub;
      const float rs = __shfl(sc, i * RPI + sub, k_wave);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        if (row < L.n_head) {
          if (A.q_norm != nullptr) x[i][c] *= rs * wq[c];
        } else if (row < n_qk) {
          if (A.k_norm != nullptr) x[i][c] *= rs * wk[c];
        }
      }
    }
  }
  if (NORMS && A.v_rms != 0 && row0 + RW > n_qk) {  // uniform
    const float rs = v_scale(v_src, L.n_head_kv * D, lane, A.eps);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        if (row0 + i * RPI + sub >= n_qk) x[i][c] *= rs;
      }
    }
  }

  // apply_rope_pairing (detail.hpp:2905-2936); pairs never overlap, so their
  // order does not matter
  if (rotates && A.pairing == k_pairs_general) {
    wave_sync();  // the norm's reads are done
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        *reinterpret_cast<float4_t *>(buf + (i * RPI + sub) * LROW + 4 * (l + c * LPR)) = x[i][c];
      }
    }
    wave_sync();
    for (int j = 0; j < RW && row0 + j < n_qk; ++j) {  // uniform
#pragma unroll
      for (int e = 0; e < NPL; ++e) {
        const int32_t pr = lane + e * k_wave;
        if (pr < A.pair_count) {
          float *b0 = buf + j * LROW + pr * A.x0_stride;
          float *b1 = buf + j * LROW + pr * A.x1_stride + A.x1_base;
          const float x0 = *b0;
          const float x1 = *b1;
          *b0 = x0 * cs[e].x - x1 * cs[e].y;
          *b1 = x0 * cs[e].y + x1 * cs[e].x;
        }
      }
    }
    wave_sync();
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        x[i][c] = *reinterpret_cast<const float4_t *>(buf + (i * RPI + sub) * LROW + 4 * (l + c * LPR));
      }
    }
  } else if (rotates && A.pairing == k_pairs_halves) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const bool turn = row0 + i * RPI + sub < n_qk;
      if constexpr (NC == 2) {  // both halves in the lane
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x0 = x[i][0][e], x1 = x[i][NC - 1][e];
          if (turn) {
            x[i][0][e] = x0 * cs[e].x - x1 * cs[e].y;
            x[i][NC - 1][e] = x0 * cs[e].y + x1 * cs[e].x;
          }
        }
      } else {  // the other half lies LPR / 2 lanes away
        const bool upper = l >= LPR / 2;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float own = x[i][0][e];
          const float other = __shfl_xor(own, LPR / 2, k_wave);
          const float x0 = upper ? other : own, x1 = upper ? own : other;
          const float y = upper ? x0 * cs[e].y + x1 * cs[e].x : x0 * cs[e].x - x1 * cs[e].y;
          x[i][0][e] = turn ? y : own;
        }
      }
    }
  } else if (rotates) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const bool turn = row0 + i * RPI + sub < n_qk;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float x0 = x[i][c][2 * e], x1 = x[i][c][2 * e + 1];
          if (turn && 2 * (l + c * LPR) + e < A.pair_count) {
            x[i][c][2 * e] = x0 * cs[2 * c + e].x - x1 * cs[2 * c + e].y;
            x[i][c][2 * e + 1] = x0 * cs[2 * c + e].y + x1 * cs[2 * c + e].x;
          }
        }
      }
    }
  }

#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int32_t row = row0 + i * RPI + sub;
    const int32_t kvh = row < n_qk ? row - L.n_head : row - n_qk;
    uint8_t *region = (row < n_qk ? A.k_pool : A.v_pool) +
                      L.region_offset(A.layer, static_cast<int32_t>(page), kvh);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int32_t d = 4 * (l + c * LPR);
      const float4_t y = x[i][c];
      if (row < L.n_head) {
        *reinterpret_cast<float4_u *>(A.q_out + (static_cast<uint64_t>(tok) * L.n_head + row) * D + d) = y;
      } else if (!Q8 && row < n_rows) {
        // store_fp16_rounded_cache (detail.hpp:3050-3055): RNE per value
        *reinterpret_cast<uint2_u *>(region + (static_cast<uint64_t>(slot) * D + d) * 2u) =
            uint2_u{as_u32(pack_half2(y.x, y.y)), as_u32(pack_half2(y.z, y.w))};
      }
      if (Q8 && row0 + RW > L.n_head) {  // uniform
        // quantize_row_q8_0_strided (kernel/detail.hpp:804-824) as
        // quantize_block32: a block is 8 lanes, which share its amax
        float amax = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) amax = fmaxf(amax, fabsf(y[e]));
        amax = fmaxf(amax, dpp<k_dpp_quad_xor1>(amax));
        amax = fmaxf(amax, dpp<k_dpp_quad_xor2>(amax));
        amax = fmaxf(amax, dpp<k_dpp_row_half_mirror>(amax));
        const float dq = amax / 127.0f;
        const float inv = dq != 0.0f ? 1.0f / dq : 0.0f;
        uint32_t w = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          int q = static_cast<int>(roundf(y[e] * inv));
          q = q < -127 ? -127 : (q > 127 ? 127 : q);
          w |= (static_cast<uint32_t>(q) & 0xFFu) << (8 * e);
        }
        if (row >= L.n_head && row < n_rows) {
          *reinterpret_cast<uint32_t *>(region + static_cast<uint64_t>(slot) * D + d) = w;
          if (l % 8 == 0) {
            reinterpret_cast<uint16_t *>(region + L.scale_plane())
                [static_cast<uint64_t>(slot) * (D / 32) + d / 32] = f32_to_f16_bits(dq);
          }
        }
      }
    }
  }
}

// Row slots per lane: as many as leave the launch k_enough_waves waves (a
// prompt chunk), one for a decode step, whose latency counts.  Measured on
// MI355X with 1 / 2 / 4 / 8 slots at most: 8 x 512 tokens of 16/8 heads of 128
// with q and k norms and halved pairs 38 / 29 / 28 / 42 us (69 with one lane
// per wave summing row after row; 4.2 TB/s at 28); 64 x 512 of 32/8 heads,
// adjacent pairs, 376 / 330 / 304 / 476 (444 before; 271, 5.4 TB/s, since such
// launches have no norm in them), on a q8_0 pool 387 / 340 / 313 / 510 (694 with
// one thread per 32-value block; now 261).  A decode
// step of 8 tokens takes 4.6 us (5.4 before, q8_0 8.3).  Waves of a workgroup
// that take one token's next rows instead of the next token's same rows were
// no faster (29 and 315 us at four slots).  Rows of 256 and 512 dims without
// norms take two at most: four leave them fewer waves and, at 10 rows a token,
// two slots in twelve empty (8 x 512 of 8/1 heads of 256 19.6 us with four, 18.6
// with two).
constexpr int k_slots_at(int head_dim, bool norms) { return head_dim > 128 && !norms ? 2 : 4; }
constexpr int64_t k_enough_waves = 4096;
template <int D, int NI, bool NORMS>
bool launch_rope_slots(const rope_append_args &A, hipStream_t st) {
  constexpr int LPR = D / 4 < k_wave ? D / 4 : k_wave;
  constexpr int RW = NI * (k_wave / LPR);
  const int32_t n_rows = A.L.n_head + 2 * A.L.n_head_kv;
  const int64_t tokens = static_cast<int64_t>(A.n_seq) * A.n_tokens;
  const int64_t parts = (n_rows + RW - 1) / RW;
  if constexpr (NI > 1) {
    if (tokens * parts < k_enough_waves || RW > n_rows) {
      return launch_rope_slots<D, NI / 2, NORMS>(A, st);
    }
  }
  const bool lds = A.q_norm != nullptr || A.k_norm != nullptr || A.pairing == k_pairs_general;
  const uint32_t lds_bytes = lds ? k_waves * RW * (D + 4) * sizeof(float) : 0;
  const dim3 grid(static_cast<uint32_t>((tokens + k_waves - 1) / k_waves), static_cast<uint32_t>(parts));
  const dim3 block(k_waves * k_wave);
  if (A.L.kv_type == EMELK_KV_F16) {
    hipLaunchKernelGGL((rope_append_kernel<D, NI, NORMS, false>), grid, block, lds_bytes, st, A);
  } else {
    hipLaunchKernelGGL((rope_append_kernel<D, NI, NORMS, true>), grid, block, lds_bytes, st, A);
  }
  return hipGetLastError() == hipSuccess;
}

template <int D>
bool launch_rope(const rope_append_args &A, hipStream_t st) {
  return A.q_norm != nullptr || A.k_norm != nullptr || A.v_rms != 0
             ? launch_rope_slots<D, k_slots_at(D, true), true>(A, st)
             : launch_rope_slots<D, k_slots_at(D, false), false>(A, st);
}

// Checks a pairing: every pair inside the head and no dim used twice.
bool pairing_ok(const emelk_rope_params &p, int32_t head_dim, int32_t pair_count, int32_t x1_base) {
  if (p.x0_stride < 0 || p.x1_stride < 0 || x1_base < 0) return false;
  std::vector<char> used(static_cast<size_t>(head_dim), 0);
  for (int32_t i = 0; i < pair_count; ++i) {
    const int64_t d0 = static_cast<int64_t>(i) * p.x0_stride;
    const int64_t d1 = static_cast<int64_t>(i) * p.x1_stride + x1_base;
    if (d0 >= head_dim || d1 >= head_dim || d0 == d1) return false;
    if (used[static_cast<size_t>(d0)] || used[static_cast<size_t>(d1)]) return false;
    used[static_cast<size_t>(d0)] = 1;
    used[static_cast<size_t>(d1)] = 1;
  }
  return true;
}

}  // namespace
}  // namespace emelk

extern "C" emel_error_type emelk_rope_table_create(const emelk_rope_params *params,
                                                   int32_t head_dim, int32_t max_positions,
                                                   void *stream, emelk_rope_table **table_out) {
  if (table_out == nullptr) return EMELK_ERR_INVALID_REQUEST;
  *table_out = nullptr;
  if (params == nullptr || head_dim <= 0 || head_dim > emelk::k_max_dim || max_positions <= 0 ||
      !(params->freq_base > 0.0f) || !std::isfinite(params->freq_base)) {
    return EMELK_ERR_INVALID_REQUEST;
  }
  const int32_t rot_dim = params->n_rot < head_dim ? params->n_rot : head_dim;
  // apply_rope_pairing leaves the vector unchanged when rot_dim <= 1
  const int32_t pair_count = rot_dim > 1 ? rot_dim / 2 : 0;
  const int64_t x1_base_wide = static_cast<int64_t>(params->x1_offset) +
                               static_cast<int64_t>(params->x1_half_rot_offset) * pair_count;
  if (x1_base_wide < 0 || x1_base_wide > head_dim) return EMELK_ERR_INVALID_REQUEST;
  const int32_t x1_base = static_cast<int32_t>(x1_base_wide);
  if (!emelk::pairing_ok(*params, head_dim, pair_count, x1_base)) return EMELK_ERR_INVALID_REQUEST;
  const uint64_t entries = static_cast<uint64_t>(max_positions) * static_cast<uint64_t>(pair_count);
  if (entries > (uint64_t{1} << 29)) return EMELK_ERR_INVALID_REQUEST;  // 4 GiB of (cos, sin)

  auto *tb = new (std::nothrow) emelk_rope_table();
  if (tb == nullptr) return EMELK_ERR_OUT_OF_MEMORY;
  tb->params = *params;
  tb->head_dim = head_dim;
  tb->pair_count = pair_count;
  tb->x1_base = x1_base;
  tb->max_positions = max_positions;
  if (entries > 0) {
    std::vector<float2> host;
    try {
      host.resize(entries);
    } catch (...) {
      delete tb;
      return EMELK_ERR_OUT_OF_MEMORY;
    }
    // the per-call recurrence of apply_rope_pairing (detail.hpp:2915-2934)
    const float theta_scale = ::powf(params->freq_base, -2.0f / static_cast<float>(rot_dim));
    for (int32_t p = 0; p < max_positions; ++p) {
      float theta = static_cast<float>(p);
      float2 *row = host.data() + static_cast<uint64_t>(p) * pair_count;
      for (int32_t i = 0; i < pair_count; ++i) {
        row[i] = make_float2(::cosf(theta), ::sinf(theta));
        theta *= theta_scale;
      }
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (hipMalloc(reinterpret_cast<void **>(&tb->dev), entries * sizeof(float2)) != hipSuccess) {
      delete tb;
      return EMELK_ERR_OUT_OF_MEMORY;
    }
    if (hipMemcpyAsync(tb->dev, host.data(), entries * sizeof(float2), hipMemcpyHostToDevice, st) !=
            hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess) {
      emelk_rope_table_destroy(tb);
      return EMELK_ERR_BACKEND;
    }
  }
  *table_out = tb;
  return EMELK_ERR_NONE;
}

extern "C" void emelk_rope_table_destroy(emelk_rope_table *table) {
  if (table == nullptr) return;
  if (table->dev != nullptr) {
    (void)hipDeviceSynchronize();
    (void)hipFree(table->dev);
  }
  delete table;
}

extern "C" int32_t emelk_rope_table_positions(const emelk_rope_table *table) {
  return table == nullptr ? 0 : table->max_positions;
}

extern "C" emel_error_type emelk_kv_qkv_rope_append(
    const emelk_kv_geometry *g, void *k_pool, void *v_pool, int32_t layer, const float *q_in,
    float *q_out, const float *k_rows, const float *v_rows, int32_t n_seq, int32_t n_tokens,
    const int32_t *positions, const uint16_t *block_tables, int32_t table_stride,
    const emelk_rope_table *rope, const float *q_norm, const float *k_norm, int32_t v_rms,
    float rms_epsilon, void *stream) {
  emelk::pool_layout L;
  if (emelk::make_pool_layout(g, L) != EMELK_ERR_NONE || k_pool == nullptr || v_pool == nullptr ||
      q_in == nullptr || q_out == nullptr || k_rows == nullptr || v_rows == nullptr ||
      positions == nullptr || block_tables == nullptr || rope == nullptr || layer < 0 ||
      layer >= L.n_layer || n_seq < 0 || n_tokens < 0 || table_stride <= 0 ||
      rope->head_dim != L.head_dim || !std::isfinite(rms_epsilon) ||
      static_cast<int64_t>(n_seq) * n_tokens > 0x7FFFFFFF) {
    return EMELK_ERR_INVALID_REQUEST;
  }
  if (n_seq == 0 || n_tokens == 0) return EMELK_ERR_NONE;
  emelk::rope_append_args A;
  A.L = L;
  A.k_pool = static_cast<uint8_t *>(k_pool);
  A.v_pool = static_cast<uint8_t *>(v_pool);
  A.layer = layer;
  A.q_in = q_in;
  A.q_out = q_out;
  A.k_rows = k_rows;
  A.v_rows = v_rows;
  A.n_seq = n_seq;
  A.n_tokens = n_tokens;
  A.positions = positions;
  A.tables = block_tables;
  A.table_stride = table_stride;
  A.rope = rope->dev;
  A.rope_positions = rope->max_positions;
  A.pair_count = rope->pair_count;
  A.x0_stride = rope->params.x0_stride;
  A.x1_stride = rope->params.x1_stride;
  A.x1_base = rope->x1_base;
  A.q_norm = q_norm;
  A.k_norm = k_norm;
  A.v_rms = v_rms;
  A.eps = rms_epsilon;
  A.pairing = A.pair_count == 0 ? emelk::k_pairs_none
              : A.x0_stride == 2 && A.x1_stride == 2 && A.x1_base == 1 ? emelk::k_pairs_adjacent
              : A.x0_stride == 1 && A.x1_stride == 1 && A.x1_base == L.head_dim / 2 &&
                      A.pair_count == L.head_dim / 2
                  ? emelk::k_pairs_halves
                  : emelk::k_pairs_general;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool ok = L.head_dim == 64    ? emelk::launch_rope<64>(A, st)
                  : L.head_dim == 128 ? emelk::launch_rope<128>(A, st)
                  : L.head_dim == 256 ? emelk::launch_rope<256>(A, st)
                                      : emelk::launch_rope<512>(A, st);
  return ok ? EMELK_ERR_NONE : EMELK_ERR_BACKEND;
}
