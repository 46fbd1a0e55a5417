// Shared by the sources of libvla_seq_gfx950.so: dtype dispatch, block reductions, error slot.
#pragma once

#include <atomic>

#include "../../include/vla_sequence_ops.h"
#include "vla_common.h"

namespace vla {
namespace seq {

void set_hip_error(int e);

#define VLA_SEQ_HIP_CHECK(expr)          \
  do {                                   \
    hipError_t e_ = (expr);              \
    if (e_ != hipSuccess) {              \
      vla::seq::set_hip_error((int)e_);  \
      return VLA_ERR_HIP;                \
    }                                    \
  } while (0)

// calls f(S{}) with the scalar traits of a dtype code; VLA_ERR_DTYPE for an unknown code
template <class F>
inline int with_dtype(int dtype, F&& f) {
  switch (dtype) {
    case VLA_F16: return f(F16{});
    case VLA_BF16: return f(BF16{});
    case VLA_F32: return f(F32{});
    default: return VLA_ERR_DTYPE;
  }
}

// LDS of a launch of so many workgroups: where they are fewer than the CUs have room for, as much as leaves room for a CU's
// share of them.  Workgroups go where there is room: four to some CUs while others have none.  Linear recurrence, us with and
// without: 8 runs of 200 rows, 16 heads of 64 x 128, float16 (512 workgroups, room for 1024) 18 + 29 and 22 + 36; 4096 rows of
// 4 heads of 128 x 128, float32 (256, room for 512) 24 + 38 and 28 + 49.
constexpr int64_t kLdsOfCu = 160 * 1024, kLdsGrain = 1280;
inline size_t spread_lds(size_t lds, int64_t workgroups) {
  const int64_t share = (workgroups + 255) / 256;
  if (share > 8) return lds;
  const size_t least = kLdsOfCu / (share + 1) / kLdsGrain * kLdsGrain + kLdsGrain;      // share + 1 of it are more than there is
  return lds > least ? lds : least;
}
// A kernel's LDS limit, raised once on each device that launches it, to what any launch may ask for.
template <class K>
inline int raise_lds(K kernel, size_t lds, std::atomic<uint64_t>& raised) {
  if (lds <= 64 * 1024) return VLA_OK;
  int dev = 0;
  VLA_SEQ_HIP_CHECK(hipGetDevice(&dev));
  const uint64_t bit = 1ull << (dev & 63);
  if (!(raised.load(std::memory_order_relaxed) & bit)) {
    VLA_SEQ_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 120 * 1024));
    raised.fetch_or(bit, std::memory_order_relaxed);
  }
  return VLA_OK;
}
// Pieces of up to `rows` new rows of num_seqs sequences, of which the host knows the sum of the lengths, in slots
// start_b / rows + b + 0, 1, ..: no more than (tokens + seqs (rows - 1)) / rows have rows.  Where the slots are even in
// number, those without may all be one XCD's, and the others' CUs have more than their share: then all count.
inline int64_t pieces_at_most(int num_tokens, int num_seqs, int rows) {
  const int64_t slots = (int64_t)num_tokens / rows + num_seqs;
  return slots % 2 ? (num_tokens + (int64_t)num_seqs * (rows - 1)) / rows : slots;
}

// Orders one wave's LDS traffic: what its lanes wrote before is visible to what they read after.
// (The hardware keeps a wave's LDS instructions in order; the fences keep the compiler from
// moving accesses of different types across the point.)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the two 16-bit values of a packed word, and back
template <class S>
__device__ __forceinline__ float lo16(uint32_t w) {
  return S::to_f32(__builtin_bit_cast(typename S::T, (uint16_t)(w & 0xffffu)));
}
template <class S>
__device__ __forceinline__ float hi16(uint32_t w) {
  return S::to_f32(__builtin_bit_cast(typename S::T, (uint16_t)(w >> 16)));
}
template <class S>
__device__ __forceinline__ uint32_t pack16(float lo, float hi) {
  return (uint32_t)__builtin_bit_cast(uint16_t, S::from_f32(lo)) |
         ((uint32_t)__builtin_bit_cast(uint16_t, S::from_f32(hi)) << 16);
}

// (which product is fused is said here, so that the sums in 32 bits are the same in every kernel; a float16 result may still be
// rounded from them at once in one kernel and by way of 32 bits in another)
__device__ __forceinline__ void turn_by(float& a, float& b, float2 sc) {
  const float a2 = fmaf(a, sc.y, -(b * sc.x));
  b = fmaf(b, sc.y, a * sc.x);
  a = a2;
}

// i / d for i < 2048 with inverse = 65536 / d rounded up, d <= 32
__device__ __forceinline__ int quotient(int i, int inverse) { return (i * inverse) >> 16; }

// Eight neighbouring pairs of a head, as two pieces of 16 bytes: pairs side by side, or the same places of the two pieces.
struct TurnPieces {
  u32x4 x, y;
};
template <class S>
__device__ __forceinline__ TurnPieces turn_eight(TurnPieces in, const float2* sines, int interleaved) {
  TurnPieces out;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const u32x4 two = *reinterpret_cast<const u32x4*>(sines + 2 * e);
    const float2 s0 = {__builtin_bit_cast(float, (uint32_t)two[0]), __builtin_bit_cast(float, (uint32_t)two[1])};
    const float2 s1 = {__builtin_bit_cast(float, (uint32_t)two[2]), __builtin_bit_cast(float, (uint32_t)two[3])};
    const uint32_t wx = interleaved ? (e < 2 ? in.x[2 * e & 3] : in.y[2 * e & 3]) : in.x[e];
    const uint32_t wy = interleaved ? (e < 2 ? in.x[(2 * e + 1) & 3] : in.y[(2 * e + 1) & 3]) : in.y[e];
    float a0 = lo16<S>(wx), b0 = interleaved ? hi16<S>(wx) : lo16<S>(wy);
    float a1 = interleaved ? lo16<S>(wy) : hi16<S>(wx), b1 = hi16<S>(wy);
    turn_by(a0, b0, s0);
    turn_by(a1, b1, s1);
    const uint32_t u0 = pack16<S>(a0, interleaved ? b0 : a1), u1 = pack16<S>(interleaved ? a1 : b0, b1);
    if (interleaved) {
      (e < 2 ? out.x : out.y)[2 * e & 3] = u0;
      (e < 2 ? out.x : out.y)[(2 * e + 1) & 3] = u1;
    } else {
      out.x[e] = u0;
      out.y[e] = u1;
    }
  }
  return out;
}

// sum over a workgroup of up to 1024 threads; red holds 16 floats; every thread gets the sum
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  if (lane == 0) red[w] = v;
  __syncthreads();
  float r = 0.f;
  for (int i = 0; i < nw; ++i) r += red[i];
  __syncthreads();
  return r;
}

// v + the value another lane holds, the lanes paired by a DPP pattern (no LDS round trip)
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  const int other = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false);
  return v + __builtin_bit_cast(float, other);
}

// the sum over each aligned group of `split` lanes (1, 2, 4, 8 or 16), in every lane of the group:
// neighbours, pairs of a quad, the mirrored half of eight, the mirrored half of sixteen
__device__ __forceinline__ void group_sums(float& a, float& b, int split) {
  if (split > 1) {
    a = dpp_add<0xB1>(a);      // quad_perm [1, 0, 3, 2]
    b = dpp_add<0xB1>(b);
  }
  if (split > 2) {
    a = dpp_add<0x4E>(a);      // quad_perm [2, 3, 0, 1]
    b = dpp_add<0x4E>(b);
  }
  if (split > 4) {
    a = dpp_add<0x141>(a);     // row_half_mirror: lane i of eight with lane 7 - i
    b = dpp_add<0x141>(b);
  }
  if (split > 8) {
    a = dpp_add<0x140>(a);     // row_mirror: lane i of sixteen with lane 15 - i
    b = dpp_add<0x140>(b);
  }
}

// one 16x16x4 fp32 matrix-core step.  lane = (g, c) = (lane >> 4, lane & 15): A operand row c,
// contraction index g; B operand column c, contraction index g; result column c, rows 4 g .. 4 g + 3
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// four values d .. d + 3 of a row of `dim`, zeros behind its end
template <class S>
__device__ __forceinline__ f32x4 load4(const typename S::T* row, int d, int dim, bool vec) {
  f32x4 r = {0.f, 0.f, 0.f, 0.f};
  if (vec) {
    if (d < dim) {
      if constexpr (sizeof(typename S::T) == 2) {
        const u32x2 x = *reinterpret_cast<const u32x2*>(row + d);
        r = f32x4{lo16<S>(x[0]), hi16<S>(x[0]), lo16<S>(x[1]), hi16<S>(x[1])};
      } else {
        r = *reinterpret_cast<const f32x4*>(row + d);
      }
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (d + e < dim) r[e] = S::to_f32(row[d + e]);
  }
  return r;
}

// 16 bytes per lane from each lane's own address into 1 KB of LDS (no register result), where `go`: a branch that the
// compiler does not see, so that the products around it stay one block
__device__ __forceinline__ void tile_dma16(const void* src, uint32_t lds_at, int go) {
  unsigned keep;
  asm volatile(
      "s_cmp_lg_u32 %3, 0\n\ts_cbranch_scc0 1f\n\ts_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0\n1:"
      : "=&s"(keep)
      : "v"(src), "s"(lds_at), "s"(__builtin_amdgcn_readfirstlane(go))
      : "memory", "scc");
}

// the larger of a lane's value and that of the lane 32 further on
__device__ __forceinline__ float max_halves(float v) {
  const uint32_t x = __builtin_bit_cast(uint32_t, v);
  const auto both = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return fmaxf(__builtin_bit_cast(float, (uint32_t)both[0]), __builtin_bit_cast(float, (uint32_t)both[1]));
}

// the sums over a wave's first 1, 2, .. lanes, each in its last lane
__device__ __forceinline__ int wave_sums(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);      // row_shr 1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);     // row_bcast 15 to rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);     // row_bcast 31 to rows 2 and 3
  return v;
}

// the sum over a wave, in every lane
__device__ __forceinline__ int wave_total(int v) { return __builtin_amdgcn_readlane(wave_sums(v), 63); }

// the largest of a wave's values, none of them negative, in every lane
__device__ __forceinline__ int wave_most(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));
  return __builtin_amdgcn_readlane(v, 63);
}

// the first row of a sequence's cache that its new rows see
__device__ __forceinline__ int first_formed(int context, int window) { return window > 0 ? max(0, context - window + 1) : 0; }

// The `rank`-th of all tiles of 2^shift rows of a step's sequences, counted from those that walk the most keys (a
// tile's level: how many tiles of keys lie ahead of its last row).  Every wave finds it for itself: a search over
// the levels for the one whose tiles hold the rank, with the sequences in the lanes' registers.  Launching one
// workgroup per tile of the longest sequence for every sequence instead left empty ones between the real ones:
// workgroups go to the shader engines of an XCD in turn, an engine that is full holds all others up, and half the
// chip stood idle for 40 of 98 us with four prompts of 2047, 1265, 483 and 1748 rows.  A sequence has at most `most` tiles,
// so that the caller's bound on all of them holds whatever the lengths on the device are.
// kGathered: a sequence's rows context .. and the keys ahead of them that its window sees lie one behind the other among
// num_rows gathered ones (`before` of them ahead of it); those that do not end there have no tiles, nor have those
// behind them (`fitting` sequences do).
constexpr int kRankedChunks = 4;
constexpr int kRankedSeqs = kRankedChunks * kWave;
struct RankedTile {
  int all, fitting;                                    // the tiles there are; below, where the rank is one of them:
  int seq, tile;
  int first_row, rows, context, before;                // the sequence's first row, its rows and what lies ahead of them
};
template <bool kGathered>
__device__ __forceinline__ RankedTile ranked_tile(int rank, int num_seqs, const int* __restrict__ query_start_loc,
                                                  const int* __restrict__ context_lens, int shift, int most,
                                                  int window = 0, int num_rows = 0) {
  const int lane = threadIdx.x & 63, chunks = (num_seqs + kWave - 1) / kWave;
  int begin[kRankedChunks], rows[kRankedChunks], context[kRankedChunks], before[kRankedChunks];
  int first[kRankedChunks], end[kRankedChunks];       // the levels of a sequence's tiles
  RankedTile r = {0, num_seqs, 0, 0, 0, 0, 0, 0};
  if (num_seqs == 1) {                                 // its last tile is the first
    r.first_row = query_start_loc[0];
    r.rows = query_start_loc[1] - r.first_row;
    r.context = context_lens[0];
    r.all = min((max(r.rows, 0) + (1 << shift) - 1) >> shift, most);
    if (kGathered && r.context + r.rows - first_formed(r.context, window) > num_rows) r.all = r.fitting = 0;
    r.tile = r.all - 1 - rank;
    return r;
  }
#pragma unroll
  for (int k = 0; k < kRankedChunks; ++k) {
    begin[k] = rows[k] = context[k] = 0;
    const int s = k * kWave + lane;
    if (k < chunks && s < num_seqs) {
      begin[k] = query_start_loc[s];
      rows[k] = query_start_loc[s + 1];
      context[k] = context_lens[s];
    }
  }
  int top = 0, behind = 0;
  if constexpr (kGathered) r.fitting = 0;
#pragma unroll
  for (int k = 0; k < kRankedChunks; ++k) {
    before[k] = first[k] = end[k] = 0;
    if (k < chunks) {
      rows[k] -= begin[k];
      first[k] = context[k] >> shift;
      end[k] = first[k] + min((max(rows[k], 0) + (1 << shift) - 1) >> shift, most);
      if constexpr (kGathered) {
        const int keys = context[k] + rows[k] - first_formed(context[k], window), sums = wave_sums(keys);
        before[k] = behind + sums - keys;
        const bool fits = behind + sums <= num_rows;
        if (!fits) end[k] = first[k];
        r.fitting += __popcll(__ballot(fits && k * kWave + lane < num_seqs));
        behind += __builtin_amdgcn_readlane(sums, 63);
      }
      r.all += end[k] - first[k];
      top = max(top, end[k]);
    }
  }
  r.all = wave_total(r.all);
  if (r.all <= rank) return r;
  auto at_least = [&](int level) {                     // tiles of this level and above
    int n = 0;
#pragma unroll
    for (int k = 0; k < kRankedChunks; ++k)
      if (k < chunks) n += max(end[k] - max(first[k], level), 0);
    return wave_total(n);
  };
  int lo = 0, hi = wave_most(top), above = 0;      // at_least(lo) > rank >= at_least(hi) = above
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1, n = at_least(mid);
    if (n > rank) {
      lo = mid;
    } else {
      hi = mid;
      above = n;
    }
  }
  int left = rank - above;
#pragma unroll
  for (int k = 0; k < kRankedChunks; ++k)
    if (k < chunks && left >= 0) {
      const bool here = first[k] <= lo && lo < end[k];
      const uint64_t mask = __ballot(here);
      const int n = __popcll(mask);
      if (left < n) {
        const uint64_t which = __ballot(here && __popcll(mask & ((1ull << lane) - 1)) == left);
        const int l = __ffsll((unsigned long long)which) - 1;
        r.seq = k * kWave + l;
        r.tile = lo - __builtin_amdgcn_readlane(first[k], l);
        r.first_row = __builtin_amdgcn_readlane(begin[k], l);
        r.rows = __builtin_amdgcn_readlane(rows[k], l);
        r.context = __builtin_amdgcn_readlane(context[k], l);
        r.before = __builtin_amdgcn_readlane(before[k], l);
      }
      left -= n;
    }
  // (the compiler does not see that these are the same for all lanes)
  for (int* x : {&r.seq, &r.tile, &r.first_row, &r.rows, &r.context, &r.before}) *x = __builtin_amdgcn_readfirstlane(*x);
  return r;
}

__device__ __forceinline__ bool finite(float x) { return fabsf(x) <= 3.402823466e38f; }

// z / (1 + exp(-z)).  exp(-z) = 2^n 2^f with the argument's rounding in f; the quotient is the hardware reciprocal's product
// and what that leaves over, divided once more.  Error against 64 bits as that of expf and a division: 3.84e-8 (root mean
// square over -20 .. 20), 1.85e-7 at most.
template <int N>
__device__ __forceinline__ void silu(float (&v)[N]) {
#pragma clang fp contract(off)
  float top = 0.f;                                         // NaN aside, which both ways hand on
#pragma unroll
  for (int k = 0; k < N; ++k) top = fmaxf(top, fabsf(v[k]));
  if (__any(top >= 87.f)) {
    // exp(-z) beyond what the reciprocal takes, where the sum is exp(-z) alone: 2^64 of it, and the rest from the quotient's
    // exponent.  And infinity, whose remainder is not a number.
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const float y = __builtin_amdgcn_fmed3f(-v[k], -100.f, 400.f), t = 1.44269504f * y, n = __builtin_rintf(t);
      const float x = __builtin_amdgcn_exp2f((t - n) + fmaf(1.92596299e-8f, y, fmaf(1.44269504f, y, -t)));
      const bool far = v[k] < -87.f;
      const float d = far ? __builtin_amdgcn_ldexpf(x, 64) : 1.f + __builtin_amdgcn_ldexpf(x, (int)n);
      const float r = __builtin_amdgcn_rcpf(d), q = v[k] * r, w = fmaf(fmaf(-d, q, v[k]), r, q);
      v[k] = far ? __builtin_amdgcn_ldexpf(w, 64 - (int)n) : v[k] == INFINITY ? v[k] : w;
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < N; ++k) {
    // n in the low bits of a sum with 1.5 2^23, from where it is added to the exponent
    const float t = -1.44269504f * v[k], at = t + 12582912.f, n = at - 12582912.f;
    const float x = __builtin_amdgcn_exp2f((t - n) + fmaf(-1.92596299e-8f, v[k], fmaf(-1.44269504f, v[k], -t)));
    const float d = 1.f + __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) + (__builtin_bit_cast(uint32_t, at) << 23));
    const float r = __builtin_amdgcn_rcpf(d), q = v[k] * r;
    v[k] = fmaf(fmaf(-d, q, v[k]), r, q);
  }
}

__device__ __forceinline__ float softplusf(float z) { return z > 20.f ? z : log1pf(expf(z)); }

}  // namespace seq
}  // namespace vla
