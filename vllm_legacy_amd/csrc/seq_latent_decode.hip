// Attention over a cached latent for single rows (decode steps) of 16-bit models: what
// latent_attention_tile_kernel (seq_latent_attention.hip) computes, where every sequence brings one row.
//
// Bound by HBM: each cache row is read once and is key and value of every head.  What the kernel is
// built for is to keep reads on their way:
//   * A workgroup's waves, two for 16 heads and four for 32, bring tiles of 16 rows by LDS-DMA into a ring of four: three
//     are under way while one is worked on, one barrier a tile, no staging registers; a CU holds two workgroups and up to
//     147 KB of rows.
//     Both waves of a set of 16 heads form all scores of a tile (the matrix cores have the time) and each half of the
//     latent sums, which leaves room for the queries in registers and nothing to join between the waves.
//   * The keys of all sequences are one line of tiles that the workgroups share out evenly, whatever
//     the lengths: a range may end inside a sequence and go on in the next.  The lengths are read on the
//     device, so a captured step may be replayed with others.  A part of a sequence leaves its sums in scratch for
//     latent_decode_merge_kernel or latent_decode_up_kernel; one that lies within a range is written out at once.
// Products on 16x16 MFMAs, lane = (g, c) = (lane >> 4, lane & 15), 16 heads to a workgroup:
//   S^T = K q^T    A = K    lane: key c, dims 32 ks + 8 g .. + 7     (LDS, 16 bytes)
//                  B = q^T  lane: head c, the same dims              (registers, loaded once a sequence)
//                  C        lane: head c, keys 4 g .. 4 g + 3
//   O^T = C^T P^T  B = P^T  lane: head c, keys 4 g .. + 3: where they lie
//                  A = C^T  lane: latent dim 16 n + c of the same keys (one transposing read of the row-major tile)
// Scores, max / sum (base 2) and accumulators are fp32; a weight enters the second product as the sum of two 16-bit
// numbers (its rounding and the rounding of what the rounding lost): the matrix cores have the time.
// 64 sequences of 4096 keys, rank 512 + 64: 61 us (4.9 TB/s) and 6 for the merge, of 1 .. 4001 keys 37 and 6; the tile
// kernel and its merge 137 and 116.  32 heads: 73 us (with 16 heads to a workgroup 101: the rows are read twice).  Each wave
// with keys and tiles of its own: 68 (the sums of 512 dims beside the queries leave no registers for reads ahead).  Reads
// of both products go in groups ahead of the products, or each would wait out its own latency (47 instead of 37).
// A DMA instruction writes 64 lanes x 16 bytes in a row, so rows are not padded: a tile is blocks of 64 dims, [block]
// [row][8 pieces of 16 bytes], and pieces change place by the row's number, on the source's side, so that the lanes
// of either read fall into different banks.
#include <algorithm>
#include <atomic>

#include "seq_common.h"

namespace vla {
namespace seq {
namespace {

constexpr int kLdUnit = 16;                       // rows of a tile: what the line of all sequences' keys is shared out in
constexpr int kLdRing = 4;                        // tiles in LDS
// Tiles of a range, at least.  Two of them instead: one sequence of 4096 keys 23 us instead of 19; eight of 4096 the same.
constexpr int kLdMinUnits = 4;
// Keys up to which every sequence stays with one workgroup (and set of heads) and there is no merge: this many; two for
// each workgroup that there is, up to kLdWholeMost; and two for each sequence, divided by its sets of heads (which read the
// same rows at different times then).  Sharing out costs the merge, a part more per workgroup and a walk over all lengths
// in every wave, and where the workgroups are many they are even without it.  us of the layer's attention (product, kernels
// and up-projection), one workgroup / shared out:
//   1 sequence of 130 keys 14 / 18, of 250 21 / 18
//   16 heads: 64 of 200 33 / 34, of 260 37 / 35; 128 of 260 39 / 40, of 400 49 / 43; 256 of 400 51 / 55, of 700 72 / 68; 512 of 700
//   110 / 118, of 2000 261 / 262, of 1 .. 2000 205 / 191; 4096 of 1 .. 200 255 / 513
//   32: 2048 of 1 .. 400 262 / 429, of 1 .. 2000 791 / 852; 64: 1024 of 1 .. 1000 491 / 512, of 1 .. 4000 1291 / 1196
//   128: 64 of 400 66 / 73; 512 of 500 441 / 413, of 1 .. 500 312 / 363, of 1 .. 2000 834 / 692; 2048 of 1 .. 1000 1646 / 1892
constexpr int kLdWhole = 192, kLdWholeEach = 2, kLdWholeMost = 512;
constexpr int kLdRanges = 512;                    // two workgroups to a CU
constexpr int kLdSlots = 1024;                    // rows looked up ahead

typedef short ld_s16x4 __attribute__((ext_vector_type(4)));
typedef ld_s16x4 __attribute__((address_space(3))) * ld_lds_s16x4;

template <class S>
struct LdMma;
template <>
struct LdMma<BF16> {
  static __device__ __forceinline__ f32x4 score(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 sum(ld_s16x4 a, ld_s16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
  }
};
template <>
struct LdMma<F16> {
  static __device__ __forceinline__ f32x4 score(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 sum(ld_s16x4 a, ld_s16x4 b, f32x4 c) {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h4, a), __builtin_bit_cast(h4, b), c, 0, 0, 0);
  }
};

struct LatentDecode {
  void* out;
  int64_t out_token_stride, out_head_stride;
  const void* q_lat;
  int64_t lat_token_stride, lat_head_stride;
  const void* q_rot;
  int64_t rot_token_stride, rot_head_stride;
  const void* cache;
  const int* block_tables;
  const int* query_start_loc;
  const int* context_lens;
  const void* gate;
  int64_t gate_stride;
  const float* sinks;
  float* parts;                // [2 * ranges][heads][rank + 4]: sums, then max and sum of weights
  int max_blocks, num_seqs, heads, rank, block_size, num_blocks, window, ranges, by_sequence;
  float scale;
};

// the keys that the row of sequence b sees, and the first of them (0 keys: the sequence has no row)
__device__ __forceinline__ int keys_of(const LatentDecode& a, int b, int& first) {
  const int p = a.context_lens[b];
  first = a.window > 0 ? max(0, p - a.window + 1) : 0;
  return a.query_start_loc[b + 1] > a.query_start_loc[b] ? max(0, p + 1 - first) : 0;
}
__device__ __forceinline__ int units_of(const LatentDecode& a, int b) {
  int first;
  return b < a.num_seqs ? (keys_of(a, b, first) + kLdUnit - 1) / kLdUnit : 0;
}
__device__ __forceinline__ int wave_scan(int v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const int o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  return v;
}
// all sequences' units and a range's share of them (every wave for itself)
__device__ __forceinline__ int units_in_all(const LatentDecode& a, int lane) {
  int mine = 0;
  for (int b = lane; b < a.num_seqs; b += 64) mine += units_of(a, b);
#pragma unroll
  for (int d = 32; d > 0; d /= 2) mine += __shfl_xor(mine, d, 64);
  return __builtin_amdgcn_readfirstlane(mine);
}
__device__ __forceinline__ int share_of(const LatentDecode& a, int total) {
  return max((total + a.ranges - 1) / a.ranges, kLdMinUnits);
}

__device__ __forceinline__ void ld_dma16(const void* src, uint32_t lds_at) {
  unsigned keep;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
      : "=&s"(keep)
      : "v"(src), "s"(lds_at)
      : "memory");
}
// all DMA but the N youngest instructions has landed
template <int N>
__device__ __forceinline__ void ld_landed() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// all DMA but that of `later` tiles (at most two) of N instructions each
template <int N>
__device__ __forceinline__ void ld_landed_but(int later) {
  if (later >= 2)
    ld_landed<2 * N>();
  else if (later == 1)
    ld_landed<N>();
  else
    ld_landed<0>();
}
// by how much the pieces of row r change place: distinct for eight rows in a row (the first product's read), and in
// pairs of pieces for four rows from a multiple of four on (the second's)
__device__ __forceinline__ int ld_turn(int r) { return ((r & 3) << 1) | ((r >> 2) & 1); }

template <class S, int LB, int RB, int HS>      // blocks of 64 latent dims and of the rotated part, sets of 16 heads
__global__ __launch_bounds__(128 * HS, 2) void latent_decode_kernel(LatentDecode a) {
  using T = typename S::T;
  using M = LdMma<S>;
  constexpr int NB = LB + RB;                    // blocks of a row
  constexpr int KS = 2 * NB;                     // steps of the first product
  constexpr int ND = 2 * LB;                     // blocks of 16 dims of the second, of each wave
  constexpr int ROW = 128 * NB;                  // bytes
  constexpr int TILE = kLdUnit * ROW;
  constexpr int C = 64 * LB;
  constexpr int W = 2 * HS;                      // waves
  constexpr int NI = TILE / 1024;                // DMA instructions of a tile: wave w gives w, w + W, ..
  extern __shared__ __align__(16) unsigned char smem[];
  int* slots_lds = reinterpret_cast<int*>(smem + kLdRing * TILE);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int half = w & 1;                                  // of the latent dims
  const int range = blockIdx.x, h = (blockIdx.y * HS + (w >> 1)) * 16 + c;
  const bool has_head = h < a.heads;
  int b = range, u = 0, u_end = a.by_sequence ? units_of(a, range) : 0, start = 0;
  if (!a.by_sequence) {
    const int total = units_in_all(a, lane), share = share_of(a, total);
    u = range * share;
    u_end = min(total, u + share);
  }
  if (u >= u_end) return;
  // the sequence that unit u lies in, and the units ahead of it
  for (int b0 = 0; !a.by_sequence; b0 += 64) {
    const int n = units_of(a, b0 + lane), up_to = start + wave_scan(n, lane);
    const unsigned long long behind = __ballot(up_to > u);
    if (behind) {
      const int at = __builtin_ctzll(behind);
      b = b0 + at;
      start = __shfl(up_to - n, at, 64);
      break;
    }
    start = __shfl(up_to, 63, 64);
  }
  b = __builtin_amdgcn_readfirstlane(b);
  start = __builtin_amdgcn_readfirstlane(start);
  const float scale2 = a.scale * 1.4426950408889634f;    // scores in base 2
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)smem;
  const int piece = 16 * ((lane & 7) ^ ld_turn(lane >> 3));
  const int key_at = c * 128, key_turn = ld_turn(c);
  const int vrow = 4 * g + (c >> 2), vturn = ld_turn(vrow);

  for (; u < u_end; ++b) {
    int first;
    const int keys = keys_of(a, b, first), units = (keys + kLdUnit - 1) / kLdUnit;
    if (units == 0) continue;
    const int seg_end = min(u_end, start + units);
    const int k_begin = (u - start) * kLdUnit, k_end = min(keys, (seg_end - start) * kLdUnit);
    const bool from_start = u == start, whole = from_start && seg_end == start + units;
    const int64_t t = a.query_start_loc[b];
    const int* table = a.block_tables + (int64_t)b * a.max_blocks;

    u32x4 qf[KS];
    {
      const int hq = min(h, a.heads - 1);
      const T* lat = (const T*)a.q_lat + t * a.lat_token_stride + hq * a.lat_head_stride + 8 * g;
      const T* rot = (const T*)a.q_rot + t * a.rot_token_stride + hq * a.rot_head_stride + 8 * g;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        qf[ks] = *reinterpret_cast<const u32x4*>(ks < 2 * LB ? lat + 32 * ks : rot + 32 * (ks - 2 * LB));
    }
    f32x4 o[ND];
#pragma unroll
    for (int n = 0; n < ND; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    if (a.sinks != nullptr && from_start && has_head) {     // the denominator's first term, counted once
      m = a.sinks[h] * 1.4426950408889634f;
      l = g == 0 ? 1.f : 0.f;
    }
    for (int k0 = k_begin; k0 < k_end; k0 += kLdSlots) {
      const int n_keys = min(kLdSlots, k_end - k0);
      __syncthreads();                                   // nobody reads the rows' places or tiles of before
      for (int i = tid; i < n_keys; i += 64 * W) {
        const int j = first + k0 + i, jb = j / a.block_size;
        const int blk = table[jb];                       // an id outside the pool reads block 0
        slots_lds[i] = ((unsigned)blk < (unsigned)a.num_blocks ? blk : 0) * a.block_size + (j - jb * a.block_size);
      }
      __syncthreads();
      __builtin_amdgcn_s_waitcnt(0x0f70);                // vmcnt(0): the loop counts DMA only
      // rows behind the end: the last key again (not used: see below)
      auto bring = [&](int i) {
        const uint32_t slot = (uint32_t)slots_lds[min(kLdUnit * i + 8 * half + (lane >> 3), n_keys - 1)];
        const unsigned char* src = (const unsigned char*)a.cache + (uint64_t)slot * ROW + piece;
        const uint32_t to = lds0 + (i & (kLdRing - 1)) * TILE;
#pragma unroll
        for (int u = 0; u < NI; u += W)
          if (u + w < NI) ld_dma16(src + 128 * ((u + w) >> 1), to + 1024 * (u + w));
      };
      const int tiles = (n_keys + kLdUnit - 1) / kLdUnit;
      for (int i = 0; i < kLdRing - 1 && i < tiles; ++i) bring(i);
      for (int i = 0; i < tiles; ++i) {
        const int later = min(kLdRing - 2, tiles - 1 - i);     // tiles that are under way behind this one
        constexpr int MOST = (NI + W - 1) / W;
        if (NI % W == 0 || w < NI % W)
          ld_landed_but<MOST>(later);
        else
          ld_landed_but<MOST - 1>(later);
        unsigned char* tile = smem + (i & (kLdRing - 1)) * TILE;
        const int live = n_keys - kLdUnit * i;           // rows of the tile that are keys
        if (live < kLdUnit) {
          // no product with what lies behind the sequence's end: a zero weight times infinity is not zero
          if (8 * half + (lane >> 3) >= live) {
#pragma unroll
            for (int u = 0; u < NI; u += W)
              if (u + w < NI) *reinterpret_cast<u32x4*>(tile + 1024 * (u + w) + 16 * lane) = u32x4{0u, 0u, 0u, 0u};
          }
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        __builtin_amdgcn_s_barrier();                    // the tile is here; the one before it is done with
        asm volatile("" ::: "memory");
        if (i + kLdRing - 1 < tiles) bring(i + kLdRing - 1);
        f32x4 st[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        // reads in groups, so that a group's latency passes once and under the products of the one before
        constexpr int SG = 6;
        u32x4 ka[2][SG];
        auto read_keys = [&](int i) {
#pragma unroll
          for (int x = 0; x < SG; ++x)
            if (SG * i + x < KS) {
              const int ks = SG * i + x;
              ka[i & 1][x] = *reinterpret_cast<const u32x4*>(tile + 2048 * (ks >> 1) + key_at + 16 * ((4 * (ks & 1) + g) ^ key_turn));
            }
        };
        read_keys(0);
#pragma unroll
        for (int i = 0; SG * i < KS; ++i) {
          read_keys(i + 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int x = 0; x < SG; ++x)
            if (SG * i + x < KS) st[x & 1] = M::score(ka[i & 1][x], qf[SG * i + x], st[x & 1]);
          __builtin_amdgcn_sched_barrier(0);
        }
        float s[4], mt = -INFINITY;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = (st[0][e] + st[1][e]) * scale2;
          s[e] = 4 * g + e < live ? v : -INFINITY;
          mt = fmaxf(mt, s[e]);
        }
        mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        const float m_new = fmaxf(m, mt);
        const float corr = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
        float psum = 0.f;
        ld_s16x4 hi, low;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // a score that is not a number stays one, also where the tile has no other and m_new is -infinity
          const float pv = s[e] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s[e] - m_new);
          psum += pv;
          const T rounded = S::from_f32(pv);
          hi[e] = __builtin_bit_cast(short, rounded);
          low[e] = __builtin_bit_cast(short, S::from_f32(pv - S::to_f32(rounded)));
        }
        l = l * corr + psum;
        m = m_new;
        if (__any(corr != 1.f)) {
#pragma unroll
          for (int n = 0; n < ND; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[n][e] *= corr;
        }
        constexpr int VG = 8;
        ld_s16x4 va[2][VG];
        auto read_values = [&](int i) {
#pragma unroll
          for (int x = 0; x < VG; ++x)
            if (VG * i + x < ND) {
              const int n = half * ND + VG * i + x;
              va[i & 1][x] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                  (ld_lds_s16x4)(tile + 2048 * (n >> 2) + 128 * vrow + 16 * ((2 * (n & 3) + ((c >> 1) & 1)) ^ vturn) + 8 * (c & 1)));
            }
        };
        read_values(0);
#pragma unroll
        for (int i = 0; VG * i < ND; ++i) {
          read_values(i + 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int x = 0; x < VG; ++x) o[VG * i + x] = M::sum(va[i & 1][x], hi, o[VG * i + x]);
#pragma unroll
          for (int x = 0; x < VG; ++x) o[VG * i + x] = M::sum(va[i & 1][x], low, o[VG * i + x]);
          __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("" ::: "memory");
      }
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    float inv = 1.f / l;
    if (a.gate != nullptr && has_head) inv /= 1.f + expf(-S::to_f32(((const T*)a.gate)[t * a.gate_stride + h]));
    float* part = a.parts + ((int64_t)(2 * range + (from_start ? 1 : 0)) * a.heads + h) * (C + 4);
    T* row = (T*)a.out + t * a.out_token_stride + h * a.out_head_stride;
    if (has_head) {
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        const int d = 16 * (half * ND + n) + 4 * g;
        if (whole) {
          const u32x2 packed = {pack16<S>(o[n][0] * inv, o[n][1] * inv), pack16<S>(o[n][2] * inv, o[n][3] * inv)};
          *reinterpret_cast<u32x2*>(row + d) = packed;
        } else {
          *reinterpret_cast<f32x4*>(part + d) = o[n];
        }
      }
      if (!whole && half == 0 && g == 0) {
        part[C] = m;
        part[C + 1] = l;
      }
    }
    u = seg_end;
    start += units;
  }
}

// The first unit of sequence b in the line of all, and a range's share; the same in every lane, which all come here.
__device__ __forceinline__ void place_of(const LatentDecode& a, int b, int& start, int& share) {
  int total = 0;
  start = 0;
  for (int i = threadIdx.x & 63; i < a.num_seqs; i += 64) {
    const int n = units_of(a, i);
    total += n;
    if (i < b) start += n;
  }
#pragma unroll
  for (int x = 32; x > 0; x /= 2) {
    total += __shfl_xor(total, x, 64);
    start += __shfl_xor(start, x, 64);
  }
  share = share_of(a, total);
}

// sum_s o_s[d] 2^(m_s - M) over the ranges s = i0 .. i1, M the largest m_s, of four sums from d + 256 j on each; the
// result is sum_s l_s 2^(m_s - M)
// EARLY: the first eight parts are asked for with their maxima, where there are registers for that.
template <int NJ, bool EARLY>
__device__ __forceinline__ float merge_parts(const LatentDecode& a, int h, int i0, int i1, int d, f32x4 (&num)[NJ]) {
  const int lane = threadIdx.x & 63, row_floats = a.rank + 4;
  auto part = [&](int s) {
    const int slot = s == i0 ? 2 * s + 1 : 2 * s;        // its first part is the last of that range
    return a.parts + ((int64_t)slot * a.heads + h) * row_floats;
  };
  constexpr int AHEAD = EARLY ? 8 : 4;                   // (where workgroups are many, sequences have few parts)
  f32x4 v[AHEAD][NJ];
  auto fetch = [&](int s0, int n, int s8) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
#pragma unroll
      for (int j = 0; j < NJ; ++j) v[s][j] = *reinterpret_cast<const f32x4*>(part(s0 + min(s8 + s, n - 1)) + d + 256 * j);
  };
  float ms = 0.f, ls = 0.f, big = -INFINITY;
  if (EARLY) {
    const int at = min(i0 + lane, i1);
    ms = part(at)[a.rank];
    ls = part(at)[a.rank + 1];
    fetch(i0, min(64, i1 - i0 + 1), 0);
    big = i0 + lane <= i1 ? ms : -INFINITY;
  }
  for (int s = i0 + (EARLY ? 64 : 0) + lane; s <= i1; s += 64) big = fmaxf(big, part(s)[a.rank]);
  big = wave_max(big);
  float den = 0.f;
#pragma unroll
  for (int j = 0; j < NJ; ++j) num[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = i0; s0 <= i1; s0 += 64) {
    const int n = min(64, i1 - s0 + 1);
    if (!EARLY || s0 > i0) {
      ms = part(min(s0 + lane, i1))[a.rank];
      ls = part(min(s0 + lane, i1))[a.rank + 1];
    }
    const float f = lane >= n || ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms - big);
    den += wave_sum(lane < n ? ls * f : 0.f);
    for (int s8 = 0; s8 < n; s8 += AHEAD) {              // several parts on their way
      if (!EARLY || s8 > 0 || s0 > i0) fetch(s0, n, s8);
#pragma unroll
      for (int s = 0; s < AHEAD; ++s) {
        const float fs = s8 + s < n ? __shfl(f, s8 + s, 64) : 0.f;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) num[j][e] = s8 + s < n ? num[j][e] + v[s][j][e] * fs : num[j][e];
      }
    }
  }
  return den;
}
template <class S>
__device__ __forceinline__ float gate_of(const LatentDecode& a, int64_t t, int h) {
  return a.gate != nullptr ? 1.f / (1.f + expf(-S::to_f32(((const typename S::T*)a.gate)[t * a.gate_stride + h]))) : 1.f;
}

// out[t, h, d] = the merged sums over the merged weights, times the gate.  rank / 4 threads to a head; a sequence that
// lies within one range is written out already.
template <class S>
__global__ __launch_bounds__(128) void latent_decode_merge_kernel(LatentDecode a) {
  using T = typename S::T;
  const int b = blockIdx.x, per = a.rank / 4, h = blockIdx.y * (128 / per) + threadIdx.x / per, d = 4 * (threadIdx.x % per);
  int start, share;
  place_of(a, b, start, share);
  const int units = units_of(a, b), i0 = start / share, i1 = (start + units - 1) / share;
  if (units == 0 || i0 == i1 || h >= a.heads) return;
  const int64_t t = a.query_start_loc[b];
  f32x4 num[1];
  const float den = merge_parts<1, true>(a, h, i0, i1, d, num);
  const float gv = gate_of<S>(a, t, h);
  const u32x2 packed = {pack16<S>(num[0][0] / den * gv, num[0][1] / den * gv), pack16<S>(num[0][2] / den * gv, num[0][3] / den * gv)};
  *reinterpret_cast<u32x2*>((T*)a.out + t * a.out_token_stride + h * a.out_head_stride + d) = packed;
}

// The merge and the heads' up-projection in one: up[t, h vdim + n] = sum_d o[t, h, d] w[h, d, n], o rounded to 16 bits as
// the merge leaves it.  A workgroup is 8 or 16 sequences and a head: a wave merges a row (or reads one that is written out
// already) into LDS, then takes 32 columns and a part of the latent dims.  The weights' rows run along n, where the
// matrix cores want them along d: a lane loads two columns of eight rows and puts the words together itself.  64
// sequences of 1 .. 4001 keys, 16 heads, rank 512, vdim 128: 10 us, where the merge, a batched library product and
// the copy that puts a token's heads side by side took 6, 10 and 4.
struct LatentUp {
  void* up;
  int64_t up_stride;
  const void* w;                       // [heads, rank, vdim]
  int vdim;
};
template <class S, int NJ, int ROWS>   // rank = 256 NJ
__global__ __launch_bounds__(64 * ROWS) void latent_decode_up_kernel(LatentDecode a, LatentUp u) {
  using T = typename S::T;
  constexpr int C = 256 * NJ, PITCH = C + 8;
  __shared__ __align__(16) T o_lds[ROWS * PITCH];
  __shared__ float part[ROWS][ROWS][34];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c = lane & 15;
  const int b0 = ROWS * blockIdx.x, h = blockIdx.y;
  const int blocks = u.vdim / 32, split = min(ROWS / blocks, C / 32), nb = w % blocks, ks0 = min(w / blocks, split - 1) * (C / 32 / split);
  const uint32_t* wr = reinterpret_cast<const uint32_t*>((const T*)u.w + ((int64_t)h * C + 32 * ks0 + 8 * g) * u.vdim + 32 * nb + 2 * c);
  constexpr int AHEAD = 4;                               // steps whose weights are on their way during the merge
  const int steps = C / 32 / split;
  uint32_t x[AHEAD][8];
#pragma unroll
  for (int ks = 0; ks < AHEAD; ++ks)
#pragma unroll
    for (int j = 0; j < 8; ++j) x[ks][j] = wr[(int64_t)(32 * min(ks, steps - 1) + j) * (u.vdim / 2)];
  int start = 0, share = 1;
  const bool parts = !a.by_sequence && a.ranges > 1;
  if (parts) place_of(a, b0 + w, start, share);
  {
    const int row = w, b = b0 + row;
    u32x2 packed[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) packed[j] = u32x2{0u, 0u};
    if (b < a.num_seqs && a.query_start_loc[b + 1] > a.query_start_loc[b]) {
      const int64_t t = a.query_start_loc[b];
      const int units = units_of(a, b), i0 = start / share, i1 = (start + units - 1) / share;
      if (parts && i0 != i1) {
        f32x4 num[NJ];
        const float den = merge_parts<NJ, ROWS == 8>(a, h, i0, i1, 4 * lane, num);
        const float gv = gate_of<S>(a, t, h);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          packed[j] = u32x2{pack16<S>(num[j][0] / den * gv, num[j][1] / den * gv), pack16<S>(num[j][2] / den * gv, num[j][3] / den * gv)};
      } else {
        const T* from = (const T*)a.out + t * a.out_token_stride + h * a.out_head_stride + 4 * lane;
#pragma unroll
        for (int j = 0; j < NJ; ++j) packed[j] = *reinterpret_cast<const u32x2*>(from + 256 * j);
      }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) *reinterpret_cast<u32x2*>(o_lds + row * PITCH + 256 * j + 4 * lane) = packed[j];
  }
  __syncthreads();
  f32x4 even = {0.f, 0.f, 0.f, 0.f}, odd = {0.f, 0.f, 0.f, 0.f};
  for (int k8 = 0; k8 < steps; k8 += AHEAD) {
#pragma unroll
    for (int ks = 0; ks < AHEAD; ++ks) {
      if (k8 + ks >= steps) break;
      const u32x4 ov = *reinterpret_cast<const u32x4*>(o_lds + c % ROWS * PITCH + 32 * (ks0 + k8 + ks) + 8 * g);
      u32x4 lo, hi;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        lo[j] = __builtin_amdgcn_perm(x[ks][2 * j + 1], x[ks][2 * j], 0x05040100);
        hi[j] = __builtin_amdgcn_perm(x[ks][2 * j + 1], x[ks][2 * j], 0x07060302);
      }
      even = LdMma<S>::score(ov, lo, even);
      odd = LdMma<S>::score(ov, hi, odd);
    }
    if (k8 + AHEAD < steps) {
#pragma unroll
      for (int ks = 0; ks < AHEAD; ++ks)
#pragma unroll
        for (int j = 0; j < 8; ++j) x[ks][j] = wr[(int64_t)(32 * min(k8 + AHEAD + ks, steps - 1) + j) * (u.vdim / 2)];
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (4 * g + i < ROWS) part[w][4 * g + i][2 * c] = even[i], part[w][4 * g + i][2 * c + 1] = odd[i];
  __syncthreads();
  for (int i = tid; i < ROWS * u.vdim / 2; i += 64 * ROWS) {
    const int row = i / (u.vdim / 2), n = 2 * (i % (u.vdim / 2)), b = b0 + row;
    if (b >= a.num_seqs || a.query_start_loc[b + 1] <= a.query_start_loc[b]) continue;
    float v0 = 0.f, v1 = 0.f;
    for (int s = 0; s < split; ++s) v0 += part[s * blocks + n / 32][row][n % 32], v1 += part[s * blocks + n / 32][row][n % 32 + 1];
    *reinterpret_cast<uint32_t*>((T*)u.up + a.query_start_loc[b] * u.up_stride + (int64_t)h * u.vdim + n) = pack16<S>(v0, v1);
  }
}

bool latent_decode_sizes(int rank, int rot) {
  return (rank == 256 || rank == 512) && (rot == 0 || rot == 64);
}
// workgroups per range: 16 heads each up to 16, 32 beyond
int head_groups(int heads) { return heads <= 16 ? 1 : (heads + 31) / 32; }

template <class S, int LB, int RB, int HS>
int launch_latent_decode(const LatentDecode& a, const LatentUp* up, hipStream_t stream) {
  constexpr size_t lds = kLdRing * kLdUnit * 128 * (LB + RB) + kLdSlots * 4;
  static std::atomic<bool> allowed{false};         // raised once per kernel, not per launch
  if (lds > 64 * 1024 && !allowed.load(std::memory_order_relaxed)) {
    VLA_SEQ_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_decode_kernel<S, LB, RB, HS>),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    allowed.store(true, std::memory_order_relaxed);
  }
  latent_decode_kernel<S, LB, RB, HS><<<dim3(a.ranges, head_groups(a.heads)), 128 * HS, lds, stream>>>(a);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  if (up != nullptr) {
    // Eight sequences to a workgroup while that leaves one for each CU at most: more of them, and registers for the first parts
    // ahead of their maxima (16 heads: 64 of 1 .. 4001 keys 9.8 us instead of 11.9, of 4000 10.4 and 13.4, one of 4000 10.7 and
    // 11.7); sixteen beyond, where weights would be read twice as often (256 of 1000 11.9, with eight 17.1; 1024 of 100 19 and 31).
    // Half the waves also take twice the steps each, which only merging outweighs where they are more than are asked for ahead:
    // with eight and with sixteen, whole sequences of 100 keys, rank 512, vdim 128 7.2 and 5.1 (32 heads, 64 sequences), 256 13.2
    // and 8.0 (128 heads, 16); vdim 64 the call of 64 sequences of 16 heads 13.9 and 14.8 (rank 256).  In parts, vdim 256, the call
    // of 32 heads, 16 sequences of 4000, 46.1 and 53.1, of 64 of 1 .. 1000 46.5 and 45.7.
    const int64_t eights = (int64_t)((a.num_seqs + 7) / 8) * a.heads;
    const bool whole = a.by_sequence || a.ranges <= 1;
    if (whole ? eights <= 256 && a.rank * up->vdim <= 512 * 64 : eights <= (up->vdim <= 128 ? 256 : 128))
      latent_decode_up_kernel<S, LB / 4, 8><<<dim3((a.num_seqs + 7) / 8, a.heads), 512, 0, stream>>>(a, *up);
    else
      latent_decode_up_kernel<S, LB / 4, 16><<<dim3((a.num_seqs + 15) / 16, a.heads), 1024, 0, stream>>>(a, *up);
    VLA_SEQ_HIP_CHECK(hipGetLastError());
  } else if (!a.by_sequence && a.ranges > 1) {
    const int heads_per = 128 / (a.rank / 4);
    latent_decode_merge_kernel<S><<<dim3(a.num_seqs, (a.heads + heads_per - 1) / heads_per), 128, 0, stream>>>(a);
    VLA_SEQ_HIP_CHECK(hipGetLastError());
  }
  return VLA_OK;
}

template <class S>
int latent_decode_go(const LatentDecode& a, const LatentUp* up, int rot, hipStream_t stream) {
  const bool wide = a.rank == 512, turned = rot == 64;
  const bool two = a.heads > 16;
#define VLA_LD(L, R) return two ? launch_latent_decode<S, L, R, 2>(a, up, stream) : launch_latent_decode<S, L, R, 1>(a, up, stream)
  if (wide && turned) VLA_LD(8, 1);
  if (wide) VLA_LD(8, 0);
  if (turned) VLA_LD(4, 1);
  VLA_LD(4, 0);
#undef VLA_LD
}

}  // namespace
}  // namespace seq
}  // namespace vla

using namespace vla;
using namespace vla::seq;

extern "C" int vla_seq_latent_decode_supported(int rank, int rot, int dtype) {
  return (dtype == VLA_F16 || dtype == VLA_BF16) && latent_decode_sizes(rank, rot) &&
         vla_seq_latent_attention_tiles_supported(rank, rot, dtype);
}

extern "C" int vla_seq_latent_decode_ranges(int num_seqs, int max_keys, int heads) {
  if (num_seqs <= 0 || heads <= 0) return 0;
  const int64_t sets = head_groups(heads), each = (int64_t)kLdWholeEach * num_seqs;
  if (max_keys <= std::max<int64_t>({kLdWhole, each / sets, std::min<int64_t>(each * sets, kLdWholeMost)})) return 0;
  const int64_t units = (int64_t)num_seqs * ((max_keys + kLdUnit - 1) / kLdUnit);
  const int64_t most = kLdRanges / head_groups(heads) > 1 ? kLdRanges / head_groups(heads) : 1;
  const int64_t want = (units + kLdMinUnits - 1) / kLdMinUnits;
  return (int)(want < most ? want : most);
}

extern "C" int64_t vla_seq_latent_decode_scratch_floats(int ranges, int heads, int rank) {
  return ranges > 1 ? (int64_t)2 * ranges * heads * (rank + 4) : 0;
}

namespace {
int latent_decode(void* out, int64_t out_token_stride, int64_t out_head_stride, const void* q_lat,
                  int64_t lat_token_stride, int64_t lat_head_stride, const void* q_rot,
                  int64_t rot_token_stride, int64_t rot_head_stride, const void* cache,
                  const int* block_tables, int max_blocks, const int* query_start_loc,
                  const int* context_lens, int num_seqs, int heads, int rank, int rot,
                  int block_size, int num_blocks, float scale, int ranges, float* scratch,
                  int64_t scratch_floats, int dtype, int window, const void* gate,
                  int64_t gate_stride, const float* sinks, void* stream, const LatentUp* up) {
  if (num_seqs == 0) return VLA_OK;
  if (gate && gate_stride < heads) return VLA_ERR_ARG;
  if (!out || !q_lat || (rot > 0 && !q_rot) || !cache || !block_tables || !query_start_loc || !context_lens ||
      num_seqs < 0 || heads <= 0 || heads > 65535 || rot < 0 || block_size <= 0 || num_blocks <= 0 ||
      (int64_t)num_blocks * block_size > 0x7fffffff || max_blocks <= 0 || ranges < 0 || ranges > kLdRanges ||
      (ranges > 1 && (!scratch || scratch_floats < vla_seq_latent_decode_scratch_floats(ranges, heads, rank))))
    return VLA_ERR_ARG;
  if ((dtype != VLA_F16 && dtype != VLA_BF16) || !latent_decode_sizes(rank, rot)) return VLA_ERR_HEAD_SIZE;
  // 16-byte loads of query and cache rows, 8-byte stores of the output, 16-byte ones of the sums
  if (((uintptr_t)q_lat % 16) || (lat_token_stride % 8) || (lat_head_stride % 8) || ((uintptr_t)cache % 16) ||
      (rot > 0 && (((uintptr_t)q_rot % 16) || (rot_token_stride % 8) || (rot_head_stride % 8))) ||
      ((uintptr_t)out % 8) || (out_token_stride % 4) || (out_head_stride % 4) || ((uintptr_t)scratch % 16))
    return VLA_ERR_ARG;
  const LatentDecode a{out, out_token_stride, out_head_stride, q_lat, lat_token_stride, lat_head_stride, q_rot,
                       rot_token_stride, rot_head_stride, cache, block_tables, query_start_loc, context_lens, gate,
                       gate_stride, sinks, scratch, max_blocks, num_seqs, heads, rank, block_size, num_blocks, window,
                       ranges > 0 ? ranges : num_seqs, ranges == 0, scale};
  return dtype == VLA_BF16 ? latent_decode_go<BF16>(a, up, rot, (hipStream_t)stream)
                           : latent_decode_go<F16>(a, up, rot, (hipStream_t)stream);
}
}  // namespace

extern "C" int vla_seq_latent_decode(void* out, int64_t out_token_stride, int64_t out_head_stride, const void* q_lat,
                                     int64_t lat_token_stride, int64_t lat_head_stride, const void* q_rot,
                                     int64_t rot_token_stride, int64_t rot_head_stride,
                                     const void* cache, const int* block_tables, int max_blocks, const int* query_start_loc,
                                     const int* context_lens, int num_seqs, int heads, int rank, int rot, int block_size,
                                     int num_blocks, float scale, int ranges, float* scratch, int64_t scratch_floats, int dtype, int window,
                                     const void* gate, int64_t gate_stride, const float* sinks, void* stream) {
  return latent_decode(out, out_token_stride, out_head_stride, q_lat, lat_token_stride, lat_head_stride, q_rot,
                       rot_token_stride, rot_head_stride, cache, block_tables, max_blocks, query_start_loc, context_lens,
                       num_seqs, heads, rank, rot, block_size, num_blocks, scale, ranges, scratch, scratch_floats, dtype,
                       window, gate, gate_stride, sinks, stream, nullptr);
}

extern "C" int vla_seq_latent_decode_up_supported(int vdim) { return vdim == 32 || vdim == 64 || vdim == 128 || vdim == 256; }

extern "C" int vla_seq_latent_decode_up(void* out, int64_t out_token_stride, int64_t out_head_stride, const void* q_lat,
                                        int64_t lat_token_stride, int64_t lat_head_stride, const void* q_rot,
                                        int64_t rot_token_stride, int64_t rot_head_stride,
                                        const void* cache, const int* block_tables, int max_blocks, const int* query_start_loc,
                                        const int* context_lens, int num_seqs, int heads, int rank, int rot, int block_size,
                                        int num_blocks, float scale, int ranges, float* scratch, int64_t scratch_floats, int dtype, int window,
                                        const void* gate, int64_t gate_stride, const float* sinks, void* stream,
                                        const void* w, void* up, int64_t up_stride, int vdim) {
  if (!w || !up || up_stride < (int64_t)heads * vdim || up_stride % 2 || ((uintptr_t)w % 4) || ((uintptr_t)up % 4))
    return VLA_ERR_ARG;
  if (!vla_seq_latent_decode_up_supported(vdim)) return VLA_ERR_HEAD_SIZE;
  const LatentUp to{up, up_stride, w, vdim};
  return latent_decode(out, out_token_stride, out_head_stride, q_lat, lat_token_stride, lat_head_stride, q_rot,
                       rot_token_stride, rot_head_stride, cache, block_tables, max_blocks, query_start_loc, context_lens,
                       num_seqs, heads, rank, rot, block_size, num_blocks, scale, ranges, scratch, scratch_floats, dtype,
                       window, gate, gate_stride, sinks, stream, &to);
}
