// Latent attention over runs of rows with every head's keys and values formed from the cached latents.
//
// Scoring the cached latent itself costs a head 2 rank + rot numbers per (query, key) pair; a head's own
// key and value cost dim + rot + vdim, and forming them rank (dim + vdim) per key and head, once for all
// queries of the run.  A run of rows therefore gathers its visible cache rows into one place
// (latent_gather_kernel), latent_form_kernel multiplies them with the two up-projections, and
// latent_prompt_kernel below is plain causal attention with keys [formed (dim) | shared rotated part
// (rot)] and values of vdim.  4096 rows of 16 heads (128 + 64, values of 128, rank 512): 143 us under the tracer on average
// (139 to 172 from box to box; 600 TFLOP/s, 840 with the remainders' product) where latent_attention_tile_kernel takes 1685,
// plus 5 us to gather (9 with 32 rows to a workgroup instead of 8) and 31 to form keys and values (the products on the query's
// side that they replace take 46).
//
// Keys come as two 16-bit numbers, the rounded one and what rounding took.  The latent kernel rounds the query's
// side, which is the same for all keys of a row and mostly cancels in the softmax; a key's rounding is its own.
// Outputs' error against 64 bits, this / one 16-bit number / the latent kernel, bf16, 1e-3: independent latents
// 2.5 / 2.8 / 2.8, with scores four times as large 2.4 / 3.8 / 3.6 (float16: an eighth of each).  One number
// per key took 136 us when two took 184.
//
// The rows of sequence b are its keys from first_b = max(0, context - window + 1) (0 without a window) to
// its last new row; sequences follow each other, so a sequence's place is the sum of the counts before
// it, which every workgroup forms for itself (nothing has to be planned on the host or copied there).
//
// latent_prompt_kernel<S, DB, VB, LB>: a workgroup is 128 query rows of one head, 32 per wave, and walks key
// tiles of 64.  Products on 32x32x16 MFMAs in transposed form (lane = (hf, c) = (lane >> 5, lane & 31)):
//   S^T = K q^T   A = K: lane: key c, dims 16 ks + 8 hf .. + 7 (LDS);  B = q^T: query c (registers)
//   O^T = V^T P^T B = P^T: the first product's result where it lies;   A = V^T: two transposing reads
// Tiles come in by LDS-DMA, keys and values in turn (one tile of each in LDS: 56 KB), without staging registers.  A DMA
// instruction writes 64 lanes x 16 bytes in a row, so rows cannot be padded; 16-byte pieces (values:
// 64-byte ones) are exchanged within a row by the row's number instead, on the source's side, so that
// the lanes of a read fall into different banks.  DMA goes out between the products, a value tile's between the first
// ones and a key tile's ahead of and between the second ones, and weights are formed between those (184 us and bursts
// behind the barriers before).
//
// Workgroups go out longest walk first over all sequences (ranked_tile), heads next to each other.  Few of
// them (prompt_form) have two groups of four waves, a CU each, that take every other tile and join their sums at the end: with
// one group, two workgroups to a CU, all 512 of a run of 4096 rows are on the chip at once and the ones with 64 tiles
// stay alone on their CUs (165 us instead of 150; 2048 rows 70 instead of 59).  Each group rounds its weights to 16 bits against
// a maximum of its own: a row's bits differ by one rounding between steps of one form and the other (errors against 64 bits
// are the same).  Counted: matrix cores 45 %, vector instructions 38 % of a CU's busy cycles, at 2.07 GHz; within a wave a
// tile's scores, maximum, weights and second product are a chain.  Taken back: the second group half a step behind the first
// (with two tiles of values: 157), raised priority for the first product (162).
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "seq_common.h"

namespace vla {
namespace seq {
namespace {

constexpr int kKeys = 64;           // keys of a tile
constexpr int kRowsPerWave = 32;
constexpr int kWaves = 4;
constexpr int kRowsPerGroup = kRowsPerWave * kWaves, kGroupShift = 7;
static_assert(kRowsPerGroup == 1 << kGroupShift, "tiles of rows are ranked by their level");
constexpr int kEarly = 4;           // a wave's DMA instructions for the next keys ahead of the softmax
constexpr int kGatherRows = 8;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef s16x4 __attribute__((address_space(3))) * lds_s16x4;

template <class S>
struct Mma;
template <>
struct Mma<BF16> {
  static __device__ __forceinline__ f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  }
};
template <>
struct Mma<F16> {
  static __device__ __forceinline__ f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
  }
};

// 0xffff for each of two 16-bit numbers that is not finite
template <class S>
__device__ __forceinline__ uint32_t odd_halves(uint32_t x) {
  constexpr uint32_t kLow = std::is_same<S, BF16>::value ? 0x7f80u : 0x7c00u, kHigh = kLow << 16;      // exponents of ones
  return ((x & kLow) == kLow ? 0xffffu : 0u) | ((x & kHigh) == kHigh ? 0xffff0000u : 0u);
}

// where sequence b's rows begin among all gathered rows (one wave; every lane gets it)
__device__ __forceinline__ int gathered_before(const int* __restrict__ query_start_loc,
                                               const int* __restrict__ context_lens, int b, int window) {
  int n = 0;
  for (int i = threadIdx.x & 63; i < b; i += kWave)
    n += context_lens[i] + query_start_loc[i + 1] - query_start_loc[i] - first_formed(context_lens[i], window);
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) n += __shfl_xor(n, m, 64);
  return __builtin_amdgcn_readfirstlane(n);
}

// rows[k] = the cache row of the k-th visible key: kGatherRows rows per workgroup, 16 bytes per lane
__global__ __launch_bounds__(256) void latent_gather_kernel(
    u32x4* __restrict__ rows, const u32x4* __restrict__ cache, const int* __restrict__ block_tables,
    int max_blocks, const int* __restrict__ query_start_loc, const int* __restrict__ context_lens,
    int pieces, int block_size, int num_blocks, int window, int num_rows, int key_first) {
  const int b = blockIdx.y;
  const int ctx = context_lens[b], first = first_formed(ctx, window) + key_first;
  const int n = ctx + query_start_loc[b + 1] - query_start_loc[b] - first;
  if ((int)blockIdx.x * kGatherRows >= n) return;
  const int base = gathered_before(query_start_loc, context_lens, b, window);
  const int* table = block_tables + (int64_t)b * max_blocks;
  const int end = min(n, num_rows - base);
  // (a second time round only where the sequence is longer than the host's lengths say)
  for (int r0 = blockIdx.x * kGatherRows; r0 < end; r0 += gridDim.x * kGatherRows) {
    const int count = min(kGatherRows, end - r0) * pieces;
    for (int i = threadIdx.x; i < count; i += 256) {
      const int r = i / pieces, v = i - r * pieces;
      const int j = first + r0 + r;
      int blk = table[j / block_size];
      blk = (unsigned)blk < (unsigned)num_blocks ? blk : 0;  // a table the host filled wrongly reads block 0
      rows[(int64_t)(base + r0 + r) * pieces + v] = cache[((int64_t)blk * block_size + j % block_size) * pieces + v];
    }
  }
}

// Every head's keys, in two numbers each, and values of the gathered rows: [num_rows, rank] times W_uk^T [rank, heads * dim]
// and W_uv [rank, heads * vdim] in one launch.  A workgroup has 256 rows and 128 columns of keys or of values, a wave 128 rows
// and 64 columns; products on 32x32x16 MFMAs with the weights as the rows, so that a lane ends with neighbouring columns of
// one row.  Stages of 32 numbers of the rank come by LDS-DMA into a ring of three (72 KB: two workgroups to a CU, one's
// results leave under the other's products), 16-byte pieces (values' weights, which lie with a head's columns
// as rows and are read transposing: 64-byte ones) exchanged by the row's number.  A key's remainder comes from the sum in the
// registers.  4096 rows of rank 512 and 16 heads of 128 + 128: 31 us, 550 TFLOP/s; a library's product per operand and a third
// for what the first lost, with a copy of the keys ahead of it and one of the values' weights, were 70.  Counted: matrix
// cores are at work in 34 % of a CU's busy cycles, vector instructions in 22 %, LDS reads in 13 %: all 512 workgroups are there at
// once, wait for their first stages together and write 50 MB of results together at the end.
constexpr int kFormRows = 256, kFormCols = 128, kFormStep = 32;
constexpr int kFormLatents = kFormRows * kFormStep * 2, kFormStage = kFormLatents + kFormCols * kFormStep * 2;
struct LatentForm {
  void* keys;
  void* keys_rest;
  void* values;
  const void* rows;             // [num_rows, row_width]: latents of `rank` and something behind them
  const void* w_uk;             // [heads * dim, rank]
  const void* w_uv;             // [heads, rank, vdim]
  int num_rows, row_width, heads, dim, vdim, rank;
  int key_tiles, tiles;         // column tiles: of keys, and all
};

template <class S>
__global__ __launch_bounds__(256, 2) void latent_form_kernel(LatentForm a) {
  using T = typename S::T;
  using M = Mma<S>;
  extern __shared__ __align__(16) unsigned char smem[];
  // an XCD's workgroups (every eighth) share an eighth of the column tiles, whose weights stay in its L2
  const int share = (a.tiles + 7) / 8, id = blockIdx.x >> 3;
  const int tile = (blockIdx.x & 7) + 8 * (id % share), m0 = id / share * kFormRows;
  if (tile >= a.tiles) return;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hf = lane >> 5, c = lane & 31, wm = w & 1, wn = w >> 1;
  const int steps = a.rank / kFormStep;
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)smem;
  const unsigned char* src[6];                             // four pieces of latents, two of weights
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int r = 16 * (4 * w + u) + (lane >> 2), piece = (lane & 3) ^ ((r >> 2) & 3);
    src[u] = (const unsigned char*)a.rows + ((int64_t)min(m0 + r, a.num_rows - 1) * a.row_width + 8 * piece) * 2;
  }
  auto form = [&](auto is_key) __attribute__((always_inline)) {
    constexpr bool KEY = decltype(is_key)::value;
    const int n_all = KEY ? a.heads * a.dim : a.heads * a.vdim;
    const int n0 = kFormCols * (KEY ? tile : tile - a.key_tiles);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i = 2 * w + u;
      if constexpr (KEY) {
        const int r = 16 * i + (lane >> 2), piece = (lane & 3) ^ ((r >> 2) & 3);
        src[4 + u] = (const unsigned char*)a.w_uk + ((int64_t)min(n0 + r, n_all - 1) * a.rank + 8 * piece) * 2;
      } else {
        const int k = 4 * i + (lane >> 4), s = lane & 15;
        const int n = min(n0 + 32 * ((s >> 2) ^ (k & 3)) + 8 * (s & 3), n_all - 8), h = n / a.vdim;
        src[4 + u] = (const unsigned char*)a.w_uv + (((int64_t)h * a.rank + k) * a.vdim + (n - h * a.vdim)) * 2;
      }
    }
    const int w_step = KEY ? 2 * kFormStep : 2 * kFormStep * a.vdim;
    auto bring = [&](int u, int step, int slot, int go) {
      tile_dma16(src[u] + (int64_t)step * (u < 4 ? 2 * kFormStep : w_step),
                 lds0 + slot * kFormStage + (u < 4 ? (4 * w + u) * 1024 : kFormLatents + (2 * w + u - 4) * 1024), go);
    };
    f32x16 acc[4][2];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mb][nb][i] = 0.f;
#pragma unroll
    for (int u = 0; u < 6; ++u) bring(u, 0, 0, 1);
#pragma unroll
    for (int u = 0; u < 6; ++u) bring(u, 1, 1, steps > 1);
    const int swap = (c >> 2) & 3, i16 = c & 15;
    // fragment i of 16 numbers of the rank: two of weights, then four of rows
    auto read = [&](const unsigned char* at, int ks, int i) {
      if (i >= 2) return *reinterpret_cast<const u32x4*>(at + (128 * wm + 32 * (i - 2) + c) * 64 + 16 * ((2 * ks + hf) ^ swap));
      if constexpr (KEY) {
        return *reinterpret_cast<const u32x4*>(at + kFormLatents + (64 * wn + 32 * i + c) * 64 + 16 * ((2 * ks + hf) ^ swap));
      } else {
        const unsigned char* p = at + kFormLatents + (16 * ks + 8 * hf + (i16 >> 2)) * (2 * kFormCols) +
                                 64 * ((2 * wn + i) ^ (i16 >> 2)) + 32 * (c >> 4) + 8 * (i16 & 3);
        const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)p));
        const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(p + 4 * 2 * kFormCols)));
        return u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
    };
    int slot = 0;
    for (int it = 0; it < steps; ++it) {
      // this stage has come (of the younger one's six pieces none need have), and the stage before it is read
      if (it + 1 < steps)
        __builtin_amdgcn_s_waitcnt(0x0076);                // vmcnt(6), lgkmcnt(0)
      else
        __builtin_amdgcn_s_waitcnt(0x0070);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const unsigned char* at = smem + slot * kFormStage;
      const int free_slot = slot == 0 ? 2 : slot - 1;
      u32x4 f[2][6];
#pragma unroll
      for (int i = 0; i < 6; ++i) f[0][i] = read(at, 0, i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (ks == 0 && i < 6) f[1][i] = read(at, 1, i);
          acc[i >> 1][i & 1] = M::run(f[ks][i & 1], f[ks][2 + (i >> 1)], acc[i >> 1][i & 1]);
          if (ks == 0 && i >= 2) bring(i - 2, it + 2, free_slot, it + 2 < steps);
          __builtin_amdgcn_sched_barrier(0);
        }
      slot = slot == 2 ? 0 : slot + 1;
    }
    // eight neighbouring columns a lane: of two groups of eight, the lower half of the wave has the first
    const int n = n0 + 64 * wn + 8 * hf;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      const int row = m0 + 128 * wm + 32 * mb + c;
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          u32x4 put, rest;
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            uint32_t hi[2], lo[2];
#pragma unroll
            for (int g = 0; g < 2; ++g) {
              const float x = acc[mb][nb][8 * j + 4 * g + 2 * e], y = acc[mb][nb][8 * j + 4 * g + 2 * e + 1];
              hi[g] = M::pack2(x, y);
              if constexpr (KEY) lo[g] = M::pack2(x - lo16<S>(hi[g]), y - hi16<S>(hi[g]));
            }
            const auto both = __builtin_amdgcn_permlane32_swap(hi[0], hi[1], false, false);
            put[e] = both[0];
            put[2 + e] = both[1];
            if constexpr (KEY) {
              const auto left = __builtin_amdgcn_permlane32_swap(lo[0], lo[1], false, false);
              rest[e] = left[0];
              rest[2 + e] = left[1];
            }
          }
          const int col = n + 32 * nb + 16 * j;
          if (row < a.num_rows && col < n_all) {
            const int64_t to = (int64_t)row * n_all + col;
            *reinterpret_cast<u32x4*>((T*)(KEY ? a.keys : a.values) + to) = put;
            if constexpr (KEY) *reinterpret_cast<u32x4*>((T*)a.keys_rest + to) = rest;
          }
        }
    }
  };
  if (tile < a.key_tiles)
    form(std::true_type{});
  else
    form(std::false_type{});
}

struct LatentPrompt {
  void* out;
  int64_t out_stride;
  const void* q;                // [T, heads * q_head]: a head's row is [plain (dim) | rotated (rot)]
  int64_t q_stride;
  const void* keys;             // [N, heads * dim]
  const void* keys_rest;        // the same: what the keys lost when they were rounded
  const void* values;           // [N, heads * vdim]
  const void* rows;             // [N, rank + rot]: the rotated part behind the latent
  const int* query_start_loc;
  const int* context_lens;
  const void* gate;
  int64_t gate_stride;
  const float* sinks;
  float* carry;                 // one sequence whose keys come in ranges: [T, heads, VD + 4], null otherwise
  int heads, dim, rot, vdim, rank, window, num_rows, row_tiles;
  int ranked_seqs, tiles;       // ranked_seqs > 0: tiles are found by their rank among at most `tiles`
  int key_first, key_total;     // the range's first key and all keys of the sequence
  float scale;
};

// for pieces of LDS rows behind a row's end
__device__ const u32x4 kNothing = {0u, 0u, 0u, 0u};

template <class S, int DB, int VB, int LB, int KG>
__global__ __launch_bounds__(256 * KG, 2) void latent_prompt_kernel(LatentPrompt a) {
  using T = typename S::T;
  using M = Mma<S>;
  constexpr int DQ = 32 * DB, VD = 32 * VB, LD = 32 * LB;
  constexpr int KB = 2 * DQ, VBYTES = 2 * VD, RB = 2 * LD;                   // bytes of a tile's rows
  constexpr int KTILE = kKeys * KB, RTILE = kKeys * RB, VTILE = kKeys * VBYTES;
  constexpr int KI = KTILE / 1024 / kWaves, RI = RTILE / 1024 / kWaves, VI = VTILE / 1024 / kWaves;    // DMA instructions per wave
  // a key row is a whole number of 256 bytes (all 64 banks), or half of one more: which pieces change place
  constexpr int KMASK = KB % 256 == 0 ? 15 : 7, KSHIFT = KB % 256 == 0 ? 0 : 1;
  constexpr int RMASK = RB % 256 == 0 ? 15 : 7, RSHIFT = RB % 256 == 0 ? 0 : 1;
  constexpr int kStep = kKeys * KG;                        // keys of a step: a tile for every group of four waves
  extern __shared__ __align__(16) unsigned char all_tiles[];
  const int h = blockIdx.x % a.heads;
  const bool ranged = a.carry != nullptr, last_range = !ranged || a.key_first + a.num_rows == a.key_total;
  int b = blockIdx.z, tile = a.row_tiles - 1 - (int)blockIdx.y;       // the longest walks first
  int t_first, run, ctx, base;
  if (a.ranked_seqs > 0) {
    const int rank = blockIdx.x / a.heads;
    const RankedTile found = ranked_tile<true>(rank, a.ranked_seqs, a.query_start_loc, a.context_lens, kGroupShift, a.row_tiles,
                                               a.window, ranged ? 0x7fffffff : a.num_rows);
    // the host gathered for other lengths than the device has: no answer for those behind, and none that looks like one
    for (int i = rank; i < (a.ranked_seqs - found.fitting) * a.row_tiles; i += a.tiles) {
      const int s = found.fitting + i / a.row_tiles, r = kRowsPerGroup * (i % a.row_tiles);
      const int n = min(kRowsPerGroup, a.query_start_loc[s + 1] - a.query_start_loc[s] - r);
      T* row = (T*)a.out + (int64_t)(a.query_start_loc[s] + r) * a.out_stride + (int64_t)h * a.vdim;
      for (int e = threadIdx.x; e < n * a.vdim; e += 256 * KG) row[e / a.vdim * a.out_stride + e % a.vdim] = S::from_f32(NAN);
    }
    if (rank >= found.all) return;
    tile = found.tile;
    t_first = found.first_row;
    run = found.rows;
    ctx = found.context;
    base = found.before;
  } else {
    t_first = a.query_start_loc[b];
    run = a.query_start_loc[b + 1] - t_first;
    ctx = a.context_lens[b];
    base = ranged ? 0 : gathered_before(a.query_start_loc, a.context_lens, b, a.window);
  }
  const int r0 = tile * kRowsPerGroup;
  if (r0 >= run) return;
  const int tid = threadIdx.x;
  const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);     // group of waves
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane((tid & 255) >> 6);
  unsigned char* smem = all_tiles + kg * (KTILE + RTILE + VTILE);
  const int hf = lane >> 5, c = lane & 31;
  const int first = first_formed(ctx, a.window) + (ranged ? a.key_first : 0);
  const int n_rows = min(kRowsPerGroup, run - r0);         // rows of this workgroup
  const int nq = min(kRowsPerWave, n_rows - kRowsPerWave * w);               // and of this wave (<= 0: none)
  const int t0 = t_first + r0 + kRowsPerWave * w;
  // positions, counted from the first gathered key
  const int p0 = ctx + r0 + kRowsPerWave * w - first, pq = p0 + c;
  const int n_keys = min(ctx + run - first, a.num_rows);
  const int p_end = min(ctx + r0 + n_rows - 1 - first, n_keys - 1);
  if (ranged ? ctx + run - first != a.key_total - a.key_first : base + ctx + run - first > a.num_rows) {
    // other lengths again
    const uint32_t nan2 = M::pack2(NAN, NAN);
    T* orow = (T*)a.out + (int64_t)(t0 + c) * a.out_stride + (int64_t)h * a.vdim + 4 * hf;
    for (int d = 0; c < nq && d + 4 * hf < a.vdim; d += 8) *reinterpret_cast<u32x2*>(orow + d) = u32x2{nan2, nan2};
    return;
  }
  const int g_first = a.window > 0 ? max(0, ctx + r0 - first - a.window + 1) : 0;    // the group's first key
  const int g_p0 = ctx + r0 - first, g_lo_last = a.window > 0 ? g_p0 + kRowsPerGroup - a.window : 0;    // the group's
  const int lo_q = a.window > 0 ? pq - a.window + 1 : 0;                       // this row's
  const int lo_last = a.window > 0 ? p0 + kRowsPerWave - a.window : 0;         // the wave's last row's
  const int lo_first = a.window > 0 ? p0 - a.window + 1 : 0;

  u32x4 qf[DQ / 16];
  const int width = a.dim + a.rot;
#pragma unroll
  for (int ks = 0; ks < DQ / 16; ++ks) {
    u32x4 v = {0u, 0u, 0u, 0u};
    const int d = 16 * ks + 8 * hf;
    if (c < nq && d < width)
      v = *reinterpret_cast<const u32x4*>((const T*)a.q + (int64_t)(t0 + c) * a.q_stride + (int64_t)h * width + d);
    qf[ks] = v;
  }
  f32x16 o[VB];
#pragma unroll
  for (int n = 0; n < VB; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[n][i] = 0.f;
  const float scale2 = a.scale * 1.4426950408889634f;      // scores in base 2; scale > 0
  float m = -INFINITY, l = 0.f;
  if (a.sinks != nullptr && kg == 0) {                     // the denominator's first term, counted in one lane half
    m = a.sinks[h] * 1.4426950408889634f;
    l = hf == 0 ? __builtin_amdgcn_exp2f(m - (m == -INFINITY ? 0.f : m)) : 0.f;      // 1, 0 or, for an infinite one, NaN
  }
  if (ranged && a.key_first > 0 && c < nq && kg == 0) {               // where the range before this one ended
    const float* carry = a.carry + ((int64_t)(t0 + c) * a.heads + h) * (VD + 4);
    m = carry[0];
    l = carry[1 + hf];
#pragma unroll
    for (int n = 0; n < VB; ++n)
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        const f32x4 got = *reinterpret_cast<const f32x4*>(carry + 4 + 32 * n + 8 * (i >> 2) + 4 * hf);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[n][i + e] = got[e];
      }
  }

  // What this lane brings in: piece `at` of a tile in LDS is row at / pieces; which 16 bytes of the row
  // stand there follows from the exchange.  Pieces past the end of a key are zeros; those past a value's repeat its
  // first ones, for columns nobody writes.  The first KI pieces are the keys', the next RI what rounding took.
  constexpr int kKeyPieces = KI + RI;
  const unsigned char* from_k[kKeyPieces];                  // where the piece of the first tile lies
  int row_k[kKeyPieces];
  int step_k[kKeyPieces];
  const int key_row = a.heads * a.dim * 2, value_row = a.heads * a.vdim * 2;
  const int lat_row = (a.rank + a.rot) * 2;
  const int64_t first_key = (int64_t)base * key_row + (int64_t)h * a.dim * 2;
#pragma unroll
  for (int u = 0; u < KI; ++u) {
    const int at = ((w * KI + u) * 1024 + 16 * lane) / 16, r = at / (KB / 16), s = at % (KB / 16);
    const int piece = (s & ~KMASK) | ((s ^ (r >> KSHIFT)) & KMASK);
    const int d = 8 * piece;
    row_k[u] = r;
    step_k[u] = d < a.dim ? key_row : d < width ? lat_row : 0;
    from_k[u] = d < a.dim   ? (const unsigned char*)a.keys + first_key + 2 * d
                : d < width ? (const unsigned char*)a.rows + (int64_t)base * lat_row + (a.rank + d - a.dim) * 2
                            : (const unsigned char*)&kNothing;
    from_k[u] += (int64_t)r * step_k[u];
  }
#pragma unroll
  for (int u = 0; u < RI; ++u) {
    const int at = ((w * RI + u) * 1024 + 16 * lane) / 16, r = at / (RB / 16), s = at % (RB / 16);
    const int piece = (s & ~RMASK) | ((s ^ (r >> RSHIFT)) & RMASK);
    const int d = 8 * piece;
    row_k[KI + u] = r;
    step_k[KI + u] = d < a.dim ? key_row : 0;
    from_k[KI + u] = d < a.dim ? (const unsigned char*)a.keys_rest + first_key + 2 * d : (const unsigned char*)&kNothing;
    from_k[KI + u] += (int64_t)r * step_k[KI + u];
  }
  // (a value row's pieces come in at the same places for every instruction, kValueRows rows further on)
  constexpr int kValueRows = 1024 / VBYTES;
  const int row_v = w * VI * kValueRows + lane / (VBYTES / 16), unit_v = VB == 4 ? row_v & 3 : (row_v >> 1) & (VB - 1);
  const int sv = lane % (VBYTES / 16), dv = 8 * ((((sv >> 2) ^ unit_v) << 2) | (sv & 3));
  const unsigned char* from_v = (const unsigned char*)a.values + (int64_t)(base + row_v) * value_row +
                                ((int64_t)h * a.vdim + (dv < a.vdim ? dv : 0)) * 2;
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)smem;
  // piece i of the tile that begins with key u0; behind the end the last key again
  auto bring_key = [&](int i, int u0, int go) {
    tile_dma16(from_k[i] + (int64_t)min(u0, n_keys - 1 - row_k[i]) * step_k[i],
               lds0 + (i < KI ? (w * KI + i) * 1024 : KTILE + (w * RI + i - KI) * 1024), go);
  };
  auto bring_value = [&](int i, int u0, int go) {
    tile_dma16(from_v + (int64_t)min(u0 + i * kValueRows, n_keys - 1 - row_v) * value_row, lds0 + KTILE + RTILE + (w * VI + i) * 1024, go);
  };
  // where this lane reads: the exchanged piece of its key row, and the unit of its value rows
  const int kx = (hf ^ ((c >> KSHIFT) & KMASK)) & KMASK;   // piece 2 ks + hf stands at 2 ks ^ kx within its group
  const int rx = (hf ^ ((c >> RSHIFT) & RMASK)) & RMASK;
  const int i16 = c & 15;
  const int vrow = 4 * hf + (i16 >> 2);
  const int vf = VB == 4 ? vrow & 3 : (vrow >> 1) & (VB - 1);
  const int vat = vrow * VBYTES + 32 * (c >> 4) + 8 * (i16 & 3);

  // Keys and values take turns: a tile's values come in under the first product, the next tile's keys under the
  // softmax and the second one.
  const unsigned char* k_lds = smem;
  const unsigned char* r_lds = smem + KTILE;
  const unsigned char* v_lds = smem + KTILE + RTILE;
  auto landed = [&]() {
    // the builtin and not asm: the compiler then knows that the query rows have arrived, and does not wait for
    // vmcnt(0), and so for the DMA just started, at their first use in every step
    __builtin_amdgcn_s_waitcnt(0x0f70);                // vmcnt(0)
    asm volatile("" ::: "memory");
    __syncthreads();
  };
  int u0 = (g_first & ~(kKeys - 1)) + kg * kKeys;
  float top = m == -INFINITY ? 0.f : m;                    // m, and 0 where nothing was seen yet
  if (u0 <= p_end)
#pragma unroll
    for (int i = 0; i < kKeyPieces; ++i) bring_key(i, u0, 1);
  for (; u0 - kg * kKeys <= p_end; u0 += kStep) {
    landed();
    const bool concerned = nq > 0 && u0 <= p_end && u0 <= p0 + nq - 1 && u0 + kKeys > lo_first;     // some key of it concerns this wave
    f32x16 st[2];
    if (concerned) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) st[kb][i] = 0.f;
      // keys are read two steps ahead of their products, and the values' DMA goes out between the products
      constexpr int kSteps = (DQ + LD) / 16;
      auto key_at = [&](int ks, int kb) {
        const int k = ks < DQ / 16 ? ks : ks - DQ / 16;
        const int slot = ks < DQ / 16 ? ((2 * k) & ~KMASK) | (((2 * k) & KMASK) ^ kx) : ((2 * k) & ~RMASK) | (((2 * k) & RMASK) ^ rx);
        return *reinterpret_cast<const u32x4*>((ks < DQ / 16 ? k_lds + (32 * kb + c) * KB : r_lds + (32 * kb + c) * RB) + 16 * slot);
      };
      u32x4 ka[3][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) ka[ks][kb] = key_at(ks, kb);
#pragma unroll
      for (int ks = 0; ks < kSteps; ++ks) {
        if (ks + 2 < kSteps) {
#pragma unroll
          for (int kb = 0; kb < 2; ++kb) ka[(ks + 2) % 3][kb] = key_at(ks + 2, kb);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) st[kb] = M::run(ka[ks % 3][kb], qf[ks < DQ / 16 ? ks : ks - DQ / 16], st[kb]);
        if (ks < VI) bring_value(ks, u0, 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int i = 0; i < VI; ++i) bring_value(i, u0, u0 <= p_end);
    }
    landed();
    const int more = u0 + kStep <= p_end;
#pragma unroll
    for (int i = 0; i < kEarly; ++i) bring_key(i, u0 + kStep, more);
    // A hidden key's weight is 0, which times an infinity or a NaN would not be: a tile that hides keys from some row
    // goes without values that are not finite.  Rows that see such a key are NaN by their scores: a key of the same
    // latent is not finite either, and it and what it lost to rounding never sum to a number (finite latents give finite
    // values: the layer looks at its weights for that).
    if (u0 + (KG - kg) * kKeys - 1 > g_p0 || u0 - kg * kKeys < g_lo_last) {      // (the same for both groups: a barrier)
#pragma unroll
      for (int u = 0; u < VI; ++u) {
        u32x4* at = reinterpret_cast<u32x4*>(smem + KTILE + RTILE + (w * VI + u) * 1024 + 16 * lane);
        u32x4 x = *at;
        uint32_t some = 0u;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t odd = odd_halves<S>(x[e]);
          x[e] &= ~odd;
          some |= odd;
        }
        if (some != 0u) *at = x;
      }
      __syncthreads();
    }
    if (!concerned) {
#pragma unroll
      for (int i = kEarly; i < kKeyPieces; ++i) bring_key(i, u0 + kStep, more);
      continue;
    }
    // Values: transposing reads, the first 16 keys' under the softmax
    u32x4 va[VB];
    auto value_at = [&](int s4, int n) {                   // keys 16 s4 .. + 15, dims 32 n ..
      // 8 rows further on the exchange is the same for four units; for two it is too (8 / 2 even)
      const unsigned char* at = v_lds + vat + 16 * s4 * VBYTES + 64 * (n ^ vf);
      const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)at));
      const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(at + 8 * VBYTES)));
      return u32x4{lo[0], lo[1], hi[0], hi[1]};
    };
#pragma unroll
    for (int n = 0; n < VB; ++n) va[n] = value_at(0, n);
    // masks only where some key of the tile is hidden from some row of the wave; nobody writes the rows behind the run's end
    if (u0 + kKeys - 1 > p0 || u0 < lo_last) {
      const int least = lo_q - u0 - 4 * hf;
      const uint32_t seen = max(pq - lo_q + 1, 0);        // (rows ahead of a range of keys see none)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          st[kb][i] = (uint32_t)(32 * kb + (i & 3) + 8 * (i >> 2) - least) < seen ? st[kb][i] : -INFINITY;
    }
    float mts[2] = {-INFINITY, -INFINITY};                 // chains of their own
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) mts[kb] = fmaxf(mts[kb], st[kb][i]);
    const float mt = max_halves(fmaxf(mts[0], mts[1])) * scale2;
    // (a maximum that may lag behind, by 8 in base 2, leaves the accumulators alone in most tiles and is 2.5 % faster, but
    // the largest weight is then no longer 1 and rounds like the others: errors grow by 1 to 2 %)
    if (__any(mt > m)) {
      const float m_new = fmaxf(m, mt);
      top = m_new == -INFINITY ? 0.f : m_new;              // nothing seen yet: every weight is 2^-inf
      const float corr = __builtin_amdgcn_exp2f(m - top);
      l *= corr;
#pragma unroll
      for (int n = 0; n < VB; ++n)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[n][i] *= corr;
      m = m_new;
    }
    // weights 8 s4 .. + 7 of this lane; the partner's half of the sum is added at the end
    auto weight2 = [&](int s4, int e) {
      const float a0 = st[s4 >> 1][8 * (s4 & 1) + 2 * e], b0 = st[s4 >> 1][8 * (s4 & 1) + 2 * e + 1];
      const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(a0, scale2, -top));
      const float y = __builtin_amdgcn_exp2f(__builtin_fmaf(b0, scale2, -top));
      l += x;
      l += y;
      return M::pack2(x, y);
    };
    u32x4 pb[2];
#pragma unroll
    for (int e = 0; e < 4; ++e) pb[0][e] = weight2(0, e);
    // the next 16 keys' weights are formed, and the next tile's keys sent for, between the products of these
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
#pragma unroll
      for (int n = 0; n < VB; ++n) {
        o[n] = M::run(va[n], pb[s4 & 1], o[n]);
        if (s4 < 3) {
          va[n] = value_at(s4 + 1, n);
#pragma unroll
          for (int e = 4 * n / VB; e < 4 * (n + 1) / VB; ++e) pb[(s4 + 1) & 1][e] = weight2(s4 + 1, e);
        }
#pragma unroll
        for (int i = kEarly; i < kKeyPieces; ++i)
          if ((i - kEarly) * 2 * VB / (kKeyPieces - kEarly) == s4 * VB + n) bring_key(i, u0 + kStep, more);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  if constexpr (KG == 2) {
    // the second group hands its sums over: registers lie lane for lane in the tiles' place
    __syncthreads();
    float* part = reinterpret_cast<float*>(all_tiles) + w * (VB * 16 + 2) * kWave + lane;
    if (kg == 1) {
      part[0] = m;
      part[kWave] = l;
#pragma unroll
      for (int n = 0; n < VB; ++n)
#pragma unroll
        for (int i = 0; i < 16; ++i) part[(2 + 16 * n + i) * kWave] = o[n][i];
    }
    __syncthreads();
    if (kg == 1) return;
    const float m2 = part[0], m_new = fmaxf(m, m2);
    const float shift = m_new == -INFINITY ? 0.f : m_new;
    const float f = __builtin_amdgcn_exp2f(m - shift), f2 = __builtin_amdgcn_exp2f(m2 - shift);
    l = l * f + part[kWave] * f2;
#pragma unroll
    for (int n = 0; n < VB; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[n][i] = o[n][i] * f + part[(2 + 16 * n + i) * kWave] * f2;
    m = m_new;
  }
  // (this lane's row and half again: what follows from them would be kept through the loop, which has no registers left)
  int me = threadIdx.x;
  asm volatile("" : "+v"(me));
  const int row = t0 + (me & 31), half = (me >> 5) & 1;
  if (!last_range) {
    if (row >= t0 + nq) return;
    float* carry = a.carry + ((int64_t)row * a.heads + h) * (VD + 4);
    if (half == 0) carry[0] = m;
    carry[1 + half] = l;
#pragma unroll
    for (int n = 0; n < VB; ++n)
#pragma unroll
      for (int i = 0; i < 16; i += 4)
        *reinterpret_cast<f32x4*>(carry + 4 + 32 * n + 8 * (i >> 2) + 4 * half) = f32x4{o[n][i], o[n][i + 1], o[n][i + 2], o[n][i + 3]};
    return;
  }
  l += __shfl_xor(l, 32, 64);
  if (row >= t0 + nq) return;
  T* orow = (T*)a.out + (int64_t)row * a.out_stride + (int64_t)h * a.vdim + 4 * half;
  float inv = 1.f / l;
  if (a.gate != nullptr) inv /= 1.f + expf(-S::to_f32(((const T*)a.gate)[(int64_t)row * a.gate_stride + h]));
#pragma unroll
  for (int n = 0; n < VB; ++n)
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      const int d = 32 * n + 8 * (i >> 2);
      if (d + 4 * half < a.vdim)
        *reinterpret_cast<u32x2*>(orow + d) =
            u32x2{M::pack2(o[n][i] * inv, o[n][i + 1] * inv), M::pack2(o[n][i + 2] * inv, o[n][i + 3] * inv)};
    }
}

template <class S, int DB, int VB, int LB, int KG>
int launch_latent_prompt_groups(const LatentPrompt& a, dim3 grid, hipStream_t stream) {
  constexpr size_t tiles = kKeys * 64 * (DB + VB + LB) * KG, sums = KG == 2 ? sizeof(float) * kWaves * (VB * 16 + 2) * kWave : 0;
  constexpr size_t lds = tiles > sums ? tiles : sums;
  static_assert(lds <= 160 * 1024, "two groups' tiles fit a CU's LDS");
  static std::atomic<bool> raised{false};           // LDS limit: raised once per kernel, not per launch
  if (lds > 64 * 1024 && !raised.load(std::memory_order_relaxed)) {
    VLA_SEQ_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_prompt_kernel<S, DB, VB, LB, KG>),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    raised.store(true, std::memory_order_relaxed);
  }
  latent_prompt_kernel<S, DB, VB, LB, KG><<<grid, 256 * KG, lds, stream>>>(a);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  return VLA_OK;
}
template <class S, int DB, int VB, int LB>
int launch_latent_prompt(const LatentPrompt& a, dim3 grid, int key_groups, hipStream_t stream) {
  return key_groups == 2 ? launch_latent_prompt_groups<S, DB, VB, LB, 2>(a, grid, stream)
                         : launch_latent_prompt_groups<S, DB, VB, LB, 1>(a, grid, stream);
}

// How many tiles of rows there are at most, how many groups of waves share a workgroup's keys, and whether a tile is found
// by its rank.  Every query row is a gathered row, too (a range's launch: one sequence).  The bound holds whatever the
// lengths on the device are: sequences have at most row_tiles tiles, and only those whose rows were gathered have any.
// Two groups where a CU has one workgroup and the walks are long enough for two (16 heads of 128 + 64, values of 128: one
// run of 512 rows 22 us with two groups, 23 with one; 16 of 128 behind 300 keys 29 and 28; 128 rows behind 2000 60 and 71;
// four heads of 64 + 32 and 64: 12 runs of 50 to 500 rows 16 and 18, 16 of 128 10 and 9.5), or where long runs have walks
// of all lengths (one of 4096 rows 152 and 165, two of 2048 78 and 83, three of 1024 behind 1000 95 and 88, 32 of 33 18
// and 10, eight of 512 42 and 31, 16 of 256 behind 2000 202 and 150; 280 workgroups of 4 narrow heads, 10 runs of 100 and 60
// of 20 behind 300, 25 and 20).
// Not by their rank where a sequence is a tile and the walks are short, as key / value prompts: 256 runs of 33 rows 72
// and 67 us, 128 of 128 101 and 98 (but one of 200 beside 60 of 10 behind 200 keys 44 and 54: the bound, which counts keys for
// rows, does not show that workgroups are empty).
struct PromptForm {
  int64_t tiles;
  int key_groups;
  bool ranked;
};
PromptForm prompt_form(int num_rows, int num_seqs, int max_query_len, int heads, int dim, int rot, int vdim, bool ranged) {
  const int64_t row_tiles = ((int64_t)max_query_len + kRowsPerGroup - 1) / kRowsPerGroup, all = num_seqs * row_tiles;
  PromptForm form;
  form.tiles = std::min(all, ranged ? row_tiles : (int64_t)num_rows / kRowsPerGroup + num_seqs);
  const int64_t workgroups = form.tiles * heads, keys = num_rows / num_seqs;
  const bool wide = dim + rot > 128 || vdim > 64;
  form.key_groups = (workgroups <= 256 && keys >= (wide ? 512 : 129)) || (workgroups <= 512 && max_query_len > 1024) ? 2 : 1;
  form.ranked = num_seqs <= kRankedSeqs && workgroups <= 0xffffff && !(row_tiles == 1 && num_seqs > 1 && keys <= 256);
  return form;
}

bool prompt_sizes(int dim, int rot, int vdim, int rank) {
  return dim > 0 && dim % 8 == 0 && rot >= 0 && rot % 8 == 0 && vdim > 0 && vdim % 8 == 0 && rank > 0 && rank % 8 == 0 &&
         dim + rot <= 192 && vdim <= 128;
}

}  // namespace
}  // namespace seq
}  // namespace vla

using namespace vla;
using namespace vla::seq;

extern "C" int vla_seq_latent_prompt_supported(int dim, int rot, int vdim, int rank, int dtype) {
  return (dtype == VLA_F16 || dtype == VLA_BF16) && prompt_sizes(dim, rot, vdim, rank);
}

extern "C" int vla_seq_latent_gather(void* rows, int num_rows, const void* cache, const int* block_tables,
                                     int max_blocks, const int* query_start_loc, const int* context_lens,
                                     int num_seqs, int max_seq_rows, int width, int block_size,
                                     int num_blocks, int window, int key_first, int dtype, void* stream) {
  if (num_seqs == 0 || num_rows == 0) return VLA_OK;
  if (!rows || !cache || !block_tables || !query_start_loc || !context_lens || num_seqs < 0 || num_seqs > 65535 ||
      num_rows < 0 || max_seq_rows <= 0 || max_blocks <= 0 || width <= 0 || block_size <= 0 || num_blocks <= 0 ||
      window < 0 || key_first < 0 || (key_first > 0 && num_seqs > 1))
    return VLA_ERR_ARG;
  if (dtype != VLA_F16 && dtype != VLA_BF16) return VLA_ERR_DTYPE;
  if (width % 8 || (uintptr_t)rows % 16 || (uintptr_t)cache % 16) return VLA_ERR_ARG;
  latent_gather_kernel<<<dim3((max_seq_rows + kGatherRows - 1) / kGatherRows, num_seqs), 256, 0, (hipStream_t)stream>>>(
      (u32x4*)rows, (const u32x4*)cache, block_tables, max_blocks, query_start_loc, context_lens, width / 8, block_size,
      num_blocks, window, num_rows, key_first);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  return VLA_OK;
}

extern "C" int vla_seq_latent_form_supported(int dim, int vdim, int rank, int row_width, int dtype) {
  return (dtype == VLA_F16 || dtype == VLA_BF16) && dim > 0 && dim % 8 == 0 && vdim > 0 && vdim % 8 == 0 && rank > 0 &&
         rank % kFormStep == 0 && row_width >= rank && row_width % 8 == 0;
}

extern "C" int vla_seq_latent_form(void* keys, void* keys_rest, void* values, const void* rows, int num_rows, int row_width,
                                  const void* w_uk, const void* w_uv, int heads, int dim, int vdim, int rank, int dtype,
                                  void* stream) {
  if (num_rows == 0) return VLA_OK;
  if (!keys || !keys_rest || !values || !rows || !w_uk || !w_uv || num_rows < 0 || heads <= 0 || dim <= 0 || vdim <= 0 ||
      rank <= 0 || row_width < rank || (int64_t)heads * dim > 0x3fffffff || (int64_t)heads * vdim > 0x3fffffff)
    return VLA_ERR_ARG;
  if (dtype != VLA_F16 && dtype != VLA_BF16) return VLA_ERR_DTYPE;
  if (!vla_seq_latent_form_supported(dim, vdim, rank, row_width, dtype)) return VLA_ERR_HEAD_SIZE;
  for (const void* p : {(const void*)keys, (const void*)keys_rest, (const void*)values, rows, w_uk, w_uv})
    if ((uintptr_t)p % 16) return VLA_ERR_ARG;
  LatentForm a;
  a.keys = keys;
  a.keys_rest = keys_rest;
  a.values = values;
  a.rows = rows;
  a.w_uk = w_uk;
  a.w_uv = w_uv;
  a.num_rows = num_rows;
  a.row_width = row_width;
  a.heads = heads;
  a.dim = dim;
  a.vdim = vdim;
  a.rank = rank;
  a.key_tiles = (heads * dim + kFormCols - 1) / kFormCols;
  a.tiles = a.key_tiles + (heads * vdim + kFormCols - 1) / kFormCols;
  const int64_t groups = ((int64_t)a.tiles + 7) / 8 * 8 * ((num_rows + (int64_t)kFormRows - 1) / kFormRows);
  if (groups > 0xffffff) return VLA_ERR_ARG;
  auto go = [&](auto s) -> int {
    using S = decltype(s);
    static std::atomic<bool> raised{false};           // LDS limit: raised once per kernel, not per launch
    if (!raised.load(std::memory_order_relaxed)) {
      VLA_SEQ_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_form_kernel<S>),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, 3 * kFormStage));
      raised.store(true, std::memory_order_relaxed);
    }
    latent_form_kernel<S><<<(unsigned)groups, 256, 3 * kFormStage, (hipStream_t)stream>>>(a);
    VLA_SEQ_HIP_CHECK(hipGetLastError());
    return VLA_OK;
  };
  return dtype == VLA_BF16 ? go(BF16{}) : go(F16{});
}

extern "C" int vla_seq_latent_prompt_form(int num_rows, int num_seqs, int max_query_len, int heads, int dim, int rot, int vdim,
                                         int ranged) {
  if (num_rows <= 0 || num_seqs <= 0 || max_query_len <= 0 || heads <= 0) return 0;
  const PromptForm form = prompt_form(num_rows, num_seqs, max_query_len, heads, dim, rot, vdim, ranged != 0);
  return form.key_groups + (form.ranked ? 4 : 0);
}

extern "C" int vla_seq_latent_prompt(void* out, int64_t out_stride, const void* q, int64_t q_stride,
                                     const void* keys, const void* keys_rest, const void* values,
                                     const void* rows, int num_rows,
                                     const int* query_start_loc, const int* context_lens, int num_seqs,
                                     int max_query_len, int heads, int dim, int rot, int vdim, int rank,
                                     float scale, int window, const void* gate, int64_t gate_stride,
                                     const float* sinks, int key_first, int key_total, float* carry, int dtype,
                                     void* stream) {
  if (num_seqs == 0 || max_query_len == 0) return VLA_OK;
  if (!out || !q || !keys || !keys_rest || !values || !rows || !query_start_loc || !context_lens || num_seqs < 0 ||
      num_seqs > 65535 || max_query_len < 0 || num_rows <= 0 || heads <= 0 || heads > 65535 || !(scale > 0.f) ||
      window < 0 || (gate && gate_stride < heads) || out_stride < (int64_t)heads * vdim ||
      q_stride < (int64_t)heads * (dim + rot))
    return VLA_ERR_ARG;
  if (dtype != VLA_F16 && dtype != VLA_BF16) return VLA_ERR_DTYPE;
  if (!prompt_sizes(dim, rot, vdim, rank)) return VLA_ERR_HEAD_SIZE;
  if ((uintptr_t)q % 16 || q_stride % 8 || (uintptr_t)keys % 16 || (uintptr_t)keys_rest % 16 || (uintptr_t)values % 16 || (uintptr_t)rows % 16 ||
      (uintptr_t)out % 8 || out_stride % 4)
    return VLA_ERR_ARG;
  // a range begins with a tile, and a tile ends with it or with the sequence
  if (carry ? num_seqs > 1 || key_first < 0 || key_first % kKeys || key_total - num_rows < key_first ||
                  (key_total - num_rows > key_first && num_rows % kKeys) || (uintptr_t)carry % 16
            : key_first != 0)
    return VLA_ERR_ARG;
  LatentPrompt a;
  a.out = out;
  a.out_stride = out_stride;
  a.q = q;
  a.q_stride = q_stride;
  a.keys = keys;
  a.keys_rest = keys_rest;
  a.values = values;
  a.rows = rows;
  a.query_start_loc = query_start_loc;
  a.context_lens = context_lens;
  a.gate = gate;
  a.gate_stride = gate_stride;
  a.sinks = sinks;
  a.carry = carry;
  a.key_first = key_first;
  a.key_total = key_total;
  a.heads = heads;
  a.dim = dim;
  a.rot = rot;
  a.vdim = vdim;
  a.rank = rank;
  a.window = window;
  a.num_rows = num_rows;
  a.row_tiles = (max_query_len + kRowsPerGroup - 1) / kRowsPerGroup;
  a.scale = scale;
  if (a.row_tiles > 65535) return VLA_ERR_ARG;
  const PromptForm form = prompt_form(num_rows, num_seqs, max_query_len, heads, dim, rot, vdim, carry != nullptr);
  a.ranked_seqs = form.ranked ? num_seqs : 0;
  a.tiles = form.ranked ? (int)form.tiles : 1;
  const int key_groups = form.key_groups;
  const dim3 grid = form.ranked ? dim3((unsigned)(heads * form.tiles)) : dim3(heads, a.row_tiles, num_seqs);
  auto go = [&](auto s) -> int {
    using S = decltype(s);
    auto with_values = [&](auto vb) -> int {
      constexpr int VB = decltype(vb)::value;
      if (dim > 128) return launch_latent_prompt<S, 6, VB, 6>(a, grid, key_groups, (hipStream_t)stream);
      return dim + rot > 128 ? launch_latent_prompt<S, 6, VB, 4>(a, grid, key_groups, (hipStream_t)stream)
                             : launch_latent_prompt<S, 4, VB, 4>(a, grid, key_groups, (hipStream_t)stream);
    };
    return vdim <= 64 ? with_values(std::integral_constant<int, 2>{}) : with_values(std::integral_constant<int, 4>{});
  };
  return dtype == VLA_BF16 ? go(BF16{}) : go(F16{});
}
