// Gated linear attention with a decay per key channel over runs of rows, in chunks of 64 rows that are worked
// on at the same time:  S_t = diag(a_t) S_(t-1) + k_t v_t^T,  o_t = S_t^T q_t,  a_t = sigmoid(W2 y_t + b)^(1/tau)
// per head, then o / rms(o) * w * silu(gate) * scale.  (Single rows and short runs: seq_linear_recurrence.hip.)
//
// A chunk's rows see its start state S through their decays from the chunk's start, and each other:
//   o_i = (q_i G_i)^T S + sum_(j <= i) A_ij v_j,    A_ij = sum_d q_i[d] k_j[d] prod_(l = j+1 .. i) a_l[d]
//   S' = diag(G) S + R,    R = sum_j (k_j prod_(l > j) a_l) v_j^T
//   gla_chunk_state_kernel  the decays' logarithms (left in scratch), G and R
//   gla_chunk_scan_kernel   S' = diag(G) S + R over a run's chunks in order, element by element; every chunk's
//                           start state takes R's place, the last one's successor the sequence's slot
//   gla_chunk_out_kernel    outputs, head norm and gate
// A chunk is four blocks of 16 rows.  Inside a block A is formed with the decays row by row; between blocks with
// the decays to a block's end, over whole blocks and from a block's start, each the exponential of a sum of
// logarithms over just those rows: nothing is divided and no sums are subtracted, so a decay of 0 beside decays of
// 1 is exact, and decays near 1 keep the precision of their logarithms (multiplied row by row they left the
// states after 4096 rows several times as far from 64 bits).
// Products run on 16x16x4 fp32 matrix cores, those with values of bfloat16 on its own (ThreeParts below).  Operands that
// later kernels read lie in scratch lane for lane.
// 4096 rows of 16 heads of 64 x 128 are 68 MB in and out and 100 MB of chunk states and decays: 74 us per call (23 + 13 + 44
// under the tracer; pieces of 256 rows walked token by token and joined by matrix products took 408).  Four workgroups share a
// CU, so that all 1024 of that step are there at once: 16-bit rows stay 16-bit in LDS (39 of 40 KB), a thread holds a channel's
// logarithms of a block in registers, A lies where its queries lay and the values where the keys were (two workgroups per CU
// and two rounds of them, with rows as 32-bit numbers beside a copy of the decays: 123 us, 42 + 23 + 66; with all products on
// the fp32 instructions 97, 31 + 23 + 52).  What bounds the first and last kernel now are vector instructions (84 and 60 % of
// a CU's busy cycles, counted; exponentials and logarithms most of them), in the last also matrix cores (24 %, most of it the
// fp32 products with the start states); the scan is a copy of the states, 34 MB in and out in 13 us.
#include <atomic>
#include <type_traits>

#include "seq_common.h"

namespace vla {
namespace seq {
namespace {

constexpr int kChunk = 64;
constexpr int kBlock = 16;
constexpr int kMaxDim = 128;
constexpr int kMaxRank = 32;
constexpr int kAMat = kChunk + 4;   // floats per row of A in LDS

struct GlaChunks {
  void* out;
  int64_t out_stride;
  const void* q;
  int64_t q_stride;
  const void* k;
  int64_t k_stride;
  const void* v;
  int64_t v_stride;
  const void* gate;
  int64_t gate_stride;
  const void* y;
  int64_t y_stride;
  const void* w2;               // [heads * dim, rank]
  const float* bias;            // [heads * dim]; null: 0
  const float* norm_weight;     // [vdim]
  float* state;                 // [slots, heads, dim, vdim]
  float* scratch;
  const int* query_start_loc;
  const int* context_lens;
  const int* state_slots;
  int num_seqs, heads, dim, vdim, rank;
  float q_scale, inv_tau, eps, out_scale;
  bool paired;                  // how tiles of columns lie in scratch: paired_column, or one after the other
};

// floats of a chunk and head: logarithms of the decays [64][dim] | G [dim] | R, then the start state [dim / 16][vdim / 16][lane][4]
__host__ __device__ __forceinline__ int64_t chunk_floats(int dim, int vdim) {
  return (int64_t)kChunk * dim + dim + (int64_t)dim * vdim;
}

// Which sequence and chunk a slot is: sequence b's chunks are slots start_b / 64 + b + 0, 1, ...
__device__ __forceinline__ bool find_chunk(const GlaChunks& a, int slot, int& b, int& chunk) {
  int lo = 0, hi = a.num_seqs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.query_start_loc[mid] / kChunk + mid <= slot)
      lo = mid;
    else
      hi = mid - 1;
  }
  b = lo;
  chunk = slot - (a.query_start_loc[b] / kChunk + b);
  return chunk >= 0 && chunk * kChunk < a.query_start_loc[b + 1] - a.query_start_loc[b];
}

// Four values of a row, aligned for one access, as they lie there and as numbers.  (Two steps: where loads stand behind
// conditions, one that is made a number at once is waited for before the next is asked for.)
template <class S>
using Four = std::conditional_t<sizeof(typename S::T) == 2, u32x2, f32x4>;
template <class S>
__device__ __forceinline__ Four<S> fetch4(const typename S::T* p) {
  return *reinterpret_cast<const Four<S>*>(p);
}
template <class S>
__device__ __forceinline__ f32x4 numbers(Four<S> x) {
  if constexpr (sizeof(typename S::T) == 2)
    return f32x4{lo16<S>(x[0]), hi16<S>(x[0]), lo16<S>(x[1]), hi16<S>(x[1])};
  else
    return x;
}

// exp(p) for p <= 0 (NaN passes): 2^n 2^f with the argument's rounding in f.  expf without what other p need, the same
// error: 2.62e-8 root mean square over -87 .. 0, 8.4e-8 at most.
__device__ __forceinline__ float exp_of_log(float p) {
#pragma clang fp contract(off)
  p = __builtin_elementwise_maximum(p, -150.f);
  const float t = 1.44269504f * p, n = __builtin_rintf(t);
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((t - n) + fmaf(1.92596299e-8f, p, fmaf(1.44269504f, p, -t))), (int)n);
}

// ln sigmoid(z) = -(max(-z, 0) + log1p(x)), x = exp(-|z|) in 0 .. 1: log1p as 2 artanh(x / (2 + x)) in two numbers, by its
// series up to the 17th power, and one rounding for the sum.  Error, root mean square and at most: 3.26e-8 and 1.35e-7 over
// -3 .. 6 (log1pf and expf 3.34e-8 and 1.35e-7), nowhere more than theirs.  No contraction: the quotient's rounding must be
// what the rest is formed from.
__device__ __forceinline__ float log_sigmoid(float z) {
#pragma clang fp contract(off)
  const float x = exp_of_log(-fabsf(z)), m = fmaxf(-z, 0.f);
  const float d = 2.f + x, lost = x - (d - 2.f), q = __builtin_amdgcn_rcpf(d), s = x * (2.f * q), y = s * s;
  const float more = fmaf(-lost, s, fmaf(-d, s, 2.f * x)) * q;
  float a = 1.f / (17.f * 65536.f);
  a = fmaf(a, y, 1.f / (15.f * 16384.f));
  a = fmaf(a, y, 1.f / (13.f * 4096.f));
  a = fmaf(a, y, 1.f / (11.f * 1024.f));
  a = fmaf(a, y, 1.f / (9.f * 256.f));
  a = fmaf(a, y, 1.f / (7.f * 64.f));
  a = fmaf(a, y, 1.f / (5.f * 16.f));
  a = fmaf(a, y, 1.f / (3.f * 4.f));
  const float hi = fmaxf(m, s), lo = fminf(m, s), t = hi + lo, lost_lo = hi < 1e30f ? lo - (t - hi) : 0.f;
  return -(t + (lost_lo + fmaf(a * y, s, more)));
}

// Values of a chunk in LDS, as they lie in memory: rows of V elements and some, so that rows 4 apart start 16 banks apart.
template <class S>
__host__ __device__ __forceinline__ int value_row(int vdim) {
  return (vdim + 31) / 32 * 32 + (sizeof(typename S::T) == 2 ? 8 : 4);
}

// Tiles of 16 value columns come in pairs that share a read: lane c has columns 2 c and 2 c + 1 of 32, the first for the one
// tile and the second for the other.  The last of an odd number of tiles stands alone and has column c.
struct TilePair {
  int at;          // where lane c reads its two values of a row
  bool alone, second;
  __device__ __forceinline__ TilePair(int pair, int tiles, int c)
      : at(2 * pair + 1 < tiles ? 32 * pair + 2 * c : 32 * pair + (c & ~1)), alone(2 * pair + 1 >= tiles), second(alone && (c & 1)) {}
  template <class S>
  __device__ __forceinline__ void read(const typename S::T* row, float& x, float& y) const {
    if constexpr (sizeof(typename S::T) == 2) {
      const uint32_t two = *reinterpret_cast<const uint32_t*>(row + at);
      x = lo16<S>(two);
      y = hi16<S>(two);
    } else {
      const float2 two = *reinterpret_cast<const float2*>(row + at);
      x = two.x;
      y = two.y;
    }
    x = second ? y : x;
  }
};
__device__ __forceinline__ int paired_column(int tile, int tiles, int c) {
  return (tile | 1) < tiles ? 32 * (tile >> 1) + 2 * c + (tile & 1) : 16 * tile + c;
}

// Products with values of bfloat16 run on its matrix cores, 32 rows at a time: a 32-bit factor is three bfloat16 numbers whose
// sum it is (8 of its 24 bits each), the value is one, every product is exact and sums are fp32 as those of the fp32
// instructions, which take five times as long (eight of 32 cycles where these take three of 16) and hold up vector
// instructions meanwhile.  An infinite value meets a factor's first part only: the others are often 0, and 0 times it is not
// a number where the factor times it is infinite.  Values come in by transposing reads: lane c has column c of a tile, rows
// 4 g .. 4 g + 3 of two blocks of 16.
template <class S>
constexpr bool kSplit = std::is_same<S, BF16>::value;
template <class S>
__device__ __forceinline__ int tile_column(int tile, int tiles, int c) {
  return kSplit<S> ? 16 * tile + c : paired_column(tile, tiles, c);
}
typedef unsigned short gla_u16x2 __attribute__((ext_vector_type(2)));
typedef short gla_s16x4 __attribute__((ext_vector_type(4)));
typedef gla_s16x4 __attribute__((address_space(3))) * gla_lds_s16x4;
struct ThreeParts {
  u32x4 part[3];                                           // the largest first
};
__device__ __forceinline__ ThreeParts three_parts(f32x4 x, f32x4 y) {
  float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]}, most = 0.f;
  ThreeParts t;
#pragma unroll
  for (int p = 0; p < 3; ++p) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      t.part[p][e] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, v[2 * e + 1]), __builtin_bit_cast(uint32_t, v[2 * e]), 0x07060302u);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (p == 0) most = fmaxf(most, fabsf(v[e]));
      v[e] -= __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v[e]) & 0xffff0000u);
    }
  }
  if (__any(most == INFINITY)) {                           // an infinity has no rest
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t w = t.part[0][e], keep = ((w & 0x7fffu) == 0x7f80u ? 0u : 0xffffu) | ((w & 0x7fff0000u) == 0x7f800000u ? 0u : 0xffff0000u);
      t.part[1][e] &= keep;
      t.part[2][e] &= keep;
    }
  }
  return t;
}
// values of lane c's column, at `rows` (the lane's row of a block and its place in it) and 16 rows further on
__device__ __forceinline__ u32x4 two_blocks(const void* rows, int pitch) {
  const char* at = (const char*)rows;
  const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((gla_lds_s16x4)(at)));
  const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((gla_lds_s16x4)(at + 16 * pitch)));
  return u32x4{lo[0], lo[1], hi[0], hi[1]};
}
// bfloat16 numbers, those that are not finite as 0
__device__ __forceinline__ u32x4 finite_only(u32x4 v) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
    v[e] &= ((v[e] & 0x7f80u) == 0x7f80u ? 0u : 0xffffu) | ((v[e] & 0x7f800000u) == 0x7f800000u ? 0u : 0xffff0000u);
  return v;
}
// rest: what the second and third parts meet
__device__ __forceinline__ f32x4 mfma_parts(const ThreeParts& a, u32x4 b, u32x4 rest, f32x4 c) {
#pragma unroll
  for (int p = 2; p >= 0; --p)
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a.part[p]), __builtin_bit_cast(bf16x8, p ? rest : b), c, 0, 0, 0);
  return c;
}

template <class S, int DT>          // DT: dim / 16
__global__ __launch_bounds__(256, DT <= 4 && sizeof(typename S::T) == 2 ? 4 : 2) void gla_chunk_state_kernel(GlaChunks a) {
  using T = typename S::T;
  extern __shared__ __align__(16) float lds[];
  constexpr int D = 16 * DT, KR = D + 4, ITEMS = (4 * D + 255) / 256;
  const int V = a.vdim, R = a.rank, VR = value_row<S>(V);
  const int RP = (R + 3) / 4 * 4;
  float* k_lds = lds;                       // [64][KR]
  float* tot = k_lds + kChunk * KR;         // [4][D]: a block's sum of logarithms
  float* y_lds = tot + 4 * D;               // [64][RP]
  int* odd_lds = (int*)(y_lds + kChunk * RP);                // [4]: a wave has met a value that is not finite
  T* v_lds = (T*)(odd_lds + 4);             // [64][VR]
  float* a_lds = (float*)(v_lds + kChunk * VR);              // [64][D]: logarithms, heads of less than 64 channels
  const int slot = blockIdx.x, h = blockIdx.y;
  int b, chunk;
  if (!find_chunk(a, slot, b, chunk)) return;
  const int run = a.query_start_loc[b + 1] - a.query_start_loc[b];
  const int t0 = a.query_start_loc[b] + chunk * kChunk, n = min(kChunk, run - chunk * kChunk);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15;
  float* mine = a.scratch + ((int64_t)slot * a.heads + h) * chunk_floats(D, V);

  // rows behind the run's end are zeros; every load is on its way before the first is waited for
  const int d = tid % D;                     // a thread has a channel's 16 rows of a block (two blocks with 128 channels)
  auto block_of = [&](int u) __attribute__((always_inline)) {
    return D >= 64 ? __builtin_amdgcn_readfirstlane((tid + 256 * u) / D) : min(tid / D, 3);
  };
  constexpr int PER = 16 / sizeof(T);
  const bool w_wide = R % PER == 0 && (uintptr_t)a.w2 % 16 == 0;
  u32x4 w_row[kMaxRank / PER];
  float wv[kMaxRank];
  const T* wr = (const T*)a.w2 + ((int64_t)h * D + d) * R;
  if (w_wide) {
#pragma unroll
    for (int r = 0; r < kMaxRank / PER; ++r) w_row[r] = *reinterpret_cast<const u32x4*>(wr + min(PER * r, R - PER));
  } else {
    T raw[kMaxRank];
#pragma unroll
    for (int r = 0; r < kMaxRank; ++r) raw[r] = wr[min(r, R - 1)];
#pragma unroll
    for (int r = 0; r < kMaxRank; ++r) wv[r] = r < R ? S::to_f32(raw[r]) : 0.f;
  }
  const float bias = a.bias != nullptr ? a.bias[(int64_t)h * D + d] : 0.f;
  const int row = tid >> 2, quarter = tid & 3;
  const int64_t t = t0 + min(row, n - 1);
  T ys[kMaxRank / 4];
#pragma unroll
  for (int u = 0; u < kMaxRank / 4; ++u) ys[u] = ((const T*)a.y)[t * a.y_stride + min(quarter + 4 * u, R - 1)];
  T ks[ITEMS][kBlock];
#pragma unroll
  for (int u = 0; u < ITEMS; ++u)
#pragma unroll
    for (int i = 0; i < kBlock; ++i)
      ks[u][i] = ((const T*)a.k + (t0 + min(kBlock * block_of(u) + i, n - 1)) * a.k_stride + (int64_t)h * D)[d];
  // four values a thread, in the order they lie in: V / 16 of them, whole for all threads
  constexpr int kMost = 8;
  Four<S> vs[kMost];
  const int per_row = V / 4, inverse = (65536 + per_row - 1) / per_row;      // (i * inverse) >> 16 is i / per_row below 2048
#pragma unroll
  for (int u = 0; u < kMost; ++u) {
    const int i = tid + 256 * min(u, V / 16 - 1), r = (i * inverse) >> 16, at = 4 * (i - r * per_row);
    vs[u] = fetch4<S>((const T*)a.v + (t0 + min(r, n - 1)) * a.v_stride + (int64_t)h * V + at);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < kMaxRank / 4; ++u)
    if (4 * u < RP) y_lds[row * RP + quarter + 4 * u] = quarter + 4 * u < R ? S::to_f32(ys[u]) : 0.f;
  __syncthreads();

  // decays, and keys times the decays behind them in their block
  if (w_wide) {
#pragma unroll
    for (int r = 0; r < kMaxRank; ++r) {
      if (r >= R)
        wv[r] = 0.f;
      else if constexpr (sizeof(T) == 2)
        wv[r] = r & 1 ? hi16<S>(w_row[r / PER][r % PER / 2]) : lo16<S>(w_row[r / PER][r % PER / 2]);
      else
        wv[r] = __builtin_bit_cast(float, (uint32_t)w_row[r / PER][r % PER]);
    }
  }
  // logarithms of rows first, first + step, ..
  auto logarithms = [&](auto& av, int first, int step) __attribute__((always_inline)) {
    constexpr int N = sizeof(av) / sizeof(av[0]);
#pragma unroll
    for (int i = 0; i < N; ++i) av[i] = bias;
#pragma unroll
    for (int r4 = 0; r4 < kMaxRank; r4 += 4) {
      if (r4 >= RP) break;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const f32x4 yv = *reinterpret_cast<const f32x4*>(y_lds + (first + step * i) * RP + r4);
#pragma unroll
        for (int e = 0; e < 4; ++e) av[i] += wv[r4 + e] * yv[e];
      }
    }
#pragma unroll
    for (int i = N - 1; i >= 0; --i) av[i] = first + step * i < n ? log_sigmoid(av[i]) * a.inv_tau : 0.f;
  };
  if constexpr (D < 64) {
    // Fewer channels' blocks than threads: their logarithms are everyone's (16 rows by a thread of each block: a workgroup of
    // 16 channels takes 2.3 us more).
    float av[D / 4];
    logarithms(av, tid / D, 256 / D);
#pragma unroll
    for (int i = 0; i < D / 4; ++i) {
      const int at = (tid / D + 256 / D * i) * D + d;
      a_lds[at] = mine[at] = av[i];
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < ITEMS; ++u) {
    const int r0 = kBlock * block_of(u);
    const bool act = D >= 64 || tid < 4 * D;
    float av[kBlock];
    if constexpr (D >= 64) {
      logarithms(av, r0, 1);
    } else {
#pragma unroll
      for (int i = 0; i < kBlock; ++i) av[i] = a_lds[(r0 + i) * D + d];
    }
    float p = 0.f;
#pragma unroll
    for (int i = kBlock - 1; i >= 0; --i) {
      if (act) {
        if (D >= 64) mine[(r0 + i) * D + d] = av[i];
        k_lds[(r0 + i) * KR + d] = r0 + i < n ? S::to_f32(ks[u][i]) * exp_of_log(p) : 0.f;
      }
      p += av[i];
    }
    if (act) tot[(r0 / kBlock) * D + d] = p;
  }
#pragma unroll
  for (int u = 0; u < kMost; ++u)
    if (16 * u < V) {
      const int i = tid + 256 * u, r = (i * inverse) >> 16, at = 4 * (i - r * per_row);
      *reinterpret_cast<Four<S>*>(v_lds + r * VR + at) = r < n ? vs[u] : Four<S>{};
    }
  if constexpr (kSplit<S>) {
    gla_u16x2 most = {0, 0};
#pragma unroll
    for (int u = 0; u < kMost; ++u)
#pragma unroll
      for (int e = 0; e < 2; ++e) most = __builtin_elementwise_max(most, __builtin_bit_cast(gla_u16x2, vs[u][e] & 0x7fff7fffu));
    const bool odd = __any(max(most[0], most[1]) >= 0x7f80);
    if (lane == 0) odd_lds[w] = odd;
  }
  __syncthreads();
  float* r_out = mine + kChunk * D + D;
  const int vt_n = V / 16, pairs = (vt_n + 1) / 2;
  bool some_odd = false;
  if constexpr (kSplit<S>) some_odd = __builtin_amdgcn_readfirstlane(odd_lds[0] | odd_lds[1] | odd_lds[2] | odd_lds[3]);
  constexpr int SHARE = DT >= 4 ? 1 : 4 / DT;              // waves that share the keys' 16 channels
  for (int dt = w / SHARE; dt < DT; dt += 4 / SHARE) {
    // the decay over the blocks behind each
    const int ch = 16 * dt + c;
    const float t3 = tot[3 * D + ch], t2 = tot[2 * D + ch] + t3, t1 = tot[D + ch] + t2;
    const float m[4] = {exp_of_log(t1), exp_of_log(t2), exp_of_log(t3), 1.f};
    if (w % SHARE == 0 && g == 0) mine[kChunk * D + ch] = exp_of_log(tot[ch] + t1);
    float kj[kBlock];
#pragma unroll
    for (int x = 0; x < kBlock; ++x) kj[x] = k_lds[(kBlock * (x >> 2) + 4 * g + (x & 3)) * KR + ch] * m[x >> 2];
    if constexpr (kSplit<S>) {
      ThreeParts kp[2];
#pragma unroll
      for (int x = 0; x < 2; ++x)
        kp[x] = three_parts(f32x4{kj[8 * x], kj[8 * x + 1], kj[8 * x + 2], kj[8 * x + 3]}, f32x4{kj[8 * x + 4], kj[8 * x + 5], kj[8 * x + 6], kj[8 * x + 7]});
      const T* at = v_lds + (4 * g + (c >> 2)) * VR + 4 * (c & 3);
      for (int vt = w % SHARE; vt < vt_n; vt += SHARE) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const u32x4 v = two_blocks(at + 32 * x * VR + 16 * vt, 2 * VR);
          u32x4 rest = v;
          if (some_odd) rest = finite_only(v);
          acc = mfma_parts(kp[x], v, rest, acc);
        }
        *reinterpret_cast<f32x4*>(r_out + ((int64_t)(dt * vt_n + vt) * 64 + lane) * 4) = acc;
      }
      continue;
    }
    for (int pair = w % SHARE; pair < pairs; pair += SHARE) {
      const TilePair tp(pair, vt_n, c);
      f32x4 acc = {0.f, 0.f, 0.f, 0.f}, acc2 = acc;
#pragma unroll
      for (int x = 0; x < kBlock; ++x) {
        float v0, v1;
        tp.read<S>(v_lds + (kBlock * (x >> 2) + 4 * g + (x & 3)) * VR, v0, v1);
        acc = mfma4(kj[x], v0, acc);
        acc2 = mfma4(kj[x], v1, acc2);
      }
      float* to = r_out + ((int64_t)(dt * vt_n + 2 * pair) * 64 + lane) * 4;
      *reinterpret_cast<f32x4*>(to) = acc;
      if (!tp.alone) *reinterpret_cast<f32x4*>(to + 256) = acc2;
    }
  }
}

// one thread: two neighbouring channels of a value column, over the run's chunks
__global__ __launch_bounds__(256) void gla_chunk_scan_kernel(GlaChunks a) {
  const int D = a.dim, V = a.vdim, vt_n = V / 16;
  const int h = blockIdx.x, b = blockIdx.z;
  const int item = blockIdx.y * 256 + threadIdx.x;         // tile, lane, which two of its four channels
  if (item >= D * V / 2) return;
  const int begin = a.query_start_loc[b], run = a.query_start_loc[b + 1] - begin;
  if (run <= 0) return;
  const int tile = item >> 7, lane = (item >> 1) & 63, g = lane >> 4, c = lane & 15;
  const int d = 16 * (tile / vt_n) + 4 * g + 2 * (item & 1), v = a.paired ? paired_column(tile % vt_n, vt_n, c) : 16 * (tile % vt_n) + c;
  float* st = a.state + (((int64_t)a.state_slots[b] * a.heads + h) * D + d) * V + v;
  f32x2 s = {0.f, 0.f};
  if (a.context_lens[b] > 0) s = f32x2{st[0], st[V]};
  const int chunks = (run + kChunk - 1) / kChunk;
  const int64_t per = chunk_floats(D, V), step = a.heads * per;
  float* p = a.scratch + ((int64_t)(begin / kChunk + b) * a.heads + h) * per + kChunk * D;
  // `ahead` chunks on their way; whole: no more than those, and nothing is asked for behind them.  Whole groups of chunks
  // have no conditions between them, behind which a wait is for everything on its way (64 chunks 23 us instead of 13).
  auto walk = [&](auto ahead, auto whole) __attribute__((always_inline)) {
    constexpr int AHEAD = decltype(ahead)::value;
    f32x2 rv[AHEAD], gv[AHEAD];
    auto fetch = [&](int u, int i) __attribute__((always_inline)) {
      const float* at = p + min(i, chunks - 1) * step;
      gv[u] = *reinterpret_cast<const f32x2*>(at + d);
      rv[u] = *reinterpret_cast<const f32x2*>(at + D + 2 * item);
    };
    auto pass = [&](int u, int i) __attribute__((always_inline)) {
      *reinterpret_cast<f32x2*>(p + i * step + D + 2 * item) = s;            // the chunk's start state
#pragma unroll
      for (int e = 0; e < 2; ++e) s[e] = gv[u][e] * s[e] + rv[u][e];
    };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) fetch(u, u);
    int i = 0;
    if constexpr (!decltype(whole)::value)
      for (; i + AHEAD <= chunks; i += AHEAD)
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
          pass(u, i + u);
          fetch(u, i + u + AHEAD);       // (behind the end a place already overwritten, whose numbers are not used)
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (i + u < chunks) pass(u, i + u);
  };
  // Short runs ask for what they have: 16 runs of one chunk (16 heads of 64 x 128) 9 us, and 24 asking for sixteen chunks each.
  using std::integral_constant;
  if (chunks <= 2)
    walk(integral_constant<int, 2>(), std::true_type());
  else if (chunks <= 5)
    walk(integral_constant<int, 5>(), std::true_type());
  else if (chunks <= 10)
    walk(integral_constant<int, 10>(), std::true_type());
  else
    walk(integral_constant<int, 8>(), std::false_type());
  st[0] = s[0];
  st[V] = s[1];
}

// r *= d in the wave's first n lanes, of which all run: four instructions fewer than a choice of the factor
__device__ __forceinline__ void times_in_lanes_below(int n, f32x4& r, f32x4 d) {
  asm volatile("s_bfm_b64 exec, %8, 0\n\tv_mul_f32 %0, %0, %4\n\tv_mul_f32 %1, %1, %5\n\tv_mul_f32 %2, %2, %6\n\t"
               "v_mul_f32 %3, %3, %7\n\ts_mov_b64 exec, -1"
               : "+&v"(r[0]), "+&v"(r[1]), "+&v"(r[2]), "+&v"(r[3])
               : "v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]), "s"(n));
}

template <class S, int DT>          // DT: dim / 16
__global__ __launch_bounds__(256, DT <= 4 && sizeof(typename S::T) == 2 ? 4 : 2) void gla_chunk_out_kernel(GlaChunks a) {
  using T = typename S::T;
  extern __shared__ __align__(16) float lds[];
  constexpr int D = 16 * DT, KR = D + 4, QR = KR > kAMat ? KR : kAMat, ITEMS = (D + 63) / 64;
  const int V = a.vdim, VR = value_row<S>(V), vt_n = V / 16;
  const int slot = blockIdx.x, h = blockIdx.y;
  int b, chunk;
  if (!find_chunk(a, slot, b, chunk)) return;
  const int run = a.query_start_loc[b + 1] - a.query_start_loc[b];
  const int t0 = a.query_start_loc[b] + chunk * kChunk, n = min(kChunk, run - chunk * kChunk);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15;
  // A wave has a block's 16 rows of queries and then, in their place, of A; keys and values are everyone's.
  float* q_own = lds + kBlock * w * QR;                    // [16][QR]
  float* a_own = q_own;                                    // [16][kAMat]
  float* tot = lds + kChunk * QR;                          // [4][D]
  float* decay_own = tot + 4 * D + kBlock * kBlock * w;    // [16][16]
  float* k_lds = tot + 4 * D + kChunk * kBlock;            // [64][KR], then the values
  T* v_lds = (T*)k_lds;                                    // [64][VR]
  const float* mine = a.scratch + ((int64_t)slot * a.heads + h) * chunk_floats(D, V);
  const float* s_in = mine + kChunk * D + D;

  const int row = tid >> 2, quarter = tid & 3;             // the wave's rows again
  const int64_t t = t0 + min(row, n - 1);
  const bool live = row < n;
  const T* qr = (const T*)a.q + t * a.q_stride + (int64_t)h * D;
  const T* kr = (const T*)a.k + t * a.k_stride + (int64_t)h * D;
  const T* vr = (const T*)a.v + t * a.v_stride + (int64_t)h * V;
  Four<S> q_raw[DT], k_raw[DT], held[8];
  f32x4 av[DT];
  float down[ITEMS][kBlock];                               // a channel's logarithms in the wave's rows
#pragma unroll
  for (int x = 0; x < DT; ++x) {
    q_raw[x] = fetch4<S>(qr + 4 * quarter + 16 * x);
    k_raw[x] = fetch4<S>(kr + 4 * quarter + 16 * x);
    av[x] = *reinterpret_cast<const f32x4*>(mine + row * D + 4 * quarter + 16 * x);
  }
#pragma unroll
  for (int u = 0; u < ITEMS; ++u)
#pragma unroll
    for (int i = 0; i < kBlock; ++i) down[u][i] = mine[(kBlock * w + i) * D + (lane + 64 * u) % D];
#pragma unroll
  for (int x = 0; x < 8; ++x) held[x] = fetch4<S>(vr + 4 * quarter + 16 * min(x, vt_n - 1));
  const float norm_mine = a.norm_weight[min(tid, V - 1)];
  __builtin_amdgcn_sched_barrier(0);
  f32x4 kv[DT];
#pragma unroll
  for (int x = 0; x < DT; ++x) {
    const int at = 4 * quarter + 16 * x;
    f32x4 qv = numbers<S>(q_raw[x]);
    kv[x] = numbers<S>(k_raw[x]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      qv[e] = live ? qv[e] * a.q_scale : 0.f;
      if (!live) kv[x][e] = 0.f;
    }
    *reinterpret_cast<f32x4*>(q_own + (lane >> 2) * QR + at) = qv;
    *reinterpret_cast<f32x4*>(k_lds + row * KR + at) = kv[x];
  }

  // A inside the block: lane (j, part) decays a quarter of k_j's channels row by row, 16 channels at a time
  const int j = lane >> 2, part = lane & 3;
  float dot[kBlock];
#pragma unroll
  for (int i = 0; i < kBlock; ++i) dot[i] = 0.f;
#pragma unroll
  for (int x = 0; x < DT; ++x) {
    wave_sync();
    *reinterpret_cast<f32x4*>(decay_own + j * kBlock + 4 * part) =
        f32x4{exp_of_log(av[x][0]), exp_of_log(av[x][1]), exp_of_log(av[x][2]), exp_of_log(av[x][3])};
    wave_sync();
    f32x4 r = kv[x];
#pragma unroll
    for (int i = 0; i < kBlock; ++i) {
      const f32x4 dv = *reinterpret_cast<const f32x4*>(decay_own + i * kBlock + 4 * part);
      const f32x4 qv = *reinterpret_cast<const f32x4*>(q_own + i * QR + 4 * part + 16 * x);
      if (i > 0) times_in_lanes_below(4 * i, r, dv);       // j < i
#pragma unroll
      for (int e = 0; e < 4; ++e) dot[i] += qv[e] * r[e];
    }
  }
  float inside[4];                                         // of rows part, part + 4, ..
#pragma unroll
  for (int i = 0; i < kBlock; i += 2) group_sums(dot[i], dot[i + 1], 4);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float x = part & 2 ? (part & 1 ? dot[4 * u + 3] : dot[4 * u + 2]) : (part & 1 ? dot[4 * u + 1] : dot[4 * u]);
    inside[u] = 4 * u + part >= j ? x : 0.f;
  }

  // queries times the decays from their block's start, keys times those to their block's end
  wave_sync();
#pragma unroll
  for (int u = 0; u < ITEMS; ++u) {
    const int ch = lane + 64 * u;
    if (ch < D) {
      float p = 0.f;
#pragma unroll
      for (int i = 0; i < kBlock; ++i) {
        p += down[u][i];
        q_own[i * QR + ch] *= exp_of_log(p);
      }
      tot[w * D + ch] = p;
      p = 0.f;
#pragma unroll
      for (int i = kBlock - 1; i >= 0; --i) {
        k_lds[(kBlock * w + i) * KR + ch] *= exp_of_log(p);
        p += down[u][i];
      }
    }
  }
  wave_sync();
  f32x4 qs[DT];
#pragma unroll
  for (int x = 0; x < DT; ++x) qs[x] = *reinterpret_cast<const f32x4*>(q_own + c * QR + 16 * x + 4 * g);
  wave_sync();
#pragma unroll
  for (int u = 0; u < 4; ++u) a_own[(4 * u + part) * kAMat + kBlock * w + j] = inside[u];
  __syncthreads();

  // the wave's rows against the blocks before them, and the product over those blocks for the start state
  f32x4 before[DT];
#pragma unroll
  for (int x = 0; x < DT; ++x) before[x] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int o = w - 1; o >= 0; --o) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < DT; ++x) {
      const f32x4 kv = *reinterpret_cast<const f32x4*>(k_lds + (kBlock * o + c) * KR + 16 * x + 4 * g);
      const f32x4 tv = *reinterpret_cast<const f32x4*>(tot + o * D + 16 * x + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc = mfma4(o == w - 1 ? qs[x][e] : qs[x][e] * exp_of_log(before[x][e]), kv[e], acc);
        before[x][e] += tv[e];
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) a_own[(4 * g + e) * kAMat + kBlock * o + c] = acc[e];
  }
  if (w > 0) {
#pragma unroll
    for (int x = 0; x < DT; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) qs[x][e] *= exp_of_log(before[x][e]);
  }
  // the start state of a tile of columns is asked for a tile ahead
  f32x4 sv[2][DT];
  auto fetch_state = [&](int vt) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < DT; ++x) sv[vt & 1][x] = *reinterpret_cast<const f32x4*>(s_in + ((int64_t)(x * vt_n + vt) * 64 + lane) * 4);
  };
  fetch_state(0);
  // the values take the keys' place, the norm's weights that of the decays inside the blocks
  float* norm = tot + 4 * D;
  if (tid < V) norm[tid] = norm_mine;
  __syncthreads();
  bool odd = false;
#pragma unroll
  for (int x = 0; x < 8; ++x)
    if (16 * x < V) {
      const Four<S> put = live ? held[x] : Four<S>{};
      *reinterpret_cast<Four<S>*>(v_lds + row * VR + 4 * quarter + 16 * x) = put;
      const f32x4 num = numbers<S>(put);
#pragma unroll
      for (int e = 0; e < 4; ++e) odd |= !finite(num[e]);
    }
  const bool some_bad = __syncthreads_or(odd);

  // Results leave through LDS, eight neighbouring columns of a row to a lane, where the rows of gates and results allow
  // it (16-bit types).  Gates and norm weights are there ahead of the stores: a load behind a store that may write the same
  // place waits for it.
  const bool wide = sizeof(T) == 2 && a.gate_stride % 8 == 0 && a.out_stride % 8 == 0 &&
                    (uintptr_t)a.gate % 16 == 0 && (uintptr_t)a.out % 16 == 0;
  constexpr int PIECES = 4;                                // 16 rows of 16 pieces over 64 lanes
  u32x4 gates[PIECES];
  const int row_of = lane >> 3, col_of = 8 * (lane & 7);   // of half the columns: rows row_of and row_of + 8
  if (wide) {
#pragma unroll
    for (int u = 0; u < PIECES; ++u) {
      const int i = min(kBlock * w + row_of + 8 * (u & 1), n - 1), col = 64 * (u >> 1) + col_of;
      if (col < V) gates[u] = *reinterpret_cast<const u32x4*>((const T*)a.gate + (int64_t)(t0 + i) * a.gate_stride + (int64_t)h * V + col);
    }
  }

  f32x4 acc[8];
  float ss[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (kSplit<S>) {
    // the wave's rows of A over one or two pairs of blocks; zeros behind its own block, which the values there meet
    const bool two = w >= 2;
    ThreeParts ap[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
      const f32x4 a0 = *reinterpret_cast<const f32x4*>(a_own + c * kAMat + 32 * x + 4 * g), a1 = *reinterpret_cast<const f32x4*>(a_own + c * kAMat + 32 * x + 16 + 4 * g);
      if (x == 0 || two) ap[x] = three_parts(2 * x <= w ? a0 : zero, 2 * x + 1 <= w ? a1 : zero);
    }
    const T* at = v_lds + (4 * g + (c >> 2)) * VR + 4 * (c & 3);
    // (behind all of these where registers are for four workgroups a CU; for two, tile by tile)
    auto with_state = [&](int vt) __attribute__((always_inline)) {
      if (vt + 1 < vt_n) fetch_state(vt + 1);
#pragma unroll
      for (int x = 0; x < DT; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[vt] = mfma4(qs[x][e], sv[vt & 1][x][e], acc[vt]);
#pragma unroll
      for (int e = 0; e < 4; ++e) ss[e] += acc[vt][e] * acc[vt][e];
    };
#pragma unroll
    for (int vt = 0; vt < 8; ++vt) {
      acc[vt] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (vt < vt_n) {
        u32x4 v0 = two_blocks(at + 16 * vt, 2 * VR), v1 = v0;
        if (two) v1 = two_blocks(at + 32 * VR + 16 * vt, 2 * VR);
        // A row's product with the rows behind it is 0 times their values, which must be finite for that; and a column
        // in which one was not stays so, as it does in the state of a walk.
        int bad = kBlock;                                  // the block's first such row in the lane's column
        if (some_bad) {
          for (int i = kBlock * (w + 1) - 1; i >= 0; --i)
            if (!finite(S::to_f32(v_lds[i * VR + 16 * vt + c]))) bad = max(i - kBlock * w, 0);
          v0 = finite_only(v0);
          v1 = finite_only(v1);
        }
        acc[vt] = mfma_parts(ap[0], v0, v0, acc[vt]);
        if (two) acc[vt] = mfma_parts(ap[1], v1, v1, acc[vt]);
        if (some_bad) {
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[vt][e] = 4 * g + e < bad ? acc[vt][e] : NAN;
        }
        if constexpr (DT > 4) with_state(vt);
      }
    }
    if constexpr (DT <= 4) {
#pragma unroll
      for (int vt = 0; vt < 8; ++vt)
        if (vt < vt_n) with_state(vt);
    }
  } else {
#pragma unroll
  for (int pair = 0; pair < 4; ++pair) {
    acc[2 * pair] = acc[2 * pair + 1] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (2 * pair < vt_n) {
      const TilePair tp(pair, vt_n, c);
      auto two = [&](int at, float& x, float& y) __attribute__((always_inline)) { tp.read<S>(v_lds + at * VR, x, y); };
      for (int o = 0; o < w; ++o) {
        const f32x4 am = *reinterpret_cast<const f32x4*>(a_own + c * kAMat + kBlock * o + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float v0, v1;
          two(kBlock * o + 4 * g + e, v0, v1);
          acc[2 * pair] = mfma4(am[e], v0, acc[2 * pair]);
          acc[2 * pair + 1] = mfma4(am[e], v1, acc[2 * pair + 1]);
        }
      }
      // A row's product with the rows behind it is 0 times their values, which must be finite for that; and a column
      // in which one was not stays so, as it does in the state of a walk.
      int bad[2] = {kBlock, kBlock};                       // the block's first such row in the lane's columns
      if (some_bad) {
        for (int i = kBlock * (w + 1) - 1; i >= 0; --i) {
          float v0, v1;
          two(i, v0, v1);
          if (!finite(v0)) bad[0] = max(i - kBlock * w, 0);
          if (!finite(v1)) bad[1] = max(i - kBlock * w, 0);
        }
      }
      const f32x4 am = *reinterpret_cast<const f32x4*>(a_own + c * kAMat + kBlock * w + 4 * g);
      f32x4 v0, v1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float x, y;
        two(kBlock * w + 4 * g + e, x, y);
        v0[e] = x;
        v1[e] = y;
      }
      if (some_bad) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v0[e] = 4 * g + e < bad[0] ? v0[e] : 0.f;
          v1[e] = 4 * g + e < bad[1] ? v1[e] : 0.f;
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[2 * pair] = mfma4(am[e], v0[e], acc[2 * pair]);
        acc[2 * pair + 1] = mfma4(am[e], v1[e], acc[2 * pair + 1]);
      }
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int vt = 2 * pair + half;
        if (vt < vt_n) {
          if (vt + 1 < vt_n) fetch_state(vt + 1);
#pragma unroll
          for (int x = 0; x < DT; ++x)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[vt] = mfma4(qs[x][e], sv[half][x][e], acc[vt]);
          if (some_bad) {
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[vt][e] = 4 * g + e < bad[half] ? acc[vt][e] : NAN;
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) ss[e] += acc[vt][e] * acc[vt][e];
        }
      }
    }
  }
  }
  group_sums(ss[0], ss[1], 16);
  group_sums(ss[2], ss[3], 16);
  // lane: its columns of rows 16 w + 4 g .. + 3
  float inv[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) inv[e] = a.out_scale / sqrtf(ss[e] / (float)V + a.eps);
  if constexpr (sizeof(T) == 2) {
    if (wide) {
      float* own = a_own;                                  // the wave's rows of A, which it alone reads and has read
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        if (64 * half >= V) break;
        wave_sync();
#pragma unroll
        for (int vt = 4 * half; vt < 4 * half + 4; ++vt)
          if (vt < vt_n)
#pragma unroll
            for (int e = 0; e < 4; ++e) own[(4 * g + e) * kAMat + tile_column<S>(vt, vt_n, c) - 64 * half] = acc[vt][e] * inv[e] * norm[tile_column<S>(vt, vt_n, c)];
        wave_sync();
#pragma unroll
        for (int r8 = 0; r8 < 2; ++r8) {
          const int r = row_of + 8 * r8, i = kBlock * w + r, col = 64 * half + col_of;
          if (i >= n || col >= V) continue;
          const f32x4 x0 = *reinterpret_cast<const f32x4*>(own + r * kAMat + col_of), x1 = *reinterpret_cast<const f32x4*>(own + r * kAMat + col_of + 4);
          const u32x4 gw = gates[2 * half + r8];
          float gv[8];
          u32x4 res;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            gv[2 * k] = lo16<S>(gw[k]);
            gv[2 * k + 1] = hi16<S>(gw[k]);
          }
          silu(gv);
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float y0 = 2 * k < 4 ? x0[2 * k & 3] : x1[2 * k & 3], y1 = 2 * k < 4 ? x0[(2 * k + 1) & 3] : x1[(2 * k + 1) & 3];
            res[k] = pack16<S>(y0 * gv[2 * k], y1 * gv[2 * k + 1]);
          }
          *reinterpret_cast<u32x4*>((T*)a.out + (int64_t)(t0 + i) * a.out_stride + (int64_t)h * V + col) = res;
        }
      }
      return;
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int i = kBlock * w + 4 * g + e;
    if (i >= n) continue;
    const T* gr = (const T*)a.gate + (int64_t)(t0 + i) * a.gate_stride + (int64_t)h * V;
    T* to = (T*)a.out + (int64_t)(t0 + i) * a.out_stride + (int64_t)h * V;
    float gt[8];
#pragma unroll
    for (int vt = 0; vt < 8; ++vt)
      if (vt < vt_n) gt[vt] = S::to_f32(gr[tile_column<S>(vt, vt_n, c)]);
#pragma unroll
    for (int vt = 0; vt < 8; ++vt)
      if (vt < vt_n) to[tile_column<S>(vt, vt_n, c)] = S::from_f32(acc[vt][e] * inv[e] * norm[tile_column<S>(vt, vt_n, c)] * (gt[vt] / (1.f + expf(-gt[vt]))));
  }
}

bool chunk_sizes(int dim, int vdim, int rank) {
  return dim >= 16 && dim <= kMaxDim && (dim & (dim - 1)) == 0 && vdim >= 16 && vdim <= 128 && vdim % 16 == 0 && rank > 0 &&
         rank <= kMaxRank;
}
int64_t chunk_slots(int num_tokens, int num_seqs) { return (int64_t)num_tokens / kChunk + num_seqs; }

template <class S, int DT>
int launch_chunks(const GlaChunks& a, int num_tokens, dim3 grid, hipStream_t stream) {
  constexpr int D = 16 * DT;
  static std::atomic<uint64_t> raised{0}, raised_out{0};
  auto spread = [&](size_t lds) { return spread_lds(lds, pieces_at_most(num_tokens, a.num_seqs, kChunk) * a.heads); };
  const size_t values = sizeof(typename S::T) * (size_t)kChunk * value_row<S>(a.vdim);
  const size_t lds = spread(sizeof(float) * ((size_t)kChunk * (D + 4 + (a.rank + 3) / 4 * 4 + (D < 64 ? D : 0)) + 4 * D + 4) + values);
  if (const int rc = raise_lds(&gla_chunk_state_kernel<S, DT>, lds, raised)) return rc;
  gla_chunk_state_kernel<S, DT><<<grid, 256, lds, stream>>>(a);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  gla_chunk_scan_kernel<<<dim3(a.heads, (D * a.vdim / 2 + 255) / 256, a.num_seqs), 256, 0, stream>>>(a);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  const size_t keys = sizeof(float) * (size_t)kChunk * (D + 4);
  const size_t lds_out = spread(sizeof(float) * ((size_t)kChunk * (D + 4 > kAMat ? D + 4 : kAMat) + 4 * D + kChunk * kBlock) + (keys > values ? keys : values));
  if (const int rc = raise_lds(&gla_chunk_out_kernel<S, DT>, lds_out, raised_out)) return rc;
  gla_chunk_out_kernel<S, DT><<<grid, 256, lds_out, stream>>>(a);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  return VLA_OK;
}

}  // namespace
}  // namespace seq
}  // namespace vla

using namespace vla;
using namespace vla::seq;

// 0 where the sizes do not fit, a launch has no room for the sequences or heads, or the chunks would want more than 4 GiB
extern "C" int64_t vla_seq_gla_chunks_scratch_floats(int num_tokens, int num_seqs, int heads, int dim, int vdim, int rank) {
  if (num_tokens <= 0 || num_seqs <= 0 || num_seqs > 65535 || heads <= 0 || heads > 65535 ||
      !chunk_sizes(dim, vdim, rank))
    return 0;
  const int64_t need = chunk_slots(num_tokens, num_seqs) * heads * chunk_floats(dim, vdim);
  return need <= ((int64_t)1 << 30) ? need : 0;
}

extern "C" int vla_seq_gla_chunks(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k,
                                  int64_t k_stride, const void* v, int64_t v_stride, const void* gate,
                                  int64_t gate_stride, const void* y, int64_t y_stride, const void* w2,
                                  const float* bias, const float* norm_weight, float* state,
                                  const int* query_start_loc, const int* context_lens, const int* state_slots,
                                  int num_tokens, int num_seqs, int num_slots, int heads, int dim, int vdim,
                                  int rank, float q_scale, float inv_tau, float eps, float out_scale,
                                  float* scratch, int64_t scratch_floats, int dtype, void* stream) {
  if (num_tokens == 0 || num_seqs == 0) return VLA_OK;
  if (!out || !q || !k || !v || !gate || !y || !w2 || !norm_weight || !state || !query_start_loc || !context_lens ||
      !state_slots || !scratch || num_tokens < 0 || num_seqs < 0 || num_seqs > 65535 || num_slots <= 0 || heads <= 0 ||
      heads > 65535 || q_stride < (int64_t)heads * dim || k_stride < (int64_t)heads * dim ||
      v_stride < (int64_t)heads * vdim || gate_stride < (int64_t)heads * vdim || out_stride < (int64_t)heads * vdim ||
      y_stride < rank)
    return VLA_ERR_ARG;
  if (!chunk_sizes(dim, vdim, rank)) return VLA_ERR_HEAD_SIZE;
  const int64_t need = vla_seq_gla_chunks_scratch_floats(num_tokens, num_seqs, heads, dim, vdim, rank);
  if (need == 0 || scratch_floats < need || (uintptr_t)scratch % 16) return VLA_ERR_ARG;
  const int quad = dtype == VLA_F32 ? 16 : 8;
  for (const void* p : {q, k, v})
    if ((uintptr_t)p % quad) return VLA_ERR_ARG;
  if (q_stride % 4 || k_stride % 4 || v_stride % 4) return VLA_ERR_ARG;
  const GlaChunks a{out, out_stride, q, q_stride, k, k_stride, v, v_stride, gate, gate_stride, y, y_stride, w2, bias,
                    norm_weight, state, scratch, query_start_loc, context_lens, state_slots, num_seqs, heads, dim, vdim,
                    rank, q_scale, inv_tau, eps, out_scale, dtype != VLA_BF16};
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)chunk_slots(num_tokens, num_seqs), heads);
  return with_dtype(dtype, [&](auto s) -> int {
    using S = decltype(s);
    switch (dim / 16) {
      case 1: return launch_chunks<S, 1>(a, num_tokens, grid, st);
      case 2: return launch_chunks<S, 2>(a, num_tokens, grid, st);
      case 4: return launch_chunks<S, 4>(a, num_tokens, grid, st);
      default: return launch_chunks<S, 8>(a, num_tokens, grid, st);
    }
  });
}
