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
// All products run on 16x16x4 fp32 matrix cores.  Operands that later kernels read lie in scratch lane for
// lane.  Bound by memory and the launches: 4096 rows of 16 heads of 64 x 128 are 68 MB in and out and 100 MB
// of chunk states and decays; 123 us per call (42 + 23 + 66 under the tracer) where the pieces of 256 rows walked
// token by token and joined by matrix products took 408.  What a workgroup's 19 and 29 us go to: waits for its rows
// (4 and 5), products (7 and 9), decays (6 and 5), the products inside a block (4), gates and stores (5).  Rows are
// asked for together and made numbers afterwards, start states a tile of columns ahead (130 us where values and W2
// were each waited for behind a condition of their own, and keys, values and y in turn).
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
template <class S>
__device__ __forceinline__ f32x4 row4(const typename S::T* p) {
  return numbers<S>(fetch4<S>(p));
}

// exp(p) for p <= 0 (NaN passes): 2^n 2^f with the argument's rounding in f.  expf without what other p need, the same
// error: 2.62e-8 root mean square over -87 .. 0, 8.4e-8 at most.
__device__ __forceinline__ float exp_of_log(float p) {
#pragma clang fp contract(off)
  p = p < -150.f ? -150.f : p;
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

template <class S, int DT>          // DT: dim / 16
__global__ __launch_bounds__(256) void gla_chunk_state_kernel(GlaChunks a) {
  using T = typename S::T;
  extern __shared__ __align__(16) float lds[];
  constexpr int D = 16 * DT, KR = D + 4;
  const int V = a.vdim, R = a.rank, VR = V + 4;
  float* k_lds = lds;                       // [64][KR]
  float* a_lds = k_lds + kChunk * KR;       // [64][D]
  float* v_lds = a_lds + kChunk * D;        // [64][VR]
  float* y_lds = v_lds + kChunk * VR;       // [64][R padded to 4]
  float* tot = y_lds + kChunk * kMaxRank;   // [4][D]: a block's sum of logarithms
  const int slot = blockIdx.x, h = blockIdx.y;
  int b, chunk;
  if (!find_chunk(a, slot, b, chunk)) return;
  const int run = a.query_start_loc[b + 1] - a.query_start_loc[b];
  const int t0 = a.query_start_loc[b] + chunk * kChunk, n = min(kChunk, run - chunk * kChunk);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int RP = (R + 3) / 4 * 4;
  float* mine = a.scratch + ((int64_t)slot * a.heads + h) * chunk_floats(D, V);

  // rows behind the run's end are zeros; every load is on its way before the first is waited for
  const int row = tid >> 2, quarter = tid & 3;
  const int64_t t = t0 + min(row, n - 1);
  const int d_mine = tid % D;                // the thread's decay channel and its row of W2, on its way with the rows
  constexpr int PER = 16 / sizeof(T);
  const bool w_wide = R % PER == 0 && (uintptr_t)a.w2 % 16 == 0;
  u32x4 w_row[kMaxRank / PER];
  float wv[kMaxRank];
  const T* wr = (const T*)a.w2 + ((int64_t)h * D + d_mine) * R;
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
  const float bias = a.bias != nullptr ? a.bias[(int64_t)h * D + d_mine] : 0.f;
  T ys[kMaxRank / 4];
#pragma unroll
  for (int u = 0; u < kMaxRank / 4; ++u) ys[u] = ((const T*)a.y)[t * a.y_stride + min(quarter + 4 * u, R - 1)];
  // four values a thread, in the order they lie in: D / 16 and V / 16 of them, whole for all threads
  constexpr int kMost = 8;
  Four<S> ks[DT], vs[kMost];
  const int per_row = V / 4, inverse = (65536 + per_row - 1) / per_row;      // (i * inverse) >> 16 is i / per_row below 2048
#pragma unroll
  for (int u = 0; u < DT; ++u) {
    const int i = tid + 256 * u, r = i / (D / 4), d = 4 * (i % (D / 4));
    ks[u] = fetch4<S>((const T*)a.k + (t0 + min(r, n - 1)) * a.k_stride + (int64_t)h * D + d);
  }
#pragma unroll
  for (int u = 0; u < kMost; ++u) {
    const int i = tid + 256 * min(u, V / 16 - 1), r = (i * inverse) >> 16, d = 4 * (i - r * per_row);
    vs[u] = fetch4<S>((const T*)a.v + (t0 + min(r, n - 1)) * a.v_stride + (int64_t)h * V + d);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < kMaxRank / 4; ++u)
    if (4 * u < RP) y_lds[row * kMaxRank + quarter + 4 * u] = quarter + 4 * u < R ? S::to_f32(ys[u]) : 0.f;
#pragma unroll
  for (int u = 0; u < DT; ++u) {
    const int i = tid + 256 * u, r = i / (D / 4), d = 4 * (i % (D / 4));
    *reinterpret_cast<f32x4*>(k_lds + r * KR + d) = r < n ? numbers<S>(ks[u]) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int u = 0; u < kMost; ++u)
    if (16 * u < V) {
      const int i = tid + 256 * u, r = (i * inverse) >> 16, d = 4 * (i - r * per_row);
      *reinterpret_cast<f32x4*>(v_lds + r * VR + d) = r < n ? numbers<S>(vs[u]) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  __syncthreads();

  // decays: a thread keeps its channel's row of W2 and walks every (256 / D)-th row
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
  for (int i = tid / D; i < kChunk; i += 256 / D) {
    float z = bias;
#pragma unroll
    for (int r4 = 0; r4 < kMaxRank; r4 += 4) {
      if (r4 >= RP) break;
      const f32x4 yv = *reinterpret_cast<const f32x4*>(y_lds + i * kMaxRank + r4);
#pragma unroll
      for (int e = 0; e < 4; ++e) z += wv[r4 + e] * yv[e];
    }
    const float ld = log_sigmoid(z) * a.inv_tau;
    a_lds[i * D + d_mine] = i < n ? ld : 0.f;
    mine[i * D + d_mine] = i < n ? ld : 0.f;
  }
  __syncthreads();

  // keys times the decays behind them: inside a block of 16 rows first, then the later blocks' products
  for (int item = tid; item < 4 * D; item += 256) {
    const int seg = item / D, d = item - seg * D;
    float av[kBlock];
#pragma unroll
    for (int i = 0; i < kBlock; ++i) av[i] = a_lds[(kBlock * seg + i) * D + d];
    float p = 0.f;
#pragma unroll
    for (int i = kBlock - 1; i >= 0; --i) {
      k_lds[(kBlock * seg + i) * KR + d] *= exp_of_log(p);
      p += av[i];
    }
    tot[seg * D + d] = p;
  }
  __syncthreads();
  for (int d = tid; d < D; d += 256) {
    const float t3 = tot[3 * D + d], t2 = tot[2 * D + d] + t3, t1 = tot[D + d] + t2;
    mine[kChunk * D + d] = exp_of_log(tot[d] + t1);
    // from here on: the decay over the blocks behind each
    tot[d] = exp_of_log(t1);
    tot[D + d] = exp_of_log(t2);
    tot[2 * D + d] = exp_of_log(t3);
    tot[3 * D + d] = 1.f;
  }
  __syncthreads();
  float* r_out = mine + kChunk * D + D;
  const int dt_n = D / 16, vt_n = V / 16;
  const int pairs = (vt_n + 1) / 2;            // two value tiles share the reads of the keys
  for (int item = w; item < dt_n * pairs; item += 4) {
    const int dt = item / pairs, vt = 2 * (item - dt * pairs), vt2 = min(vt + 1, vt_n - 1);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f}, acc2 = acc;
#pragma unroll
    for (int seg = 0; seg < 4; ++seg) {
      const float m = tot[seg * D + 16 * dt + c];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = kBlock * seg + 4 * g + e;
        const float kj = k_lds[j * KR + 16 * dt + c] * m;
        acc = mfma4(kj, v_lds[j * VR + 16 * vt + c], acc);
        acc2 = mfma4(kj, v_lds[j * VR + 16 * vt2 + c], acc2);
      }
    }
    *reinterpret_cast<f32x4*>(r_out + ((int64_t)(dt * vt_n + vt) * 64 + lane) * 4) = acc;
    if (vt2 != vt) *reinterpret_cast<f32x4*>(r_out + ((int64_t)(dt * vt_n + vt2) * 64 + lane) * 4) = acc2;
  }
}

// one thread: four neighbouring channels of a value column, over the run's chunks
__global__ __launch_bounds__(256) void gla_chunk_scan_kernel(GlaChunks a) {
  const int D = a.dim, V = a.vdim, vt_n = V / 16;
  const int h = blockIdx.x, b = blockIdx.z;
  const int item = blockIdx.y * 256 + threadIdx.x;         // tile, lane
  if (item >= D * V / 4) return;
  const int begin = a.query_start_loc[b], run = a.query_start_loc[b + 1] - begin;
  if (run <= 0) return;
  const int tile = item >> 6, lane = item & 63, g = lane >> 4, c = lane & 15;
  const int d = 16 * (tile / vt_n) + 4 * g, v = 16 * (tile % vt_n) + c;
  float* st = a.state + (((int64_t)a.state_slots[b] * a.heads + h) * D + d) * V + v;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  if (a.context_lens[b] > 0)
    s = f32x4{st[0], st[V], st[2 * V], st[3 * V]};
  const int chunks = (run + kChunk - 1) / kChunk;
  const int64_t per = chunk_floats(D, V), step = a.heads * per;
  float* p = a.scratch + ((int64_t)(begin / kChunk + b) * a.heads + h) * per + kChunk * D;
  constexpr int AHEAD = 8;
  f32x4 rv[AHEAD], gv[AHEAD];
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) {
    const float* at = p + min(u, chunks - 1) * step;
    gv[u] = *reinterpret_cast<const f32x4*>(at + d);
    rv[u] = *reinterpret_cast<const f32x4*>(at + D + 4 * item);
  }
  for (int i = 0; i < chunks; i += AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (i + u < chunks) {
        *reinterpret_cast<f32x4*>(p + (i + u) * step + D + 4 * item) = s;    // the chunk's start state
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = gv[u][e] * s[e] + rv[u][e];
        const float* at = p + min(i + u + AHEAD, chunks - 1) * step;
        // (behind the end this is a place already overwritten, and what it gives is not used)
        gv[u] = *reinterpret_cast<const f32x4*>(at + d);
        rv[u] = *reinterpret_cast<const f32x4*>(at + D + 4 * item);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) st[e * V] = s[e];
}

template <class S, int DT>          // DT: dim / 16
__global__ __launch_bounds__(256) void gla_chunk_out_kernel(GlaChunks a) {
  using T = typename S::T;
  extern __shared__ __align__(16) float lds[];
  constexpr int D = 16 * DT, KR = D + 4;
  const int V = a.vdim, VR = V + 4, vt_n = V / 16;
  float* q_lds = lds;                                      // [64][KR]
  float* a_mat = q_lds + kChunk * KR;                      // [64][kAMat]
  float* tot = a_mat + kChunk * kAMat;                     // [4][D]
  float* k_lds = tot + 4 * D;                              // [64][KR], later v [64][VR] from here on
  float* a_lds = k_lds + kChunk * KR;                      // [64][D]
  float* v_lds = k_lds;
  const int slot = blockIdx.x, h = blockIdx.y;
  int b, chunk;
  if (!find_chunk(a, slot, b, chunk)) return;
  const int run = a.query_start_loc[b + 1] - a.query_start_loc[b];
  const int t0 = a.query_start_loc[b] + chunk * kChunk, n = min(kChunk, run - chunk * kChunk);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15;
  const float* mine = a.scratch + ((int64_t)slot * a.heads + h) * chunk_floats(D, V);
  const float* s_in = mine + kChunk * D + D;

  const int row = tid >> 2, quarter = tid & 3;
  const int64_t t = t0 + min(row, n - 1);
  const bool live = row < n;
  const T* qr = (const T*)a.q + t * a.q_stride + (int64_t)h * D;
  const T* kr = (const T*)a.k + t * a.k_stride + (int64_t)h * D;
  const T* vr = (const T*)a.v + t * a.v_stride + (int64_t)h * V;
  {
    f32x4 qv[DT], kv[DT], av[DT];
#pragma unroll
    for (int x = 0; x < DT; ++x) {
      const int d = 4 * quarter + 16 * x;
      qv[x] = row4<S>(qr + d);
      kv[x] = row4<S>(kr + d);
      av[x] = *reinterpret_cast<const f32x4*>(mine + row * D + d);
    }
#pragma unroll
    for (int x = 0; x < DT; ++x) {
      const int d = 4 * quarter + 16 * x;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        qv[x][e] = live ? qv[x][e] * a.q_scale : 0.f;
        if (!live) kv[x][e] = 0.f;
      }
      *reinterpret_cast<f32x4*>(q_lds + row * KR + d) = qv[x];
      *reinterpret_cast<f32x4*>(k_lds + row * KR + d) = kv[x];
      *reinterpret_cast<f32x4*>(a_lds + row * D + d) = f32x4{exp_of_log(av[x][0]), exp_of_log(av[x][1]), exp_of_log(av[x][2]), exp_of_log(av[x][3])};
    }
  }
  __syncthreads();

  // A inside the wave's block of 16 rows: lane (j, part) decays a quarter of k_j's channels row by row
  {
    const int j = lane >> 2, part = lane & 3, r0 = kBlock * w;
    f32x4 r[DT];
#pragma unroll
    for (int x = 0; x < DT; ++x) r[x] = *reinterpret_cast<const f32x4*>(k_lds + (r0 + j) * KR + 4 * part + 16 * x);
#pragma unroll 4
    for (int i = 0; i < kBlock; ++i) {
      float dot = 0.f, none = 0.f;
#pragma unroll
      for (int x = 0; x < DT; ++x) {
        const f32x4 av = *reinterpret_cast<const f32x4*>(a_lds + (r0 + i) * D + 4 * part + 16 * x);
        const f32x4 qv = *reinterpret_cast<const f32x4*>(q_lds + (r0 + i) * KR + 4 * part + 16 * x);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          r[x][e] *= i > j ? av[e] : 1.f;
          dot += qv[e] * r[x][e];
        }
      }
      group_sums(dot, none, 4);
      if (part == 0) a_mat[(r0 + i) * kAMat + r0 + j] = i >= j ? dot : 0.f;
    }
  }
  __syncthreads();

  // queries times the decays from their block's start, keys times those to their block's end
  for (int item = tid; item < 4 * D; item += 256) {
    const int seg = item / D, d = item - seg * D;
    float av[kBlock];
#pragma unroll
    for (int i = 0; i < kBlock; ++i) av[i] = mine[(kBlock * seg + i) * D + d];
    float p = 0.f;
#pragma unroll
    for (int i = 0; i < kBlock; ++i) {
      p += av[i];
      q_lds[(kBlock * seg + i) * KR + d] *= exp_of_log(p);
    }
    tot[seg * D + d] = p;
    p = 0.f;
#pragma unroll
    for (int i = kBlock - 1; i >= 0; --i) {
      k_lds[(kBlock * seg + i) * KR + d] *= exp_of_log(p);
      p += av[i];
    }
  }
  __syncthreads();

  // the wave's rows against the blocks before them, and the product over those blocks for the start state
  f32x4 before[DT];
#pragma unroll
  for (int x = 0; x < DT; ++x) before[x] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int o = w - 1; o >= 0; --o) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < DT; ++x) {
      const f32x4 qv = *reinterpret_cast<const f32x4*>(q_lds + (kBlock * w + c) * KR + 16 * x + 4 * g);
      const f32x4 kv = *reinterpret_cast<const f32x4*>(k_lds + (kBlock * o + c) * KR + 16 * x + 4 * g);
      const f32x4 tv = *reinterpret_cast<const f32x4*>(tot + o * D + 16 * x + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc = mfma4(qv[e] * exp_of_log(before[x][e]), kv[e], acc);
        before[x][e] += tv[e];
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) a_mat[(kBlock * w + 4 * g + e) * kAMat + kBlock * o + c] = acc[e];
  }
  // the values take the keys' and the decays' place
  Four<S> held[8];
#pragma unroll
  for (int x = 0; x < 8; ++x)
    if (16 * x < V) held[x] = fetch4<S>(vr + 4 * quarter + 16 * x);
  // the start state of a tile of columns is asked for a tile ahead
  f32x4 sv[2][DT];
  auto fetch_state = [&](int vt) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < DT; ++x) sv[vt & 1][x] = *reinterpret_cast<const f32x4*>(s_in + ((int64_t)(x * vt_n + vt) * 64 + lane) * 4);
  };
  fetch_state(0);
  __syncthreads();
  bool odd = false;
#pragma unroll
  for (int x = 0; x < 8; ++x)
    if (16 * x < V) {
      const f32x4 put = live ? numbers<S>(held[x]) : f32x4{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<f32x4*>(v_lds + row * VR + 4 * quarter + 16 * x) = put;
#pragma unroll
      for (int e = 0; e < 4; ++e) odd |= !finite(put[e]);
    }
  const bool some_bad = __syncthreads_or(odd);

  // Results leave through LDS, eight neighbouring columns of a row to a lane, where the rows of gates and results allow
  // it (16-bit types).  Gates and norm weights are there ahead of the stores: a load behind a store that may write the same
  // place waits for it.
  const bool wide = sizeof(T) == 2 && a.gate_stride % 8 == 0 && a.out_stride % 8 == 0 &&
                    (uintptr_t)a.gate % 16 == 0 && (uintptr_t)a.out % 16 == 0;
  constexpr int PIECES = 4;                                // 16 rows of 16 pieces over 64 lanes
  u32x4 gates[PIECES];
  float norm[8];
  const int row_of = lane >> 3, col_of = 8 * (lane & 7);   // of half the columns: rows row_of and row_of + 8
#pragma unroll
  for (int vt = 0; vt < 8; ++vt)
    if (vt < vt_n) norm[vt] = a.norm_weight[16 * vt + c];
  if (wide) {
#pragma unroll
    for (int u = 0; u < PIECES; ++u) {
      const int i = min(kBlock * w + row_of + 8 * (u & 1), n - 1), col = 64 * (u >> 1) + col_of;
      if (col < V) gates[u] = *reinterpret_cast<const u32x4*>((const T*)a.gate + (int64_t)(t0 + i) * a.gate_stride + (int64_t)h * V + col);
    }
  }

  f32x4 acc[8];
  f32x4 qs[DT];
#pragma unroll
  for (int x = 0; x < DT; ++x) {
    qs[x] = *reinterpret_cast<const f32x4*>(q_lds + (kBlock * w + c) * KR + 16 * x + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) qs[x][e] *= exp_of_log(before[x][e]);
  }
  float ss[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int vt = 0; vt < 8; ++vt) {
    acc[vt] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (vt < vt_n) {
      if (vt + 1 < vt_n) fetch_state(vt + 1);
      for (int o = 0; o < w; ++o) {
        const f32x4 am = *reinterpret_cast<const f32x4*>(a_mat + (kBlock * w + c) * kAMat + kBlock * o + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[vt] = mfma4(am[e], v_lds[(kBlock * o + 4 * g + e) * VR + 16 * vt + c], acc[vt]);
      }
      // A row's product with the rows behind it is 0 times their values, which must be finite for that; and a column
      // in which one was not stays so, as it does in the state of a walk.
      int bad = kBlock;                                    // the block's first such row in column c
      if (some_bad) {
        for (int j = kBlock * (w + 1) - 1; j >= 0; --j)
          if (!finite(v_lds[j * VR + 16 * vt + c])) bad = max(j - kBlock * w, 0);
      }
      const f32x4 am = *reinterpret_cast<const f32x4*>(a_mat + (kBlock * w + c) * kAMat + kBlock * w + 4 * g);
      f32x4 vv;
#pragma unroll
      for (int e = 0; e < 4; ++e) vv[e] = v_lds[(kBlock * w + 4 * g + e) * VR + 16 * vt + c];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[vt] = mfma4(am[e], 4 * g + e < bad ? vv[e] : 0.f, acc[vt]);
#pragma unroll
      for (int x = 0; x < DT; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[vt] = mfma4(qs[x][e], sv[vt & 1][x][e], acc[vt]);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[vt][e] = 4 * g + e < bad ? acc[vt][e] : NAN;
#pragma unroll
      for (int e = 0; e < 4; ++e) ss[e] += acc[vt][e] * acc[vt][e];
    }
  }
  group_sums(ss[0], ss[1], 16);
  group_sums(ss[2], ss[3], 16);
  // lane: column 16 vt + c of rows 16 w + 4 g .. + 3
  float inv[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) inv[e] = a.out_scale / sqrtf(ss[e] / (float)V + a.eps);
  if constexpr (sizeof(T) == 2) {
    if (wide) {
      float* own = a_mat + kBlock * w * kAMat;             // the wave's rows of A, which it alone reads and has read
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        if (64 * half >= V) break;
        wave_sync();
#pragma unroll
        for (int vt = 4 * half; vt < 4 * half + 4; ++vt)
          if (vt < vt_n)
#pragma unroll
            for (int e = 0; e < 4; ++e) own[(4 * g + e) * kAMat + 16 * (vt - 4 * half) + c] = acc[vt][e] * inv[e] * norm[vt];
        wave_sync();
#pragma unroll
        for (int r8 = 0; r8 < 2; ++r8) {
          const int r = row_of + 8 * r8, i = kBlock * w + r, col = 64 * half + col_of;
          if (i >= n || col >= V) continue;
          const f32x4 x0 = *reinterpret_cast<const f32x4*>(own + r * kAMat + col_of), x1 = *reinterpret_cast<const f32x4*>(own + r * kAMat + col_of + 4);
          const u32x4 gw = gates[2 * half + r8];
          u32x4 res;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float g0 = lo16<S>(gw[k]), g1 = hi16<S>(gw[k]);
            const float y0 = 2 * k < 4 ? x0[2 * k & 3] : x1[2 * k & 3], y1 = 2 * k < 4 ? x0[(2 * k + 1) & 3] : x1[(2 * k + 1) & 3];
            res[k] = pack16<S>(y0 * (g0 / (1.f + expf(-g0))), y1 * (g1 / (1.f + expf(-g1))));
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
    const T* gr = (const T*)a.gate + (int64_t)(t0 + i) * a.gate_stride + (int64_t)h * V + c;
    T* to = (T*)a.out + (int64_t)(t0 + i) * a.out_stride + (int64_t)h * V + c;
    float gt[8];
#pragma unroll
    for (int vt = 0; vt < 8; ++vt)
      if (vt < vt_n) gt[vt] = S::to_f32(gr[16 * vt]);
#pragma unroll
    for (int vt = 0; vt < 8; ++vt)
      if (vt < vt_n) to[16 * vt] = S::from_f32(acc[vt][e] * inv[e] * norm[vt] * (gt[vt] / (1.f + expf(-gt[vt]))));
  }
}

bool chunk_sizes(int dim, int vdim, int rank) {
  return dim >= 16 && dim <= kMaxDim && (dim & (dim - 1)) == 0 && vdim >= 16 && vdim <= 128 && vdim % 16 == 0 && rank > 0 &&
         rank <= kMaxRank;
}
int64_t chunk_slots(int num_tokens, int num_seqs) { return (int64_t)num_tokens / kChunk + num_seqs; }

template <class K>
int raise_lds(K kernel, size_t lds, std::atomic<size_t>& allowed) {
  if (lds > allowed.load(std::memory_order_relaxed)) {
    VLA_SEQ_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    allowed.store(lds, std::memory_order_relaxed);
  }
  return VLA_OK;
}

template <class S, int DT>
int launch_chunks(const GlaChunks& a, dim3 grid, hipStream_t stream) {
  constexpr int D = 16 * DT;
  static std::atomic<size_t> allowed{64 * 1024}, allowed_out{64 * 1024};   // raised once per kernel, not per launch
  const size_t lds = sizeof(float) * ((size_t)kChunk * (D + 4 + D + a.vdim + 4 + kMaxRank) + 4 * D);
  if (const int rc = raise_lds(&gla_chunk_state_kernel<S, DT>, lds, allowed)) return rc;
  gla_chunk_state_kernel<S, DT><<<grid, 256, lds, stream>>>(a);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  gla_chunk_scan_kernel<<<dim3(a.heads, (D * a.vdim / 4 + 255) / 256, a.num_seqs), 256, 0, stream>>>(a);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  const size_t keys = (size_t)kChunk * (D + 4 + D), values = (size_t)kChunk * (a.vdim + 4);
  const size_t lds_out = sizeof(float) * ((size_t)kChunk * (D + 4) + kChunk * kAMat + 4 * D + (keys > values ? keys : values));
  if (const int rc = raise_lds(&gla_chunk_out_kernel<S, DT>, lds_out, allowed_out)) return rc;
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
                    rank, q_scale, inv_tau, eps, out_scale};
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)chunk_slots(num_tokens, num_seqs), heads);
  return with_dtype(dtype, [&](auto s) -> int {
    using S = decltype(s);
    switch (dim / 16) {
      case 1: return launch_chunks<S, 1>(a, grid, st);
      case 2: return launch_chunks<S, 2>(a, grid, st);
      case 4: return launch_chunks<S, 4>(a, grid, st);
      default: return launch_chunks<S, 8>(a, grid, st);
    }
  });
}
