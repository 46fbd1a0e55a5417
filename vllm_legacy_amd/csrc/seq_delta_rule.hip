// Gated delta rule: per head a state S [dim, vdim] in fp32 that every token first decays, then
// corrects towards its value along its key, then reads with its query:
//   S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q
// with k and q made unit vectors per head (q also times dim^-1/2), beta = sigmoid(b),
// g = exp(-exp(A_log) softplus(dt + dt_bias)).  The head's o is RMS-normed over vdim, weighted and
// gated with silu before it leaves.  Several value heads may share one query / key head.
//
// One workgroup per (head, sequence, group of value columns) walks the sequence's rows of the step.
// A column of S (one value dimension) never meets another, so a head's columns are spread over
// workgroups, and thread (j, r) keeps R rows of column j in registers -- rows 4 (ii split + r) ..
// + 3 for ii < R / 4, so that the `split` threads of a column, neighbours in a wave, read whole
// lines of the state and of the staged keys -- and they add their partial dot products with lane
// exchanges.  Rows go through LDS in chunks: queries, keys, values and the per-token numbers of a
// chunk are staged and normed together, and the walk then needs no barrier per token.  With
//   dk = S^T k and dq = S^T q taken from the state before the token,
//   u = beta (v - g dk),   o = g dq + (k . q) u,   S <- g S + k u^T
// is the same update with both dot products read from one state.  Steps whose runs have at most
// four rows (decode steps) skip the staging: the lanes of a column read their rows of the query and
// key themselves and the unit norms are lane sums.  The walk leaves o in fp32; a
// second launch norms each head's o over vdim, weighs and gates it.  The state is stored
// [slot, head, vdim, dim], so a thread's rows are contiguous.  Everything is fp32.
//
// Longer runs (heads of at most 256 rows) go in blocks of 32 rows.  With L_ij the product of g over
// rows j + 1 .. i of a block (formed as that product: decays that underflow beside decays of 1 are
// exact) and G_i the one over rows 0 .. i:
//   B_ij = beta_i (k_i . k_j) L_ij  (j < i),   A_ij = (q_i . k_j) L_ij  (j <= i)
//   T = (I + B)^-1 diag(beta)                                            (32 x 32, lower triangular)
//   U = T V - W S,   O = A U + Q~ S      W = T (G k),   Q~ = G q
//   S <- G_31 S + K^^T U                 K^_j = L_31,j k_j
// Everything but the last two lines' products with S and U depends on the block alone:
// delta_block_prepare_kernel forms it for all blocks at once, one workgroup per block and head, and
// leaves W, Q~, K^, G_31, A and T V in scratch; delta_block_walk_kernel goes over a run's blocks in
// order, a workgroup per 16 columns of S, whose rows its four waves share and keep in registers.  All
// products run on 16x16x4 matrix cores: what the preparation forms and K^^T U in 64 bits, those with S in 32.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "seq_common.h"

namespace vla {
namespace seq {
namespace {

constexpr int kMaxChunk = 32;
constexpr int kMaxSplit = 16;

template <class SI>
struct DeltaRows {
  const typename SI::T* q;
  int64_t q_stride;
  const typename SI::T* k;
  int64_t k_stride;
  const typename SI::T* v;
  int64_t v_stride;
  const typename SI::T* gate;
  int64_t gate_stride;
  const typename SI::T* beta;
  int64_t beta_stride;
  const typename SI::T* dt;
  int64_t dt_stride;
};

template <class SI, int R>
__global__ __launch_bounds__(256) void delta_rule_kernel(
    float* __restrict__ o, DeltaRows<SI> in, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, float* __restrict__ state,
    const int* __restrict__ query_start_loc, const int* __restrict__ context_lens,
    const int* __restrict__ state_slots, int heads, int kv_heads, int dim, int vdim, int split,
    int cols, int chunk) {
  extern __shared__ __align__(16) float lds[];
  const int dp = split * R;                       // padded dim
  float* q_lds = lds;                             // [chunk][dp]
  float* k_lds = q_lds + chunk * dp;              // [chunk][dp]
  float* v_lds = k_lds + chunk * dp;              // [chunk][cols]
  float* num = v_lds + chunk * cols;              // [chunk][5]: g, beta, k scale, q scale, k . q

  // the column group runs fastest: workgroups that run together touch one stretch of the state
  const int h = blockIdx.y, b = blockIdx.z, j0 = blockIdx.x * cols;
  const int g_head = h / (heads / kv_heads);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
  const int jl = tid / split, r = tid - jl * split;
  const int j = j0 + jl;
  const bool col = jl < cols && j < vdim;
  const int ncols = min(cols, vdim - j0);
  const int start = query_start_loc[b], end = query_start_loc[b + 1];
  float* st = state + (((int64_t)state_slots[b] * heads + h) * vdim + (col ? j : 0)) * dim;
  const bool whole = dim == dp && (dim & 3) == 0;  // no padded rows: four rows per access
  const bool resume = context_lens[b] > 0;
  float s[R];
#pragma unroll
  for (int ii = 0; ii < R / 4; ++ii) {
    const int d = 4 * (ii * split + r);
    f32x4 got = {0.f, 0.f, 0.f, 0.f};
    if (col && resume) {
      if (whole) {
        got = *reinterpret_cast<const f32x4*>(st + d);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < dim) got[e] = st[d + e];
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s[4 * ii + e] = got[e];
  }
  const float decay_rate = expf(a_log[h]), bias = dt_bias[h];
  const float q_unit = 1.f / sqrtf((float)dim);

  // A chunk's rows come through registers: they are asked for before the walk over the chunk
  // ahead of them, and land in LDS when that walk is done.
  constexpr int PF = 8;                           // pieces of four rows / of values a thread stages
  f32x4 pq[PF], pk[PF];
  float pv[PF], pb = 0.f, pd = 0.f;
  const int quads = dp / 4;                        // a power of two, as split and R are
  const int quad_shift = __ffs(quads) - 1;
  const bool vec = whole && (in.q_stride & 3) == 0 && (in.k_stride & 3) == 0 &&
                   ((uintptr_t)in.q & 15) == 0 && ((uintptr_t)in.k & 15) == 0;
  auto fetch = [&](int t0, int n) {
    const int pieces = max(n * quads, n * ncols);
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      if (u * (int)blockDim.x >= pieces) break;    // a short chunk (a decode step) stops early
      const int i = tid + u * blockDim.x;
      f32x4 q4 = {0.f, 0.f, 0.f, 0.f}, k4 = {0.f, 0.f, 0.f, 0.f};
      if (i < n * quads) {
        const int tc = i >> quad_shift, d = 4 * (i & (quads - 1));
        const typename SI::T* qr = in.q + (int64_t)(t0 + tc) * in.q_stride + (int64_t)g_head * dim + d;
        const typename SI::T* kr = in.k + (int64_t)(t0 + tc) * in.k_stride + (int64_t)g_head * dim + d;
        if (vec) {
          q4 = *reinterpret_cast<const f32x4*>(qr);
          k4 = *reinterpret_cast<const f32x4*>(kr);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (d + e < dim) {
              q4[e] = SI::to_f32(qr[e]);
              k4[e] = SI::to_f32(kr[e]);
            }
        }
      }
      pq[u] = q4;
      pk[u] = k4;
      pv[u] = 0.f;
      if (i < n * ncols) {
        const int tc = i / ncols, d = i - tc * ncols;
        pv[u] = SI::to_f32(in.v[(int64_t)(t0 + tc) * in.v_stride + (int64_t)h * vdim + j0 + d]);
      }
    }
    if (tid < n) {
      pb = SI::to_f32(in.beta[(int64_t)(t0 + tid) * in.beta_stride + h]);
      pd = SI::to_f32(in.dt[(int64_t)(t0 + tid) * in.dt_stride + h]);
    }
  };
  auto land = [&](int n) {
    const int pieces = max(n * quads, n * ncols);
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      if (u * (int)blockDim.x >= pieces) break;
      const int i = tid + u * blockDim.x;
      if (i < n * quads) {
        *reinterpret_cast<f32x4*>(q_lds + 4 * i) = pq[u];
        *reinterpret_cast<f32x4*>(k_lds + 4 * i) = pk[u];
      }
      if (i < n * ncols) {
        const int tc = i / ncols, d = i - tc * ncols;
        v_lds[tc * cols + d] = pv[u];
      }
    }
    if (tid < n) {
      num[tid * 5 + 0] = expf(-decay_rate * softplusf(pd + bias));
      num[tid * 5 + 1] = 1.f / (1.f + expf(-pb));
    }
  };
  // the unit norms of a chunk's queries and keys and their product: four lanes per token, each
  // summing every fourth row (a token's walk starts 4 tc rows in, so that the tokens of a wave
  // read different banks; the padded rows are zeros)
  auto norms = [&](int n) {
    const int tc = tid >> 2, part = tid & 3;
    float qq = 0.f, kk = 0.f, kq = 0.f;
    if (tc < n) {
      int d = (part + 4 * tc) & (dp - 1);
#pragma unroll 8
      for (int i = 0; i < quads; ++i) {
        const float qv = q_lds[tc * dp + d], kv = k_lds[tc * dp + d];
        qq += qv * qv;
        kk += kv * kv;
        kq += kv * qv;
        d += 4;
        d = d >= dp ? d - dp : d;
      }
    }
    qq = dpp_add<0x4E>(dpp_add<0xB1>(qq));
    kk = dpp_add<0x4E>(dpp_add<0xB1>(kk));
    kq = dpp_add<0x4E>(dpp_add<0xB1>(kq));
    if (tc < n && part == 0) {
      const float ks = 1.f / sqrtf(kk + 1e-6f), qs = q_unit / sqrtf(qq + 1e-6f);
      num[tc * 5 + 2] = ks;
      num[tc * 5 + 3] = qs;
      num[tc * 5 + 4] = kq * ks * qs;
    }
  };
  fetch(start, min(chunk, end - start));
  land(min(chunk, end - start));
  __syncthreads();
  norms(min(chunk, end - start));
  __syncthreads();
  for (int t0 = start; t0 < end; t0 += chunk) {
    const int n = min(chunk, end - t0);
    const int n_next = min(chunk, end - t0 - chunk);
    if (n_next > 0) fetch(t0 + chunk, n_next);
    float* orow = o + ((int64_t)t0 * heads + h) * vdim + (col ? j : 0);
    for (int tc = 0; tc < n; ++tc) {
      const float g = num[tc * 5 + 0], be = num[tc * 5 + 1], ks = num[tc * 5 + 2], qs = num[tc * 5 + 3],
                  kq = num[tc * 5 + 4];
      float kv[R];
      float dk0 = 0.f, dk1 = 0.f, dq0 = 0.f, dq1 = 0.f;
#pragma unroll
      for (int ii = 0; ii < R / 4; ++ii) {
        const f32x4 k4 = *reinterpret_cast<const f32x4*>(k_lds + tc * dp + 4 * (ii * split + r));
        const f32x4 q4 = *reinterpret_cast<const f32x4*>(q_lds + tc * dp + 4 * (ii * split + r));
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          kv[4 * ii + e] = k4[e];
          kv[4 * ii + e + 1] = k4[e + 1];
          dk0 += s[4 * ii + e] * k4[e];
          dk1 += s[4 * ii + e + 1] * k4[e + 1];
          dq0 += s[4 * ii + e] * q4[e];
          dq1 += s[4 * ii + e + 1] * q4[e + 1];
        }
      }
      float dk = dk0 + dk1, dq = dq0 + dq1;
      group_sums(dk, dq, split);
      const float u = be * (v_lds[tc * cols + (col ? jl : 0)] - g * ks * dk);
      const float ku = ks * u;
#pragma unroll
      for (int i = 0; i < R; ++i) s[i] = g * s[i] + kv[i] * ku;
      if (col && r == 0) orow[(int64_t)tc * heads * vdim] = g * qs * dq + kq * u;
    }
    if (n_next > 0) {
      __syncthreads();
      land(n_next);
      __syncthreads();
      norms(n_next);
      __syncthreads();
    }
  }
  if (col) {
#pragma unroll
    for (int ii = 0; ii < R / 4; ++ii) {
      const int d = 4 * (ii * split + r);
      if (whole) {
        const f32x4 put = {s[4 * ii], s[4 * ii + 1], s[4 * ii + 2], s[4 * ii + 3]};
        *reinterpret_cast<f32x4*>(st + d) = put;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < dim) st[d + e] = s[4 * ii + e];
      }
    }
  }
}

constexpr int kStepRows = 4;        // runs of at most this many rows go token by token beside blocks

// Runs of a few rows (decode steps): no staging.  The `split` lanes of a column hold all rows between
// them, so a token's unit norms are lane sums of what they read for the dot products anyway.  LIMIT: runs of more
// than kStepRows rows are the block kernels' (a form of its own: the state's loads would wait for the run's length,
// 129 decode rows of 16 heads of 128 x 128 54.6 us per call, 53.0 without).
template <class SI, int R, bool LIMIT>
__global__ __launch_bounds__(256) void delta_rule_step_kernel(
    float* __restrict__ o, DeltaRows<SI> in, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, float* __restrict__ state,
    const int* __restrict__ query_start_loc, const int* __restrict__ context_lens,
    const int* __restrict__ state_slots, int heads, int kv_heads, int dim, int vdim, int split,
    int cols) {
  const int h = blockIdx.y, b = blockIdx.z, j0 = blockIdx.x * cols;
  const int g_head = h / (heads / kv_heads);
  const int tid = threadIdx.x;
  const int jl = tid / split, r = tid - jl * split;
  const int j = j0 + jl;
  const bool col = jl < cols && j < vdim;
  const int start = query_start_loc[b], end = query_start_loc[b + 1];
  if (LIMIT && end - start > kStepRows) return;
  float* st = state + (((int64_t)state_slots[b] * heads + h) * vdim + (col ? j : 0)) * dim;
  const bool whole = dim == split * R && (dim & 3) == 0;
  const bool vec = whole && (in.q_stride & 3) == 0 && (in.k_stride & 3) == 0 &&
                   ((uintptr_t)in.q & 15) == 0 && ((uintptr_t)in.k & 15) == 0;
  const bool resume = context_lens[b] > 0;
  float s[R];
#pragma unroll
  for (int ii = 0; ii < R / 4; ++ii) {
    const int d = 4 * (ii * split + r);
    f32x4 got = {0.f, 0.f, 0.f, 0.f};
    if (col && resume) {
      if (whole) {
        got = *reinterpret_cast<const f32x4*>(st + d);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < dim) got[e] = st[d + e];
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s[4 * ii + e] = got[e];
  }
  const float decay_rate = expf(a_log[h]), bias = dt_bias[h];
  const float q_unit = 1.f / sqrtf((float)dim);
  for (int t = start; t < end; ++t) {
    float kv[R], qv[R];
#pragma unroll
    for (int ii = 0; ii < R / 4; ++ii) {
      const int d = 4 * (ii * split + r);
      const typename SI::T* qr = in.q + (int64_t)t * in.q_stride + (int64_t)g_head * dim + d;
      const typename SI::T* kr = in.k + (int64_t)t * in.k_stride + (int64_t)g_head * dim + d;
      f32x4 q4 = {0.f, 0.f, 0.f, 0.f}, k4 = {0.f, 0.f, 0.f, 0.f};
      if (vec) {
        q4 = *reinterpret_cast<const f32x4*>(qr);
        k4 = *reinterpret_cast<const f32x4*>(kr);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < dim) {
            q4[e] = SI::to_f32(qr[e]);
            k4[e] = SI::to_f32(kr[e]);
          }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        qv[4 * ii + e] = q4[e];
        kv[4 * ii + e] = k4[e];
      }
    }
    const float vj = SI::to_f32(in.v[(int64_t)t * in.v_stride + (int64_t)h * vdim + (col ? j : 0)]);
    const float be = 1.f / (1.f + expf(-SI::to_f32(in.beta[(int64_t)t * in.beta_stride + h])));
    const float g = expf(-decay_rate * softplusf(SI::to_f32(in.dt[(int64_t)t * in.dt_stride + h]) + bias));
    float qq = 0.f, kk = 0.f, kq = 0.f, dk = 0.f, dq = 0.f, none = 0.f;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      qq += qv[i] * qv[i];
      kk += kv[i] * kv[i];
      kq += kv[i] * qv[i];
      dk += s[i] * kv[i];
      dq += s[i] * qv[i];
    }
    group_sums(qq, kk, split);
    group_sums(kq, none, split);
    group_sums(dk, dq, split);
    const float ks = 1.f / sqrtf(kk + 1e-6f), qs = q_unit / sqrtf(qq + 1e-6f);
    const float u = be * (vj - g * ks * dk);
    const float ku = ks * u;
#pragma unroll
    for (int i = 0; i < R; ++i) s[i] = g * s[i] + kv[i] * ku;
    if (col && r == 0) o[((int64_t)t * heads + h) * vdim + j] = g * qs * dq + kq * ks * qs * u;
  }
  if (col) {
#pragma unroll
    for (int ii = 0; ii < R / 4; ++ii) {
      const int d = 4 * (ii * split + r);
      if (whole) {
        const f32x4 put = {s[4 * ii], s[4 * ii + 1], s[4 * ii + 2], s[4 * ii + 3]};
        *reinterpret_cast<f32x4*>(st + d) = put;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < dim) st[d + e] = s[4 * ii + e];
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Blocks of 32 rows
constexpr int kRows = 32;
constexpr int kMaxBlockDim = 256;
constexpr int kMat = 36;            // floats per row of a 32 x 32 matrix in LDS
constexpr int kMatB = 34;           // and of one in 64 bits
constexpr int kMatT = 18;           // and of a 16 x 16 one

struct DeltaBlocks {
  float* o;                         // [T][heads * vdim]
  DeltaRows<F32> in;
  const float* a_log;
  const float* dt_bias;
  float* state;
  float* scratch;
  const int* query_start_loc;
  const int* context_lens;
  const int* state_slots;
  int num_seqs, heads, kv_heads, dim, vdim;
  int step_rows;                    // runs of at most this many rows are the step kernel's
  bool vec_qk, vec_state;
};

// A block's operands lie in scratch as the walk's waves take them, lane for lane: [16 x 16 tile][lane][4].
// (Lanes side by side in memory matter: with lanes 64 bytes apart the walk below took 192 us.)
// Floats of a block's scratch: W | Q~ | K^ (each 32 x DP) | a place for stores nobody wants (padded to 4) | A (its
// three lower 16 x 16 tiles, and G_31 as the fourth of every lane) | T V (32 x VP) | from which row on a column is not
// finite (VP)
__host__ __device__ __forceinline__ int64_t delta_block_floats(int dp, int vp) {
  return (int64_t)3 * kRows * dp + 4 + 4 * 256 + kRows * vp + vp;
}

// Which sequence and block a block slot is: sequence b's blocks are slots start_b / 32 + b + 0, 1, ...
__device__ __forceinline__ bool find_delta_block(const DeltaBlocks& a, int slot, int& b, int& block) {
  int lo = 0, hi = a.num_seqs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.query_start_loc[mid] / kRows + mid <= slot)
      lo = mid;
    else
      hi = mid - 1;
  }
  b = lo;
  block = slot - (a.query_start_loc[b] / kRows + b);
  return block >= 0 && block * kRows < a.query_start_loc[b + 1] - a.query_start_loc[b];
}

// LDS of the prepare kernel: keys, then queries, whose place the waves' partial products take and then the
// 32 x 32 matrices, then L (column 32: G), decays, betas, what makes keys and queries unit rows, and
// which rows are not finite
__host__ __device__ constexpr int delta_prepare_shared_floats(int dp) {
  return kRows * (dp + 4) > 4 * 6 * 256 ? kRows * (dp + 4) : 4 * 6 * 256;
}
__host__ __device__ constexpr size_t delta_prepare_lds_floats(int dp) {
  return (size_t)kRows * (dp + 4) + delta_prepare_shared_floats(dp) + kRows * kMat + 6 * kRows;
}

// one 16x16x4 matrix-core step in 64 bits: operands as mfma4's, lane (g, c) ends with column c, rows g + 4 i
typedef double f64x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f64x4 mfma4_f64(double a, double b, f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Bound by 64-bit matrix-core instructions (four tenths of its cycles), as many vector ones and the waits between them: a
// workgroup by itself takes 13 us.  Heads of 128: 47 KB of LDS and 168 registers, so that three workgroups share a CU
// (two with the partial products beside the queries: 90 us instead of 78 for 153 blocks of 16 heads).
template <int DX>
__global__ __launch_bounds__(256, DX <= 2 ? 3 : 1) void delta_block_prepare_kernel(DeltaBlocks a) {
  constexpr int DP = 64 * DX, RS = DP + 4;
  extern __shared__ __align__(16) float lds[];
  float* k_lds = lds;                                      // [32][RS]
  float* q_lds = k_lds + kRows * RS;                       // [32][RS]
  float* part = q_lds;                                     // [4 waves][6 tiles][64 lanes][4]
  double* b_mat = reinterpret_cast<double*>(part);         // B, strictly lower
  double* t_mat = b_mat + kRows * kMatB;                   // the 16 x 16 blocks on the diagonal of (I + B)^-1
  double* p_mat = t_mat + 2 * 16 * kMatT;                  // [4 waves]: one between two products
  float* l_mat = part + delta_prepare_shared_floats(DP);   // [32][kMat]
  float* g_lds = l_mat + kRows * kMat;                     // [32]
  float* beta_lds = g_lds + kRows;                         // [32]
  float* ks_lds = beta_lds + kRows;                        // [32]
  float* qs_lds = ks_lds + kRows;                          // [32]
  float* odd_lds = qs_lds + kRows;                         // [2][32]: decay or beta, key
  const int slot = blockIdx.x, h = blockIdx.y;
  int b, block;
  if (!find_delta_block(a, slot, b, block)) return;
  const int run = a.query_start_loc[b + 1] - a.query_start_loc[b];
  if (run <= a.step_rows) return;
  const int t0 = a.query_start_loc[b] + block * kRows, n = min(kRows, run - block * kRows);
  const int D = a.dim, V = a.vdim, hg = h / (a.heads / a.kv_heads);
  const int vb = (V + 15) / 16;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 4, c = lane & 15;
  float* out = a.scratch + ((int64_t)slot * a.heads + h) * delta_block_floats(DP, 16 * vb);
  float* w_out = out;                                      // [DP / 16][2][lane][4]: row c, head row 4 g + e
  float* q_out = w_out + kRows * DP;                       // the same
  float* k_out = q_out + kRows * DP;                       // [DP / 16][2][lane][4]: head row pc (below), row 4 g + e
  float* a_out = k_out + kRows * DP + 4;                   // [wave][lane][three tiles, G_31]
  float* u_out = a_out + 4 * 256;                          // [vb][2][lane][4]: column c, row 4 g + e
  const int row = tid >> 3, eighth = tid & 7;              // 8 neighbouring lanes share a row

  // a wave's columns of v, rows 4 g .. and 16 + 4 g ..: the first two tiles are asked for at the start.  What lies behind
  // the run or the columns is left out where the values are used: chosen here, each load would be waited for behind a
  // branch of its own.
  auto fetch_v = [&](float (&to)[2][4], int vt) {
    const int col = 16 * vt + c;
    const float* vr = a.in.v + (int64_t)h * V + min(col, V - 1);
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 16 * it + 4 * g + e;
        to[it][e] = vr[(int64_t)(t0 + min(j, n - 1)) * a.in.v_stride];
      }
  };

  // rows (zeros behind the run's end) and their factors, decays and betas: every load ahead of everything else, and
  // none behind a branch of its own
  f32x4 qv[2 * DX], kv[2 * DX];
  float v_a[2][4], v_b[2][4];
  {
    const bool live = row < n;
    const int64_t t = t0 + (live ? row : 0);
    const float* qr = a.in.q + t * a.in.q_stride + (int64_t)hg * D;
    const float* kr = a.in.k + t * a.in.k_stride + (int64_t)hg * D;
    const int64_t tr = t0 + min(tid & 31, n - 1);
    const float z = a.in.dt[tr * a.in.dt_stride + h] + a.dt_bias[h], bt = a.in.beta[tr * a.in.beta_stride + h];
    const float al = a.a_log[h];
    if (a.vec_qk) {
#pragma unroll
      for (int x = 0; x < 2 * DX; ++x) {
        const int d = min(4 * eighth + 32 * x, D - 4);
        qv[x] = *reinterpret_cast<const f32x4*>(qr + d);
        kv[x] = *reinterpret_cast<const f32x4*>(kr + d);
      }
    } else {
#pragma unroll
      for (int x = 0; x < 2 * DX; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int d = min(4 * eighth + 32 * x + e, D - 1);
          qv[x][e] = qr[d];
          kv[x][e] = kr[d];
        }
    }
    fetch_v(v_a, min(w, vb - 1));
    fetch_v(v_b, min(w + 4, vb - 1));
    // Rows with a key, decay or beta that is not finite take no part in the products, where 0 times them would
    // reach the rows ahead of them; U of the first of them and of all rows behind it is NaN.
    if (tid < kRows) {
      const float gd = expf(-expf(al) * softplusf(z)), be = 1.f / (1.f + expf(-bt));
      const bool odd = tid < n && !(finite(gd) && finite(be));
      g_lds[tid] = tid < n && !odd ? gd : 1.f;
      beta_lds[tid] = tid < n && !odd ? be : 0.f;
      odd_lds[tid] = odd ? 1.f : 0.f;
    }
    float qq = 0.f, kk = 0.f, odd = 0.f, none = 0.f;
#pragma unroll
    for (int x = 0; x < 2 * DX; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (4 * eighth + 32 * x + e >= D) qv[x][e] = kv[x][e] = 0.f;
        odd = finite(kv[x][e]) ? odd : 1.f;
        qq += qv[x][e] * qv[x][e];
        kk += kv[x][e] * kv[x][e];
      }
    group_sums(qq, kk, 8);
    group_sums(odd, none, 8);
    const float qs = live ? 1.f / (sqrtf(qq + 1e-6f) * sqrtf((float)D)) : 0.f;
    const bool whole = live && finite(kk);               // (a sum that overflows makes a unit row of zeros)
    const float ks = whole ? 1.f / sqrtf(kk + 1e-6f) : 0.f;
#pragma unroll
    for (int x = 0; x < 2 * DX; ++x) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        qv[x][e] = live ? qv[x][e] : 0.f;
        kv[x][e] = whole ? kv[x][e] : 0.f;
      }
      *reinterpret_cast<f32x4*>(q_lds + row * RS + 4 * eighth + 32 * x) = qv[x];
      *reinterpret_cast<f32x4*>(k_lds + row * RS + 4 * eighth + 32 * x) = kv[x];
    }
    if (eighth == 0) {
      ks_lds[row] = ks;
      qs_lds[row] = qs;
      odd_lds[kRows + row] = live ? odd : 0.f;
    }
  }
  __syncthreads();
  const uint64_t odd_rows = __ballot(lane < kRows && odd_lds[lane & 31] + odd_lds[kRows + (lane & 31)] > 0.f);
  const int odd_from = odd_rows ? __builtin_ctzll(odd_rows) : kRows;

  // k_i . k_j and q_i . k_j, lower 16 x 16 tiles; every wave takes a quarter of the head's rows (a lane
  // holds four neighbouring ones: the contraction index may be relabelled as long as both operands are).  In 64
  // bits and of the rows as they are, as are L, T, W and T V, each rounded once: an error in one of them is in all
  // columns of u alike and, where keys are alike, in every u behind it.  Relative errors against 64 bits of outputs /
  // states after 1024 rows of 128 x 128 with slow decays, in 1e-7: token by token, this, and all of it in 32 bits:
  // independent keys 1.9 / 1.7, 1.5 / 1.4, 2.4 / 2.2; keys with a common part as large as the rest 2.0 / 1.8,
  // 1.7 / 1.6, 2.9 / 2.7; with one three times as large 2.4 / 2.0, 2.1 / 2.1, 4.4 / 4.1; eight times 3.3 / 2.2, 2.9 / 2.6.
  // T, W and T V in 32 bits are 8 us less per call of the size below, and 2.7 / 3.2 for keys of three times.
  {
    // L: lane j of wave 0 walks down column j (lane 32: from the block's start)
    if (w == 0) {
      f32x4 gv[kRows / 4];
#pragma unroll
      for (int i = 0; i < kRows / 4; ++i) gv[i] = *reinterpret_cast<const f32x4*>(g_lds + 4 * i);
      const int j = lane < kRows ? lane : -1;
      double r = 1.;
      if (lane <= kRows) {
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
          r *= i > j ? (double)gv[i >> 2][i & 3] : 1.;
          l_mat[i * kMat + lane] = (float)r;
        }
      }
    }
    f64x4 acc[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) acc[i] = f64x4{0., 0., 0., 0.};
#pragma unroll
    for (int x = 0; x < DX; ++x) {
      const int d = 16 * (w * DX + x) + 4 * g;
      const f32x4 k0 = *reinterpret_cast<const f32x4*>(k_lds + c * RS + d);
      const f32x4 k1 = *reinterpret_cast<const f32x4*>(k_lds + (16 + c) * RS + d);
      const f32x4 q0 = *reinterpret_cast<const f32x4*>(q_lds + c * RS + d);
      const f32x4 q1 = *reinterpret_cast<const f32x4*>(q_lds + (16 + c) * RS + d);
      qv[x] = q0;                                          // again: for Q~, which needs G
      qv[DX + x] = q1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const double k0d = k0[e], k1d = k1[e], q0d = q0[e], q1d = q1[e];
        acc[0] = mfma4_f64(k0d, k0d, acc[0]);
        acc[1] = mfma4_f64(k1d, k0d, acc[1]);
        acc[2] = mfma4_f64(k1d, k1d, acc[2]);
        acc[3] = mfma4_f64(q0d, k0d, acc[3]);
        acc[4] = mfma4_f64(q1d, k0d, acc[4]);
        acc[5] = mfma4_f64(q1d, k1d, acc[5]);
      }
    }
    __syncthreads();                                       // the sums take the queries' place
    // [tile][lane of mfma4's result][4]
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) part[((w * 6 + i) * 64 + 16 * e + c) * 4 + g] = (float)acc[i][e];
  }
  __syncthreads();
  f64x4 sum[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int at = min(tid + 256 * u, 6 * 64 - 1);
    sum[u] = f64x4{0., 0., 0., 0.};
#pragma unroll
    for (int ow = 0; ow < 4; ++ow) {
      const f32x4 got = *reinterpret_cast<const f32x4*>(part + (ow * 6 * 64 + at) * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[u][e] += (double)got[e];
    }
  }
  // Q~, from the operands of the products above
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const float gq = l_mat[(16 * it + c) * kMat + kRows] * qs_lds[16 * it + c];
#pragma unroll
    for (int x = 0; x < DX; ++x) {
      const f32x4 q4 = qv[it * DX + x];
      *reinterpret_cast<f32x4*>(q_out + (((w * DX + x) * 2 + it) * 64 + lane) * 4) =
          f32x4{gq * q4[0], gq * q4[1], gq * q4[2], gq * q4[3]};
    }
  }
  __syncthreads();                                         // the matrices take the partial products' place
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int at = tid + 256 * u, tile = at >> 6, kind = tile % 3;
    if (at < 6 * 64) {
      const int i0 = kind > 0 ? 16 : 0, j0 = kind > 1 ? 16 : 0, j = j0 + c;
      double got[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const double unit = sum[u][e] * (double)(tile < 3 ? ks_lds : qs_lds)[i0 + 4 * g + e] * (double)ks_lds[j];
        got[e] = unit * (double)l_mat[(i0 + 4 * g + e) * kMat + j];
      }
      if (tile < 3) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = i0 + 4 * g + e;
          b_mat[i * kMatB + j] = i > j ? (double)beta_lds[i] * got[e] : 0.;
        }
      } else {
        // A as the walk's waves take it: wave c & 3 meets contraction index 4 (c >> 2) + (c & 3)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          a_out[((c & 3) * 64 + ((c >> 2) << 4) + 4 * g + e) * 4 + kind] = i0 + 4 * g + e >= j ? (float)got[e] : 0.f;
      }
    }
  }
  __syncthreads();

  // waves 0 and 1 invert the diagonal blocks of I + B, waves 2 and 3 leave K^.  Lane (g, c) holds rows
  // 4 g .. 4 g + 3 of column c: four rows become final at a time, within a lane, and go to the rows
  // below through lane exchanges
  if (w < 2) {
    const int at = 16 * w;
    f64x4 bv[4][4];                                        // [e][chunk]: B's row 4 g + e
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int ch = 0; ch < 4; ++ch)
#pragma unroll
        for (int f = 0; f < 4; ++f) bv[e][ch][f] = b_mat[(at + 4 * g + e) * kMatB + at + 4 * ch + f];
    double x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = 4 * g + e == c ? 1. : 0.;
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) {
      // rows 4 ch .. 4 ch + 3, right in the lanes g == ch (the others' results are not used)
      double y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        y[e] = x[e];
#pragma unroll
        for (int f = 0; f < e; ++f) y[e] -= bv[e][ch][f] * y[f];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = g == ch ? y[e] : x[e];
        y[e] = __shfl(y[e], 16 * ch + c, 64);
      }
      // the chunk's own block is skipped, the ones above are zeros of B
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int f = 0; f < 4; ++f) x[e] -= (g > ch ? bv[e][ch][f] : 0.) * y[f];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) t_mat[(at + 4 * g + e) * kMatT + c] = x[e];
  } else {
    const float g_last = l_mat[(kRows - 1) * kMat + kRows];
    for (int i = tid - 128; i < 256; i += 128) a_out[4 * i + 3] = g_last;
    for (int i = tid - 128; i < DP * (kRows / 4); i += 128) {
      const int d = 16 * (i >> 7) + 4 * (i & 3) + ((i >> 2) & 3), j = 4 * ((i >> 4) & 7);    // i: tile, half, lane (row pc)
      const f32x4 lv = *reinterpret_cast<const f32x4*>(l_mat + (kRows - 1) * kMat + j);
      const f32x4 ks = *reinterpret_cast<const f32x4*>(ks_lds + j);
      f32x4 kh;
#pragma unroll
      for (int e = 0; e < 4; ++e) kh[e] = (float)((double)lv[e] * (double)ks[e] * (double)k_lds[(j + e) * RS + d]);
      *reinterpret_cast<f32x4*>(k_out + 4 * i) = kh;
    }
  }
  __syncthreads();
  // Row `pc` of an operand is row c of a 64-bit product, so that a lane's four results are neighbours: rows g + 4 i of
  // the product are rows 4 g + i.
  const int pc = 4 * (c & 3) + (c >> 2);
  // the block below them: -T22 (B21 T11), every wave for itself
  double t21[4];
  {
    f64x4 acc = {0., 0., 0., 0.}, neg = {0., 0., 0., 0.};
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = mfma4_f64(b_mat[(16 + pc) * kMatB + 4 * g + e], t_mat[(4 * g + e) * kMatT + c], acc);
    // acc is the next product's B operand where it lies: column c, contraction index 4 g + e
#pragma unroll
    for (int e = 0; e < 4; ++e) neg = mfma4_f64(t_mat[(16 + pc) * kMatT + 4 * g + e], acc[e], neg);
    // from column c, rows 4 g + e to row pc, columns 4 g + e
    double* mine = p_mat + w * 16 * kMatT;
#pragma unroll
    for (int e = 0; e < 4; ++e) mine[(4 * g + e) * kMatT + c] = -neg[e];
    wave_sync();
#pragma unroll
    for (int e = 0; e < 4; ++e) t21[e] = mine[pc * kMatT + 4 * g + e];
  }

  // rows of T diag(beta) as operands: 0: rows 0 .. 15; 1 and 2: rows 16 .. 31 with the first and the
  // second half of the contraction
  double tv[3][4], gj[2][4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const double be0 = beta_lds[4 * g + e], be1 = beta_lds[16 + 4 * g + e];
    tv[0][e] = t_mat[pc * kMatT + 4 * g + e] * be0;
    tv[1][e] = t21[e] * be0;
    tv[2][e] = t_mat[(16 + pc) * kMatT + 4 * g + e] * be1;
  }
#pragma unroll
  for (int jt = 0; jt < 2; ++jt)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      gj[jt][e] = (double)l_mat[(16 * jt + 4 * g + e) * kMat + kRows] * (double)ks_lds[16 * jt + 4 * g + e];
#pragma unroll
  for (int x = 0; x < DX; ++x) {
    const int tile = w + 4 * x;
    f64x4 xt[2];
#pragma unroll
    for (int it = 0; it < 2; ++it) xt[it] = f64x4{0., 0., 0., 0.};
    // transposed, so that a lane ends with four neighbouring rows of the head of one token (row pc)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double ka = (double)k_lds[(4 * g + e) * RS + 16 * tile + pc] * gj[0][e];
      const double kb = (double)k_lds[(16 + 4 * g + e) * RS + 16 * tile + pc] * gj[1][e];
      xt[0] = mfma4_f64(ka, tv[0][e], xt[0]);
      xt[1] = mfma4_f64(ka, tv[1][e], xt[1]);
      xt[1] = mfma4_f64(kb, tv[2][e], xt[1]);
    }
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      f32x4 put;
#pragma unroll
      for (int e = 0; e < 4; ++e) put[e] = (float)xt[it][e];
      *reinterpret_cast<f32x4*>(w_out + ((tile * 2 + it) * 64 + 16 * g + pc) * 4) = put;
    }
  }
  for (int vt = w; vt < vb; vt += 4) {
    int from = odd_from;                                   // column c's first row that is not finite
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 16 * it + 4 * g + e;
        asm volatile("" : "+v"(v_a[it][e]));
        v_a[it][e] = j < n && 16 * vt + c < V ? v_a[it][e] : 0.f;
        if (!finite(v_a[it][e])) {
          from = min(from, j);
          v_a[it][e] = 0.f;
        }
      }
    if (__any(from < kRows)) {
      from = min(from, __shfl_xor(from, 16, 64));
      from = min(from, __shfl_xor(from, 32, 64));
    }
    if (g == 0) u_out[kRows * 16 * vb + 16 * vt + c] = (float)from;
    f64x4 xt[2];
#pragma unroll
    for (int it = 0; it < 2; ++it) xt[it] = f64x4{0., 0., 0., 0.};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double va = v_a[0][e], vb2 = v_a[1][e];
      xt[0] = mfma4_f64(tv[0][e], va, xt[0]);
      xt[1] = mfma4_f64(tv[1][e], va, xt[1]);
      xt[1] = mfma4_f64(tv[2][e], vb2, xt[1]);
    }
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      f32x4 put;
#pragma unroll
      for (int e = 0; e < 4; ++e) put[e] = 16 * it + 4 * g + e < from ? (float)xt[it][e] : NAN;
      *reinterpret_cast<f32x4*>(u_out + ((vt * 2 + it) * 64 + lane) * 4) = put;
#pragma unroll
      for (int e = 0; e < 4; ++e) v_a[it][e] = v_b[it][e];
    }
    if (vt + 8 < vb) fetch_v(v_b, vt + 8);
  }
}

// a value that is the same for all lanes, where a choice by it should be no branch
__device__ __forceinline__ int lane_value(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// What bounds it: a wave has 35 matrix-core instructions of 32 cycles per block and 16 of 64 (2140 of about 3300 cycles
// of 128 x 128) in a chain product -> LDS -> barrier -> LDS -> product, one wave per SIMD and nobody to fill its
// waits.  So the next block's loads go out between the products (56 KB per block and workgroup: sent at once they held a
// wave up for 1250 cycles), the product for the outputs stands where the exchange of U is on its way, and the
// state of 16 rows and the block before's outputs are formed under the 64-bit products.  No value of a block may be
// copied from turn to turn (its load would be waited for right there), and the first block's loads keep the order of
// the loop's, which waits for what both orders have in common.
// Two prompts of 2999 and 1854 tokens, 16 heads of 128 x 128 (94 blocks in a row), under the tracer, which lets no launch
// begin before the one ahead of it has ended: the walk 179 us, 1.9 us per block (212 with the loads at once and choices by
// branches), the prepare kernel 79, the norms 20 and the step kernel's empty launch 5; a call, whose launches overlap,
// 251 (333), where the token-by-token walk of the same prompts takes 1079.
// What a block adds to the state is summed in 64 bits: in 32 a call is 20 us less and states are 1.2 times as far
// from 64 bits as token by token where keys share a part three times as large as the rest (1.0).
template <int DX>
__global__ __launch_bounds__(256, DX <= 2 ? 2 : 1) void delta_block_walk_kernel(DeltaBlocks a) {
  constexpr int DP = 64 * DX;
  __shared__ __align__(16) float u_part[2][4][2][64][4];   // a wave's part of W S
  __shared__ __align__(16) float o_part[2][4][2][4][64];   // of the outputs, by component
  // heads run fastest: the workgroups of a head's columns, which read the same scratch, share an XCD
  // (and its L2) whenever the number of heads is a multiple of 8
  const int h = blockIdx.x, v0 = 16 * blockIdx.y, b = blockIdx.z;
  const int t_begin = a.query_start_loc[b], run = a.query_start_loc[b + 1] - t_begin;
  if (run <= a.step_rows) return;
  const int D = a.dim, V = a.vdim, vp = (V + 15) / 16 * 16;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = v0 + c;
  const int64_t per = delta_block_floats(DP, vp);
  const float* base = a.scratch + ((int64_t)(t_begin / kRows + b) * a.heads + h) * per;
  const int64_t step = (int64_t)a.heads * per;
  float* st = a.state + (((int64_t)a.state_slots[b] * a.heads + h) * V + (col < V ? col : 0)) * D;
  const bool resume = a.context_lens[b] > 0;
  f32x4 s[DX];
#pragma unroll
  for (int x = 0; x < DX; ++x) {
    const int d = 16 * (w * DX + x) + 4 * g;
    s[x] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (resume && col < V) s[x] = load4<F32>(st, d, D, a.vec_state);
  }
  const int blocks = (run + kRows - 1) / kRows;
  struct Block {
    f32x4 wv[DX][2], qv[DX][2], kv[DX][2], u[2], av;
    float from;
  };
  const int at_x = w * DX * 2 * 256 + 4 * lane, at_a = 4 * (w * 64 + lane), at_u = blockIdx.y * 2 * 256 + 4 * lane;
  // piece j of a block, in the order that the walk wants them: W, Q~, T V, K^, A and the rest
  constexpr int kHalves = 2 * DX, kPieces = 3 * kHalves + 4, kFirst = 2 * kHalves;
  auto fetch = [&](Block& f, const float* p, int j) __attribute__((always_inline)) {
    const float* pa = p + 3 * kRows * DP;
    const int x = (j % kHalves) >> 1, it = j & 1;
    if (j < kHalves)
      f.wv[x][it] = *reinterpret_cast<const f32x4*>(p + at_x + 256 * j);
    else if (j < kFirst)
      f.qv[x][it] = *reinterpret_cast<const f32x4*>(p + kRows * DP + at_x + 256 * (j - kHalves));
    else if (j < kFirst + 2)
      f.u[it] = *reinterpret_cast<const f32x4*>(pa + 4 + 4 * 256 + at_u + 256 * it);
    else if (j < kFirst + 2 + kHalves)
      f.kv[((j - 2) % kHalves) >> 1][it] = *reinterpret_cast<const f32x4*>(p + 2 * kRows * DP + at_x + 256 * (j - 2 - kFirst));
    else if (j == kPieces - 2)
      f.av = *reinterpret_cast<const f32x4*>(pa + 4 + at_a);
    else
      f.from = pa[4 + 4 * 256 + kRows * vp + col];
  };
  // wave w finishes rows 16 it + 4 g + w of a block's outputs; what has no place goes to the block's pad
  const int64_t row_step = (int64_t)a.heads * V;
  float* o_at = a.o + ((int64_t)(t_begin + 4 * g + w) * a.heads + h) * V + (col < V ? col : 0);
  float* nowhere = a.scratch + ((int64_t)(t_begin / kRows + b) * a.heads + h) * per + 3 * kRows * DP;
  // column c is NaN from its first row on that is not finite, as the state that a walk reads it with
  const float row_w = (float)(4 * g + w);
  const unsigned rows_here = col < V ? run : 0;
  auto finish_read = [&](int i, float (&o)[2][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int ow = 0; ow < 4; ++ow) o[it][ow] = o_part[i & 1][ow][it][w][lane];
  };
  auto finish = [&](int i, const float (&o)[2][4], float from) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const float sum = (o[it][0] + o[it][1]) + (o[it][2] + o[it][3]);
      const bool live = (unsigned)(i * kRows + 16 * it + 4 * g + w) < rows_here;      // (block -1 has none)
      *(live ? o_at + (i * kRows + 16 * it) * row_step : nowhere) = row_w + 16.f * it < from ? sum : NAN;
    }
  };
  const int own = lane_value(w);
  auto advance = [&](const Block& f, Block& next, const float* next_at, int i) __attribute__((always_inline)) {
    const int buf = i & 1;
    // sums in several parts: half the roundings in a row
    constexpr int kParts = DX > 1 ? 2 : 1;
    f32x4 xu[2][kParts], xo[2][kParts];
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int p = 0; p < kParts; ++p) xu[it][p] = xo[it][p] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < DX; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int it = 0; it < 2; ++it) {
          xu[it][x % kParts] = mfma4(f.wv[x][it][e], s[x][e], xu[it][x % kParts]);
          if (it == 0 && e % 2 == 0) fetch(next, next_at, 2 * x + e / 2);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
    for (int it = 0; it < 2; ++it) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if constexpr (kParts > 1) xu[it][0][e] += xu[it][1][e];
      *reinterpret_cast<f32x4*>(&u_part[buf][w][it][lane][0]) = xu[it][0];
    }
    __syncthreads();
    f32x4 p[2][4];
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int ow = 0; ow < 4; ++ow) p[it][ow] = *reinterpret_cast<const f32x4*>(&u_part[buf][ow][it][lane][0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < DX; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int it = 0; it < 2; ++it) {
          xo[it][x % kParts] = mfma4(f.qv[x][it][e], s[x][e], xo[it][x % kParts]);
          if (it == 0 && e % 2 == 0) fetch(next, next_at, kHalves + 2 * x + e / 2);
          __builtin_amdgcn_sched_barrier(0);
        }
    float done[2][4];
    finish_read(i - 1, done);                              // (ahead of the first block: what nobody wants)
    __builtin_amdgcn_sched_barrier(0);
    f32x4 u[2];
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        u[it][e] = f.u[it][e] - ((p[it][0][e] + p[it][1][e]) + (p[it][2][e] + p[it][3][e]));
    // A U: the wave takes contraction index 4 g + w, so that the sum over waves is the whole product.  A row's product
    // with the rows behind it is 0 times their U: those that are not finite stay out.
    float us[2];
#pragma unroll
    for (int it = 0; it < 2; ++it) {
#pragma unroll
      for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(u[it][e]));       // (chosen, not worked out again behind branches)
      const float even = own & 2 ? u[it][2] : u[it][0], odd = own & 2 ? u[it][3] : u[it][1];
      us[it] = own & 1 ? odd : even;
    }
    const float u0 = row_w < f.from ? us[0] : 0.f, u1 = row_w + 16.f < f.from ? us[1] : 0.f;
    f32x4 av = f.av;
    asm volatile("" : "+v"(av));                            // (whole: a part by itself would be copied from block to block)
    xo[0][0] = mfma4(av[0], u0, xo[0][0]);
    xo[1][0] = mfma4(av[1], u0, xo[1][0]);
    xo[1][0] = mfma4(av[2], u1, xo[1][0]);
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (kParts > 1) xo[it][0][e] += xo[it][1][e];
        o_part[buf][w][it][e][lane] = xo[it][0][e];
      }
    // What the block adds is summed by itself, in 64 bits: one rounding of the state per block.  One 16 rows after the
    // other, so that a state is formed under the next one's products, as are the outputs of the block before.
    f64x4 ds[DX];
#pragma unroll
    for (int x = 0; x < DX; ++x) {
      ds[x] = f64x4{0., 0., 0., 0.};
#pragma unroll
      for (int it = 0; it < 2; ++it)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ds[x] = mfma4_f64((double)f.kv[x][it][e], (double)u[it][e], ds[x]);
          constexpr int kLeft = kPieces - kFirst, kProducts = 8 * DX;
          const int at = 8 * x + 4 * it + e;
          if (at == kProducts / 2 - 1) finish(i - 1, done, next.from);     // (next has the block before in its place)
#pragma unroll
          for (int j = 0; j < kLeft; ++j)
            if (j * kProducts / kLeft == at) fetch(next, next_at, kFirst + j);
          if (x > 0 && it == 0) s[x - 1][e] = (float)((double)av[3] * (double)s[x - 1][e] + ds[x - 1][e]);
          __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s[DX - 1][e] = (float)((double)av[3] * (double)s[DX - 1][e] + ds[DX - 1][e]);
  };
  // two blocks in turn, so that one is asked for while the other is worked on
  Block f0, f1;
#pragma unroll
  for (int j = 0; j < kPieces; ++j) {
    fetch(f0, base, j);
    __builtin_amdgcn_sched_barrier(0);                     // (the loop waits for the order that it finds here, too)
  }
  const float* at = base;
  for (int i = 0; i < blocks; i += 2) {
    at += i + 1 < blocks ? step : 0;
    advance(f0, f1, at, i);
    if (i + 1 >= blocks) break;
    at += i + 2 < blocks ? step : 0;
    advance(f1, f0, at, i + 1);
  }
  const float from = at[3 * kRows * DP + 4 + 4 * 256 + kRows * vp + col];      // (f0's would be copied, and waited for, in each turn)
  __syncthreads();
  float done[2][4];
  finish_read(blocks - 1, done);
  finish(blocks - 1, done, from);
  if (col < V) {
#pragma unroll
    for (int x = 0; x < DX; ++x) {
      const int d = 16 * (w * DX + x) + 4 * g;
      if (a.vec_state) {
        if (d < D) *reinterpret_cast<f32x4*>(st + d) = s[x];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < D) st[d + e] = s[x][e];
      }
    }
  }
}

template <int DX>
int launch_delta_blocks(const DeltaBlocks& a, int num_tokens, int64_t slots, hipStream_t stream) {
  // Heads of more than 192: as if lengths were even, since no more than two share a CU and a second round of a few costs no
  // more than uneven shares do (4 heads of 256, 16 runs of 100 rows 23 us, with two to some CUs 31).
  const int64_t even = (int64_t)a.num_seqs * ((num_tokens + (int64_t)a.num_seqs * kRows - 1) / ((int64_t)a.num_seqs * kRows));
  const size_t lds = spread_lds(delta_prepare_lds_floats(64 * DX) * sizeof(float),
                                (DX > 3 ? even : pieces_at_most(num_tokens, a.num_seqs, kRows)) * a.heads);
  static std::atomic<uint64_t> raised{0};
  if (const int rc = raise_lds(&delta_block_prepare_kernel<DX>, lds, raised)) return rc;
  delta_block_prepare_kernel<DX><<<dim3((unsigned)slots, a.heads), 256, lds, stream>>>(a);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  delta_block_walk_kernel<DX><<<dim3(a.heads, (a.vdim + 15) / 16, a.num_seqs), 256, 0, stream>>>(a);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  return VLA_OK;
}

int64_t delta_block_slots(int num_tokens, int num_seqs) { return (int64_t)num_tokens / kRows + num_seqs; }

// out = dtype(o / sqrt(mean_v(o^2) + eps) * weight * silu(gate)) per (token, head): one wave each
template <class SI, class SO>
__global__ __launch_bounds__(256) void delta_head_norm_kernel(
    typename SO::T* __restrict__ out, int64_t out_stride, const float* __restrict__ o,
    const typename SI::T* __restrict__ gate, int64_t gate_stride, const float* __restrict__ weight,
    float eps, int rows, int heads, int vdim) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);     // token * heads + head
  if (row >= rows) return;
  const int64_t t = row / heads;
  const int h = (int)(row - t * heads);
  const float* orow = o + row * vdim;
  float ss = 0.f;
  for (int d = lane; d < vdim; d += kWave) ss += orow[d] * orow[d];
  ss = wave_sum(ss);
  const float inv = 1.f / sqrtf(ss / (float)vdim + eps);
  for (int d = lane; d < vdim; d += kWave) {
    const float gt = SI::to_f32(gate[t * gate_stride + (int64_t)h * vdim + d]);
    out[t * out_stride + (int64_t)h * vdim + d] = SO::from_f32(orow[d] * inv * weight[d] * (gt / (1.f + expf(-gt))));
  }
}

// The same for heads of up to 256 values, four per lane: `lanes` neighbours share a (token, head), 16, 32
// or 64 of them.  Bound by HBM: 4853 tokens of 16 heads of 128 are 99 MB.
template <class SO>
__global__ __launch_bounds__(256) void delta_head_norm_vec_kernel(
    typename SO::T* __restrict__ out, int64_t out_stride, const float* __restrict__ o,
    const float* __restrict__ gate, int64_t gate_stride, const float* __restrict__ weight, float eps,
    int rows, int heads, int vdim, int lanes) {
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / lanes;      // token * heads + head
  const int d = 4 * (threadIdx.x & (lanes - 1));
  const bool live = row < rows && d < vdim;
  const int64_t t = (row < rows ? row : 0) / heads;
  const int h = (int)((row < rows ? row : 0) - t * heads);
  f32x4 x = {0.f, 0.f, 0.f, 0.f}, gt = x, wt = x;
  if (live) {
    x = *reinterpret_cast<const f32x4*>(o + row * vdim + d);
    gt = *reinterpret_cast<const f32x4*>(gate + t * gate_stride + (int64_t)h * vdim + d);
    wt = *reinterpret_cast<const f32x4*>(weight + d);
  }
  float ss = x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3], none = 0.f;
  group_sums(ss, none, 16);
  if (lanes > 16) ss += __shfl_xor(ss, 16, 64);
  if (lanes > 32) ss += __shfl_xor(ss, 32, 64);
  const float inv = 1.f / sqrtf(ss / (float)vdim + eps);
  if (!live) return;
  float y[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = x[e] * inv * wt[e] * (gt[e] / (1.f + expf(-gt[e])));
  typename SO::T* dst = out + t * out_stride + (int64_t)h * vdim + d;
  if constexpr (sizeof(typename SO::T) == 2)
    *reinterpret_cast<u32x2*>(dst) = u32x2{pack16<SO>(y[0], y[1]), pack16<SO>(y[2], y[3])};
  else
    *reinterpret_cast<f32x4*>(dst) = f32x4{y[0], y[1], y[2], y[3]};
}

std::atomic<int> g_delta_kernel{0};

// Blocks pay from about a block's rows on (us on the GPU, calls back to back, 16 heads of 128, token by token / in
// blocks: one run of 33 rows 21 / 23, 48 rows 24 / 23, 100 rows 43 / 28; six runs of 64 rows 55 / 44; 32 runs of 33
// rows 140 / 114, of 64 217 / 129; one of 33 beside 31 single rows 50 / 41).  Their scratch is 69 KB per block and head of 128 x 128;
// a step that would want more than 4 GiB of it walks token by token.  (The 1 KB of a block and head where G_31 lies is not
// counted, so that the line lies where it did before: steps of up to 4.06 GiB at 128 x 128, 4.14 at 64 x 16, go in blocks.)
constexpr int kBlockMinRows = 33;

int64_t delta_out_floats(int num_tokens, int heads, int vdim) {
  return ((int64_t)num_tokens * heads * vdim + 3) / 4 * 4;
}

bool wants_blocks(int mode, int num_tokens, int num_seqs, int max_query_len, int heads, int dim, int vdim) {
  if (mode != 0 || dim > kMaxBlockDim || max_query_len < kBlockMinRows || (vdim + 15) / 16 > 65535) return false;
  return delta_block_slots(num_tokens, num_seqs) * heads *
             (delta_block_floats((dim + 63) / 64 * 64, (vdim + 15) / 16 * 16) - 256) <= ((int64_t)1 << 30);
}

int pow2_at_least(int n) {
  int p = 1;
  while (p < n) p <<= 1;
  return p;
}

}  // namespace
}  // namespace seq
}  // namespace vla

using namespace vla;
using namespace vla::seq;

namespace {

// scratch_floats < 0: as many as vla_seq_delta_rule_scratch_floats says, which holds no blocks
int delta_rule_scan(
    void* out, int64_t out_stride, int out_dtype, const void* q, int64_t q_stride, const void* k,
    int64_t k_stride, const void* v, int64_t v_stride, const void* gate, int64_t gate_stride,
    const void* beta, int64_t beta_stride, const void* dt, int64_t dt_stride, int in_dtype,
    const float* a_log, const float* dt_bias, const float* norm_weight, float* state,
    const int* query_start_loc, const int* context_lens, const int* state_slots, int num_tokens,
    int num_seqs, int max_query_len, int num_slots, int heads, int kv_heads, int dim, int vdim,
    float eps, float* scratch, int64_t scratch_floats, void* stream) {
  if (num_seqs == 0 || num_tokens == 0) return VLA_OK;
  if (!out || !q || !k || !v || !gate || !beta || !dt || !a_log || !dt_bias || !norm_weight ||
      !state || !scratch || !query_start_loc || !context_lens || !state_slots || num_seqs < 0 ||
      num_seqs > 65535 || num_tokens < 0 || num_slots <= 0 || heads <= 0 || kv_heads <= 0 ||
      heads % kv_heads != 0 || dim <= 0 || vdim <= 0 || out_stride < (int64_t)heads * vdim ||
      q_stride < (int64_t)kv_heads * dim || k_stride < (int64_t)kv_heads * dim ||
      v_stride < (int64_t)heads * vdim || gate_stride < (int64_t)heads * vdim ||
      beta_stride < heads || dt_stride < heads)
    return VLA_ERR_ARG;
  // the rows that enter the recurrence are fp32 (the caller's projections leave them so)
  if (in_dtype != VLA_F32) return VLA_ERR_DTYPE;
  // the fewest rows per thread (8, 16, 32, 64) whose column groups are at most kMaxSplit lanes
  int rows = 0, split = 0;
  for (int r = 8; r <= 64; r *= 2) {
    const int sp = pow2_at_least((dim + r - 1) / r);
    if (sp <= kMaxSplit) {
      rows = r;
      split = sp;
      break;
    }
  }
  if (rows == 0) return VLA_ERR_HEAD_SIZE;
  // a workgroup of 256 threads: 256 / split columns of one head
  const int cols = 256 / split < vdim ? 256 / split : vdim;
  const int threads = (cols * split + 63) / 64 * 64;
  const int col_groups = (vdim + cols - 1) / cols;
  if (heads > 65535) return VLA_ERR_ARG;
  // a chunk fits LDS, a thread's staging registers (8 pieces of four rows, 8 values) and four
  // threads per token
  const size_t per_token = (size_t)(2 * split * rows + cols + 5) * sizeof(float);
  int chunk = kMaxChunk;
  chunk = std::min<int64_t>(chunk, 60 * 1024 / per_token);
  chunk = std::min(chunk, 8 * threads * 4 / (split * rows));
  chunk = std::min(chunk, 8 * threads / cols);
  chunk = std::min(chunk, threads / 4);
  if (max_query_len > 0) chunk = std::min(chunk, max_query_len);
  if (chunk < 1) return VLA_ERR_HEAD_SIZE;
  const size_t lds = chunk * per_token;
  using SI = F32;
  const DeltaRows<SI> in{(const float*)q, q_stride, (const float*)k, k_stride, (const float*)v, v_stride,
                         (const float*)gate, gate_stride, (const float*)beta, beta_stride,
                         (const float*)dt, dt_stride};
  const dim3 grid(col_groups, heads, num_seqs);
  // runs of at most four rows take the kernel without staging (modes 1 / 2: always / never, for tests)
  const int mode = g_delta_kernel.load(std::memory_order_relaxed);
  const bool blocks = scratch_floats >= 0 && wants_blocks(mode, num_tokens, num_seqs, max_query_len, heads, dim, vdim);
  // (a lone run goes in blocks however short it is: max_query_len may be more than its rows)
  const bool steps = blocks ? num_seqs > 1 : mode == 1 || (mode == 0 && max_query_len > 0 && max_query_len <= kStepRows);
  const int64_t out_floats = delta_out_floats(num_tokens, heads, vdim);
  if (blocks) {
    DeltaBlocks a;
    a.o = scratch;
    a.in = in;
    a.a_log = a_log;
    a.dt_bias = dt_bias;
    a.state = state;
    a.scratch = scratch + out_floats;
    a.query_start_loc = query_start_loc;
    a.context_lens = context_lens;
    a.state_slots = state_slots;
    a.num_seqs = num_seqs;
    a.heads = heads;
    a.kv_heads = kv_heads;
    a.dim = dim;
    a.vdim = vdim;
    a.step_rows = steps ? kStepRows : 0;
    auto fours = [&](const void* p, int64_t stride) {              // four values per access
      return dim % 4 == 0 && stride % 4 == 0 && (uintptr_t)p % 16 == 0;
    };
    a.vec_qk = fours(q, q_stride) && fours(k, k_stride);
    a.vec_state = fours(state, 0);
    const int64_t slots = delta_block_slots(num_tokens, num_seqs);
    if ((uintptr_t)scratch % 16 || scratch_floats < out_floats + slots * heads * delta_block_floats((dim + 63) / 64 * 64, (vdim + 15) / 16 * 16))
      return VLA_ERR_ARG;
    int rc = VLA_OK;
    switch ((dim + 63) / 64) {
      case 1: rc = launch_delta_blocks<1>(a, num_tokens, slots, (hipStream_t)stream); break;
      case 2: rc = launch_delta_blocks<2>(a, num_tokens, slots, (hipStream_t)stream); break;
      case 3: rc = launch_delta_blocks<3>(a, num_tokens, slots, (hipStream_t)stream); break;
      default: rc = launch_delta_blocks<4>(a, num_tokens, slots, (hipStream_t)stream); break;
    }
    if (rc != VLA_OK) return rc;
  }
  if (steps) {
    auto launch_step = [&](auto kernel) {
      kernel<<<grid, threads, 0, (hipStream_t)stream>>>(scratch, in, a_log, dt_bias, state, query_start_loc,
                                                        context_lens, state_slots, heads, kv_heads, dim, vdim,
                                                        split, cols);
    };
    auto step_of = [&](auto limit) {
      constexpr bool kLimit = decltype(limit)::value;
      switch (rows) {
        case 8: launch_step(delta_rule_step_kernel<SI, 8, kLimit>); break;
        case 16: launch_step(delta_rule_step_kernel<SI, 16, kLimit>); break;
        case 32: launch_step(delta_rule_step_kernel<SI, 32, kLimit>); break;
        default: launch_step(delta_rule_step_kernel<SI, 64, kLimit>); break;
      }
    };
    if (blocks)
      step_of(std::true_type{});
    else
      step_of(std::false_type{});
  }
  auto launch = [&](auto kernel) {
    kernel<<<grid, threads, lds, (hipStream_t)stream>>>(scratch, in, a_log, dt_bias, state, query_start_loc,
                                                        context_lens, state_slots, heads, kv_heads, dim,
                                                        vdim, split, cols, chunk);
  };
  if (!steps && !blocks) {
    switch (rows) {
      case 8: launch(delta_rule_kernel<SI, 8>); break;
      case 16: launch(delta_rule_kernel<SI, 16>); break;
      case 32: launch(delta_rule_kernel<SI, 32>); break;
      default: launch(delta_rule_kernel<SI, 64>); break;
    }
  }
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  return with_dtype(out_dtype, [&](auto so) {
    using SO = decltype(so);
    const int64_t head_rows = (int64_t)num_tokens * heads;
    const int quads = sizeof(typename SO::T) == 2 ? 8 : 16;         // bytes a lane writes
    if (vdim % 4 == 0 && vdim <= 256 && gate_stride % 4 == 0 && (uintptr_t)gate % 16 == 0 && out_stride % 4 == 0 &&
        (uintptr_t)out % quads == 0 && (uintptr_t)norm_weight % 16 == 0 && (uintptr_t)scratch % 16 == 0) {
      const int lanes = vdim <= 64 ? 16 : vdim <= 128 ? 32 : 64;
      delta_head_norm_vec_kernel<SO><<<(unsigned)((head_rows * lanes + 255) / 256), 256, 0, (hipStream_t)stream>>>(
          (typename SO::T*)out, out_stride, scratch, (const float*)gate, gate_stride, norm_weight, eps, (int)head_rows,
          heads, vdim, lanes);
      VLA_SEQ_HIP_CHECK(hipGetLastError());
      return VLA_OK;
    }
    delta_head_norm_kernel<SI, SO><<<(unsigned)((head_rows + 3) / 4), 256, 0, (hipStream_t)stream>>>(
        (typename SO::T*)out, out_stride, scratch, (const float*)gate, gate_stride, norm_weight, eps,
        (int)head_rows, heads, vdim);
    VLA_SEQ_HIP_CHECK(hipGetLastError());
    return VLA_OK;
  });
}

}  // namespace

extern "C" int64_t vla_seq_delta_rule_scratch_floats(int num_tokens, int heads, int vdim) {
  return (int64_t)num_tokens * heads * vdim;
}

extern "C" int64_t vla_seq_delta_rule_block_scratch_floats(int num_tokens, int num_seqs, int max_query_len, int heads,
                                                           int dim, int vdim) {
  const int64_t o = delta_out_floats(num_tokens, heads, vdim);
  if (!wants_blocks(g_delta_kernel.load(std::memory_order_relaxed), num_tokens, num_seqs, max_query_len, heads, dim, vdim))
    return o;
  return o + delta_block_slots(num_tokens, num_seqs) * heads * delta_block_floats((dim + 63) / 64 * 64, (vdim + 15) / 16 * 16);
}

extern "C" int vla_seq_delta_rule_scan(
    void* out, int64_t out_stride, int out_dtype, const void* q, int64_t q_stride, const void* k,
    int64_t k_stride, const void* v, int64_t v_stride, const void* gate, int64_t gate_stride,
    const void* beta, int64_t beta_stride, const void* dt, int64_t dt_stride, int in_dtype,
    const float* a_log, const float* dt_bias, const float* norm_weight, float* state,
    const int* query_start_loc, const int* context_lens, const int* state_slots, int num_tokens,
    int num_seqs, int max_query_len, int num_slots, int heads, int kv_heads, int dim, int vdim,
    float eps, float* scratch, void* stream) {
  return delta_rule_scan(out, out_stride, out_dtype, q, q_stride, k, k_stride, v, v_stride, gate, gate_stride, beta, beta_stride,
                         dt, dt_stride, in_dtype, a_log, dt_bias, norm_weight, state, query_start_loc, context_lens,
                         state_slots, num_tokens, num_seqs, max_query_len, num_slots, heads, kv_heads, dim, vdim, eps,
                         scratch, -1, stream);
}

extern "C" int vla_seq_delta_rule_scan_blocks(
    void* out, int64_t out_stride, int out_dtype, const void* q, int64_t q_stride, const void* k,
    int64_t k_stride, const void* v, int64_t v_stride, const void* gate, int64_t gate_stride,
    const void* beta, int64_t beta_stride, const void* dt, int64_t dt_stride, int in_dtype,
    const float* a_log, const float* dt_bias, const float* norm_weight, float* state,
    const int* query_start_loc, const int* context_lens, const int* state_slots, int num_tokens,
    int num_seqs, int max_query_len, int num_slots, int heads, int kv_heads, int dim, int vdim,
    float eps, float* scratch, int64_t scratch_floats, void* stream) {
  if (scratch_floats < 0) return VLA_ERR_ARG;
  return delta_rule_scan(out, out_stride, out_dtype, q, q_stride, k, k_stride, v, v_stride, gate, gate_stride, beta, beta_stride,
                         dt, dt_stride, in_dtype, a_log, dt_bias, norm_weight, state, query_start_loc, context_lens,
                         state_slots, num_tokens, num_seqs, max_query_len, num_slots, heads, kv_heads, dim, vdim, eps,
                         scratch, scratch_floats, stream);
}

// 0: pick per step; 1: always the kernel without staging; 2: never (tests run both)
extern "C" int vla_seq_set_delta_kernel(int mode) {
  if (mode < 0 || mode > 2) return VLA_ERR_ARG;
  g_delta_kernel.store(mode, std::memory_order_relaxed);
  return VLA_OK;
}
