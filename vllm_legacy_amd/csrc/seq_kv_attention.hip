// Causal softmax attention over paged key and value caches with rotary positions on queries and
// keys, values that are rotated by their own position when they are cached (the head's output is
// turned back by the query's position), an optional sliding window that may keep a sequence's
// first tokens visible, optional chunks (a row sees the keys of its own chunk of positions only), an
// optional cap on the scores (cap * tanh(score / cap)), an optional sink per head (one more term in the
// softmax denominator that has no value) and a sigmoid gate of one number per head.  rotary_kv_write
// can also norm the whole query and key rows, or every head, before it rotates them and blend the
// values with another layer's values of the same tokens.
//
// With a window and `keep_first` kept tokens, query position p sees j <= p with p - j < window or
// j < keep_first; with chunks, j >= p - p % chunk (both: the later of the two bounds).  The kernels walk such a key set through one index u: with lo the window's first
// key and nk = min(keep_first, lo), u < nk is key u and u >= nk is key lo + u - nk.
//
// Caches: keys [num_blocks, block_size, kv_heads, dim] and values [num_blocks, block_size, kv_heads,
// vdim] in the model dtype, token-major rows.  rotary_kv_write rotates the step's queries in place
// and writes the rotated keys and values to their slots; the attention kernels then read every
// query row's keys from the caches, so prompts, portions of prompts and decode steps are one case
// and a position's result cannot depend on how its sequence was cut into steps.  Angles, scores,
// softmax and the weighted sum are fp32.
//
// kv_attention_kernel: one wave per (token, query head), any dtype and head size up to 256.  A
// tile is 64 keys: lane j scores key j against the query held in LDS, the wave reduces max / sum
// (online softmax across tiles), then lane d accumulates sum_j p_j v_j[d] with coalesced reads.
#include <atomic>
#include <type_traits>

#include "seq_common.h"

namespace vla {
namespace seq {
namespace {

constexpr int kMaxDim = 512;
constexpr int kMaxPairs = kMaxDim / 2;
constexpr int kHeadsPerGroup = 4;

// the pair (a, b) turned by angle: (a cos - b sin, b cos + a sin)
__device__ __forceinline__ void turn(float& a, float& b, float angle) {
  float s, c;
  sincosf(angle, &s, &c);
  const float a2 = a * c - b * s;
  b = b * c + a * s;
  a = a2;
}
// cap * tanh(s / cap): libm's tanh in the fp32 kernel, one exponential and one reciprocal in the
// matrix-core kernels (absolute error of a few 1e-7 times cap)
__device__ __forceinline__ float cap_score(float s, float cap) { return cap * tanhf(s / cap); }
__device__ __forceinline__ float cap_score_fast(float s, float cap, float two_log2e_over_cap) {
  const float e = __builtin_amdgcn_exp2f(s * two_log2e_over_cap);   // e^(2 s / cap); inf and 0 are fine
  return cap - 2.f * cap * __builtin_amdgcn_rcpf(e + 1.f);
}

// the first key position p sees (kept tokens apart): its window's, or its chunk's, whichever is later;
// never decreases with p
__device__ __forceinline__ int first_key(int p, int window, int chunk) {
  int lo = window > 0 ? max(0, p - window + 1) : 0;
  if (chunk > 0) lo = max(lo, p - p % chunk);
  return lo;
}

// element indices of pair i among `span` rotated elements
__device__ __forceinline__ void pair_index(int i, int span, int interleaved, int& ia, int& ib) {
  if (interleaved) {
    ia = 2 * i;
    ib = 2 * i + 1;
  } else {
    ia = i;
    ib = i + span / 2;
  }
}

// One workgroup per token: every head's rotated pairs, then the elements that are not rotated.  A token's sines
// and cosines are the same for all heads: formed once, in LDS (5543 rows of 16 + 4 heads of 128: 25 us, 27.5
// when every pair of every head formed its own).
template <class S>
__global__ __launch_bounds__(256) void rotary_kv_write_kernel(
    typename S::T* __restrict__ q, int64_t q_stride, const typename S::T* __restrict__ k,
    int64_t k_stride, const typename S::T* __restrict__ v, int64_t v_stride,
    typename S::T* __restrict__ key_cache, typename S::T* __restrict__ value_cache,
    const int64_t* __restrict__ positions, const int64_t* __restrict__ slot_mapping,
    const float* __restrict__ inv_freq, const float* __restrict__ value_inv_freq, int heads,
    int kv_heads, int dim, int vdim, int rot_dims, int interleaved, int64_t num_slots,
    const float* __restrict__ q_norm, const float* __restrict__ k_norm, float norm_eps,
    const typename S::T* __restrict__ v_other, int64_t v_other_stride,
    const float* __restrict__ v_blend, int head_norm) {
  using T = typename S::T;
  extern __shared__ float head_inv[];     // head_norm: 1 / rms of every query head, then of every key head
  __shared__ float red[16];
  __shared__ float2 sines[kMaxPairs];
  const int t = blockIdx.x;
  const float p = (float)positions[t];
  int64_t slot = slot_mapping[t];
  const bool cached = slot >= 0 && slot < num_slots;
  const int half = rot_dims / 2;
  const int rest = dim - rot_dims;
  for (int f = threadIdx.x; f < min(half, kMaxPairs); f += blockDim.x) {
    float2 sc;
    sincosf(p * inv_freq[f], &sc.x, &sc.y);
    sines[f] = sc;
  }
  __syncthreads();
  auto sine_of = [&](int f) {
    float2 sc;
    if (f < kMaxPairs)
      sc = sines[f];
    else
      sincosf(p * inv_freq[f], &sc.x, &sc.y);
    return sc;
  };
  T* qr = q + (int64_t)t * q_stride;
  const T* kr = k + (int64_t)t * k_stride;
  // RMS norm over the whole row (all heads at once) with a weight per element, before the rotation
  float q_inv = 1.f, k_inv = 1.f;
  if (head_norm) {
    // a quarter wave per head
    const int sub = threadIdx.x & 15;
    for (int h = threadIdx.x >> 4; h < heads + kv_heads; h += 16) {
      const T* hr = h < heads ? qr + h * dim : kr + (h - heads) * dim;
      float ss = 0.f;
      for (int d = sub; d < dim; d += 16) {
        const float x = S::to_f32(hr[d]);
        ss += x * x;
      }
#pragma unroll
      for (int m = 8; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, 16);
      if (sub == 0) head_inv[h] = 1.f / sqrtf(ss / (float)dim + norm_eps);
    }
    __syncthreads();
  }
  // factor of element i of query / key head h
  auto q_factor = [&](int h, int i) {
    return (head_norm ? head_inv[h] : q_inv) * (q_norm != nullptr ? q_norm[h * dim + i] : 1.f);
  };
  auto k_factor = [&](int h, int i) {
    return (head_norm ? head_inv[heads + h] : k_inv) * (k_norm != nullptr ? k_norm[h * dim + i] : 1.f);
  };
  const bool q_normed = head_norm || q_norm != nullptr, k_normed = head_norm || k_norm != nullptr;
  if (!head_norm && q_norm != nullptr) {
    float ss = 0.f;
    for (int i = threadIdx.x; i < heads * dim; i += blockDim.x) {
      const float x = S::to_f32(qr[i]);
      ss += x * x;
    }
    q_inv = 1.f / sqrtf(block_sum(ss, red) / (float)(heads * dim) + norm_eps);
  }
  if (!head_norm && k_norm != nullptr) {
    float ss = 0.f;
    for (int i = threadIdx.x; i < kv_heads * dim; i += blockDim.x) {
      const float x = S::to_f32(kr[i]);
      ss += x * x;
    }
    k_inv = 1.f / sqrtf(block_sum(ss, red) / (float)(kv_heads * dim) + norm_eps);
  }
  for (int i = threadIdx.x; i < heads * half; i += blockDim.x) {
    const int h = i / half, f = i - h * half;
    int ia, ib;
    pair_index(f, rot_dims, interleaved, ia, ib);
    float a = S::to_f32(qr[h * dim + ia]), b = S::to_f32(qr[h * dim + ib]);
    if (q_normed) {
      a *= q_factor(h, ia);
      b *= q_factor(h, ib);
    }
    turn_by(a, b, sine_of(f));
    qr[h * dim + ia] = S::from_f32(a);
    qr[h * dim + ib] = S::from_f32(b);
  }
  if (q_normed) {
    for (int i = threadIdx.x; i < heads * rest; i += blockDim.x) {
      const int h = i / rest, d = rot_dims + (i - h * rest);
      qr[h * dim + d] = S::from_f32(S::to_f32(qr[h * dim + d]) * q_factor(h, d));
    }
  }
  if (!cached) return;
  T* kc = key_cache + slot * (int64_t)kv_heads * dim;
  for (int i = threadIdx.x; i < kv_heads * half; i += blockDim.x) {
    const int h = i / half, f = i - h * half;
    int ia, ib;
    pair_index(f, rot_dims, interleaved, ia, ib);
    float a = S::to_f32(kr[h * dim + ia]), b = S::to_f32(kr[h * dim + ib]);
    if (k_normed) {
      a *= k_factor(h, ia);
      b *= k_factor(h, ib);
    }
    turn_by(a, b, sine_of(f));
    kc[h * dim + ia] = S::from_f32(a);
    kc[h * dim + ib] = S::from_f32(b);
  }
  for (int i = threadIdx.x; i < kv_heads * rest; i += blockDim.x) {
    const int h = i / rest, d = rot_dims + (i - h * rest);
    if (k_normed)
      kc[h * dim + d] = S::from_f32(S::to_f32(kr[h * dim + d]) * k_factor(h, d));
    else
      kc[h * dim + d] = kr[h * dim + d];
  }
  const T* vr = v + (int64_t)t * v_stride;
  T* vc = value_cache + slot * (int64_t)kv_heads * vdim;
  if (v_other != nullptr) {
    // the cached value is (1 - lambda) v + lambda v_other, v_other another layer's values of this token
    const float lam = v_blend[0];
    const T* vo = v_other + (int64_t)t * v_other_stride;
    for (int i = threadIdx.x; i < kv_heads * vdim; i += blockDim.x)
      vc[i] = S::from_f32((1.f - lam) * S::to_f32(vr[i]) + lam * S::to_f32(vo[i]));
    return;
  }
  if (value_inv_freq == nullptr) {
    for (int i = threadIdx.x; i < kv_heads * vdim; i += blockDim.x) vc[i] = vr[i];
    return;
  }
  const int vhalf = vdim / 2;
  for (int i = threadIdx.x; i < kv_heads * vhalf; i += blockDim.x) {
    const int h = i / vhalf, f = i - h * vhalf;
    int ia, ib;
    pair_index(f, vdim, interleaved, ia, ib);
    float a = S::to_f32(vr[h * vdim + ia]), b = S::to_f32(vr[h * vdim + ib]);
    turn(a, b, p * value_inv_freq[f]);
    vc[h * vdim + ia] = S::from_f32(a);
    vc[h * vdim + ib] = S::from_f32(b);
  }
  if (vdim & 1) {
    for (int h = threadIdx.x; h < kv_heads; h += blockDim.x)
      vc[h * vdim + vdim - 1] = vr[h * vdim + vdim - 1];
  }
}

// The same for 16-bit rows at multiples of 16 bytes without norms, blends or rotated values (rows_fit): one wave per token, 16
// bytes an access, pair 8 j .. + 7 of a head to a lane.  The kernel above is a chain of loads, each behind the store
// before it; here all of a token's rows (up to 4 x 64 pieces of queries) are asked for ahead of its sines.
// 5543 rows of 16 + 4 heads of 128 are 68 MB: 25 us above, 14 here.
constexpr int kRowPairs = 128;           // pairs of a head (and floats of LDS per token)
constexpr int kTurnWaves = 4;
struct RotaryRows {
  void* q;
  int64_t q_stride;
  const void* k;
  int64_t k_stride;
  const void* v;
  int64_t v_stride;
  void* key_cache;
  void* value_cache;
  const int64_t* positions;
  const int64_t* slot_mapping;
  const float* inv_freq;
  int64_t num_slots;
  int num_tokens, heads, kv_heads, dim, vdim, rot_dims, interleaved;
};

bool rows_fit(const RotaryRows& a) {
  const int eighth = a.rot_dims / 16;    // pieces of pairs of a head
  const uintptr_t at = (uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.key_cache | (uintptr_t)a.value_cache;
  return a.rot_dims > 0 && a.rot_dims % 16 == 0 && a.rot_dims / 2 <= kRowPairs && (int64_t)a.heads * eighth <= 2048 &&
         (int64_t)a.kv_heads * eighth <= 2048 && a.dim % 8 == 0 && a.dim - a.rot_dims <= 256 &&
         (int64_t)a.kv_heads * (a.dim - a.rot_dims) <= 2048 * 8 && (int64_t)a.kv_heads * a.vdim <= (1 << 20) &&
         (int64_t)a.kv_heads * a.vdim % 8 == 0 && (a.q_stride | a.k_stride | a.v_stride) % 8 == 0 && at % 16 == 0;
}

template <class S>
__global__ __launch_bounds__(64 * kTurnWaves) void rotary_kv_rows_kernel(RotaryRows a) {
  using T = typename S::T;
  __shared__ __align__(16) float2 sines[kTurnWaves][kRowPairs];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t = blockIdx.x * (blockDim.x >> 6) + w;
  if (t >= a.num_tokens) return;                     // a whole wave; no workgroup barriers below
  const int half = a.rot_dims / 2, eighth = half / 8, rest = (a.dim - a.rot_dims) / 8;
  const int inverse = (65536 + eighth - 1) / eighth;
  const int nq = a.heads * eighth, nk = a.kv_heads * eighth, nv = a.kv_heads * a.vdim / 8;
  const float p = (float)a.positions[t];
  const int64_t slot = a.slot_mapping[t];
  const bool cached = slot >= 0 && slot < a.num_slots;
  T* qr = (T*)a.q + (int64_t)t * a.q_stride;
  const T* kr = (const T*)a.k + (int64_t)t * a.k_stride;
  const T* vr = (const T*)a.v + (int64_t)t * a.v_stride;
  T* kc = (T*)a.key_cache + (cached ? slot : 0) * (int64_t)a.kv_heads * a.dim;
  T* vc = (T*)a.value_cache + (cached ? slot : 0) * (int64_t)a.kv_heads * a.vdim;
  const int second = a.interleaved ? 8 : half;       // elements from a lane's first piece to its second
  // item i: pairs 8 j .. + 7 of head h
  auto where = [&](int i, int& j) {
    const int h = quotient(i, inverse);
    j = i - h * eighth;
    return h * a.dim + (a.interleaved ? 16 : 8) * j;
  };
  auto fetch = [&](const T* row, int i) {
    int j;
    const T* at = row + where(i, j);
    return TurnPieces{*reinterpret_cast<const u32x4*>(at), *reinterpret_cast<const u32x4*>(at + second)};
  };
  auto turn_into = [&](T* row, int i, TurnPieces in) {
    int j;
    T* at = row + where(i, j);
    const TurnPieces out = turn_eight<S>(in, &sines[w][8 * j], a.interleaved);
    *reinterpret_cast<u32x4*>(at) = out.x;
    *reinterpret_cast<u32x4*>(at + second) = out.y;
  };
  constexpr int QU = 4, VU = 2;
  TurnPieces qp[QU], kp;
  u32x4 vp[VU];
#pragma unroll
  for (int u = 0; u < QU; ++u)
    if (kWave * u < nq) qp[u] = fetch(qr, min(lane + kWave * u, nq - 1));
  kp = fetch(kr, min(lane, nk - 1));
#pragma unroll
  for (int u = 0; u < VU; ++u)
    if (kWave * u < nv) vp[u] = *reinterpret_cast<const u32x4*>(vr + 8 * min(lane + kWave * u, nv - 1));
  for (int f = lane; f < half; f += kWave) {
    float2 sc;
    sincosf(p * a.inv_freq[f], &sc.x, &sc.y);
    sines[w][f] = sc;
  }
  wave_sync();
#pragma unroll
  for (int u = 0; u < QU; ++u)
    if (lane + kWave * u < nq) turn_into(qr, lane + kWave * u, qp[u]);
  for (int i = lane + QU * kWave; i < nq; i += kWave) turn_into(qr, i, fetch(qr, i));
  if (!cached) return;
  if (lane < nk) turn_into(kc, lane, kp);
  for (int i = lane + kWave; i < nk; i += kWave) turn_into(kc, i, fetch(kr, i));
  if (rest > 0) {
    const int inverse_rest = (65536 + rest - 1) / rest;
    for (int i = lane; i < a.kv_heads * rest; i += kWave) {
      const int h = quotient(i, inverse_rest), d = h * a.dim + a.rot_dims + 8 * (i - h * rest);
      *reinterpret_cast<u32x4*>(kc + d) = *reinterpret_cast<const u32x4*>(kr + d);
    }
  }
#pragma unroll
  for (int u = 0; u < VU; ++u)
    if (lane + kWave * u < nv) *reinterpret_cast<u32x4*>(vc + 8 * (lane + kWave * u)) = vp[u];
  for (int i = lane + VU * kWave; i < nv; i += kWave)
    *reinterpret_cast<u32x4*>(vc + 8 * i) = *reinterpret_cast<const u32x4*>(vr + 8 * i);
}

// The epilogue every attention kernel of this file shares: o_lds holds one head's normalized
// output [vdim] in fp32; turn pair m back by the query's position, gate, write.
template <class S>
__device__ __forceinline__ void write_head_output(typename S::T* __restrict__ orow,
                                                  const float* __restrict__ o_lds, int vdim, float p,
                                                  const float* __restrict__ out_inv_freq,
                                                  int interleaved, float gate, int first, int step) {
  const int vhalf = vdim / 2;
  for (int d = first; d < vdim; d += step) {
    float val = o_lds[d];
    if (out_inv_freq != nullptr && d < 2 * vhalf) {
      int f, other;
      bool is_a;
      if (interleaved) {
        f = d >> 1;
        is_a = (d & 1) == 0;
        other = d ^ 1;
      } else {
        is_a = d < vhalf;
        f = is_a ? d : d - vhalf;
        other = is_a ? d + vhalf : d - vhalf;
      }
      float s, c;
      sincosf(p * out_inv_freq[f], &s, &c);
      // turned by the negative angle: (a cos + b sin, b cos - a sin)
      val = is_a ? val * c + o_lds[other] * s : val * c - o_lds[other] * s;
    }
    orow[d] = S::from_f32(val * gate);
  }
}

template <class S, int kAccum>    // kAccum values per lane: rows of up to 64 kAccum
__global__ __launch_bounds__(kWave* kHeadsPerGroup) void kv_attention_kernel(
    typename S::T* __restrict__ out, int64_t out_stride, const typename S::T* __restrict__ q,
    int64_t q_stride, const typename S::T* __restrict__ gate, int64_t gate_stride,
    const typename S::T* __restrict__ key_cache, const typename S::T* __restrict__ value_cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ token_seq,
    const int64_t* __restrict__ positions, const float* __restrict__ out_inv_freq, int interleaved,
    int heads, int kv_heads, int dim, int vdim, int block_size, int num_blocks, int window,
    float scale, int keep_first, float softcap, int chunk, const float* __restrict__ sinks) {
  __shared__ float q_lds[kHeadsPerGroup][kWave * kAccum];
  __shared__ float p_lds[kHeadsPerGroup][kWave];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int t = blockIdx.x;
  const int h = blockIdx.y * kHeadsPerGroup + w;
  if (h >= heads) return;  // whole wave; no workgroup barrier below
  const int g = h / (heads / kv_heads);
  const int p = (int)positions[t];
  const int* table = block_tables + (int64_t)token_seq[t] * max_blocks;
  const int lo = first_key(p, window, chunk);
  const int nk = min(keep_first, lo);         // kept keys ahead of the window
  const int total = nk + p - lo + 1;
  auto key_of = [&](int u) { return u < nk ? u : u - nk + lo; };
  for (int d = lane; d < dim; d += kWave)
    q_lds[w][d] = S::to_f32(q[(int64_t)t * q_stride + (int64_t)h * dim + d]) * scale;
  wave_sync();
  // a block id outside the pool (a table the host filled wrongly) reads block 0 instead of faulting
  auto token_row = [&](int j) {
    int b = table[j / block_size];
    b = (unsigned)b < (unsigned)num_blocks ? b : 0;
    return ((int64_t)b * block_size + j % block_size) * kv_heads + g;
  };

  float acc[kAccum];
#pragma unroll
  for (int c = 0; c < kAccum; ++c) acc[c] = 0.f;
  // a sink is a term of the denominator that was there first
  float m = sinks != nullptr ? sinks[h] : -INFINITY, l = sinks != nullptr ? 1.f : 0.f;
  for (int u0 = 0; u0 < total; u0 += kWave) {
    const int u = u0 + lane;
    float s = -INFINITY;
    if (u < total) {
      const typename S::T* kr = key_cache + token_row(key_of(u)) * dim;
      float dot = 0.f;
      for (int d = 0; d < dim; ++d) dot += q_lds[w][d] * S::to_f32(kr[d]);
      s = softcap > 0.f ? cap_score(dot, softcap) : dot;
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float pj = u < total ? expf(s - m_new) : 0.f;
    const float corr = expf(m - m_new);  // first tile: exp(-inf) = 0
    l = l * corr + wave_sum(pj);
    m = m_new;
    wave_sync();
    p_lds[w][lane] = pj;
    wave_sync();
#pragma unroll
    for (int c = 0; c < kAccum; ++c) acc[c] *= corr;
    const int n = min(kWave, total - u0);
    for (int jj = 0; jj < n; ++jj) {
      const typename S::T* vr = value_cache + token_row(key_of(u0 + jj)) * vdim;
      const float pv = p_lds[w][jj];
#pragma unroll
      for (int c = 0; c < kAccum; ++c) {
        const int d = lane + c * kWave;
        if (d < vdim) acc[c] += pv * S::to_f32(vr[d]);
      }
    }
  }
  wave_sync();
  const float inv = 1.f / l;
#pragma unroll
  for (int c = 0; c < kAccum; ++c) {
    const int d = lane + c * kWave;
    if (d < vdim) q_lds[w][d] = acc[c] * inv;   // the query is done with
  }
  wave_sync();
  float gv = 1.f;
  if (gate != nullptr) gv = 1.f / (1.f + expf(-S::to_f32(gate[(int64_t)t * gate_stride + h])));
  write_head_output<S>(out + (int64_t)t * out_stride + (int64_t)h * vdim, q_lds[w], vdim, (float)p,
                       out_inv_freq, interleaved, gv, lane, kWave);
}


// ---------------------------------------------------------------------------------------------
// Matrix-core kernels for 16-bit models.  Both products run in transposed form on 32x32x8 MFMAs,
// lane = (hf, c) = (lane >> 5, lane & 31):
//   S^T = K q^T   A = K    lane: key c, dims 8 ks + 4 hf .. + 3
//                 B = q^T  lane: query c, the same dims (registers, loaded once)
//                 C        lane: query c, keys (i & 3) + 8 (i >> 2) + 4 hf, i = 0 .. 15
//   O^T = V^T P^T A = V^T  lane: value dim 32 n + c, keys 8 s + 4 hf .. + 3
//                 B = P^T  lane: query c, the same keys = registers 4 s .. 4 s + 3 of C above
//                 C        lane: query c, dims 32 n + (i & 3) + 8 (i >> 2) + 4 hf
// so a lane owns one query's scores, running max / sum and output column, and both elements of
// every rotated output pair (neighbours when interleaved; vdim / 2 = 16 (vdim / 32) apart
// otherwise, which moves n and i >> 2 but neither hf nor c).  Scores leave the first product in
// fp32 and stay there; a weight enters the second product as the sum of two 16-bit numbers (its
// rounding and the rounding of what the rounding lost).
template <class S>
struct Mfma8;
template <>
struct Mfma8<BF16> {
  typedef short V4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ f32x16 run(u32x2 a, u32x2 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(V4, a), __builtin_bit_cast(V4, b), c,
                                                    0, 0, 0);
  }
};
template <>
struct Mfma8<F16> {
  typedef _Float16 V4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ f32x16 run(u32x2 a, u32x2 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(V4, a), __builtin_bit_cast(V4, b), c, 0,
                                                0, 0);
  }
};
template <class S>
__device__ __forceinline__ uint32_t bits16(float v) {
  return (uint32_t)__builtin_bit_cast(uint16_t, S::from_f32(v));
}
template <class S>
__device__ __forceinline__ float from_bits16(uint32_t b) {
  return S::to_f32(__builtin_bit_cast(typename S::T, (uint16_t)b));
}

constexpr int kTile = 32;
std::atomic<int> g_kv_kernel{0};

// dim index of register i of output block n for lane half hf
__device__ __forceinline__ constexpr int out_dim(int n, int i, int hf) {
  return 32 * n + (i & 3) + 8 * (i >> 2) + 4 * hf;
}

// Turns the output pairs a lane holds back by the query's position (o[n][i] normalized already).
template <int VB>
__device__ __forceinline__ void turn_back(f32x16 (&o)[VB], int hf, float p,
                                          const float* __restrict__ out_inv_freq, int interleaved) {
  constexpr int VD = 32 * VB;
  if (interleaved) {
#pragma unroll
    for (int n = 0; n < VB; ++n)
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        float s, c;
        sincosf(p * out_inv_freq[out_dim(n, i, hf) >> 1], &s, &c);
        const float a = o[n][i], b = o[n][i + 1];
        o[n][i] = a * c + b * s;
        o[n][i + 1] = b * c - a * s;
      }
  } else {
    // partner of dim d < VD / 2 is d + 16 VB: block n + VB / 2 (and, for odd VB, i + 8)
#pragma unroll
    for (int n = 0; n < VB; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int d = 32 * n + (i & 3) + 8 * (i >> 2);      // without 4 hf: same for both halves
        if (d < VD / 2) {
          const int d2 = d + VD / 2;
          const int n2 = d2 / 32, r2 = d2 % 32;
          const int i2 = (r2 & 3) + 4 * (r2 >> 3);
          float s, c;
          sincosf(p * out_inv_freq[d + 4 * hf], &s, &c);
          const float a = o[n][i], b = o[n2][i2];
          o[n][i] = a * c + b * s;
          o[n2][i2] = b * c - a * s;
        }
      }
  }
}

// kv_attention_tile_kernel<S, DB, VB>: runs of rows (prompts, portions), on 32x32x16 MFMAs.  One
// workgroup per (sequence, tile of query rows, KV head, chunk of its query heads).  Its four waves
// are (query head of the chunk) x (block of 32 consecutive rows): 4 x 1 for groups of three heads
// and more, 2 x 2 for two, 1 x 4 for one, so a tile is 32, 64 or 128 rows.  Keys and values from
// the first row's window start to the last row walk through LDS in tiles of 64; the rows' places in
// the paged caches are looked up once per tile by 64 threads, two tiles ahead.
//   S^T = K q^T   A = K    lane: key c of a 32-key block, dims 16 ks + 8 hf .. + 7   (LDS, 16 bytes)
//                 B = q^T  lane: query c, the same dims (registers, loaded once)
//                 C        lane: query c, keys (i & 3) + 8 (i >> 2) + 4 hf, i = 0 .. 15
//   O^T = V^T P^T B = P^T  lane: query c, registers 8 s .. 8 s + 7 of C = keys 16 s + 4 hf + {0..3, 8..11}
//                 A = V^T  lane: value dim 32 n + c of the same eight keys (two transposing reads
//                          of the row-major tile)
// The k index of the second product is a free relabelling of the keys, so the weights go from the
// first product's result to the second's operand without leaving the lane.  Scores, running
// max / sum (base 2) and the accumulators are fp32; a weight enters the second product rounded to
// the model dtype.
//
// Bound by the vector port and the chain from the scores over their maximum to the second product: a wave alone takes
// 3000 cycles for a tile (1024 of products, 1200 of vector instructions), two that share a SIMD 4500 for one each; counted over
// the kernel, vector instructions take 50 % of a CU's busy cycles and matrix cores 35 %, at 2.3 GHz.  Tiles come in by LDS-DMA: no staging registers, no waits before the stores to LDS, one barrier per tile, two
// tiles in LDS (64 KB at most and the rows' places: two workgroups share a CU and one's softmax runs under
// the other's products).  A DMA instruction writes 64 lanes x 16 bytes in a row, so rows cannot be padded: 16-byte
// pieces of a key row and 64-byte units of a value row are exchanged by the row's number on the source's
// side, so that the lanes of a read fall into different banks.  The next tile's DMA goes out between the first products
// (sent at once it holds a wave up for 700 cycles), weights are formed between the second ones.  What is the same for
// all lanes is told to the compiler, or every choice of a mask or a scale copies the 32 scores.  Workgroups go out
// longest walk first over all sequences, groups of heads next to each other: each XCD's L2 holds few heads' keys.
// Where the workgroups are few, each has two groups of four waves (KG = 2) that take every other tile and join their
// sums at the end.  Four prompts of up to 2047 rows, 16 heads on 4 of 128: 65 us (104 with DMA in a burst, masks for
// all tiles of a run's last rows and a grid as long as the longest prompt for each; 172 with tiles staged through
// registers into padded rows).
template <class S>
struct Mfma16;
template <>
struct Mfma16<BF16> {
  static __device__ __forceinline__ f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                   c, 0, 0, 0);
  }
};
template <>
struct Mfma16<F16> {
  static __device__ __forceinline__ f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                  0, 0, 0);
  }
};

constexpr int kKeys = 64;     // keys per staged tile
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef s16x4 __attribute__((address_space(3))) * lds_s16x4;

// two fp32 -> one word of two model-dtype values (round to nearest even), as one packed convert
template <class S>
__device__ __forceinline__ uint32_t pack2(float a, float b);
template <>
__device__ __forceinline__ uint32_t pack2<F16>(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
}
template <>
__device__ __forceinline__ uint32_t pack2<BF16>(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// which units of 64 bytes of a value row change place: rows whose units would meet in the banks
template <int VB>
__device__ __forceinline__ int value_exchange(int r) {
  return VB == 4 ? r & 3 : VB == 2 ? (r >> 1) & 1 : 0;
}

template <class S, int DB, int VB, int KG>
__global__ __launch_bounds__(256 * KG, 2) void kv_attention_tile_kernel(
    typename S::T* __restrict__ out, int64_t out_stride, const typename S::T* __restrict__ q,
    int64_t q_stride, const typename S::T* __restrict__ gate, int64_t gate_stride,
    const typename S::T* __restrict__ key_cache, const typename S::T* __restrict__ value_cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ query_start_loc,
    const int* __restrict__ context_lens, const float* __restrict__ out_inv_freq, int interleaved,
    int heads, int kv_heads, int head_groups, int block_size, int num_blocks, int window, float scale, int head_waves,
    int keep_first, float softcap, int chunk, const float* __restrict__ sinks, int v_row, int v_first,
    int last_tile, int ranked_seqs, int first_rank) {
  using T = typename S::T;
  using M = Mfma16<S>;
  constexpr int D = 32 * DB, VD = 32 * VB;
  constexpr int KB = 2 * D, VBYTES = 2 * VD;           // bytes of a tile's rows
  constexpr int kStep = kKeys * KG;                    // keys of a step: a tile for every group of four waves
  constexpr int KTILE = kKeys * KB, VTILE = kKeys * VBYTES, STAGE = KTILE + VTILE;
  // which 16-byte pieces of a key row change place: the rows of 16 lanes begin at one, two or four places
  // among the banks, and the exchange spreads those that begin at the same one
  constexpr int KMASK = DB == 4 ? 15 : DB == 2 ? 7 : 3, KSHIFT = DB == 4 ? 0 : DB == 2 ? 1 : 2;
  // two tiles for every group of waves: one is read while the next lands
  __shared__ __align__(16) unsigned char all_tiles[KG * 2 * STAGE];
  __shared__ uint32_t all_rows[KG][2][kKeys];          // the cache row (slot) of each key of a tile
  const int yb = blockIdx.x % head_groups;
  const int row_blocks = 4 / head_waves;              // blocks of 32 query rows per workgroup
  const int tile_rows = kTile * row_blocks;
  // the last tiles of a run have the most keys to walk: they are dispatched first
  int b = blockIdx.x / head_groups, tile_x = last_tile - (int)blockIdx.y;
  int first_row, run, context;
  if (ranked_seqs > 0) {
    const int rank = first_rank + b;
    const RankedTile found = ranked_tile<false>(rank, ranked_seqs, query_start_loc, context_lens, __builtin_ctz(tile_rows), last_tile + 1);
    if (rank >= found.all) return;
    b = found.seq;
    tile_x = found.tile;
    first_row = found.first_row;
    run = found.rows;
    context = found.context;
  } else {
    if (ranked_seqs < 0) {                            // in the order of the rows
      const int at = first_rank + b;
      b = at / (last_tile + 1);
      tile_x = last_tile - (at - b * (last_tile + 1));
    }
    first_row = query_start_loc[b];
    run = query_start_loc[b + 1] - first_row;
    context = context_lens[b];
  }
  const int t_first = first_row + tile_rows * tile_x;
  const int n_tile = min(tile_rows, run - tile_rows * tile_x);
  if (n_tile <= 0) return;
  const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);      // group of waves
  const int tid = threadIdx.x & 255, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* tiles = all_tiles + kg * 2 * STAGE;
  auto& rows_lds = all_rows[kg];
  const int hf = lane >> 5, c = lane & 31;
  const int group = heads / kv_heads;
  const int chunks = (group + head_waves - 1) / head_waves;
  const int g = yb / chunks;
  const int h = g * group + (yb % chunks) * head_waves + w % head_waves;
  const int rb = w / head_waves;                      // this wave's block of rows
  const int t0 = t_first + kTile * rb;
  const int nq = min(kTile, n_tile - kTile * rb);     // <= 0: no rows for this wave
  const bool active = h < g * group + group && nq > 0;
  const int p_first = context + tile_rows * tile_x, p_last = p_first + n_tile - 1;
  const int p0 = p_first + kTile * rb;                // this wave's first position
  const int pq = p0 + c;
  // (the compiler does not see that a remainder is the same for all lanes, and would take every branch on it for one
  // that is not)
  const int j_lo = __builtin_amdgcn_readfirstlane(first_key(p_first, window, chunk));
  const int lo_q = first_key(pq, window, chunk);      // this lane's row's first key
  // of the wave's first row and of its last
  const int lo_first = __builtin_amdgcn_readfirstlane(first_key(p0, window, chunk));
  const int lo_last = __builtin_amdgcn_readfirstlane(first_key(p0 + kTile - 1, window, chunk));
  // the keys this workgroup walks, through one index: the kept first tokens that lie ahead of the
  // first row's window, then the window's first key to the last row
  const int nk = min(keep_first, j_lo);
  const int total = nk + p_last - j_lo + 1;
  auto key_of = [&](int u) { return u < nk ? u : u - nk + j_lo; };
  // in that index, a row sees u <= last and (u >= least or u < kept); the same for the wave's rows together
  const int kept = nk == j_lo ? keep_first : nk;
  const int last_q = pq + nk - j_lo, least_q = lo_q + nk - j_lo;
  const int last_first = p0 + nk - j_lo, last_last = last_first + nq - 1;
  const int least_first = lo_first + nk - j_lo, least_last = lo_last + nk - j_lo;
  const int* table = block_tables + (int64_t)b * max_blocks;
  const float scale2 = scale * 1.4426950408889634f;   // scores in base 2
  const float cap2 = softcap * 1.4426950408889634f, cap_arg = softcap > 0.f ? 2.f * 1.4426950408889634f / softcap : 0.f;
  // a positive scale is left to the exponent's fused product; otherwise scores are scaled before the maximum
  const bool late = softcap <= 0.f && scale2 > 0.f;

  f32x16 o[VB];
#pragma unroll
  for (int n = 0; n < VB; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[n][i] = 0.f;
  float m = -INFINITY, top = 0.f, l = 0.f;            // top: m, and 0 where nothing was seen yet
  if (sinks != nullptr && active && kg == 0) {     // the denominator's first term, counted in one lane half
    m = sinks[h] * 1.4426950408889634f;
    top = m == -INFINITY ? 0.f : m;                   // (a sink that counts for nothing, also where base 2 overflows)
    l = hf == 0 ? __builtin_amdgcn_exp2f(m - top) : 0.f;       // 1, 0 or, for an infinite one, NaN
  }

  // the first wave looks the rows of a tile up: the block id is read one step before it is used
  const bool shifts = (block_size & (block_size - 1)) == 0;
  const int shift = __builtin_ctz(block_size);
  struct Place {
    int blk, at;
  };
  auto look_up = [&](int u0) {
    const int j = key_of(min(u0 + lane, total - 1));   // behind the end: the last key again, masked
    const int nb = shifts ? j >> shift : j / block_size;
    return Place{table[nb], j - nb * block_size};      // not looked at yet: that would wait for it, and for the DMA
  };
  auto store_row = [&](Place p, int buf) {
    const int blk = (unsigned)p.blk < (unsigned)num_blocks ? p.blk : 0;
    rows_lds[buf][lane] = (uint32_t)blk * (uint32_t)block_size + (uint32_t)p.at;      // a card holds fewer than 2^32 rows
  };
  // what this lane brings in: the row of a tile, and the piece of it that stands at the lane's place
  constexpr int kPieces = DB + VB;                     // DMA instructions of a wave
  int row_of[kPieces];
  const unsigned char* from[kPieces];                  // where the piece of cache row 0 lies
#pragma unroll
  for (int u = 0; u < DB; ++u) {
    const int at = (w * DB + u) * 64 + lane, r = at / (KB / 16), p = at % (KB / 16);
    row_of[u] = r;
    from[u] = (const unsigned char*)key_cache + (size_t)g * KB + 16 * ((p & ~KMASK) | ((p ^ (r >> KSHIFT)) & KMASK));
  }
#pragma unroll
  for (int u = 0; u < VB; ++u) {
    const int at = (w * VB + u) * 64 + lane, r = at / (VBYTES / 16), p = at % (VBYTES / 16);
    row_of[DB + u] = r;
    from[DB + u] = (const unsigned char*)value_cache + (size_t)g * (2 * v_row) + 2 * v_first +
                   16 * ((((p >> 2) ^ value_exchange<VB>(r)) << 2) | (p & 3));
  }
  const uint32_t key_row = (uint32_t)kv_heads * KB, value_row = (uint32_t)kv_heads * 2 * v_row;
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)tiles;
  uint32_t slot[kPieces];
  auto slots_of = [&](int buf) {                       // the rows of the tile that is brought in next
#pragma unroll
    for (int i = 0; i < kPieces; ++i) slot[i] = DB == VB && i >= DB ? slot[i - DB] : rows_lds[buf][row_of[i]];
  };
  auto bring = [&](int i, int buf, int go) {           // piece i of that tile into buffer buf
    const uint32_t to = lds0 + buf * STAGE + (i < DB ? (w * DB + i) * 1024 : KTILE + (w * VB + i - DB) * 1024);
    tile_dma16(from[i] + (uint64_t)slot[i] * (i < DB ? key_row : value_row), to, go);
  };
  // where this lane reads: the exchanged piece of its key row, and the unit of its value rows
  const int kx = (hf ^ (c >> KSHIFT)) & KMASK;         // piece 2 ks + hf stands at 2 ks ^ kx within its group
  const int i16 = c & 15;
  const int vr = 4 * hf + (i16 >> 2);
  const int vf = value_exchange<VB>(vr);               // 8 and 16 rows further on it is the same
  const int vat = vr * VBYTES + 32 * (c >> 4) + 8 * (i16 & 3);

  // One barrier per tile.  Behind it in step `it`: tile `it` is in its buffer, the rows of tile it + 1 are in
  // rows_lds[(it + 1) & 1], and the first wave holds the block ids of tile it + 2.
  // (the first three ids are asked for together, ahead of the query rows: nothing waits for more than it needs)
  Place next = {0, 0}, first = {0, 0}, second = {0, 0};
  if (w == 0) {
    const int u = kg * kKeys;
    first = look_up(u);
    second = look_up(u + kStep);
    next = look_up(u + 2 * kStep);
  }
  __builtin_amdgcn_sched_barrier(0);
  u32x4 qf[D / 16];
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (active && c < nq)
      v = *reinterpret_cast<const u32x4*>(q + (int64_t)(t0 + c) * q_stride + (int64_t)h * D + 16 * ks + 8 * hf);
    qf[ks] = v;
  }
  __builtin_amdgcn_sched_barrier(0);
  if (w == 0) {
    store_row(first, 0);
    store_row(second, 1);
  }
  __syncthreads();
  slots_of(0);
#pragma unroll
  for (int i = 0; i < kPieces; ++i) bring(i, 0, kg * kKeys < total);
  const int steps = (total + kStep - 1) / kStep;
  // the loop once for scores that go to the exponent as they are and once for the others: both in one cost the
  // first 32 moves a step
  auto walk = [&](auto scaled_late) {
  constexpr bool kLate = decltype(scaled_late)::value;
  for (int it = 0; it < steps; ++it) {
    const int u0 = it * kStep + kg * kKeys;
    // the builtin and not asm: the compiler then knows that the query rows have arrived, and does not wait for
    // vmcnt(0), and so for the DMA just started, at their first use in every step
    __builtin_amdgcn_s_waitcnt(0x0f70);                // vmcnt(0)
    asm volatile("" ::: "memory");
    __syncthreads();
    const int more = __builtin_amdgcn_readfirstlane(u0 + kStep < total), into = (it + 1) & 1;
    slots_of(into);
    const unsigned char* k_lds = tiles + (it & 1) * STAGE;
    const unsigned char* v_lds = k_lds + KTILE;
    // a tile that no row of this wave sees is none of its business
    const bool concerned = active && u0 < total && u0 <= last_last && (u0 < kept || u0 + kKeys > least_first);
    f32x16 st[2];
    if (concerned) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) st[kb][i] = 0.f;
      // keys are read two steps ahead of their products, which the compiler would not do by itself, and the next
      // tile's DMA goes out between the products: a burst of it holds a wave up for longer than half of them take
      auto key_at = [&](int ks, int kb) {
        const int piece = ((2 * ks) & ~KMASK) | (((2 * ks) & KMASK) ^ kx);
        return *reinterpret_cast<const u32x4*>(k_lds + (32 * kb + c) * KB + 16 * piece);
      };
      u32x4 ka[3][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) ka[ks][kb] = key_at(ks, kb);
#pragma unroll
      for (int ks = 0; ks < 2 * DB; ++ks) {
        if (ks + 2 < 2 * DB) {
#pragma unroll
          for (int kb = 0; kb < 2; ++kb) ka[(ks + 2) % 3][kb] = key_at(ks + 2, kb);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) st[kb] = M::run(ka[ks % 3][kb], qf[ks], st[kb]);
#pragma unroll
        for (int i = 0; i < kPieces; ++i)
          if (i * (2 * DB) / kPieces == ks) bring(i, into, more);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int i = 0; i < kPieces; ++i) bring(i, into, more);
    }
    if (w == 0) {
      store_row(next, it & 1);                         // (the rows of tile `it` were read ahead of the barrier)
      next = look_up(u0 + 3 * kStep);
    }
    if (!concerned) continue;
    // Values: a transposing read of the row-major tile.  A group of 16 lanes reads 4 keys x 16 dims, 8 bytes per
    // lane (key i16 >> 2, dims 4 (i16 & 3) .. + 3), and every lane receives the four keys of dim i16 of the group.
    u32x4 va[2][VB];
    auto value_at = [&](int s4, int n) {               // keys 16 s4 .. + 15, dims 32 n ..
      const unsigned char* at = v_lds + vat + 16 * s4 * VBYTES + 64 * (n ^ vf);
      const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)at));
      const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(at + 8 * VBYTES)));
      return u32x4{lo[0], lo[1], hi[0], hi[1]};
    };
#pragma unroll
    for (int n = 0; n < VB; ++n) va[0][n] = value_at(0, n);
    if constexpr (!kLate) {
      if (softcap > 0.f) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i) st[kb][i] = cap_score_fast(st[kb][i] * scale, cap2, cap_arg);
      } else {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i) st[kb][i] *= scale2;
      }
    }
    // Masks, only where some key of the tile is hidden from some row of the wave, against numbers that are known when
    // it is compiled; rows behind the run's end (c >= nq) may see anything, nobody writes them.
    if (u0 + kKeys - 1 > last_first || (u0 < least_last && u0 + kKeys > kept)) {
      const int last = last_q - u0 - 4 * hf, least = least_q - u0 - 4 * hf, held = kept - u0 - 4 * hf;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int e = 32 * kb + (i & 3) + 8 * (i >> 2);
          st[kb][i] = e <= last && (e >= least || e < held) ? st[kb][i] : -INFINITY;
        }
    }
    float mts[2] = {-INFINITY, -INFINITY};             // chains of their own
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) mts[kb] = fmaxf(mts[kb], st[kb][i]);
    const float mt = max_halves(fmaxf(mts[0], mts[1])) * (kLate ? scale2 : 1.f);
    // (a maximum that may lag behind, by 8 in base 2, leaves the accumulators alone in most tiles and is 2.5 % faster, but
    // the largest weight is then no longer 1 and rounds like the others: errors grow by 1 to 2 %)
    if (__any(mt > m)) {
      const float m_new = fmaxf(m, mt);
      top = m_new == -INFINITY ? 0.f : m_new;          // nothing seen yet: every weight is 2^-inf
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
      const float a0 = st[s4 >> 1][8 * (s4 & 1) + 2 * e];
      const float b0 = st[s4 >> 1][8 * (s4 & 1) + 2 * e + 1];
      const float a = __builtin_amdgcn_exp2f(kLate ? __builtin_fmaf(a0, scale2, -top) : a0 - top);
      const float b = __builtin_amdgcn_exp2f(kLate ? __builtin_fmaf(b0, scale2, -top) : b0 - top);
      l += a;
      l += b;
      return pack2<S>(a, b);
    };
    u32x4 pb[2];
#pragma unroll
    for (int e = 0; e < 4; ++e) pb[0][e] = weight2(0, e);
    // the next 16 keys' weights are formed between the products of these
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      if (s4 < 3) {
#pragma unroll
        for (int n = 0; n < VB; ++n) va[(s4 + 1) & 1][n] = value_at(s4 + 1, n);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < VB; ++n) {
        o[n] = M::run(va[s4 & 1][n], pb[s4 & 1], o[n]);
        if (s4 < 3) {
#pragma unroll
          for (int e = 4 * n / VB; e < 4 * (n + 1) / VB; ++e) pb[(s4 + 1) & 1][e] = weight2(s4 + 1, e);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  };
  if (late)
    walk(std::true_type{});
  else
    walk(std::false_type{});
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
  }
  if (!active) return;
  l += __shfl_xor(l, 32, 64);
  if (c >= nq) return;
  const float inv = 1.f / l;
#pragma unroll
  for (int n = 0; n < VB; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[n][i] *= inv;
  if (out_inv_freq != nullptr) turn_back<VB>(o, hf, (float)pq, out_inv_freq, interleaved);
  float gv = 1.f;
  if (gate != nullptr) gv = 1.f / (1.f + expf(-S::to_f32(gate[(int64_t)(t0 + c) * gate_stride + h])));
  T* orow = out + (int64_t)(t0 + c) * out_stride + (int64_t)h * v_row + v_first;
  if (((uintptr_t)out | (uintptr_t)(out_stride * 2)) % 8 == 0) {
#pragma unroll
    for (int n = 0; n < VB; ++n)
#pragma unroll
      for (int i = 0; i < 16; i += 4)
        *reinterpret_cast<u32x2*>(orow + out_dim(n, i, hf)) =
            u32x2{pack2<S>(o[n][i] * gv, o[n][i + 1] * gv), pack2<S>(o[n][i + 2] * gv, o[n][i + 3] * gv)};
  } else {
#pragma unroll
    for (int n = 0; n < VB; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) orow[out_dim(n, i, hf)] = S::from_f32(o[n][i] * gv);
  }
}

// kv_attention_heads_kernel<S, DB, VB>: single rows (decode steps).  One workgroup per (row, KV
// head, chunk of up to 32 of its query heads): the 32 columns of the products hold the chunk's
// query heads, so each key and value byte is read once per KV head whatever the group size.  The
// kRowWaves waves split the window's tiles (wave w takes tiles w, w + kRowWaves, ...), each with
// its own key and value tiles in LDS and its own running max / sum / output, merged at the end.
constexpr int kRowWaves = 8;

template <class S, int DB, int VB>
__global__ __launch_bounds__(64 * kRowWaves) void kv_attention_heads_kernel(
    typename S::T* __restrict__ out, int64_t out_stride, const typename S::T* __restrict__ q,
    int64_t q_stride, const typename S::T* __restrict__ gate, int64_t gate_stride,
    const typename S::T* __restrict__ key_cache, const typename S::T* __restrict__ value_cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ token_seq,
    const int64_t* __restrict__ positions, const float* __restrict__ out_inv_freq, int interleaved,
    int heads, int kv_heads, int block_size, int num_blocks, int window, float scale,
    int merge_heads, int keep_first, float softcap, int chunk, const float* __restrict__ sinks,
    int v_row, int v_first) {
  using T = typename S::T;
  using M = Mfma8<S>;
  constexpr int D = 32 * DB, VD = 32 * VB;
  constexpr int KROW = D + 4, VROW = VD + 4;
  constexpr int WAVE_ELEMS = kTile * (KROW + VROW);       // one wave's two tiles, in elements
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int hf = lane >> 5, c = lane & 31;
  T* k_lds = reinterpret_cast<T*>(smem) + (size_t)w * WAVE_ELEMS;
  T* v_lds = k_lds + kTile * KROW;
  const int t = blockIdx.x;
  const int group = heads / kv_heads;
  const int chunks = (group + 31) / 32;
  const int g = blockIdx.y / chunks;
  const int h0 = g * group + (blockIdx.y % chunks) * 32;
  const int nh = min(32, g * group + group - h0);
  const int p = (int)positions[t];
  const int* table = block_tables + (int64_t)token_seq[t] * max_blocks;
  const int lo = first_key(p, window, chunk);
  const int nk = min(keep_first, lo);         // kept keys ahead of the window
  const int total = nk + p - lo + 1;
  const float cap_arg = softcap > 0.f ? 2.f * 1.4426950408889634f / softcap : 0.f;
  const bool live = c < nh;
  u32x2 qf[D / 8];
#pragma unroll
  for (int ks = 0; ks < D / 8; ++ks) {
    u32x2 v = {0u, 0u};
    if (live)
      v = *reinterpret_cast<const u32x2*>(q + (int64_t)t * q_stride + (int64_t)(h0 + c) * D + 8 * ks + 4 * hf);
    qf[ks] = v;
  }
  f32x16 o[VB];
#pragma unroll
  for (int n = 0; n < VB; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[n][i] = 0.f;
  float m = -INFINITY, l = 0.f;
  if (sinks != nullptr && live && w == 0) {   // the denominator's first term, counted by one wave's lane half
    m = sinks[h0 + c];
    l = hf == 0 ? 1.f : 0.f;
  }

  // A wave's share of a tile is D / 8 + VD / 8 pieces of 8 bytes per lane, all issued before any
  // is used and one tile ahead.  Lanes 0..31 look the 32 tokens of the tile up once and hand the
  // row numbers round with shuffles.
  constexpr int KP = D / 8, VP = VD / 8;
  u32x2 xk[KP], xv[VP];
  auto fetch = [&](int u0) {
    const int ur = u0 + c;
    long long row = -1;
    if (ur < total) {
      const int jr = ur < nk ? ur : ur - nk + lo;
      int blk = table[jr / block_size];
      blk = (unsigned)blk < (unsigned)num_blocks ? blk : 0;
      row = ((long long)blk * block_size + jr % block_size) * kv_heads + g;
    }
#pragma unroll
    for (int u = 0; u < KP; ++u) {
      const int i = lane + kWave * u;
      const int r = i / (D / 4), v = i % (D / 4);
      const long long rb = __shfl(row, r, 64);
      const u32x2 got = *reinterpret_cast<const u32x2*>(key_cache + (rb >= 0 ? rb * D + 4 * v : 0));
      xk[u] = rb >= 0 ? got : u32x2{0u, 0u};
    }
#pragma unroll
    for (int u = 0; u < VP; ++u) {
      const int i = lane + kWave * u;
      const int r = i / (VD / 4), v = i % (VD / 4);
      const long long rb = __shfl(row, r, 64);
      const u32x2 got = *reinterpret_cast<const u32x2*>(value_cache + (rb >= 0 ? rb * v_row + v_first + 4 * v : 0));
      xv[u] = rb >= 0 ? got : u32x2{0u, 0u};
    }
  };
  fetch(w * kTile);
  for (int u0 = w * kTile; u0 < total; u0 += kRowWaves * kTile) {
#pragma unroll
    for (int u = 0; u < KP; ++u) {
      const int i = lane + kWave * u;
      const int r = i / (D / 4), v = i % (D / 4);
      *reinterpret_cast<u32x2*>(k_lds + r * KROW + 4 * v) = xk[u];
    }
#pragma unroll
    for (int u = 0; u < VP; ++u) {
      const int i = lane + kWave * u;
      const int r = i / (VD / 4), v = i % (VD / 4);
      *reinterpret_cast<u32x2*>(v_lds + r * VROW + 4 * v) = xv[u];
    }
    if (u0 + kRowWaves * kTile < total) fetch(u0 + kRowWaves * kTile);
    wave_sync();
    f32x16 st;
#pragma unroll
    for (int i = 0; i < 16; ++i) st[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < D / 8; ++ks) {
      const u32x2 a = *reinterpret_cast<const u32x2*>(k_lds + c * KROW + 8 * ks + 4 * hf);
      st = M::run(a, qf[ks], st);
    }
    float mt = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int u = u0 + (i & 3) + 8 * (i >> 2) + 4 * hf;
      float v = st[i] * scale;
      if (softcap > 0.f) v = cap_score_fast(v, softcap, cap_arg);
      st[i] = (live && u < total) ? v : -INFINITY;
      mt = fmaxf(mt, st[i]);
    }
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    const float m_new = fmaxf(m, mt);
    const float corr = m_new == -INFINITY ? 1.f : expf(m - m_new);
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      st[i] = m_new == -INFINITY ? 0.f : expf(st[i] - m_new);
      psum += st[i];
    }
    l = l * corr + psum;
    m = m_new;
#pragma unroll
    for (int n = 0; n < VB; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[n][i] *= corr;
#pragma unroll
    for (int s8 = 0; s8 < 4; ++s8) {
      uint32_t hb[4], lb[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float pv = st[4 * s8 + e];
        hb[e] = bits16<S>(pv);
        lb[e] = bits16<S>(pv - from_bits16<S>(hb[e]));
      }
      const u32x2 hi = {hb[0] | (hb[1] << 16), hb[2] | (hb[3] << 16)};
      const u32x2 lo2 = {lb[0] | (lb[1] << 16), lb[2] | (lb[3] << 16)};
#pragma unroll
      for (int n = 0; n < VB; ++n) {
        // V^T operand from the row-major tile: value dim 32 n + c of keys 8 s8 + 4 hf .. + 3
        const uint16_t* col = reinterpret_cast<const uint16_t*>(v_lds) + (8 * s8 + 4 * hf) * VROW + 32 * n + c;
        const u32x2 a = {(uint32_t)col[0] | ((uint32_t)col[VROW] << 16),
                         (uint32_t)col[2 * VROW] | ((uint32_t)col[3 * VROW] << 16)};
        o[n] = M::run(a, hi, o[n]);
        o[n] = M::run(a, lo2, o[n]);
      }
    }
    wave_sync();
  }
  l += __shfl_xor(l, 32, 64);
  // merge the waves through LDS (the tiles are done with): [wave][head][2 + VD]
  __syncthreads();
  float* merge = reinterpret_cast<float*>(smem);
  if (live) {
    float* mine = merge + ((size_t)w * merge_heads + c) * (2 + VD);
    if (hf == 0) {
      mine[0] = m;
      mine[1] = l;
    }
#pragma unroll
    for (int n = 0; n < VB; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) mine[2 + out_dim(n, i, hf)] = o[n][i];
  }
  __syncthreads();
  auto merged = [&](int hh, int d) {
    float mm = -INFINITY;
    for (int ww = 0; ww < kRowWaves; ++ww) mm = fmaxf(mm, merge[((size_t)ww * merge_heads + hh) * (2 + VD)]);
    float ll = 0.f, ov = 0.f;
    for (int ww = 0; ww < kRowWaves; ++ww) {
      const float* src = merge + ((size_t)ww * merge_heads + hh) * (2 + VD);
      const float f = src[0] == -INFINITY ? 0.f : expf(src[0] - mm);
      ll += src[1] * f;
      ov += src[2 + d] * f;
    }
    return ov / ll;
  };
  for (int i = tid; i < nh * VD; i += 64 * kRowWaves) {
    const int hh = i / VD, d = i - hh * VD;
    float val = merged(hh, d);
    if (out_inv_freq != nullptr) {
      const bool is_a = interleaved ? (d & 1) == 0 : d < VD / 2;
      const int other = interleaved ? (d ^ 1) : (is_a ? d + VD / 2 : d - VD / 2);
      const int f = interleaved ? d >> 1 : (is_a ? d : d - VD / 2);
      float s, c2;
      sincosf((float)p * out_inv_freq[f], &s, &c2);
      const float ov = merged(hh, other);
      val = is_a ? val * c2 + ov * s : val * c2 - ov * s;
    }
    if (gate != nullptr) val *= 1.f / (1.f + expf(-S::to_f32(gate[(int64_t)t * gate_stride + h0 + hh])));
    out[(int64_t)t * out_stride + (int64_t)(h0 + hh) * v_row + v_first + d] = S::from_f32(val);
  }
}

// kv_decode_kernel<S, DB, VB>: single rows again, for heads of 64 or 128 and values of 64 or 128 with at
// most 16 query heads to a KV head, on 16x16x32 MFMAs (16 columns: the group's query heads; the 32x32
// ones above leave 28 of 32 columns idle at a group of 4).  Bound by HBM: every key and value is read once.
//   S^T = K q^T    A = K    lane (g, c) = (lane >> 4, lane & 15): key c, dims 32 ks + 8 g .. + 7
//                  B = q^T  lane: head c, the same dims (registers)
//                  C        lane: head c, keys 4 g .. 4 g + 3
//   O^T = V^T P^T  B = P^T  lane: head c, keys 4 g .. + 3 of both halves of the tile, where they lie
//                  A = V^T  lane: value dim 16 n + c of the same keys (two transposing reads)
// A weight enters as the sum of two 16-bit numbers, as in the kernel above.  The four waves take tiles of 32
// keys in turn, each through its own two LDS buffers: while one tile is worked on the next is on its way, and the one
// behind that is asked for, keys and values each, as soon as their place is free.  64 KB on their way per CU
// without a staging register, and no barrier in the loop.  A DMA instruction writes 64 lanes x 16
// bytes in a row, so rows are not padded: 16-byte pieces of a key row and 32-byte units of a value row
// are exchanged by the row's number, on the source's side, for reads without bank conflicts.  The block
// table's part waits in LDS, because a table load inside the loop would have to wait for the DMA ahead of
// it.  Few rows over long contexts: the keys of a row are shared out to `splits` workgroups, whose sums
// kv_decode_merge_kernel joins.
// 64 rows of 4096 keys, 16 / 4 heads of 128 (537 MB): 95 us = 5.6 TB/s (the kernel above 122; without the
// nontemporal hint 108; a tile asked for only when the one before it is done with, also without the hint, 106).
constexpr int kDecodeWaves = 4;
constexpr int kDecodeHeads = 16;
constexpr int kDecodeKeys = 32;
constexpr int kDecodeMinSplitKeys = 256;      // keys of a split, at least

template <class S>
struct Mma16x16;
template <>
struct Mma16x16<BF16> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <>
struct Mma16x16<F16> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

struct KvDecode {
  void* out;
  int64_t out_stride;
  const void* q;
  int64_t q_stride;
  const void* gate;
  int64_t gate_stride;
  const void* key_cache;
  const void* value_cache;
  const int* block_tables;
  int max_blocks;
  const int* token_seq;
  const int64_t* positions;
  const float* out_inv_freq;
  const float* sinks;
  float* parts;                 // [splits][T][heads][2 + VD]
  int interleaved, num_tokens, heads, kv_heads, block_size, num_blocks, window, keep_first, chunk, v_row, v_first;
  int splits, table_slots;
  float scale, softcap;
};

// a head's output dim d (ov: its pair's other dim) turned back, gated and stored
template <class S>
__device__ __forceinline__ void finish_decode(const KvDecode& a, int64_t t, int h, int d, int vd, float val, float ov) {
  if (a.out_inv_freq != nullptr) {
    const bool is_a = a.interleaved ? (d & 1) == 0 : d < vd / 2;
    const int f = a.interleaved ? d >> 1 : (is_a ? d : d - vd / 2);
    float s, c;
    sincosf((float)a.positions[t] * a.out_inv_freq[f], &s, &c);
    val = is_a ? val * c + ov * s : val * c - ov * s;
  }
  using T = typename S::T;
  if (a.gate != nullptr) val *= 1.f / (1.f + expf(-S::to_f32(((const T*)a.gate)[t * a.gate_stride + h])));
  ((T*)a.out)[t * a.out_stride + (int64_t)h * a.v_row + a.v_first + d] = S::from_f32(val);
}
__device__ __forceinline__ int pair_of(const KvDecode& a, int d, int vd) {
  return a.interleaved ? (d ^ 1) : (d < vd / 2 ? d + vd / 2 : d - vd / 2);
}

// 16 bytes per lane from each lane's own address into 1 KB of LDS (no register result); NT: read once, not kept
template <bool NT>
__device__ __forceinline__ void kv_dma16(const void* src, uint32_t lds_at) {
  unsigned keep;
  if constexpr (NT)
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt\n\ts_mov_b32 m0, %0"
        : "=&s"(keep)
        : "v"(src), "s"(lds_at)
        : "memory");
  else
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
        : "=&s"(keep)
        : "v"(src), "s"(lds_at)
        : "memory");
}
// all DMA but the N youngest instructions has landed
template <int N>
__device__ __forceinline__ void kv_dma_landed() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <class S, int DB, int VB, bool NT>
__global__ __launch_bounds__(64 * kDecodeWaves) void kv_decode_kernel(KvDecode a) {
  using T = typename S::T;
  using M = Mma16x16<S>;
  constexpr int D = 32 * DB, VD = 32 * VB;
  constexpr int KB = 2 * D, VBYTES = 2 * VD;               // bytes of a row of one KV head
  constexpr int KTILE = kDecodeKeys * KB, STAGE = KTILE + kDecodeKeys * VBYTES;
  constexpr int KI = KTILE / 1024, VI = STAGE / 1024 - KI; // DMA instructions of a tile
  constexpr int KP = KB / 16, VP = VBYTES / 16;            // pieces of a row
  static_assert((DB == 2 || DB == 4) && (VB == 2 || VB == 4), "rows of 128 or 256 bytes");
  extern __shared__ __align__(16) unsigned char smem[];
  int* table_lds = reinterpret_cast<int*>(smem + kDecodeWaves * 2 * STAGE);
  const int t = blockIdx.x, g_kv = blockIdx.y, split = blockIdx.z;
  const int group = a.heads / a.kv_heads, h0 = g_kv * group;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int p = (int)a.positions[t];
  const int* table = a.block_tables + (int64_t)a.token_seq[t] * a.max_blocks;
  const int lo = first_key(p, a.window, a.chunk);
  const int nk = min(a.keep_first, lo);                    // kept keys ahead of the window
  const int total = nk + p - lo + 1;
  const int share = ((total + a.splits - 1) / a.splits + kDecodeKeys - 1) / kDecodeKeys * kDecodeKeys;
  const int u_begin = split * share, u_end = min(total, u_begin + share);
  auto key_of = [&](int u) { return u < nk ? u : u - nk + lo; };
  const bool live = c < group;

  u32x4 qf[DB];
#pragma unroll
  for (int ks = 0; ks < DB; ++ks) {
    qf[ks] = u32x4{0u, 0u, 0u, 0u};
    if (live) qf[ks] = *reinterpret_cast<const u32x4*>((const T*)a.q + (int64_t)t * a.q_stride + (int64_t)(h0 + c) * D + 32 * ks + 8 * g);
  }
  // the blocks of the kept keys, then those of the rest of this share; an id outside the pool (a table the
  // host filled wrongly) reads block 0
  const int kept_blocks = u_begin < nk ? (nk + a.block_size - 1) / a.block_size : 0;
  const int first_block = key_of(max(u_begin, nk)) / a.block_size;
  if (u_begin < u_end) {
    const int last_block = key_of(u_end - 1) / a.block_size;
    const int n = min(a.table_slots, kept_blocks + max(0, last_block - first_block + 1));
    for (int i = tid; i < n; i += 64 * kDecodeWaves) {
      const int blk = table[i < kept_blocks ? i : i - kept_blocks + first_block];
      table_lds[i] = (unsigned)blk < (unsigned)a.num_blocks ? blk : 0;
    }
  }
  __syncthreads();

  f32x4 o[2 * VB];
#pragma unroll
  for (int n = 0; n < 2 * VB; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr float kLog2e = 1.4426950408889634f;
  const float scale2 = a.scale * kLog2e;                   // scores in base 2
  const float cap2 = a.softcap * kLog2e, cap_arg = a.softcap > 0.f ? 2.f * kLog2e / a.softcap : 0.f;
  float m = -INFINITY, l = 0.f;
  if (a.sinks != nullptr && live && w == 0 && split == 0) {     // the denominator's first term, counted once
    m = a.sinks[h0 + c] * kLog2e;
    l = g == 0 ? 1.f : 0.f;
  }
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)smem + w * 2 * STAGE;
  const unsigned char* mine = smem + w * 2 * STAGE;
  const uint32_t key_step = (uint32_t)a.kv_heads * KB, value_step = (uint32_t)a.kv_heads * a.v_row * 2;
  const unsigned char* keys = (const unsigned char*)a.key_cache + (size_t)g_kv * KB;
  const unsigned char* values = (const unsigned char*)a.value_cache + ((size_t)g_kv * a.v_row + a.v_first) * 2;
  // where a tile's keys lie (lane & 31: the key); behind the end: the last key again
  auto places = [&](int u0) {
    const int j = key_of(min(u0 + (lane & 31), u_end - 1));
    const int blk = j / a.block_size;
    const int at = j < lo ? blk : blk - first_block + kept_blocks;
    return table_lds[min(at, a.table_slots - 1)] * a.block_size + (j - blk * a.block_size);
  };
  // a tile's DMA: a lane's rows and pieces (a piece's place within the row is exchanged by the row's number)
  auto bring_keys = [&](int slot, int buf) {
#pragma unroll
    for (int u = 0; u < KI; ++u) {
      const int r = u * (64 / KP) + lane / KP, s = lane % KP;
      const int piece = s ^ (KP == 16 ? r & 15 : (r >> 1) & 7);
      const uint32_t row = (uint32_t)__shfl(slot, r, 64);
      kv_dma16<NT>(keys + (uint64_t)row * key_step + 16 * piece, lds0 + buf * STAGE + 1024 * u);
    }
  };
  auto bring_values = [&](int slot, int buf) {
#pragma unroll
    for (int u = 0; u < VI; ++u) {
      const int r = u * (64 / VP) + lane / VP, s = lane % VP;
      const int piece = (((s >> 1) ^ (VP == 16 ? r & 7 : (r >> 1) & 3)) << 1) | (s & 1);
      const uint32_t row = (uint32_t)__shfl(slot, r, 64);
      kv_dma16<NT>(values + (uint64_t)row * value_step + 16 * piece, lds0 + buf * STAGE + KTILE + 1024 * u);
    }
  };
  const int kx = KP == 16 ? c & 15 : (c >> 1) & 7;         // key rows c and 16 + c
  const int vrow = 4 * g + (c >> 2);                       // value rows vrow and 16 + vrow
  const int vx = VP == 16 ? vrow & 7 : (vrow >> 1) & 3;
  // Two tiles are under way: the keys of tile it + 2 are asked for as soon as those of tile `it` are used,
  // its values behind tile it's values.
  constexpr int STEP = kDecodeWaves * kDecodeKeys;
  int u0 = u_begin + w * kDecodeKeys;
  if (u0 < u_end) {
    const int slot = places(u0);
    bring_keys(slot, 0);
    bring_values(slot, 0);
  }
  if (u0 + STEP < u_end) {
    const int slot = places(u0 + STEP);
    bring_keys(slot, 1);
    bring_values(slot, 1);
  }
  for (int buf = 0; u0 < u_end; u0 += STEP, buf ^= 1) {
    const bool ahead = u0 + 2 * STEP < u_end;
    const int slot = ahead ? places(u0 + 2 * STEP) : 0;
    if (u0 + STEP < u_end)
      kv_dma_landed<KI + 2 * VI>();
    else
      kv_dma_landed<0>();
    const unsigned char* k_lds = mine + buf * STAGE;
    const unsigned char* v_lds = k_lds + KTILE;
    f32x4 st[2];
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      st[kh] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < DB; ++ks) {
        const u32x4 ka = *reinterpret_cast<const u32x4*>(k_lds + (16 * kh + c) * KB + 16 * ((4 * ks + g) ^ kx));
        st[kh] = M::run(ka, qf[ks], st[kh]);
      }
    }
    if (ahead) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the keys are read
      bring_keys(slot, buf);
    }
    float mt = -INFINITY;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = st[kh][e] * scale2;
        if (a.softcap > 0.f) v = cap_score_fast(st[kh][e] * a.scale, cap2, cap_arg);
        st[kh][e] = u0 + 16 * kh + 4 * g + e < u_end ? v : -INFINITY;
        mt = fmaxf(mt, st[kh][e]);
      }
    mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    const float m_new = fmaxf(m, mt);
    const float shift = m_new == -INFINITY ? 0.f : m_new;
    const float corr = __builtin_amdgcn_exp2f(m - shift);
    u32x4 hi, low;
    float psum = 0.f;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int e2 = 0; e2 < 2; ++e2) {
        uint32_t hb[2], lb[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float pv = __builtin_amdgcn_exp2f(st[kh][2 * e2 + e] - shift);
          psum += pv;
          hb[e] = bits16<S>(pv);
          lb[e] = bits16<S>(pv - from_bits16<S>(hb[e]));
        }
        hi[2 * kh + e2] = hb[0] | (hb[1] << 16);
        low[2 * kh + e2] = lb[0] | (lb[1] << 16);
      }
    l = l * corr + psum;
    if (__any(m_new != m)) {
#pragma unroll
      for (int n = 0; n < 2 * VB; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[n][e] *= corr;
    }
    m = m_new;
    if (ahead)
      kv_dma_landed<2 * KI + VI>();
    else
      kv_dma_landed<0>();
#pragma unroll
    for (int n = 0; n < 2 * VB; ++n) {
      const unsigned char* at = v_lds + vrow * VBYTES + 32 * (n ^ vx) + 8 * (c & 3);
      // 16 rows further on the exchange is the same
      const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)at);
      const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(at + 16 * VBYTES));
      const u32x2 x0 = __builtin_bit_cast(u32x2, v0), x1 = __builtin_bit_cast(u32x2, v1);
      const u32x4 va = {x0[0], x0[1], x1[0], x1[1]};
      o[n] = M::run(va, hi, o[n]);
      o[n] = M::run(va, low, o[n]);
    }
    if (ahead) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // and the values
      bring_values(slot, buf);
    }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  // merge the waves through LDS (the tiles are done with): [wave][head][2 + VD]
  __syncthreads();
  float* merge = reinterpret_cast<float*>(smem);
  if (live) {
    float* to = merge + (w * kDecodeHeads + c) * (2 + VD);
    if (g == 0) {
      to[0] = m;
      to[1] = l;
    }
#pragma unroll
    for (int n = 0; n < 2 * VB; ++n)
#pragma unroll
      for (int e = 0; e < 4; ++e) to[2 + 16 * n + 4 * g + e] = o[n][e];
  }
  __syncthreads();
  auto merged = [&](int hh, int d, float& mm, float& ll) {
    mm = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < kDecodeWaves; ++ww) mm = fmaxf(mm, merge[(ww * kDecodeHeads + hh) * (2 + VD)]);
    float ov = 0.f;
    ll = 0.f;
#pragma unroll
    for (int ww = 0; ww < kDecodeWaves; ++ww) {
      const float* src = merge + (ww * kDecodeHeads + hh) * (2 + VD);
      const float f = src[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(src[0] - mm);
      ll += src[1] * f;
      ov += src[2 + d] * f;
    }
    return ov;
  };
  for (int i = tid; i < group * VD; i += 64 * kDecodeWaves) {
    const int hh = i / VD, d = i - hh * VD;
    float mm, ll;
    const float ov = merged(hh, d, mm, ll);
    if (a.splits > 1) {
      float* to = a.parts + (((int64_t)split * a.num_tokens + t) * a.heads + h0 + hh) * (2 + VD);
      to[2 + d] = ov;
      if (d == 0) {
        to[0] = mm;
        to[1] = ll;
      }
    } else {
      const float other = a.out_inv_freq != nullptr ? merged(hh, pair_of(a, d, VD), mm, ll) / ll : 0.f;
      finish_decode<S>(a, t, h0 + hh, d, VD, ov / ll, other);
    }
  }
}

template <class S, int VB>
__global__ __launch_bounds__(32 * VB) void kv_decode_merge_kernel(KvDecode a) {
  constexpr int VD = 32 * VB;
  const int64_t t = blockIdx.x;
  const int h = blockIdx.y, d = threadIdx.x;
  const int64_t step = (int64_t)a.num_tokens * a.heads * (2 + VD);
  const float* src = a.parts + (t * a.heads + h) * (2 + VD);
  float mm = -INFINITY;
  for (int s = 0; s < a.splits; ++s) mm = fmaxf(mm, src[s * step]);
  float ll = 0.f, val = 0.f, ov = 0.f;
  const int other = pair_of(a, d, VD);
#pragma unroll 4
  for (int s = 0; s < a.splits; ++s) {
    const float f = src[s * step] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(src[s * step] - mm);
    ll += src[s * step + 1] * f;
    val += src[s * step + 2 + d] * f;
    if (a.out_inv_freq != nullptr) ov += src[s * step + 2 + other] * f;
  }
  finish_decode<S>(a, t, h, d, VD, val / ll, ov / ll);
}

// Workgroups that a row's keys are shared out to: as many as bring the launch to one per CU, none with fewer
// than kDecodeMinSplitKeys keys.  max_keys 0 (unknown): one.  The merge is a launch and a scratch allocation more,
// about 4 us per call, which up to 2048 keys are not worth (16 / 4 heads of 128, us per call, shared / one
// workgroup: 2 rows of 512 keys 45 / 40, of 2048 44 / 40, of 4096 45 / 65; 8 rows of 2048 42 / 42, of 4096
// 43 / 68; 32 rows of 1024 43 / 38, of 4096 59 / 70).
int decode_splits(int num_tokens, int kv_heads, int max_keys) {
  const int64_t groups = (int64_t)num_tokens * kv_heads;
  if (groups >= 256 || max_keys <= VLA_KV_WHOLE_KEYS) return 1;
  return (int)std::max<int64_t>(1, std::min<int64_t>((256 + groups - 1) / groups, max_keys / kDecodeMinSplitKeys));
}

bool decode_sizes(int dim, int vdim, int heads, int kv_heads) {
  return (dim == 64 || dim == 128) && (vdim == 64 || vdim == 128) && heads / kv_heads <= kDecodeHeads;
}

template <class S, int DB, int VB, bool NT>
int launch_decode_one(const KvDecode& a, hipStream_t stream) {
  const size_t tiles = (size_t)kDecodeWaves * 2 * kDecodeKeys * 64 * (DB + VB);
  const size_t merge = (size_t)kDecodeWaves * kDecodeHeads * (2 + 32 * VB) * sizeof(float);
  const size_t lds = std::max(tiles + a.table_slots * sizeof(int), merge);
  static std::atomic<size_t> allowed{64 * 1024};   // raised once per kernel, not per launch
  if (lds > allowed.load(std::memory_order_relaxed)) {
    VLA_SEQ_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&kv_decode_kernel<S, DB, VB, NT>),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    allowed.store(160 * 1024, std::memory_order_relaxed);
  }
  kv_decode_kernel<S, DB, VB, NT><<<dim3(a.num_tokens, a.kv_heads, a.splits), 64 * kDecodeWaves, lds, stream>>>(a);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  if (a.splits > 1) {
    kv_decode_merge_kernel<S, VB><<<dim3(a.num_tokens, a.heads), 32 * VB, 0, stream>>>(a);
    VLA_SEQ_HIP_CHECK(hipGetLastError());
  }
  return VLA_OK;
}

// keys and values of a launch that Infinity Cache (256 MiB) cannot hold are read past it
template <class S, int DB, int VB>
int launch_decode(const KvDecode& a, int max_keys, hipStream_t stream) {
  const int64_t bytes = (int64_t)a.num_tokens * max_keys * a.kv_heads * 64 * (DB + VB);
  return bytes > ((int64_t)256 << 20) ? launch_decode_one<S, DB, VB, true>(a, stream)
                                      : launch_decode_one<S, DB, VB, false>(a, stream);
}

template <class S, int DB, int VB>
int launch_heads_one(dim3 grid, hipStream_t stream, typename S::T* out, int64_t out_stride,
                     const typename S::T* q, int64_t q_stride, const typename S::T* gate,
                     int64_t gate_stride, const typename S::T* key_cache,
                     const typename S::T* value_cache, const int* block_tables, int max_blocks,
                     const int* token_seq, const int64_t* positions, const float* out_inv_freq,
                     int interleaved, int heads, int kv_heads, int block_size, int num_blocks,
                     int window, float scale, int keep_first, float softcap, int chunk,
                     const float* sinks, int v_row, int v_first) {
  constexpr int D = 32 * DB, VD = 32 * VB;
  const int group = heads / kv_heads;
  const int merge_heads = group < 32 ? group : 32;
  const size_t tiles = (size_t)kRowWaves * kTile * (D + 4 + VD + 4) * sizeof(typename S::T);
  const size_t merge = (size_t)kRowWaves * merge_heads * (2 + VD) * sizeof(float);
  const size_t lds = tiles > merge ? tiles : merge;
  if (lds > 160 * 1024) return VLA_ERR_HEAD_SIZE;
  static std::atomic<size_t> allowed{64 * 1024};   // raised once per kernel, not per launch
  if (lds > allowed.load(std::memory_order_relaxed)) {
    VLA_SEQ_HIP_CHECK(hipFuncSetAttribute(
        reinterpret_cast<const void*>(&kv_attention_heads_kernel<S, DB, VB>),
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    allowed.store(lds, std::memory_order_relaxed);
  }
  kv_attention_heads_kernel<S, DB, VB><<<grid, 64 * kRowWaves, lds, stream>>>(
      out, out_stride, q, q_stride, gate, gate_stride, key_cache, value_cache, block_tables,
      max_blocks, token_seq, positions, out_inv_freq, interleaved, heads, kv_heads, block_size,
      num_blocks, window, scale, merge_heads, keep_first, softcap, chunk, sinks, v_row, v_first);
  VLA_SEQ_HIP_CHECK(hipGetLastError());
  return VLA_OK;
}

struct TileGrid {
  int64_t tiles;        // at most this many tiles of rows, of all sequences
  int of_longest;       // and of one
  int num_seqs, head_waves, head_groups, key_groups;
  bool ranked;          // a tile is found by its rank, not by the grid
  bool in_order;        // the grid goes through the rows in order, not through the last tiles of all sequences first
};

// num_rows rows in all, walks of at most `keys` keys.
// Two groups of four waves, one workgroup a CU, share a workgroup's keys where there are few workgroups: of 16 heads on 4
// of 128, a run of 2047 rows (256 of them) takes 44 us instead of 52, one of 4096 (512) 103 instead of 114, 16 of 96 to
// 256 rows behind up to 3000 keys (436) 63 instead of 76; 700 fill the chip with independent ones (62 instead of 73).
// Between one and two workgroups a CU it needs walks of some length: 40 runs of up to 100 rows 22 us with two groups, 14 with
// one; behind 300 keys 27 and 21; a run of 256 rows beside 60 of 20 19 and 14.
// By their rank, so that none is empty and the longest walks go out first: not where no workgroup is empty and the walks are
// short: the search is a wait for memory more, 256 runs of 33 rows take 42 us with it and 39 without, 128 of 64 48
// and 39; (one sequence does without in any case).
// In the order of the rows where all runs are the same whole tiles of rows of 4 KB or more: tiles of the same number lie at the
// same distance from each other and meet in the same memory channels (128 runs of 64 rows 26 us, last tiles first 47; 64
// of 128 28 and 43).  Others keep that order: of 60 rows 28 and 27, 400 runs of 128 rows of 8 heads of 64 46 and 42.
TileGrid tile_grid(int num_seqs, int max_query_len, int64_t num_rows, int heads, int kv_heads, int dim, int64_t keys) {
  TileGrid to;
  const int group = heads / kv_heads;
  to.num_seqs = num_seqs;
  to.head_waves = group >= 3 ? 4 : group;      // waves of a workgroup that are heads
  const int tile_rows = kTile * (4 / to.head_waves);
  to.head_groups = kv_heads * ((group + to.head_waves - 1) / to.head_waves);
  to.of_longest = (max_query_len + tile_rows - 1) / tile_rows;
  const int64_t all = (int64_t)num_seqs * to.of_longest;
  to.tiles = std::min(all, num_rows / tile_rows + num_seqs);
  const int64_t workgroups = to.head_groups * to.tiles;
  to.key_groups = workgroups <= 256 || (workgroups <= 512 && keys > 512) ? 2 : 1;
  to.in_order = keys <= 128 && (int64_t)heads * dim >= 2048 && max_query_len % tile_rows == 0 &&
                num_rows == (int64_t)num_seqs * max_query_len;
  to.ranked = num_seqs <= kRankedSeqs && !to.in_order && !(to.tiles == all && keys <= 256);
  return to;
}

// the most keys that a workgroup's rows walk
int64_t walked_keys(int max_blocks, int block_size, int window, int keep_first, int chunk) {
  int64_t keys = (int64_t)max_blocks * block_size;
  if (window > 0) keys = std::min(keys, (int64_t)window + 4 * kTile + keep_first);
  if (chunk > 0) keys = std::min(keys, (int64_t)chunk + 4 * kTile + keep_first);
  return keys;
}

template <class S, int DB, int VB>
int launch_tiles_one(TileGrid to, hipStream_t stream, typename S::T* out, int64_t out_stride,
                     const typename S::T* q, int64_t q_stride, const typename S::T* gate,
                     int64_t gate_stride, const typename S::T* key_cache,
                     const typename S::T* value_cache, const int* block_tables, int max_blocks,
                     const int* qsl, const int* ctx, const float* out_inv_freq, int interleaved,
                     int heads, int kv_heads, int block_size, int num_blocks, int window,
                     float scale, int keep_first, float softcap, int chunk,
                     const float* sinks, int v_row, int v_first) {
  auto go = [&](dim3 grid, int b0, int last_tile, int ranked_seqs, int first_rank) -> int {
    auto* kernel = to.key_groups == 2 ? &kv_attention_tile_kernel<S, DB, VB, 2> : &kv_attention_tile_kernel<S, DB, VB, 1>;
    kernel<<<grid, 256 * to.key_groups, 0, stream>>>(
        out, out_stride, q, q_stride, gate, gate_stride, key_cache, value_cache, block_tables + (int64_t)b0 * max_blocks,
        max_blocks, qsl + b0, ctx + b0, out_inv_freq, interleaved, heads, kv_heads, to.head_groups, block_size, num_blocks,
        window, scale, to.head_waves, keep_first, softcap, chunk, sinks, v_row, v_first, last_tile, ranked_seqs, first_rank);
    VLA_SEQ_HIP_CHECK(hipGetLastError());
    return VLA_OK;
  };
  // a launch counts its threads in 32 bits: more than 16.7 million groups of heads go in several launches
  const int64_t most = std::max(1, 0xffffff / (to.head_groups * to.key_groups));
  if (to.ranked || to.in_order) {
    for (int64_t r = 0; r < to.tiles; r += most) {
      const int rc = go(dim3(to.head_groups * (unsigned)std::min(most, to.tiles - r)), 0, to.of_longest - 1,
                        to.ranked ? to.num_seqs : -1, (int)r);
      if (rc != VLA_OK) return rc;
    }
    return VLA_OK;
  }
  // grid: (sequences x groups of heads, row tiles); more tiles than a grid's second side takes go in several
  // launches, the last rows first
  constexpr int kSide = 65535;
  for (int64_t b0 = 0; b0 < to.num_seqs; b0 += most)
    for (int left = to.of_longest; left > 0; left -= kSide) {
      const dim3 grid(to.head_groups * (unsigned)std::min(most, to.num_seqs - b0), std::min(left, kSide));
      const int rc = go(grid, (int)b0, left - 1, 0, 0);
      if (rc != VLA_OK) return rc;
    }
  return VLA_OK;
}

// dim / 32 and vdim / 32 in 1 .. 4 -> the instantiation
#define VLA_KV_BY_SIZE(FN, S, db, vb, ...)                         \
  switch ((db) * 4 + (vb)-5) {                                     \
    case 0: return FN<S, 1, 1>(__VA_ARGS__);                       \
    case 1: return FN<S, 1, 2>(__VA_ARGS__);                       \
    case 2: return FN<S, 1, 3>(__VA_ARGS__);                       \
    case 3: return FN<S, 1, 4>(__VA_ARGS__);                       \
    case 4: return FN<S, 2, 1>(__VA_ARGS__);                       \
    case 5: return FN<S, 2, 2>(__VA_ARGS__);                       \
    case 6: return FN<S, 2, 3>(__VA_ARGS__);                       \
    case 7: return FN<S, 2, 4>(__VA_ARGS__);                       \
    case 8: return FN<S, 3, 1>(__VA_ARGS__);                       \
    case 9: return FN<S, 3, 2>(__VA_ARGS__);                       \
    case 10: return FN<S, 3, 3>(__VA_ARGS__);                      \
    case 11: return FN<S, 3, 4>(__VA_ARGS__);                      \
    case 12: return FN<S, 4, 1>(__VA_ARGS__);                      \
    case 13: return FN<S, 4, 2>(__VA_ARGS__);                      \
    case 14: return FN<S, 4, 3>(__VA_ARGS__);                      \
    case 15: return FN<S, 4, 4>(__VA_ARGS__);                      \
    default: return VLA_ERR_HEAD_SIZE;                             \
  }

template <class S, class... A>
int launch_heads(int db, int vb, A... a) {
  VLA_KV_BY_SIZE(launch_heads_one, S, db, vb, a...)
}
template <class S, class... A>
int launch_tiles(int db, int vb, A... a) {
  VLA_KV_BY_SIZE(launch_tiles_one, S, db, vb, a...)
}

// Values of more than 128 dims go in slices: each a launch that forms the same weights again and sums
// its columns (values that turn back pair columns across slices and do not).
constexpr int kSliceBlocks = 4;
bool mfma_sizes(int dim, int vdim, bool turned) {
  return dim % 32 == 0 && dim >= 32 && dim <= 128 && vdim % 32 == 0 && vdim >= 32 &&
         vdim <= (turned ? 32 * kSliceBlocks : kMaxDim);
}
// f(vdim / 32 of the slice, first column) for slices of about equal size
template <class F>
int by_value_slices(int vdim, F&& f) {
  const int blocks = vdim / 32, slices = (blocks + kSliceBlocks - 1) / kSliceBlocks;
  for (int s = 0; s < slices; ++s) {
    const int first = blocks * s / slices, end = blocks * (s + 1) / slices;
    const int rc = f(end - first, 32 * first);
    if (rc != VLA_OK) return rc;
  }
  return VLA_OK;
}

}  // namespace
}  // namespace seq
}  // namespace vla

using namespace vla;
using namespace vla::seq;

extern "C" int vla_seq_rotary_kv_write_form(const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                                            int64_t v_stride, const void* key_cache, const void* value_cache, int heads,
                                            int kv_heads, int dim, int vdim, int rot_dims, int dtype) {
  if (dtype != VLA_BF16 && dtype != VLA_F16) return 0;
  return rows_fit(RotaryRows{(void*)q, q_stride, k, k_stride, v, v_stride, (void*)key_cache, (void*)value_cache, nullptr, nullptr,
                             nullptr, 0, 0, heads, kv_heads, dim, vdim, rot_dims, 0});
}

extern "C" int vla_seq_rotary_kv_write(void* q, int64_t q_stride, const void* k, int64_t k_stride,
                                       const void* v, int64_t v_stride, void* key_cache,
                                       void* value_cache, const int64_t* positions,
                                       const int64_t* slot_mapping, const float* inv_freq,
                                       const float* value_inv_freq, int num_tokens, int heads,
                                       int kv_heads, int dim, int vdim, int rot_dims,
                                       int interleaved, int block_size, int num_blocks, int dtype,
                                       const float* q_norm, const float* k_norm, float norm_eps,
                                       const void* v_other, int64_t v_other_stride,
                                       const float* v_blend, int head_norm, void* stream) {
  if (num_tokens == 0) return VLA_OK;
  if (!q || !k || !v || !key_cache || !value_cache || !positions || !slot_mapping || num_tokens < 0 ||
      heads <= 0 || kv_heads <= 0 || dim <= 0 || vdim <= 0 || rot_dims < 0 || rot_dims > dim ||
      (rot_dims & 1) || (rot_dims > 0 && !inv_freq) || block_size <= 0 || num_blocks <= 0 ||
      q_stride < (int64_t)heads * dim || k_stride < (int64_t)kv_heads * dim ||
      v_stride < (int64_t)kv_heads * vdim ||
      (v_other && (!v_blend || value_inv_freq || v_other_stride < (int64_t)kv_heads * vdim)))
    return VLA_ERR_ARG;
  return with_dtype(dtype, [&](auto s) {
    using S = decltype(s);
    using T = typename S::T;
    if constexpr (sizeof(T) == 2) {
      const RotaryRows a{q, q_stride, k, k_stride, v, v_stride, key_cache, value_cache, positions, slot_mapping, inv_freq,
                         (int64_t)num_blocks * block_size, num_tokens, heads, kv_heads, dim, vdim, rot_dims, interleaved};
      if (!head_norm && !q_norm && !k_norm && !v_other && !value_inv_freq && rows_fit(a)) {
        // few tokens: a workgroup each, so that each has a CU
        const int waves = num_tokens < 1024 ? 1 : kTurnWaves;
        rotary_kv_rows_kernel<S><<<(unsigned)(((int64_t)num_tokens + waves - 1) / waves), 64 * waves, 0, (hipStream_t)stream>>>(a);
        VLA_SEQ_HIP_CHECK(hipGetLastError());
        return (int)VLA_OK;
      }
    }
    const size_t lds = head_norm ? sizeof(float) * ((size_t)heads + kv_heads) : 0;
    rotary_kv_write_kernel<S><<<num_tokens, 256, lds, (hipStream_t)stream>>>(
        (T*)q, q_stride, (const T*)k, k_stride, (const T*)v, v_stride, (T*)key_cache,
        (T*)value_cache, positions, slot_mapping, inv_freq, value_inv_freq, heads, kv_heads, dim,
        vdim, rot_dims, interleaved, (int64_t)num_blocks * block_size, q_norm, k_norm, norm_eps,
        (const T*)v_other, v_other_stride, v_blend, head_norm);
    VLA_SEQ_HIP_CHECK(hipGetLastError());
    return (int)VLA_OK;
  });
}

namespace {

// scratch null: one workgroup per row and KV head, whatever max_keys says
int kv_attention(void* out, int64_t out_stride, const void* q, int64_t q_stride,
                                    const void* gate, int64_t gate_stride, const void* key_cache,
                                    const void* value_cache, const int* block_tables,
                                    int max_blocks, const int* token_seq, const int64_t* positions,
                                    const float* out_inv_freq, int interleaved, int num_tokens,
                                    int heads, int kv_heads, int dim, int vdim, int block_size,
                                    int num_blocks, int window, float scale, int dtype,
                                    int keep_first, float softcap, int chunk, const float* sinks,
                                    int max_keys, float* scratch, int64_t scratch_floats, void* stream) {
  if (num_tokens == 0) return VLA_OK;
  if (!out || !q || !key_cache || !value_cache || !block_tables || !token_seq || !positions ||
      num_tokens < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || block_size <= 0 ||
      num_blocks <= 0 || max_blocks <= 0 || out_stride < (int64_t)heads * vdim ||
      q_stride < (int64_t)heads * dim || (gate && gate_stride < heads) || keep_first < 0 ||
      !(softcap >= 0.f))
    return VLA_ERR_ARG;
  if (window <= 0 && chunk <= 0) keep_first = 0;
  if (dim <= 0 || dim > kMaxDim || vdim <= 0 || vdim > kMaxDim) return VLA_ERR_HEAD_SIZE;
  return with_dtype(dtype, [&](auto s) {
    using S = decltype(s);
    using T = typename S::T;
    if constexpr (sizeof(T) == 2) {
      // 16-bit rows on the matrix cores when the head sizes and the alignment allow
      if (g_kv_kernel.load(std::memory_order_relaxed) == 0 && mfma_sizes(dim, vdim, out_inv_freq != nullptr) &&
          ((uintptr_t)q % 8) == 0 && ((q_stride * 2) % 8) == 0 && ((uintptr_t)key_cache % 8) == 0 &&
          ((uintptr_t)value_cache % 8) == 0) {
        const int splits = scratch ? decode_splits(num_tokens, kv_heads, max_keys) : 1;
        // blocks of a share, and of the kept keys, that the kernel has to keep in LDS: 160 KB less its tiles
        const int64_t slots = (max_blocks + splits - 1) / splits + kDecodeKeys / block_size + 3 + keep_first / block_size + 1;
        const size_t tiles = (size_t)kDecodeWaves * 2 * kDecodeKeys * 2 * (dim + vdim);
        if (decode_sizes(dim, vdim, heads, kv_heads) && tiles + slots * 4 <= 160 * 1024 &&
            (uint64_t)num_blocks * block_size < ((uint64_t)1 << 31) && (uint64_t)kv_heads * std::max(dim, vdim) * 2 < ((uint64_t)1 << 32) &&
            num_tokens <= 0x7fffffff && kv_heads <= 65535 && heads <= 65535 && (uintptr_t)q % 16 == 0 && q_stride % 8 == 0 &&
            (uintptr_t)key_cache % 16 == 0 && (uintptr_t)value_cache % 16 == 0) {
          if (splits > 1 && scratch_floats < (int64_t)splits * num_tokens * heads * (2 + vdim)) return (int)VLA_ERR_ARG;
          KvDecode a;
          a.out = out;
          a.out_stride = out_stride;
          a.q = q;
          a.q_stride = q_stride;
          a.gate = gate;
          a.gate_stride = gate_stride;
          a.key_cache = key_cache;
          a.value_cache = value_cache;
          a.block_tables = block_tables;
          a.max_blocks = max_blocks;
          a.token_seq = token_seq;
          a.positions = positions;
          a.out_inv_freq = out_inv_freq;
          a.sinks = sinks;
          a.parts = scratch;
          a.interleaved = interleaved;
          a.num_tokens = num_tokens;
          a.heads = heads;
          a.kv_heads = kv_heads;
          a.block_size = block_size;
          a.num_blocks = num_blocks;
          a.window = window;
          a.keep_first = keep_first;
          a.chunk = chunk;
          a.v_row = vdim;
          a.v_first = 0;
          a.splits = splits;
          a.table_slots = (int)slots;
          a.scale = scale;
          a.softcap = softcap;
          if (dim == 128)
            return vdim == 128 ? launch_decode<S, 4, 4>(a, max_keys, (hipStream_t)stream) : launch_decode<S, 4, 2>(a, max_keys, (hipStream_t)stream);
          return vdim == 128 ? launch_decode<S, 2, 4>(a, max_keys, (hipStream_t)stream) : launch_decode<S, 2, 2>(a, max_keys, (hipStream_t)stream);
        }
        const int group = heads / kv_heads;
        const dim3 grid(num_tokens, kv_heads * ((group + 31) / 32));
        const int rc = by_value_slices(vdim, [&](int vb, int v_first) {
          return launch_heads<S>(dim / 32, vb, grid, (hipStream_t)stream, (T*)out, out_stride, (const T*)q,
                                 q_stride, (const T*)gate, gate_stride, (const T*)key_cache,
                                 (const T*)value_cache, block_tables, max_blocks, token_seq, positions,
                                 out_inv_freq, interleaved, heads, kv_heads, block_size, num_blocks,
                                 window, scale, keep_first, softcap, chunk, sinks, vdim, v_first);
        });
        if (rc != VLA_ERR_HEAD_SIZE) return rc;
      }
    }
    const dim3 grid(num_tokens, (heads + kHeadsPerGroup - 1) / kHeadsPerGroup);
    auto plain = [&](auto kernel) {
      kernel<<<grid, kWave * kHeadsPerGroup, 0, (hipStream_t)stream>>>(
          (T*)out, out_stride, (const T*)q, q_stride, (const T*)gate, gate_stride, (const T*)key_cache,
          (const T*)value_cache, block_tables, max_blocks, token_seq, positions, out_inv_freq,
          interleaved, heads, kv_heads, dim, vdim, block_size, num_blocks, window, scale, keep_first,
          softcap, chunk, sinks);
    };
    if (dim <= 256 && vdim <= 256)
      plain(kv_attention_kernel<S, 4>);
    else
      plain(kv_attention_kernel<S, kMaxDim / kWave>);
    VLA_SEQ_HIP_CHECK(hipGetLastError());
    return VLA_OK;
  });
}

}  // namespace

extern "C" int vla_seq_kv_attention(void* out, int64_t out_stride, const void* q, int64_t q_stride,
                                    const void* gate, int64_t gate_stride, const void* key_cache,
                                    const void* value_cache, const int* block_tables,
                                    int max_blocks, const int* token_seq, const int64_t* positions,
                                    const float* out_inv_freq, int interleaved, int num_tokens,
                                    int heads, int kv_heads, int dim, int vdim, int block_size,
                                    int num_blocks, int window, float scale, int dtype,
                                    int keep_first, float softcap, int chunk, const float* sinks,
                                    void* stream) {
  return kv_attention(out, out_stride, q, q_stride, gate, gate_stride, key_cache, value_cache, block_tables, max_blocks, token_seq,
                      positions, out_inv_freq, interleaved, num_tokens, heads, kv_heads, dim, vdim, block_size, num_blocks, window,
                      scale, dtype, keep_first, softcap, chunk, sinks, 0, nullptr, 0, stream);
}

extern "C" int64_t vla_seq_kv_attention_scratch_floats(int num_tokens, int heads, int kv_heads, int dim, int vdim,
                                                       int max_keys, int dtype) {
  if ((dtype != VLA_F16 && dtype != VLA_BF16) || heads <= 0 || kv_heads <= 0 || heads % kv_heads ||
      !decode_sizes(dim, vdim, heads, kv_heads))
    return 0;
  const int splits = decode_splits(num_tokens, kv_heads, max_keys);
  return splits > 1 ? (int64_t)splits * num_tokens * heads * (2 + vdim) : 0;
}

extern "C" int vla_seq_kv_attention_shared(void* out, int64_t out_stride, const void* q, int64_t q_stride,
                                    const void* gate, int64_t gate_stride, const void* key_cache,
                                    const void* value_cache, const int* block_tables,
                                    int max_blocks, const int* token_seq, const int64_t* positions,
                                    const float* out_inv_freq, int interleaved, int num_tokens,
                                    int heads, int kv_heads, int dim, int vdim, int block_size,
                                    int num_blocks, int window, float scale, int dtype,
                                    int keep_first, float softcap, int chunk, const float* sinks,
                                    int max_keys, float* scratch, int64_t scratch_floats, void* stream) {
  return kv_attention(out, out_stride, q, q_stride, gate, gate_stride, key_cache, value_cache, block_tables, max_blocks, token_seq,
                      positions, out_inv_freq, interleaved, num_tokens, heads, kv_heads, dim, vdim, block_size, num_blocks, window,
                      scale, dtype, keep_first, softcap, chunk, sinks, max_keys, scratch, scratch_floats, stream);
}

// 0: pick per shape; 1: always the one-wave-per-(row, head) kernel (tests run both)
extern "C" int vla_seq_set_kv_attention_kernel(int mode) {
  if (mode < 0 || mode > 1) return VLA_ERR_ARG;
  g_kv_kernel.store(mode, std::memory_order_relaxed);
  return VLA_OK;
}

extern "C" int vla_seq_kv_attention_tiles_supported(int dim, int vdim, int turned, int dtype) {
  return (dtype == VLA_F16 || dtype == VLA_BF16) && mfma_sizes(dim, vdim, turned != 0) &&
         g_kv_kernel.load(std::memory_order_relaxed) == 0;
}

extern "C" int vla_seq_kv_attention_tiles_form(int num_seqs, int max_query_len, int64_t num_rows, int heads, int kv_heads, int dim,
                                               int max_blocks, int block_size, int window, int keep_first, int chunk) {
  if (num_seqs <= 0 || max_query_len <= 0 || num_rows < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 ||
      dim <= 0 || max_blocks <= 0 || block_size <= 0)
    return 0;
  const TileGrid to = tile_grid(num_seqs, max_query_len, num_rows, heads, kv_heads, dim,
                                walked_keys(max_blocks, block_size, window, window > 0 || chunk > 0 ? keep_first : 0, chunk));
  return to.key_groups + (to.ranked ? 4 : 0) + (to.in_order ? 8 : 0);
}

extern "C" int vla_seq_kv_attention_tiles(
    void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* gate,
    int64_t gate_stride, const void* key_cache, const void* value_cache, const int* block_tables,
    int max_blocks, const int* query_start_loc, const int* context_lens, const float* out_inv_freq,
    int interleaved, int num_seqs, int max_query_len, int heads, int kv_heads, int dim, int vdim,
    int block_size, int num_blocks, int window, float scale, int dtype, int keep_first,
    float softcap, int chunk, const float* sinks, void* stream) {
  return vla_seq_kv_attention_tiles_of(out, out_stride, q, q_stride, gate, gate_stride, key_cache, value_cache, block_tables,
                                       max_blocks, query_start_loc, context_lens, out_inv_freq, interleaved, num_seqs,
                                       max_query_len, (int64_t)num_seqs * max_query_len, heads, kv_heads, dim, vdim, block_size,
                                       num_blocks, window, scale, dtype, keep_first, softcap, chunk, sinks, stream);
}

extern "C" int vla_seq_kv_attention_tiles_of(
    void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* gate,
    int64_t gate_stride, const void* key_cache, const void* value_cache, const int* block_tables,
    int max_blocks, const int* query_start_loc, const int* context_lens, const float* out_inv_freq,
    int interleaved, int num_seqs, int max_query_len, int64_t num_rows, int heads, int kv_heads, int dim, int vdim,
    int block_size, int num_blocks, int window, float scale, int dtype, int keep_first,
    float softcap, int chunk, const float* sinks, void* stream) {
  if (num_seqs == 0 || max_query_len == 0) return VLA_OK;
  if (keep_first < 0 || !(softcap >= 0.f)) return VLA_ERR_ARG;
  if (window <= 0 && chunk <= 0) keep_first = 0;
  if (!out || !q || !key_cache || !value_cache || !block_tables || !query_start_loc || !context_lens ||
      num_seqs < 0 || num_seqs > 65535 || max_query_len < 0 || num_rows < 0 || heads <= 0 || kv_heads <= 0 ||
      heads % kv_heads != 0 || block_size <= 0 || num_blocks <= 0 || max_blocks <= 0 ||
      out_stride < (int64_t)heads * vdim || q_stride < (int64_t)heads * dim ||
      (gate && gate_stride < heads))
    return VLA_ERR_ARG;
  if ((dtype != VLA_F16 && dtype != VLA_BF16) || !mfma_sizes(dim, vdim, out_inv_freq != nullptr))
    return VLA_ERR_HEAD_SIZE;
  // 8-byte fragment loads: query rows and cache rows must allow them
  if (((uintptr_t)q % 8) || ((q_stride * 2) % 8) || ((uintptr_t)key_cache % 8) ||
      ((uintptr_t)value_cache % 8))
    return VLA_ERR_ARG;
  // 16-byte fragment loads: query rows and cache rows must allow them
  if (((uintptr_t)q % 16) || ((q_stride * 2) % 16) || ((uintptr_t)key_cache % 16) ||
      ((uintptr_t)value_cache % 16))
    return VLA_ERR_ARG;
  const TileGrid to = tile_grid(num_seqs, max_query_len, num_rows, heads, kv_heads, dim,
                                walked_keys(max_blocks, block_size, window, keep_first, chunk));
  auto go = [&](auto tag) {
    using S = decltype(tag);
    using T = typename S::T;
    return by_value_slices(vdim, [&](int vb, int v_first) -> int {
      return launch_tiles<S>(dim / 32, vb, to, (hipStream_t)stream, (T*)out, out_stride, (const T*)q, q_stride,
                             (const T*)gate, gate_stride, (const T*)key_cache, (const T*)value_cache, block_tables,
                             max_blocks, query_start_loc, context_lens, out_inv_freq, interleaved, heads, kv_heads,
                             block_size, num_blocks, window, scale, keep_first, softcap, chunk, sinks, vdim, v_first);
    });
  };
  return dtype == VLA_BF16 ? go(BF16{}) : go(F16{});
}
