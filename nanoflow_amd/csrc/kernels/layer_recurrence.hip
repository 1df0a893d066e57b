// Linear recurrences of the layer-stack pipeline: a state S [dim][vdim] per head, fp32.  A token scales
// the state's rows, adds the outer product of its key and value, and reads the state with its query:
// after the update (FIXED_DECAY), or before it with the token's own key weighted by u (TOKEN_DECAY).
// With S the state before the token, both reads are
//     o = c (q . S) + b v,     b = q . k  or  q . (u * k),     c = the decay  or  1.
// Everything between the loaded projections and the stored output is fp32: rotation, decays,
// products, state, the per-head norm and the gate (both left out where no gate is given).
//
// recur_seq_kernel: one workgroup per (request, head) holds the head's state in registers and walks
// the request's rows, a few at a time through LDS.  Decode (one row): the state is streamed in, used,
// and streamed out once, through the caches (us, ordinary stores and these: 16 requests of 32 heads of 64 x 64, 8 MB, 7.4 -> 5.7, 64 17.0 -> 14.2, 256 60.5 ->
// 58.5, 16 of 16 heads of 128 x 128 10.0 -> 7.8; 0.5 to 4 MB 5.0 to 5.5 and 5.0 to 5.2).
//
// Portions of prompts are cut into chunks that are computed side by side, in three launches:
//   recur_chunk_state_kernel  what every chunk adds to a state that enters it as zero, and the factor the
//                             entering state is multiplied by;
//   recur_chunk_scan_kernel   the state that enters each chunk (one pass over the chunks per element), and
//                             the state the request leaves behind;
//   recur_chunk_out_kernel    every chunk's outputs from its entering state.
// Heads of 128 x 128 under fixed decays and of 64 x 64 under decays of the token have forms of their own in bf16 (recurrence_fixed.h, recurrence_token.h); in this one,
// the general one, inside a chunk the state lives in MFMA accumulators (v_mfma_f32_16x16x4_f32: products and sums in fp32)
// and 16 tokens are taken at a time:  o = (decayed q) S + A v,  S <- decays * S + (decayed k)^T v,  A[i][j] =
// q_i . k_j times the decay between the two.  An accumulator's rows 4g + r are the k index g of the r-th
// MFMA that multiplies by it, so S and A are operands where they lie.  A token's own decays enter as
// q 2^(L before i) and k 2^-(L through j), L counted from the start of the 16 tokens; where some L is
// below -100 fewer tokens are taken at a time.
#include <algorithm>
#include <cmath>

#include "layer_common.h"

namespace nf {

constexpr int kMaxStateDim = 256;

struct RecurrenceDims {
  int kp, vp;  // dim and vdim padded to 16
};
__host__ __device__ inline RecurrenceDims padded(int dim, int vdim) { return {(dim + 15) / 16 * 16, (vdim + 15) / 16 * 16}; }

// Element d of a row's head vector `src`, rotated to position `pos`.
template <class T>
__device__ __forceinline__ float load_rotated(const T* src, int d, const nf_rotation& rot, int pos) {
  const float y = Act<T>::load(src + d);
  const int half = rot.dims / 2;
  if (d >= 2 * half) return y;
  const int f = rot.interleaved ? d >> 1 : (d < half ? d : d - half);
  const bool first = rot.interleaved ? !(d & 1) : d < half;
  const float other = Act<T>::load(src + (rot.interleaved ? d ^ 1 : (first ? d + half : d - half)));
  const float cs = rot.table[((size_t)pos * half + f) * 2], sn = rot.table[((size_t)pos * half + f) * 2 + 1];
  return first ? y * cs - other * sn : y * cs + other * sn;
}

// log2 of the factor that key channel `col` (over all heads) is multiplied by at a row.  Limited to
// 2^-126: a smaller factor leaves nothing of a state in fp32, and sums of logs stay finite.
__device__ __forceinline__ float token_log2_decay(const nf_recurrence_args& a, int row, int col) {
  float z = a.w0[col];
  for (int s = 0; s < a.z_shares; ++s) z += a.z[((size_t)s * a.total_rows + row) * a.z_ld + col];
  return fmaxf(-expf(z) * 1.44269504088896340736f, -126.f);
}

template <class T, int NP, int KIND>
__global__ __launch_bounds__(1024) void recur_seq_kernel(nf_recurrence_args a, int tb) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const RecurrenceDims pd = padded(a.dim, a.vdim);
  const int req = a.req_begin + blockIdx.x, h = blockIdx.y;
  const int ns = blockDim.x / 256, vw = ns * 64;
  float* sq = lds;                   // [tb][kp]
  float* sk = sq + tb * pd.kp;       // [tb][kp]
  float* sw = sk + tb * pd.kp;       // [tb][kp] (TOKEN_DECAY)
  float* sv = sw + (KIND == NF_RECURRENCE_TOKEN_DECAY ? tb * pd.kp : 0);  // [tb][vw]
  float* sp = sv + tb * vw;          // [tb][4][vw]
  float* sb = sp + tb * 4 * vw;      // [tb]

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n_waves = blockDim.x >> 6;
  const int slice = tid >> 8, col = slice * 64 + (tid & 15) * 4, krow = (tid & 255) >> 4, swave = (tid & 255) >> 6;
  const int row0 = a.input_indptr[req], row1 = a.input_indptr[req + 1];
  if (row0 >= row1) return;
  const int slot = a.state_slots[req], np = pd.kp / 16;
  float* state = a.state + ((size_t)slot * a.heads + h) * pd.kp * pd.vp;
  const bool fresh = a.positions[row0] == 0;
  const float decay = KIND == NF_RECURRENCE_FIXED_DECAY ? exp2f(a.log2_decay[h]) : 1.f;

  float4_t S[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int k = krow + 16 * i;
    S[i] = float4_t{0.f, 0.f, 0.f, 0.f};
    if (!fresh && k < pd.kp && col < pd.vp) S[i] = *reinterpret_cast<const float4_t*>(state + (size_t)k * pd.vp + col);
  }

  for (int r0 = row0; r0 < row1; r0 += tb) {
    const int n = min(tb, row1 - r0);
    for (int e = tid; e < n * pd.kp; e += blockDim.x) {
      const int t = e / pd.kp, d = e % pd.kp, row = r0 + t;
      float q = 0.f, k = 0.f, w = 1.f;
      if (d < a.dim) {
        const T* qp = (const T*)a.q + (size_t)row * a.q_ld + (size_t)h * a.dim;
        const T* kp = (const T*)a.k + (size_t)row * a.k_ld + (size_t)h * a.dim;
        if constexpr (KIND == NF_RECURRENCE_FIXED_DECAY) {
          const int pos = a.positions[row];
          q = load_rotated(qp, d, a.rot, pos);
          k = load_rotated(kp, d, a.rot, pos) * a.k_scale;
        } else {
          q = Act<T>::load(qp + d);
          k = Act<T>::load(kp + d);
          w = exp2f(token_log2_decay(a, row, h * a.dim + d));
        }
      }
      sq[e] = q;
      sk[e] = k;
      if constexpr (KIND == NF_RECURRENCE_TOKEN_DECAY) sw[e] = w;
    }
    for (int e = tid; e < n * vw; e += blockDim.x) {
      const int t = e / vw, c = e % vw;
      sv[e] = c < a.vdim ? Act<T>::load((const T*)a.v + (size_t)(r0 + t) * a.v_ld + (size_t)h * a.vdim + c) : 0.f;
    }
    __syncthreads();
    for (int t = wave; t < n; t += n_waves) {
      float b = 0.f;
      for (int d = lane; d < a.dim; d += 64)
        b += sq[t * pd.kp + d] * sk[t * pd.kp + d] * (KIND == NF_RECURRENCE_TOKEN_DECAY ? a.u[(size_t)h * a.dim + d] : 1.f);
      b = wave_sum(b);
      if (lane == 0) sb[t] = b;
    }
    for (int t = 0; t < n; ++t) {
      const float4_t v = *reinterpret_cast<const float4_t*>(sv + t * vw + col);
      float4_t o{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        if (i >= np) continue;  // the state has np x 16 rows
        const int k = krow + 16 * i;
        const float w = KIND == NF_RECURRENCE_TOKEN_DECAY ? sw[t * pd.kp + k] : decay;
        o += S[i] * sq[t * pd.kp + k];
        S[i] = S[i] * w + v * sk[t * pd.kp + k];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = sum_over_near_lane_groups(o[e]);
      if (lane < 16) *reinterpret_cast<float4_t*>(sp + (t * 4 + swave) * vw + col) = o;
    }
    if (r0 + tb >= row1) {  // on its way while the rows are normed
      // The state has long been there; said once, ahead of the branches, it spares a wait for each store ahead of the next.
      __builtin_amdgcn_s_waitcnt(0x0F70);
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int k = krow + 16 * i;
        if (k >= pd.kp || col >= pd.vp) continue;
        store_through(state, (uint32_t)(pd.kp * pd.vp * sizeof(float)), (uint32_t)((k * pd.vp + col) * sizeof(float)), S[i]);
      }
    }
    __syncthreads();
    // per row: the four partial sums, the current token's own term, norm, gate
    for (int t = wave; t < n; t += n_waves) {
      const int row = r0 + t;
      float o[kMaxStateDim / 64], sqs = 0.f;
#pragma unroll
      for (int e = 0; e < kMaxStateDim / 64; ++e) {
        const int c = e * 64 + lane;
        o[e] = 0.f;
        if (c < a.vdim) {
          const float* p = sp + (size_t)t * 4 * vw + c;
          o[e] = (p[0] + p[vw] + p[2 * vw] + p[3 * vw]) * decay + sb[t] * sv[t * vw + c];
        }
        sqs += o[e] * o[e];
      }
      const float inv = a.g ? a.out_scale / sqrtf(wave_sum(sqs) / (float)a.vdim + a.eps) : a.out_scale;
#pragma unroll
      for (int e = 0; e < kMaxStateDim / 64; ++e) {
        const int c = e * 64 + lane;
        if (c >= a.vdim) continue;
        const int hc = h * a.vdim + c;
        float y = o[e] * inv;
        if (a.g) y *= silu<T>(Act<T>::load((const T*)a.g + (size_t)row * a.g_ld + hc));
        if (a.norm_weight) y *= a.norm_weight[hc];
        Act<T>::store((T*)a.out + (size_t)row * a.out_ld + a.out_col + hc, y);
      }
    }
    __syncthreads();
  }
  if (a.shift_x && h == 0)
    for (int c = tid * 4; c < a.shift_ld; c += blockDim.x * 4)
      *reinterpret_cast<float4_t*>(a.shift_state + (size_t)slot * a.shift_ld + c) =
          *reinterpret_cast<const float4_t*>(a.shift_x + (size_t)(row1 - 1) * a.shift_ld + c);
}

template <class T, int KIND>
static int launch_seq(const nf_recurrence_args& a, hipStream_t s) {
  const RecurrenceDims pd = padded(a.dim, a.vdim);
  const int ns = (pd.vp + 63) / 64, vw = ns * 64;
  // decode: one row per request; else as many rows at a time as 64 KB of LDS hold, at most 8
  auto lds_of = [&](int tb) {
    return ((size_t)tb * pd.kp * (KIND == NF_RECURRENCE_TOKEN_DECAY ? 3 : 2) + (size_t)tb * vw * 5 + tb) * sizeof(float);
  };
  int tb = a.rows == a.req_num ? 1 : 8;
  while (tb > 1 && lds_of(tb) > 64 * 1024) tb /= 2;
  const dim3 grid((unsigned)a.req_num, (unsigned)a.heads);
  auto go = [&](auto np) {
    recur_seq_kernel<T, decltype(np)::value, KIND><<<grid, ns * 256, lds_of(tb), s>>>(a, tb);
    return check_launch("nf_linear_recurrence");
  };
  const int np = pd.kp / 16;
  if (np <= 2) return go(ic<2>{});
  if (np <= 4) return go(ic<4>{});
  if (np <= 8) return go(ic<8>{});
  return go(ic<16>{});
}

// ---------------------------------------------------------------- chunks of a prompt's portion
constexpr int kStep = 16;           // tokens per step inside a chunk
constexpr float kMinStepLog2 = -100.f;

struct ChunkSpan {
  int req, row0, n, slot;  // request, first row, rows (0: no such chunk), index of its chunk in the workspace
};
// Chunk `slot` of the launch: chunks of `len` rows, request after request.
__device__ __forceinline__ ChunkSpan find_chunk(const nf_recurrence_args& a, int slot, int len) {
  int c = slot;
  for (int r = a.req_begin; r < a.req_begin + a.req_num; ++r) {
    const int row0 = a.input_indptr[r], rows = a.input_indptr[r + 1] - row0, n = (rows + len - 1) / len;
    if (c < n) return {r, row0 + c * len, min(len, rows - c * len), slot};
    c -= n;
  }
  return {-1, 0, 0, slot};
}

// Workspace: [chunks][heads] states in fragment order -- tile (kt, vt) of 16 x 16, lane, four rows -- then
// (TOKEN_DECAY) [chunks][heads][kp] factors.
__device__ __forceinline__ float* chunk_states(const nf_recurrence_args& a, const RecurrenceDims& pd, int slot, int h) {
  return (float*)a.workspace + ((size_t)slot * a.heads + h) * pd.kp * pd.vp;
}
__device__ __forceinline__ float* chunk_factors(const nf_recurrence_args& a, const RecurrenceDims& pd, int max_chunks, int slot, int h) {
  return (float*)a.workspace + (size_t)max_chunks * a.heads * pd.kp * pd.vp + ((size_t)slot * a.heads + h) * pd.kp;
}

}  // namespace nf

#include "recurrence_fixed.h"
#include "recurrence_token.h"

namespace nf {

template <int KIND, int NKT, int NVT>
struct ChunkShape {
  static constexpr int KP = NKT * 16, VP = 4 * NVT * 16;
  static constexpr int kPitch = KP + 4, vPitch = VP + 4;
  static constexpr int kGroups = (kStep * KP / 4 + 255) / 256;  // four-element groups per thread of a staged q or k
  static constexpr int vGroups = kStep * VP / 4 / 256;
  static constexpr int kPairs = (kStep * KP / 2 + 255) / 256;   // rotation pairs per thread
  static constexpr int kParts = 256 / KP, kPartTok = kStep / kParts;  // TOKEN_DECAY: thread = (channel, part of the tokens)
};

template <int KIND, int NKT, int NVT, bool kQ>
struct ChunkLds {
  using C = ChunkShape<KIND, NKT, NVT>;
  static constexpr bool kToken = KIND == NF_RECURRENCE_TOKEN_DECAY;
  __attribute__((aligned(16))) float q[kQ ? kStep * C::kPitch : 4];            // raw, or times 2^(L before the token)
  __attribute__((aligned(16))) float k[kStep * C::kPitch];                     // raw, or times 2^(decay to the end of the step)
  __attribute__((aligned(16))) float kb[kQ && kToken ? kStep * C::kPitch : 4];  // k 2^-(L through it)
  __attribute__((aligned(16))) float v[kStep * C::vPitch];
  __attribute__((aligned(16))) float o[kQ ? kStep * C::vPitch : 4];
  __attribute__((aligned(16))) float keep[C::KP];                              // TOKEN_DECAY: factor of a state row over the step
  float part[kToken ? C::kParts : 1][C::KP];
  float bonus[kStep];
  __attribute__((aligned(16))) float ss[kStep][4];
};

// A step's rows in registers: requested one step ahead, so that their latency passes under the step before.
// Loads are never branched around: rows and columns past the end read a valid place and are masked when they are
// written to LDS.
template <class T, int KIND, int NKT, int NVT, bool kQ>
struct StepLoads {
  using C = ChunkShape<KIND, NKT, NVT>;
  typename Act<T>::raw4 q[kQ ? C::kGroups : 1], k[C::kGroups], v[C::vGroups], g[kQ ? C::vGroups : 1];
  float cs[KIND == NF_RECURRENCE_FIXED_DECAY ? C::kPairs : 1], sn[KIND == NF_RECURRENCE_FIXED_DECAY ? C::kPairs : 1];
  float z[KIND == NF_RECURRENCE_TOKEN_DECAY ? C::kPartTok : 1];

  // rows [row, last] exist
  __device__ __forceinline__ void request(const nf_recurrence_args& a, int h, int row, int last) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int i = 0; i < C::kGroups; ++i) {
      const int e = i * 256 + tid, t = e / (C::KP / 4), c = e % (C::KP / 4) * 4;
      const size_t r = (size_t)min(row + t, last);
      const int cc = c < a.dim ? c : 0;
      if constexpr (kQ) q[i] = Act<T>::load_raw4((const T*)a.q + r * a.q_ld + h * a.dim + cc);
      k[i] = Act<T>::load_raw4((const T*)a.k + r * a.k_ld + h * a.dim + cc);
    }
#pragma unroll
    for (int i = 0; i < C::vGroups; ++i) {
      const int e = i * 256 + tid, t = e / (C::VP / 4), c = e % (C::VP / 4) * 4;
      const size_t r = (size_t)min(row + t, last);
      const int cc = c < a.vdim ? c : 0;
      v[i] = Act<T>::load_raw4((const T*)a.v + r * a.v_ld + h * a.vdim + cc);
      if constexpr (kQ) g[i] = Act<T>::load_raw4((const T*)(a.g ? a.g : a.v) + r * (a.g ? a.g_ld : a.v_ld) + h * a.vdim + cc);
    }
    if constexpr (KIND == NF_RECURRENCE_FIXED_DECAY) {
      const int half = a.rot.dims / 2;
      if (half > 0) {
#pragma unroll
        for (int i = 0; i < C::kPairs; ++i) {
          const int e = i * 256 + tid, t = e / (C::KP / 2), f = min(e % (C::KP / 2), half - 1);
          const float* tab = a.rot.table + ((size_t)a.positions[min(row + t, last)] * half + f) * 2;
          cs[i] = tab[0];
          sn[i] = tab[1];
        }
      }
    } else {
      const int c = tid % C::KP, part = tid / C::KP;
#pragma unroll
      for (int i = 0; i < C::kPartTok; ++i) {
        const size_t r = (size_t)min(row + part * C::kPartTok + i, last);
        const int cc = h * a.dim + (c < a.dim ? c : 0);
        z[i] = a.z[r * a.z_ld + cc];
        for (int s = 1; s < a.z_shares; ++s) z[i] += a.z[((size_t)s * a.total_rows + r) * a.z_ld + cc];
      }
    }
  }

  // The first n rows to LDS, the others as zeros.
  __device__ __forceinline__ void store(const nf_recurrence_args& a, ChunkLds<KIND, NKT, NVT, kQ>& s, int n) const {
    const float4_t zero{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < C::kGroups; ++i) {
      const int e = i * 256 + (int)threadIdx.x, t = e / (C::KP / 4), c = e % (C::KP / 4) * 4;
      if (C::KP < 64 && t >= kStep) continue;
      const bool live = t < n && c < a.dim;
      if constexpr (kQ) *reinterpret_cast<float4_t*>(s.q + t * C::kPitch + c) = live ? Act<T>::widen4(q[i]) : zero;
      *reinterpret_cast<float4_t*>(s.k + t * C::kPitch + c) = live ? Act<T>::widen4(k[i]) * a.k_scale : zero;
    }
#pragma unroll
    for (int i = 0; i < C::vGroups; ++i) {
      const int e = i * 256 + (int)threadIdx.x, t = e / (C::VP / 4), c = e % (C::VP / 4) * 4;
      *reinterpret_cast<float4_t*>(s.v + t * C::vPitch + c) = t < n && c < a.vdim ? Act<T>::widen4(v[i]) : zero;
    }
  }

  // FIXED_DECAY, after store() and a barrier: q and k rotated where they lie.
  __device__ __forceinline__ void rotate(const nf_recurrence_args& a, ChunkLds<KIND, NKT, NVT, kQ>& s) const {
    const int half = a.rot.dims / 2;
#pragma unroll
    for (int i = 0; i < C::kPairs; ++i) {
      const int e = i * 256 + (int)threadIdx.x, t = e / (C::KP / 2), f = e % (C::KP / 2);
      if (f >= half || t >= kStep) continue;
      const int c1 = t * C::kPitch + (a.rot.interleaved ? 2 * f : f), c2 = c1 + (a.rot.interleaved ? 1 : half);
      const float k1 = s.k[c1], k2 = s.k[c2];
      s.k[c1] = k1 * cs[i] - k2 * sn[i];
      s.k[c2] = k2 * cs[i] + k1 * sn[i];
      if constexpr (kQ) {
        const float q1 = s.q[c1], q2 = s.q[c2];
        s.q[c1] = q1 * cs[i] - q2 * sn[i];
        s.q[c2] = q2 * cs[i] + q1 * sn[i];
      }
    }
  }
};

// What a thread of a TOKEN_DECAY chunk keeps of its key channel.
struct ChannelDecay {
  float w0, lw[kStep], before, total;
};

// TOKEN_DECAY, between two barriers after store(): the log2 decays of this thread's tokens, their sum to LDS, and the
// tokens' bonus terms from raw q and k.
template <class T, int NKT, int NVT, bool kQ>
__device__ __forceinline__ void decay_sums(const nf_recurrence_args& a, ChunkLds<NF_RECURRENCE_TOKEN_DECAY, NKT, NVT, kQ>& s,
                                           const StepLoads<T, NF_RECURRENCE_TOKEN_DECAY, NKT, NVT, kQ>& ld, ChannelDecay& d, int h,
                                           int n) {
  using C = ChunkShape<NF_RECURRENCE_TOKEN_DECAY, NKT, NVT>;
  const int c = threadIdx.x % C::KP, part = threadIdx.x / C::KP;
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < C::kPartTok; ++i) {
    const float l = fmaxf(-expf(ld.z[i] + d.w0) * 1.44269504088896340736f, -126.f);
    d.lw[i] = part * C::kPartTok + i < n && c < a.dim ? l : 0.f;
    sum += d.lw[i];
  }
  s.part[part][c] = sum;
  if constexpr (kQ) {
    const int t = threadIdx.x >> 4, l = threadIdx.x & 15;
    float b = 0.f;
    for (int e = l; e < a.dim; e += 16) b += s.q[t * C::kPitch + e] * s.k[t * C::kPitch + e] * a.u[(size_t)h * a.dim + e];
    b = sum_of_16(b);
    if (l == 0) s.bonus[t] = b;
  }
}

// The channel's decay before this thread's tokens and over the step; whether it stays above kMinStepLog2.
template <int NKT, int NVT, bool kQ>
__device__ __forceinline__ bool decay_totals(ChunkLds<NF_RECURRENCE_TOKEN_DECAY, NKT, NVT, kQ>& s, ChannelDecay& d) {
  using C = ChunkShape<NF_RECURRENCE_TOKEN_DECAY, NKT, NVT>;
  const int c = threadIdx.x % C::KP, part = threadIdx.x / C::KP;
  d.before = d.total = 0.f;
#pragma unroll
  for (int p = 0; p < C::kParts; ++p) {
    const float x = s.part[p][c];
    if (p < part) d.before += x;
    d.total += x;
  }
  return d.total >= kMinStepLog2;
}

// q, k and k's quotient form from raw q and k.
template <int NKT, int NVT, bool kQ>
__device__ __forceinline__ void decay_apply(ChunkLds<NF_RECURRENCE_TOKEN_DECAY, NKT, NVT, kQ>& s, const ChannelDecay& d) {
  using C = ChunkShape<NF_RECURRENCE_TOKEN_DECAY, NKT, NVT>;
  const int c = threadIdx.x % C::KP, part = threadIdx.x / C::KP;
  float after = 0.f;  // sums of later tokens only: no difference of large sums
#pragma unroll
  for (int p = C::kParts - 1; p > 0; --p)
    if (p > part) after += s.part[p][c];
  float before = d.before;
#pragma unroll
  for (int i = 0; i < C::kPartTok; ++i) {
    float own_after = after;
#pragma unroll
    for (int j = C::kPartTok - 1; j > 0; --j)
      if (j > i) own_after += d.lw[j];
    const int at = (part * C::kPartTok + i) * C::kPitch + c;
    const float k = s.k[at];
    s.k[at] = k * __builtin_amdgcn_exp2f(own_after);
    if constexpr (kQ) {
      s.q[at] *= __builtin_amdgcn_exp2f(before);
      before += d.lw[i];
      s.kb[at] = k * __builtin_amdgcn_exp2f(-before);
    }
  }
  if (part == 0) s.keep[c] = __builtin_amdgcn_exp2f(d.total);
}

// S <- keep * S + k^T v over the step; the wavefront's NVT column tiles.
template <int KIND, int NKT, int NVT, bool kQ>
__device__ __forceinline__ void update_state(float4_t (&S)[NKT][NVT], const ChunkLds<KIND, NKT, NVT, kQ>& s, int n, float ld2,
                                             const float (&vr)[NVT][4]) {
  using C = ChunkShape<KIND, NKT, NVT>;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  float kf[4];  // FIXED_DECAY: decay from the token to the end of the step
  float keep_all = 1.f;
  if constexpr (KIND == NF_RECURRENCE_FIXED_DECAY) {
#pragma unroll
    for (int r = 0; r < 4; ++r) kf[r] = 4 * g + r < n ? __builtin_amdgcn_exp2f((float)(n - 1 - 4 * g - r) * ld2) : 0.f;
    keep_all = __builtin_amdgcn_exp2f((float)n * ld2);
  }
#pragma unroll
  for (int kt = 0; kt < NKT; ++kt) {
    float4_t keep{keep_all, keep_all, keep_all, keep_all};
    if constexpr (KIND == NF_RECURRENCE_TOKEN_DECAY) keep = *reinterpret_cast<const float4_t*>(s.keep + kt * 16 + 4 * g);
    float k[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      k[r] = s.k[(4 * g + r) * C::kPitch + kt * 16 + l16];
      if constexpr (KIND == NF_RECURRENCE_FIXED_DECAY) k[r] *= kf[r];
    }
#pragma unroll
    for (int vt = 0; vt < NVT; ++vt) {
      S[kt][vt] *= keep;
#pragma unroll
      for (int r = 0; r < 4; ++r) S[kt][vt] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[r], vr[vt][r], S[kt][vt], 0, 0, 0);
    }
  }
}

// The bound of two workgroups a CU keeps the state in VGPRs: with more room the compiler moves it to accumulation
// registers, and every scaling of it through moves between the two files.
template <class T, int KIND, int NKT, int NVT>
__global__ __launch_bounds__(256, 2) void recur_chunk_state_kernel(nf_recurrence_args a, int len, int max_chunks) {
  using C = ChunkShape<KIND, NKT, NVT>;
  constexpr bool kToken = KIND == NF_RECURRENCE_TOKEN_DECAY;
  __shared__ ChunkLds<KIND, NKT, NVT, false> s;
  const RecurrenceDims pd = padded(a.dim, a.vdim);
  const int h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
  const ChunkSpan ch = find_chunk(a, blockIdx.x, len);
  if (ch.n == 0) return;
  const float ld2 = kToken ? 0.f : a.log2_decay[h];
  const int last = ch.row0 + ch.n - 1;
  StepLoads<T, KIND, NKT, NVT, false> ld;
  ld.request(a, h, ch.row0, last);
  ChannelDecay d;
  const int channel = threadIdx.x % C::KP;
  if constexpr (kToken) d.w0 = a.w0[h * a.dim + (channel < a.dim ? channel : 0)];
  float log2_all = 0.f;
  float4_t S[NKT][NVT];
#pragma unroll
  for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
    for (int vt = 0; vt < NVT; ++vt) S[kt][vt] = float4_t{0.f, 0.f, 0.f, 0.f};
  for (int t0 = 0; t0 < ch.n; t0 += kStep) {
    const int n = min(kStep, ch.n - t0);
    __syncthreads();
    ld.store(a, s, n);
    if constexpr (kToken) {
      decay_sums<T, NKT, NVT, false>(a, s, ld, d, h, n);
      __syncthreads();
      decay_totals<NKT, NVT, false>(s, d);  // every factor formed here is at most 1, whatever the logs
      log2_all += d.total;
      decay_apply<NKT, NVT, false>(s, d);
    } else {
      __syncthreads();
      ld.rotate(a, s);
    }
    if (t0 + kStep < ch.n) ld.request(a, h, ch.row0 + t0 + kStep, last);
    __syncthreads();
    float vr[NVT][4];
#pragma unroll
    for (int vt = 0; vt < NVT; ++vt)
#pragma unroll
      for (int r = 0; r < 4; ++r) vr[vt][r] = s.v[(4 * g + r) * C::vPitch + (wave * NVT + vt) * 16 + l16];
    update_state<KIND, NKT, NVT, false>(S, s, n, ld2, vr);
  }
  float* dst = chunk_states(a, pd, ch.slot, h);
  const int v_tiles = pd.vp / 16;
#pragma unroll
  for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
    for (int vt = 0; vt < NVT; ++vt) {
      const int tile = wave * NVT + vt;
      if (kt * 16 < pd.kp && tile < v_tiles) *reinterpret_cast<float4_t*>(dst + ((size_t)(kt * v_tiles + tile) * 64 + lane) * 4) = S[kt][vt];
    }
  if constexpr (kToken)
    if ((int)threadIdx.x < pd.kp) chunk_factors(a, pd, max_chunks, ch.slot, h)[threadIdx.x] = exp2f(log2_all);
}

// kForm: the states lie as recurrence_fixed.h or recurrence_token.h, of the kind, has them
template <int KIND, bool kForm = false>
__global__ __launch_bounds__(256) void recur_chunk_scan_kernel(nf_recurrence_args a, int len, int max_chunks) {
  const RecurrenceDims pd = padded(a.dim, a.vdim);
  const int req = a.req_begin + blockIdx.x, h = blockIdx.y;
  const int row0 = a.input_indptr[req], rows = a.input_indptr[req + 1] - row0;
  if (rows <= 0) return;
  int slot0 = 0;
  for (int r = a.req_begin; r < req; ++r) slot0 += (a.input_indptr[r + 1] - a.input_indptr[r] + len - 1) / len;
  const int chunks = (rows + len - 1) / len, state_slot = a.state_slots[req];
  const int f4 = blockIdx.z * 256 + threadIdx.x, e = f4 * 4;  // four rows of a column, in fragment order
  if (e < pd.kp * pd.vp) {
    const int v_tiles = pd.vp / 16, lane = f4 & 63, tile = f4 >> 6;
    int k = tile / v_tiles * 16 + (lane >> 4) * 4, c = tile % v_tiles * 16 + (lane & 15);
    if constexpr (kForm) KIND == NF_RECURRENCE_FIXED_DECAY ? fixed_place(f4, &k, &c) : token_place(f4, &k, &c);
    float* state = a.state + ((size_t)state_slot * a.heads + h) * pd.kp * pd.vp + (size_t)k * pd.vp + c;
    const float ld2 = KIND == NF_RECURRENCE_FIXED_DECAY ? a.log2_decay[h] : 0.f;
    float4_t cur{0.f, 0.f, 0.f, 0.f};
    if (a.positions[row0] != 0)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        cur[r] = state[(size_t)r * pd.vp];
        if constexpr (kForm && KIND == NF_RECURRENCE_FIXED_DECAY) cur[r] = __builtin_canonicalizef(cur[r]);  // NaN shows in the upper half, all that `split` has of it
      }
    constexpr int kAhead = 4;  // loads do not depend on the running state
    for (int c0 = 0; c0 < chunks; c0 += kAhead) {
      float4_t add[kAhead], f[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        const int ci = min(c0 + i, chunks - 1);
        add[i] = *reinterpret_cast<const float4_t*>(chunk_states(a, pd, slot0 + ci, h) + e);
        if constexpr (KIND == NF_RECURRENCE_TOKEN_DECAY) {
          f[i] = *reinterpret_cast<const float4_t*>(chunk_factors(a, pd, max_chunks, slot0 + ci, h) + k);
        } else {
          const float x = exp2f((float)min(len, rows - ci * len) * ld2);
          f[i] = float4_t{x, x, x, x};
        }
      }
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        if (c0 + i >= chunks) continue;
        *reinterpret_cast<float4_t*>(chunk_states(a, pd, slot0 + c0 + i, h) + e) = cur;
        cur = cur * f[i] + add[i];
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) state[(size_t)r * pd.vp] = cur[r];
  }
  if (a.shift_x && h == 0 && blockIdx.z == 0)
    for (int c = threadIdx.x * 4; c < a.shift_ld; c += 1024)
      *reinterpret_cast<float4_t*>(a.shift_state + (size_t)state_slot * a.shift_ld + c) =
          *reinterpret_cast<const float4_t*>(a.shift_x + (size_t)(row0 + rows - 1) * a.shift_ld + c);
}

template <class T, int KIND, int NKT, int NVT>
__global__ __launch_bounds__(256, 2) void recur_chunk_out_kernel(nf_recurrence_args a, int len) {
  using C = ChunkShape<KIND, NKT, NVT>;
  constexpr bool kToken = KIND == NF_RECURRENCE_TOKEN_DECAY;
  __shared__ ChunkLds<KIND, NKT, NVT, true> s;
  const RecurrenceDims pd = padded(a.dim, a.vdim);
  const int h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
  const ChunkSpan ch = find_chunk(a, blockIdx.x, len);
  if (ch.n == 0) return;
  const float ld2 = kToken ? 0.f : a.log2_decay[h];
  const int last = ch.row0 + ch.n - 1;
  StepLoads<T, KIND, NKT, NVT, true> ld;
  ld.request(a, h, ch.row0, last);
  ChannelDecay d;
  const int channel = threadIdx.x % C::KP;
  if constexpr (kToken) d.w0 = a.w0[h * a.dim + (channel < a.dim ? channel : 0)];
  float4_t S[NKT][NVT];
  const float* src = chunk_states(a, pd, ch.slot, h);
  const int v_tiles = pd.vp / 16;
#pragma unroll
  for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
    for (int vt = 0; vt < NVT; ++vt) {
      const int tile = wave * NVT + vt;
      const bool in = kt * 16 < pd.kp && tile < v_tiles;
      S[kt][vt] = *reinterpret_cast<const float4_t*>(src + ((size_t)(in ? kt * v_tiles + tile : 0) * 64 + lane) * 4);
      if (!in) S[kt][vt] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
  int n;
  for (int t0 = 0; t0 < ch.n; t0 += n) {
    n = min(kStep, ch.n - t0);
    const int row = ch.row0 + t0;
    for (;;) {
      __syncthreads();
      ld.store(a, s, n);
      __syncthreads();
      if constexpr (kToken) {
        decay_sums<T, NKT, NVT, true>(a, s, ld, d, h, n);
        __syncthreads();
        const bool ok = decay_totals<NKT, NVT, true>(s, d);
        if (__syncthreads_or(!ok) && n > 1) {
          n = n > 4 ? 4 : 1;
          continue;
        }
        decay_apply<NKT, NVT, true>(s, d);
      } else {
        ld.rotate(a, s);
      }
      break;
    }
    typename Act<T>::raw4 gate[C::vGroups];
#pragma unroll
    for (int i = 0; i < C::vGroups; ++i) gate[i] = ld.g[i];
    if (t0 + n < ch.n) ld.request(a, h, row + n, last);
    __syncthreads();
    // A^T[j][i] in fragment form: lane holds j = 4g + r of i = l16; and the part of o that the entering state gives
    float4_t at{0.f, 0.f, 0.f, 0.f}, o[NVT];
#pragma unroll
    for (int vt = 0; vt < NVT; ++vt) o[vt] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt) {
      const float4_t q = *reinterpret_cast<const float4_t*>(s.q + l16 * C::kPitch + kt * 16 + 4 * g);
      const float4_t k = *reinterpret_cast<const float4_t*>((kToken ? s.kb : s.k) + l16 * C::kPitch + kt * 16 + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        at = __builtin_amdgcn_mfma_f32_16x16x4f32(k[r], q[r], at, 0, 0, 0);
#pragma unroll
        for (int vt = 0; vt < NVT; ++vt) o[vt] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[r], S[kt][vt][r], o[vt], 0, 0, 0);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 4 * g + r, i = l16;
      if constexpr (!kToken) {
        at[r] = j <= i ? at[r] * __builtin_amdgcn_exp2f((float)(i - j) * ld2) : 0.f;
      } else {
        at[r] = j < i ? at[r] : 0.f;
        if (j == i) at[r] = s.bonus[i];
      }
      if (j >= n || i >= n) at[r] = 0.f;
    }
    if constexpr (!kToken) {  // row i = 4g + r of o: the entering state has decayed i + 1 times
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float f = __builtin_amdgcn_exp2f((float)(4 * g + r + 1) * ld2);
#pragma unroll
        for (int vt = 0; vt < NVT; ++vt) o[vt][r] *= f;
      }
    }
    float vr[NVT][4];
#pragma unroll
    for (int vt = 0; vt < NVT; ++vt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        vr[vt][r] = s.v[(4 * g + r) * C::vPitch + (wave * NVT + vt) * 16 + l16];
        o[vt] = __builtin_amdgcn_mfma_f32_16x16x4f32(at[r], vr[vt][r], o[vt], 0, 0, 0);
      }
    if (t0 + n < ch.n) update_state<KIND, NKT, NVT, true>(S, s, n, ld2, vr);  // what the last step leaves, the scan has

    // per-head norm over all columns, gate; through LDS, so that rows are written in whole runs
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float ss = 0.f;
#pragma unroll
      for (int vt = 0; vt < NVT; ++vt) {
        ss += o[vt][r] * o[vt][r];
        s.o[(4 * g + r) * C::vPitch + (wave * NVT + vt) * 16 + l16] = o[vt][r];
      }
      ss = sum_of_16(ss);
      if (l16 == 0) s.ss[4 * g + r][wave] = ss;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < C::vGroups; ++i) {
      const int e = i * 256 + (int)threadIdx.x, t = e / (C::VP / 4), c = e % (C::VP / 4) * 4;
      const float4_t part = *reinterpret_cast<const float4_t*>(s.ss[t]);
      const float inv = a.g ? a.out_scale / sqrtf((part[0] + part[1] + part[2] + part[3]) / (float)a.vdim + a.eps) : a.out_scale;
      float4_t y = *reinterpret_cast<const float4_t*>(s.o + t * C::vPitch + c) * inv;
      if (a.norm_weight && c < a.vdim) y *= *reinterpret_cast<const float4_t*>(a.norm_weight + h * a.vdim + c);
      const float4_t g4 = Act<T>::widen4(gate[i]);
#pragma unroll
      for (int x = 0; x < 4; ++x) y[x] *= a.g ? silu<T>(g4[x]) : 1.f;
      if (t < n && c < a.vdim)
        Act<T>::store4((T*)a.out + (size_t)(row + t) * a.out_ld + a.out_col + (size_t)h * a.vdim + c, y);
    }
  }
}

// Chunk length and count of a launch, or 0 chunks where the sequential kernel is the better one (few rows per request,
// states beyond the tiles) or the workspace is too small.
struct ChunkPlan {
  int len, chunks;
};
static size_t chunk_bytes(int heads, int dim, int vdim) {
  const RecurrenceDims pd = padded(dim, vdim);
  return (size_t)heads * (pd.kp * pd.vp + pd.kp) * sizeof(float);
}
constexpr int kMinChunk = 64, kMaxChunkRequests = 64;
static ChunkPlan chunk_plan(const nf_recurrence_args& a) {
  const RecurrenceDims pd = padded(a.dim, a.vdim);
  if (pd.kp > 128 || pd.vp > 128 || (long long)a.rows < 24ll * a.req_num || !a.workspace) return {0, 0};
  // rows are read and written four elements at a time
  const size_t four = 4 * (a.dtype == NF_BF16 ? 2 : 4);
  const uintptr_t at = (uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.g | (uintptr_t)a.out;
  if ((a.dim | a.vdim | a.q_ld | a.k_ld | a.v_ld | (a.g ? a.g_ld : 0) | a.out_ld | a.out_col) % 4 || at % four ||
      (uintptr_t)a.norm_weight % 16)
    return {0, 0};
  int len = kMinChunk;
  // longer chunks, fewer states through memory, as long as every CU has the workgroups it can hold
  const int enough = pd.kp * pd.vp > 64 * 64 ? 512 : 1024;
  while (len < 256 && (long long)(a.rows / (2 * len)) * a.heads >= enough) len *= 2;
  const int chunks = a.rows / len + a.req_num;
  if ((size_t)chunks * chunk_bytes(a.heads, a.dim, a.vdim) > a.workspace_bytes) return {0, 0};
  return {len, chunks};
}

template <class T, int KIND, int NKT, int NVT>
static int launch_chunks(const nf_recurrence_args& a, const ChunkPlan& p, hipStream_t s) {
  const RecurrenceDims pd = padded(a.dim, a.vdim);
  const dim3 grid((unsigned)p.chunks, (unsigned)a.heads);
  recur_chunk_state_kernel<T, KIND, NKT, NVT><<<grid, 256, 0, s>>>(a, p.len, p.chunks);
  int rc = check_launch("nf_linear_recurrence (chunk states)");
  if (rc) return rc;
  const unsigned parts = (unsigned)((pd.kp * pd.vp / 4 + 255) / 256);
  recur_chunk_scan_kernel<KIND><<<dim3((unsigned)a.req_num, (unsigned)a.heads, parts), 256, 0, s>>>(a, p.len, p.chunks);
  rc = check_launch("nf_linear_recurrence (chunk scan)");
  if (rc) return rc;
  recur_chunk_out_kernel<T, KIND, NKT, NVT><<<grid, 256, 0, s>>>(a, p.len);
  return check_launch("nf_linear_recurrence (chunk outputs)");
}

// Fixed decays on the 16-bit matrix instructions (recurrence_fixed.h): heads of 128 x 128 in bf16, neither rotated nor gated, rows read and written 16 bytes at
// a time; wherever the fp32 form takes chunks, for it was slower at every number of rows (all of 16 heads, us, fp32 form and this: 40 rows 25.8, 14.6; 500 rows 42, 24; 2047
// 67, 38; 8000 195, 113; 8 requests of 256 72, 49; fewer heads were not timed: of a long prompt they leave CUs idle in either form).  Halves of a chunk where requests hardly fill one and the CUs are not all taken: 128 rows 20.1 -> 16.9 us,
// but 2 x 300 25.7 -> 27.0.
static ChunkPlan fixed_plan(const nf_recurrence_args& a) {
  if (a.dtype != NF_BF16 || a.kind != NF_RECURRENCE_FIXED_DECAY || a.dim != kFixedDim || a.vdim != kFixedDim || a.rot.dims != 0 || a.g) return {0, 0};
  if ((a.q_ld | a.k_ld | a.v_ld | a.out_ld | a.out_col) % 8 || ((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.out) % 16) return {0, 0};
  if (std::max(std::max(a.q_ld, a.k_ld), a.v_ld) >= 1 << 24) return {0, 0};  // a chunk's rows within 32-bit offsets
  const bool brief = a.rows <= 160ll * a.req_num && ((long long)a.rows / kFixedChunk + a.req_num) * a.heads <= cu_count();
  const int len = brief ? kFixedChunk / 2 : kFixedChunk, chunks = a.rows / len + a.req_num;
  if ((size_t)chunks * chunk_bytes(a.heads, a.dim, a.vdim) > a.workspace_bytes) return {0, 0};
  return {len, chunks};
}
static int launch_fixed(const nf_recurrence_args& a, const ChunkPlan& p, hipStream_t s) {
  static bool attr_set = false;  // benign race: the call is idempotent
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(recur_fixed_state_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 2 * FixedTile::bytes);
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void*>(recur_fixed_out_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kFixedOutLds);
    if (e != hipSuccess) {
      set_error("nf_linear_recurrence: cannot reserve %d bytes of LDS: %s", kFixedOutLds, hipGetErrorString(e));
      return NF_ERR_RUNTIME;
    }
    attr_set = true;
  }
  const dim3 grid((unsigned)p.chunks, (unsigned)a.heads);
  recur_fixed_state_kernel<<<grid, 512, 2 * FixedTile::bytes, s>>>(a, p.len);
  int rc = check_launch("nf_linear_recurrence (chunk states)");
  if (rc) return rc;
  recur_chunk_scan_kernel<NF_RECURRENCE_FIXED_DECAY, true><<<dim3((unsigned)a.req_num, (unsigned)a.heads, kFixedDim * kFixedDim / 1024), 256, 0, s>>>(a, p.len, p.chunks);
  rc = check_launch("nf_linear_recurrence (chunk scan)");
  if (rc) return rc;
  recur_fixed_out_kernel<<<grid, 512, kFixedOutLds, s>>>(a, p.len);
  return check_launch("nf_linear_recurrence (chunk outputs)");
}

// Decays of every token, 64 tokens at a time (recurrence_token.h): heads of 64 x 64 in bf16, rows read and written 16 bytes at a time; wherever the general form
// takes chunks, for it was slower at every number of rows (all of 32 heads, us, general form and this: 40 rows 21.1, 14.1; 129 rows 28.0, 16.3; 500 rows 32, 20; 3000 85, 60;
// 8000, in its chunks of 256, 173, 135; 8 requests of 256 61, 48; 2047 rows of which most blocks decay below 2^-100, its steps then of four tokens or one, 597, 72).
static ChunkPlan token_plan(const nf_recurrence_args& a) {
  if (a.dtype != NF_BF16 || a.kind != NF_RECURRENCE_TOKEN_DECAY || a.dim != kTokenDim || a.vdim != kTokenDim) return {0, 0};
  if ((a.q_ld | a.k_ld | a.v_ld | (a.g ? a.g_ld : 0) | a.out_ld | a.out_col) % 8 || a.z_ld % 4 ||
      ((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.g | (uintptr_t)a.out | (uintptr_t)a.z | (uintptr_t)a.w0 | (uintptr_t)a.u) % 16)
    return {0, 0};
  if (std::max(a.k_ld, a.v_ld) >= 1 << 24) return {0, 0};  // a chunk's rows within 32-bit offsets
  const int chunks = a.rows / kTokenChunk + a.req_num;
  if ((size_t)chunks * chunk_bytes(a.heads, a.dim, a.vdim) > a.workspace_bytes) return {0, 0};
  return {kTokenChunk, chunks};
}
static int launch_token(const nf_recurrence_args& a, const ChunkPlan& p, hipStream_t s) {
  const dim3 grid((unsigned)p.chunks, (unsigned)a.heads);
  recur_token_state_kernel<<<grid, 4 * kTokenChunk, 0, s>>>(a, p.chunks);
  int rc = check_launch("nf_linear_recurrence (chunk states)");
  if (rc) return rc;
  recur_chunk_scan_kernel<NF_RECURRENCE_TOKEN_DECAY, true><<<dim3((unsigned)a.req_num, (unsigned)a.heads, kTokenDim * kTokenDim / 1024), 256, 0, s>>>(a, p.len, p.chunks);
  rc = check_launch("nf_linear_recurrence (chunk scan)");
  if (rc) return rc;
  recur_token_out_kernel<<<grid, 4 * kTokenChunk, 0, s>>>(a);
  return check_launch("nf_linear_recurrence (chunk outputs)");
}

template <class T, int KIND>
static int launch_recurrence(nf_recurrence_args a, hipStream_t s) {
  if (KIND == NF_RECURRENCE_TOKEN_DECAY) a.k_scale = 1.f;
  const ChunkPlan p = chunk_plan(a);
  if (p.chunks == 0) return launch_seq<T, KIND>(a, s);
  if constexpr (std::is_same_v<T, bf16_t> && KIND == NF_RECURRENCE_FIXED_DECAY) {
    const ChunkPlan f = fixed_plan(a);
    if (f.chunks > 0) return launch_fixed(a, f, s);
  }
  if constexpr (std::is_same_v<T, bf16_t> && KIND == NF_RECURRENCE_TOKEN_DECAY) {
    const ChunkPlan f = token_plan(a);
    if (f.chunks > 0) return launch_token(a, f, s);
  }
  const RecurrenceDims pd = padded(a.dim, a.vdim);
  const bool wide = pd.vp > 64;
  if (pd.kp <= 32) return wide ? launch_chunks<T, KIND, 2, 2>(a, p, s) : launch_chunks<T, KIND, 2, 1>(a, p, s);
  if (pd.kp <= 64) return wide ? launch_chunks<T, KIND, 4, 2>(a, p, s) : launch_chunks<T, KIND, 4, 1>(a, p, s);
  return wide ? launch_chunks<T, KIND, 8, 2>(a, p, s) : launch_chunks<T, KIND, 8, 1>(a, p, s);
}

}  // namespace nf

using namespace nf;

extern "C" {

size_t nf_recurrence_state_elements(int dim, int vdim) {
  if (dim <= 0 || vdim <= 0) return 0;
  const RecurrenceDims pd = padded(dim, vdim);
  return (size_t)pd.kp * pd.vp;
}

size_t nf_recurrence_workspace_bytes(int heads, int dim, int vdim, int max_rows, int max_requests) {
  if (heads <= 0 || dim <= 0 || vdim <= 0 || max_rows <= 0) return 0;
  const size_t chunks = (size_t)max_rows / kMinChunk + std::min(max_requests, kMaxChunkRequests);
  return chunks * chunk_bytes(heads, dim, vdim);
}

int nf_linear_recurrence(const nf_recurrence_args* args, nf_stream_t stream) {
  const char* who = "nf_linear_recurrence";
  NF_REQUIRE(args, "%s: null pointer", who);
  const nf_recurrence_args& a = *args;
  NF_REQUIRE(a.dtype == NF_F32 || a.dtype == NF_BF16, "%s: unknown dtype %d", who, a.dtype);
  NF_REQUIRE(a.kind == NF_RECURRENCE_FIXED_DECAY || a.kind == NF_RECURRENCE_TOKEN_DECAY, "%s: unknown kind %d", who, a.kind);
  NF_REQUIRE(a.heads > 0 && a.heads <= 65535 && a.dim > 0 && a.vdim > 0 && a.dim <= kMaxStateDim && a.vdim <= kMaxStateDim,
             "%s: %d heads of %d x %d (at most %d)", who, a.heads, a.dim, a.vdim, kMaxStateDim);
  NF_REQUIRE(a.req_num >= 0 && a.req_begin >= 0 && a.rows >= a.req_num && a.row_begin >= 0, "%s: %d requests with %d rows",
             who, a.req_num, a.rows);
  NF_REQUIRE(a.q_ld >= a.heads * a.dim && a.k_ld >= a.heads * a.dim && a.v_ld >= a.heads * a.vdim &&
                 (!a.g || a.g_ld >= a.heads * a.vdim) &&
                 a.out_col >= 0 && a.out_col + a.heads * a.vdim <= a.out_ld,
             "%s: row strides too small", who);
  if (a.req_num == 0) return NF_OK;
  NF_REQUIRE(a.q && a.k && a.v && (a.g || !a.norm_weight) && a.state && a.out && a.input_indptr && a.positions && a.state_slots,
             "%s: null pointer", who);
  if (a.kind == NF_RECURRENCE_FIXED_DECAY) {
    NF_REQUIRE(a.log2_decay && a.rot.dims >= 0 && a.rot.dims % 2 == 0 && a.rot.dims <= a.dim && (a.rot.dims == 0 || a.rot.table),
               "%s: decay or rotation missing", who);
  } else {
    NF_REQUIRE(a.z && a.w0 && a.u && a.z_shares >= 1 && a.z_shares <= kMaxShares && a.z_ld >= a.heads * a.dim &&
                   a.total_rows >= a.row_begin + a.rows,
               "%s: token decay inputs missing", who);
  }
  NF_REQUIRE(!a.shift_x || (a.shift_state && a.shift_ld > 0 && a.shift_ld % 4 == 0), "%s: shift state missing", who);
  hipStream_t s = (hipStream_t)stream;
  if (a.dtype == NF_BF16)
    return a.kind == NF_RECURRENCE_FIXED_DECAY ? launch_recurrence<bf16_t, NF_RECURRENCE_FIXED_DECAY>(a, s)
                                               : launch_recurrence<bf16_t, NF_RECURRENCE_TOKEN_DECAY>(a, s);
  return a.kind == NF_RECURRENCE_FIXED_DECAY ? launch_recurrence<float, NF_RECURRENCE_FIXED_DECAY>(a, s)
                                             : launch_recurrence<float, NF_RECURRENCE_TOKEN_DECAY>(a, s);
}

}  // extern "C"
