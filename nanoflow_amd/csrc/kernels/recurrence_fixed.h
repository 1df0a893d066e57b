#pragma once
// Chunks of prompts under one fixed decay per head, on the 16-bit matrix instructions: bf16 q, k and v of 128 features a head that enter as they are (no
// rotation, no gate).  (included by layer_recurrence.hip)
//
// What bounded the fp32 form was its MFMAs (16 x 16 x 4 takes as long as 16 x 16 x 32 in bf16) and the states' way through memory.  Here a chunk of 128 tokens
// is taken at once:
//     o_i = d^(i+1) q_i S + sum over j <= i of d^(i-j) (q_i . k_j) v_j,    S <- d^n S + sum of k_j (d^(n-1-j) v_j)
// q, k and v are exact operands.  The others -- state, decayed scores, decayed values -- are fp32 numbers, each taken apart into three bf16 numbers of
// eight bits whose sum it is (`split`), so their products are exact as well and the sums are fp32, as they were: three MFMAs for one, at an eighth of its cost
// per token.  2047 tokens of 16 heads (us, fp32 form -> this): chunk states 18.8 -> 11.1, scan 13.5 -> 9.5 over half as many states, outputs 35.5 -> 17.0; the
// states' error against 64 bits 9.6e-8 -> 7.0e-8.
// A token's infinities and NaN reach the tokens of its 16 and later ones, as in the fp32 form.  But an infinity against a number of which eight bits are the whole
// meets zeros as that number's other parts, and tokens of a whole chunk meet one by one: so a wavefront whose sums are not all finite takes the others again 16 tokens
// at a time in fp32 (`fixed_steps`), as the fp32 form does.  (The figures are without that check, 40 vector instructions a wavefront and phase.)

namespace nf {

constexpr int kFixedDim = 128, kFixedChunk = 128;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// x = hi + mid + lo, each with its lower 16 bits zero: eight bits of the significand at a time, cut off, so that nothing is rounded.  What is not finite
// stays in hi alone.
struct Split {
  uint32_t hi, mid, lo;
};
__device__ __forceinline__ Split split(float x) {
  const uint32_t hi = __float_as_uint(x) & 0xffff0000u;
  float r = x - __uint_as_float(hi);
  r = r == r ? r : 0.f;
  const uint32_t mid = __float_as_uint(r) & 0xffff0000u;
  return Split{hi, mid, __float_as_uint(r - __uint_as_float(mid))};
}
// The bf16 numbers of a (lower half) and b.
__device__ __forceinline__ uint32_t pair_of(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// Eight fp32 operands as three bf16 ones, by place: hi, mid, lo.
struct Triple {
  u32x4 part[3];
};
__device__ __forceinline__ Triple triple_of(const float (&x)[8]) {
  Split s[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) s[e] = split(x[e]);
  Triple t;
  t.part[0] = u32x4{pair_of(s[0].hi, s[1].hi), pair_of(s[2].hi, s[3].hi), pair_of(s[4].hi, s[5].hi), pair_of(s[6].hi, s[7].hi)};
  t.part[1] = u32x4{pair_of(s[0].mid, s[1].mid), pair_of(s[2].mid, s[3].mid), pair_of(s[4].mid, s[5].mid), pair_of(s[6].mid, s[7].mid)};
  t.part[2] = u32x4{pair_of(s[0].lo, s[1].lo), pair_of(s[2].lo, s[3].lo), pair_of(s[4].lo, s[5].lo), pair_of(s[6].lo, s[7].lo)};
  return t;
}
template <class A, class B>
__device__ __forceinline__ float4_t mfma_bf16(const A& a, const B& b, float4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Whether all sums of the wavefront are finite; and x with what is not as y has it.
template <int n>
__device__ __forceinline__ bool all_finite(const float4_t (&x)[n]) {
  float4_t zero{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < n; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) zero[r] = __builtin_fmaf(x[i][r], 0.f, zero[r]);
  return !__any(zero[0] + zero[1] + (zero[2] + zero[3]) != 0.f);  // true of a NaN
}
__device__ __forceinline__ void mend(float4_t& x, const float4_t& y) {
#pragma unroll
  for (int r = 0; r < 4; ++r) x[r] = fabsf(x[r]) < INFINITY ? x[r] : y[r];
}

// Rows of 128 bf16 in LDS, 16 chunks of 16 bytes permuted within a row by its number in 16: a chunk of 16 neighbouring rows, and 32 bytes of 16 rows
// that a transposing read takes, lie in different banks.
struct FixedTile {
  static constexpr int bytes = kFixedChunk * 256;
  static __device__ __forceinline__ int perm(int row) { return ((row & 3) << 1) | ((row >> 2) & 1) | (row & 8); }
  static __device__ __forceinline__ uint32_t chunk(int row, int c) { return (uint32_t)(row * 256 + ((c ^ perm(row & 15)) << 4)); }
  // Rows [0, n) of a head, `ld` elements apart, by 8 wavefronts, four rows an instruction; the others as zeros.
  static __device__ __forceinline__ void load(const void* src, int ld, int n, uint32_t lds, int wave, int lane) {
    const rsrc_t r = make_rsrc(src, ((size_t)(n - 1) * ld + kFixedDim) * 2);
#pragma unroll
    for (int i = 0; i < kFixedChunk / 32; ++i) {
      const int row = (i * 8 + wave) * 4 + (lane >> 4);
      const uint32_t off = (uint32_t)row * (uint32_t)ld * 2u + (uint32_t)(((lane & 15) ^ perm(row & 15)) << 4);
      load16_to_lds(r, row < n ? off : kOob, __builtin_amdgcn_readfirstlane(lds + (i * 8 + wave) * 1024));
    }
  }
  static __device__ __forceinline__ float one(const uint8_t* tile, int row, int col) {
    return bf16_bits_to_f32(*reinterpret_cast<const uint16_t*>(tile + chunk(row, col >> 3) + (col & 7) * 2));
  }
  // What an MFMA operand of four tokens each is made of: tokens first .. first + 3 of the lane's column of 16-column unit u; the lane group's
  // lanes read four rows of 32 bytes between them.
  static __device__ __forceinline__ short4_t column(const uint8_t* tile, int first, int u, int i16) {
    return lds_read_tr16(tile + chunk(first + (i16 >> 2), 2 * u + ((i16 & 3) >> 1)) + (i16 & 1) * 8);
  }
};
typedef short short8_t __attribute__((ext_vector_type(8)));
__device__ __forceinline__ short8_t join(short4_t lo, short4_t hi) { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }

// A chunk's state lies as the outputs' MFMAs take it: [16 columns of v][32 rows of k][lane][8], lane (l16, lq) with column l16, rows 4 lq .. + 3 and 16 + 4 lq .. + 3.
// Column and first of the four rows of the float4 at index f4:
__device__ __forceinline__ void fixed_place(int f4, int* k, int* c) {
  const int lane = (f4 >> 1) & 63, tile = f4 >> 7;
  *k = (tile & 3) * 32 + (f4 & 1) * 16 + (lane >> 4) * 4;
  *c = (tile >> 2) * 16 + (lane & 15);
}

// A chunk as the fp32 form takes it, for 16 columns of v from `col` on: S [row of k 16 kt + 4 lq + r][column l16] before the 16 tokens from t0 on, and after
// them; outputs(t0, S) has the former.
template <class F>
__device__ __forceinline__ void fixed_steps(const nf_recurrence_args& a, const uint8_t* kt, const uint8_t* vt, float ld2, int n, int col, int l16, int lq, float4_t (&S)[8],
                                            F&& outputs) {
#pragma unroll 1
  for (int t0 = 0; t0 < n; t0 += 16) {
    outputs(t0, S);
    const int some = min(16, n - t0);
    const float keep = __builtin_amdgcn_exp2f((float)some * ld2);
#pragma unroll
    for (int i = 0; i < 8; ++i) S[i] *= keep;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 4 * lq + r;
      const float v = FixedTile::one(vt, t0 + t, col + l16), f = t < some ? __builtin_amdgcn_exp2f((float)(some - 1 - t) * ld2) : 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) S[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(FixedTile::one(kt, t0 + t, i * 16 + l16) * a.k_scale * f, v, S[i], 0, 0, 0);
    }
  }
}

// What a chunk adds to the state.  A wavefront has 16 columns of v, all rows of k.
__global__ __launch_bounds__(512) void recur_fixed_state_kernel(nf_recurrence_args a, int len) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t tiles[];
  const int h = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, lq = lane >> 4;
  const ChunkSpan ch = find_chunk(a, blockIdx.x, len);
  if (ch.n == 0) return;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)tiles;
  const uint8_t *kt = tiles, *vt = tiles + FixedTile::bytes;
  FixedTile::load((const uint16_t*)a.k + (size_t)ch.row0 * a.k_ld + h * kFixedDim, a.k_ld, ch.n, lds0, wave, lane);
  FixedTile::load((const uint16_t*)a.v + (size_t)ch.row0 * a.v_ld + h * kFixedDim, a.v_ld, ch.n, lds0 + FixedTile::bytes, wave, lane);
  const float ld2 = a.log2_decay[h];
  float4_t S[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) S[i] = float4_t{0.f, 0.f, 0.f, 0.f};
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
#pragma unroll
  for (int t0 = 0; t0 < kFixedChunk; t0 += 32) {
    if (t0 >= ch.n) break;
    const short8_t v8 = join(FixedTile::column(vt, t0 + lq * 8, wave, l16), FixedTile::column(vt, t0 + lq * 8 + 4, wave, l16));
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int after = ch.n - 1 - (t0 + lq * 8 + e);  // tokens past the last one are zeros
      v[e] = bf16_bits_to_f32((uint16_t)v8[e]) * (a.k_scale * __builtin_amdgcn_exp2f((float)max(after, 0) * ld2));
    }
    const Triple w = triple_of(v);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const short8_t k8 = join(FixedTile::column(kt, t0 + lq * 8, i, l16), FixedTile::column(kt, t0 + lq * 8 + 4, i, l16));
#pragma unroll
      for (int p = 2; p >= 0; --p) S[i] = mfma_bf16(k8, w.part[p], S[i]);
    }
  }
  if (!all_finite(S)) {
    float4_t again[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) again[i] = float4_t{0.f, 0.f, 0.f, 0.f};
    fixed_steps(a, kt, vt, ld2, ch.n, wave * 16, l16, lq, again, [](int, const float4_t (&)[8]) {});
#pragma unroll
    for (int i = 0; i < 8; ++i) mend(S[i], again[i]);
  }
  float* dst = chunk_states(a, {kFixedDim, kFixedDim}, ch.slot, h);
#pragma unroll
  for (int i = 0; i < 8; ++i) *reinterpret_cast<float4_t*>(dst + ((size_t)(wave * 4 + i / 2) * 64 + lane) * 8 + (i & 1) * 4) = S[i];
}

// A chunk's outputs from the state that enters it.  Four wavefronts have the chunk's first 64 tokens, four the others; of these, each one's scores
// of 16 tokens, then 32 columns of all 64 outputs.
constexpr int kFixedScores = 3 * 2 * 4 * 1024;  // a group's decayed scores against 64 tokens: [part][32 tokens before][16 tokens][lane][16 bytes]
constexpr int kFixedOutLds = 3 * FixedTile::bytes + 2 * kFixedScores;
__global__ __launch_bounds__(512) void recur_fixed_out_kernel(nf_recurrence_args a, int len) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t tiles[];
  const int h = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, lq = lane >> 4;
  const ChunkSpan ch = find_chunk(a, blockIdx.x, len);
  if (ch.n == 0) return;
  const int group = wave >> 2, w4 = wave & 3;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)tiles;
  uint8_t* qt = tiles;
  const uint8_t *kt = tiles + FixedTile::bytes, *vt = tiles + 2 * FixedTile::bytes;
  uint8_t* scores = tiles + 3 * FixedTile::bytes + group * kFixedScores;
  FixedTile::load((const uint16_t*)a.q + (size_t)ch.row0 * a.q_ld + h * kFixedDim, a.q_ld, ch.n, lds0, wave, lane);
  FixedTile::load((const uint16_t*)a.k + (size_t)ch.row0 * a.k_ld + h * kFixedDim, a.k_ld, ch.n, lds0 + FixedTile::bytes, wave, lane);
  FixedTile::load((const uint16_t*)a.v + (size_t)ch.row0 * a.v_ld + h * kFixedDim, a.v_ld, ch.n, lds0 + 2 * FixedTile::bytes, wave, lane);
  const float ld2 = a.log2_decay[h];
  const float* src = chunk_states(a, {kFixedDim, kFixedDim}, ch.slot, h);
  auto raw_at = [&](int c, int b, int e) { return *reinterpret_cast<const float4_t*>(src + ((size_t)((w4 * 2 + c) * 4 + b) * 64 + lane) * 8 + e * 4); };
  float4_t raw[2][4][2];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 2; ++e) raw[c][b][e] = raw_at(c, b, e);
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  const bool some = group * 64 < ch.n;  // this group has tokens

  // ---- the entering state's part: columns of v (rows of the MFMA's result) x tokens
  float4_t o[2][4];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int t = 0; t < 4; ++t) o[c][t] = float4_t{0.f, 0.f, 0.f, 0.f};
  if (some) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      Triple s[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const float x[8] = {raw[c][b][0][0], raw[c][b][0][1], raw[c][b][0][2], raw[c][b][0][3], raw[c][b][1][0], raw[c][b][1][1], raw[c][b][1][2], raw[c][b][1][3]};
        s[c] = triple_of(x);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int row = group * 64 + t * 16 + l16, at = b * 4 + (lq >> 1);
        const short8_t q8 = join(*reinterpret_cast<const short4_t*>(qt + FixedTile::chunk(row, at) + (lq & 1) * 8),
                                 *reinterpret_cast<const short4_t*>(qt + FixedTile::chunk(row, at + 2) + (lq & 1) * 8));
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
          for (int c = 0; c < 2; ++c) o[c][t] = mfma_bf16(s[c].part[p], q8, o[c][t]);
      }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float f = __builtin_amdgcn_exp2f((float)(group * 64 + t * 16 + l16 + 1) * ld2);
#pragma unroll
      for (int c = 0; c < 2; ++c) o[c][t] *= f;
    }
  }

  // ---- the chunk's own tokens, 64 at a time
  u32x4 q8[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) q8[b] = *reinterpret_cast<const u32x4*>(qt + FixedTile::chunk(group * 64 + w4 * 16 + l16, b * 4 + lq));
  for (int jb = 0; jb < 2; ++jb) {
    const bool mine = some && jb <= group, diagonal = jb == group;
    if (mine) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {  // 32 tokens
        if (diagonal && 2 * p > w4) continue;
        float x[8];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          float4_t s{0.f, 0.f, 0.f, 0.f};
          if (!diagonal || 2 * p + j <= w4)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
              const u32x4 k8 = *reinterpret_cast<const u32x4*>(kt + FixedTile::chunk(jb * 64 + (2 * p + j) * 16 + l16, b * 4 + lq));
              s = mfma_bf16(k8, q8[b], s);
            }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int back = (group - jb) * 64 + w4 * 16 + l16 - ((2 * p + j) * 16 + lq * 4 + r);  // tokens between the two
            x[j * 4 + r] = back >= 0 ? s[r] * (a.k_scale * __builtin_amdgcn_exp2f((float)back * ld2)) : 0.f;
          }
        }
        const Triple w = triple_of(x);
#pragma unroll
        for (int e = 0; e < 3; ++e) *reinterpret_cast<u32x4*>(scores + ((e * 2 + p) * 4 + w4) * 1024 + lane * 16) = w.part[e];
      }
    }
    __syncthreads();
    if (mine) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        short8_t v8[2], half[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const short4_t lo = FixedTile::column(vt, jb * 64 + p * 32 + lq * 4, w4 * 2 + c, l16), hi = FixedTile::column(vt, jb * 64 + p * 32 + 16 + lq * 4, w4 * 2 + c, l16);
          v8[c] = join(lo, hi);
          half[c] = join(lo, short4_t{0, 0, 0, 0});
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (diagonal && 2 * p > t) continue;
          const bool first = diagonal && 2 * p == t;  // the second 16 tokens come after these: their values stay out of it
#pragma unroll
          for (int e = 2; e >= 0; --e) {
            const u32x4 s8 = *reinterpret_cast<const u32x4*>(scores + ((e * 2 + p) * 4 + t) * 1024 + lane * 16);
#pragma unroll
            for (int c = 0; c < 2; ++c) o[c][t] = mfma_bf16(first ? half[c] : v8[c], s8, o[c][t]);
          }
        }
      }
    }
    if (jb == 0) __syncthreads();
  }
  if (some)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if (all_finite(o[c])) continue;
      const int col = (w4 * 2 + c) * 16;
      float4_t S[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) S[i] = raw_at(c, i >> 1, i & 1);
      fixed_steps(a, kt, vt, ld2, min(ch.n, group * 64 + 64), col, l16, lq, S, [&](int t0, const float4_t (&S)[8]) {
        if (t0 < group * 64) return;
        const int n = min(16, ch.n - t0);
        float4_t at{0.f, 0.f, 0.f, 0.f}, y{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float q = FixedTile::one(qt, t0 + l16, i * 16 + 4 * lq + r);
            at = __builtin_amdgcn_mfma_f32_16x16x4f32(FixedTile::one(kt, t0 + l16, i * 16 + 4 * lq + r) * a.k_scale, q, at, 0, 0, 0);
            y = __builtin_amdgcn_mfma_f32_16x16x4f32(S[i][r], q, y, 0, 0, 0);
          }
        y *= __builtin_amdgcn_exp2f((float)(l16 + 1) * ld2);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 4 * lq + r;
          const float x = j <= l16 && l16 < n ? at[r] * __builtin_amdgcn_exp2f((float)(l16 - j) * ld2) : 0.f;
          y = __builtin_amdgcn_mfma_f32_16x16x4f32(FixedTile::one(vt, t0 + j, col + l16), x, y, 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (t == (t0 >> 4 & 3)) mend(o[c][t], y);
      });
    }
  __syncthreads();

  // ---- through LDS, where q was: a token's 128 columns are written together
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float4_t y = o[c][t] * a.out_scale;
      const int row = group * 64 + t * 16 + l16, at = (w4 * 2 + c) * 2 + (lq >> 1);
      *reinterpret_cast<u32x2*>(qt + FixedTile::chunk(row, at) + (lq & 1) * 8) = u32x2{f32_to_bf16_pair(y[0], y[1]), f32_to_bf16_pair(y[2], y[3])};
    }
  __syncthreads();
  uint16_t* dst = (uint16_t*)a.out + (size_t)ch.row0 * a.out_ld + a.out_col + h * kFixedDim;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = i * 32 + (threadIdx.x >> 4), at = threadIdx.x & 15;
    if (row < ch.n) *reinterpret_cast<u32x4*>(dst + (size_t)row * a.out_ld + at * 8) = *reinterpret_cast<const u32x4*>(qt + FixedTile::chunk(row, at));
  }
}

}  // namespace nf
