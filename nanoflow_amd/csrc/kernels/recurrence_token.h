#pragma once
// Chunks of prompts under decays of every token and key channel: bf16 q, k, v and gate, heads of 64 x 64.  (included by layer_recurrence.hip)
//
// What bounded the general form was a chain of steps of 16 tokens, each with six barriers, and four wavefronts that all worked out the same scores.  Here
// a chunk of 64 tokens is taken at once, a wavefront to each block of 16:
//     o_i = (q_i 2^(L before i)) S + sum over j < i of (q_i . k_j 2^(L from j + 1 to before i)) v_j + (q_i . u k_i) v_i
// L, the sums of log2 decays, are scans over the lanes of a wavefront.  Within a block the scores are products of q 2^(L before i) and k 2^-(L through j), both from the
// block's start, or, where some channel's L is below -100, worked out one by one.  Between blocks no factor is above 1: k has decayed to the end of its own block,
// q from the start of its own, and the blocks between the two multiply q.  Scores and the state's part are MFMAs in fp32; the values are exact in bf16, so scores and
// decayed keys are taken apart into three bf16 numbers each (recurrence_fixed.h) where they meet them, and nothing is rounded that was not.  Sums that are not
// finite are taken again block after block in fp32, for the reasons given there: they are then what the general form's steps of 16 tokens leave.  (Its outputs take fewer
// where a channel decays below 2^-100 over 16; an infinity that it still has there is NaN in its states from the next chunk on.  The
// figures below are without the check, 20 vector instructions a wavefront.)
// 2019 tokens of 32 heads in two requests (us, general form -> this): chunk states 15.2 -> 11.3, scan 8.4 (bytes), outputs 35.8 -> 23.5; the states' error against
// 64 bits 7.3e-8 -> 6.2e-8.  The outputs are bound by what their wavefronts issue (some 1250 vector instructions for 16 tokens, and 92 to 152 matrix ones, 122 on average), little of it side
// by side; the same on 8 wavefronts and chunks of 128 took 32: the last block has seven before it.

namespace nf {

constexpr int kTokenDim = 64, kBlocks = 4, kTokenChunk = 16 * kBlocks;
typedef uint32_t words4_t __attribute__((ext_vector_type(4)));

template <int kCtrl>
__device__ __forceinline__ float dpp_or_zero(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xf, 0xf, true));
}
// Within 16 lanes: the value n lanes before (up) or after (down), zero past the end.
template <int n>
__device__ __forceinline__ float lanes_up(float x) { return dpp_or_zero<0x110 + n>(x); }
template <int n>
__device__ __forceinline__ float lanes_down(float x) { return dpp_or_zero<0x100 + n>(x); }
// token_log2_decay of the sum, limited to what matters: 2^y times the exponential of what y, z log2 e rounded, leaves out.
__device__ __forceinline__ float log2_decay_of(float z, float w0) {
  const float x = fmaxf(fminf(z + w0, 64.f), -128.f), y = x * 1.44269504088896340736f;  // what is no number: the largest decay
  const float rest = __builtin_fmaf(x, 1.9259629911266175e-8f, __builtin_fmaf(x, 1.44269502162933349609f, -y)), e = __builtin_amdgcn_exp2f(y);
  return fmaxf(-1.44269504088896340736f * __builtin_fmaf(e, rest * 0.69314718055994530942f, e), -126.f);
}

// Rows of 64 bf16 in LDS, eight pieces of 16 bytes; those of every second pair of rows are swapped, so that a transposing read of four rows takes each bank
// once.
struct TokenTile {
  static __device__ __forceinline__ uint32_t piece(int row, int c) { return (uint32_t)(row * 128 + ((c ^ ((row >> 1) & 1)) << 4)); }
  // Rows [0, n) of a head, `ld` elements apart, by four wavefronts, eight rows an instruction; the others as zeros.
  static __device__ __forceinline__ void load(const void* src, int ld, int n, uint32_t lds, int wave, int lane) {
    const rsrc_t r = make_rsrc(src, ((size_t)(n - 1) * ld + kTokenDim) * 2);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = (i * kBlocks + wave) * 8 + (lane >> 3);
      const uint32_t off = (uint32_t)row * (uint32_t)ld * 2u + (uint32_t)(((lane & 7) ^ ((row >> 1) & 1)) << 4);
      load16_to_lds(r, row < n ? off : kOob, __builtin_amdgcn_readfirstlane(lds + (i * kBlocks + wave) * 1024));
    }
  }
  // Tokens first .. first + 3 of the lane's column: lane i16 has column 16 u + i16, or (spread) 16 (i16 / 4) + 4 u + i16 % 4, by which a wavefront's
  // results give every lane 16 columns beside each other.
  static __device__ __forceinline__ short4_t column(const uint8_t* tile, int first, int u, int i16) {
    return lds_read_tr16(tile + piece(first + (i16 >> 2), 2 * u + ((i16 & 3) >> 1)) + (i16 & 1) * 8);
  }
  static __device__ __forceinline__ int spread_column(int u, int i16) { return 16 * (i16 >> 2) + 4 * u + (i16 & 3); }
  static __device__ __forceinline__ float one(const uint8_t* tile, int row, int col) {
    return bf16_bits_to_f32(*reinterpret_cast<const uint16_t*>(tile + piece(row, col >> 3) + (col & 7) * 2));
  }
  static __device__ __forceinline__ short4_t spread(const uint8_t* tile, int first, int u, int i16) {
    return lds_read_tr16(tile + piece(first + (i16 >> 2), 2 * (i16 & 3) + (u >> 1)) + (u & 1) * 8);
  }
};

// A chunk's state lies as the outputs' MFMAs take it: [4 columns in 16][4 rows in 16][lane][4], lane (l16, g) with column 16 (l16 / 4) + 4 vt + l16 % 4 and rows
// 16 g + 4 kt .. + 3.  Column and first of the four rows of the float4 at index f4:
__device__ __forceinline__ void token_place(int f4, int* k, int* c) {
  const int lane = f4 & 63, kt = (f4 >> 6) & 3, vt = f4 >> 8;
  *k = (lane >> 4) * 16 + kt * 4;
  *c = ((lane & 15) >> 2) * 16 + vt * 4 + (lane & 3);
}

// What a chunk adds to the state, and the factors of the entering one.  A wavefront has 16 rows of k, all columns of v.
__global__ __launch_bounds__(kTokenChunk * 4, 4) void recur_token_state_kernel(nf_recurrence_args a, int max_chunks) {
  __shared__ __attribute__((aligned(1024))) uint8_t tiles[2 * kBlocks * 2048];
  const int h = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, g = lane >> 4;
  const ChunkSpan ch = find_chunk(a, blockIdx.x, kTokenChunk);
  if (ch.n == 0) return;
  const int channel = wave * 16 + l16;
  float own[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) own[i] = a.z[(size_t)(ch.row0 + min(g * 16 + i, ch.n - 1)) * a.z_ld + h * kTokenDim + channel];
  const float w0 = a.w0[h * kTokenDim + channel];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)tiles;
  const uint8_t *kt = tiles, *vt = tiles + kBlocks * 2048;
  TokenTile::load((const uint16_t*)a.k + (size_t)ch.row0 * a.k_ld + h * kTokenDim, a.k_ld, ch.n, lds0, wave, lane);
  TokenTile::load((const uint16_t*)a.v + (size_t)ch.row0 * a.v_ld + h * kTokenDim, a.v_ld, ch.n, lds0 + kBlocks * 2048, wave, lane);
  for (int s = 1; s < a.z_shares; ++s)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      own[i] += a.z[((size_t)s * a.total_rows + ch.row0 + min(g * 16 + i, ch.n - 1)) * a.z_ld + h * kTokenDim + channel];
  // own becomes the decay of the lane's later tokens, sum that of all of them
  float sum = 0.f;
#pragma unroll
  for (int i = 15; i >= 0; --i) {
    const float l = log2_decay_of(own[i], w0) * (g * 16 + i < ch.n ? 1.f : 0.f);  // no branch around the exponential
    own[i] = sum;
    sum += l;
  }
  const float beside = __shfl_xor(sum, 16, 64), pair = (g & 1) ? beside + sum : sum + beside, other = __shfl_xor(pair, 32, 64);
  const float after = ((g & 1) ? 0.f : beside) + (g < 2 ? other : 0.f);
  const RecurrenceDims pd{kTokenDim, kTokenDim};
  if (g == 0) chunk_factors(a, pd, max_chunks, ch.slot, h)[channel] = exp2f(pair + other);
  float4_t S[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) S[c] = float4_t{0.f, 0.f, 0.f, 0.f};
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  Triple w[2];
  short8_t v8[2][4];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int first = g * 16 + s * 8;
    const short8_t k8 = join(TokenTile::column(kt, first, wave, l16), TokenTile::column(kt, first + 4, wave, l16));
    float k[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) k[e] = bf16_bits_to_f32((uint16_t)k8[e]) * __builtin_amdgcn_exp2f(own[s * 8 + e] + after);
    w[s] = triple_of(k);
#pragma unroll
    for (int c = 0; c < 4; ++c) v8[s][c] = join(TokenTile::spread(vt, first, c, l16), TokenTile::spread(vt, first + 4, c, l16));
  }
#pragma unroll
  for (int p = 2; p >= 0; --p)  // the small parts of all tokens first: fewer roundings of a large sum
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int c = 0; c < 4; ++c) S[c] = mfma_bf16(w[s].part[p], v8[s][c], S[c]);
  if (!all_finite(S)) {
    // Token after token, its decay worked out again: what is kept in registers for this would cost every launch a workgroup a CU.
    float4_t again[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) again[c] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int blk = 0; blk < kBlocks; ++blk) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float keep = __builtin_amdgcn_exp2f(__shfl(sum, blk * 16 + 4 * g + r, 64));
#pragma unroll
        for (int c = 0; c < 4; ++c) again[c][r] *= keep;
      }
      float later = 0.f;
#pragma unroll 1
      for (int i = 15; i >= 0; --i) {  // the lanes of a group have its block's tokens
        const int t = g * 16 + i;
        const size_t row = ch.row0 + min(t, ch.n - 1);
        float z = a.z[row * a.z_ld + h * kTokenDim + channel];
        for (int s = 1; s < a.z_shares; ++s) z += a.z[((size_t)s * a.total_rows + row) * a.z_ld + h * kTokenDim + channel];
        const float k = TokenTile::one(kt, t, channel) * __builtin_amdgcn_exp2f(later);
#pragma unroll
        for (int c = 0; c < 4; ++c)
          again[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(g == blk ? k : 0.f, g == blk ? TokenTile::one(vt, t, TokenTile::spread_column(c, l16)) : 0.f, again[c], 0, 0, 0);
        later += t < ch.n ? log2_decay_of(z, a.w0[h * kTokenDim + channel]) : 0.f;
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) mend(S[c], again[c]);
  }
  float* dst = chunk_states(a, pd, ch.slot, h);
#pragma unroll
  for (int c = 0; c < 4; ++c) *reinterpret_cast<float4_t*>(dst + ((size_t)(c * 4 + g) * 64 + wave * 16 + l16) * 4) = S[c];
}

// A chunk's outputs from the state that enters it.
struct TokenOutLds {
  static constexpr int state = kBlocks * 2048, keys = state + kTokenDim * kTokenDim * 4, totals = keys + (kBlocks - 1) * 4096, bytes = totals + kBlocks * 256;
};
// Three workgroups a CU leave registers for everything; of four, with two registers spilled, the launch took 24.8 us for 24.1.
__global__ __launch_bounds__(kTokenChunk * 4, 3) void recur_token_out_kernel(nf_recurrence_args a) {
  using L = TokenOutLds;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[L::bytes];
  const int h = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, g = lane >> 4;
  const ChunkSpan ch = find_chunk(a, blockIdx.x, kTokenChunk);
  if (ch.n == 0) return;
  // later blocks have more to do: not on the same SIMD in every workgroup of a CU
  const int blk = (wave + (int)blockIdx.x + (int)blockIdx.y) & (kBlocks - 1), t = blk * 16 + l16;
  const bool live = t < ch.n;
  const size_t row = (size_t)ch.row0 + (live ? t : ch.n - 1);
  const int col = h * kTokenDim + g * 16;  // a lane's 16 channels, and columns of v
  float lw[16];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const float4_t z = *reinterpret_cast<const float4_t*>(a.z + row * a.z_ld + col + 4 * c);
#pragma unroll
    for (int r = 0; r < 4; ++r) lw[4 * c + r] = z[r];
  }
  float4_t w0[4], u[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    w0[c] = *reinterpret_cast<const float4_t*>(a.w0 + col + 4 * c);
    u[c] = *reinterpret_cast<const float4_t*>(a.u + col + 4 * c);
  }
  words4_t k8[2], q8[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    k8[c] = *reinterpret_cast<const words4_t*>((const uint16_t*)a.k + row * a.k_ld + col + 8 * c);
    q8[c] = *reinterpret_cast<const words4_t*>((const uint16_t*)a.q + row * a.q_ld + col + 8 * c);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  TokenTile::load((const uint16_t*)a.v + (size_t)ch.row0 * a.v_ld + h * kTokenDim, a.v_ld, ch.n, lds0, wave, lane);
  const rsrc_t state = make_rsrc(chunk_states(a, {kTokenDim, kTokenDim}, ch.slot, h), kTokenDim * kTokenDim * 4);
#pragma unroll
  for (int i = 0; i < 16 / kBlocks; ++i) {
    const int at = (i * kBlocks + wave) * 1024;
    load16_to_lds(state, (uint32_t)(at + lane * 16), __builtin_amdgcn_readfirstlane(lds0 + L::state + at));
  }
  for (int s = 1; s < a.z_shares; ++s)
#pragma unroll
    for (int c = 0; c < 4; ++c)
    {
      const float4_t more = *reinterpret_cast<const float4_t*>(a.z + ((size_t)s * a.total_rows + row) * a.z_ld + col + 4 * c);
#pragma unroll
      for (int r = 0; r < 4; ++r) lw[4 * c + r] += more[r];
    }

  // ---- decays, and the block's own scores: rows j = 4 g + r, column i = l16
  float q[16];
  float4_t own{0.f, 0.f, 0.f, 0.f};
  {
    float k[16], through[16], bonus = 0.f;
    float4_t total[4], kh[4];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        k8[c][e] = live ? k8[c][e] : 0u;
        q8[c][e] = live ? q8[c][e] : 0u;
      }
    const float one = live ? 1.f : 0.f;
    bool low = false;
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const uint32_t kw = k8[c >> 3][(c >> 1) & 3], qw = q8[c >> 3][(c >> 1) & 3];
      k[c] = __uint_as_float((c & 1) ? kw & 0xffff0000u : kw << 16);
      q[c] = __uint_as_float((c & 1) ? qw & 0xffff0000u : qw << 16);
      lw[c] = log2_decay_of(lw[c], w0[c >> 2][c & 3]) * one;  // no branch around the exponential
      bonus += q[c] * k[c] * u[c >> 2][c & 3];
      float to = lw[c];
      to += lanes_up<1>(to);
      to += lanes_up<2>(to);
      to += lanes_up<4>(to);
      to += lanes_up<8>(to);
      through[c] = to;
      low |= to < kMinStepLog2;
    }
    bonus = sum_over_near_lane_groups(bonus);
    if (blk + 1 < kBlocks) {
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        float from = lw[c];  // a sum of later tokens only: no difference of large sums
        from += lanes_down<1>(from);
        from += lanes_down<2>(from);
        from += lanes_down<4>(from);
        from += lanes_down<8>(from);
        kh[c >> 2][c & 3] = k[c] * __builtin_amdgcn_exp2f(lanes_down<1>(from));
        total[c >> 2][c & 3] = from;  // the block's, in its first lane
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        *reinterpret_cast<float4_t*>(lds + L::keys + (blk * 4 + c) * 1024 + lane * 16) = kh[c];
        if (l16 == 0) *reinterpret_cast<float4_t*>(lds + L::totals + blk * 256 + g * 64 + c * 16) = total[c];
      }
    }
    if (__any(low)) {
      float between[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) between[c] = 0.f;
#pragma unroll 1
      for (int d = 1; d < 16; ++d) {
        const int from = (lane & 48) | ((l16 - d) & 15);
        float s = 0.f;
#pragma unroll
        for (int c = 0; c < 16; ++c) {
          s += q[c] * __builtin_amdgcn_exp2f(between[c]) * __shfl(k[c], from, 64);
          const float l = __shfl(lw[c], from, 64);
          between[c] += d <= l16 ? l : 0.f;
        }
        s = sum_over_near_lane_groups(s);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (4 * g + r == l16 - d) own[r] = s;
      }
#pragma unroll
      for (int c = 0; c < 16; ++c) q[c] *= __builtin_amdgcn_exp2f(between[c]);
    } else {
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        q[c] *= __builtin_amdgcn_exp2f(lanes_up<1>(through[c]));
        own = __builtin_amdgcn_mfma_f32_16x16x4f32(k[c] * __builtin_amdgcn_exp2f(-through[c]), q[c], own, 0, 0, 0);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) own[r] = 4 * g + r < l16 ? own[r] : 4 * g + r == l16 ? bonus : 0.f;
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  if (blk * 16 >= ch.n) return;
  words4_t gate[2];
#pragma unroll
  for (int c = 0; c < 2; ++c)
    gate[c] = a.g ? *reinterpret_cast<const words4_t*>((const uint16_t*)a.g + row * a.g_ld + col + 8 * c) : words4_t{0, 0, 0, 0};

  // ---- earlier blocks, the nearest first: columns of v (rows of the results) x tokens
  float4_t o[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) o[c] = float4_t{0.f, 0.f, 0.f, 0.f};
  float4_t ahead[4];  // decays of the blocks since
#pragma unroll
  for (int c = 0; c < 4; ++c) ahead[c] = float4_t{0.f, 0.f, 0.f, 0.f};
  float now[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) now[c] = q[c];
  auto scores_of = [&](int b) {
    float4_t s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float4_t k = *reinterpret_cast<const float4_t*>(lds + L::keys + (b * 4 + c) * 1024 + lane * 16);
#pragma unroll
      for (int r = 0; r < 4; ++r) s = __builtin_amdgcn_mfma_f32_16x16x4f32(k[r], now[4 * c + r], s, 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      ahead[c] += *reinterpret_cast<const float4_t*>(lds + L::totals + b * 256 + g * 64 + c * 16);
#pragma unroll
      for (int r = 0; r < 4; ++r) now[4 * c + r] = q[4 * c + r] * __builtin_amdgcn_exp2f(ahead[c][r]);
    }
    return s;
  };
#pragma unroll 1
  for (int p = blk >> 1; p >= 0; --p) {
    const bool first = blk == 2 * p;  // the second 16 tokens come after these: their values stay out of it
    float4_t s1{0.f, 0.f, 0.f, 0.f};
    if (blk == 2 * p + 1) s1 = own;
    else if (!first) s1 = scores_of(2 * p + 1);
    const float4_t s0 = first ? own : scores_of(2 * p);
    const float x[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
    const Triple w = triple_of(x);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const short4_t lo = TokenTile::spread(lds, p * 32 + g * 4, c, l16);
      short4_t hi = TokenTile::spread(lds, p * 32 + 16 + g * 4, c, l16);
      if (first) hi = short4_t{0, 0, 0, 0};
      const short8_t v8 = join(lo, hi);
#pragma unroll
      for (int e = 2; e >= 0; --e) o[c] = mfma_bf16(v8, w.part[e], o[c]);
    }
  }

  // ---- the entering state
  float4_t weight[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) weight[c] = a.norm_weight ? *reinterpret_cast<const float4_t*>(a.norm_weight + col + 4 * c) : float4_t{1.f, 1.f, 1.f, 1.f};
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    float4_t s[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) s[c] = *reinterpret_cast<const float4_t*>(lds + L::state + (c * 4 + b) * 1024 + lane * 16);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(s[c][r], now[4 * b + r], o[c], 0, 0, 0);
  }

  if (!all_finite(o)) {
#pragma unroll 1
    for (int c = 0; c < 4; ++c) {
      const int col_v = TokenTile::spread_column(c, l16);
      float4_t s[4], y{0.f, 0.f, 0.f, 0.f};  // s: rows 16 g + 4 kt + r of k, column col_v; y: columns 16 g + 4 c + r of the token l16
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) s[kt] = *reinterpret_cast<const float4_t*>(lds + L::state + (c * 4 + kt) * 1024 + lane * 16);
#pragma unroll 1
      for (int b = 0; b < blk; ++b)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
          const float4_t total = *reinterpret_cast<const float4_t*>(lds + L::totals + b * 256 + g * 64 + kt * 16);
#pragma unroll
          for (int r = 0; r < 4; ++r) s[kt][r] *= __builtin_amdgcn_exp2f(total[r]);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float k = *reinterpret_cast<const float*>(lds + L::keys + (b * 4 + kt) * 1024 + ((l16 >> 2) * 16 + 4 * g + r) * 16 + (l16 & 3) * 4);
            s[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(k, TokenTile::one(lds, b * 16 + 4 * g + r, col_v), s[kt], 0, 0, 0);
          }
        }
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) y = __builtin_amdgcn_mfma_f32_16x16x4f32(s[kt][r], q[4 * kt + r], y, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) y = __builtin_amdgcn_mfma_f32_16x16x4f32(TokenTile::one(lds, blk * 16 + 4 * g + r, col_v), own[r], y, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i == c) mend(o[i], y);
    }
  }

  // ---- norm over the head's columns, gate
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) ss += o[c][r] * o[c][r];
  ss = sum_over_near_lane_groups(ss);
  const float inv = a.g ? a.out_scale / sqrtf(ss / (float)kTokenDim + a.eps) : a.out_scale;
  float4_t y[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) y[c] = o[c] * inv * weight[c];
  if (a.g) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float4_t g4 = Act<bf16_t>::widen4(u32x2{gate[c >> 1][(c & 1) * 2], gate[c >> 1][(c & 1) * 2 + 1]});
#pragma unroll
      for (int r = 0; r < 4; ++r) y[c][r] *= silu<bf16_t>(g4[r]);
    }
  }
  words4_t y8[2];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    y8[c >> 1][(c & 1) * 2] = f32_to_bf16_pair(y[c][0], y[c][1]);
    y8[c >> 1][(c & 1) * 2 + 1] = f32_to_bf16_pair(y[c][2], y[c][3]);
  }
  if (!live) return;
  words4_t* dst = reinterpret_cast<words4_t*>((uint16_t*)a.out + row * a.out_ld + a.out_col + col);
  dst[0] = y8[0];
  dst[1] = y8[1];
}

}  // namespace nf
