#pragma once
// GEMMs of at most 64 rows: the weights are read once and that is the time (a product of 16 x 4096 x 4096 takes 0.2 us of
// the matrix cores and 4.8 us of HBM), so this kernel is a weight stream with MFMAs beside it.
//
// A workgroup owns NT tiles of 16 weight rows (output columns) and AR rows of A over the WHOLE of K; its wavefronts share K
// out in units of 64, and their sums meet in LDS at the end, where the epilogue follows: no fp32 shares in memory, no second
// launch.  Every wavefront streams its own units through a ring of its own in LDS (S units, `buffer_load ... lds`), waits for
// nobody until the end and refills a slot as soon as its fragments are in registers.  An instruction fetches 8 rows of 128
// bytes: whole lines, with the non-temporal hint, reach 6.3 - 7.0 TB/s where fragments loaded straight into registers
// (16 rows of 64 bytes) stop at 5.0 (the gate/up pair of 1 x 14336 x 4096: 37 us against 47).  Weights may be [K][N] as well
// (kBCol false): rows of NT * 32 bytes per k, read back through the transposing LDS read.  That stream is slower than tiles
// which are split over K where those can be (16 x 4096 x 14336: 50 us against 26) and runs where they cannot.
//
// The sum of an output element is taken in the same order whatever the tile: eight classes of units (unit mod 8), each in the
// order of k, neighbouring classes added first, then the pairs, then those.  A row's result does not depend on how many rows come
// with it, nor on the weights' layout: the tiles for [K][N] weights take their slabs in this order (kClasses in gemm_impl.h).
//
// Measured against the tiles and the split over K that it replaces (us, one launch after the other on streamed weights):
//   rows x N x K              before   here         rows x N x K              before   here
//   1 x 4096 x 4096             14.3    7.4         64 x 4096 x 4096            15.5   12.0
//   1 x 6144 x 4096             14.5    9.9         64 x 6144 x 4096            17.8   17.0
//   1 x 4096 x 14336            25.1   19.6         64 x 2048 x 2048            11.1    6.2
//   1 x 14336 x 4096 (pair)     47.4   37.2         64 x 14336 x 4096           54.4   27.9
//   16 x 14336 x 4096 (pair)    48.0   38.7         64 x 14336 x 4096 (pair)    61.5   50.4
//   16 x 128256 x 4096         173    153.5         16 x 14336 x 4096           49.1   21.1
// (included by gemm_impl.h, between its kernels and its entry functions)

namespace nf {

constexpr int kRowsMax = 64;       // rows of A
// e4m3 operands: a unit is 128 k, a lane's two chunks of it go through one MFMA, and the sums are multiplied by a scale per row of A
// and one per output column.
struct RowsF8 {
  static __device__ __forceinline__ float widen(uint32_t bits) { return h2f_bits(bits); }  // C and D are fp16
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) { return pack_f16x2(lo, hi); }
  static __device__ __forceinline__ float rounded(float x) { return __half2float(__float2half_rn(x)); }
  static __device__ __forceinline__ float4_t finish(float4_t v) { return v; }
};
struct RowsScales {
  const float *a = nullptr, *b = nullptr, *b1 = nullptr;
};
constexpr int kRowsClasses = 8;    // K is summed in this many interleaved classes of units

template <int AR, int NT, int NW, int NB, int S>
struct RowsSmem {
  static constexpr int w_bytes = NB * NT * 2048, slot = w_bytes + AR * 128, ring = NW * S * slot;
  static constexpr int tiles = NB * ((AR + 15) / 16) * NT;                // accumulator tiles of a wavefront
  static constexpr int pass = (tiles < 8 ? tiles : 8) / NB;               // output tiles whose sums meet at a time
  static constexpr int bytes = ring > kRowsClasses * pass * NB * 1024 ? ring : kRowsClasses * pass * NB * 1024;
  static_assert(bytes <= 160 * 1024 && NB * ((AR + 15) / 16) * NT % (pass * NB) == 0, "rows tile");
};

// The tile of AR rows (8, 16, 32, 48 or 64) from row m0 and NT * 16 output columns from n0.  NB: 2 = two weight matrices.  a_row(m): byte
// offset of row m in A, kOob past the last one (nothing is fetched then).  store(m, n, v): what becomes of the sums v[NB] of row
// m, columns n .. n + 3.
template <class E, int AR, int NT, int NW, int NB, int S, bool kBCol, class ARow, class Store>
__device__ __forceinline__ void rows_tile(const rsrc_t a_rsrc, const rsrc_t (&b_rsrc)[NB], const uint32_t row_bytes, const int N,
                                          const int m0, const int n0, ARow&& a_row, Store&& store) {
  using SM = RowsSmem<AR, NT, NW, NB, S>;
  constexpr int MT = (AR + 15) / 16, PAR = kRowsClasses / NW;  // classes per wavefront
  constexpr bool kF8 = std::is_same_v<E, RowsF8>;
  static_assert(NW * PAR == kRowsClasses && (S % PAR == 0 || S == 1), "classes take turns in the ring's slots");
  constexpr int R = S > PAR ? S : PAR;  // units of a round
  static_assert(!kF8 || kBCol, "e4m3 weights are k-contiguous");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, lq = lane >> 4;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const uint32_t mine_lds = __builtin_amdgcn_readfirstlane(lds0 + wave * (S * SM::slot));
  const uint8_t* mine = smem + wave * (S * SM::slot);
  const int units = (int)((row_bytes + 127) / 128);

  // Rows of 128 bytes (A, [N][K] weights): lane -> row lane / 8 of the instruction's 8, position lane % 8, which holds chunk
  // position ^ ((row >> 1) & 7) of the 16-row tile (an odd instruction has its rows 8..15): fragment reads without conflicts.
  const int r8 = lane >> 3;
  const uint32_t kc[2] = {(uint32_t)((lane & 7) ^ (r8 >> 1)) * 16u, (uint32_t)((lane & 7) ^ ((r8 >> 1) | 4)) * 16u};
  uint32_t a_off[AR / 8], b_off[NT * 2];
  // [K][N] weights: 64 k rows of NT * 32 bytes, as they lie; columns from N on belong to the next row and are not stored
  constexpr int CPR = NT * 2;  // 16-byte chunks of such a row
#pragma unroll
  for (int j = 0; j < NT * 2; ++j) {
    if constexpr (kBCol) b_off[j] = (uint32_t)(n0 + j * 8 + r8) * row_bytes + kc[j & 1];
    else b_off[j] = ((uint32_t)((j * 64 + lane) / CPR) * (uint32_t)N + n0 + (j * 64 + lane) % CPR * 8) * 2u;
  }
  // Weight rows past the last one lie past the end of the buffer and read as zero.
  auto issue_b = [&](auto s_c, int u) {
    constexpr int s = decltype(s_c)::value;
    const uint32_t kb = (uint32_t)u * 128u;
    const bool in = u < units;
    const bool ok[2] = {in && kb + kc[0] < row_bytes, in && kb + kc[1] < row_bytes};
    static_for<NB>([&](auto b_c) {
      static_for<NT * 2>([&](auto j_c) {
        constexpr int b = decltype(b_c)::value, j = decltype(j_c)::value, dst = s * SM::slot + (b * NT * 2 + j) * 1024;
        if constexpr (kBCol) load16_to_lds<dst, true>(b_rsrc[b], ok[j & 1] ? b_off[j] + kb : kOob, mine_lds);
        else load16_to_lds<dst, (NT >= 4)>(b_rsrc[b], in ? b_off[j] + (uint32_t)u * 64u * (uint32_t)N * 2u : kOob, mine_lds);
      });
    });
  };
  auto issue_a = [&](auto s_c, int u) {
    constexpr int s = decltype(s_c)::value;
    const uint32_t kb = (uint32_t)u * 128u;
    const bool in = u < units;
    const bool ok[2] = {in && kb + kc[0] < row_bytes, in && kb + kc[1] < row_bytes};
    static_for<AR / 8>([&](auto i_c) {
      constexpr int i = decltype(i_c)::value;
      load16_to_lds<s * SM::slot + SM::w_bytes + i * 1024>(a_rsrc, ok[i & 1] && a_off[i] != kOob ? a_off[i] + kc[i & 1] + kb : kOob, mine_lds);
    });
  };

  float4_t acc[PAR][NB][MT][NT];
#pragma unroll
  for (int p = 0; p < PAR; ++p)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[p][b][i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  const uint32_t f_row = (uint32_t)l16 * 128u, f_swz = (l16 >> 1) & 7;
  // eight rows of A stand for sixteen: the upper half of the products is not stored
  const uint32_t af_row = AR == 8 ? (uint32_t)(l16 & 7) * 128u : f_row, a_swz = AR == 8 ? (l16 & 7) >> 1 : f_swz;
  auto consume = [&](auto s_c, auto p_c) {
    constexpr int s = decltype(s_c)::value, P = decltype(p_c)::value;
    const uint8_t* slot = mine + s * SM::slot;
    half8_t w[2][NB][NT], a[2][MT];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          if constexpr (kBCol) {
            w[h][b][j] = *reinterpret_cast<const half8_t*>(slot + (b * NT + j) * 2048 + f_row + (((h * 4 + lq) ^ f_swz) << 4));
          } else {  // k rows h * 32 + lq * 8 .. + 7, columns j * 16 .. + 15
            const uint8_t* p = slot + b * NT * 2048 + (h * 32 + lq * 8 + (l16 >> 2)) * (NT * 32) + j * 32 + (l16 & 3) * 8;
            typedef short short8_t __attribute__((ext_vector_type(8)));
            const short4_t lo = lds_read_tr16(p), hi = lds_read_tr16(p + 4 * NT * 32);
            w[h][b][j] = __builtin_bit_cast(half8_t, (short8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
          }
        }
#pragma unroll
      for (int i = 0; i < MT; ++i)
        a[h][i] = *reinterpret_cast<const half8_t*>(slot + SM::w_bytes + i * 2048 + af_row + (((h * 4 + lq) ^ a_swz) << 4));
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the fragments are in registers, the slot may be refilled
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kF8) {
      typedef int v4i32 __attribute__((ext_vector_type(4)));
      typedef int v8i32 __attribute__((ext_vector_type(8)));
      auto both = [](half8_t lo, half8_t hi) {
        return (v8i32)__builtin_shufflevector(__builtin_bit_cast(v4i32, lo), __builtin_bit_cast(v4i32, hi), 0, 1, 2, 3, 4, 5, 6, 7);
      };
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int i = 0; i < MT; ++i)
            acc[P][b][i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(both(w[0][b][j], w[1][b][j]), both(a[0][i], a[1][i]),
                                                                                    acc[P][b][i][j], 0, 0, 0, 0, 0, 0);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[P][b][i][j] = E::mfma16(w[h][b][j], a[h][i], acc[P][b][i][j]);
    }
  };
  // vmcnt(n): all but the n youngest loads of this wavefront have landed
  auto wait_but = [](auto n_c) {
    constexpr int n = decltype(n_c)::value;
    static_assert(n < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (n & 15) | ((n >> 4) << 14));
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int kA = AR / 8, kLoads = SM::slot / 1024;
  // The weights of the first S units are under way before the rows of A are looked up, which may take a load of its own.
  static_for<S>([&](auto s_c) { issue_b(s_c, wave + decltype(s_c)::value * NW); });
#pragma unroll
  for (int i = 0; i < kA; ++i) a_off[i] = a_row(m0 + i * 8 + r8);
  static_for<S>([&](auto s_c) { issue_a(s_c, wave + decltype(s_c)::value * NW); });
  int u = wave + S * NW;
  auto round = [&](auto first_c) {  // units past the last one read as zero
    static_for<R>([&](auto r_c) {
      constexpr int r = decltype(r_c)::value, s = r % S;
      wait_but(ic<decltype(first_c)::value && r < S ? (S - 1 - r) * kA + r * kLoads : (S - 1) * kLoads>{});  // the slot has landed
      consume(ic<s>{}, ic<r % PAR>{});
      issue_b(ic<s>{}, u);
      issue_a(ic<s>{}, u);
      u += NW;
    });
  };
  if (wave < units) round(ic<1>{});
  for (int done = wave + NW * R; done < units; done += NW * R) round(ic<0>{});
  __builtin_amdgcn_s_waitcnt(0x0070);
  __syncthreads();

  // The classes' sums, SM::pass output tiles at a time: [class][tile][matrix][lane].  Lane (l16, lq) of a tile has columns
  // lq * 4 .. + 3 of row l16; items are handed out along the rows.
  constexpr int TP = SM::pass;
  float4_t* red = reinterpret_cast<float4_t*>(smem);
  static_for<MT * NT / TP>([&](auto g_c) {
    constexpr int g = decltype(g_c)::value;
    if (g) __syncthreads();
    static_for<PAR * TP * NB>([&](auto q_c) {
      constexpr int q = decltype(q_c)::value, p = q / (TP * NB), t = q / NB % TP, b = q % NB, tt = g * TP + t;
      red[(((wave + p * NW) * TP + t) * NB + b) * 64 + lane] = acc[p][b][tt / NT][tt % NT];
    });
    __syncthreads();
    for (int it = threadIdx.x; it < TP * 64; it += NW * 64) {
      const int t = it >> 6, ln = (it & 3) * 16 + ((it >> 2) & 15), tt = g * TP + t;
      float4_t v[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        float4_t sum[kRowsClasses];
#pragma unroll
        for (int c = 0; c < kRowsClasses; ++c) sum[c] = red[((c * TP + t) * NB + b) * 64 + ln];
#pragma unroll
        for (int d = 1; d < kRowsClasses; d *= 2)
#pragma unroll
          for (int c = 0; c < kRowsClasses; c += 2 * d) sum[c] += sum[c + d];
        v[b] = sum[0];
      }
      const int row = tt / NT * 16 + (ln & 15), n = n0 + tt % NT * 16 + (ln >> 4) * 4;
      if (row < AR && n < N) store(m0 + row, n, v);
    }
  });
}

// kSums: D is float, sums as they are.  A, B, B1: elements of E's operand type.
template <class E, int AR, int NT, int NW, int NB, int S, bool kBCol, bool kSums>
__global__ __launch_bounds__(NW * 64) void gemm_rows_kernel(const void* __restrict__ A, const void* __restrict__ B,
                                                            const void* __restrict__ B1, const uint16_t* C, uint16_t* D, int M,
                                                            int N, int K, float alpha, float beta, int ldc, int tiles_m, int tiles_n,
                                                            RowsScales scales) {
  constexpr bool kF8 = std::is_same_v<E, RowsF8>;
  const int total = tiles_m * tiles_n, logical = xcd_order(blockIdx.x, total);
  if (logical >= total) return;
  const uint32_t row_bytes = (uint32_t)K * (kF8 ? 1u : 2u);  // of A and of [N][K] weights
  rsrc_t b_rsrc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) b_rsrc[b] = make_rsrc(b ? B1 : B, (size_t)N * row_bytes);
  // the m tiles of a weight panel side by side: the panel is fetched once
  rows_tile<E, AR, NT, NW, NB, S, kBCol>(
      make_rsrc(A, (size_t)M * row_bytes), b_rsrc, row_bytes, N, logical % tiles_m * AR, logical / tiles_m * (NT * 16),
      [&](int m) { return m < M ? (uint32_t)m * row_bytes : kOob; },
      [&](int m, int n, float4_t(&v)[NB]) {
        if (m >= M) return;
        if constexpr (kSums) {
          *reinterpret_cast<float4_t*>(reinterpret_cast<float*>(D) + (size_t)m * N + n) = v[0];
        } else {
          if constexpr (kF8) {
            const float row_scale = scales.a[m];
            v[0] = v[0] * (*reinterpret_cast<const float4_t*>(scales.b + n) * alpha) * row_scale;
            if constexpr (NB == 2) v[1] = v[1] * *reinterpret_cast<const float4_t*>(scales.b1 + n) * row_scale;
          }
          float4_t o;
          if constexpr (NB == 2) {
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = swiglu_rounded<E>(v[0][e], v[NB - 1][e]);
          } else {
            o = kF8 ? v[0] : v[0] * alpha;
            if (beta != 0.f) {
              const u32x2 c = *reinterpret_cast<const u32x2*>(C + (size_t)m * ldc + n);
              o[0] += beta * E::widen(c.x & 0xffffu);
              o[1] += beta * E::widen(c.x >> 16);
              o[2] += beta * E::widen(c.y & 0xffffu);
              o[3] += beta * E::widen(c.y >> 16);
            }
            o = E::finish(o);
          }
          *reinterpret_cast<u32x2*>(D + (size_t)m * N + n) = u32x2{E::pack2(o[0], o[1]), E::pack2(o[2], o[3])};
        }
      });
}

template <class E, int AR, int NT, int NW, int NB, int S, bool kBCol, bool kSums>
static int launch_rows(const void* A, const void* B, const void* B1, const uint16_t* C, uint16_t* D, int M, int N, int K,
                       float alpha, float beta, int ldc, hipStream_t stream, const RowsScales& scales = {}) {
  using SM = RowsSmem<AR, NT, NW, NB, S>;
  auto kern = gemm_rows_kernel<E, AR, NT, NW, NB, S, kBCol, kSums>;
  static bool attr_set = false;  // benign race: the call is idempotent
  if (!attr_set) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, SM::bytes);
    if (e != hipSuccess) {
      set_error("gemm: cannot reserve %d bytes of LDS: %s", SM::bytes, hipGetErrorString(e));
      return NF_ERR_RUNTIME;
    }
    attr_set = true;
  }
  const int tiles_m = (M + AR - 1) / AR, tiles_n = (N + NT * 16 - 1) / (NT * 16);
  kern<<<(tiles_m * tiles_n + 7) / 8 * 8, NW * 64, SM::bytes, stream>>>(A, B, B1, C, D, M, N, K, alpha, beta, ldc, tiles_m, tiles_n, scales);
  return check_launch("gemm (few rows) launch");
}

// Which launches run here: at most 64 rows against k-contiguous weights with K >= 1536 (three units a class; below, the plain tile
// is as good).  Every workgroup reads its rows of A over all of K, so from 17 rows on that traffic counts: a long
// contraction against a narrow N is better off split over K between workgroups (64 x 4096 x 14336: 26.4 us against 37.5;
// 64 x 8192 x 8192: even at 31), and from 33 rows on more workgroups than CUs re-read A once too often (64 x 128256 x 4096: 215
// us against 181 on 64 x 256 tiles).
static bool rows_pay(int M, int N, int K, int row_bytes = 0) {
  if (row_bytes == 0) row_bytes = K * 2;  // of 16-bit operands
  if (M <= 0 || M > kRowsMax || row_bytes < 3 * kRowsClasses * 128) return false;
  if (M <= 16) return true;
  if (row_bytes > 8192 && N < 8192) return false;
  return M <= 32 || (N + 63) / 64 <= cu_count();
}
// fp16 and bf16 launches that may come with either layout: from 9 rows on not against 33 to 44 columns a CU and K >= 4096, where [K][N]
// weights have no tiles in this order that are as fast (16 x 10240 x 8192: 42 us in 4 shares, 31.6 as splitk_plan_narrow says, 34.6 on
// 64 x 256; k-contiguous ones 36.2 here, 35.2 and 37.6).
static bool in_a_gap(int N, int K) { return N > 32 * cu_count() && N <= 44 * cu_count() && K >= 4096; }
static bool few_pay(int M, int N, int K) { return rows_pay(M, N, K) && (M <= 8 || !in_a_gap(N, K)); }

// With a workspace there is another choice: few columns against a long contraction are few workgroups, each with all of K to take in, and
// better off split (splitk_plan_narrow; 16 x 1024 x 14336 17.6 us here, 11.2 so, 16 x 2048 x 14336 19.6 and 15.6, one row of it 13.9 and
// 15.2, 8 x 512 x 14336 12.7 and 8.9, 16 x 1024 x 8192 9.5 and 8.7, 16 x 2048 x 8192 10.9 and 11.8; [K][N] weights 1 x 2048 x 14336 18.7
// and 15.7).
static bool narrow_and_deep(int M, int N, int K) { return M <= 16 && K >= 8192 && N <= (K > 8192 ? 8 : 4) * cu_count(); }

// The gate/up pair of 17 to 64 rows: a workgroup of 32 columns is one a CU, and its rows of A come with every one, so between 48 and 64 columns a CU two nearly full
// rounds of them lose to one round of twice the width, whose LDS holds a ring of one: 64 x 14336 x 4096 52 -> 46 us, 64 x 16384 x 4096 59 -> 52, 40 x
// 16384 x 4096 57 -> 51, 32 x 16384 x 4096 58 -> 55, e4m3 64 x 14336 x 4096 32 -> 29, 24 x 14336 x 4096 26 -> 24.  Below, the second round is
// short enough to cost less (64 x 8192 x 4096, which has none: 28 and 41; 40 x 11264 x 4096 44 and 46); above, both take as many bytes a
// round and the shorter ring shows (64 x 18432 x 4096 66 and 72), as it does on rows beyond 10 KB (17 x 15360 x 8192 92 and 104, e4m3 17 x 15360 x 16384
// 85 and 95).  Up to 32 rows, of 5 sizes against 9 widths and 6 depths: 0.86 to 1.01 of the time, but weight rows whole multiples of 4 KB apart, which
// few of the memory's channels hold at a time, 0.95 to 1.08 between 50 and 62 columns a CU (17 x 14336 x 4096 45 and 48; 0.80 to 0.90 at 64).  The sums keep their order.
static bool wide_pair(int M, int N, int row_bytes) {
  const int cus = cu_count();
  if (M <= 16 || N < 48 * cus || N > 64 * cus || row_bytes > 10240) return false;
  return M > 32 || row_bytes % 4096 != 0 || N <= 50 * cus || N > 62 * cus;
}

// The same for the gate/up pair of 16-bit or e4m3 (f8) operands.  Few columns against a long contraction, or workgroups that spill over
// into another round, lose to the tiles and their split over K: 64 x 512 x 14336 63 us against 20, 16 x 4096 x 14336 56 against 46, 64 x
// 10240 x 8192 86 against 73, e4m3 64 x 512 x 14336 29 against 15.  Both sides by what they take in: here a workgroup's rows of both weights and of A over the whole of K at
// 50 GB/s, round after round, or all weights at 6.4 TB/s; there 10 us (e4m3: 9) and the weights at 6.  Fitted to 132 and 531 launches
// of 1 to 64 rows, 64 to 28672 columns, K of 2048 to 14336, on 32 columns a workgroup, and within 5 % of the faster one except e4m3 against 16384 x 4096
// (35 us, 31); wide pairs, priced with 64, are the faster ones in 90 launches of 33 to 64 rows (64 x 12288 x 4096 60 -> 50, 48 x 13312 x 4096 65 -> 53, e4m3 64 x
// 13312 x 8192 64 -> 50; [K][N] weights the same with a workspace, 66 -> 50 without).
// More than 32 rows against more than 64 columns a CU, and e4m3 rows below 4 KB there from 17 rows on, are the tiles' (64 x 28672 x 8192 181 us
// against 168, e4m3 64 x 28672 x 3072 49 against 37).
static bool rows_pay_dual(int M, int N, int row_bytes, bool f8) {
  if (M <= 0 || M > kRowsMax || row_bytes < 3 * kRowsClasses * 128) return false;
  const int cus = cu_count(), cols = wide_pair(M, N, row_bytes) ? 64 : M <= 8 ? 16 : 32, ar = M <= 8 ? 8 : M <= 16 ? 16 : M <= 32 ? 32 : 64;
  const bool beyond = N > 64 * cus;
  if ((beyond && (M > 32 || (f8 && M > 16 && row_bytes < 4096))) || (row_bytes > 16384 && N < 16 * cus)) return false;
  if (!f8 && M > 8 && in_a_gap(N, row_bytes / 2)) return false;
  const int rounds = ((N + cols - 1) / cols + cus - 1) / cus;
  const double weights = 2.0 * N * row_bytes, intake = (double)rounds * (2 * cols + ar) * row_bytes;
  return std::max(weights / 6.4e6, intake / 50e3) * 1.1 + 1.0 + (f8 ? rounds : 0) < (f8 ? 9.0 : 10.0) + weights / 6e6;
}

// Rounds of workgroups times what one of them reads (16-row panels of weights and of A).
static int rows_cost(int N, int nt, int m_tiles, int a_panels) { return ((N + nt * 16 - 1) / (nt * 16) * m_tiles + cu_count() - 1) / cu_count() * (nt + a_panels); }

template <class E, bool kSums>
static int dispatch_rows(const void* A, const void* B, const uint16_t* C, uint16_t* D, int M, int N, int K, float alpha, float beta,
                         int ldc, hipStream_t s, const RowsScales& sc = {}) {
  // Short e4m3 rows against many columns want workgroups of 32, whatever the rounds say: 16 are over too soon (1 x 28672 x 4096 25.0 us, 21.9
  // so, 4 x 20480 x 6144 22.8 and 21.3; from 8 KB on the same in both), and 64 have few wavefronts a CU (17 x 28672 x 4096 25.7 and
  // 23.9, 17 x 57344 x 4096 47.5 and 40.7; but 32 x 28672 x 6144 34.1 and 36.5).
  const bool f8 = std::is_same_v<E, RowsF8>, brief = f8 && K < 8192 && N > 64 * cu_count();
  if (M <= 8)  // a tie goes to fewer, wider workgroups (1 x 6144 x 4096: 9.9 us against 11.2)
    return !brief && rows_cost(N, 1, 1, 0) < rows_cost(N, 2, 1, 0) ? launch_rows<E, 8, 1, 8, 1, 3, true, kSums>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s, sc)
                                                         : launch_rows<E, 8, 2, 8, 1, 2, true, kSums>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s, sc);
  if (M <= 16)
    return rows_cost(N, 1, 1, 1) < rows_cost(N, 2, 1, 1) ? launch_rows<E, 16, 1, 8, 1, 2, true, kSums>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s, sc)
                                                         : launch_rows<E, 16, 2, 4, 1, 2, true, kSums>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s, sc);
  const bool pairs = f8 && M <= 32 && K <= 4096 && N > 96 * cu_count();
  const int half = (M + 31) / 32;  // m tiles of 32 rows
  const int c1 = rows_cost(N, 1, half, 2), c2 = rows_cost(N, 2, half, 2);
  const int w2 = M <= 32 ? 1 << 30 : rows_cost(N, 2, 1, 4), w4 = rows_cost(N, 4, 1, M <= 32 ? 2 : 4);
  const int best = std::min(std::min(c1, c2), std::min(w2, w4));
  if (best == c1 && !pairs) return launch_rows<E, 32, 1, 8, 1, 2, true, kSums>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s, sc);
  if (best == c2 || pairs) return launch_rows<E, 32, 2, 4, 1, 2, true, kSums>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s, sc);
  if (best == w2) return launch_rows<E, 64, 2, 4, 1, 2, true, kSums>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s, sc);
  return M <= 32 ? launch_rows<E, 32, 4, 4, 1, 2, true, kSums>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s, sc)
                 : launch_rows<E, 64, 4, 4, 1, 2, true, kSums>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s, sc);
}

template <class E>
static int dispatch_rows_dual(const void* A, const void* Bg, const void* Bu, uint16_t* out, int M, int N, int K, hipStream_t s,
                              const RowsScales& sc = {}) {
  if (M <= 8) return launch_rows<E, 8, 1, 8, 2, 2, true, false>(A, Bg, Bu, nullptr, out, M, N, K, 1.f, 0.f, N, s, sc);
  if (M <= 16) return launch_rows<E, 16, 2, 4, 2, 2, true, false>(A, Bg, Bu, nullptr, out, M, N, K, 1.f, 0.f, N, s, sc);
  const bool wide = wide_pair(M, N, K * (std::is_same_v<E, RowsF8> ? 1 : 2));
  if (M <= 32)
    return wide ? launch_rows<E, 32, 4, 4, 2, 1, true, false>(A, Bg, Bu, nullptr, out, M, N, K, 1.f, 0.f, N, s, sc)
                : launch_rows<E, 32, 2, 4, 2, 2, true, false>(A, Bg, Bu, nullptr, out, M, N, K, 1.f, 0.f, N, s, sc);
  if (wide) return launch_rows<E, 64, 4, 4, 2, 1, true, false>(A, Bg, Bu, nullptr, out, M, N, K, 1.f, 0.f, N, s, sc);
  return launch_rows<E, 64, 2, 4, 2, 2, true, false>(A, Bg, Bu, nullptr, out, M, N, K, 1.f, 0.f, N, s, sc);
}

// Up to 64 rows where few_pay says no: narrow tiles (64 x 64, of [K][N] weights 64 x 128), two workgroups a CU, and as many shares of K
// as give every CU `per_cu` of 64 x 64 (64 x 4096 x 14336: 4 shares 27.6 us, 8 29.2, 64 x 256 tiles in 16 29.9; on [K][N] weights 8 shares
// 27.9, 4 37, 64 x 256 in 16 29.8: both layouts take 8, for the same bits).
static int splitk_plan_narrow(int N, int K, int per_cu, int* k_per) {
  if (K <= 4096) return 1;
  const int shares = std::min(std::min(per_cu * cu_count() / ((N + 63) / 64), K / 512), kMaxShares);
  if (shares < 2) return 1;
  *k_per = ((K + shares - 1) / shares + BK - 1) / BK * BK;
  return (K + *k_per - 1) / *k_per;
}

// [K][N] weights where k-contiguous ones run on the weight stream, in its order of sums: 64 x 128 tiles, two workgroups a CU, in 2, 4 or 8
// shares of the classes, no more than `most` (what the workspace holds) and fewer against more columns, whose sums are to be written.
// Against 64 x 256 tiles in runs of K, 1 to 64 rows: 4096 x 4096 13.2 .. 15.8 -> 10.7 .. 13.7 us, 6144 x 4096 14.7 .. 18.1 -> 14.6 ..
// 17.4, 4096 x 14336 24.9 .. 29.7 -> 22.6 .. 27.8, 12288 x 4096 22.4 .. 26.0 -> 23.1 .. 26.6.  The stream, in the longest pieces of a k row
// that still give the CUs work, where nothing is to be split, against more than 64 columns a CU and in the gap below 6144: 28672 x 4096
// 43 -> 40 us, 128256 x 4096 171 -> 160; without a workspace 4096 x 4096 40 -> 16.
template <class E>
static int launch_classes(const uint16_t* A, const uint16_t* B, const uint16_t* C, uint16_t* D, int M, int N, int K, float alpha, float beta,
                          int ldc, int most, float* P, hipStream_t s) {
  const int tiles = (N + 127) / 128, cus = cu_count();
  int shares = tiles <= cus / 8 || in_a_gap(N, K) ? 8 : tiles <= cus / 4 ? 4 : tiles <= cus / 2 ? 2 : 1;
  if (most >= 8 && N > 16 * cus && N <= 22 * cus)  // 5120 x 5120: 15.3 us, 16.2 in 4 shares of the others
    return launch_splitk<E, 64, 256, 1, 4, false, false, kWholeCu, 1>(A, B, C, D, M, N, K, alpha, beta, ldc, 8, 0, P, s);
  if (in_a_gap(N, K) && K < 6144) shares = 1;
  while (shares > most) shares /= 2;
  if (shares > 1) return launch_splitk<E, 64, 128, 2, 2, false, false, kHalfCu, 2>(A, B, C, D, M, N, K, alpha, beta, ldc, shares, 0, P, s);
  auto rows = [&](auto ar_c) {
    constexpr int AR = decltype(ar_c)::value;
    if (N <= 16 * cus) return launch_rows<E, AR, 1, 8, 1, 1, false, false>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s);
    if (N <= 32 * cus) return launch_rows<E, AR, 2, 8, 1, 1, false, false>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s);
    if constexpr (AR <= 32)
      if (N > 64 * cus) return launch_rows<E, AR, 8, 8, 1, 1, false, false>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s);
    return launch_rows<E, AR, 4, 8, 1, 1, false, false>(A, B, nullptr, C, D, M, N, K, alpha, beta, ldc, s);
  };
  return M <= 8 ? rows(ic<8>{}) : M <= 16 ? rows(ic<16>{}) : M <= 32 ? rows(ic<32>{}) : rows(ic<64>{});
}

// The same for the pair: 64 x 128 tiles (1 to 64 rows of 8192 x 8192 57 .. 63 -> 53 .. 61 us), or the stream, also against few columns and a
// short contraction (32 x 2048 x 2048 14.4 -> 12.5; 28672 x 8192 167 -> 157).
template <class E>
static int launch_classes_dual(const uint16_t* A, const uint16_t* Bg, const uint16_t* Bu, uint16_t* out, int M, int N, int K, int most, float* P,
                               hipStream_t s) {
  const int cus = cu_count(), shares = most >= 8 ? 8 : most >= 4 ? 4 : 2;
  const bool narrow = N <= 4 * cus && K < 4096;
  if (most > 1 && !narrow) return launch_splitk<E, 64, 128, 2, 2, false, true, kWholeCu, 2>(A, Bg, nullptr, out, M, N, K, 1.f, 0.f, N, shares, 0, P, s, Bu);
  auto rows = [&](auto ar_c) {
    constexpr int AR = decltype(ar_c)::value;
    if (narrow) return launch_rows<E, AR, 2, 8, 2, 1, false, false>(A, Bg, Bu, nullptr, out, M, N, K, 1.f, 0.f, N, s);
    if constexpr (AR <= 32)
      if (N > 64 * cus) return launch_rows<E, AR, 8, 4, 2, 1, false, false>(A, Bg, Bu, nullptr, out, M, N, K, 1.f, 0.f, N, s);
    return launch_rows<E, AR, 4, 4, 2, 1, false, false>(A, Bg, Bu, nullptr, out, M, N, K, 1.f, 0.f, N, s);
  };
  return M <= 8 ? rows(ic<8>{}) : M <= 16 ? rows(ic<16>{}) : M <= 32 || narrow ? rows(ic<32>{}) : rows(ic<64>{});
}

}  // namespace nf
