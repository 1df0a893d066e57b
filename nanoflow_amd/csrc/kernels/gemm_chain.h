#pragma once
// Routed grouped products on workgroups that stay for the whole launch (16-bit operands, k-contiguous weights, tile lists of 128 rows): 128 x 256
// tiles on eight wavefronts, one workgroup a CU, and the rings of operand slabs run on from a tile into the workgroup's next one.
//
// What bounds it: the weights' way from HBM (32 experts of 4096 x 2048 are 537 MB, at 5-6 TB/s 95 us of the 206) and the matrix pipe at the
// power cap (128 us of MFMAs), which the lookahead of two slabs overlaps in part.  Three things differ from gemm_tile on these tiles, all measured
// on 32 experts, 4 of them a token:
//   - The rows of weights are whole multiples of 4 KB apart where K is a multiple of 2048, and workgroups that walk K in step then ask a few of the
//     memory's channels at a time (eight rows of 128 bytes an instruction: 4.4 TB/s; each workgroup at another k: 6.1).  So every column tile starts K
//     at a slab of its own and goes round; the tiles that share its weights start at the same one.
//   - A workgroup's next tile is on its way while the last slabs of one are multiplied, and its sums leave the registers as 16-byte
//     stores without LDS: a tile's start and end (6 us of 40 at 2048 deep) are hidden or gone.
//   - An expert's rows are shared out evenly over its tiles, in steps of 32, and only live rows are multiplied.
// us, without a profiler and against what would run instead, two workgroups of 128 x 128 a CU (2048 deep) or a 128 x 256 one on eight wavefronts (3584), turned
// as well: 1946 rows, gated 4096 x 2048 and a 33rd expert for all 231 -> 211, 2048 x 2048 back 118 -> 114; 2047 rows and identities among the choices, 2048 x
// 2048 with GELU 115 -> 114, back 111 -> 109 (their layer 461 -> 451); 2048 rows of 4096 x 3584 324 -> 315.  Under a profiler's clocks the third and fourth lose 2 to 7 %.
// Measured and left: 256 x 256 tiles of as many wavefronts (200 of the 210, but 108 us for 79 where experts have a little more than 256 rows), four
// wavefronts (the compiler moves 128 sums between register files at every branch), rings of four stages (240 for 215: they fill the memory's queues), the
// non-temporal hint on weights that two tiles share, a wavefront that asks for lines ahead of the loads (249 -> 311).
#include "gemm_impl.h"

namespace nf {

struct ChainTile {
  int group, m_base, end, n_base, row0;  // rows [m_base, end) of the group, whose first row is row0; end 0: no tile, every operand reads as zeros
  int turn;                              // the slab of K that comes first
};

template <int BM, int BN>
struct ChainSmem {
  static constexpr int stages = 3, a_bytes = BM * 128, b_bytes = BN * 128, b_ring = stages * a_bytes;
  static constexpr size_t bytes = (size_t)b_ring + stages * (size_t)b_bytes;
};
static_assert(BK == 64, "the loop looks three slabs ahead: contractions of 192 and more");

// Tiles first, first + stride, .. below `end`; place(i) says where tile i lies.  LDS rows and their swizzle are gemm_tile's; row tile q of a
// wavefront is rows (q * WM + wm) * 16 .. of the tile, so that its first rows lie in all row waves alike.
template <class E, int BM, int BN, int WM, int WN, class Place>
__device__ __forceinline__ void gemm_chain(const nf_grouped_gemm_args& a, int first, int end, int stride, Place place) {
  using SM = ChainSmem<BM, BN>;
  constexpr int NS = SM::stages, NW = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16, CH = TN / 2;
  constexpr int AL = BM / (8 * NW), BL = BN / (8 * NW), HA = (AL + 1) / 2, HB = (BL + 1) / 2;  // loads of a slab, and those of a first half
  constexpr int G = 4, TNG = TN / G;
  constexpr bool kPairs = std::is_same_v<E, BF16Gated>;
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && TN % G == 0 && AL + BL < 64, "tile shape");
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const uint32_t smem_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN, l16 = lane & 15, lq = lane >> 4;
  const int K = a.K, N = a.N, lda = a.lda, ldd = a.ldd, nslab = (K + BK - 1) / BK;
  const bool gather = a.gather;

  using acc_t = typename AccVec<G>::type;
  acc_t acc[TM][TNG];
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TNG; ++j) acc[i][j] = acc_t{};
  };
  clear();

  // the tile that is multiplied, the one whose loads follow on its, and the one whose rows are looked up at the end of the first
  int at = first + 2 * stride;
  ChainTile cur = place(first), nxt = place(first + stride), third = place(at);

  // ---- loads, as gemm_tile's.  What a tile needs from global memory beforehand -- its rows of A, and their weights for the epilogue -- is asked for
  // ahead of the stores of the tile two before it and waited for behind them: any wait of the compiler's own elsewhere would be for the slabs in
  // flight as well.
  const int kc = ((lane & 7) ^ (((lane >> 4) & 3) | ((wave & 1) << 2))) * 8;
  auto tile_row = [&](int t) { return (t * NW + wave) * 8 + (lane >> 3); };
  int index[AL];
  auto fetch_rows = [&](const ChainTile& t) {
#pragma unroll
    for (int i = 0; i < AL; ++i) {
      const int r = t.m_base + tile_row(i);
      index[i] = gather ? a.routing.row_of[t.row0 + (r < t.end ? r : 0)] : r;
    }
  };
  constexpr int WT = kPairs ? TM : 0;  // weights: gated experts only
  float weight[TM], next_weight[TM];
  auto fetch_weights = [&](const ChainTile& t) {
#pragma unroll
    for (int i = 0; i < WT; ++i) {
      const int r = t.m_base + (i * WM + wm) * 16 + l16;
      next_weight[i] = a.weigh ? a.routing.row_weight[t.row0 + (r < t.end ? r : 0)] : 1.f;
    }
  };
  auto land = [&] {
#pragma unroll
    for (int i = 0; i < AL; ++i) asm volatile("" : "+v"(index[i]));
#pragma unroll
    for (int i = 0; i < WT; ++i) asm volatile("" : "+v"(next_weight[i]));
  };
  uint32_t a_off[AL], b_off[BL];
  rsrc_t a_rsrc, b_rsrc;
  int ka = 0, kb = 0;  // slab of K that the activation / weight loads are at
  auto aim_a = [&](const ChainTile& t) {
    ka = t.turn;
    const size_t extent = t.end > 0 ? ((size_t)((gather ? a.M : t.end) - 1) * lda + K) * 2 : 0;
    a_rsrc = make_rsrc((const uint16_t*)a.a + (gather ? 0 : (size_t)t.row0 * lda), extent);
    const uint32_t past = (uint32_t)((extent + 15) & ~(size_t)15);  // rows past the tile's last one read as zero
#pragma unroll
    for (int i = 0; i < AL; ++i) a_off[i] = (t.m_base + tile_row(i) < t.end ? ((uint32_t)index[i] * (uint32_t)lda + kc) * 2u : past) + ka * (BK * 2u);
  };
  auto aim_b = [&](const ChainTile& t) {
    kb = t.turn;
    b_rsrc = make_rsrc((const uint16_t*)a.b + (size_t)t.group * N * K, t.end > 0 ? (size_t)N * K * 2 : 0);
#pragma unroll
    for (int i = 0; i < BL; ++i) b_off[i] = ((uint32_t)(t.n_base + tile_row(i)) * (uint32_t)K + kc) * 2u + kb * (BK * 2u);
  };
  auto a_lds = [&](int stage) { return __builtin_amdgcn_readfirstlane(smem_lds + stage * SM::a_bytes + wave * 1024); };
  auto b_lds = [&](int stage) { return __builtin_amdgcn_readfirstlane(smem_lds + SM::b_ring + stage * SM::b_bytes + wave * 1024); };
  auto after = [&](int k) { return k + 1 == nslab ? 0 : k + 1; };
  auto k_ok = [&](int k) { return k * BK + kc < K; };
  auto advance = [&](int k) { return k + 1 == nslab ? -(nslab - 1) * (BK * 2) : BK * 2; };
  uint32_t pend = 0;
  auto load_prepare = [&](auto t_c, bool ok, int by) {
    constexpr int t = decltype(t_c)::value;
    uint32_t& off = t < AL ? a_off[t < AL ? t : 0] : b_off[t < AL ? 0 : t - AL];
    pend = ok ? off : kOob;
    off += by;
  };
  auto load_issue = [&](auto t_c, uint32_t st) {
    constexpr int t = decltype(t_c)::value;
    if constexpr (t < AL) load16_to_lds<t * NW * 1024>(a_rsrc, pend, st);
    else load16_to_lds<(t - AL) * NW * 1024>(b_rsrc, pend, st);
  };
  auto load_run = [&](auto l0_c, auto n_c, uint32_t st, int k) {
    static_for<decltype(n_c)::value>([&](auto i_c) {
      load_prepare(ic<decltype(l0_c)::value + decltype(i_c)::value>{}, k_ok(k), advance(k));
      load_issue(ic<decltype(l0_c)::value + decltype(i_c)::value>{}, st);
    });
  };

  half8_t af[2][TM], bh[2][CH];  // by k-step, and by sub-step
  const uint32_t a_rd = (uint32_t)(wm * 16 + l16) * 128u, b_rd = (uint32_t)(wn * (BN / WN) + l16) * 128u;
  uint32_t swz[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) swz[kk] = (uint32_t)(((kk * 4 + lq) ^ ((l16 >> 1) & 7)) << 4);
  auto read_a = [&](auto q_c, auto k2_c, const uint8_t* sa) {
    constexpr int q = decltype(q_c)::value, k2 = decltype(k2_c)::value;
    af[k2][q] = *reinterpret_cast<const half8_t*>(sa + a_rd + swz[k2] + q * WM * 16 * 128);
  };
  auto read_b = [&](auto c_c, auto k2_c, auto h_c, const uint8_t* sb) {
    constexpr int c = decltype(c_c)::value, k2 = decltype(k2_c)::value, h = decltype(h_c)::value;
    bh[h][c] = *reinterpret_cast<const half8_t*>(sb + b_rd + swz[k2] + (h * CH + c) * 16 * 128);
  };
  // Sub-step kk of a slab, as gemm_tile's: k-step kk / 2 on half kk % 2 of the column tiles, `live` row tiles; fragments of what
  // follows from sa / sb (all row tiles of the next slab's first k-step: it may be another tile's), NL loads from L0 on into the stage at `st`.
  auto step = [&](auto live_c, auto kk_c, auto l0_c, auto nl_c, uint32_t st, int k, const uint8_t* sa, const uint8_t* sb) {
    constexpr int L = decltype(live_c)::value, kk = decltype(kk_c)::value, L0 = decltype(l0_c)::value, NL = decltype(nl_c)::value;
    constexpr int K2 = kk >> 1, H = kk & 1, NM = CH * L, NXT = (kk + 1) & 3;
    constexpr int A0 = kk == 1 ? L / 2 : 0, A1 = kk == 0 ? L / 2 : kk == 1 ? L : kk == 3 ? TM : 0, NRA = A1 - A0, NRD = NRA + CH, S = NRD + 2 * NL;
    const bool ok = k_ok(k);
    const int by = advance(k);
    static_for<NM>([&](auto n_c) {
      constexpr int n = decltype(n_c)::value, c = n / L, i = n % L, j = H * CH + c;
      acc_put<j % G, 4 * G>(acc[i][j / G], E::mfma16(bh[H][c], af[K2][i], acc_get<j % G>(acc[i][j / G])));
      constexpr int lo = n * S / NM, hi = (n + 1) * S / NM;
      static_for<hi - lo>([&](auto d_c) {
        constexpr int q = lo + decltype(d_c)::value;
        if constexpr (q < NRA) read_a(ic<A0 + q>{}, ic<(kk == 3 ? 0 : 1)>{}, sa);
        else if constexpr (q < NRD) read_b(ic<q - NRA>{}, ic<(NXT >> 1)>{}, ic<(NXT & 1)>{}, sb);
        else if constexpr ((q - NRD) % 2 == 0) load_prepare(ic<L0 + (q - NRD) / 2>{}, ok, by);
        else load_issue(ic<L0 + (q - NRD) / 2>{}, st);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto meet = [&] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // vmcnt(a slab's loads), lgkmcnt(0): everything up to the next slab has landed, the slab behind it may be in flight.  Stores and lookups of a
  // tile's end count as loads: then more is waited for, never less.
  constexpr int kNextSlab = 0x0070 | ((AL + BL) & 15) | (((AL + BL) >> 4) << 14);

  // ---- the first tile's first slabs: activations and weights of 0 and 1, and the first half of 2's activations, as the slabs before would have
  fetch_rows(cur);
  fetch_weights(cur);
  land();
#pragma unroll
  for (int i = 0; i < WT; ++i) weight[i] = next_weight[i];
  aim_a(cur);
  aim_b(cur);
  fetch_rows(nxt);
  fetch_weights(nxt);
  land();
  static_for<NS - 1>([&](auto s_c) {
    constexpr int s = decltype(s_c)::value;
    load_run(ic<0>{}, ic<AL>{}, a_lds(s), ka);
    load_run(ic<AL>{}, ic<BL>{}, b_lds(s), kb);
    ka = after(ka);
    if (s + 1 < NS - 1) kb = after(kb);
  });
  __builtin_amdgcn_s_waitcnt(kNextSlab);
  meet();
  static_for<TM>([&](auto q_c) { read_a(q_c, ic<0>{}, smem); });
  static_for<CH>([&](auto c_c) { read_b(c_c, ic<0>{}, ic<0>{}, smem + SM::b_ring); });
  load_run(ic<0>{}, ic<HA>{}, a_lds(NS - 1), ka);

  // One slab, from LDS stage `cs`.  It asks for the second half of the activations and all weights of the slab two ahead and, past the barrier, when
  // everybody is done with this stage, for the first half of the activations of the slab three ahead.  NA / NB: those
  // activations / weights are the first of the next tile.
  int cs = 0;
  auto slab = [&](auto live_c, auto na_c, auto nb_c) {
    const int cs1 = cs + 1 == NS ? 0 : cs + 1, cs2 = cs == 0 ? NS - 1 : cs - 1;
    const uint8_t *sa = smem + cs * SM::a_bytes, *sb = smem + SM::b_ring + cs * SM::b_bytes;
    step(live_c, ic<0>{}, ic<HA>{}, ic<AL - HA>{}, a_lds(cs2), ka, sa, sb);
    kb = after(kb);
    if constexpr (decltype(nb_c)::value) aim_b(nxt);
    step(live_c, ic<1>{}, ic<AL>{}, ic<HB>{}, b_lds(cs2), kb, sa, sb);
    step(live_c, ic<2>{}, ic<AL + HB>{}, ic<BL - HB>{}, b_lds(cs2), kb, sa, sb);
    ka = after(ka);
    if constexpr (decltype(na_c)::value) aim_a(nxt);
    __builtin_amdgcn_s_waitcnt(kNextSlab);
    meet();
    step(live_c, ic<3>{}, ic<0>{}, ic<HA>{}, a_lds(cs), ka, smem + cs1 * SM::a_bytes, smem + SM::b_ring + cs1 * SM::b_bytes);
    cs = cs1;
  };
  auto slabs = [&](auto live_c) {
    using T = std::true_type;
    using F = std::false_type;
    for (int s = 0; s < nslab - 3; ++s) slab(live_c, F{}, F{});
    slab(live_c, T{}, F{});
    slab(live_c, F{}, T{});
    slab(live_c, F{}, F{});
  };

  // The sums of a tile that is done.  A lane has 4 neighbouring columns of a row in each MFMA tile; two column tiles (of pairs, which leave half the
  // columns, four) are turned between the four lane groups, so that a lane stores 16 bytes and 64 of a row are together.
  auto store = [&](int live, const ChainTile& t) {
    typedef unsigned int u32v4_t __attribute__((ext_vector_type(4)));
    constexpr int PER = kPairs ? 4 : 2;
    GroupEpilogue ep;
    if constexpr (kPairs) {
      ep.slope = a.gated.slope;
      ep.shift = a.gated.shift;
      if (a.gated.limits) ep.limit = ((const __attribute__((address_space(4))) float*)a.gated.limits)[t.group];
    }
    const int out = kPairs ? N / 2 : N;
    const __amdgpu_buffer_rsrc_t d_rsrc =
        __builtin_amdgcn_make_buffer_rsrc((uint16_t*)a.d + (size_t)(t.row0 + t.m_base) * ldd, 0, ((t.end - t.m_base - 1) * ldd + out) * 2, 0x00020000);
    auto swap = [](uint32_t& x, uint32_t& y, auto far_c) {  // y's lower and x's upper half wave, or every other 16 lanes
      const auto r = decltype(far_c)::value ? __builtin_amdgcn_permlane32_swap(x, y, false, false) : __builtin_amdgcn_permlane16_swap(x, y, false, false);
      x = r[0];
      y = r[1];
    };
    static_for<TM>([&](auto i_c) {
      constexpr int i = decltype(i_c)::value;
      if (i >= live) return;
      const uint32_t row = (uint32_t)((i * WM + wm) * 16 + l16) * (uint32_t)ldd;  // rows past the tile's last one lie past the buffer's end
      static_for<TN / PER>([&](auto j_c) {
        constexpr int j = decltype(j_c)::value * PER;
        uint32_t v[4];
        static_for<PER>([&](auto e_c) {
          constexpr int e = decltype(e_c)::value;
          const float4_t x = acc_get<(j + e) % G>(acc[i][(j + e) / G]);
          if constexpr (kPairs) {
            const float4_t w = x * weight[i];
            v[e] = E::pack2(ep.gated(w[0], w[1]), ep.gated(w[2], w[3]));
          } else {
            const float4_t y = E::finish(x);
            v[2 * e] = E::pack2(y[0], y[1]);
            v[2 * e + 1] = E::pack2(y[2], y[3]);
          }
        });
        swap(v[0], v[2], std::true_type{});
        swap(v[1], v[3], std::true_type{});
        swap(v[0], v[kPairs ? 1 : 2], std::false_type{});
        swap(v[kPairs ? 2 : 1], v[3], std::false_type{});
        const int col = (t.n_base + wn * (BN / WN) + j * 16) / (kPairs ? 2 : 1) + lq * 8;
        __builtin_amdgcn_raw_buffer_store_b128(u32v4_t{v[0], v[1], v[2], v[3]}, d_rsrc, col < out ? (row + col) * 2u : kOob, 0, 0);
      });
    });
  };

  for (;;) {
    static_assert(TM == 4, "as many forms of the loop as row tiles");
    const int live = (cur.end - cur.m_base + 16 * WM - 1) / (16 * WM);
    if (live == 4) slabs(ic<4>{});
    else if (live == 3) slabs(ic<3>{});
    else if (live == 2) slabs(ic<2>{});
    else slabs(ic<1>{});
    const ChainTile done = cur;
    cur = nxt;
    nxt = third;
    const bool more = cur.end > 0;
    float w[TM];
#pragma unroll
    for (int i = 0; i < WT; ++i) w[i] = next_weight[i];
    if (more) {
      fetch_rows(nxt);
      fetch_weights(nxt);
      at += stride;
      third = place(at);
    }
    store(live, done);
    if (!more) break;
    clear();
#pragma unroll
    for (int i = 0; i < WT; ++i) weight[i] = w[i];
    land();
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // what was asked for past the last tile lands, as zeros, before the LDS is another workgroup's
}

}  // namespace nf
