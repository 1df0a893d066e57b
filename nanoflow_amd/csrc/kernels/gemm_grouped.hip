// Grouped GEMMs on k-contiguous weights, D_g = act(A_g . B_g^T): the experts of a mixture (every group has the
// rows its router chose, found through the routing's tile list and gathered while they are loaded) and
// per-head products (every group has all rows and columns of its own).
//
// bf16: the tiles of the plain GEMM family; an m tile never spans two groups.  fp32: gemm_f32's tile.
#include "gemm_f32_tile.h"
#include "gemm_chain.h"

namespace {

struct TilePlace {
  int group, m_base, rows, n_tile;  // rows: of the group
  size_t row0;                      // the group's first row in A (routed, not gathered) and in D
};

// Tile `logical` of the launch; group -1: past the end.  Inside a routed group the m tiles are fastest: they run side by
// side and share a panel of the expert's weights, which is read once.
// kSpread: every XCD takes an eighth of every group's panels instead of its own run of the launch's tiles, for launches whose tiles
// cost very unlike: the last XCD would have all of an expert that every token goes to (256 rows, 32 experts of 2048 x 2048 and
// such a one: 92 -> 75 us).  An eighth is a run of neighbours: every eighth panel is 25 % slower (64 rows of 3584 x 4096: 182 us,
// 139).  And the last expert's panels come first where there are at most 30 rows an expert: an expert that every token goes to follows the
// others, and its tiles of 128 x 32 are a launch's longest (4 of 32 of 2048 x 2048 beside such a one, us, first expert first -> last first: 24 tokens
// 47.5 -> 44.4, 49 58.5 -> 49.1, 80 55.8 -> 47.6, 128 53.8 -> 51.5, 200 59.1 -> 58.5; of more rows they take the CUs' intake from the streams: 230 60.9 and 61.9,
// 256 63.1 and 66.0; without such a one 47.1 to 51.7 and 47.2 to 52.0).
template <int BM, bool kSpread = false>
__device__ __forceinline__ TilePlace find_tile(const nf_grouped_gemm_args& a, int bid, int tiles_n) {
  const int tiles_m = (a.M + BM - 1) / BM;
  const int per = (tiles_n + 7) / 8, start = kSpread ? bid % 8 * per : 0;
  if constexpr (kSpread) {
    tiles_n = min(per, tiles_n - start);
    if (tiles_n <= 0) return {-1, 0, 0, 0, 0};
  }
  const int m_tiles = a.routing.n_tiles ? *a.routing.n_tiles : tiles_m * a.groups;
  const int total = m_tiles * tiles_n;
  if (bid / 8 >= (kSpread ? total : (total + 7) / 8)) return {-1, 0, 0, 0, 0};
  const int logical = !kSpread ? xcd_order(bid, total) : a.max_rows <= 30 * a.groups ? total - 1 - bid / 8 : bid / 8;
  if (logical >= total) return {-1, 0, 0, 0, 0};
  const int mt = logical / tiles_n, n_tile = logical % tiles_n;
  if (a.routing.n_tiles) {
    const int g = a.routing.tile_group[mt], row0 = a.routing.offsets[g], rows = a.routing.offsets[g + 1] - row0;
    const int i = logical - (mt - a.routing.tile_row[mt] / BM) * tiles_n, tiles = (rows + BM - 1) / BM;
    return {g, i % tiles * BM, rows, i / tiles + start, (size_t)row0};
  }
  return {mt / tiles_m, mt % tiles_m * BM, a.M, n_tile + start, 0};
}

// The BM x BN tile of a group from row t.m_base and column n_base.
template <class E, int BM, int BN, int WM, int WN, int kCap, bool kTurn>
__device__ __forceinline__ void grouped_tile(const nf_grouped_gemm_args& a, const TilePlace& t, int n_base) {
  const bool routed = a.routing.n_tiles != nullptr;
  const int32_t* rows = routed && a.gather ? a.routing.row_of + t.row0 : nullptr;
  const uint16_t* A = (const uint16_t*)a.a + (routed ? (rows ? 0 : t.row0 * a.lda) : (size_t)t.group * a.a_group);
  uint16_t* D = (uint16_t*)a.d + (routed ? t.row0 * a.ldd : (size_t)t.group * a.d_group);
  GroupEpilogue ep;
  if (routed && a.weigh) ep.row_scale = a.routing.row_weight + t.row0;
  if constexpr (std::is_same_v<E, BF16Gated>) {
    ep.slope = a.gated.slope;
    ep.shift = a.gated.shift;
    if (a.gated.limits) ep.limit = a.gated.limits[t.group];
  }
  // Weight rows are whole multiples of 4 KB apart where K is a multiple of 2048, and workgroups that walk K in step then ask a few of the memory's
  // channels at a time (a stream of 8 rows of 128 bytes an instruction: 4.4 TB/s, 6.1 with every workgroup at another k).  So every column tile
  // of an expert starts K at a slab of its own and goes round; the m tiles that share its weights start at the same one.
  const int turn = kTurn ? (t.n_tile + t.group * 4) % ((a.K + BK - 1) / BK) : 0;
  gemm_tile<E, BM, BN, WM, WN, false, true, false, true, kCap, false, 0, kTurn>(A, (const uint16_t*)a.b + (size_t)t.group * a.N * a.K, nullptr, nullptr, D,
                                                               t.rows, a.N, a.K, 1.f, 0.f, a.N, t.m_base, n_base, a.lda, a.K,
                                                               a.ldd, rows, a.M, ep, 0, 1, turn);
}

// kFit: a tile with at most half its rows is half as high, with the same sums: of uneven experts many are, and a tile of 2048 deep takes
// less than its place in a round (748 rows, 5 of 32 experts and 8 identities, 28 to 300 rows each, a layer 401 -> 387 us; 560 rows, 2 of 8
// experts of 14336 x 2048 140 -> 129; 800 rows, 4 of 32 of 2048 x 2048, nearly all with more than 64, 71 and 71).
template <class E, int BM, int BN, int WM, int WN, int kCap, bool kFit, bool kTurn>
__global__ __launch_bounds__(WM * WN * 64, kCap == kHalfCu ? 2 : 1) void gemm_grouped_kernel(nf_grouped_gemm_args a, int tiles_n) {
  const TilePlace t = find_tile<BM>(a, blockIdx.x, tiles_n);
  if (t.group < 0) return;
  if constexpr (kFit) {
    static_assert(GemmSmem<BM / 2, BN, 1, kCap>::bytes <= GemmSmem<BM, BN, 1, kCap>::bytes, "both heights run in the same LDS");
    if (t.rows - t.m_base <= BM / 2) return grouped_tile<E, BM / 2, BN, WM, WN, kCap, kTurn>(a, t, t.n_tile * BN);
  }
  grouped_tile<E, BM, BN, WM, WN, kCap, kTurn>(a, t, t.n_tile * BN);
}

unsigned grid_of(const nf_grouped_gemm_args& a, int bm, int tiles_n) {
  const long long m_tiles = a.routing.n_tiles ? (long long)a.max_rows / bm + std::min(a.groups, a.max_rows) : (long long)((a.M + bm - 1) / bm) * a.groups;
  return (unsigned)((m_tiles * tiles_n + 7) / 8 * 8);
}

// Experts with few rows (tile lists of 64): the weight stream of gemm_rows.h, 32 output columns of an expert a workgroup, on a tile
// that fits the rows that are there.  An expert with more of them than that (one that every token goes to) has 128 x 32 tiles,
// which leave the other half of its entries in the list out.
constexpr int kFewRows = 48;  // three 16-row tiles beside 32 columns: 80 KB of ring, two workgroups a CU
template <class E, bool kSpread>
__global__ __launch_bounds__(256) void gemm_grouped_rows_kernel(nf_grouped_gemm_args a, int tiles_n) {
  const TilePlace t = find_tile<64, kSpread>(a, blockIdx.x, tiles_n);
  if (t.group < 0) return;
  const int32_t* from = a.gather ? a.routing.row_of + t.row0 : nullptr;
  const uint16_t* A = (const uint16_t*)a.a + (from ? 0 : t.row0 * a.lda);
  uint16_t* D = (uint16_t*)a.d + t.row0 * a.ldd;
  const float* row_scale = a.weigh ? a.routing.row_weight + t.row0 : nullptr;
  GroupEpilogue ep;
  if constexpr (std::is_same_v<E, BF16Gated>) {
    ep.slope = a.gated.slope;
    ep.shift = a.gated.shift;
    if (a.gated.limits) ep.limit = a.gated.limits[t.group];
  }
  const rsrc_t a_rsrc = make_rsrc(A, ((size_t)((from ? a.M : t.rows) - 1) * a.lda + a.K) * 2);
  const rsrc_t b_rsrc[1] = {make_rsrc((const uint16_t*)a.b + (size_t)t.group * a.N * a.K, (size_t)a.N * a.K * 2)};
  const int end = t.rows;
  auto pass = [&](auto rows_c, int m0) {
    rows_tile<E, decltype(rows_c)::value, 2, 4, 1, 2, true>(
        a_rsrc, b_rsrc, (uint32_t)a.K * 2u, a.N, m0, t.n_tile * 32,
        [&](int m) { return m < end ? (uint32_t)(from ? from[m] : m) * (uint32_t)a.lda * 2u : kOob; },
        [&](int m, int n, float4_t(&v)[1]) {
          if (m >= end) return;
          if (row_scale) v[0] *= row_scale[m];
          if constexpr (std::is_same_v<E, BF16Gated>) {
            *reinterpret_cast<uint32_t*>(D + (size_t)m * a.ldd + n / 2) = E::pack2(ep.gated(v[0][0], v[0][1]), ep.gated(v[0][2], v[0][3]));
          } else {
            const float4_t o = E::finish(v[0]);
            *reinterpret_cast<u32x2*>(D + (size_t)m * a.ldd + n) = u32x2{E::pack2(o[0], o[1]), E::pack2(o[2], o[3])};
          }
        });
  };
  if (t.rows > kFewRows) {
    if (t.m_base % 128 == 0) grouped_tile<E, 128, 32, 4, 1, kHalfCu, false>(a, t, t.n_tile * 32);
  } else if (t.rows <= 16) {
    pass(ic<16>{}, t.m_base);
  } else if (t.rows <= 32) {
    pass(ic<32>{}, t.m_base);
  } else {
    pass(ic<kFewRows>{}, t.m_base);
  }
}

template <class E, bool kSpread>
int launch_grouped_rows(const nf_grouped_gemm_args& a, hipStream_t s) {
  constexpr int lds = RowsSmem<kFewRows, 2, 4, 1, 2>::bytes;
  static_assert(GemmSmem<128, 32, 1, kHalfCu>::bytes <= lds, "the other tile runs in the same LDS");
  auto kern = gemm_grouped_rows_kernel<E, kSpread>;
  static bool attr_set = false;  // benign race: the call is idempotent
  if (!attr_set) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      set_error("nf_gemm_grouped: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
      return NF_ERR_RUNTIME;
    }
    attr_set = true;
  }
  const int tiles_n = (a.N + 31) / 32;
  kern<<<grid_of(a, 64, kSpread ? (tiles_n + 7) / 8 * 8 : tiles_n), 256, lds, s>>>(a, tiles_n);
  return check_launch("nf_gemm_grouped");
}

template <int kAct>
__global__ __launch_bounds__(256) void gemm_grouped_f32_kernel(nf_grouped_gemm_args a, int tiles_n) {
  const TilePlace t = find_tile<kF32Tile>(a, blockIdx.x, tiles_n);
  if (t.group < 0) return;
  const bool routed = a.routing.n_tiles != nullptr;
  const int32_t* rows = routed && a.gather ? a.routing.row_of + t.row0 : nullptr;
  const float* A = (const float*)a.a + (routed ? (rows ? 0 : t.row0 * a.lda) : (size_t)t.group * a.a_group);
  float* D = (float*)a.d + (routed ? t.row0 * a.ldd : (size_t)t.group * a.d_group);
  RowEpilogue ep;
  if (routed && a.weigh) ep.row_scale = a.routing.row_weight + t.row0;
  if constexpr (kAct == NF_ACT_GATED) {
    ep.slope = a.gated.slope;
    ep.shift = a.gated.shift;
    if (a.gated.limits) ep.limit = a.gated.limits[t.group];
  }
  gemm_f32_tile<kAct>(A, (const float*)a.b + (size_t)t.group * a.N * a.K, nullptr, D, t.rows, a.N, a.K, a.lda, a.K, a.ldd, rows, t.m_base,
                      t.n_tile * kF32Tile, ep);
}

template <class E, int BM, int BN, int WM, int WN, int kCap, bool kFit, bool kTurn>
int launch_grouped_of(const nf_grouped_gemm_args& a, hipStream_t s) {
  using SM = GemmSmem<BM, BN, 1, kCap>;
  auto kern = gemm_grouped_kernel<E, BM, BN, WM, WN, kCap, kFit, kTurn>;
  static bool attr_set = false;  // benign race: the call is idempotent
  if (!attr_set) {
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)SM::bytes);
    if (e != hipSuccess) {
      set_error("nf_gemm_grouped: cannot reserve %zu bytes of LDS: %s", SM::bytes, hipGetErrorString(e));
      return NF_ERR_RUNTIME;
    }
    attr_set = true;
  }
  const int tiles_n = (a.N + BN - 1) / BN;
  kern<<<grid_of(a, BM, tiles_n), WM * WN * 64, SM::bytes, s>>>(a, tiles_n);
  return check_launch("nf_gemm_grouped");
}

// Turned contractions: experts whose weights are at least 128 MB, half the last-level cache, which the memory's channels set the pace of (time
// turned over straight 0.80 to 1.00, 748 rows, 5 of 32 experts of 2048 x 2048 90 -> 80 us; experts of 200 rows and more 1.00).  Of fewer weights, and where K is no
// multiple of 2048, the offsets that go round only cost (8 of 2048 x 2048 19.0 us and 20.0, 4 of 256 x 4096 28.4 and 30.7; 8 of 768 x 1408, of which none
// turn, 12.9 and 13.6), nor do the tiles of the one expert beside a weight stream gain.
template <class E, int BM, int BN, int WM, int WN, int kCap = kWholeCu, bool kFit = false>
int launch_grouped(const nf_grouped_gemm_args& a, hipStream_t s) {
  return a.routing.n_tiles && a.K % 2048 == 0 && (size_t)a.groups * a.N * a.K * 2 >= (size_t)128 << 20
             ? launch_grouped_of<E, BM, BN, WM, WN, kCap, kFit, true>(a, s)
             : launch_grouped_of<E, BM, BN, WM, WN, kCap, kFit, false>(a, s);
}

// Each XCD takes a run of the launch's tiles (m tiles of an expert fastest), its workgroups every n-th of them.
template <class E, int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(WM * WN * 64, 1) void gemm_chain_kernel(nf_grouped_gemm_args a, int tiles_n) {
  typedef const __attribute__((address_space(4))) int32_t* list_t;  // read-only: by scalar loads, which the operands' waits do not count
  const list_t n_tiles = (list_t)a.routing.n_tiles, groups = (list_t)a.routing.tile_group, tile_row = (list_t)a.routing.tile_row, offsets = (list_t)a.routing.offsets;
  const int total = n_tiles[0] * tiles_n, per = (total + 7) / 8, x = blockIdx.x % 8, end = min((x + 1) * per, total);
  const int first = x * per + blockIdx.x / 8, nslab = (a.K + BK - 1) / BK;
  if (first >= end) return;
  gemm_chain<E, BM, BN, WM, WN>(a, first, end, gridDim.x / 8, [&](int logical) {
    if (logical >= end) return ChainTile{0, 0, 0, 0, 0, 0};
    const int mt = logical / tiles_n, g = groups[mt], row0 = offsets[g], rows = offsets[g + 1] - row0;
    const int i = logical - (mt - tile_row[mt] / BM) * tiles_n, tiles = (rows + BM - 1) / BM, n_tile = i / tiles;
    const int h = ((rows + tiles - 1) / tiles + 16 * WM - 1) / (16 * WM) * (16 * WM), m_base = i % tiles * h;
    return ChainTile{g, m_base, min(rows, m_base + h), n_tile * BN, row0, (n_tile + g * 4) % nslab};
  });
}

template <class E>
int launch_chain(const nf_grouped_gemm_args& a, hipStream_t s) {
  constexpr int BM = 128, BN = 256;
  using SM = ChainSmem<BM, BN>;
  auto kern = gemm_chain_kernel<E, BM, BN, 2, 4>;
  static bool attr_set = false;  // benign race: the call is idempotent
  if (!attr_set) {
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)SM::bytes);
    if (e != hipSuccess) {
      set_error("nf_gemm_grouped: cannot reserve %zu bytes of LDS: %s", SM::bytes, hipGetErrorString(e));
      return NF_ERR_RUNTIME;
    }
    attr_set = true;
  }
  const int tiles_n = (a.N + BN - 1) / BN;
  kern<<<std::min(grid_of(a, BM, tiles_n), (unsigned)std::max(cu_count() / 8 * 8, 8)), 512, SM::bytes, s>>>(a, tiles_n);
  return check_launch("nf_gemm_grouped");
}

// Tile lists of 128 rows that run on gemm_chain.h.  Contractions beyond 2048 against whole column tiles do, where a 128 x 256 tile on eight wavefronts
// stands against it: 0.93 to 1.04 of its time over 80 launches of more than a round, 2112 to 8192 deep, 0.99 in the mean; below a round it has its even
// shares of an expert's rows alone, 0.93 where they are 150 and 1.05 to 1.10 where they fill a tile (800 of 8 experts of 512 x 2304).
// At 2048 two workgroups of 128 x 128 a CU stand against it, which leave less of a round idle: it pays where its own rounds, of which there must be more
// than one, are at least four fifths full of columns that are there (0.87 to 1.02 of their time; 1.1 to 1.5 rounds 1.00, 2.0 to 2.4 0.99 to 1.01; in
// one round 0.84 to 0.98, but 1.04 to 1.26 where the 128 x 128 tiles are no more than the CUs).  The rows of
// an expert are not known here: half a tile each over the sorted rows, among which are those of identity choices, that no expert has: with a fifth
// of them a launch taken for full rounds can be 1.09 of the other form's time.  Below 2048 neither wins.
bool chain_pays(const nf_grouped_gemm_args& a) {
  if (a.K < 2048 || a.N < 256 || a.ldd > 1 << 22 || (a.act == NF_ACT_GATED ? a.N % 16 != 0 : a.weigh)) return false;
  if (a.K > 2048) return a.N % 256 == 0;
  const double m_tiles = a.max_rows / 128.0 + a.groups * 0.5, rounds = m_tiles * ((a.N + 255) / 256) / cu_count(), filled = m_tiles * a.N / 256.0 / cu_count();
  return rounds > 1 && std::ceil(rounds) <= 1.25 * filled;
}

template <class E>
int dispatch_grouped(const nf_grouped_gemm_args& a, int tile_rows, hipStream_t s) {
  if (a.routing.n_tiles) {
    // Few rows an expert: as gemm_rows.h.  Its workgroups re-read an expert's rows for every 32 columns, which the larger tiles do
    // not, so from 17 rows on it pays for short contractions only.  32 experts, 4 of them a token, us against 64 x 256 tiles:
    //   N x K         1 token   16 tokens   64 tokens   256 tokens (32 rows an expert)
    //   2048 x 2048   19 -> 13   59 -> 46    65 -> 47    66 -> 56
    //   4096 x 3584   44 -> 21  136 -> 116  159 -> 139  165 -> 185: not taken
    // 64 tokens, 2 of 8 of 4096 x 14336 (16 rows an expert): 202 -> 156.
    // Where it ends: 2048 deep 40 rows an expert 67 -> 61.5, 48 rows 68 -> 71 (4096 x 2048: 126 -> 114, 126 -> 131); 1536 deep 17 rows
    // 41 -> 41, 24 rows 41 -> 42.5, 40 rows 41 -> 50.  The line between: 16 rows at 1536, 40 at 2048.
    const long long rows = a.max_rows, groups = a.groups;
    const int most = a.K < 1536 ? 0 : a.K <= 2048 ? 16 + (a.K - 1536) * 24 / 512 : 16;
    if (tile_rows == 64 && rows <= most * groups)
      return a.N >= 512 ? launch_grouped_rows<E, true>(a, s) : launch_grouped_rows<E, false>(a, s);
    // Short contractions: a third of a tile's time is its start and its end, so two workgroups share a CU and one runs under the
    // other's (2000 rows, 8 of 64 experts of 1024 x 1024: 80 -> 62 us; 1946 rows, 5 of 33 gated experts of 4096 x 2048: 242 ->
    // 225).  Longer ones want the larger tile's lower LDS traffic (512 rows, 4 of 32 of 4096 x 3584: 187 us against 205).
    if (tile_rows == 128 && chain_pays(a)) return launch_chain<E>(a, s);
    if (a.K <= 2048)
      return tile_rows == 64 ? launch_grouped<E, 64, 128, 2, 2, kHalfCu>(a, s) : launch_grouped<E, 128, 128, 2, 2, kHalfCu, true>(a, s);
  }
  // One workgroup a CU: eight wavefronts (us, four -> eight: 16 heads of 128 x 512 for 128 rows 8.1 -> 6.4, of 576 x 128 5.1 -> 4.4; 256 rows, 4 of 33 experts of
  // 2048 x 4096 156 -> 131, the contraction turned among it).  Two a CU gain nothing by it (1946 rows, 33 experts of 3072 x 1536 144 and 155).
  if (tile_rows == 64) return a.N <= 128 ? launch_grouped<E, 64, 128, 2, 4>(a, s) : launch_grouped<E, 64, 256, 2, 4>(a, s);
  return a.N > 128 && a.N % 256 == 0 ? launch_grouped<E, 128, 256, 2, 4>(a, s) : launch_grouped<E, 128, 128, 2, 4>(a, s);
}

}  // namespace

extern "C" {

// Rows of an m tile: what the routing's tile list has to be made for.  From 96 slots an expert on most experts have more than 64 rows, and two
// tiles of 64 pass their weights twice.  us on 128 / 64 rows: 32 experts of 4096 x 3584 at 100 slots 186 / 219 and at 117 223 / 253, 8 of
// 4096 x 4096 at 117 76 / 106, 32 of 2048 x 2560 at 110 109 / 118; 2048 deep and less 64 rows win up to 120 (2048 x 2048 at 117 95 / 84),
// but the list is made before the contraction is known.
int nf_grouped_tile_rows(int dtype, int rows, int groups) {
  if (dtype == NF_F32) return kF32Tile;
  return (long long)rows <= 96ll * std::max(groups, 1) ? 64 : 128;
}

int nf_gemm_grouped(const nf_grouped_gemm_args* args, nf_stream_t stream) {
  const char* who = "nf_gemm_grouped";
  NF_REQUIRE(args, "%s: null pointer", who);
  const nf_grouped_gemm_args& a = *args;
  NF_REQUIRE(a.dtype == NF_F32 || a.dtype == NF_BF16, "%s: unknown dtype %d", who, a.dtype);
  NF_REQUIRE(a.act == NF_ACT_NONE || a.act == NF_ACT_GELU || a.act == NF_ACT_SQUARED_RELU || a.act == NF_ACT_GATED, "%s: unknown activation %d", who, a.act);
  NF_REQUIRE(a.groups > 0 && a.M >= 0 && a.N > 0 && a.K > 0 && a.N % 8 == 0 && a.K % 8 == 0 && a.lda >= a.K && a.ldd >= (a.act == NF_ACT_GATED ? a.N / 2 : a.N) && a.lda % 8 == 0 &&
                 a.ldd % 8 == 0 && a.a_group % 8 == 0 && a.d_group % 8 == 0,
             "%s: bad shape: %d groups, M=%d N=%d K=%d, strides %d %d", who, a.groups, a.M, a.N, a.K, a.lda, a.ldd);
  const bool routed = a.routing.n_tiles != nullptr;
  NF_REQUIRE(!routed || (a.routing.tile_group && a.routing.tile_row && a.routing.offsets && a.max_rows >= 0 && (!a.gather || a.routing.row_of)),
             "%s: incomplete routing", who);
  NF_REQUIRE(!a.weigh || (routed && a.routing.row_weight), "%s: no weights of the sorted rows", who);
  if (a.M == 0 || (routed && a.max_rows == 0)) return NF_OK;
  NF_REQUIRE(a.a && a.b && a.d, "%s: null pointer", who);
  NF_REQUIRE(((uintptr_t)a.a | (uintptr_t)a.b | (uintptr_t)a.d) % 16 == 0, "%s: operands must be 16-byte aligned", who);
  const int a_rows = routed && !a.gather ? a.max_rows : a.M;
  NF_REQUIRE(((size_t)a_rows + 256) * ((size_t)a.lda + 512) * 2 < 0xFFFFFF00ull && ((size_t)a.N + 256) * ((size_t)a.K + 512) * 2 < 0xFFFFFF00ull,
             "%s: an operand exceeds the 4 GiB buffer-addressing limit", who);
  const int tile_rows = a.dtype == NF_F32 || routed ? nf_grouped_tile_rows(a.dtype, a.max_rows, a.groups) : a.M <= 96 ? 64 : 128;
  NF_REQUIRE(!routed || a.routing.tile_rows == tile_rows, "%s: the tile list is for tiles of %d rows, not %d", who, a.routing.tile_rows, tile_rows);
  hipStream_t s = (hipStream_t)stream;
  if (a.dtype == NF_F32) {
    const int tiles_n = (a.N + kF32Tile - 1) / kF32Tile;
    auto kern = a.act == NF_ACT_GELU           ? gemm_grouped_f32_kernel<NF_ACT_GELU>
                : a.act == NF_ACT_SQUARED_RELU ? gemm_grouped_f32_kernel<NF_ACT_SQUARED_RELU>
                : a.act == NF_ACT_GATED        ? gemm_grouped_f32_kernel<NF_ACT_GATED>
                                               : gemm_grouped_f32_kernel<NF_ACT_NONE>;
    kern<<<grid_of(a, kF32Tile, tiles_n), 256, 0, s>>>(a, tiles_n);
    return check_launch(who);
  }
  if (a.act == NF_ACT_SQUARED_RELU) return dispatch_grouped<BF16SquaredRelu>(a, tile_rows, s);
  if (a.act == NF_ACT_GATED) return dispatch_grouped<BF16Gated>(a, tile_rows, s);
  return a.act == NF_ACT_GELU ? dispatch_grouped<BF16Gelu>(a, tile_rows, s) : dispatch_grouped<BF16>(a, tile_rows, s);
}

}  // extern "C"
