// Routing of a mixture of experts: scores, choice, and the order of the chosen rows by expert.
//
// route_rows_kernel: one wavefront per token, its scores in registers (fp32 softmax over all outputs, or a sigmoid of each), groups of
//   outputs closed by the rank of their largest entry, the `top` largest taken one after the other (up to 64 outputs: all at once, by rank), then the
//   experts that every token has.  What bounds it is a chain of dependent steps: loads that are all on their way before the first is waited for, and lanes that
//   meet without LDS, took both launches from 11.6 to 9.1 us (256 rows of 32 outputs in 8 groups, 4 a token, 16 shares), 11.9 to 9.9 (2047 rows of 40, 5 a
//   token), 8.2 to 6.5 (one row).  (Timed of 1, 4 and 16 shares.  All but the first are requested kMaxShares - 1 at a time, those past the last as the last again, from
//   the caches.)
// route_plan_kernel: counts the rows of every expert, places them (an expert's rows consecutive)
//   and lists the m tiles of the grouped product.  The place of a row inside its expert's run
//   depends on the order of LDS atomics; nothing computed from it does.
#include <algorithm>
#include <cmath>

#include "layer_common.h"

namespace nf {

constexpr int kMaxOutputs = 1024, kMaxTop = 64;

__device__ __forceinline__ float lane_value(float x, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane)); }

template <int kPer>  // outputs per lane
__global__ __launch_bounds__(256) void route_rows_kernel(nf_route_args a, int32_t* __restrict__ choice, float* __restrict__ weight) {
  __shared__ float entry[4][kPer > 1 ? kPer * 64 : 1], best_of[4][kPer > 1 ? kPer * 64 : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, t = blockIdx.x * 4 + wave;
  const bool live = t < a.rows;
  const float* __restrict__ z = a.z + (size_t)(live ? t : 0) * a.ld;
  const int shares = a.shares, outputs = a.outputs, per_token = a.top + a.always;
  const size_t slice = (size_t)a.rows * a.ld;
  float s[kPer], c[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) c[i] = a.correction ? a.correction[min(i * 64 + lane, outputs - 1)] : 0.f;
  // lane p: share p of the score of the experts that every token has
  const float gate_share = a.always > 0 && !a.always_plain && lane < shares ? z[lane * slice + outputs] : 0.f;
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int o = i * 64 + lane;
    const float* at = z + min(o, outputs - 1);
    float sum = at[0];
    if (shares > 1) {
      float part[kMaxShares];  // in flight together: with a branch around each the compiler lets them wait for each other
#pragma unroll
      for (int p = 1; p < kMaxShares; ++p) part[p] = at[(size_t)min(p, shares - 1) * slice];
#pragma unroll
      for (int p = 1; p < kMaxShares; ++p) sum += p < shares ? part[p] : 0.f;
    }
    s[i] = o < outputs ? sum : -INFINITY;
    mx = fmaxf(mx, s[i]);
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const bool is = i * 64 + lane < outputs;
    if (a.scores == NF_SCORES_SIGMOID) s[i] = is ? 1.f / (1.f + expf(-s[i])) : 0.f;
    else s[i] = is ? expf(s[i] - mx) : 0.f;
    sum += s[i];
  }
  sum = a.scores == NF_SCORES_SIGMOID ? 1.f : wave_sum(sum);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int o = i * 64 + lane;
    s[i] /= sum;
    c[i] = o < outputs ? s[i] + c[i] : -INFINITY;
  }
  if constexpr (kPer == 1) {
    // An output a lane: its rank is the number of those ahead of it, read lane by lane into scalar registers, and the wavefront needs neither LDS nor a chain of
    // `top` maxima.
    float mine = c[0] > -INFINITY ? c[0] : -INFINITY;  // what is no number is not chosen
    const int even = (outputs + 7) / 8 * 8;            // the lanes past the outputs are ahead of no one
    if (a.groups > 1) {
      const int size = outputs / a.groups, group = lane / size;
      float best = -INFINITY;
#pragma unroll 8
      for (int o = 0; o < even; ++o) {
        const float x = lane_value(mine, o);
        best = o >= group * size && o < group * size + size ? fmaxf(best, x) : best;
      }
      int ahead = 0;  // groups with a larger entry, or as large and before it
      for (int g = 0; g < a.groups; ++g) {
        const float x = lane_value(best, g * size);
        ahead += x > best || (x == best && g < group);
      }
      if (ahead >= a.keep_groups) mine = -INFINITY;
    }
    if (!live) return;
    int ahead = 0;  // larger scores, and as large ones before it
#pragma unroll 8
    for (int o = 0; o < even; ++o) {
      const float x = lane_value(mine, o);
      ahead += x > mine || (x == mine && o < lane);
    }
    const bool some = mine > -INFINITY;
    const int chosen = (int)__popcll(__ballot(some));
    if (some && ahead < a.top) {
      choice[(size_t)t * per_token + ahead] = lane;
      weight[(size_t)t * per_token + ahead] = s[0] * a.scale;
    }
    if (lane >= chosen && lane < a.top) {  // scores that are no numbers: a valid index all the same
      choice[(size_t)t * per_token + lane] = 0;
      weight[(size_t)t * per_token + lane] = 0.f * a.scale;
    }
  } else {
    if (a.groups > 1) {  // the same for every wavefront: the barriers are met by all
      const int size = outputs / a.groups;
#pragma unroll
      for (int i = 0; i < kPer; ++i) entry[wave][i * 64 + lane] = c[i];
      __syncthreads();
      for (int g = lane; g < a.groups; g += 64) {
        float b = entry[wave][g * size];
        for (int e = 1; e < size; ++e) b = fmaxf(b, entry[wave][g * size + e]);
        best_of[wave][g] = b;
      }
      __syncthreads();
      for (int g = lane; g < a.groups; g += 64) {
        const float b = best_of[wave][g];
        int ahead = 0;  // groups with a larger entry, or as large and before it
        for (int o = 0; o < a.groups; ++o) ahead += best_of[wave][o] > b || (best_of[wave][o] == b && o < g);
        entry[wave][g] = ahead < a.keep_groups ? 1.f : 0.f;
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int o = i * 64 + lane;
        if (o < outputs && entry[wave][o / size] == 0.f) c[i] = -INFINITY;
      }
    }
    if (!live) return;
    for (int k = 0; k < a.top; ++k) {
      float best = -INFINITY, w = 0.f;
      int at = 0x7fffffff;
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        if (c[i] > best) {  // the smallest of equal ones: i ascends
          best = c[i];
          at = i * 64 + lane;
          w = s[i];
        }
#pragma unroll
      for (int m = 32; m > 0; m >>= 1) {
        const float b2 = __shfl_xor(best, m, 64), w2 = __shfl_xor(w, m, 64);
        const int a2 = __shfl_xor(at, m, 64);
        if (b2 > best || (b2 == best && a2 < at)) {
          best = b2;
          at = a2;
          w = w2;
        }
      }
      if (at >= outputs) at = 0, w = 0.f;  // scores that are no numbers: a valid index all the same
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        if (i * 64 + lane == at) c[i] = -INFINITY;
      if (lane == 0) {
        choice[(size_t)t * per_token + k] = at;
        weight[(size_t)t * per_token + k] = w * a.scale;
      }
    }
  }
  float g = 0.f;
  for (int p = 0; p < shares; ++p) g += lane_value(gate_share, p);
  if (lane < a.always) {
    choice[(size_t)t * per_token + a.top + lane] = outputs + lane;
    weight[(size_t)t * per_token + a.top + lane] = a.always_plain ? 1.f : 1.f / (1.f + expf(-g));
  }
}

// The sum over a wavefront's lanes up to this one: within 16 lanes, then the last of 16 to the next 16, then the last of 32 to the next 32.
__device__ __forceinline__ int sum_to_lane(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
  return x + __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
}

// experts: of the grouped product, the last `always` of which have every token's row, in the tokens' order.
// What bounds it is what one CU can read and write, so every workgroup places a share of the entries, kPlanChunk at a time, all of which every workgroup
// counts: those ahead of its own apart from the rest (us, one workgroup for all -> this: 1946 rows of 5 10.8 -> 7.3, 2047 of 5 9.3 -> 6.8; 748
// rows of 5 5.4 -> 5.0, 256 of 5 4.7 and 4.7; an empty launch takes 4).
// held: for arrays that share memory with the choices or weights.  One workgroup, which has read both when it writes the sorted rows: they stay in LDS till then,
// up to kHeldEntries; an entry's place is written by the thread that has read the entry.
constexpr int kPlanChunk = 1024, kPlanGroups = 32, kHeldEntries = 16384;
__global__ __launch_bounds__(kPlanChunk) void route_plan_kernel(nf_routing r, int rows, int top, int always, int experts, bool held) {
  extern __shared__ int held_rows[];  // [n] rows, [n] weights
  __shared__ int ahead[kMaxOutputs], count[kMaxOutputs], first[kMaxOutputs], wave_rows[16], wave_tiles[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, routed = experts - always, per_token = top + always, n = rows * per_token;
  const int chunks = (n - 1) / kPlanChunk + 1, per_group = (chunks + gridDim.x - 1) / gridDim.x;
  const int c0 = min((int)blockIdx.x * per_group, chunks), c1 = min(c0 + per_group, chunks);
  int own = 0;
  float weight = 0.f;
  auto read_own = [&](int c) {
    const int i = min(c * kPlanChunk + tid, n - 1);
    own = r.choice[i];
    weight = r.weight[i];
  };
  if (c0 < c1) read_own(c0);
  ahead[tid] = 0;
  count[tid] = tid >= routed && tid < experts ? rows : 0;
  __syncthreads();
  constexpr int kAhead = 8;  // choices of a thread requested at once
  for (int c = 0; c < chunks; c += kAhead) {
    int e[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) e[k] = c + k < chunks ? r.choice[min((c + k) * kPlanChunk + tid, n - 1)] : experts;
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      if (c + k == chunks - 1 && tid >= n - (chunks - 1) * kPlanChunk) e[k] = experts;
      if (e[k] < routed) atomicAdd(c + k < c0 ? &ahead[e[k]] : &count[e[k]], 1);  // those of every token are past the outputs
    }
  }
  __syncthreads();
  // exclusive sums over the experts: rows, tiles
  const int before = ahead[tid], c = count[tid] + before, tiles = (c + r.tile_rows - 1) / r.tile_rows;
  int rows_to = sum_to_lane(c), tiles_to = sum_to_lane(tiles);
  if (lane == 63) {
    wave_rows[wave] = rows_to;
    wave_tiles[wave] = tiles_to;
  }
  __syncthreads();
  if (wave * 64 < experts)  // no one reads what the others have
    for (int w = 0; w < wave; ++w) {
      rows_to += wave_rows[w];
      tiles_to += wave_tiles[w];
    }
  first[tid] = rows_to - c + before;  // nobody's entries are ahead of another's at the experts of every token
  if (blockIdx.x == 0 && tid < experts) {
    const int tile0 = tiles_to - tiles;
    r.offsets[tid + 1] = rows_to;
    if (tid == 0) r.offsets[0] = 0;
    if (tid == experts - 1) *r.n_tiles = tiles_to;
    for (int i = 0; i < tiles; ++i) {
      r.tile_group[tile0 + i] = tid;
      r.tile_row[tile0 + i] = i * r.tile_rows;
    }
  }
  __syncthreads();
  for (int c = c0; c < c1; ++c) {
    const int i = c * kPlanChunk + tid;
    if (i < n) {
      const int t = i / per_token, k = i - t * per_token;
      int at = -1;
      if (k >= top) at = first[routed + k - top] + t;
      else if (own < routed) at = atomicAdd(&first[own], 1);
      if (at >= 0 && held) {
        held_rows[at] = t;
        held_rows[n + at] = (int)__float_as_uint(weight);
      } else if (at >= 0) {
        r.row_of[at] = t;
        if (r.row_weight) r.row_weight[at] = weight;
      }
      r.place[i] = at;
    }
    if (c + 1 < c1) read_own(c + 1);
  }
  if (held) {
    __syncthreads();
    int sorted = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) sorted += wave_rows[w];
    for (int i = tid; i < sorted; i += kPlanChunk) {
      r.row_of[i] = held_rows[i];
      if (r.row_weight) r.row_weight[i] = __uint_as_float((uint32_t)held_rows[n + i]);
    }
  }
}

}  // namespace nf

using namespace nf;

extern "C" {

int nf_routing_max_tiles(int sorted_rows, int experts, int tile_rows) {
  return sorted_rows > 0 && tile_rows > 0 ? sorted_rows / tile_rows + std::min(experts, sorted_rows) : 0;
}

int nf_route(const nf_route_args* args, const nf_routing* routing, nf_stream_t stream) {
  const char* who = "nf_route";
  NF_REQUIRE(args && routing, "%s: null pointer", who);
  const nf_route_args& a = *args;
  NF_REQUIRE(a.outputs > 0 && a.outputs <= kMaxOutputs && a.experts > 0 && a.experts <= a.outputs && a.top > 0 && a.always >= 0 &&
                 a.top <= a.outputs && a.top + a.always <= kMaxTop && a.experts + a.always <= kMaxOutputs,
             "%s: top %d and %d more of %d outputs, %d experts (at most %d outputs, %d per token)", who, a.top, a.always, a.outputs, a.experts,
             kMaxOutputs, kMaxTop);
  NF_REQUIRE(a.groups <= 1 || (a.outputs % a.groups == 0 && a.keep_groups > 0 && a.keep_groups <= a.groups &&
                               a.top <= a.outputs / a.groups * a.keep_groups),
             "%s: top %d of the outputs of %d of %d groups of %d", who, a.top, a.keep_groups, a.groups, a.outputs);
  const int per_token = a.top + a.always;
  NF_REQUIRE(a.rows >= 0 && (long long)a.rows * per_token < (1ll << 31) && a.ld >= a.outputs + (a.always > 0 && !a.always_plain) && a.shares >= 1 &&
                 a.shares <= kMaxShares && routing->tile_rows > 0,
             "%s: rows=%d ld=%d shares=%d tile_rows=%d", who, a.rows, a.ld, a.shares, routing->tile_rows);
  NF_REQUIRE(a.scores == NF_SCORES_SOFTMAX || a.scores == NF_SCORES_SIGMOID, "%s: unknown scores %d", who, a.scores);
  if (a.rows == 0) return NF_OK;
  const nf_routing& r = *routing;
  NF_REQUIRE(a.z && r.choice && r.weight && r.place && r.row_of && r.offsets && r.tile_group && r.tile_row && r.n_tiles, "%s: null pointer", who);
  hipStream_t s = (hipStream_t)stream;
  auto go = [&](auto per) {
    route_rows_kernel<decltype(per)::value><<<(a.rows + 3) / 4, 256, 0, s>>>(a, r.choice, r.weight);
    return check_launch(who);
  };
  const int per = (a.outputs + 63) / 64;
  const int rc = per <= 1 ? go(ic<1>{}) : per <= 2 ? go(ic<2>{}) : per <= 4 ? go(ic<4>{}) : per <= 8 ? go(ic<8>{}) : go(ic<16>{});
  if (rc) return rc;
  const size_t n = (size_t)a.rows * per_token;
  const long long chunks = (long long)(n + kPlanChunk - 1) / kPlanChunk;
  auto shares = [&](const void* out) {  // memory with what the plan reads
    auto over = [&](const void* in) { return out && (uintptr_t)out < (uintptr_t)in + n * 4 && (uintptr_t)in < (uintptr_t)out + n * 4; };
    return over(r.choice) || over(r.weight);
  };
  const bool alone = shares(r.place) || shares(r.row_of) || shares(r.row_weight), held = alone && n <= kHeldEntries;
  if (held) {
    static bool attr_set = false;  // benign race: the call is idempotent
    if (!attr_set) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(route_plan_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kHeldEntries * 8);
      if (e != hipSuccess) {
        set_error("%s: cannot reserve %d bytes of LDS: %s", who, kHeldEntries * 8, hipGetErrorString(e));
        return NF_ERR_RUNTIME;
      }
      attr_set = true;
    }
  }
  route_plan_kernel<<<alone ? 1u : (unsigned)std::min<long long>(chunks, kPlanGroups), kPlanChunk, held ? n * 8 : 0, s>>>(r, a.rows, a.top, a.always,
                                                                                                                        a.experts + a.always, held);
  return check_launch("nf_route (plan)");
}

}  // extern "C"
