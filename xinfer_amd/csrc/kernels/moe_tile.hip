// Routed experts' products for many rows an expert (prompt portions), bfloat16: tiles of up to 256 rows
// of one expert each, walked like the dense many-row product's (tile_core.h): rows and weights go into an LDS
// ring by loads that write LDS, whose lanes name their own addresses, so that the rows of a tile are read where they lie,
// through `order` in the first product and side by side in the second.
//
//   gated       out bfloat16 [P, N] = act(gate) * up: a wave's rows of w are gate rows and the up rows of the same
//               features, so that both sums of an element meet in a lane; one rounding
//   activated   out bfloat16 [P, N] = act(up)
//   plain       out float32 [P, N], rows in slot order
//
// An expert's rows are shared out evenly over its tiles, and a tile goes through the lowest of six walks (64 to 256 rows) that
// holds it; how high tiles may be is chosen on the device from the counts, for each product by its rounds of workgroups.
// (Tiles of one height for all, chosen from the average: 410 pairs an expert filled two of 256 to 80%, and 490 in four of
// 128 ran at 0.8 of the larger ones' rate.)  Both products and what stands around them, us, one height | this: 8 gated experts
// of 6144 at width 4096, 39 to 761 pairs each 584 | 539, 163 to 622 595 | 576, 410 596 | 552, 78 to 1,522 989 | 969, 512 584 | 570, 1,024
// 1,061 | 1,060; without a gate 130 to 634 519 | 457, 260 to 1,268 932 | 838, 1,536 1,116 | 1,161; 16 of 4096 at 2048, 512 each 302 | 290, 1,024 539 |
// 548, 156 to 3,044 919 | 983 (192 rows where 256 are ahead: the one load of 125 with more than 5% lost); 8 of 1536 at 1024, 1,024 each
// 113 | 104, 512 55 | 57.  (All of these with two stages of w in flight; with three 1 to 10% less: tile_core.h.)  What is left: rows past an expert's in
// the tiles (7%), the last round of workgroups, and 1.1 PFLOP/s in between where the dense walk has 1.4: a tile's w is shared by the few
// tiles of its expert.
//
// A workgroup owns a tile and BN rows of w; the number of tiles is known on the device alone, and the grid is the most
// there can be.  Nothing is read on the host.  (As many workgroups as compute units, each taking its die's next tile by a counter:
// level to 8% behind, 349 | 382 us at 30 to 200 pairs each: a tile then starts behind the counter's round trip.)
// The vendor library's products an expert, which were here before, came to 0.3 to 0.6 PFLOP/s at 200 to 500 rows, with a
// gather, an activation pass and a read of the row counts on the host around them.
#include "moe_act.h"
#include "moe_pairs.h"
#include "tile_core.h"

namespace xi {
namespace tile {

constexpr int kUnits = 256;
constexpr int kHeights = 5;
// heights that an expert's rows may be cut into, highest first, and the height of the walk that a tile of `rows` takes
__host__ __device__ constexpr int height(int i) { return i == 0 ? 256 : i == 1 ? 224 : i == 2 ? 192 : i == 3 ? 160 : 128; }
__device__ __forceinline__ int lowest(int rows) { return rows <= 64 ? 64 : rows <= 128 ? 128 : (rows + 31) & ~31; }
// a round's time, in rows: 1.95 us for 64 k of 256 rows, and what a tile costs beyond its products.  Measured with two stages of w in flight: since there are
// three, tiles of 192 rows and more take up to a tenth less and lower ones do not, which these prices do not know.
__device__ __forceinline__ int tile_time(int high) { return high + 16; }

// ceil(n / d), n and d > 0, of up to 2^22: the float quotient is one off at most (the compiler's division is three times as many instructions).
__device__ __forceinline__ int share(int n, int d) {
  const int m = n + d - 1;
  int q = (int)((float)m * __builtin_amdgcn_rcpf((float)d));
  const int left = m - q * d;
  q += left >= d ? 1 : left < 0 ? -1 : 0;
  return q;
}

// The pairs in the order of their experts, and the tiles of the two products: of product i up to high[i] rows (0: chosen here), an expert's all
// of one height but the last.  One workgroup, so a chain of dependent instructions: a wave a height, and divisions by a float's reciprocal (2,048
// pairs on 8 experts 8.8 us with all heights in every thread, 6.6 so; the sort alone, whose tiles were of one height, 4.3).
__global__ __launch_bounds__(kSortThreads) void moe_plan_kernel(const int* __restrict__ idx, int P, int E, int I, int high1, int high2,
                                                                int columns1, int columns2, int* __restrict__ order,
                                                                int* __restrict__ slot_of, int* __restrict__ tiles1,
                                                                int* __restrict__ tiles2, int most1, int most2) {
  __shared__ int count[kSortExperts], cursor[kSortExperts], across[3][kSortThreads / kWave];
  __shared__ float tiles_of[kHeights], time_of[kHeights];      // of every height: the tiles, and the mean time of one
  const int A = E + I, e = threadIdx.x, lane = e & 63, wave = e >> 6;
  moe_count_pairs(idx, P, A, count);
  const int pairs = e < A ? count[e] : 0, routed = e < E ? pairs : 0;
  int high[2] = {high1, high2};
  bool even[2] = {false, false};       // the tiles take about as long as the highest ones would
  if (high1 == 0 || high2 == 0) {
    for (int h = wave; h < kHeights; h += blockDim.x >> 6) {
      const int up_to = h == 0 ? height(0) : h == 1 ? height(1) : h == 2 ? height(2) : h == 3 ? height(3) : height(4);
      int t = 0, cost = 0;
      for (int x = lane; x < E; x += kWave) {
        const int n = share(count[x], up_to);
        t += n;
        cost += n ? n * tile_time(lowest(share(count[x], n))) : 0;
      }
      t += lane_xor<32>(t), cost += lane_xor<32>(cost);
      t += lane_xor<16>(t), cost += lane_xor<16>(cost);
      t += lane_xor<8>(t), cost += lane_xor<8>(cost);
      t += lane_xor<4>(t), cost += lane_xor<4>(cost);
      t += lane_xor<2>(t), cost += lane_xor<2>(cost);
      t += lane_xor<1>(t), cost += lane_xor<1>(cost);
      if (lane == 0) {
        tiles_of[h] = (float)t;
        time_of[h] = t ? (float)cost * __builtin_amdgcn_rcpf((float)t) : 0.f;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (high[i]) continue;
      float least = 0.f;
      const float columns = (float)(i ? columns2 : columns1) * (1.f / kUnits);
#pragma unroll
      for (int h = 0; h < kHeights; ++h) {
        const float cost = ceilf(tiles_of[h] * columns) * time_of[h];
        if (h == 0 || cost < least) {
          least = cost;
          high[i] = height(h);
          even[i] = time_of[h] >= 0.97f * (float)tile_time(height(h));
        }
      }
    }
  }
  const int n1 = routed ? share(routed, high[0]) : 0, n2 = routed ? share(routed, high[1]) : 0;
  int before[3] = {pairs, n1, n2};
  int busy = 0;
  if (high[0] == high[1] && high[0] <= 64) {        // the same list twice, and one order for all (8 pairs on 1,000 experts, a layer: 17.4 -> 16.6 us)
    int both[2] = {pairs, n1};
    moe_sums_before(both, A, across);
    before[0] = both[0], before[1] = before[2] = both[1];
  } else {
    moe_sums_before(before, A, across);
    busy = __syncthreads_count(routed > 0);
  }
  if (e == A - 1) {
    tiles1[5 * most1] = before[1] + n1;
    tiles2[5 * most2] = before[2] + n2;
    tiles1[5 * most1 + 1] = 2 * (before[1] + n1) > 3 * busy ? 1 + even[0] : 0;
    tiles2[5 * most2 + 1] = 2 * (before[2] + n2) > 3 * busy ? 1 + even[1] : 0;
  }
  if (e < A) cursor[e] = before[0];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int n = i ? n2 : n1, rows = n ? share(routed, n) : 0, most = i ? most2 : most1;
    int* to = (i ? tiles2 : tiles1) + before[1 + i];
    for (int t = 0; t < n; ++t) {
      to[t] = e;
      to[most + t] = before[0] + t * rows;
      to[2 * most + t] = routed - t * rows < rows ? routed - t * rows : rows;
      to[3 * most + t] = before[1 + i];
      to[4 * most + t] = n;
    }
  }
  moe_place_pairs(idx, P, A, cursor, order, slot_of);
}

// One tile: BM rows of x by BN rows of w (gated: BN / 2 features), rings of S and SW stages.
template <int BM, int BN, int S, int SW, int FORM, int ACT, int WGM = 2, int WGN = 4>
__device__ __forceinline__ void moe_one_tile(const bf16* __restrict__ x, const int* __restrict__ order, int top,
                                             const bf16* __restrict__ w, int e, int row0, int rows, int tn_i, void* __restrict__ out,
                                             int N, int K, const float* __restrict__ in_wt, unsigned char* smem) {
  constexpr bool GATED = FORM == 1, GATHER = FORM != 0;
  using W = Walk<BM, BN, WGM, WGN, S, SW>;
  constexpr int TM = W::TM, TN = W::TN;
  constexpr int TF = GATED ? TN / 2 : TN, WF = 16 * TF;            // 16-feature tiles of a wave, and its features
  static_assert(!GATED || TN % 2 == 0, "half of a wave's rows of w are gate rows");
  // (opaque, so that nothing made from them is made in front of the choice between the walks and held in registers through all)
  asm volatile("" : "+s"(row0), "+s"(rows), "+s"(tn_i));
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, j = lane >> 4;
  const int wm = wave % WGM, wn = wave / WGM;
  const int f0 = tn_i * (WGN * WF);                                  // the first feature
  unsigned ld_off[W::LPW];
  W::offsets(ld_off, [&](bool is_w, int p) {
    int row;
    if (is_w) {
      int f = GATED ? f0 + WF * (p / (2 * WF)) + p % WF : f0 + p;
      f = f < N ? f : N - 1;
      row = GATED && (p & WF) ? N + f : f;
    } else {
      const int slot = row0 + (p < rows ? p : rows - 1);
      row = GATHER ? order[slot] / top : slot;
    }
    return (unsigned)((size_t)row * K * 2);
  });
  f32x4 acc[TN][TM];
  W::run(w + (size_t)e * (GATED ? 2 : 1) * N * K, x, ld_off, K / 64, smem, acc);
  typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
#pragma unroll
  for (int b = 0; b < TM; ++b) {
    const int m = (wm * TM + b) * 16 + r;
    if (m >= rows) continue;
    const int slot = row0 + m;
    // a weight on the expert's INPUT: the products are linear, so it multiplies their sums before the activation
    const float wi = (GATHER && in_wt) ? in_wt[order[slot]] : 1.f;
#pragma unroll
    for (int a = 0; a < TF; ++a) {
      const int n = f0 + WF * wn + 16 * a + 4 * j;
      if (n >= N) continue;                    // (N is a multiple of 4)
      if (FORM == 0) {
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(out) + (size_t)slot * N + n) = acc[a][b];
      } else {
        bf16x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = moe_act_m<ACT>(wi * acc[a][b][i]);
          o[i] = (__bf16)(GATED ? v * (wi * acc[GATED ? TF + a : a][b][i]) : v);
        }
        *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(out) + (size_t)slot * N + n) = o;
      }
    }
  }
}

// Rows of w and stages of the tiles of up to 16 rows: two workgroups of four waves a compute unit, 70 KB on their way each.  Decode steps are
// bound by the stream of the touched experts' weights: with tiles of 64 rows a third of what came into LDS was copies of the few rows of x, one
// workgroup a compute unit left a gap at every round's start, and columns of 128 features of the down product were fewer than the compute
// units.  16 pairs on 8 gated experts of 6144 at width 4096 219 -> 206 us, without a gate 167 -> 148; 8 on 16 of 4096 at 2048 68 -> 57.
constexpr int few_wide(int form) { return form == 1 ? 128 : 64; }
constexpr int few_stages(int form) { return form == 1 ? 4 : 7; }

// HIGH 64: tiles of up to 64 rows by 128 rows of w; 16: of up to 16 rows by 64 features; 0: of up to 256 by 256, each in the lowest walk that
// holds it.
template <int HIGH, int FORM, int ACT>
__global__ __launch_bounds__(HIGH == 16 ? 256 : 512, HIGH == 16 ? 2 : 1) void moe_tile_kernel(const bf16* __restrict__ x, const int* __restrict__ order, int top,
                                                          const bf16* __restrict__ w, const int* __restrict__ tiles, int most,
                                                          void* __restrict__ out, int N, int K, int columns,
                                                          const float* __restrict__ in_wt) {
  extern __shared__ __align__(1024) unsigned char smem[];
  const int n_tiles = tiles[5 * most], die = blockIdx.x & 7, in_die = blockIdx.x >> 3;
  int tile, column;
  // the place `place` of those of the experts' tiles with `width` columns: an expert's lie together, its tiles innermost
  auto find = [&](int place, int width) {
    const int some = place / width, first = tiles[3 * most + some], count = tiles[4 * most + some], q = place - first * width;
    column = q / count;
    tile = first + (q - column * count);
  };
  const int order_of = HIGH ? 2 : tiles[5 * most + 1];
  if (order_of == 2) {
    // Consecutive places a die, an expert after the other: a die's L2 holds an expert's rows and the rows of w that its tiles share.  For
    // tiles that take about as long as each other (within 3%, the list says): 16 experts of 4096 at width 2048, 1,024 rows each 577 us the other way,
    // 547 so, 2,048 each 1,139 and 1,075; 8 gated ones of 1536 at width 1024, 1,024 each 114 and 108.
    const int total = n_tiles * columns, per_die = (total + 7) >> 3, place = die * per_die + in_die;
    if (in_die >= per_die || place >= total) return;
    find(place, columns);
  } else {
    // Tiles of unequal height: every die gets the same columns of all experts, so that the heights come out even over the dies; columns that do
    // not share out go round in tiles, and so do all where few experts have a second tile to share w with (64 rows an expert
    // 290 us in that order, 310 an expert after the other).
    const int whole = order_of == 1 ? columns >> 3 : 0, rest = columns - 8 * whole;
    if (in_die < whole * n_tiles) {
      find(in_die, whole);
      column += die * whole;
    } else {
      const int per_die = (rest * n_tiles + 7) >> 3, i = in_die - whole * n_tiles, place = die * per_die + i;
      if (i >= per_die || place >= rest * n_tiles) return;
      column = place / n_tiles;
      tile = place - column * n_tiles;
      column += 8 * whole;
    }
  }
  const int e = tiles[tile], row0 = tiles[most + tile], rows = tiles[2 * most + tile];
#define XI_ONE(BM, BN, S, SW) moe_one_tile<BM, BN, S, SW, FORM, ACT>(x, order, top, w, e, row0, rows, column, out, N, K, in_wt, smem)
  if constexpr (HIGH == 16) {
    moe_one_tile<16, few_wide(FORM), few_stages(FORM), few_stages(FORM), FORM, ACT, 1, 4>(x, order, top, w, e, row0, rows, column, out, N, K, in_wt, smem);
  } else if constexpr (HIGH == 64) {
    XI_ONE(64, 128, 6, 6);
  } else {
    if (rows > 224) XI_ONE(256, 256, 2, 3);
    else if (rows > 192) XI_ONE(224, 256, 2, 3);
    else if (rows > 160) XI_ONE(192, 256, 2, 3);
    else if (rows > 128) XI_ONE(160, 256, 3, 3);
    else if (rows > 64) XI_ONE(128, 256, 3, 3);
    else XI_ONE(64, 256, 3, 4);
  }
#undef XI_ONE
}

}  // namespace tile
}  // namespace xi

using namespace xi;

extern "C" {

int xi_moe_tiles_most(int P, int E, int bm);         // moe_mfma.hip

// Sizes that `xi_moe_tile` takes: K in whole tiles of 64, N in fours, offsets within an expert's weights and within the rows
// (rows_x of K) in 32 bits.
int xi_moe_tile_takes(long long rows_x, int N, int K, int gated) {
  return rows_x > 0 && N > 0 && N % 4 == 0 && K > 0 && K % 64 == 0 && rows_x * K * 2 < (1LL << 32) &&
         (gated ? 2LL : 1LL) * N * K * 2 < (1LL << 32);
}

// idx int32 [P] (expert of every pair; E .. E + I - 1: identity experts) -> order, slot_of int32 [P] and the tiles of the two products, int32
// [5 most + 2] each: expert, first slot and rows of each, the first tile of its expert and how many that has, how many there are in all, and
// their order over the dies, for tiles of more than 64 rows in either product: 0 up to one and a half an expert with any, 2 where they are of
// about one height, 1 otherwise.  high: most rows of a tile, 0: chosen from the counts on the
// device, of 128 to 256, for that many columns of workgroups; most: xi_moe_tiles_most for high or for 128.
int xi_moe_plan(const int* idx, int P, int E, int I, int high1, int high2, int columns1, int columns2, int* order, int* slot_of, int* tiles1,
                int* tiles2, int most1, int most2, hipStream_t stream) {
  auto fits = [](int h) { return h == 0 || h == 16 || h == 64 || h == 128 || h == 256; };
  XI_CHECK(P > 0 && E > 0 && I >= 0 && E + I <= kSortExperts && fits(high1) && fits(high2) && columns1 > 0 && columns2 > 0,
           "moe_plan: bad sizes pairs=%d experts=%d rows=%d, %d", P, E, high1, high2);
  XI_CHECK(most1 >= xi_moe_tiles_most(P, E, high1 ? high1 : 128) && most2 >= xi_moe_tiles_most(P, E, high2 ? high2 : 128),
           "moe_plan: too few tiles");
  tile::moe_plan_kernel<<<1, moe_sort_threads(P, E + I), 0, stream>>>(idx, P, E, I, high1, high2, columns1, columns2, order, slot_of, tiles1, tiles2,
                                                        most1, most2);
  XI_LAUNCH_CHECK("moe_plan");
  return 0;
}

// Columns of workgroups of a product of N features in tiles of up to `high` rows (0: chosen on the device).
int xi_moe_tile_columns(int N, int high, int gated) {
  const int features = high == 16 ? 64 : (high == 64 ? 128 : 256) / (gated ? 2 : 1);
  return (N + features - 1) / features;
}

// The operands of `xi_moe_group` (moe_mfma.hip) for the tiles of `xi_moe_plan` with this `high`; rows_x: rows of A.
int xi_moe_tile(const void* A, long long rows_x, const int* order, int top, const void* W, const int* tiles, int most, void* out,
                int N, int K, int high, int form, int act, const float* in_wt, hipStream_t stream) {
  XI_CHECK(xi_moe_tile_takes(rows_x, N, K, form == 1) && top > 0 && most > 0 && (high == 0 || high == 16 || high == 64 || high == 128 || high == 256),
           "moe_tile: bad sizes N=%d K=%d top=%d tiles=%d rows=%d", N, K, top, most, high);
  XI_CHECK(act >= 0 && act <= 2 && form >= 0 && form <= 2, "moe_tile: unknown activation %d or form %d", act, form);
  XI_CHECK(tiles && order, "moe_tile: an operand is missing");
  auto on16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  XI_CHECK(on16(A) && on16(W) && on16(out), "moe_tile: operands must start on 16 bytes");
  const int columns = xi_moe_tile_columns(N, high, form == 1);
  XI_CHECK((long long)most * columns <= 0x3fffffffLL, "moe_tile: too many tiles");
  const long long places = 8 * ((long long)most * (columns / 8) + ((long long)most * (columns % 8) + 7) / 8);
  const unsigned wgs = (unsigned)(high == 64 || high == 16 ? ((long long)most * columns + 7) / 8 * 8 : places);
#define XI_MT(HIGH, FORM, ACT)                                                                                              \
  do {                                                                                                                      \
    auto kern = tile::moe_tile_kernel<HIGH, FORM, ACT>;                                                                      \
    const size_t lds = HIGH == 16 ? tile::Walk<16, tile::few_wide(FORM), 1, 4, tile::few_stages(FORM)>::LDS                  \
                       : HIGH ? tile::Walk<64, 128, 2, 4, 6>::LDS : tile::Walk<256, 256, 2, 4, 2, 3>::LDS;                     \
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);      \
    XI_CHECK(e == hipSuccess, "moe_tile: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));                      \
    kern<<<wgs, HIGH == 16 ? 256 : 512, lds, stream>>>((const bf16*)A, order, top, (const bf16*)W, tiles, most, out, N, K, columns, in_wt); \
  } while (0)
#define XI_MT_FORM(HIGH)                                \
  do {                                                  \
    if (form == 0) XI_MT(HIGH, 0, 0);                    \
    else if (form == 1 && act == 0) XI_MT(HIGH, 1, 0);   \
    else if (form == 1 && act == 1) XI_MT(HIGH, 1, 1);   \
    else if (form == 1) XI_MT(HIGH, 1, 2);               \
    else if (act == 0) XI_MT(HIGH, 2, 0);                \
    else if (act == 1) XI_MT(HIGH, 2, 1);                \
    else XI_MT(HIGH, 2, 2);                              \
  } while (0)
  if (high == 16) XI_MT_FORM(16);
  else if (high == 64) XI_MT_FORM(64);
  else XI_MT_FORM(0);
#undef XI_MT_FORM
#undef XI_MT
  XI_LAUNCH_CHECK("moe_tile");
  return 0;
}

}  // extern "C"
