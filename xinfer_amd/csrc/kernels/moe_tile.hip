// Routed experts' products for many rows an expert (prompt portions), bfloat16: the tiles of `moe_sort` (moe_mfma.hip),
// up to BM rows of one expert each, walked like the dense many-row product's (tile_core.h): rows and weights go into an LDS
// ring by loads that write LDS, whose lanes name their own addresses, so that the rows of a tile are read where they lie,
// through `order` in the first product and side by side in the second.
//
//   gated       out bfloat16 [P, N] = act(gate) * up: a wave's rows of w are gate rows and the up rows of the same
//               features, so that both sums of an element meet in a lane; one rounding
//   activated   out bfloat16 [P, N] = act(up)
//   plain       out float32 [P, N], rows in slot order
//
// A workgroup owns a tile and BN rows of w.  Workgroups of one die get consecutive places in the order (expert, rows of
// w, tile), so that its L2 holds what they share; the number of tiles is known on the device alone, and the grid is the most
// there can be.  Nothing is read on the host.
// The vendor library's products an expert, which were here before, came to 0.3 to 0.6 PFLOP/s at 200 to 500 rows, with a
// gather, an activation pass and a read of the row counts on the host around them.
#include "moe_act.h"
#include "tile_core.h"

namespace xi {
namespace tile {

// BM rows of x by BN rows of w (gated: BN / 2 features), a ring of S stages.
template <int BM, int BN, int S, int FORM, int ACT>
__global__ __launch_bounds__(512, 1) void moe_tile_kernel(const bf16* __restrict__ x, const int* __restrict__ order, int top,
                                                          const bf16* __restrict__ w, const int* __restrict__ tile_expert,
                                                          const int* __restrict__ tile_row0, const int* __restrict__ tile_rows,
                                                          const int* __restrict__ n_tiles, const int* __restrict__ tile_first,
                                                          const int* __restrict__ tile_count, void* __restrict__ out, int N, int K,
                                                          int tiles_n, int parts, const float* __restrict__ in_wt) {
  constexpr bool GATED = FORM == 1, GATHER = FORM != 0;
  constexpr int WGM = 2, WGN = 4;
  using W = Walk<BM, BN, WGM, WGN, S>;
  constexpr int TM = W::TM, TN = W::TN;
  constexpr int TF = GATED ? TN / 2 : TN, WF = 16 * TF;            // 16-feature tiles of a wave, and its features
  static_assert(TN % 2 == 0, "half of a wave's rows of w are gate rows");
  extern __shared__ __align__(1024) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, j = lane >> 4;
  const int wm = wave % WGM, wn = wave / WGM;
  const int total = *n_tiles * parts * tiles_n, per_die = (total + 7) >> 3;
  const int in_die = blockIdx.x >> 3, place = (blockIdx.x & 7) * per_die + in_die;
  if (in_die >= per_die || place >= total) return;
  // the places of an expert's tiles lie together: those of a tile's expert are first * parts * tiles_n and on
  const int some = place / tiles_n / parts, first = tile_first[some] * parts, count = tile_count[some] * parts;
  const int q = place - first * tiles_n, tn_i = q / count, piece = first + (q - tn_i * count), tile = piece / parts;
  const int skip = (piece - tile * parts) * BM;                      // this part's rows of the tile
  const int e = tile_expert[tile], row0 = tile_row0[tile] + skip, rows = tile_rows[tile] - skip;
  if (rows <= 0) return;
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
    if (m >= rows) continue;                   // (rows may go on in the tile's next part: m < BM)
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

}  // namespace tile
}  // namespace xi

using namespace xi;

extern "C" {

// Sizes that `xi_moe_tile` takes: K in whole tiles of 64, N in fours, offsets within an expert's weights and within the rows
// (rows_x of K) in 32 bits.
int xi_moe_tile_takes(long long rows_x, int N, int K, int gated) {
  return rows_x > 0 && N > 0 && N % 4 == 0 && K > 0 && K % 64 == 0 && rows_x * K * 2 < (1LL << 32) &&
         (gated ? 2LL : 1LL) * N * K * 2 < (1LL << 32);
}

// The operands of `xi_moe_group` (moe_mfma.hip) for tiles of bm = 64, 128 or 256 rows, with the tiles' `first` and `count` of `xi_moe_sort`;
// rows_x: rows of A.  parts: a tile of `xi_moe_sort` has parts * bm rows at most and is that many workgroups' (bm: of one).
int xi_moe_tile(const void* A, long long rows_x, const int* order, int top, const void* W, const int* tile_expert, const int* tile_row0,
                const int* tile_rows, const int* n_tiles, const int* tile_first, const int* tile_count, int tiles_most, void* out, int N,
                int K, int bm, int parts, int form, int act, const float* in_wt, hipStream_t stream) {
  XI_CHECK(xi_moe_tile_takes(rows_x, N, K, form == 1) && top > 0 && tiles_most > 0 && (bm == 64 || bm == 128 || bm == 256) && parts >= 1 && parts <= 4,
           "moe_tile: bad sizes N=%d K=%d top=%d tiles=%d rows=%d", N, K, top, tiles_most, bm);
  XI_CHECK(act >= 0 && act <= 2 && form >= 0 && form <= 2, "moe_tile: unknown activation %d or form %d", act, form);
  XI_CHECK(tile_first && tile_count && n_tiles && order, "moe_tile: an operand is missing");
  auto on16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  XI_CHECK(on16(A) && on16(W) && on16(out), "moe_tile: operands must start on 16 bytes");
  const int bn = bm == 64 ? 128 : 256, features = form == 1 ? bn / 2 : bn;
  const int tiles_n = (N + features - 1) / features;
  const long long wgs = ((long long)tiles_most * parts * tiles_n + 7) / 8 * 8;
  XI_CHECK(wgs <= 0x7fffffffLL, "moe_tile: too many workgroups");
#define XI_MT(BM, BN, S, FORM, ACT)                                                                                         \
  do {                                                                                                                      \
    auto kern = tile::moe_tile_kernel<BM, BN, S, FORM, ACT>;                                                                \
    const size_t lds = tile::Walk<BM, BN, 2, 4, S>::LDS;                                                                    \
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);      \
    XI_CHECK(e == hipSuccess, "moe_tile: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));                      \
    kern<<<(unsigned)wgs, 512, lds, stream>>>((const bf16*)A, order, top, (const bf16*)W, tile_expert, tile_row0, tile_rows, \
                                              n_tiles, tile_first, tile_count, out, N, K, tiles_n, parts, in_wt);           \
  } while (0)
#define XI_MT_FORM(...)                                        \
  do {                                                         \
    if (form == 0) XI_MT(__VA_ARGS__, 0, 0);                   \
    else if (form == 1 && act == 0) XI_MT(__VA_ARGS__, 1, 0);  \
    else if (form == 1 && act == 1) XI_MT(__VA_ARGS__, 1, 1);  \
    else if (form == 1) XI_MT(__VA_ARGS__, 1, 2);              \
    else if (act == 0) XI_MT(__VA_ARGS__, 2, 0);               \
    else if (act == 1) XI_MT(__VA_ARGS__, 2, 1);               \
    else XI_MT(__VA_ARGS__, 2, 2);                             \
  } while (0)
  if (bm == 64) XI_MT_FORM(64, 128, 6);
  else if (bm == 128) XI_MT_FORM(128, 256, 3);
  else XI_MT_FORM(256, 256, 2);
#undef XI_MT_FORM
#undef XI_MT
  XI_LAUNCH_CHECK("moe_tile");
  return 0;
}

}  // extern "C"
