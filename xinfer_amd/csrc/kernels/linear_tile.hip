// y[M, N] = x[M, K] @ w[N, K]^T in bfloat16 for many rows (prompt portions, decode steps of more
// than 128 requests) on the gfx950 matrix cores, with split K for narrow outputs.
//
// The vendor library serves these products well where the output gives it as many tiles as the
// chip has compute units; a narrow output does not (2,048 rows by 4,096 features are 128 of its
// tiles for 256 units, 256 rows 16), and its own choice of kernel does not cut K.  Here a workgroup
// of eight waves owns a tile of BM rows by BN features (128 by 256, 256 by 128, or 256 by 256) and
// one of KS slices of K, tiles x slices filling the compute units; with slices the result is
// float32 partial sums [KS, M, N] that the consumer adds in slice order (the fused add + RMSNorm,
// the q/k kernel), without them one bfloat16 rounding of the float32 sum.
//
// Tiles of 64 k reach LDS through loads that write LDS themselves (`global_load_lds_dwordx4`:
// every lane asks for one 16-byte chunk, a wave's 64 chunks land in 1 KB of consecutive LDS, no
// register holds a tile), into rings of two or three stages of x and three or more of w (160 KB of
// LDS: tile_core.h); a tile is waited for with a count, not by draining the queue, and one barrier a tile orders
// the stage's reuse.  Rows of 128 bytes cannot be padded then, so the 16-byte chunks of row p are
// permuted: chunk c sits at place c ^ ((p >> 1) & 7), and the 16 lanes that read an operand together
// (16 rows, one chunk each) fall into 16 different 16-byte groups of the 64 banks (the counters
// show no bank conflict).
//
// A wave multiplies 64 features by 64 rows (128 rows in the tile of 256 by 256) as 4 x 4 (4 x 8)
// v_mfma_f32_16x16x32_bf16 tiles per 32-wide k step: A = 16 rows of w, B = 16 rows of x, so that a
// lane holds four consecutive features of one row of the result.  The operands of a tile's two
// steps live in two sets of registers, each read from LDS while the matrix cores work on the other
// set, and both these reads and the loads of the tile S ahead are issued one at a time between the products: a wave that
// asks for all its loads at once waits until the load unit has taken them before it issues its
// first product (5 to 10% of the kernel's time).
//
// Measured on MI355X (random operands, the clock under load about 1.8 GHz): 2,048 rows by
// N = 4096, K = 12288 in 172 us (1.2 PFLOP/s; the library 174), K = 4096 in 68 us (the library 64);
// 4,096 x 4,096 x 4,096 in tiles of 256 by 256 102 us (1.35; the library 92), operands in a cache: the matrix cores are
// busy 63% of the time, LDS serves the tiles' 48 to 64 KB of writes and 128 to 192 KB of reads a
// tile (without the barrier or without the wait for the loads it is no faster).  With weights from memory, as in a model, what
// bounds it is how long they have been asked for when they are wanted (tile_core.h).  Where it is ahead of the library is the narrow output at few rows, whose tiles
// leave most of the chip idle unless K is cut: 256 rows of N = 4096, K = 12288 in 30 us against 41.
// A long K whose output is less than a round of such tiles (down projections of 1,025 to 2,688 rows) goes in the lowest tiles that
// still are one round, 96 to 224 rows by 256 features: 1,727 rows of N = 5120, K = 17408 in 11 x 20 tiles of 160 rows 255 to 261 us
// (1.2 PFLOP/s, its loads into LDS at 57 GB/s a compute unit, which bounds tiles up to that height), the library 473; 256 rows 401;
// four slices of 128 rows 309 and the reader's four float32 parts.
// Not kept: the tiles' k shared out evenly over the compute units, whoever comes last at a tile adding up its parts (345 us there:
// workgroups at different places of K share nothing in L2, and the parts go through memory); v_mfma_f32_32x32x16_bf16 (4,096 cubed 114
// us); a ring of five stages of 32 k (113); tiles of 32 k with two workgroups a compute unit (0.85 PFLOP/s against 0.95 at 4,096
// cubed); the tiles going memory -> registers -> LDS (0.83); four waves of twice the tile each
// (0.80, and 7% behind with the reads between the products); the operands of one step only in registers (the second step's reads then wait: -8%).
//
// Products of a few MB at up to 1,024 rows (and any of one round of them: `kernels.small_tile_plan`) go in tiles of 64 x 64, 64 x 128 or 128 x 128 with
// rings of four to eight stages: a workgroup has 128 to 144 KB on their way from its first clocks on, which for 512 k of 64 x 64 is all it
// will need, and the time is a kernel's start, one way to memory and the results' way out.  With slices of K the reader adds partial sums.
// Rows, N, K, us, weights from memory, the library | the tiles for 128 rows a block (linear_mid) | this: 256, 1024, 2048 8.4 | 15.6 | 5.8 (four
// slices of 64 x 64), 256, 1024, 3072 9.7 | 16.6 | 7.3, 256, 4096, 1024 12.0 | 17.1 | 8.1 (whole), 512, 2048, 4096 21.7 | - | 15.8 (20.1 in six slices of
// 256 x 256), 1024, 1024, 1024 8.9 | - | 6.9, 128, 1024, 2048 8.5 | 8.1 | 4.7, 64, 1024, 1024 8.5 | 5.0 | 4.3.
//
// Workgroups go round the chip's eight dies; consecutive workgroup numbers of one die are mapped
// to tiles that share rows of w, then of x, so that a die's L2 holds what its workgroups share.
// The value of an output element depends on (K, the slices) alone: never on M, on the tile shape or
// on what else is in the batch (a sum over a slice runs in ascending k, 32 at a time).
//
// Reference call site: candle matmul in /root/reference/src/models/layers/linear.rs:76-124
// (vendor BLAS).
#include "moe_act.h"
#include "tile_core.h"

namespace xi {
namespace tile {

constexpr int kSliceK = 64;        // K is cut into slices in tiles of this many

// BM rows of x by BN rows of w a workgroup; see Walk.
template <int BM, int BN, int WGM, int WGN, int S, int SW, bool PARTIAL>
__global__ __launch_bounds__(64 * WGM * WGN, 1) void linear_tile_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ w, void* __restrict__ yv, int M, int N, int K, int tiles_m,
    int tiles_n, int slices, int k_tiles_all) {
  using W = Walk<BM, BN, WGM, WGN, S, SW>;
  constexpr int TM = W::TM, TN = W::TN;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, j = lane >> 4;
  const int wm = wave % WGM, wn = wave / WGM;

  // ---- which tile and slice: workgroup numbers b, b + 8, b + 16, .. run on one die; they get
  // consecutive places in the order (slice, tile of features, tile of rows)
  const int total = tiles_m * tiles_n * slices;
  const int q8 = total >> 3, r8 = total & 7, die = blockIdx.x & 7;
  const int place = die * q8 + (die < r8 ? die : r8) + (blockIdx.x >> 3);
  const int per_slice = tiles_m * tiles_n;
  const int slice = place / per_slice;
  const int in_slice = place - slice * per_slice;
  const int tn_i = in_slice / tiles_m, tm_i = in_slice - tn_i * tiles_m;
  const int m0 = tm_i * BM, n0 = tn_i * BN;
  // slice s of the K / 64 tiles: [s * tiles / slices, (s + 1) * tiles / slices), one tile at least
  const int kt_begin = (int)((long long)slice * k_tiles_all / slices);
  const int k_tiles = (int)((long long)(slice + 1) * k_tiles_all / slices) - kt_begin;
  const size_t k0 = (size_t)kt_begin * kSliceK;

  unsigned ld_off[W::LPW];
  W::offsets(ld_off, [&](bool is_w, int p) {      // (rows past the end: the last row)
    const int first = is_w ? n0 : m0, last = (is_w ? N : M) - 1;
    const int row = first + p > last ? last : first + p;
    return (unsigned)(((size_t)(row - first) * K) * 2);
  });
  f32x4 acc[TN][TM];
  W::run(w + (size_t)n0 * K + k0, x + (size_t)m0 * K + k0, ld_off, k_tiles, smem, acc);

  // ---- a lane holds features n .. n + 3 of row m of every 16 x 16 tile
  const int mw = m0 + wm * TM * 16 + r, nw = n0 + wn * TN * 16 + 4 * j;
#pragma unroll
  for (int b = 0; b < TM; ++b) {
    const int m = mw + 16 * b;
    if (m >= M) continue;
#pragma unroll
    for (int a = 0; a < TN; ++a) {
      const int n = nw + 16 * a;
      if (n >= N) continue;          // (N is a multiple of 4)
      const f32x4 v = acc[a][b];
      if (PARTIAL) {
        float* y = reinterpret_cast<float*>(yv) + ((size_t)slice * M + m) * N + n;
        *reinterpret_cast<f32x4*>(y) = v;
      } else {
        bf16* y = reinterpret_cast<bf16*>(yv) + (size_t)m * N + n;
        typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
        bf16x4 o;
        o[0] = (__bf16)v[0];
        o[1] = (__bf16)v[1];
        o[2] = (__bf16)v[2];
        o[3] = (__bf16)v[3];
        *reinterpret_cast<bf16x4*>(y) = o;
      }
    }
  }
}

// The feed-forward's first product with its activation (in place of a product of 2 N features, a pass that reads them again and
// writes half, and their two launches): w [2 N, K] = [gate; up], y bfloat16 [M, N] = act(gate) * up of the
// float32 sums, one rounding.  A workgroup owns BM rows of x and BN / 2 features; a wave's rows of w are gate rows and the up
// rows of the same features (as in moe_tile.hip).  Bound by the walk, as above, and by how evenly the tiles fill rounds of 256
// workgroups; measured at N=17408, K=5120 against the library and the activation's pass: 1,024 rows 288 us (1.27 PFLOP/s) / 408,
// 2,048 rows 537 / 619; at N=3072, K=1024: 256 rows in tiles of 64 by 64 9.3 / 16.9, 1,024 in 128 by 128 17.3 / 22.8, 2,048 in
// 256 by 128 27.5 / 35.2.
template <int BM, int BN, int S, int SW, int ACT>
__device__ __forceinline__ void gated_tile(const bf16* x, const bf16* w, bf16* y, int M, int N, int K, int m0, int f0, unsigned char* smem) {
  constexpr int WGM = 2, WGN = 4;
  using W = Walk<BM, BN, WGM, WGN, S, SW>;
  constexpr int TM = W::TM, TN = W::TN, TF = TN / 2, WF = 16 * TF;
  static_assert(TN % 2 == 0, "half of a wave's rows of w are gate rows");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, j = lane >> 4;
  const int wm = wave % WGM, wn = wave / WGM;
  unsigned ld_off[W::LPW];
  W::offsets(ld_off, [&](bool is_w, int p) {
    int row;
    if (is_w) {
      int f = f0 + WF * (p / (2 * WF)) + p % WF;
      f = f < N ? f : N - 1;
      row = (p & WF) ? N + f : f;
    } else {
      row = m0 + p < M ? m0 + p : M - 1;
    }
    return (unsigned)((size_t)row * K * 2);
  });
  f32x4 acc[TN][TM];
  W::run(w, x, ld_off, K / kSliceK, smem, acc);
  typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
#pragma unroll
  for (int b = 0; b < TM; ++b) {
    const int m = m0 + (wm * TM + b) * 16 + r;
    if (m >= M) continue;
#pragma unroll
    for (int a = 0; a < TF; ++a) {
      const int n = f0 + WF * wn + 16 * a + 4 * j;
      if (n >= N) continue;                    // (N is a multiple of 4)
      bf16x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = (__bf16)(moe_act_m<ACT>(acc[a][b][i]) * acc[TF + a][b][i]);
      *reinterpret_cast<bf16x4*>(y + (size_t)m * N + n) = o;
    }
  }
}

// Tiles of BM rows by BN / 2 features, the rows innermost.  Workgroup numbers of one die get consecutive places: its L2 holds the
// rows of w they share.
template <int BM, int BN, int S, int SW, int ACT>
__global__ __launch_bounds__(512, 1) void gated_tile_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                            bf16* __restrict__ y, int M, int N, int K, int tiles_m) {
  extern __shared__ __align__(1024) unsigned char smem[];
  const int total = gridDim.x, q8 = total >> 3, r8 = total & 7, die = blockIdx.x & 7;
  const int place = die * q8 + (die < r8 ? die : r8) + (blockIdx.x >> 3);
  const int tn_i = place / tiles_m;
  gated_tile<BM, BN, S, SW, ACT>(x, w, y, M, N, K, (place - tn_i * tiles_m) * BM, tn_i * (BN / 2), smem);
}

// Tiles of 256 rows by 128 features, of which the last ones, a round of workgroups that would leave half of the compute units or
// more idle, are cut into `parts` (2: halves of the rows; 4: and of the features).  `whole`: the tiles in front of those.
// N=17408, K=5120, 2,048 rows (4.25 rounds): 665 us uncut, 583 cut (563 with the walk as it is now); N=25600 (6.25 rounds): 962
// and 846 (819); with three stages of w 537 and 779.
template <int ACT>
__global__ __launch_bounds__(512, 1) void gated_tile_rest_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                                 bf16* __restrict__ y, int M, int N, int K, int tiles_m, int whole,
                                                                 int parts) {
  extern __shared__ __align__(1024) unsigned char smem[];
  const int b = blockIdx.x;
  if (b < whole) {                             // (a multiple of 256)
    const int place = (b & 7) * (whole >> 3) + (b >> 3), tn_i = place / tiles_m;
    gated_tile<256, 256, 2, 3, ACT>(x, w, y, M, N, K, (place - tn_i * tiles_m) * 256, tn_i * 128, smem);
    return;
  }
  const int piece = b - whole, place = whole + piece / parts, part = piece % parts, tn_i = place / tiles_m;
  const int m0 = (place - tn_i * tiles_m) * 256 + 128 * (part & 1), f0 = tn_i * 128 + 64 * (part >> 1);
  if (m0 >= M || f0 >= N) return;
  if (parts == 2) gated_tile<128, 256, 3, 3, ACT>(x, w, y, M, N, K, m0, f0, smem);
  else gated_tile<128, 128, 4, 5, ACT>(x, w, y, M, N, K, m0, f0, smem);
}

}  // namespace tile
}  // namespace xi

using namespace xi;

extern "C" {

// Whether the tiled product takes a shape: K in whole tiles of 64, a tile a slice at least, N in fours.
int xi_linear_tile_takes(int M, int N, int K, int slices) {
  return M > 0 && N > 0 && N % 4 == 0 && slices >= 1 && K > 0 && K % tile::kSliceK == 0 && K / tile::kSliceK >= slices;
}

// x [M, K], w [N, K] bfloat16.  slices == 1 and partial == 0: y bfloat16 [M, N].  Otherwise y is
// float32 [slices, M, N], the sums over the slices of K: slice s takes the tiles of 64 k from
// s * (K / 64) / slices up to (s + 1) * (K / 64) / slices (whole numbers: the slices differ by a tile
// at most).  shape 0: tiles of 128 rows by 256
// features; 1: 256 rows by 128 features; 2: 256 by 256; 7, 8, 9: 64 by 64, 64 by 128, 128 by 128; without slices also 4,
// 5, 6: 96, 160 and 224 rows by 256 features.
int xi_linear_tile(const void* x, const void* w, void* y, int M, int N, int K, int slices, int partial, int shape,
                   hipStream_t stream) {
  XI_CHECK(xi_linear_tile_takes(M, N, K, slices), "linear_tile: M=%d N=%d K=%d in %d slices is not taken (K in tiles of "
           "64, a tile a slice at least, N a multiple of 4)", M, N, K, slices);
  XI_CHECK(partial || slices == 1, "linear_tile: %d slices need the float32 partial sums", slices);
  XI_CHECK((shape >= 0 && shape <= 2) || (shape >= 4 && shape <= 6 && !partial) || (shape >= 7 && shape <= 9), "linear_tile: unknown tile shape %d", shape);
  XI_CHECK((size_t)K * 2 * 256 < ((size_t)1 << 32), "linear_tile: K=%d is too long for 32-bit offsets within a tile", K);
  static const int heights[10] = {128, 256, 256, 0, 96, 160, 224, 64, 64, 128}, widths[10] = {256, 128, 256, 0, 256, 256, 256, 64, 128, 128};
  const int bm = heights[shape], bn = widths[shape];
  const int tiles_m = (M + bm - 1) / bm, tiles_n = (N + bn - 1) / bn;
  const long long total = (long long)tiles_m * tiles_n * slices;
  XI_CHECK(total <= 0x7fffffffLL, "linear_tile: too many workgroups");
#define XI_TILE(BM, BN, WGM, WGN, S, SW, PARTIAL)                                                             \
  do {                                                                                                            \
    auto kern = tile::linear_tile_kernel<BM, BN, WGM, WGN, S, SW, PARTIAL>;                                    \
    const size_t lds = tile::Walk<BM, BN, WGM, WGN, S, SW>::LDS;                                                      \
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);  \
    XI_CHECK(e == hipSuccess, "linear_tile: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));         \
    kern<<<(unsigned)total, 64 * WGM * WGN, lds, stream>>>((const bf16*)x, (const bf16*)w, y, M, N, K, tiles_m,   \
                                                           tiles_n, slices, K / tile::kSliceK);                   \
  } while (0)
  if (shape == 0) {
    if (partial) XI_TILE(128, 256, 2, 4, 3, 3, true);
    else XI_TILE(128, 256, 2, 4, 3, 3, false);
  } else if (shape == 1) {
    if (partial) XI_TILE(256, 128, 4, 2, 3, 4, true);
    else XI_TILE(256, 128, 4, 2, 3, 4, false);
  } else if (shape == 2) {
    if (partial) XI_TILE(256, 256, 2, 4, 2, 3, true);
    else XI_TILE(256, 256, 2, 4, 2, 3, false);
  } else if (shape == 4) XI_TILE(96, 256, 2, 4, 3, 3, false);
  else if (shape == 5) XI_TILE(160, 256, 2, 4, 3, 3, false);
  else if (shape == 6) XI_TILE(224, 256, 2, 4, 2, 3, false);
  else if (shape == 7) {
    if (partial) XI_TILE(64, 64, 2, 4, 8, 8, true);
    else XI_TILE(64, 64, 2, 4, 8, 8, false);
  } else if (shape == 8) {
    if (partial) XI_TILE(64, 128, 2, 4, 6, 6, true);
    else XI_TILE(64, 128, 2, 4, 6, 6, false);
  } else {
    if (partial) XI_TILE(128, 128, 2, 4, 4, 5, true);
    else XI_TILE(128, 128, 2, 4, 4, 5, false);
  }
#undef XI_TILE
  XI_LAUNCH_CHECK("linear_tile");
  return 0;
}

// Whether the gated product takes a shape: K in whole tiles of 64, N in fours, offsets within x and w in 32 bits.
int xi_linear_gated_tile_takes(int M, int N, int K) {
  return M > 0 && N > 0 && N % 4 == 0 && K > 0 && K % tile::kSliceK == 0 && 2LL * M * K < (1LL << 32) && 4LL * N * K < (1LL << 32);
}

// x [M, K], w [2 N, K] = [gate; up], y [M, N] bfloat16 = act(gate) * up; act: 0 silu, 1 gelu (tanh form).  shape 0: 64 rows
// by 64 features a workgroup; 1: 128 by 128; 2: 256 by 128, the last tiles cut where they would be a round of a few workgroups.
int xi_linear_gated_tile(const void* x, const void* w, void* y, int M, int N, int K, int act, int shape, hipStream_t stream) {
  XI_CHECK(xi_linear_gated_tile_takes(M, N, K), "linear_gated_tile: M=%d N=%d K=%d is not taken", M, N, K);
  XI_CHECK((act == 0 || act == 1) && shape >= 0 && shape <= 2, "linear_gated_tile: unknown activation %d or shape %d", act, shape);
  auto on16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  XI_CHECK(on16(x) && on16(w) && (reinterpret_cast<uintptr_t>(y) & 7) == 0, "linear_gated_tile: operands must start on 16 bytes");
  const int bm = shape == 0 ? 64 : shape == 1 ? 128 : 256, features = shape == 0 ? 64 : 128;
  const int tiles_m = (M + bm - 1) / bm;
  const long long tiles = (long long)tiles_m * ((N + features - 1) / features);
  XI_CHECK(tiles <= 0x3fffffffLL, "linear_gated_tile: too many workgroups");
#define XI_GT_LAUNCH(KERN, LDS, WGS, ...)                                                                                    \
  do {                                                                                                                       \
    auto kern = KERN;                                                                                                        \
    const size_t lds = LDS;                                                                                                  \
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);       \
    XI_CHECK(e == hipSuccess, "linear_gated_tile: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));              \
    kern<<<(unsigned)(WGS), 512, lds, stream>>>((const bf16*)x, (const bf16*)w, (bf16*)y, M, N, K, __VA_ARGS__);             \
  } while (0)
#define XI_GT(BM, BN, S, SW)                                                                                                  \
  do {                                                                                                                       \
    constexpr size_t bytes = tile::Walk<BM, BN, 2, 4, S, SW>::LDS;                                                           \
    if (act == 0) XI_GT_LAUNCH((tile::gated_tile_kernel<BM, BN, S, SW, 0>), bytes, tiles, tiles_m);                              \
    else XI_GT_LAUNCH((tile::gated_tile_kernel<BM, BN, S, SW, 1>), bytes, tiles, tiles_m);                                       \
  } while (0)
  const long long whole = tiles / 256 * 256, rest = tiles - whole;
  if (shape == 0) XI_GT(64, 128, 6, 6);
  else if (shape == 1) XI_GT(128, 256, 3, 3);
  else if (whole == 0 || rest == 0 || rest > 128) XI_GT(256, 256, 2, 3);
  else {
    const int parts = rest <= 64 ? 4 : 2;
    constexpr size_t bytes = tile::Walk<256, 256, 2, 4, 2, 3>::LDS;       // the most of the three walks
    static_assert(bytes >= tile::Walk<128, 256, 2, 4, 3>::LDS && bytes >= tile::Walk<128, 128, 2, 4, 4, 5>::LDS, "");
    if (act == 0) XI_GT_LAUNCH(tile::gated_tile_rest_kernel<0>, bytes, whole + rest * parts, tiles_m, (int)whole, parts);
    else XI_GT_LAUNCH(tile::gated_tile_rest_kernel<1>, bytes, whole + rest * parts, tiles_m, (int)whole, parts);
  }
#undef XI_GT
#undef XI_GT_LAUNCH
  XI_LAUNCH_CHECK("linear_gated_tile");
  return 0;
}

}  // extern "C"
