// y[M,N] = x[M,K] @ w[N,K]^T for the true 32-bit path, on the matrix cores' float32 form
// (v_mfma_f32_16x16x4_f32: float32 products, float32 accumulation, no reduced-precision mode), and
// a plain FMA kernel for bfloat16 operands (reference tests of the bfloat16 kernels use it).
//
// The value of an output element depends on K alone, never on M, on the kernel that makes it, on
// the tile it falls in or on what else is in the batch: both float32 kernels cut K into the same (up
// to) eight chunks of kc = 32 * ceil(K / 256), run a chunk as one chain of matrix instructions over
// 16 k at a time, the four instructions of which take k = e, e + 4, e + 8, e + 12 for e = 0 .. 3
// (a lane's 16-byte load holds four consecutive k, element e of it is instruction e's operand), and
// add the chunks in ascending order.  Missing k are zeros.
//
//   few rows  (M <= 64)  a workgroup owns 16 or 32 features and all rows, its eight waves a chunk
//             each; operands go straight from memory into registers, 16 bytes a lane, some steps
//             ahead; the chunks meet in LDS.  Bound by the weights' bytes
//             beside x, which every tile of features reads again: 3.4 (N = 6144, K = 4096) to 5.3 TB/s
//             (N = 151936) of weights at 8 rows.
//   tile      a workgroup of four waves owns BM rows by BN features; tiles of 32 k go through
//             registers into two LDS buffers, one barrier a tile.  The matrix cores (157 TFLOP/s)
//             are busy 67 to 71% of the time in tiles of 64 x 64 and 56% in those of 32 x 64; a
//             step's operands are read together in front of its products, and half of the 36 to
//             48% of the time that LDS is active is bank conflicts.
//
// Reference call site: candle matmul, /root/reference/src/models/layers/linear.rs:76-124.
#include "common.h"

namespace xi {

// ---- bfloat16 operands: one FMA chain an output element, in ascending k ---------------------------------
constexpr int BM = 64, BN = 64, BK = 16, TM = 4, TN = 4;

template <typename TO, bool ADD>
__global__ __launch_bounds__(256) void gemm_tn_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                      TO* __restrict__ y, int M, int N, int K) {
  __shared__ float xs[BK][BM + 4];
  __shared__ float ws[BK][BN + 4];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * BM;
  const int n0 = blockIdx.x * BN;
  const int tx = tid % 16;  // n direction
  const int ty = tid / 16;  // m direction
  float acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = 0.f;

  const int lr = tid / 4;        // 0..63: row of the tile this thread loads
  const int lk = (tid % 4) * 4;  // 0,4,8,12: first k of the four it loads
  for (int k0 = 0; k0 < K; k0 += BK) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k = k0 + lk + q;
      const int m = m0 + lr;
      const int n = n0 + lr;
      xs[lk + q][lr] = (m < M && k < K) ? to_float(x[(size_t)m * K + k]) : 0.f;
      ws[lk + q][lr] = (n < N && k < K) ? to_float(w[(size_t)n * K + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < BK; ++kk) {
      float a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = xs[kk][ty * TM + i];
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j] = ws[kk][tx * TN + j];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + ty * TM + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + tx * TN + j;
      if (n >= N) continue;
      const size_t o = (size_t)m * N + n;
      if (ADD)
        y[o] = from_float<TO>(to_float(y[o]) + acc[i][j]);
      else
        y[o] = from_float<TO>(acc[i][j]);
    }
  }
}

// ---- float32 ------------------------------------------------------------------------------------------
namespace f32 {

typedef __attribute__((ext_vector_type(4))) float f4;

constexpr int kChunks = 8;
// k of a chunk: a multiple of 32, at most eight chunks
__host__ __device__ __forceinline__ int chunk_k(int K) { return (K + 32 * kChunks - 1) / (32 * kChunks) * 32; }

// Four consecutive k of a row from k on; VEC: K % 4 == 0 and rows on 16 bytes.  Past K: zeros.
template <bool VEC>
__device__ __forceinline__ f4 load4(const float* __restrict__ row, int k, int K) {
  if constexpr (VEC) {
    return k < K ? *reinterpret_cast<const f4*>(row + k) : f4{0.f, 0.f, 0.f, 0.f};
  } else {
    f4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = k + e < K ? row[k + e] : 0.f;
    return v;
  }
}

constexpr unsigned kNowhere = 0x80000000u;

// A pointer that is the same in all lanes, in scalar registers (a buffer descriptor has to be).
__device__ __forceinline__ float* uniform(const float* p) {
  const unsigned long long a = (unsigned long long)(uintptr_t)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a), hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
  return reinterpret_cast<float*>((uintptr_t)(((unsigned long long)hi << 32) | lo));
}

// Four consecutive floats `at` bytes into a buffer, of which the first `n` count (the others, and what lies past the
// buffer's end, are zeros).  VEC: n is a multiple of 4.
template <bool VEC>
__device__ __forceinline__ f4 buffer4(__amdgpu_buffer_rsrc_t d, unsigned at, int n) {
  if constexpr (VEC) {
    return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(d, n > 0 ? at : kNowhere, 0, 0));
  } else {
    f4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(d, n > e ? at + 4u * e : kNowhere, 0, 0));
    return v;
  }
}

// y (+)= v for features n .. n + 3 of row m; `whole`: N % 4 == 0 and y on 16 bytes.
__device__ __forceinline__ void put4(float* __restrict__ y, size_t m, int n, int N, f4 v, bool add, bool whole) {
  float* p = y + m * N + n;
  if (whole && n + 3 < N) {
    f4* q = reinterpret_cast<f4*>(p);
    *q = add ? *q + v : v;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n + e < N) p[e] = add ? p[e] + v[e] : v[e];
}

// FT tiles of 16 features and RT tiles of 16 rows a workgroup.  Lane (r, j) = (l & 15, l >> 4) of wave c brings row r of
// every tile, k 16 i + 4 j .. + 3 of its chunk's blocks; a lane of the result holds features 4 j .. 4 j + 3 of row r.
// A workgroup walks the tiles b, b + gridDim.x, ..; a step is KS k of one of them, and the operands of S steps, past a
// tile's end those of the next tile, are in registers or on their way.  The chunks' sums meet in one of two LDS buffers,
// one barrier a tile.
template <int FT, int RT, int KS, int S, bool VEC>
__global__ __launch_bounds__(64 * kChunks, 2) void few_rows_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                   float* __restrict__ y, int M, int N, int K, int tiles,
                                                                   int add, int whole) {
  constexpr int NB = KS / 16;      // blocks of 16 k in a step
  __shared__ f4 part[2][kChunks][FT * RT][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, j = lane >> 4;
  const int kc = chunk_k(K);
  const int kb = wave * kc, ke = kb + kc < K ? kb + kc : K;
  const int steps = (kc + KS - 1) / KS;
  // Loads through buffer descriptors: what lies past the descriptor's end reads zeros, and so does a lane that is sent
  // there, so that rows, features and k past the end need no branch.  Offsets stay below kNowhere (the host checks).
  const auto xd = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), 0, M * K * 4, 0x00027000);
  const unsigned lane0 = ((unsigned)r * (unsigned)K + 4u * j) * 4u, tile16 = 16u * (unsigned)K * 4u;
  f4 acc[FT][RT], wv[S][FT][NB], xv[S][RT][NB];
  int ft = blockIdx.x, fs = 0;     // the tile and step that is asked for next
  auto fetch = [&](f4 (&wn)[FT][NB], f4 (&xn)[RT][NB]) {
    const int n0 = ft * 16 * FT, left = N - n0;
    const int bytes = __builtin_amdgcn_readfirstlane((left <= 0 ? 0 : left < 16 * FT ? left : 16 * FT) * K * 4);
    const auto wd = __builtin_amdgcn_make_buffer_rsrc(uniform(w + (size_t)(left > 0 ? n0 : 0) * K), 0, bytes, 0x00027000);
    const int k0 = kb + fs * KS;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int kk = k0 + 16 * i + 4 * j;
      const unsigned at = lane0 + (unsigned)(k0 + 16 * i) * 4u;
#pragma unroll
      for (int f = 0; f < FT; ++f) wn[f][i] = buffer4<VEC>(wd, at + f * tile16, ke - kk);
#pragma unroll
      for (int t = 0; t < RT; ++t) xn[t][i] = buffer4<VEC>(xd, at + t * tile16, ke - kk);
    }
    if (++fs == steps) {
      fs = 0;
      ft += gridDim.x;
    }
  };
  auto clear = [&] {
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
      for (int t = 0; t < RT; ++t) acc[f][t] = f4{0.f, 0.f, 0.f, 0.f};
  };
  clear();
#pragma unroll
  for (int s = 0; s < S; ++s) fetch(wv[s], xv[s]);
  int tile = blockIdx.x, step = 0, buf = 0;
  for (;;) {                       // (the grid has no more workgroups than there are tiles)
#pragma unroll
    for (int s = 0; s < S; ++s) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int f = 0; f < FT; ++f)
#pragma unroll
            for (int t = 0; t < RT; ++t)
              acc[f][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[s][f][i][e], xv[s][t][i][e], acc[f][t], 0, 0, 0);
      fetch(wv[s], xv[s]);
      if (++step < steps) continue;
      step = 0;
#pragma unroll
      for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int t = 0; t < RT; ++t) part[buf][wave][f * RT + t][lane] = acc[f][t];
      clear();
      __syncthreads();
      for (int p = wave; p < FT * RT; p += kChunks) {
        f4 sum = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < kChunks; ++c) sum += part[buf][c][p][lane];
        const int m = 16 * (p % RT) + r, n = tile * 16 * FT + 16 * (p / RT) + 4 * j;
        if (m < M && n < N) put4(y, m, n, N, sum, add, whole);
      }
      buf ^= 1;                    // (the buffer is written again two tiles on, behind the next tile's barrier)
      tile += gridDim.x;
      if (tile >= tiles) return;
    }
  }
}

// BM_ rows of x by BN_ features, four waves of half of each.  A tile of 32 k lies in LDS as two blocks of 16 k, a row's 64
// bytes side by side: the 64 lanes of an operand read take 1 KB in one piece.
template <int BM_, int BN_, bool VEC>
__global__ __launch_bounds__(256, 1) void tile_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                      float* __restrict__ y, int M, int N, int K, int tiles_m, int add, int whole) {
  constexpr int ROWS = BM_ + BN_, LOADS = ROWS * 8 / 256;
  constexpr int WM = BM_ / 32, WN = BN_ / 32;              // 16 x 16 tiles of a wave
  constexpr int BLOCK = ROWS * 16 + 32;                    // floats of a block of 16 k (the second one starts in other banks)
  __shared__ __align__(16) float lds[2][2 * BLOCK];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, j = lane >> 4;
  // workgroup numbers b, b + 8, .. run on one die: they get consecutive places, rows of x innermost, so that a die's L2
  // holds the rows of w that its workgroups share
  const int total = gridDim.x, q8 = total >> 3, r8 = total & 7, die = blockIdx.x & 7;
  const int place = die * q8 + (die < r8 ? die : r8) + (blockIdx.x >> 3);
  const int m0 = (place % tiles_m) * BM_, n0 = (place / tiles_m) * BN_;
  const float* row[LOADS];
  int at[LOADS], kk[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int idx = tid + 256 * i, p = idx >> 3, c = idx & 7;        // row of the tile, 16-byte piece of its 32 k
    const bool is_w = p < BN_;
    const int g = is_w ? (n0 + p < N ? n0 + p : N - 1) : (m0 + p - BN_ < M ? m0 + p - BN_ : M - 1);
    row[i] = (is_w ? w : x) + (size_t)g * K;
    kk[i] = 4 * c;
    at[i] = (c >> 2) * BLOCK + p * 16 + (c & 3) * 4;
  }
  const int w_rd = ((wave >> 1) * WN * 16 + r) * 16 + 4 * j, x_rd = (BN_ + (wave & 1) * WM * 16 + r) * 16 + 4 * j;
  f4 acc[WN][WM], sum[WN][WM];
#pragma unroll
  for (int a = 0; a < WN; ++a)
#pragma unroll
    for (int b = 0; b < WM; ++b) acc[a][b] = sum[a][b] = f4{0.f, 0.f, 0.f, 0.f};
  f4 next[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) next[i] = load4<VEC>(row[i], kk[i], K);
#pragma unroll
  for (int i = 0; i < LOADS; ++i) *reinterpret_cast<f4*>(&lds[0][at[i]]) = next[i];
  __syncthreads();
  const int kc = chunk_k(K);
  int buf = 0, chunk_end = kc;
  for (int k0 = 0; k0 < K; k0 += 32) {
    const bool more = k0 + 32 < K;
    if (more) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) next[i] = load4<VEC>(row[i], k0 + 32 + kk[i], K);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      f4 wa[WN], xb[WM];
#pragma unroll
      for (int a = 0; a < WN; ++a) wa[a] = *reinterpret_cast<const f4*>(&lds[buf][s * BLOCK + w_rd + a * 256]);
#pragma unroll
      for (int b = 0; b < WM; ++b) xb[b] = *reinterpret_cast<const f4*>(&lds[buf][s * BLOCK + x_rd + b * 256]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int a = 0; a < WN; ++a)
#pragma unroll
          for (int b = 0; b < WM; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wa[a][e], xb[b][e], acc[a][b], 0, 0, 0);
    }
    if (k0 + 32 >= chunk_end || !more) {       // the chunk's chain joins the sum
      chunk_end += kc;
#pragma unroll
      for (int a = 0; a < WN; ++a)
#pragma unroll
        for (int b = 0; b < WM; ++b) {
          sum[a][b] += acc[a][b];
          acc[a][b] = f4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (more) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) *reinterpret_cast<f4*>(&lds[buf ^ 1][at[i]]) = next[i];
    }
    __syncthreads();
    buf ^= 1;
  }
#pragma unroll
  for (int b = 0; b < WM; ++b) {
    const int m = m0 + ((wave & 1) * WM + b) * 16 + r;
    if (m >= M) continue;
#pragma unroll
    for (int a = 0; a < WN; ++a) {
      const int n = n0 + ((wave >> 1) * WN + a) * 16 + 4 * j;
      if (n < N) put4(y, m, n, N, sum[a][b], add, whole);
    }
  }
}

// 0: few rows, 16 features a workgroup; 1: few rows, 32; 2, 3, 4: tiles of 32 x 64, 64 x 64, 128 x 128 (rows x features).
//
// Few rows, MI355X, us at 8 rows (16 | 32 features a workgroup): N = 4096, K = 4096: 20 | 28; N = 6144: 31 | 30; N = 24576: 85 | 85;
// at 1 row 17 | 24, 27 | 28, 72 | 79, at 40 rows 37 | 46, 64 | 46, 177 | 131: half as many reads of x a feature against half as many
// workgroups.  (The FMA kernel that was here took 845 us for N = 4096, K = 12288 at 8 rows where this takes 49.)  From 49 rows
// on a wide output is bound by the matrix cores: N = 24576 at 64 rows 165 us here, 147 in tiles of 32 x 64.
// Tiles: rounds of 256 workgroups times a tile's products, a tile of 32 x 64 taking 1.12 and one of 128 x 128 1.05 of its
// share: 562 rows, N = 4096: 238 | 244 | 328 us, N = 24576: 1161 | 1099 | 1330; 2,048 rows, N = 24576: 4078 | 3724 | 3985
// (111 TFLOP/s; the FMA kernel 30).
int form_for(int M, int N) {
  if (M <= 48 || (M <= 64 && N < 16384)) return M >= 8 && N >= 6144 ? 1 : 0;
  constexpr int bm[3] = {32, 64, 128}, bn[3] = {64, 64, 128};
  constexpr double more[3] = {1.12, 1.0, 1.05};
  int best = 0;
  double least = 0;
  for (int i = 0; i < 3; ++i) {
    const long long wgs = ((long long)M + bm[i] - 1) / bm[i] * (((long long)N + bn[i] - 1) / bn[i]);
    const double cost = (double)((wgs + 255) / 256) * bm[i] * bn[i] * more[i];
    if (i == 0 || cost < least) {
      least = cost;
      best = i;
    }
  }
  return 2 + best;
}

}  // namespace f32
}  // namespace xi

using namespace xi;

extern "C" {

// The form that a float32 product of these sizes takes (see f32::form_for).
int xi_gemm_f32_form(int M, int N) { return f32::form_for(M, N); }

// form: of a float32 product, -1: chosen here.
int xi_gemm_tn(const void* x, const void* w, void* y, int M, int N, int K, int in_dtype, int out_dtype, int accumulate, int form,
               hipStream_t stream) {
  XI_CHECK(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
  if (M == 0) return 0;
  if (in_dtype == kF32 && out_dtype == kF32) {
    if (form < 0) form = f32::form_for(M, N);
    if (form < 2 && K >= (1 << 23)) form = 2;        // (64 rows of the few-rows kernel's offsets stay below 2^31)
    XI_CHECK(form <= 4 && (form >= 2 || M <= 64), "gemm: form %d does not take %d rows", form, M);
    XI_CHECK(K <= (1 << 30) && N <= (1 << 30) && M <= (1 << 30), "gemm: sizes M=%d N=%d K=%d are too large", M, N, K);
    auto on16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vec = K % 4 == 0 && on16(x) && on16(w);
    const int whole = N % 4 == 0 && on16(y);
    const float *xf = (const float*)x, *wf = (const float*)w;
    float* yf = (float*)y;
    if (form < 2) {
      const int rt = (M + 15) / 16;
#define XI_FEW(FT, RT, KS, S)                                                                                             \
  do {                                                                                                                  \
    const int tiles = (N + 16 * FT - 1) / (16 * FT);                                                                    \
    const unsigned wgs = (unsigned)(tiles < 256 ? tiles : 256);                                                         \
    if (vec) f32::few_rows_kernel<FT, RT, KS, S, true><<<wgs, 64 * f32::kChunks, 0, stream>>>(xf, wf, yf, M, N, K, tiles, accumulate, whole); \
    else f32::few_rows_kernel<FT, RT, KS, 2, false><<<wgs, 64 * f32::kChunks, 0, stream>>>(xf, wf, yf, M, N, K, tiles, accumulate, whole);    \
  } while (0)
      if (form == 0) {
        if (rt == 1) XI_FEW(1, 1, 64, 4);
        else if (rt == 2) XI_FEW(1, 2, 32, 4);
        else if (rt == 3) XI_FEW(1, 3, 32, 4);
        else XI_FEW(1, 4, 32, 3);
      } else {
        if (rt == 1) XI_FEW(2, 1, 64, 3);
        else if (rt == 2) XI_FEW(2, 2, 32, 4);
        else if (rt == 3) XI_FEW(2, 3, 32, 3);
        else XI_FEW(2, 4, 32, 3);
      }
#undef XI_FEW
    } else {
      const int bm = form == 2 ? 32 : form == 3 ? 64 : 128, bn = form == 4 ? 128 : 64;
      const int tiles_m = (M + bm - 1) / bm;
      const long long wgs = (long long)tiles_m * ((N + bn - 1) / bn);
      XI_CHECK(wgs <= 0x7fffffffLL, "gemm: M=%d by N=%d is too large for one launch", M, N);
#define XI_TILE(BM_, BN_)                                                                                              \
  do {                                                                                                                 \
    if (vec) f32::tile_kernel<BM_, BN_, true><<<(unsigned)wgs, 256, 0, stream>>>(xf, wf, yf, M, N, K, tiles_m, accumulate, whole); \
    else f32::tile_kernel<BM_, BN_, false><<<(unsigned)wgs, 256, 0, stream>>>(xf, wf, yf, M, N, K, tiles_m, accumulate, whole);   \
  } while (0)
      if (form == 2) XI_TILE(32, 64);
      else if (form == 3) XI_TILE(64, 64);
      else XI_TILE(128, 128);
#undef XI_TILE
    }
    XI_LAUNCH_CHECK("gemm");
    return 0;
  }
  dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
  XI_CHECK(grid.y <= 65535u, "gemm: M=%d is too large for one launch", M);
#define XI_GEMM(TO)                                                                                                      \
  do {                                                                                                                   \
    if (accumulate) gemm_tn_kernel<TO, true><<<grid, 256, 0, stream>>>((const bf16*)x, (const bf16*)w, (TO*)y, M, N, K);   \
    else gemm_tn_kernel<TO, false><<<grid, 256, 0, stream>>>((const bf16*)x, (const bf16*)w, (TO*)y, M, N, K);             \
  } while (0)
  if (in_dtype == kBF16 && out_dtype == kBF16) XI_GEMM(bf16);
  else if (in_dtype == kBF16 && out_dtype == kF32) XI_GEMM(float);
  else XI_CHECK(false, "gemm: unsupported dtypes in=%d out=%d", in_dtype, out_dtype);
#undef XI_GEMM
  XI_LAUNCH_CHECK("gemm");
  return 0;
}

}  // extern "C"
