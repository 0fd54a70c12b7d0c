// A selective state space over the long portions of a step in bfloat16, on the matrix cores: S <- a_t S + d_t k_t v_t^T,
// o_t = S^T q_t with one step size d_t = softplus(raw_t + bias) and one decay a_t = exp(-exp(A) d_t) a token and head
// (recurrence.hip has the walk token by token).  A portion is taken in chunks of 64 tokens, one after the other.  With
// L_i = sum_(t <= i) log a_t inside the chunk and S the state in front of it,
//
//   o_i = exp(L_i) q_i S + sum_(j <= i) [exp(L_i - L_j) d_j (q_i . k_j)] v_j
//   S  <- exp(L_last) S + sum_j k_j [exp(L_last - L_j) d_j v_j]^T
//
// A workgroup of eight waves owns a portion, a head and 32 value columns, and keeps its part of the state in registers from
// chunk to chunk (a wave 16 key channels by 32 columns): states neither travel to memory nor wait for another launch, which
// the three launches over chunks side by side pay with four passes over 4 dk dv bytes a head and chunk (134 MB a pass at 128
// heads of 128 by 64 over 2,048 tokens).
//
// q, k and v enter the products as the bfloat16 they are.  What is float32 in the walk (the scores with their decays, the
// decayed values, the state) enters as three bfloat16 that add up to it, three products instead of one, with float32 sums;
// the logarithms are summed in 64 bits, so that the difference of two long sums is as good as the product of the decays
// between them.  Relative error of the results against 64 bits over portions of 32 to 200 tokens: 1.6e-7 to 2.3e-7, the walk
// 1.6e-7 to 9.8e-7 (tests/test_gpu_step_chunks.py).
//
// A chunk with an infinite or undefined operand, a step size of 2^33 and more, or scores, decayed values or a state's results of 2^64
// and more is walked token by token instead (from the operands in LDS and the state in front of it): a masked score times a value
// without a bound is undefined and would reach the tokens in front of that value, and so are three bfloat16 that add up to an
// infinite number.  Below these sizes the chunk's numbers stay in float32's range wherever the walk's do.
//
// Measured on MI355X, us against the walk in three launches: 128 heads of 128 by 64 over 2,048 tokens 131 (1,051), over
// 8,192 517 (4,016), 32 heads over 2,048 124 (289), three portions of 1,974 tokens together 181 (1,040); a portion of 32 tokens
// of 32 heads 22 (43), which is why it starts there (STEP_FROM).  A chunk takes 4.0 us: three barriers, about 370 KB of operand
// reads from LDS a workgroup and the vector instructions of the splits, with two waves a SIMD; its 38 matrix instructions a
// wave are a sixth of it, and looking for what has no bound 4% (as sums of absolute values; as comparisons 8%).
#include "common.h"

namespace xi {
namespace step {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kTok = 64, kCols = 32, kWaves = 8, kSumWave = 2;
constexpr int kRow = kTok + 8;                 // bf16 of a row over tokens in LDS

struct Args {
  const bf16 *q, *k, *v, *raw;
  long long q_stride, k_stride, v_stride, raw_stride;
  const float *bias, *rate_log;
  float* state;
  long long slot_stride;
  const long long* slots;
  const int *first, *last;
  float* out;
  int H, dv, group_heads, least;
  float scale, k_scale;                        // q_scale * k_scale; k_scale
};

__device__ __forceinline__ bf16x8 ld8(const __bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }

__device__ __forceinline__ float pow2(double x) { return __builtin_amdgcn_exp2f((float)x); }

// x = the sum of three bfloat16 (to its last bit or two)
__device__ __forceinline__ void split3(float x, __bf16& a, __bf16& b, __bf16& c) {
  a = (__bf16)x;
  x -= (float)a;
  b = (__bf16)x;
  c = (__bf16)(x - (float)b);
}

template <int DKS>                             // key channels in steps of 32
__global__ __launch_bounds__(64 * kWaves, 1) void step_chunks_kernel(const Args A) {
  constexpr int DK = 32 * DKS, QR = DK + 8;    // bf16 of a row over channels in LDS
  constexpr int KI = (kTok * DK / 8 + 64 * kWaves - 1) / (64 * kWaves);      // 16-byte pieces of q, k a thread
  extern __shared__ __align__(16) unsigned char smem[];
  __bf16* qs = reinterpret_cast<__bf16*>(smem);              // [kTok][QR]
  __bf16* ks = qs + kTok * QR;                               // [kTok][QR]
  __bf16* kt = ks + kTok * QR;                               // [DK][kRow]: a channel a row
  __bf16* vt = kt + DK * kRow;                               // [kCols][kRow]: a value column a row
  __bf16* wt = vt + kCols * kRow;                            // [3][kCols][kRow]: the decayed values
  __bf16* ps = wt + 3 * kCols * kRow;                        // [3][kTok][kRow]: the decayed scores
  __bf16* ss = ps + 3 * kTok * kRow;                         // [3][kCols][QR]: the state, a column a row
  double* Ls2 = reinterpret_cast<double*>(ss + 3 * kCols * QR);     // [2][kTok]: this chunk's and the next one's
  float* ds2 = reinterpret_cast<float*>(Ls2 + 2 * kTok);     // [2][kTok]
  int* large = reinterpret_cast<int*>(ds2 + 2 * kTok);       // [2]: this chunk, the next one is walked token by token
  float* part = reinterpret_cast<float*>(wt);                // [DK / 16][kTok][kCols], in the place of wt, ps and ss: the walk's results
  const int p = blockIdx.x, h = blockIdx.y, col0 = blockIdx.z * kCols;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, j = lane >> 4;
  const int t_end = A.last[p];
  if (t_end - A.first[p] < A.least) return;    // (walked token by token, by another launch)
  const int qk0 = (h / A.group_heads) * DK;
  const float bias = A.bias[h], rate = -expf(A.rate_log[h]);
  float* S = A.state + (size_t)A.slots[p] * A.slot_stride + (size_t)h * DK * A.dv;
  const bool owns = 16 * wave < DK;            // this wave's 16 channels of the state
  const int vwave = wave - (kWaves - kCols / 8);      // the last four waves bring the values, 8 columns each (the others: < 0)
  // the state's tiles: channel 16 wave + 4 j + i, column 16 b + r
  f32x4 st[2];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) st[b][i] = owns ? S[(size_t)(16 * wave + 4 * j + i) * A.dv + col0 + 16 * b + r] : 0.f;
  if (tid < 2) large[tid] = 0;
  __syncthreads();
  auto keep_state = [&] {
    if (!owns) return;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      bf16x4 x[3];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        __bf16 hi, mid, lo;
        split3(st[b][i], hi, mid, lo);
        x[0][i] = hi;
        x[1][i] = mid;
        x[2][i] = lo;
      }
#pragma unroll
      for (int s = 0; s < 3; ++s) *reinterpret_cast<bf16x4*>(ss + (s * kCols + 16 * b + r) * QR + 16 * wave + 4 * j) = x[s];
    }
  };
  keep_state();
  // the tiles above the diagonal that are read beside one on it are zeros and stay so
  auto clear_above = [&] {
    for (int i = tid; i < 3 * kTok * 16; i += 64 * kWaves) {
      const int row = (i >> 4) % kTok, at = row < 16 ? 16 : row >= 32 && row < 48 ? 48 : -1;
      if (at >= 0) ps[(i >> 4) * kRow + at + (i & 15)] = (__bf16)0.f;
    }
  };
  clear_above();
  // what a thread brings of a chunk: q by rows; k and v a token a lane, so that their 2-byte stores by channel lie side by side
  typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
  u32x4 nq[KI], nk[KI], nv = {0u, 0u, 0u, 0u};
  float nraw = 0.f;
  auto piece = [](const bf16* at, bool there) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (there) v = *reinterpret_cast<const u32x4*>(at);
    return v;
  };
  auto ask = [&](int t0) {
    const int n = t_end - t0;
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const int idx = tid + 64 * kWaves * i;
      const int qt = idx / (DK / 8), qc = 8 * (idx % (DK / 8)), kc = 8 * (idx >> 6);
      nq[i] = piece(A.q + (size_t)(t0 + qt) * A.q_stride + qk0 + qc, qt < kTok && qt < n);
      nk[i] = piece(A.k + (size_t)(t0 + lane) * A.k_stride + qk0 + kc, kc < DK && lane < n);
    }
    if (vwave >= 0) nv = piece(A.v + (size_t)(t0 + lane) * A.v_stride + (size_t)h * A.dv + col0 + 8 * vwave, lane < n);
  };
  // the step sizes are asked for two chunks ahead, and summed one ahead, by a wave that has one tile of scores and no values
  auto ask_raw = [&](int t0) {
    if (wave == kSumWave) nraw = t0 + lane < t_end ? to_float(A.raw[(size_t)(t0 + lane) * A.raw_stride + h]) : 0.f;
  };
  auto sum_steps = [&](int t0, int buf) {
    if (wave != kSumWave) return;
    const bool there = t0 + lane < t_end;
    const float x = nraw + bias;
    const float d = there ? fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))) : 0.f;
    const float la = rate * d;
    // (e^-10000 is 0 in float32: a token that forgets everything still does, and the sums keep the later tokens' digits)
    double L = there ? (double)(la < -1e4f ? -1e4f : la) * 1.4426950408889634 : 0.0;      // base 2 from here on
#pragma unroll
    for (int off = 1; off < kTok; off <<= 1) {
      const double up = __shfl_up(L, off, kWave);
      if (lane >= off) L += up;
    }
    if (there && !(x < 0x1p33f)) large[buf] = 1;
    Ls2[buf * kTok + lane] = L;                // (tokens past the chunk's end: the last one's)
    ds2[buf * kTok + lane] = d;
  };
  auto half = [](u32x4 u, int e) {             // the e-th of eight bfloat16
    const unsigned w = u[e >> 1];
    return __builtin_bit_cast(__bf16, (unsigned short)(e & 1 ? w >> 16 : w & 0xffffu));
  };
  const int t_begin = A.first[p];
  ask_raw(t_begin);
  ask(t_begin);
  sum_steps(t_begin, 0);
  ask_raw(t_begin + kTok);
  int buf = 0;
  for (int t0 = t_begin; t0 < t_end; t0 += kTok, buf ^= 1) {
    const int n = t_end - t0 < kTok ? t_end - t0 : kTok;
    const double* Ls = Ls2 + buf * kTok;
    const float* ds = ds2 + buf * kTok;
    // ---- the chunk into LDS
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const int idx = tid + 64 * kWaves * i;
      const int qt = idx / (DK / 8), qc = 8 * (idx % (DK / 8)), kc = 8 * (idx >> 6);
      if (qt < kTok) *reinterpret_cast<u32x4*>(qs + qt * QR + qc) = nq[i];
      if (kc < DK) {
        *reinterpret_cast<u32x4*>(ks + lane * QR + kc) = nk[i];
#pragma unroll
        for (int e = 0; e < 8; ++e) kt[(kc + e) * kRow + lane] = half(nk[i], e);
      }
    }
    if (vwave >= 0) {
#pragma unroll
      for (int e = 0; e < 8; ++e) vt[(8 * vwave + e) * kRow + lane] = half(nv, e);
    }
    __syncthreads();
    const u32x4 cv = nv;
    if (t0 + kTok < t_end) ask(t0 + kTok);
    // ---- the decayed values, the scores with their decays, and what the state gives
    const double all = Ls[kTok - 1];
    float sizes = 0.f;                         // of what this lane has seen of the chunk, added up: undefined if one of them is
    if (vwave >= 0) {
      const float w = pow2(all - Ls[lane]) * ds[lane] * A.k_scale;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        __bf16 x[3];
        const float wv = w * (float)half(cv, e);
        sizes += fabsf(wv);                    // (a decay of 0 times a value without a bound is undefined)
        split3(wv, x[0], x[1], x[2]);
#pragma unroll
        for (int s = 0; s < 3; ++s) wt[(s * kCols + 8 * vwave + e) * kRow + lane] = x[s];
      }
    }
    // the ten tiles of 16 queries by 16 keys on and below the diagonal, one a wave and a second one for two of them;
    // a lane holds keys 16 kt_ + 4 j .. + 3 of query 16 qt_ + r
    for (int tile = wave; tile < 10; tile += kWaves) {
      const int qt_ = tile < 1 ? 0 : tile < 3 ? 1 : tile < 6 ? 2 : 3, kt_ = tile - qt_ * (qt_ + 1) / 2;
      f32x4 sc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < DKS; ++s)
        sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ld8(ks + (16 * kt_ + r) * QR + 32 * s + 8 * j),
                                                     ld8(qs + (16 * qt_ + r) * QR + 32 * s + 8 * j), sc, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) sizes += fabsf(sc[i]);       // (a q or k without a bound is in a score on the diagonal)
      const int qi = 16 * qt_ + r, k0 = 16 * kt_ + 4 * j;
      const double lq = Ls[qi];
      bf16x4 x[3];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float pv = k0 + i <= qi ? sc[i] * (pow2(lq - Ls[k0 + i]) * (ds[k0 + i] * A.scale)) : 0.f;
        __bf16 hi, mid, lo;
        split3(pv, hi, mid, lo);
        x[0][i] = hi;
        x[1][i] = mid;
        x[2][i] = lo;
      }
#pragma unroll
      for (int s = 0; s < 3; ++s) *reinterpret_cast<bf16x4*>(ps + (s * kTok + qi) * kRow + k0) = x[s];
    }
    if (t0 + kTok < t_end) {
      sum_steps(t0 + kTok, buf ^ 1);
      ask_raw(t0 + 2 * kTok);
    }
    const int rt = wave >> 1, ct = wave & 1;   // this wave's rows (tokens) of the results and half of the columns
    f32x4 os[3] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int s = 0; s < DKS; ++s) {
      const bf16x8 qa = ld8(qs + (16 * rt + r) * QR + 32 * s + 8 * j);
#pragma unroll
      for (int x = 0; x < 3; ++x)
        os[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa, ld8(ss + (x * kCols + 16 * ct + r) * QR + 32 * s + 8 * j), os[x], 0, 0, 0);
    }
    f32x4 o = (os[2] + os[1]) + os[0];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sizes += fabsf(o[i]);                    // (so is what a state without a bound gives)
      o[i] *= pow2(Ls[16 * rt + 4 * j + i]) * (A.scale / A.k_scale);
    }
    if (!(sizes < 0x1p64f)) large[buf] = 1;
    __syncthreads();
    const int walk = large[buf];
    // ---- the results, and the state behind the chunk
#pragma unroll
    for (int s = 0; s < kTok / 32; ++s) {
      if (32 * s > 16 * rt + 15) break;        // keys behind all of the rows
      const bf16x8 vb = ld8(vt + (16 * ct + r) * kRow + 32 * s + 8 * j);
#pragma unroll
      for (int x = 2; x >= 0; --x)
        o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ld8(ps + (x * kTok + 16 * rt + r) * kRow + 32 * s + 8 * j), vb, o, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tok = 16 * rt + 4 * j + i;
      if (tok < n) A.out[((size_t)(t0 + tok) * A.H + h) * A.dv + col0 + 16 * ct + r] = o[i];
    }
    const f32x4 front[2] = {st[0], st[1]};
    if (owns) {
      const float f = pow2(all);
#pragma unroll
      for (int b = 0; b < 2; ++b) st[b] *= f;
#pragma unroll
      for (int s = 0; s < kTok / 32; ++s) {
        const bf16x8 ka = ld8(kt + (16 * wave + r) * kRow + 32 * s + 8 * j);
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int x = 2; x >= 0; --x)
            st[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, ld8(wt + (x * kCols + 16 * b + r) * kRow + 32 * s + 8 * j), st[b], 0, 0, 0);
      }
    }
    if (walk) {
      __syncthreads();
      st[0] = front[0];
      st[1] = front[1];
      if (owns) {
        const float q_scale = A.scale / A.k_scale;
        for (int t = 0; t < n; ++t) {
          const float d = ds[t], a = expf(rate * d);
          float acc[2] = {0.f, 0.f};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int at = t * QR + 16 * wave + 4 * j + i;
            const float kv = (float)ks[at] * A.k_scale, qv = (float)qs[at] * q_scale;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              st[b][i] = fmaf(a, st[b][i], kv * ((float)vt[(16 * b + r) * kRow + t] * d));
              acc[b] = fmaf(st[b][i], qv, acc[b]);
            }
          }
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            acc[b] += lane_xor<16>(acc[b]);
            acc[b] += lane_xor<32>(acc[b]);
            if (j == 0) part[(wave * kTok + t) * kCols + 16 * b + r] = acc[b];
          }
        }
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 4; ++i) {            // (over what this thread has stored above)
        const int tok = 16 * rt + 4 * j + i;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < DK / 16; ++w) sum += part[(w * kTok + tok) * kCols + 16 * ct + r];
        if (tok < n) A.out[((size_t)(t0 + tok) * A.H + h) * A.dv + col0 + 16 * ct + r] = sum;
      }
      __syncthreads();
      if (tid == 0) large[buf] = 0;
      clear_above();
    }
    keep_state();
    __syncthreads();                           // (the next chunk overwrites k, v and the decayed values)
  }
  if (owns) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[(size_t)(16 * wave + 4 * j + i) * A.dv + col0 + 16 * b + r] = st[b][i];
  }
}

}  // namespace step
}  // namespace xi

using namespace xi;

extern "C" {

// Head sizes that the kernel takes (rows in whole 16-byte pieces besides: the caller's strides and pointers).
int xi_step_chunks_takes(int dk, int dv) { return dk > 0 && dk <= 128 && dk % 32 == 0 && dv > 0 && dv % 32 == 0; }

// q, k [T, .] with (H / group_heads) dk columns, v [T, .] with H dv, raw [T, .] with H, bfloat16 rows `*_stride` elements apart;
// bias, rate_log float32 [H]; portion p: tokens first[p] .. last[p] - 1, its request's state at state + slots[p] * slot_stride
// ([H, dk, dv] float32, read and left behind the portion); out float32 [T, H, dv].  Portions of fewer than `least` tokens are
// left alone.
int xi_step_chunks(const void* q, long long q_stride, const void* k, long long k_stride, const void* v, long long v_stride,
                   const void* raw, long long raw_stride, const float* bias, const float* rate_log, float* state, long long slot_stride,
                   const long long* slots, const int* first, const int* last, int n_portions, float* out, int H, int dk, int dv,
                   int group_heads, int least, float q_scale, float k_scale, hipStream_t stream) {
  XI_CHECK(xi_step_chunks_takes(dk, dv) && H > 0 && H <= 65535 && group_heads > 0 && H % group_heads == 0 && dv / step::kCols <= 65535,
           "step_chunks: %d heads of %d by %d in groups of %d are not taken", H, dk, dv, group_heads);
  XI_CHECK(q_stride % 8 == 0 && k_stride % 8 == 0 && v_stride % 8 == 0 &&
               ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) & 15) == 0,
           "step_chunks: rows in whole 16-byte pieces");
  XI_CHECK(slot_stride >= (long long)H * dk * dv && raw && bias && rate_log && state && slots && first && last && out && n_portions >= 0,
           "step_chunks: an operand is missing");
  XI_CHECK(k_scale != 0.f, "step_chunks: keys with a factor of 0");
  if (n_portions == 0) return 0;
  const step::Args A{(const bf16*)q, (const bf16*)k, (const bf16*)v, (const bf16*)raw, q_stride, k_stride, v_stride, raw_stride, bias,
                     rate_log, state, slot_stride, slots, first, last, out, H, dv, group_heads, least, q_scale * k_scale, k_scale};
  const dim3 grid((unsigned)n_portions, (unsigned)H, (unsigned)(dv / step::kCols));
#define XI_SC(DKS)                                                                                                           \
  do {                                                                                                                       \
    const size_t qr = 32 * DKS + 8;                                                                                          \
    const size_t lds = 2 * (2 * step::kTok * qr + (32 * DKS + 4 * step::kCols + 3 * step::kTok) * step::kRow + 3 * step::kCols * qr) + \
                       2 * step::kTok * 12 + 8;                                                                               \
    const hipError_t e = hipFuncSetAttribute((const void*)step::step_chunks_kernel<DKS>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                             (int)lds);                                                                      \
    XI_CHECK(e == hipSuccess, "step_chunks: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(e));                    \
    step::step_chunks_kernel<DKS><<<grid, 64 * step::kWaves, lds, stream>>>(A);                                              \
  } while (0)
  if (dk == 32) XI_SC(1);
  else if (dk == 64) XI_SC(2);
  else if (dk == 96) XI_SC(3);
  else XI_SC(4);
#undef XI_SC
  XI_LAUNCH_CHECK("step_chunks");
  return 0;
}

}  // extern "C"
