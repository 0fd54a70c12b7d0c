// Paged causal GQA attention of the true 32-bit path on the matrix cores' float32 form
// (v_mfma_f32_16x16x4_f32), for head sizes in steps of 16 up to 256.  What a token sees, the options
// of the score and the layouts are those of `attention_generic_kernel` (attention_generic.hip), which
// serves every other size, and whose one lane a key reads K a number at a time, once a query head.
//
// A workgroup of eight waves owns the query heads of one kv head for a tile of up to 16 / (heads on the
// kv head) tokens side by side in the step, at most 16 (token, head) rows: the columns of the matrix
// instructions, for which a key is read once.  Keys are taken in blocks of 16 at multiples of 16
// positions; block b goes to wave b % 8, and the eight waves' results are merged in wave order: what a
// token gets is fixed by its position, window and chunk alone, never by its tile or by what else is in
// the step.
//
//   S^T[key, row]    A = K rows (a lane brings four consecutive dims, element e of them is the e-th
//                    instruction's operand), B = the rows' queries, read from LDS; a lane holds keys
//                    4 j .. 4 j + 3 of row r.
//   O^T[dim, row]    B = the weights as they lie (instruction v takes keys v, v + 4, v + 8, v + 12 of the
//                    block), A = V: a lane brings dims 4 r .. 4 r + 3 of a key, element e belongs to
//                    tile e, whose 16 rows are the dims 4 i + e of 64.
//
// A block's K is asked for a block ahead, its V before its scores are made: a wave would wait for the
// page number, K and V one after the other.
//
// Measured on MI355X, 32 heads of 128 on 8 kv heads, against one lane a key (us): prompts of 200, 127, 54,
// 172 and 9 tokens 81 (396), a prompt of 1,024 245 (1,990; 32 kv heads 424, 2,220), 8 single tokens at up
// to 330 keys 18 (54), one at 4,096 keys 125 (738).  Bound by the chain of a block (page, K, scores, sum,
// V) in the few waves that a long head leaves room for; the matrix instructions are a third of it.
//
// A value that a token does not see never reaches it, not even with a weight of 0 (an infinite or
// undefined one would): in a block that some token of the tile does not see in full, each token's
// product is made by itself, with the nearest key that it sees in the place of one that it does not,
// and only its own columns keep it.  What no token of the tile sees is not read.  Where requests meet in a
// tile, a block that all of one's tokens see in full is one product, which their columns keep (16 heads of
// 128, 300 tokens and one behind contexts of 2,000: 260 us, 592 with a product a token there).
#include "common.h"

namespace xi {
namespace attn_f32 {

typedef __attribute__((ext_vector_type(4))) float f4;
constexpr int kWaves = 8, kBlock = 16;

// Bytes of LDS for `rows` (token, head) rows of heads of d and dv.
constexpr size_t lds_bytes(int rows, int d, int dv) { return ((size_t)kWaves * (rows * dv + 2 * 16) + 16 * (d + 4)) * sizeof(float); }

// DT: 16-dim tiles that the registers have room for (head sizes up to 16 DT)
template <int DT>
__global__ __launch_bounds__(64 * kWaves, 1) void attention_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_pages, const int* __restrict__ tok_seq, const int* __restrict__ positions,
    float* __restrict__ out, float scale, int window, int page_size, int n_tok, int lead, int tile_tokens, int nq, int nkv, int d, int dv,
    float softcap, const float* __restrict__ slopes, const float* __restrict__ sinks, int values_in_keys, int chunk) {
  constexpr int DG = (DT + 3) / 4;                  // groups of 64 value dims
  extern __shared__ float lds[];                    // m and l [kWaves][16] each, then q [16][d + 4], then [kWaves][rows][dv]
  float *m_s = lds, *l_s = lds + kWaves * 16, *q_s = lds + 2 * kWaves * 16, *acc_s = q_s + 16 * (d + 4);
  const int group = nq / nkv, kvh = blockIdx.y, hb = blockIdx.z * 16;
  const int heads = group - hb < 16 ? group - hb : 16;
  const int bx = blockIdx.x, t0 = bx < lead ? bx : lead + (bx - lead) * tile_tokens;
  const int t1 = bx < lead ? t0 + 1 : t0 + tile_tokens < n_tok ? t0 + tile_tokens : n_tok;
  const int rows = (t1 - t0) * heads;               // row: token by token, its heads side by side
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, j = lane >> 4;
  const int mine = r < rows ? r : rows - 1;         // (columns past the rows: nobody stores what they make)
  const int t = t0 + mine / heads, h = kvh * group + hb + mine % heads;
  auto first_seen = [&](int pos) {
    int lo = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    if (chunk > 0) lo = max(lo, pos - pos % chunk);
    return lo;
  };
  const int pos = positions[t], lo = first_seen(pos);
  const int vd = values_in_keys ? d : dv;           // floats of a row of the values' pool
  const float* vbase = values_in_keys ? k_cache : v_cache;
  const int nd = d / 16;

  // the rows' queries; a row's 16-byte pieces lie in other banks than the next row's
  const float* qp = q + ((size_t)t * nq + h) * d + 4 * j;
  float* qr = q_s + r * (d + 4) + 4 * j;
  for (int i = wave; i < nd; i += kWaves) *reinterpret_cast<f4*>(qr + 16 * i) = *reinterpret_cast<const f4*>(qp + 16 * i);
  f4 o[DG][4];
#pragma unroll
  for (int g = 0; g < DG; ++g)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[g][e] = f4{0.f, 0.f, 0.f, 0.f};
  const float slope = slopes ? slopes[h] : 0.f;
  const float inv_cap = softcap > 0.f ? 1.f / softcap : 0.f;
  float m = -INFINITY, l = 0.f;
  __syncthreads();

  // a tile's tokens are of one request, but where two meet: then each request's are walked by themselves
  for (int ta = t0; ta < t1;) {
    const int seq = tok_seq[ta];
    int tb = ta, low = 0x7fffffff, lo_most = 0, pos_least = 0x7fffffff, high = 0;      // the first key that any, that every
    for (; tb < t1 && tok_seq[tb] == seq; ++tb) {                                      // token sees, and the last ones
      const int p = positions[tb], f = first_seen(p);
      low = min(low, f);
      lo_most = max(lo_most, f);
      pos_least = min(pos_least, p);
      high = max(high, p);
    }
    const bool one = ta == t0 && tb == t1, own = t >= ta && t < tb;
    const int* bt = block_tables + (size_t)seq * max_pages;
    const int last = high / kBlock;
    int b = low / kBlock + ((wave - low / kBlock) & (kWaves - 1));
    // the row of the lane's key of block bb in either pool
    auto row_of = [&](int bb) {
      const int key = bb * kBlock + (lane & (kBlock - 1));
      const int seen = key < low ? low : key > high ? high : key;
      return (bt[seen / page_size] * nkv + kvh) * page_size + seen % page_size;
    };
    constexpr bool kEarly = DT <= 8;                // (larger heads: no registers for V ahead of its use)
    f4 ka[DT], va[kEarly ? 4 : 1][DG];
    auto ask_k = [&](int row) {
      const float* kp = k_cache + (size_t)__shfl(row, r, kWave) * d + 4 * j;
#pragma unroll
      for (int i = 0; i < DT; ++i)
        if (i < nd) ka[i] = *reinterpret_cast<const f4*>(kp + 16 * i);
    };
    auto ask_v = [&](int row, int v, f4 (&to)[DG]) {
      const float* vp = vbase + (size_t)__shfl(row, 4 * j + v, kWave) * vd + 4 * r;
#pragma unroll
      for (int g = 0; g < DG; ++g)
        if (64 * g < dv) to[g] = 64 * g + 4 * r < dv ? *reinterpret_cast<const f4*>(vp + 64 * g) : f4{0.f, 0.f, 0.f, 0.f};
    };
    int row = b <= last ? row_of(b) : 0, row_next = 0;
    if (b <= last) ask_k(row);
    for (; b <= last; b += kWaves) {
      const bool full = b * kBlock >= lo_most && b * kBlock + kBlock - 1 <= pos_least, whole = one && full;
      const bool more = b + kWaves <= last;
      if (more) row_next = row_of(b + kWaves);
      if (kEarly && whole) {
#pragma unroll
        for (int v = 0; v < 4; ++v) ask_v(row, v, va[kEarly ? v : 0]);
      }
      __builtin_amdgcn_sched_barrier(0);
      f4 s = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < DT; ++i)
        if (i < nd) {
          const f4 qv = *reinterpret_cast<const f4*>(qr + 16 * i);
#pragma unroll
          for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[i][e], qv[e], s, 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
      if (more) ask_k(row_next);
      __builtin_amdgcn_sched_barrier(0);
      float most = -INFINITY;
      bool sees[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int kk = b * kBlock + 4 * j + v;
        sees[v] = own && kk >= lo && kk <= pos;
        float z = s[v] * scale;
        if (softcap > 0.f) z = softcap * tanhf(z * inv_cap);
        if (slopes) z -= slope * (float)(pos - kk);
        s[v] = z;
        if (sees[v]) most = fmaxf(most, z);
      }
      most = fmaxf(most, lane_xor<16>(most));
      most = fmaxf(most, lane_xor<32>(most));
      const bool any = own && (b + 1) * kBlock > lo && b * kBlock <= pos;       // (a block that a row does not see leaves it as it is)
      const float m_new = any ? fmaxf(m, most) : m;
      const float top = m_new == -INFINITY ? 0.f : m_new;         // (scores of -inf alone so far: weights of 0)
      float sum = 0.f;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        s[v] = sees[v] ? expf(s[v] - top) : 0.f;
        sum += s[v];
      }
      sum += lane_xor<16>(sum);
      sum += lane_xor<32>(sum);
      const float corr = any ? expf(m - top) : 1.f;               // exp(-inf) = 0 on the first block
      l = l * corr + sum;
      m = m_new;
#pragma unroll
      for (int g = 0; g < DG; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[g][e] *= corr;
      if (whole) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          if (!kEarly) ask_v(row, v, va[0]);
#pragma unroll
          for (int g = 0; g < DG; ++g)
            if (64 * g < dv) {
#pragma unroll
              for (int e = 0; e < 4; ++e) o[g][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[kEarly ? v : 0][g][e], s[v], o[g][e], 0, 0, 0);
            }
        }
      } else {
        const int per = full ? tb - ta : 1;
        for (int x = ta; x < tb; x += per) {     // (beside another request's tokens: one product for all of this one's)
          const int px = positions[x], lx = first_seen(px);
          if ((b + 1) * kBlock <= lx || b * kBlock > px) continue;
          const int key = b * kBlock + (lane & (kBlock - 1));
          const int seen = key < lx ? lx : key > px ? px : key;
          const int rx = (bt[seen / page_size] * nkv + kvh) * page_size + seen % page_size;
          f4 ox[DG][4];
#pragma unroll
          for (int g = 0; g < DG; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) ox[g][e] = o[g][e];
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            ask_v(rx, v, va[kEarly ? v : 0]);
#pragma unroll
            for (int g = 0; g < DG; ++g)
              if (64 * g < dv) {
#pragma unroll
                for (int e = 0; e < 4; ++e) ox[g][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[kEarly ? v : 0][g][e], s[v], ox[g][e], 0, 0, 0);
              }
          }
#pragma unroll
          for (int g = 0; g < DG; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[g][e] = (unsigned)(t - x) < (unsigned)per ? ox[g][e] : o[g][e];
        }
      }
      row = row_next;
    }
    ta = tb;
  }
  if (j == 0) {
    m_s[wave * 16 + r] = m;
    l_s[wave * 16 + r] = l;
  }
  if (r < rows) {
#pragma unroll
    for (int g = 0; g < DG; ++g)
#pragma unroll
      for (int v = 0; v < 4; ++v) {                 // dims 64 g + 4 (4 j + v) + e of row r
        const int dim = 64 * g + 16 * j + 4 * v;
        if (dim < dv)
          *reinterpret_cast<f4*>(&acc_s[(wave * rows + r) * dv + dim]) = f4{o[g][0][v], o[g][1][v], o[g][2][v], o[g][3][v]};
      }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < rows * dv; i += 64 * kWaves) {
    const int row = i / dv, dim = i - row * dv, head = kvh * group + hb + row % heads;
    const float sink = sinks ? sinks[head] : -INFINITY;
    float mm = sink;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) mm = fmaxf(mm, m_s[w * 16 + row]);
    float ll = 0.f, total = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float mw = m_s[w * 16 + row];
      const float f = mw == -INFINITY ? 0.f : expf(mw - mm);
      ll += l_s[w * 16 + row] * f;
      total += acc_s[(w * rows + row) * dv + dim] * f;
    }
    if (sinks) ll += expf(sink - mm);
    out[((size_t)(t0 + row / heads) * nq + head) * dv + dim] = total / ll;
  }
}

}  // namespace attn_f32
}  // namespace xi

using namespace xi;

extern "C" {

// Head sizes that `xi_attention_f32` takes.
int xi_attention_f32_takes(int nq, int nkv, int d, int dv) {
  return nkv > 0 && nq % nkv == 0 && d > 0 && d % 16 == 0 && d <= 256 && dv > 0 && dv % 16 == 0 && dv <= 256;
}

// The limit that is set on the dynamic LDS of the kernel for these head sizes: what its widest heads take.
int xi_attention_f32_lds(int d, int dv) {
  const int most = (d > dv ? d : dv) <= 64 ? 64 : (d > dv ? d : dv) <= 128 ? 128 : 256;
  return (int)attn_f32::lds_bytes(16, most, most);
}

// Tokens a workgroup for `rest` tokens of `seqs` requests: one where a request brings fewer than four on average, else the fewest with
// which the workgroups are one round of the compute units, at most 16 (token, head) rows: what a tile saves are reads of keys, what it
// costs are the blocks on its diagonal, a product a token.  Measured, us, 16 heads of 128, tokens a workgroup 1 | 2 | 4 | 8 | 16 (one lane
// a key): a prompt of 20: 14.0 | 10.0 | 12.5 | 18.7 | 30.5 (13.1); of 128: 64 | 41 | 28 | 21 | 33 (57); of 2,048: 4,435 | 2,313 | 1,313 | 809
// | 569 (3,781); 300 tokens behind 1,700: 1,119 | 603 | 323 | 214 | 170 (1,293).
int xi_attention_f32_tile(int rest, int seqs, int nq, int nkv) {
  const int heads = nq / nkv < 16 ? nq / nkv : 16, most = 16 / heads;
  const long long a_token = (long long)nkv * ((nq / nkv + 15) / 16);
  int tile = 1;
  if ((long long)seqs * 4 <= rest)
    while (tile < most && ((long long)rest + tile - 1) / tile * a_token > 256) ++tile;
  return tile;
}

// The operands of `xi_attention_generic` in float32 with as many key heads as value heads; K and V rows of whole 16-byte pieces.
// n_seqs: rows of block_tables; lead: tokens at the front that have a workgroup each (single tokens of `lead` requests, which would
// be walked one after the other in a tile: 30 at 4,000 keys in front of a prompt of 512, 16 heads of 128, 440 us, 3,059 in tiles).  tile: tokens a workgroup of the others (a token's bits do not depend on it), 0: chosen.
int xi_attention_f32(const float* q, const float* k_cache, const float* v_cache, const int* block_tables, int max_pages,
                     const int* tok_seq, const int* positions, float* out, float scale, int window, int page_size, int n_tok, int nq,
                     int nkv, int d, int dv, float softcap, const float* slopes, const float* sinks, int values_in_keys, int chunk,
                     int n_seqs, int lead, int tile, hipStream_t stream) {
  XI_CHECK(n_tok >= 0 && nq > 0 && page_size > 0 && max_pages > 0, "attention_f32: bad sizes T=%d nq=%d page=%d max_pages=%d", n_tok, nq,
           page_size, max_pages);
  XI_CHECK(xi_attention_f32_takes(nq, nkv, d, dv) && nkv <= 65535, "attention_f32: %d heads of %d and %d on %d kv heads", nq, d, dv, nkv);
  XI_CHECK(!values_in_keys || dv <= d, "attention_f32: values that are the keys' first dims need dv <= d");
  XI_CHECK(window >= 0 && chunk >= 0 && softcap >= 0.f, "attention_f32: window %d, chunks of %d, soft cap %g", window, chunk, (double)softcap);
  auto on16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  XI_CHECK(on16(q) && on16(k_cache) && (values_in_keys || on16(v_cache)), "attention_f32: operands must start on 16 bytes");
  if (n_tok == 0) return 0;
  const int heads = nq / nkv < 16 ? nq / nkv : 16;
  const int most_tokens = 16 / heads;
  XI_CHECK(lead >= 0 && lead <= n_tok && tile >= 0 && tile <= most_tokens, "attention_f32: %d tokens a workgroup, %d of %d alone", tile, lead, n_tok);
  const int rest = n_tok - lead;
  if (tile == 0) tile = xi_attention_f32_tile((int)rest, n_seqs - lead, nq, nkv);
  dim3 grid((unsigned)(lead + (rest + tile - 1) / tile), (unsigned)nkv, (unsigned)((nq / nkv + 15) / 16));
  XI_CHECK(grid.z <= 65535u, "attention_f32: too many heads (%d)", nq);
  const size_t lds = attn_f32::lds_bytes(tile * heads, d, dv);
  const int most = d > dv ? d : dv;
#define XI_AF(DT)                                                                                                             \
  do {                                                                                                                        \
    if (lds > 65536) {     /* always the most this kernel may want: another thread's launch may lie between */                \
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_f32::attention_f32_kernel<DT>),              \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, xi_attention_f32_lds(d, dv));      \
      XI_CHECK(e == hipSuccess, "attention_f32: %s", hipGetErrorString(e));                                                   \
    }                                                                                                                         \
    attn_f32::attention_f32_kernel<DT><<<grid, 64 * attn_f32::kWaves, lds, stream>>>(                                         \
        q, k_cache, v_cache, block_tables, max_pages, tok_seq, positions, out, scale, window, page_size, n_tok, lead, tile, nq, nkv, d, dv, softcap, \
        slopes, sinks, values_in_keys, chunk);                                                                                \
  } while (0)
  if (most <= 64) XI_AF(4);
  else if (most <= 128) XI_AF(8);
  else XI_AF(16);
#undef XI_AF
  XI_LAUNCH_CHECK("attention_f32");
  return 0;
}

}  // extern "C"
