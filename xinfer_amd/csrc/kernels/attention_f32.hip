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
// A block's K is asked for a block ahead, its V before its scores are made: a wave would wait for the page number, K and V one after the
// other.  The page numbers of a wave's next 64 blocks are one load, a lane a block (pages in whole blocks; others are looked up key by key);
// heads of whole tiles (WHOLE: 64, 80, 96, 112, 128, 256) are a kernel without tests around their loads, behind which the compiler waits for more
// than it needs.
//
// Measured on MI355X, 32 heads of 128 on 8 kv heads, against a page's number looked up for every block and tests around every load (us):
// prompts of 200, 127, 54, 172 and 9 tokens 67.6 (79.4), a prompt of 1,024 208 (248), 8 single tokens at up to 330 keys 15.9 (17.3), one at
// 4,096 keys 99 (125); 16 heads on 8, a prompt of 1,024, heads of 64 71 (113), a prompt of 512, heads of 256 118 (182).  One lane a key took 396,
// 1,990, 54 and 738 for the first four.  Counters: on prompts a unit issues an instruction in half of its busy cycles (vector ones in 36%; matrix cores
// busy 12%), for 8 single tokens in a third (23%; 20%, of whose 16 columns a decode step uses the heads of a kv head): what bounds it is a block's
// chain (K, scores, their sums over lanes, V) in the two waves a SIMD that its registers leave room for.
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

// DT: 16-dim tiles that the registers have room for (head sizes up to 16 DT); SINGLE: every workgroup has one token;
// WHOLE: both head sizes are 16 DT
template <int DT, bool SINGLE, bool WHOLE>
__global__ __launch_bounds__(64 * kWaves, 1) void attention_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_pages, const int* __restrict__ tok_seq, const int* __restrict__ positions,
    float* __restrict__ out, float scale, int window, int page_size, int n_tok, int lead, int tile_tokens, int nq, int nkv, int d_, int dv_,
    float softcap, const float* __restrict__ slopes, const float* __restrict__ sinks, int values_in_keys, int chunk) {
  constexpr int DG = (DT + 3) / 4;                  // groups of 64 value dims
  const int d = WHOLE ? 16 * DT : d_, dv = WHOLE ? 16 * DT : dv_;
  extern __shared__ float lds[];                    // m and l [kWaves][16] each, then q [16][d + 4], then [kWaves][rows][dv]
  float *m_s = lds, *l_s = lds + kWaves * 16, *q_s = lds + 2 * kWaves * 16, *acc_s = q_s + 16 * (d + 4);
  const int group = nq / nkv, kvh = blockIdx.y, hb = blockIdx.z * 16;
  const int heads = group - hb < 16 ? group - hb : 16;
  const int bx = blockIdx.x, t0 = bx < lead ? bx : lead + (bx - lead) * tile_tokens;
  const int t1 = SINGLE || bx < lead ? t0 + 1 : t0 + tile_tokens < n_tok ? t0 + tile_tokens : n_tok;
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
  constexpr int kQ = (DT + kWaves - 1) / kWaves;
  constexpr bool kHold = DT > 4 && DT <= 8;         // (in registers from then on)
  f4 qx[kQ], qh[kHold ? DT : 1];
#pragma unroll
  for (int i = 0; i < kQ; ++i)
    if (wave + i * kWaves < nd) qx[i] = *reinterpret_cast<const f4*>(qp + 16 * (wave + i * kWaves));
  f4 o[DG][4];
#pragma unroll
  for (int g = 0; g < DG; ++g)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[g][e] = f4{0.f, 0.f, 0.f, 0.f};
  const float slope = slopes ? slopes[h] : 0.f;
  const float inv_cap = softcap > 0.f ? 1.f / softcap : 0.f;
  float m = -INFINITY, l = 0.f;
  const bool in_page = page_size % kBlock == 0;

  // a tile's tokens are of one request, but where two meet: then each request's are walked by themselves
  for (int ta = t0; ta < t1;) {
    const int seq = tok_seq[ta];
    int tb = ta, low = 0x7fffffff, lo_most = 0, pos_least = 0x7fffffff, high = 0;      // the first key that any, that every
    for (; tb < t1 && (SINGLE || tok_seq[tb] == seq); ++tb) {                          // token sees, and the last ones
      const int p = positions[tb], f = first_seen(p);
      low = min(low, f);
      lo_most = max(lo_most, f);
      pos_least = min(pos_least, p);
      high = max(high, p);
    }
    const bool one = ta == t0 && tb == t1, own = t >= ta && t < tb;
    const int* bt = block_tables + (size_t)seq * max_pages;
    const int last = high / kBlock;
    const int b0 = low / kBlock + ((wave - low / kBlock) & (kWaves - 1));
    // Pages in whole blocks: lane i keeps what is added to a key of the wave's block b0 + kWaves (64 n + i) to give its row, so that 64
    // blocks' pages are one trip to memory.
    int place = 0;
    auto ask_pages = [&](int from) {
      const int bb = from + kWaves * lane < last ? from + kWaves * lane : last, page = bb * kBlock / page_size;
      place = (bt[page] * nkv + kvh - page) * page_size;
    };
    // the row in either pool of the lane's key of block b, or of the nearest one from `from` to `to`
    auto row_of = [&](int b, int at, int from, int to) {           // (at: what belongs to block b's page)
      const int key = b * kBlock + (lane & (kBlock - 1));
      const int seen = key < from ? from : key > to ? to : key;
      if (in_page) return at + seen;
      return (bt[seen / page_size] * nkv + kvh) * page_size + seen % page_size;
    };
    constexpr bool kEarly = DT <= 8;                // (larger heads: no registers for V ahead of its use)
    constexpr int kSlots = SINGLE && kEarly ? 2 : 1;               // blocks whose operands have registers
    f4 ka[kSlots][DT], va[kSlots][kEarly ? 4 : 1][DG];
    int row[kSlots], at[kSlots], row_next = 0, at_next = 0;
    auto ask_k = [&](int row, f4 (&to)[DT]) {
      const float* kp = k_cache + (size_t)__shfl(row, r, kWave) * d + 4 * j;
#pragma unroll
      for (int i = 0; i < DT; ++i)
        if (i < nd) to[i] = *reinterpret_cast<const f4*>(kp + 16 * i);
    };
    auto ask_v = [&](int row, int v, f4 (&to)[DG]) {
      const float* vp = vbase + (size_t)__shfl(row, 4 * j + v, kWave) * vd + 4 * r;
#pragma unroll
      for (int g = 0; g < DG; ++g)
        if (64 * g < dv) to[g] = 64 * g + 4 * r < dv ? *reinterpret_cast<const f4*>(vp + 64 * g) : f4{0.f, 0.f, 0.f, 0.f};
    };
    auto full = [&](int b) { return b * kBlock >= lo_most && b * kBlock + kBlock - 1 <= pos_least; };
    // (a token by itself: what it does not see of a block reads its nearest key already)
    auto whole = [&](int b) { return SINGLE || (one && full(b)); };
    auto ask_vs = [&](int b, int slot) {
      if (kEarly && whole(b)) {
#pragma unroll
        for (int v = 0; v < 4; ++v) ask_v(row[slot], v, va[slot][kEarly ? v : 0]);
      }
    };
    // Block b, the wave's n-th: its K (two slots: and V) is in the slot or on its way there; the slot's next block is asked for.
    auto next_row = [&](int b, int n) {
      if (in_page && ((n + kSlots) & 63) == 0) ask_pages(b + kSlots * kWaves);
      at_next = __builtin_amdgcn_readlane(place, (n + kSlots) & 63);
      return row_of(b + kSlots * kWaves, at_next, low, high);
    };
    auto block = [&](int b, int n, auto slot_c) {
      constexpr int slot = decltype(slot_c)::value;
      const bool more = b + kSlots * kWaves <= last;
      if (kSlots == 1) {
        if (more) row_next = next_row(b, n);
        ask_vs(b, slot);
      }
      __builtin_amdgcn_sched_barrier(0);
      f4 s = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < DT; ++i)
        if (i < nd) {
          const f4 qv = kHold ? qh[kHold ? i : 0] : *reinterpret_cast<const f4*>(qr + 16 * i);
#pragma unroll
          for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[slot][i][e], qv[e], s, 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
        if (kSlots > 1) row_next = next_row(b, n);
        ask_k(row_next, ka[slot]);
      }
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
      if (whole(b)) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          if (!kEarly) ask_v(row[slot], v, va[slot][0]);
#pragma unroll
          for (int g = 0; g < DG; ++g)
            if (64 * g < dv) {
#pragma unroll
              for (int e = 0; e < 4; ++e) o[g][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[slot][kEarly ? v : 0][g][e], s[v], o[g][e], 0, 0, 0);
            }
        }
      } else {
        const int per = full(b) ? tb - ta : 1;
        for (int x = ta; x < tb; x += per) {     // (beside another request's tokens: one product for all of this one's)
          const int px = positions[x], lx = first_seen(px);
          if ((b + 1) * kBlock <= lx || b * kBlock > px) continue;
          const int rx = row_of(b, at[slot], lx, px);
          f4 ox[DG][4];
#pragma unroll
          for (int g = 0; g < DG; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) ox[g][e] = o[g][e];
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            ask_v(rx, v, va[slot][kEarly ? v : 0]);
#pragma unroll
            for (int g = 0; g < DG; ++g)
              if (64 * g < dv) {
#pragma unroll
                for (int e = 0; e < 4; ++e) ox[g][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[slot][kEarly ? v : 0][g][e], s[v], ox[g][e], 0, 0, 0);
              }
          }
#pragma unroll
          for (int g = 0; g < DG; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[g][e] = (unsigned)(t - x) < (unsigned)per ? ox[g][e] : o[g][e];
        }
      }
      row[slot] = row_next;
      at[slot] = at_next;
      if (kSlots > 1 && more) ask_vs(b + kSlots * kWaves, slot);
    };
    if (in_page) ask_pages(b0);
#pragma unroll
    for (int s = 0; s < kSlots; ++s)
      if (b0 + s * kWaves <= last) {
        at[s] = __builtin_amdgcn_readlane(place, s);
        row[s] = row_of(b0 + s * kWaves, at[s], low, high);
        ask_k(row[s], ka[s]);
        if (kSlots > 1) ask_vs(b0 + s * kWaves, s);
      }
    if (ta == t0) {                // (asked for above, wanted now)
#pragma unroll
      for (int i = 0; i < kQ; ++i)
        if (wave + i * kWaves < nd) *reinterpret_cast<f4*>(qr + 16 * (wave + i * kWaves)) = qx[i];
      __syncthreads();
      if constexpr (kHold)
#pragma unroll
        for (int i = 0; i < DT; ++i)
          if (i < nd) qh[i] = *reinterpret_cast<const f4*>(qr + 16 * i);
    }
    for (int n = 0, b = b0; b <= last; n += kSlots, b += kSlots * kWaves) {
      block(b, n, std::integral_constant<int, 0>{});
      if constexpr (kSlots > 1)
        if (b + kWaves <= last) block(b + kWaves, n + 1, std::integral_constant<int, kSlots - 1>{});
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
  // Single tokens with their operands two blocks ahead where half of the compute units are idle: 64 and 128 workgroups of up to 400 keys 15.9 | 18.5
  // us, 17.3 | 19.4 one block ahead; at 256 memory is what they wait for (23.3 | 22.7) and at 512 the kernel of the tiles is ahead, 40.3 | 44.4.
  const bool single = (rest == 0 || tile == 1) && (long long)grid.x * grid.y * grid.z <= 128;
  const size_t lds = attn_f32::lds_bytes(tile * heads, d, dv);
  const int most = d > dv ? d : dv;
#define XI_AF(DT)                                                                                                             \
  do {                                                                                                                        \
    const bool whole = d == 16 * DT && dv == d;                                                                               \
    if (single && whole) XI_AF1(DT, true, true);                                                                              \
    else if (single) XI_AF1(DT, true, false);                                                                                 \
    else if (whole) XI_AF1(DT, false, true);                                                                                  \
    else XI_AF1(DT, false, false);                                                                                            \
  } while (0)
#define XI_AFW(DT)                                                                                                            \
  do {                                                                                                                        \
    if (single) XI_AF1(DT, true, true);                                                                                       \
    else XI_AF1(DT, false, true);                                                                                             \
  } while (0)
#define XI_AF1(DT, SINGLE, WHOLE)                                                                                                    \
  do {                                                                                                                        \
    if (lds > 65536) {     /* always the most this kernel may want: another thread's launch may lie between */                \
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_f32::attention_f32_kernel<DT, SINGLE, WHOLE>),              \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, xi_attention_f32_lds(d, dv));      \
      XI_CHECK(e == hipSuccess, "attention_f32: %s", hipGetErrorString(e));                                                   \
    }                                                                                                                         \
    attn_f32::attention_f32_kernel<DT, SINGLE, WHOLE><<<grid, 64 * attn_f32::kWaves, lds, stream>>>(                                         \
        q, k_cache, v_cache, block_tables, max_pages, tok_seq, positions, out, scale, window, page_size, n_tok, lead, tile, nq, nkv, d, dv, softcap, \
        slopes, sinks, values_in_keys, chunk);                                                                                \
  } while (0)
  // Sizes between 64 and 128 have kernels of their own: in the one for 128 the tests on every load cost more than its other steps give wherever
  // many single tokens wait for memory: 64 heads of 96 on 8, 32 tokens at 330 keys 22.5 us, 19.5 so (21.3 with a page looked up for every block and the
  // tests), a prompt of 1,024 378, 317 (368).  Values of another size than the keys stay there: 32 heads of 128 with values of 64, the same 25.2 (23.2).
  if (most <= 64) XI_AF(4);
  else if (d == dv && d == 80) XI_AFW(5);
  else if (d == dv && d == 96) XI_AFW(6);
  else if (d == dv && d == 112) XI_AFW(7);
  else if (most <= 128) XI_AF(8);
  else XI_AF(16);
#undef XI_AF
#undef XI_AF1
  XI_LAUNCH_CHECK("attention_f32");
  return 0;
}

}  // extern "C"
