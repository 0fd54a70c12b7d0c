// The walk of a bfloat16 tile product over K that the many-row kernels share (linear_tile.hip says what it is
// and what it was measured against; moe_tile.hip takes the rows of x and w from other places): BM rows of
// x by BN rows of w, tiles of 64 k brought into LDS rings by loads that write LDS, two sets of operand
// registers a wave.
#pragma once
#include <type_traits>

#include "common.h"

namespace xi {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

namespace tile {

// (A load that writes LDS wants one wait state behind a scalar write of m0, which the compiler gives its own loads and cannot give inside an asm.)
__device__ __forceinline__ void load_lds16(const void* base, unsigned lane_off, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_off), "s"(base), "s"(lds_addr)
               : "memory", "m0");
}

template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// f(0), f(1), .. f(N - 1) with the number as a constant
template <int I, int N, typename F>
__device__ __forceinline__ void steps(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    steps<I + 1, N>(f);
  }
}

__device__ __forceinline__ bf16x8 lds8(const unsigned char* p) { return *reinterpret_cast<const bf16x8*>(p); }

// BM rows of x by BN rows of w a workgroup, BK = 64 k a tile; WGM x WGN waves, each (BM / WGM) by (BN / WGN); rings of S stages of x and
// of SW (S or S + 1) of w.  What a tile waits for is the way from memory, and that is w's: x is in a cache, read by every workgroup of its rows.  A
// stage is asked for again when its tile has been read, S - 1 tiles' time before it is needed (1.6 us for 256 by 256, two stages), and w
// that comes from memory takes longer than that.  A third stage of w alone fits the 160 KB (tiles of 192 to 256 rows).
// Two stages of both | the third of w, us, every call its own weights: gated, N=17408 K=5120, 512 rows 190 | 174, 2,048 579 | 537; N=12288 K=4096, 2,048
// rows 312 | 297; 2,048 rows of N=4096 K=12288 272 | 220, of N=5120 K=5120 121 | 102; 2,400 rows of N=5120 K=17408 in tiles of 224 374 | 343; 8 gated
// experts of 6144 at width 4096, 300 to 660 pairs each 625 | 576 (all pairs on one expert's weights, which a cache holds, took 536 of 636); without a gate
// 473 | 438; at width 1024 and 2048 1 to 2%.  A load a line of the tiles four ahead instead, to bring them into L2, costs the load unit 10%.
template <int BM, int BN, int WGM, int WGN, int S, int SW = S>
struct Walk {
  static constexpr int BK = 64, kBK = BK;
  static constexpr int kRowBytes = BK * 2;
  static constexpr int CPR = BK / 8;                                // 16-byte chunks of a row
  static constexpr int PS = 1;                                      // rows that share a 256-byte phase differ in place: p >> PS
  static constexpr int RPL = 1024 / kRowBytes;                      // rows a wave-wide load brings
  static constexpr int KSTEPS = BK / 32;
  static constexpr int NWV = WGM * WGN;
  static constexpr int TM = BM / WGM / 16, TN = BN / WGN / 16;      // 16 x 16 tiles of a wave
  static constexpr int WBYTES = BN * kRowBytes, XBYTES = BM * kRowBytes;
  static constexpr int WI = WBYTES / 1024, XI = XBYTES / 1024;      // wave-wide loads of a tile
  // every wave issues the same number of loads a tile, x's first (where they do not come out even, the last few bring the last chunk again)
  static constexpr int LX = (XI + NWV - 1) / NWV, LW = (WI + NWV - 1) / NWV, LPW = LX + LW;
  static constexpr int LDS = SW * WBYTES + S * XBYTES;
  static_assert(SW * LPW < 64 && S >= 2 && (SW == S || SW == S + 1) && LDS <= 160 * 1024, "the tiles in flight must fit the load counter");
  static_assert(BM % (16 * WGM) == 0 && BN % (16 * WGN) == 0, "whole 16 x 16 tiles a wave");

  // which of w's (t >= LX) or of x's
  static __device__ __forceinline__ int load_number(int wave, int t) {
    const bool is_w = t >= LX;
    const int i = wave + NWV * (is_w ? t - LX : t), n = is_w ? WI : XI;
    return n % NWV == 0 || i < n ? i : n - 1;
  }

  // What a lane brings of every tile: per load t of its wave the byte offset of its chunk from the operand's base.
  // `offset(is_w, p)`: of row p of the tile (rows past the end: of any row; nobody stores what they make).
  template <typename F>
  static __device__ __forceinline__ void offsets(unsigned (&ld_off)[LPW], F offset) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int t = 0; t < LPW; ++t) {
      const bool is_w = t >= LX;
      const int p = RPL * load_number(wave, t) + lane / CPR;      // row within the operand's tile
      const int ch = (lane % CPR) ^ ((p >> PS) & (CPR - 1));       // the chunk that belongs at this lane's place
      ld_off[t] = offset(is_w, p) + (unsigned)(ch * 16);
    }
  }

  // acc (features of w down, rows of x across: a lane holds features 4 j .. 4 j + 3 of row r of a 16 x 16 tile) = the sums
  // over k_tiles tiles of 64 k from wbase and xbase on.
  static __device__ __forceinline__ void run(const bf16* wbase, const bf16* xbase, const unsigned (&ld_off)[LPW], int k_tiles,
                                             unsigned char* smem, f32x4 (&acc)[TN][TM]) {
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, j = lane >> 4;
    const int wm = wave % WGM, wn = wave / WGM;

    // the t-th of this wave's loads of tile kt, into stage st
    auto fetch_one = [&](int kt, int st, int t) {
      const int ii = load_number(wave, t);
      const bool is_w = t >= LX;
      // (the same in all lanes of a wave: made a scalar by hand)
      const unsigned long long a = (unsigned long long)(uintptr_t)((is_w ? wbase : xbase) + (size_t)kt * kBK);
      const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a), hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
      load_lds16(reinterpret_cast<const void*>((uintptr_t)(((unsigned long long)hi << 32) | lo)), ld_off[t],
                 __builtin_amdgcn_readfirstlane(lds0 + (unsigned)(is_w ? st * WBYTES : SW * WBYTES + st * XBYTES) + (unsigned)ii * 1024u));
    };

    // where this lane reads its operands within a stage: row r of a 16-row tile, chunk 4 ks + j at
    // its permuted place (16 rows further on the permutation is the same)
    unsigned rd[KSTEPS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) rd[ks] = (unsigned)(r * kRowBytes + 16 * ((4 * ks + j) ^ ((r >> PS) & (CPR - 1))));
    const unsigned w_rd = (unsigned)(wn * TN * 16) * kRowBytes;
    const unsigned x_rd = SW * WBYTES + (unsigned)(wm * TM * 16) * kRowBytes;

#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
      for (int b = 0; b < TM; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto read = [&](int ks, bf16x8 (&wa)[TN], bf16x8 (&xb)[TM]) {
#pragma unroll
      for (int a = 0; a < TN; ++a) wa[a] = lds8(smem + w_rd + rd[ks] + a * 16 * kRowBytes);
#pragma unroll
      for (int b = 0; b < TM; ++b) xb[b] = lds8(smem + x_rd + rd[ks] + b * 16 * kRowBytes);
    };
    constexpr int NM = TN * TM, READS = TN + TM;
    // A step's products, wa x xb, with the reads of the next step's operands between them, in the order in which its products
    // want them and done by three quarters of these, and `load(i)` before product i.  (A wave with products to issue goes
    // before one that waits to: setprio, 1 to 3%.)
    auto step = [&](const bf16x8 (&wa)[TN], const bf16x8 (&xb)[TM], const unsigned char* Tw, const unsigned char* Tx, int ks,
                    bf16x8 (&wn_)[TN], bf16x8 (&xn_)[TM], auto load) {
      __builtin_amdgcn_s_setprio(1);
      steps<0, NM>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        constexpr int SPAN = NM * 3 / 4;      // (a half or all of them: level to 5% behind)
        steps<0, READS>([&](auto oc) {
          constexpr int o = decltype(oc)::value;
          if constexpr (o * SPAN / READS == i) {
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (o == 0) wn_[0] = lds8(Tw + w_rd + rd[ks]);
            else if constexpr (o <= TM) xn_[o - 1] = lds8(Tx + x_rd + rd[ks] + (o - 1) * 16 * kRowBytes);
            else wn_[o - TM] = lds8(Tw + w_rd + rd[ks] + (o - TM) * 16 * kRowBytes);
          }
        });
        load(ic);
        acc[i / TM][i % TM] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[i / TM], xb[i % TM], acc[i / TM][i % TM], 0, 0, 0);
      });
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
    };

    // The walk, one barrier a tile.  A tile's two 32-wide steps have their operands in two sets of
    // registers; each set is read from LDS between the products of the other: the second step's
    // between the first step's, the next tile's first step's (behind the barrier that says the tile
    // has landed) between the second step's, and there too the loads of the tile S ahead.  One at a
    // time: eight waves that leave the barrier and ask for a whole set at once keep LDS busy for
    // half a step while the matrix cores have nothing (tiles of 256 by 256, 3,000 x 5120 x 17408:
    // 428 us so, 414 one at a time; 2,048 x 12288 x 4096 gated 334 and 320), and a wave that asks
    // for all its loads at once waits until the load unit has taken them (it takes a compute unit's
    // 48 to 64 KB a tile at about 55 bytes a clock).  Tiles past the slice's last are asked for all
    // the same (from the last one's place) and read too, so that the number of loads in flight and
    // the code do not depend on where the walk is.
    static_assert(KSTEPS == 2, "two sets of operand registers, one a step");
#pragma unroll
    for (int p = 0; p < SW; ++p)
#pragma unroll
      for (int t = p < S ? 0 : LX; t < LPW; ++t) fetch_one(p < k_tiles ? p : k_tiles - 1, p, t);
    bf16x8 wa0[TN], xb0[TM], wa1[TN], xb1[TM];
    wait_loads<(S - 1) * LPW + (SW - S) * LW>();       // this wave's loads of the first tile have landed
    __syncthreads();                   // everybody's have
    read(0, wa0, xb0);
    int st = 0, sw = 0;                // the tile's stages
    for (int kt = 0; kt < k_tiles; ++kt) {
      step(wa0, xb0, smem + sw * WBYTES, smem + st * XBYTES, 1, wa1, xb1, [](auto) {});
      // this wave's loads of the next tile have landed (behind its x only w of later tiles was asked for, or whole later tiles)
      wait_loads<(S - 2) * LPW + (SW - S) * LW>();
      __builtin_amdgcn_s_waitcnt(0xC07F);   // (lgkmcnt(0): the operands above are in registers)
      __syncthreads();                 // everybody's: the next tile is whole, and this tile's stage is free
      const int filled = st, filled_w = sw;
      const int nxt = kt + S < k_tiles ? kt + S : k_tiles - 1, nxt_w = kt + SW < k_tiles ? kt + SW : k_tiles - 1;
      st = st + 1 == S ? 0 : st + 1;
      sw = sw + 1 == SW ? 0 : sw + 1;
      __builtin_amdgcn_sched_barrier(0);
      step(wa1, xb1, smem + sw * WBYTES, smem + st * XBYTES, 0, wa0, xb0, [&](auto ic) {
        steps<0, LPW>([&](auto tc) {
          constexpr int t = decltype(tc)::value;
          if constexpr (t * NM / LPW == decltype(ic)::value) {
            __builtin_amdgcn_sched_barrier(0);
            fetch_one(t < LX ? nxt : nxt_w, t < LX ? filled : filled_w, t);
          }
        });
      });
    }
    wait_loads<0>();     // the tiles asked for past the end are still on their way into LDS
  }
};

}  // namespace tile
}  // namespace xi
