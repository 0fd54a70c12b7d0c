// The parts of the rows' sums of squares that a product behind a folded norm needs at its end (linear_thin.hip, linear_mid.hip), brought into
// LDS by loads that write LDS.  They are the first thing such a kernel asks for, and every instruction in
// front of its first weights is time without traffic: 32 tested loads a thread for one row of 256 parts were 0.9 us of a product of 3.5
// (1,024 wide), one load a wave is 0.1.
#pragma once
#include "common.h"

namespace xi {

// Most numbers, rounded up to whole loads of 64.
constexpr int fold_parts_room(int n) { return (n + kWave - 1) / kWave * kWave; }

// n numbers from `from` on into `to` (LDS, room for fold_parts_room(n)), by WAVES waves.  The caller waits for them (they are the oldest of its
// loads) and for the other waves.  (s_nop: the wait state that such a load wants behind a scalar write of m0.)
template <int WAVES>
__device__ __forceinline__ void fetch_fold_parts(const float* __restrict__ from, int n, float* to, int wave, int lane) {
  const unsigned lds = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)to);
  for (int i = wave * kWave; i < n; i += WAVES * kWave) {
    const int at = i + lane < n ? i + lane : n - 1;
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(at * 4u), "s"(from), "s"(lds + 4u * i) : "memory", "m0");
  }
}

// 1 / rms of the row whose `parts` parts start at `row`: sixteen neighbouring lanes share them out, the lane `sub` those from sub on in steps of
// sixteen, in this order, and add theirs up by halves.
__device__ __forceinline__ float fold_inverse(const float* row, int parts, int sub, float inv_h, float eps) {
  float t = 0.f;
#pragma unroll 8
  for (int p = sub; p < parts; p += 16) t += row[p];
  t += lane_xor<8>(t);
  t += lane_xor<4>(t);
  t += lane_xor<2>(t);
  t += lane_xor<1>(t);
  return rsqrtf(t * inv_h + eps);
}

// All but the last N of this wave's loads have landed.  N is at most what is issued between those that are waited for and here: a count of more
// than are on their way waits for none, and loads of read-only operands are the compiler's to move behind an asm (of the slots asked for at a
// kernel's start one goes into the branch that has a second tile).
template <int N>
__device__ __forceinline__ void wait_all_but() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

}  // namespace xi
