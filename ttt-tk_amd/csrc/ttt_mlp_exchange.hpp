// Exchange of partial sums between two workgroups of one (batch, head), and what it needs to know about their placement.
// A word is sent as it is; its slot holds an impossible value (a NaN that is never sent) before and after, so the receiver
// polls the data itself and puts the mark back: no flags, nothing to order.
#pragma once
#include "ttt_mlp_common.hpp"

namespace ttt {

typedef __attribute__((address_space(1))) uint64_t* gword64_t;
constexpr uint32_t WD_EMPTY = 0xffffffffu;
// Two fp32 values as one 8-byte word of the exchange; the mark itself is never sent (a NaN stays a NaN).
TTT_DEV uint64_t wd_pack(float a, float b) {
  const uint32_t lo = min(__builtin_bit_cast(uint32_t, a), WD_EMPTY - 1), hi = min(__builtin_bit_cast(uint32_t, b), WD_EMPTY - 1);
  return (static_cast<uint64_t>(hi) << 32) | lo;
}
TTT_DEV float wd_lo(uint64_t x) { return __builtin_bit_cast(float, static_cast<uint32_t>(x)); }
TTT_DEV float wd_hi(uint64_t x) { return __builtin_bit_cast(float, static_cast<uint32_t>(x >> 32)); }
// A word for the other CU.  On one XCD the L2 is where both meet: the L1 writes through, so a plain store (wavefront scope)
// reaches it and the partner's agent-scope load is answered by it (2.9 k clocks for 16 KiB both ways; agent-scope stores
// 3.4-4.5 k).  For the same reason counters need no release where all of a pair share an XCD (give in ttt_mlp_fwd_wide.hip,
// BWW_GIVEN in ttt_mlp_bwd_wide.hip): a wave's vmcnt(0) says that its stores are in the L2, a barrier collects the waves,
// and the reader's acquire drops what its own L1 holds.  This is how gfx950 works, not what the memory model promises;
// `near` false (no common XCD) takes agent scope and release fences throughout.
TTT_DEV void wd_put(gword64_t q, uint64_t x, bool near) {
  if (near) __hip_atomic_store(q, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  else __hip_atomic_store(q, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Waits until the N words of every lane have arrived.  False: gave up (status word raised).
template <int N>
TTT_DEV bool wd_take(gword64_t q, uint64_t (&w)[N], int* status, uint64_t limit) {
  uint64_t t0 = 0;
  for (unsigned n = 0;; n++) {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < N; k++) w[k] = __hip_atomic_load(q + 64 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int k = 0; k < N; k++) ok = ok && static_cast<uint32_t>(w[k]) != WD_EMPTY && static_cast<uint32_t>(w[k] >> 32) != WD_EMPTY;
    if (__all(ok)) return true;
    const uint64_t now = wall_clock64();
    if (n == 0) t0 = now;
    else if (now - t0 > limit || ((n & 63) == 0 && __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
      raise_status(status);
      return false;
    }
  }
}

// Every workgroup of a pair says which XCD it runs on; the exchanging ones find out whether all n share one.
TTT_DEV void say_xcd(int* word) {
  unsigned xcc;
  asm volatile("s_getreg_b32 %0, hwreg(20, 0, 4)" : "=s"(xcc));   // XCC_ID
  __hip_atomic_store(word, static_cast<int>(xcc) + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// (by a whole wave) alive = false: gave up waiting for one of them
TTT_DEV bool on_one_xcd(int* words, int n, int lane, int* status, uint64_t limit, bool& alive) {
  bool ok = true, here = true;
  if (lane < n) {
    int x;
    const uint64_t t0 = wall_clock64();
    while ((x = __hip_atomic_load(words + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0) {
      if (__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 || wall_clock64() - t0 > limit) {
        raise_status(status);
        ok = false;
        break;
      }
    }
    here = x == __builtin_amdgcn_readfirstlane(x);
  }
  alive = __all(ok);
  return __all(here);
}
// The workgroups that work for several pairs: each adds itself to a pair's word, a byte per XCD; true: all `total` of them are on
// the caller's.
TTT_DEV void say_worker(int* word) {
  unsigned xcc;
  asm volatile("s_getreg_b32 %0, hwreg(20, 0, 4)" : "=s"(xcc));   // XCC_ID
  __hip_atomic_fetch_add(reinterpret_cast<uint64_t*>(word), 1ull << (8 * (xcc & 7)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
TTT_DEV bool workers_here(int* word, int total, int* status, uint64_t limit, bool& alive) {
  unsigned xcc;
  asm volatile("s_getreg_b32 %0, hwreg(20, 0, 4)" : "=s"(xcc));
  uint64_t x;
  bool ok = true;
  const uint64_t t0 = wall_clock64();
  while (((x = __hip_atomic_load(reinterpret_cast<uint64_t*>(word), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) * 0x0101010101010101ull) >> 56 <
         static_cast<uint64_t>(total)) {
    if (__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 || wall_clock64() - t0 > limit) {
      raise_status(status);
      ok = false;
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  alive = __all(ok) && alive;
  return __all(((x >> (8 * (xcc & 7))) & 255) == static_cast<uint64_t>(total));
}
// One thread: waits until `word` has reached `target` and orders what follows after it.  False: gave up.
TTT_DEV bool wait_word(int* word, int target, int* status, uint64_t limit) {
  const uint64_t t0 = wall_clock64();
  while (__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
    if (__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 || wall_clock64() - t0 > limit) {
      raise_status(status);
      return false;
    }
    __builtin_amdgcn_s_sleep(4);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  return true;
}

}  // namespace ttt
