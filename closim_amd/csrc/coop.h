// coop.h — one launch whose work-groups exchange data: a whole inner solve in
// one kernel for meshes so small that launches and kernel boundaries are most
// of the time.
#pragma once

#include "common.h"
#include "ticket.h"

namespace cloth {

// Each work-group publishes a few words; one wave of each polls all
// work-groups' words until none is empty, which also is a grid barrier.  The
// words, and vectors that other work-groups read, are written with relaxed
// agent-scope stores: they reach the point where the XCDs' caches are
// coherent, so no cache is written back, and a store counts as done once its
// wave has waited for it (coop_drain).  Vectors are read with plain loads
// after an agent-scope acquire fence.  Measured per exchange (256 threads a
// work-group): 1.1 us for 2 work-groups, 1.2 us for 8, 1.7 us for 32, 2.1 us
// for 64; a counter barrier with agent-scope release and acquire fences and a
// read of the partials 1.7, 1.7, 3.6 and 5.7 us.
constexpr unsigned kCoopMaxBlocks = 64;
constexpr unsigned kCoopWords = 8;
constexpr unsigned kCoopSets = 4;
constexpr unsigned kCoopSpin = 1u << 20;  // polls before an exchange gives up (about a second)
constexpr uint64_t kCoopEmpty = ~0ull;

struct CoopSlots {
  uint64_t w[kCoopSets][kCoopWords][kCoopMaxBlocks];  // set to all ones before each launch
  uint64_t gave_up;                                   // not all ones: some work-group waited in vain
};
struct CoopExchange {
  CoopSlots* s;
  uint32_t polls;  // before an exchange gives up
};

template <class T>
__device__ __forceinline__ T coop_load(const T* p) {
  return __hip_atomic_load(const_cast<T*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void coop_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// waits until this wave's stores have reached the coherence point
__device__ __forceinline__ void coop_drain() { __builtin_amdgcn_s_waitcnt(0x0f70); }
// a double as a word that is never the empty marker
__device__ __forceinline__ uint64_t coop_word(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  return u == kCoopEmpty ? 0x7ff8000000000000ull : u;
}

// By one full wave of each work-group (at most kCoopMaxBlocks of them): lane
// b receives work-group b's words (zeros past the last work-group).  `turn`
// counts the exchanges from 0; the words rotate through kCoopSets sets, and a
// work-group empties its words of the set two exchanges old, which everyone
// has read (each published its words of the exchange in between).  False when
// the others do not come.
template <int NW>
__device__ __forceinline__ bool coop_exchange(const CoopExchange& ex, uint32_t& turn, const uint64_t (&mine)[NW],
                                              uint64_t (&got)[NW]) {
  static_assert(NW <= (int)kCoopWords, "slot words");
  CoopSlots* s = ex.s;
  const uint32_t lane = threadIdx.x % kWave, set = turn % kCoopSets, old = (turn + 2) % kCoopSets;
  turn++;
  coop_drain();  // the words emptied last time are, before these can be seen
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < NW; k++) coop_store(&s->w[set][k][blockIdx.x], mine[k]);
  }
  if (lane < kCoopWords) coop_store(&s->w[old][lane][blockIdx.x], kCoopEmpty);
  const bool in = lane < gridDim.x;
#pragma unroll
  for (int k = 0; k < NW; k++) got[k] = in ? kCoopEmpty : 0;
  for (uint32_t i = 0; i < ex.polls; i++) {
    bool wait = false;
    if (in)
#pragma unroll
      for (int k = 0; k < NW; k++) {
        if (got[k] == kCoopEmpty) got[k] = coop_load(&s->w[set][k][lane]);
        wait = wait || got[k] == kCoopEmpty;
      }
    if (!__ballot(wait)) return true;
    if ((i & 1023u) == 1023u && coop_load(&s->gave_up) != kCoopEmpty) return false;
  }
  if (lane == 0) coop_store(&s->gave_up, (uint64_t)1);
  return false;
}

static_assert(CoopTicket::kRound == kXcds, "a ticket counts rounds over the XCDs");

// One solver's exchange: its slots, and the compute units it may wait on
// (those the device has now: a partition or a mask may leave fewer than 256).
struct CoopState {
  DevBuf<CoopSlots> slots;
  int device = -1;
  unsigned cus = 0;
  uint32_t polls = kCoopSpin;
  bool gave_up = false;  // an exchange of this solver waited in vain: no such launches any more
  void setup() {  // on the current device
    CS_HIP(hipGetDevice(&device));
    int n = 0;
    CS_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device));
    cus = n > 0 ? (unsigned)n : 0;
  }
};

}  // namespace cloth
