// sort.hip — stable LSD radix sort (8-bit digits) with LDS ranking.
//
// Per pass: (1) per-tile digit histogram in LDS, written digit-major;
// (2) one-block exclusive scan of the histogram; (3) each tile re-reads its
// keys and ranks them stably with wave64 ballots (match mask per digit) plus
// per-wave LDS digit counts, then scatters.  Up to kBlockSortMax pairs are
// sorted by one work-group in one launch instead (k_sort_block).
#include <algorithm>

#include "sort.h"

namespace cloth {

constexpr int kSortBlock = 256;
constexpr int kWaves = kSortBlock / kWave;
static_assert(kSortBlock == (int)kRadix, "a tile is kRadix keys per item");

template <int kItems>
__global__ void __launch_bounds__(kSortBlock) k_radix_hist(const uint64_t* __restrict__ keys, size_t n, int shift,
                                                           uint32_t* __restrict__ hist, unsigned nblocks) {
  __shared__ uint32_t h[kRadix];
  for (int i = threadIdx.x; i < kRadix; i += kSortBlock) h[i] = 0;
  __syncthreads();
  const size_t base = (size_t)blockIdx.x * (kSortBlock * kItems);
  for (int it = 0; it < kItems; it++) {
    const size_t i = base + (size_t)it * kSortBlock + threadIdx.x;
    if (i < n) atomicAdd(&h[(keys[i] >> shift) & 0xff], 1u);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < kRadix; d += kSortBlock) hist[(size_t)d * nblocks + blockIdx.x] = h[d];
}

// Exclusive prefix of one value per thread of a 1024-thread block; *total
// receives the block's sum.
__device__ __forceinline__ uint32_t block_scan(uint32_t x, uint32_t* total) {
  __shared__ uint32_t s_wave[16], s_total;
  const uint32_t lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
  uint32_t v = x;
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t y = __shfl_up(v, d, kWave);
    if (lane >= (uint32_t)d) v += y;
  }
  if (lane == kWave - 1) s_wave[wid] = v;
  __syncthreads();
  if (wid == 0) {
    uint32_t w = lane < 16 ? s_wave[lane] : 0;
    for (int d = 1; d < 16; d <<= 1) {
      const uint32_t y = __shfl_up(w, d, kWave);
      if (lane >= (uint32_t)d) w += y;
    }
    if (lane < 16) s_wave[lane] = w;
    if (lane == 15) s_total = w;
  }
  __syncthreads();
  const uint32_t before = (wid ? s_wave[wid - 1] : 0) + v - x;
  *total = s_total;
  __syncthreads();
  return before;
}

// Exclusive scan of `cnt` u32 in place, one block of 1024 threads, four
// consecutive values per thread and round (35,000 entries: 35 us when each
// thread walked its own run of 35, 12 us here).
__global__ void __launch_bounds__(1024) k_scan_one_block(uint32_t* a, size_t cnt) {
  uint32_t carry = 0;
  for (size_t base = 0; base < cnt; base += 4096) {
    const size_t i = base + (size_t)threadIdx.x * 4;
    uint32_t v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = i + k < cnt ? a[i + k] : 0;
    uint32_t total;
    uint32_t run = carry + block_scan(v[0] + v[1] + v[2] + v[3], &total);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (i + k < cnt) a[i + k] = run;
      run += v[k];
    }
    carry += total;
  }
}

// The whole sort by one work-group: key digits and positions packed into a
// word per pair, in registers (wave w holds a contiguous run of the pairs, 64
// per round), ranked like k_radix_scatter with per-wave digit counts, and
// permuted through LDS between the passes.  Short sorts are latency: three
// launches a pass took 25 us for 5,000 pairs (five passes of the contact keys
// 125 us), this one 38 us in all.
constexpr int kBlockSortThreads = 1024, kBlockSortWaves = kBlockSortThreads / kWave, kBlockSortItems = 16;
constexpr size_t kBlockSortMax = (size_t)kBlockSortThreads * kBlockSortItems;
constexpr int kPosBits = 14;
static_assert(kBlockSortMax == (size_t)1 << kPosBits, "positions fill their bits");
constexpr size_t kBlockSortLds = kBlockSortMax * 8 + (size_t)kBlockSortWaves * kRadix * 4;

__global__ void __launch_bounds__(kBlockSortThreads) k_sort_block(const uint64_t* __restrict__ kin,
                                                                  const uint32_t* __restrict__ vin, uint32_t n,
                                                                  int begin_bit, int bits, uint64_t* __restrict__ kout,
                                                                  uint32_t* __restrict__ vout) {
  extern __shared__ __align__(16) unsigned char sort_lds[];
  uint64_t* buf = reinterpret_cast<uint64_t*>(sort_lds);
  uint32_t* cnt = reinterpret_cast<uint32_t*>(buf + kBlockSortMax);  // [wave][digit]
  const uint32_t tid = threadIdx.x, lane = tid % kWave, wid = tid / kWave;
  const uint32_t rounds = (n + kBlockSortThreads - 1) / kBlockSortThreads;
  const uint32_t first = wid * rounds * kWave + lane;  // + 64 per round
  const uint64_t lt_mask = lane ? ((~0ull) >> (64 - lane)) : 0ull;
  const uint64_t mask = (1ull << bits) - 1;
  uint64_t w[kBlockSortItems];
  uint32_t rank[kBlockSortItems];
#pragma unroll
  for (int r = 0; r < kBlockSortItems; r++) {
    const uint32_t i = first + r * kWave;
    w[r] = (uint32_t)r < rounds && i < n ? (((kin[i] >> begin_bit) & mask) << kPosBits) | i : 0;
  }
  for (int shift = kPosBits; shift < kPosBits + bits; shift += 8) {
    for (uint32_t k = tid; k < kBlockSortWaves * (uint32_t)kRadix; k += kBlockSortThreads) cnt[k] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kBlockSortItems; r++) {
      if ((uint32_t)r < rounds) {
        const bool valid = first + r * kWave < n;
        const uint32_t digit = (uint32_t)(w[r] >> shift) & 0xffu;
        uint64_t match = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; bit++) {
          const uint64_t bset = __ballot(valid && ((digit >> bit) & 1));
          match &= ((digit >> bit) & 1) ? bset : ~bset;
        }
        const uint32_t before = __popcll(match & lt_mask);
        uint32_t* c = &cnt[wid * kRadix + digit];
        rank[r] = *c + before;
        __builtin_amdgcn_wave_barrier();
        if (valid && before == 0) *c = rank[r] + __popcll(match);
        __builtin_amdgcn_wave_barrier();
      }
    }
    __syncthreads();
    // exclusive scan in (digit, wave) order: four waves of one digit per thread
    {
      uint32_t v[4];
      uint32_t* c = &cnt[(tid % 4) * 4 * kRadix + tid / 4];
#pragma unroll
      for (int k = 0; k < 4; k++) v[k] = c[k * kRadix];
      uint32_t total;
      uint32_t run = block_scan(v[0] + v[1] + v[2] + v[3], &total);
#pragma unroll
      for (int k = 0; k < 4; k++) {
        c[k * kRadix] = run;
        run += v[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kBlockSortItems; r++) {
      if ((uint32_t)r < rounds && first + r * kWave < n)
        buf[cnt[wid * kRadix + ((uint32_t)(w[r] >> shift) & 0xffu)] + rank[r]] = w[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kBlockSortItems; r++) {
      const uint32_t i = first + r * kWave;
      if ((uint32_t)r < rounds && i < n) w[r] = buf[i];
    }
    // (the next pass writes the counts before, and buf after, barriers)
  }
#pragma unroll
  for (int r = 0; r < kBlockSortItems; r++) {
    const uint32_t i = first + r * kWave;
    if ((uint32_t)r < rounds && i < n) {
      const uint32_t p = (uint32_t)w[r] & (uint32_t)(kBlockSortMax - 1);
      kout[i] = kin[p];
      vout[i] = vin[p];
    }
  }
}

bool sort_setup() {
  int dev = 0, optin = 0, base = 0;
  CS_HIP(hipGetDevice(&dev));
  if (hipDeviceGetAttribute(&optin, hipDeviceAttributeSharedMemPerBlockOptin, dev) != hipSuccess) optin = 0;
  CS_HIP(hipDeviceGetAttribute(&base, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  const size_t need = kBlockSortLds + 1024;  // with its static LDS
  if (need > (size_t)std::max(optin, base)) return false;
  return need <= (size_t)base ||
         hipFuncSetAttribute(reinterpret_cast<const void*>(&k_sort_block), hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)kBlockSortLds) == hipSuccess;
}

template <int kItems>
__global__ void __launch_bounds__(kSortBlock) k_radix_scatter(const uint64_t* __restrict__ kin,
                                                              const uint32_t* __restrict__ vin, size_t n, int shift,
                                                              const uint32_t* __restrict__ hist, unsigned nblocks,
                                                              uint64_t* __restrict__ kout, uint32_t* __restrict__ vout) {
  __shared__ uint32_t base_off[kRadix];
  __shared__ uint32_t running[kRadix];
  __shared__ uint32_t wave_cnt[kWaves][kRadix];
  for (int d = threadIdx.x; d < kRadix; d += kSortBlock) {
    base_off[d] = hist[(size_t)d * nblocks + blockIdx.x];
    running[d] = 0;
  }
  const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
  const uint64_t lt_mask = lane ? ((~0ull) >> (64 - lane)) : 0ull;
  const size_t base = (size_t)blockIdx.x * (kSortBlock * kItems);
  for (int it = 0; it < kItems; it++) {
    for (int d = threadIdx.x; d < kWaves * kRadix; d += kSortBlock) (&wave_cnt[0][0])[d] = 0;
    __syncthreads();
    const size_t i = base + (size_t)it * kSortBlock + threadIdx.x;
    const bool valid = i < n;
    uint64_t key = 0;
    uint32_t val = 0, digit = 0;
    if (valid) {
      key = kin[i];
      val = vin[i];
      digit = (uint32_t)((key >> shift) & 0xff);
    }
    // lanes holding the same digit (valid lanes only)
    uint64_t match = __ballot(valid);
#pragma unroll
    for (int bit = 0; bit < 8; bit++) {
      const uint64_t bset = __ballot(valid && ((digit >> bit) & 1));
      match &= ((digit >> bit) & 1) ? bset : ~bset;
    }
    const uint32_t rank_in_wave = __popcll(match & lt_mask);
    if (valid && rank_in_wave == 0) wave_cnt[wid][digit] = __popcll(match);
    __syncthreads();
    if (valid) {
      uint32_t off = running[digit] + rank_in_wave;
      for (int w = 0; w < wid; w++) off += wave_cnt[w][digit];
      const size_t dst = (size_t)base_off[digit] + off;
      kout[dst] = key;
      vout[dst] = val;
    }
    __syncthreads();
    for (int d = threadIdx.x; d < kRadix; d += kSortBlock) {
      uint32_t t = 0;
      for (int w = 0; w < kWaves; w++) t += wave_cnt[w][d];
      running[d] += t;
    }
    __syncthreads();
  }
}

bool radix_sort_pairs(hipStream_t st, uint64_t* keys, uint32_t* vals, uint64_t* keys_tmp, uint32_t* vals_tmp,
                      size_t n, int begin_bit, int end_bit, SortScratch& scratch) {
  if (n <= 1 || end_bit <= begin_bit) return false;
  const int bits = end_bit - begin_bit;
  if (scratch.block_sort && n <= kBlockSortMax && bits + kPosBits <= 64) {
    // (whole digits, as the passes below: bits past end_bit take part too)
    const int whole = std::min((bits + 7) / 8 * 8, 64 - kPosBits);
    hipLaunchKernelGGL(k_sort_block, dim3(1), dim3(kBlockSortThreads), kBlockSortLds, st, keys, vals, (uint32_t)n,
                       begin_bit, whole, keys_tmp, vals_tmp);
    CS_LAUNCH_CHECK();
    return true;
  }
  const unsigned nblocks = (unsigned)radix_tiles(n);
  const size_t entries = (size_t)kRadix * nblocks;
  const bool small = radix_items(n) == 4;
  if (scratch.hist_cap < entries) throw HipError("radix sort scratch too small");
  bool in_tmp = false;
  for (int shift = begin_bit; shift < end_bit; shift += 8) {
    const uint64_t* ki = in_tmp ? keys_tmp : keys;
    const uint32_t* vi = in_tmp ? vals_tmp : vals;
    uint64_t* ko = in_tmp ? keys : keys_tmp;
    uint32_t* vo = in_tmp ? vals : vals_tmp;
    hipLaunchKernelGGL(small ? k_radix_hist<4> : k_radix_hist<16>, dim3(nblocks), dim3(kSortBlock), 0, st, ki, n,
                       shift, scratch.hist, nblocks);
    hipLaunchKernelGGL(k_scan_one_block, dim3(1), dim3(1024), 0, st, scratch.hist, entries);
    hipLaunchKernelGGL(small ? k_radix_scatter<4> : k_radix_scatter<16>, dim3(nblocks), dim3(kSortBlock), 0, st, ki,
                       vi, n, shift, scratch.hist, nblocks, ko, vo);
    CS_LAUNCH_CHECK();
    in_tmp = !in_tmp;
  }
  return in_tmp;
}

}  // namespace cloth
