// index_sort.h -- the positions of an index tensor ordered by value, those of one value in increasing position.
//
// A stable radix sort of 11 bits a pass, least significant first: two passes for values below 4 M (one below 2048, three
// beyond), and which it is the kernels find out themselves, so that the host neither waits nor has to know.  A pass is two
// launches: index_count_kernel counts each tile's digits, index_scatter_kernel works out where the tile's entries go from the
// counts of all tiles and moves them.  Launches of passes that no value needs return at once.
//
// The sizes are those where launches and their latency are all that counts (65536 entries are 256 KB, which a few CUs read
// out of their L2): tiles of 2048 entries to a block of 16 waves, so that 32 blocks share that and each reads 128 KB of counts.
// Ranks within a wave come from ballots, one per bit of the digit, and so need no atomics and keep the order.
//
// Whole sorts in us, here | rocPRIM's radix_sort_pairs, which sorts blocks of these sizes and merges them:
//   entries  8193: 24 | 24    20000: 24 | 35    65536, values below 2048: 19 | 38, below 4 M: 28 | 38, any: 38 | 38
//   entries 12000: 25 | 26    32768: 25 | 35   262144, values below 2048: 28 | 93, below 4 M: 47 | 93, any: 65 | 93
// Six empty launches take 16.  Values beyond 4 M cost a third pass, 33 us at 8193 entries; the library's time steps up between
// 12000 and 20000 and from there these kernels are not slower for any values, so the line lies at 16384.  The upper end is where
// the counts that every block reads become as many as the entries.
#pragma once

#include "common.h"

namespace cthip {

constexpr uint32_t kSortDigitBits = 11, kSortDigits = 1u << kSortDigitBits;
constexpr uint32_t kSortTile = 2048, kSortThreads = 1024, kSortWaves = kSortThreads / 64, kSortRounds = kSortTile / kSortThreads;
constexpr uint32_t kSortMinEntries = 16384;                       // more than that
constexpr uint32_t kSortMaxTiles = 128;                           // two words of `bits` to a lane
constexpr uint32_t kSortMaxEntries = kSortMaxTiles * kSortTile;

struct IndexSort {
  const int32_t* index;
  uint32_t n, tiles;
  int32_t* key[2];        // the last pass writes to [0]
  int32_t* position[2];
  uint32_t* counts;       // [tiles][kSortDigits / 2], two counts to a word
  uint32_t* bits;         // [tiles]: the bits that are set in any value of the tile
};

inline size_t index_sort_array(uint32_t n) { return ((size_t)n * 4 + 255) / 256 * 256; }
inline size_t index_sort_bytes(uint32_t n) {
  const size_t tiles = (n + kSortTile - 1) / kSortTile;
  return 4 * index_sort_array(n) + tiles * kSortDigits * 2 + kSortMaxTiles * 4;
}

__device__ inline int index_sort_passes(const IndexSort& a) {
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t v = lane < a.tiles ? a.bits[lane] : 0u;
  if (lane + 64 < a.tiles) v |= a.bits[lane + 64];
  return __ballot(v >> (2 * kSortDigitBits)) ? 3 : __ballot(v >> kSortDigitBits) ? 2 : 1;
}

template <int PASS>
__global__ void __launch_bounds__(kSortThreads) index_count_kernel(const IndexSort a) {
  __shared__ uint32_t count[kSortDigits];
  __shared__ uint32_t any;
  const int32_t* src = a.index;
  if constexpr (PASS > 0) {
    const int passes = index_sort_passes(a);
    if (PASS >= passes) return;
    src = a.key[(passes - PASS) & 1];
  }
  for (uint32_t d = threadIdx.x; d < kSortDigits; d += kSortThreads) count[d] = 0;
  if (threadIdx.x == 0) any = 0;
  __syncthreads();
  uint32_t seen = 0;
#pragma unroll
  for (uint32_t r = 0; r < kSortRounds; ++r) {
    const uint32_t i = blockIdx.x * kSortTile + r * kSortThreads + threadIdx.x;
    if (i < a.n) {
      const uint32_t v = (uint32_t)src[i];
      atomicAdd(&count[(v >> (PASS * kSortDigitBits)) & (kSortDigits - 1)], 1u);
      seen |= v;
    }
  }
  if constexpr (PASS == 0) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) seen |= __shfl_xor(seen, m, 64);
    if ((threadIdx.x & 63u) == 0) atomicOr(&any, seen);
  }
  __syncthreads();
  a.counts[blockIdx.x * (kSortDigits / 2) + threadIdx.x] = count[2 * threadIdx.x] | count[2 * threadIdx.x + 1] << 16;
  if (PASS == 0 && threadIdx.x == 0) a.bits[blockIdx.x] = any;
}

template <int PASS>
__global__ void __launch_bounds__(kSortThreads) index_scatter_kernel(const IndexSort a) {
  static_assert(kSortDigits == 2 * kSortThreads, "a thread has two digits");
  __shared__ uint32_t own[kSortWaves][kSortDigits / 2];   // the waves' counts, two to a word, then where they begin
  __shared__ uint32_t base[kSortDigits];                  // where the tile's entries of a digit go
  __shared__ uint32_t wave_total[kSortWaves];
  const int passes = index_sort_passes(a);
  if (PASS >= passes) return;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
  const int from = (passes - PASS) & 1, to = from ^ 1;
  const int32_t* src = PASS == 0 ? a.index : a.key[from];
  for (uint32_t k = 0; k < kSortWaves; ++k) own[k][tid] = 0;
  __syncthreads();

  typedef uint16_t __attribute__((may_alias)) Count;
  Count* mine = reinterpret_cast<Count*>(own[w]);
  uint32_t value[kSortRounds], rank[kSortRounds];
  int32_t position[kSortRounds];
#pragma unroll
  for (uint32_t r = 0; r < kSortRounds; ++r) {
    const uint32_t i = blockIdx.x * kSortTile + w * (64 * kSortRounds) + r * 64 + lane;
    const bool valid = i < a.n;
    value[r] = valid ? (uint32_t)src[i] : 0u;
    position[r] = valid ? (PASS == 0 ? (int32_t)i : a.position[from][i]) : 0;
    const uint32_t d = (value[r] >> (PASS * kSortDigitBits)) & (kSortDigits - 1);
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (uint32_t b = 0; b < kSortDigitBits; ++b) {
      const bool set = (d >> b) & 1u;
      const uint64_t sets = __ballot(set);
      peers &= set ? sets : ~sets;
    }
    const uint32_t ahead = (uint32_t)__popcll(peers & ((1ull << lane) - 1));
    const uint32_t earlier = mine[d];
    rank[r] = earlier + ahead;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // all lanes have read before the first of each digit adds
    __builtin_amdgcn_wave_barrier();
    if (valid && ahead == 0) mine[d] = (Count)(earlier + (uint32_t)__popcll(peers));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }

  // digits 2 tid and 2 tid + 1: how many there are, and how many of them in earlier tiles
  uint32_t total0 = 0, total1 = 0, prior0 = 0, prior1 = 0;
#pragma unroll 8
  for (uint32_t t = 0; t < a.tiles; ++t) {
    const uint32_t word = a.counts[t * (kSortDigits / 2) + tid];
    if (t < blockIdx.x) {
      prior0 += word & 0xffffu;
      prior1 += word >> 16;
    }
    total0 += word & 0xffffu;
    total1 += word >> 16;
  }
  uint32_t sum = total0 + total1;   // of the digits up to this thread's, within the wave
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    const uint32_t lower = __shfl_up(sum, m, 64);
    if (lane >= (uint32_t)m) sum += lower;
  }
  if (lane == 63) wave_total[w] = sum;
  __syncthreads();   // and the waves' counts are complete
  uint32_t before = sum - total0 - total1;
  for (uint32_t k = 0; k < w; ++k) before += wave_total[k];
  base[2 * tid] = before + prior0;
  base[2 * tid + 1] = before + total0 + prior1;
  uint32_t run = 0;   // two sums of at most 2048
  for (uint32_t k = 0; k < kSortWaves; ++k) {
    const uint32_t word = own[k][tid];
    own[k][tid] = run;
    run += word;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < kSortRounds; ++r) {
    const uint32_t i = blockIdx.x * kSortTile + w * (64 * kSortRounds) + r * 64 + lane;
    const uint32_t d = (value[r] >> (PASS * kSortDigitBits)) & (kSortDigits - 1);
    const uint32_t at = base[d] + mine[d] + rank[r];
    if (i < a.n && at < a.n) {   // the second never fails unless another stream writes the index meanwhile
      a.key[to][at] = (int32_t)value[r];
      a.position[to][at] = position[r];
    }
  }
}

// Six launches on `block` of index_sort_bytes(n); 1 <= n <= kSortMaxEntries.
inline void index_sort(hipStream_t s, const int32_t* index, uint32_t n, void* block, const int32_t** key,
                       const int32_t** position) {
  IndexSort a;
  a.index = index;
  a.n = n;
  a.tiles = (n + kSortTile - 1) / kSortTile;
  char* at = static_cast<char*>(block);
  const size_t array = index_sort_array(n);
  for (int k = 0; k < 2; ++k) {
    a.key[k] = reinterpret_cast<int32_t*>(at + (2 * k) * array);
    a.position[k] = reinterpret_cast<int32_t*>(at + (2 * k + 1) * array);
  }
  a.counts = reinterpret_cast<uint32_t*>(at + 4 * array);
  a.bits = a.counts + (size_t)a.tiles * (kSortDigits / 2);
  const dim3 grid(a.tiles), threads(kSortThreads);
  hipLaunchKernelGGL(index_count_kernel<0>, grid, threads, 0, s, a);
  hipLaunchKernelGGL(index_scatter_kernel<0>, grid, threads, 0, s, a);
  hipLaunchKernelGGL(index_count_kernel<1>, grid, threads, 0, s, a);
  hipLaunchKernelGGL(index_scatter_kernel<1>, grid, threads, 0, s, a);
  hipLaunchKernelGGL(index_count_kernel<2>, grid, threads, 0, s, a);
  hipLaunchKernelGGL(index_scatter_kernel<2>, grid, threads, 0, s, a);
  *key = a.key[0];
  *position = a.position[0];
}

}  // namespace cthip
