// Stable LSD radix sort, the rasterizer's depth sort and tile sort (the
// reference's radix_histogram.comp, radix_scatter.comp and scan_blocks.comp,
// driven by src/core/radix_sort.cpp:58-96). Per digit pass, three launches:
//
//   histogram  per tile of 2048 or 4096 keys, how many hold each digit, stored
//              digit-major (hist[digit * tiles + tile]);
//   scan       one workgroup per digit: the exclusive sum over tiles in place,
//              and the digit's total;
//   scatter    per tile: where each digit starts (the exclusive sum of the
//              digit totals), plus the tile's offset, plus each key's rank
//              among the tile's keys of its digit.
//
// Ranking uses wave64 ballots instead of the reference's barrier-separated
// 1-bit splits: for each digit bit a lane's ballot, and-ed together, gives the
// lanes of its wave holding the same digit, and its rank among them is the
// popcount below it. Each wave ranks a quarter of the tile's keys in
// order, keeping its running digit counts in LDS, so the sort is stable, as
// the tile lists need (test_radix_sort.cpp:15-60 checks the reference's
// against std::stable_sort). The tile's keys then go through LDS in digit
// order, so that each digit's run is written to memory contiguously.
//
// Counts may live in device memory (the tile entries are only known on the
// device): grids are sized for the capacity and tiles past the count exit.
//
// Up to kCountedSortKeys keys the same passes take one launch each
// (radix_pass_kernel): whoever writes the keys also counts each pass's digits per
// tile of 4096 keys, with atomics (digit_count.hpp), the first pass's as the keys
// are made and every later one's as the pass before stores them, and a tile sums
// the tiles' counts itself. At these sizes a launch's own 4 us is most of a pass:
// the kernels of the depth sort took 66 us for 100k keys in 12 launches and take
// 46 in 4, 61 and 41 for 30k. Past it every tile sums too many tiles' counts, one
// after another, and the three-launch passes are the faster ones.
#include "device.hpp"
#include "kernels.hpp"
#include "blockscan.hpp"
#include "digit_count.hpp"

#include <utility>

namespace vsplat {

namespace {

constexpr uint32_t kSortThreads = 256;
// Keys per thread: 8 (tiles of 2048) below kLargeSort keys, 16 (tiles of 4096)
// from there; the larger tiles halve the histogram and its scan, but at 1M keys
// they would leave the 256 compute units short of work.
constexpr uint32_t kSortPerThreadSmall = 8, kSortPerThreadLarge = 16;
constexpr uint32_t kLargeSort = 4u << 20;
constexpr uint32_t kScanThreads = 1024;

__device__ __forceinline__ uint32_t count_of(const uint32_t *countDev, uint32_t countHost) {
  return countDev != nullptr ? *countDev : countHost;
}

// The wave's lanes (of those that have a key) that hold this lane's digit. Per
// digit bit: the bit as a mask (0 or ~0), its ballot straight from one compare,
// and for either half of the lanes the ones that agree; four instructions.
template <uint32_t Bits> __device__ __forceinline__ uint64_t lanes_of_digit(uint32_t digit, bool valid) {
  const uint64_t all = __builtin_amdgcn_ballot_w64(valid);
  uint32_t low = static_cast<uint32_t>(all), high = static_cast<uint32_t>(all >> 32);
#pragma unroll
  for (uint32_t b = 0; b < Bits; ++b) {
    const uint32_t bit = static_cast<uint32_t>(static_cast<int32_t>(digit << (31u - b)) >> 31);
    const uint64_t ones = __builtin_amdgcn_ballot_w64(bit != 0u);
    low &= ~(static_cast<uint32_t>(ones) ^ bit);
    high &= ~(static_cast<uint32_t>(ones >> 32) ^ bit);
  }
  return (static_cast<uint64_t>(high) << 32) | low;
}

template <uint32_t Bits, uint32_t PerThread>
__global__ __launch_bounds__(kSortThreads) void radix_histogram_kernel(const uint32_t *__restrict__ keys, const uint32_t *countDev,
                                                                       uint32_t countHost, uint32_t shift, uint32_t tiles,
                                                                       uint32_t *__restrict__ hist) {
  constexpr uint32_t kRadix = 1u << Bits;
  constexpr uint32_t kSortTile = kSortThreads * PerThread;
  __shared__ uint32_t counts[kRadix];
  for (uint32_t d = threadIdx.x; d < kRadix; d += kSortThreads) counts[d] = 0;
  __syncthreads();
  const uint32_t count = count_of(countDev, countHost);
  const uint32_t base = blockIdx.x * kSortTile;
  if (base < count) {
#pragma unroll
    for (uint32_t r = 0; r < PerThread; ++r) {
      const uint32_t i = base + r * kSortThreads + threadIdx.x;
      if (i < count) atomicAdd(&counts[(keys[i] >> shift) & (kRadix - 1u)], 1u);
    }
  }
  __syncthreads();
  for (uint32_t d = threadIdx.x; d < kRadix; d += kSortThreads) hist[d * tiles + blockIdx.x] = counts[d];
}

// One workgroup per digit: the exclusive sum of that digit's counts over the
// tiles, in place, and the digit's total.
__global__ __launch_bounds__(kScanThreads) void radix_scan_kernel(uint32_t *__restrict__ hist, uint32_t tiles,
                                                                  uint32_t *__restrict__ totals) {
  __shared__ uint32_t waveTotals[kScanThreads / 64];
  uint32_t *row = hist + static_cast<size_t>(blockIdx.x) * tiles;
  uint32_t carry = 0;
  for (uint32_t start = 0; start < tiles; start += kScanThreads) {
    const uint32_t t = start + threadIdx.x;
    const uint32_t v = t < tiles ? row[t] : 0u;
    uint32_t exclusive;
    const uint32_t sum = block_exclusive_sum(v, exclusive, waveTotals);
    if (t < tiles) row[t] = carry + exclusive;
    carry += sum;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

template <uint32_t Bits, uint32_t PerThread>
__global__ __launch_bounds__(kSortThreads) void radix_scatter_kernel(const uint32_t *__restrict__ keysIn, const uint32_t *__restrict__ valsIn,
                                                                     uint32_t *__restrict__ keysOut, uint32_t *__restrict__ valsOut,
                                                                     const uint32_t *countDev, uint32_t countHost, uint32_t shift,
                                                                     uint32_t tiles, const uint32_t *__restrict__ hist,
                                                                     const uint32_t *__restrict__ totals) {
  constexpr uint32_t kRadix = 1u << Bits;
  constexpr uint32_t kWaves = kSortThreads / 64;
  constexpr uint32_t kSortTile = kSortThreads * PerThread;
  constexpr uint32_t kWaveKeys = kSortTile / kWaves; // consecutive keys per wave
  __shared__ uint32_t digitBase[kRadix]; // the digit's global start for this tile, less its start within the tile
  __shared__ uint32_t waveCount[kWaves][kRadix];
  __shared__ uint32_t waveTotals[kWaves];
  __shared__ uint32_t sortedKeys[kSortTile], sortedValues[kSortTile];
  const uint32_t count = count_of(countDev, countHost);
  const uint32_t tileStart = blockIdx.x * kSortTile;
  if (tileStart >= count) return; // the same for the whole workgroup
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;

  // Where this tile's keys of each digit go: the digit's start plus the tile's offset.
  const uint32_t total = threadIdx.x < kRadix ? totals[threadIdx.x] : 0u;
  uint32_t start;
  block_exclusive_sum(total, start, waveTotals);
  if (threadIdx.x < kRadix) digitBase[threadIdx.x] = start + hist[threadIdx.x * tiles + blockIdx.x];
  for (uint32_t x = threadIdx.x; x < kWaves * kRadix; x += kSortThreads) (&waveCount[0][0])[x] = 0;
  __syncthreads();

  // Rank within the wave's 512 keys, in order.
  const uint64_t below = (uint64_t{1} << lane) - 1u;
  uint32_t key[PerThread], val[PerThread], rank[PerThread];
  const uint32_t first = tileStart + wave * kWaveKeys + lane;
#pragma unroll
  for (uint32_t r = 0; r < PerThread; ++r) {
    const uint32_t i = first + r * 64;
    key[r] = i < count ? keysIn[i] : 0u;
    val[r] = i < count ? valsIn[i] : 0u;
  }
#pragma unroll
  for (uint32_t r = 0; r < PerThread; ++r) {
    const bool valid = first + r * 64 < count;
    const uint32_t digit = (key[r] >> shift) & (kRadix - 1u);
    const uint64_t same = lanes_of_digit<Bits>(digit, valid);
    const uint32_t lower = static_cast<uint32_t>(__popcll(same & below));
    __builtin_amdgcn_wave_barrier();
    const uint32_t prior = waveCount[wave][digit];
    rank[r] = prior + lower;
    __builtin_amdgcn_wave_barrier();
    if (valid && lower == 0) waveCount[wave][digit] = prior + static_cast<uint32_t>(__popcll(same));
  }
  __syncthreads();
  // Per digit: where its keys start within the tile (in digit order), and each
  // wave's offset from there.
  {
    const uint32_t d = threadIdx.x;
    uint32_t tileCount = 0;
    if (d < kRadix) {
#pragma unroll
      for (uint32_t w = 0; w < kWaves; ++w) tileCount += waveCount[w][d];
    }
    uint32_t localStart;
    block_exclusive_sum(tileCount, localStart, waveTotals);
    if (d < kRadix) {
      digitBase[d] -= localStart;
      uint32_t running = localStart;
#pragma unroll
      for (uint32_t w = 0; w < kWaves; ++w) {
        const uint32_t c = waveCount[w][d];
        waveCount[w][d] = running;
        running += c;
      }
    }
  }
  __syncthreads();
  // The tile's keys in digit order in LDS, then written out run by run: a
  // digit's keys are consecutive in both, so neighbouring threads store to
  // neighbouring addresses.
#pragma unroll
  for (uint32_t r = 0; r < PerThread; ++r) {
    if (first + r * 64 < count) {
      const uint32_t at = waveCount[wave][(key[r] >> shift) & (kRadix - 1u)] + rank[r];
      sortedKeys[at] = key[r];
      sortedValues[at] = val[r];
    }
  }
  __syncthreads();
  const uint32_t inTile = count - tileStart < kSortTile ? count - tileStart : kSortTile;
#pragma unroll
  for (uint32_t r = 0; r < PerThread; ++r) {
    const uint32_t j = r * kSortThreads + threadIdx.x;
    if (j < inTile) {
      const uint32_t k = sortedKeys[j];
      const uint32_t dst = digitBase[(k >> shift) & (kRadix - 1u)] + j;
      keysOut[dst] = k;
      valsOut[dst] = sortedValues[j];
    }
  }
}

constexpr uint32_t kPassThreads = 512, kPassPerThread = kCountedTile / kPassThreads;

// One whole pass over a tile of kCountedTile keys: `counts` holds every tile's
// digits (kCountedStride words a tile), nextCounts receives those of the next
// pass, whose digit is the bits from nextShift under nextMask (none: the last pass).
template <uint32_t Bits>
__global__ __launch_bounds__(kPassThreads) void radix_pass_kernel(const uint32_t *__restrict__ keysIn, const uint32_t *__restrict__ valsIn,
                                                                  uint32_t *__restrict__ keysOut, uint32_t *__restrict__ valsOut,
                                                                  const uint32_t *countDev, uint32_t countHost, uint32_t shift,
                                                                  const uint32_t *__restrict__ counts, uint32_t nextShift, uint32_t nextMask,
                                                                  uint32_t *__restrict__ nextCounts) {
  constexpr uint32_t kRadix = 1u << Bits, kWaves = kPassThreads / 64, kGroups = kPassThreads / kRadix;
  constexpr uint32_t kWaveKeys = kCountedTile / kWaves; // consecutive keys per wave
  __shared__ uint32_t digitBase[kRadix]; // the digit's global start for this tile, less its start within the tile
  __shared__ uint32_t waveCount[kWaves][kRadix];
  __shared__ uint32_t waveTotals[kWaves];
  __shared__ uint32_t sorted[2 * kCountedTile];
  uint32_t *const sortedKeys = sorted, *const sortedValues = sorted + kCountedTile;
  const uint32_t count = count_of(countDev, countHost);
  const uint32_t tileStart = blockIdx.x * kCountedTile;
  if (tileStart >= count) return; // the same for the whole workgroup
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;

  // The tile's keys, in flight while the counts are summed.
  uint32_t key[kPassPerThread], val[kPassPerThread], rank[kPassPerThread];
  const uint32_t first = tileStart + wave * kWaveKeys + lane;
#pragma unroll
  for (uint32_t r = 0; r < kPassPerThread; ++r) {
    const uint32_t i = first + r * 64;
    key[r] = i < count ? keysIn[i] : 0u;
    val[r] = i < count ? valsIn[i] : 0u;
  }
  // Each digit's keys in the tiles before this one and in all, kGroups threads a
  // digit (their partial sums meet in sortedKeys, which is not in use yet).
  {
    const uint32_t tiles = (count + kCountedTile - 1u) / kCountedTile, d = threadIdx.x % kRadix;
    uint32_t before = 0, all = 0;
#pragma unroll 8
    for (uint32_t t = threadIdx.x / kRadix; t < tiles; t += kGroups) {
      const uint32_t c = counts[t * kCountedStride + d];
      before += t < blockIdx.x ? c : 0u;
      all += c;
    }
    sortedKeys[threadIdx.x] = before;
    sortedKeys[kPassThreads + threadIdx.x] = all;
  }
  for (uint32_t x = threadIdx.x; x < kWaves * kRadix; x += kPassThreads) (&waveCount[0][0])[x] = 0;
  __syncthreads();
  uint32_t before = 0, total = 0;
  if (threadIdx.x < kRadix) {
#pragma unroll 4
    for (uint32_t g = 0; g < kGroups; ++g) {
      before += sortedKeys[g * kRadix + threadIdx.x];
      total += sortedKeys[kPassThreads + g * kRadix + threadIdx.x];
    }
  }
  uint32_t start;
  block_exclusive_sum(total, start, waveTotals);
  if (threadIdx.x < kRadix) digitBase[threadIdx.x] = start + before;

  // Rank within the wave's keys, in order.
  const uint64_t below = (uint64_t{1} << lane) - 1u;
#pragma unroll
  for (uint32_t r = 0; r < kPassPerThread; ++r) {
    const bool valid = first + r * 64 < count;
    const uint32_t digit = (key[r] >> shift) & (kRadix - 1u);
    const uint64_t same = lanes_of_digit<Bits>(digit, valid);
    const uint32_t lower = static_cast<uint32_t>(__popcll(same & below));
    __builtin_amdgcn_wave_barrier();
    const uint32_t prior = waveCount[wave][digit];
    rank[r] = prior + lower;
    __builtin_amdgcn_wave_barrier();
    if (valid && lower == 0) waveCount[wave][digit] = prior + static_cast<uint32_t>(__popcll(same));
  }
  __syncthreads();
  {
    const uint32_t d = threadIdx.x;
    uint32_t tileCount = 0;
    if (d < kRadix) {
#pragma unroll
      for (uint32_t w = 0; w < kWaves; ++w) tileCount += waveCount[w][d];
    }
    uint32_t localStart;
    block_exclusive_sum(tileCount, localStart, waveTotals);
    if (d < kRadix) {
      digitBase[d] -= localStart;
      uint32_t running = localStart;
#pragma unroll
      for (uint32_t w = 0; w < kWaves; ++w) {
        const uint32_t c = waveCount[w][d];
        waveCount[w][d] = running;
        running += c;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < kPassPerThread; ++r) {
    if (first + r * 64 < count) {
      const uint32_t at = waveCount[wave][(key[r] >> shift) & (kRadix - 1u)] + rank[r];
      sortedKeys[at] = key[r];
      sortedValues[at] = val[r];
    }
  }
  __syncthreads();
  const uint32_t inTile = count - tileStart < kCountedTile ? count - tileStart : kCountedTile;
  uint32_t slot[kPassPerThread]; // the counter of the next pass that the key adds to
#pragma unroll
  for (uint32_t r = 0; r < kPassPerThread; ++r) {
    const uint32_t j = r * kPassThreads + threadIdx.x;
    if (j < inTile) {
      const uint32_t k = sortedKeys[j];
      const uint32_t dst = digitBase[(k >> shift) & (kRadix - 1u)] + j;
      keysOut[dst] = k;
      valsOut[dst] = sortedValues[j];
      slot[r] = (dst / kCountedTile) * (nextMask + 1u) + ((k >> nextShift) & nextMask);
    }
  }
  if (nextMask == 0u) return; // the last pass (uniform)
  // The next pass's digits by destination tile: counted in LDS, two 16-bit
  // counters a word (a tile holds 4096 keys), then added to the view's.
  uint32_t *const tally = sortedKeys;
  static_assert(kCountedSortKeys / kCountedTile * kCountedStride / 2 <= 2 * kCountedTile, "the tally fits the sorted keys and values");
  const uint32_t words = ((count + kCountedTile - 1u) / kCountedTile * (nextMask + 1u) + 1u) / 2u;
  __syncthreads();
  for (uint32_t x = threadIdx.x; x < words; x += kPassThreads) tally[x] = 0u;
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < kPassPerThread; ++r) {
    if (r * kPassThreads + threadIdx.x < inTile) atomicAdd(&tally[slot[r] / 2u], (slot[r] & 1u) ? 0x10000u : 1u);
  }
  __syncthreads();
  for (uint32_t x = threadIdx.x; x < words; x += kPassThreads) {
    const uint32_t two = tally[x];
#pragma unroll
    for (uint32_t h = 0; h < 2; ++h) {
      const uint32_t n = h == 0 ? two & 0xFFFFu : two >> 16, at = 2u * x + h;
      if (n != 0u) atomicAdd(&nextCounts[at / (nextMask + 1u) * kCountedStride + (at & nextMask)], n);
    }
  }
}

// ---- Passes with a digit of up to 11 bits, for sorts of more than kCountedSortKeys
// keys: the tile sort on a grid of at most kTileSortTiles tiles, in one pass whose
// digit is the whole tile, and the depth sort in three (10, 10 and 11 bits; 11, 11 and 10 where depths can be negative):
//
//   count    per chunk of keys, how many have each digit (hist[chunk * stride + digit]);
//   scan     the exclusive sums over the chunks, in place, and each digit's keys;
//   scatter  the ranks as in radix_scatter_kernel, and from the totals each tile's
//            range, which has no kernel of its own then.
//
// The tile sort's chunk is 8 entries a tile (8192 for up to 2^10 tiles, 16384 for up
// to 2^11), so that the counts stay an eighth of the entries; the scatter takes it in
// parts of 8192, a workgroup each. The depth sort's is 4096 keys: 1M keys are then
// 245 workgroups. Each XCD takes consecutive chunks, so that a digit's
// neighbouring runs meet in one XCD's cache. What bounds them is the ranking's
// instructions and the runs' partial lines; three workgroups a CU (80
// registers) hide the one behind the other, two took a tenth longer.
//
// The tile sort against two passes of 5 or 6 bits and the kernel for the ranges (us):
// 63 to 33 for 3.4M entries on 920 tiles, 186 to 119 for 15.4M and 305 to 184 for 25M
// on 2040 tiles (400 MB read and written, 77 at the rate of a copy). At 2646 tiles (2.6M
// entries, counts of 2^12 tiles, one workgroup a CU) it is 57 against 53, and up to
// kCountedSortKeys entries the counted passes need no more launches. The depth sort
// against four passes of 8 bits: 85 to 67 for 1M keys, 145 to 107 for 3M, 70 to 58 for
// 400k (11 bits in every pass: 75, 126, 63).
constexpr uint32_t kChunkThreads = 512, kDepthChunk = 4096;
constexpr uint32_t kScanDigits = 16;
__host__ __device__ __forceinline__ uint32_t digit_stride(uint32_t digits) { return (digits + kScanDigits - 1u) / kScanDigits * kScanDigits; }
typedef uint16_t __attribute__((may_alias)) Half;

// The chunk of a workgroup (one past the last where it has none): XCD x, which runs
// workgroups x, x + 8, ..., takes the x-th eighth of the chunks, Parts workgroups each.
__device__ __forceinline__ uint32_t chunks_of(uint32_t count, uint32_t chunk) { return count / chunk + (count % chunk != 0u ? 1u : 0u); }
template <uint32_t Parts> __device__ __forceinline__ uint32_t chunk_of_block(uint32_t chunks) {
  const uint32_t each = (chunks + kRasterXcds - 1u) / kRasterXcds, k = blockIdx.x / kRasterXcds / Parts;
  return k < each ? (blockIdx.x % kRasterXcds) * each + k : chunks;
}

template <uint32_t Bits, uint32_t kChunk>
__global__ __launch_bounds__(kChunkThreads) void digit_count_kernel(const uint32_t *__restrict__ keys, const uint32_t *__restrict__ countDev,
                                                                    uint32_t countHost, uint32_t shift, uint32_t digits, uint32_t mask,
                                                                    uint32_t *__restrict__ hist) {
  constexpr uint32_t kQuads = kChunk / kChunkThreads / 4;
  __shared__ uint32_t counts[1u << Bits];
  const uint32_t count = count_of(countDev, countHost), chunks = chunks_of(count, kChunk), chunk = chunk_of_block<1>(chunks);
  if (chunk >= chunks) return; // the same for the whole workgroup
  const uint32_t inChunk = count - chunk * kChunk < kChunk ? count - chunk * kChunk : kChunk;
  const uint32_t *const chunkKeys = keys + chunk * kChunk;
  uint4 k[kQuads];
#pragma unroll
  for (uint32_t r = 0; r < kQuads; ++r) {
    const uint32_t i = (r * kChunkThreads + threadIdx.x) * 4u;
    if (i + 4u <= inChunk) {
      k[r] = *reinterpret_cast<const uint4 *>(chunkKeys + i);
    } else {
      k[r] = make_uint4(i < inChunk ? chunkKeys[i] : 0u, i + 1u < inChunk ? chunkKeys[i + 1u] : 0u, i + 2u < inChunk ? chunkKeys[i + 2u] : 0u, 0u);
    }
  }
  for (uint32_t d = threadIdx.x; d < digits; d += kChunkThreads) counts[d] = 0u;
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < kQuads; ++r) {
    const uint32_t i = (r * kChunkThreads + threadIdx.x) * 4u;
    if (i < inChunk) atomicAdd(&counts[(k[r].x >> shift) & mask], 1u);
    if (i + 1u < inChunk) atomicAdd(&counts[(k[r].y >> shift) & mask], 1u);
    if (i + 2u < inChunk) atomicAdd(&counts[(k[r].z >> shift) & mask], 1u);
    if (i + 3u < inChunk) atomicAdd(&counts[(k[r].w >> shift) & mask], 1u);
  }
  __syncthreads();
  for (uint32_t d = threadIdx.x; d < digits; d += kChunkThreads) hist[static_cast<size_t>(chunk) * digit_stride(digits) + d] = counts[d];
}

// A workgroup takes kScanDigits neighbouring digits; the chunks are dealt out in
// runs to its 64 groups of as many threads.
constexpr uint32_t kScanGroups = kScanThreads / kScanDigits;
__global__ __launch_bounds__(kScanThreads) void digit_scan_kernel(uint32_t *__restrict__ hist, const uint32_t *__restrict__ countDev, uint32_t countHost,
                                                                  uint32_t chunkSize, uint32_t digits, uint32_t *__restrict__ totals) {
  __shared__ uint32_t sums[kScanGroups][kScanDigits];
  const uint32_t chunks = chunks_of(count_of(countDev, countHost), chunkSize), stride = digit_stride(digits);
  const uint32_t t = threadIdx.x % kScanDigits, g = threadIdx.x / kScanDigits, digit = blockIdx.x * kScanDigits + t;
  const uint32_t each = (chunks + kScanGroups - 1u) / kScanGroups;
  const uint32_t begin = g * each < chunks ? g * each : chunks, end = begin + each < chunks ? begin + each : chunks;
  uint32_t *const column = hist + digit;
  uint32_t sum = 0;
#pragma unroll 16
  for (uint32_t c = begin; c < end; ++c) sum += column[static_cast<size_t>(c) * stride];
  sums[g][t] = sum;
  __syncthreads();
  uint32_t running = 0, total = 0;
#pragma unroll 16
  for (uint32_t k = 0; k < kScanGroups; ++k) {
    const uint32_t v = sums[k][t];
    running += k < g ? v : 0u;
    total += v;
  }
#pragma unroll 16
  for (uint32_t c = begin; c < end; ++c) {
    const uint32_t v = column[static_cast<size_t>(c) * stride];
    column[static_cast<size_t>(c) * stride] = running;
    running += v;
  }
  if (g == 0 && digit < digits) totals[digit] = total;
}

// A chunk's word by a 32-bit offset from its (uniform) start.
__device__ __forceinline__ uint32_t word_at(const uint32_t *__restrict__ chunk, uint32_t i) {
  return *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(chunk) + i * 4u);
}

// valsIn may be null: the values are then the keys' places. ranges may be null.
template <uint32_t Bits, uint32_t kChunk, uint32_t kPart>
__global__ __launch_bounds__(kChunkThreads, 6) void digit_scatter_kernel(
    const uint32_t *__restrict__ keysIn, const uint32_t *__restrict__ valsIn, uint32_t *__restrict__ keysOut, uint32_t *__restrict__ valsOut,
    const uint32_t *__restrict__ countDev, uint32_t countHost, uint32_t shift, uint32_t digits, uint32_t mask,
    const uint32_t *__restrict__ hist, const uint32_t *__restrict__ totals, uint2 *__restrict__ ranges) {
  constexpr uint32_t kPartPerThread = kPart / kChunkThreads, kParts = kChunk / kPart;
  constexpr uint32_t kWaves = kChunkThreads / 64, kRadix = 1u << Bits;
  constexpr uint32_t kOwn = kRadix / kChunkThreads; // consecutive digits per thread
  constexpr uint32_t kWaveKeys = kPart / kWaves;  // consecutive keys per wave
  constexpr uint32_t kCountWords = kWaves * kRadix / 2;
  __shared__ uint32_t digitBase[kRadix]; // where the digit's keys of this part go, less their start within the part
  __shared__ uint32_t waveTotals[kWaves];
  // Each wave's keys per digit in 16 bits (two digits a word), then the part's
  // keys, then its values, in digit order.
  __shared__ uint32_t shared[kCountWords > kPart ? kCountWords : kPart];
  const uint32_t count = count_of(countDev, countHost), chunks = chunks_of(count, kChunk), chunk = chunk_of_block<kParts>(chunks);
  const uint32_t part = blockIdx.x / kRasterXcds % kParts, at = chunk * kChunk + part * kPart;
  if (chunk >= chunks || at >= count) return; // the same for the whole workgroup
  const uint32_t inPart = count - at < kPart ? count - at : kPart;
  const uint32_t *const partKeys = keysIn + at;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, first = wave * kWaveKeys + lane;
  Half *const waveCount = reinterpret_cast<Half *>(shared) + wave * kRadix;
  uint32_t key[kPartPerThread], place[kPartPerThread / 2]; // place: each key's rank, then its place in the part, in 16 bits
#pragma unroll
  for (uint32_t r = 0; r < kPartPerThread; ++r) {
    key[r] = word_at(partKeys, first + r * 64 < inPart ? first + r * 64 : inPart - 1u);
  }
  for (uint32_t x = threadIdx.x; x < kCountWords; x += kChunkThreads) shared[x] = 0u;

  // Where this part's keys of each of the thread's digits go: past the chunk's
  // earlier parts, whose keys are counted again here.
  const uint32_t d = kOwn * threadIdx.x;
  {
    uint32_t n[kOwn], sum = 0, start;
#pragma unroll
    for (uint32_t o = 0; o < kOwn; ++o) {
      n[o] = d + o < digits ? totals[d + o] : 0u;
      sum += n[o];
    }
    block_exclusive_sum(sum, start, waveTotals);
#pragma unroll
    for (uint32_t o = 0; o < kOwn; ++o) {
      if (d + o < digits) digitBase[d + o] = start + hist[static_cast<size_t>(chunk) * digit_stride(digits) + d + o];
      if (ranges != nullptr && chunk == 0 && n[o] != 0u) ranges[d + o] = make_uint2(start, start + n[o]);
      start += n[o];
    }
  }
  __syncthreads();
  if (kParts > 1) {
    for (uint32_t i = threadIdx.x * 4u; i < part * kPart; i += kChunkThreads * 4u) {
      const uint4 k = *reinterpret_cast<const uint4 *>(keysIn + chunk * kChunk + i);
      atomicAdd(&digitBase[(k.x >> shift) & mask], 1u);
      atomicAdd(&digitBase[(k.y >> shift) & mask], 1u);
      atomicAdd(&digitBase[(k.z >> shift) & mask], 1u);
      atomicAdd(&digitBase[(k.w >> shift) & mask], 1u);
    }
    __syncthreads(); // before the starts within the part are taken off
  }

  // Rank within the wave's keys, in order.
  const uint64_t below = (uint64_t{1} << lane) - 1u;
#pragma unroll
  for (uint32_t r = 0; r < kPartPerThread; ++r) {
    const bool valid = first + r * 64 < inPart;
    const uint32_t digit = (key[r] >> shift) & mask;
    const uint64_t same = lanes_of_digit<Bits>(digit, valid);
    const uint32_t lower = static_cast<uint32_t>(__popcll(same & below));
    __builtin_amdgcn_wave_barrier();
    const uint32_t prior = waveCount[digit];
    place[r / 2] = r % 2 == 0 ? prior + lower : place[r / 2] | ((prior + lower) << 16);
    // The rank is formed here and the counter's address again later: kept for
    // later, the lanes' masks and the addresses take 48 registers more.
    asm volatile("" : "+v"(place[r / 2]), "+v"(key[r]));
    __builtin_amdgcn_wave_barrier();
    if (valid && lower == 0) waveCount[digit] = static_cast<Half>(prior + static_cast<uint32_t>(__popcll(same)));
  }
  __syncthreads();
  // Per digit: where its keys start within the part, and each wave's start from there.
  {
    uint32_t n[kOwn] = {}, sum = 0, start;
#pragma unroll
    for (uint32_t o = 0; o < kOwn; o += 2) {
#pragma unroll
      for (uint32_t w = 0; w < kWaves; ++w) {
        const uint32_t two = shared[(w * kRadix + d + o) / 2];
        n[o] += two & 0xFFFFu;
        n[o + 1] += two >> 16;
      }
      sum += n[o] + n[o + 1];
    }
    block_exclusive_sum(sum, start, waveTotals);
#pragma unroll
    for (uint32_t o = 0; o < kOwn; o += 2) {
      uint32_t low = start, high = start + n[o];
      digitBase[d + o] -= low;
      digitBase[d + o + 1] -= high;
      start = high + n[o + 1];
#pragma unroll
      for (uint32_t w = 0; w < kWaves; ++w) {
        const uint32_t two = shared[(w * kRadix + d + o) / 2];
        shared[(w * kRadix + d + o) / 2] = low | (high << 16);
        low += two & 0xFFFFu;
        high += two >> 16;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < kPartPerThread; ++r) {
    place[r / 2] += static_cast<uint32_t>(waveCount[(key[r] >> shift) & mask]) << (r % 2 * 16);
  }
  uint32_t val[kPartPerThread];
#pragma unroll
  for (uint32_t r = 0; r < kPartPerThread; ++r) {
    const uint32_t x = first + r * 64 < inPart ? first + r * 64 : inPart - 1u;
    val[r] = valsIn != nullptr ? word_at(valsIn + at, x) : at + x;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < kPartPerThread; ++r) {
    if (first + r * 64 < inPart) shared[(place[r / 2] >> (r % 2 * 16)) & 0xFFFFu] = key[r];
  }
  __syncthreads();
  uint32_t dst[kPartPerThread];
#pragma unroll
  for (uint32_t r = 0; r < kPartPerThread; ++r) {
    const uint32_t j = r * kChunkThreads + threadIdx.x;
    if (j < inPart) {
      const uint32_t k = shared[j];
      dst[r] = digitBase[(k >> shift) & mask] + j;
      keysOut[dst[r]] = k;
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < kPartPerThread; ++r) {
    if (first + r * 64 < inPart) shared[(place[r / 2] >> (r % 2 * 16)) & 0xFFFFu] = val[r];
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < kPartPerThread; ++r) {
    const uint32_t j = r * kChunkThreads + threadIdx.x;
    if (j < inPart) valsOut[dst[r]] = shared[j];
  }
}

uint32_t div_up(uint64_t a, uint32_t b) { return static_cast<uint32_t>((a + b - 1) / b); }

template <uint32_t Bits, uint32_t Chunk, uint32_t Part>
void digit_pass(hipStream_t stream, const uint32_t *kIn, const uint32_t *vIn, uint32_t *kOut, uint32_t *vOut, const uint32_t *countDev,
                uint32_t capacity, uint32_t shift, uint32_t bits, uint32_t digits, uint32_t *scratch, uint2 *ranges) {
  const uint32_t blocks = div_up(div_up(capacity, Chunk), kRasterXcds) * kRasterXcds, mask = (1u << bits) - 1u;
  uint32_t *totals = scratch, *hist = scratch + digit_stride(digits);
  hipLaunchKernelGGL((digit_count_kernel<Bits, Chunk>), dim3(blocks), dim3(kChunkThreads), 0, stream, kIn, countDev, capacity, shift, digits,
                     mask, hist);
  hipLaunchKernelGGL(digit_scan_kernel, dim3(digit_stride(digits) / kScanDigits), dim3(kScanThreads), 0, stream, hist, countDev, capacity, Chunk,
                     digits, totals);
  hipLaunchKernelGGL((digit_scatter_kernel<Bits, Chunk, Part>), dim3(blocks * (Chunk / Part)), dim3(kChunkThreads), 0, stream, kIn, vIn, kOut,
                     vOut, countDev, capacity, shift, digits, mask, hist, totals, ranges);
}

template <uint32_t Bits>
void counted_pass(hipStream_t stream, const uint32_t *kIn, const uint32_t *vIn, uint32_t *kOut, uint32_t *vOut, const uint32_t *countDev,
                  uint32_t capacity, uint32_t shift, const uint32_t *counts, uint32_t nextShift, uint32_t nextMask, uint32_t *nextCounts) {
  hipLaunchKernelGGL(radix_pass_kernel<Bits>, dim3(div_up(capacity, kCountedTile)), dim3(kPassThreads), 0, stream, kIn, vIn, kOut, vOut,
                     countDev, capacity, shift, counts, nextShift, nextMask, nextCounts);
}

template <uint32_t Bits, uint32_t PerThread>
void sort_pass(hipStream_t stream, const uint32_t *kIn, const uint32_t *vIn, uint32_t *kOut, uint32_t *vOut, const uint32_t *countDev,
               uint32_t capacity, uint32_t shift, uint32_t *scratch) {
  constexpr uint32_t kRadix = 1u << Bits;
  const uint32_t tiles = div_up(capacity, kSortThreads * PerThread);
  uint32_t *totals = scratch;
  uint32_t *hist = scratch + 256;
  hipLaunchKernelGGL((radix_histogram_kernel<Bits, PerThread>), dim3(tiles), dim3(kSortThreads), 0, stream, kIn, countDev, capacity,
                     shift, tiles, hist);
  hipLaunchKernelGGL(radix_scan_kernel, dim3(kRadix), dim3(kScanThreads), 0, stream, hist, tiles, totals);
  hipLaunchKernelGGL((radix_scatter_kernel<Bits, PerThread>), dim3(tiles), dim3(kSortThreads), 0, stream, kIn, vIn, kOut, vOut,
                     countDev, capacity, shift, tiles, hist, totals);
}

template <uint32_t Bits>
void sort_pass(hipStream_t stream, const uint32_t *kIn, const uint32_t *vIn, uint32_t *kOut, uint32_t *vOut, const uint32_t *countDev,
               uint32_t capacity, uint32_t shift, uint32_t *scratch) {
  if (capacity >= kLargeSort) {
    sort_pass<Bits, kSortPerThreadLarge>(stream, kIn, vIn, kOut, vOut, countDev, capacity, shift, scratch);
  } else {
    sort_pass<Bits, kSortPerThreadSmall>(stream, kIn, vIn, kOut, vOut, countDev, capacity, shift, scratch);
  }
}

} // namespace

size_t radix_sort_scratch_words(uint64_t capacity) {
  return 256 + static_cast<size_t>(div_up(capacity, kSortThreads * kSortPerThreadSmall)) * 256u;
}

bool tile_sort_one_pass(uint64_t capacity, uint32_t tiles) { return capacity > kCountedSortKeys && tiles <= kTileSortTiles; }

size_t tile_sort_scratch_words(uint64_t capacity, uint32_t tiles) {
  if (!tile_sort_one_pass(capacity, tiles)) return radix_sort_scratch_words(capacity);
  return static_cast<size_t>(digit_stride(tiles)) * (1 + div_up(capacity, tiles <= kTileSortTiles / 2 ? 4 * kTileSortTiles : 8 * kTileSortTiles));
}
bool tile_sort_from_tmp(uint64_t capacity, uint32_t tileBits, uint32_t tiles) {
  return tile_sort_one_pass(capacity, tiles) || radix_sort_from_tmp(tileBits);
}

void launch_tile_sort(hipStream_t stream, uint32_t *keys, uint32_t *values, uint32_t *tmpKeys, uint32_t *tmpValues,
                      const uint32_t *countDev, uint32_t capacity, uint32_t tileBits, uint32_t tiles, uint32_t *scratch, uint32_t *counts,
                      uint2 *ranges) {
  if (capacity == 0) return;
  if (!tile_sort_one_pass(capacity, tiles)) {
    launch_radix_sort(stream, keys, values, tmpKeys, tmpValues, countDev, capacity, tileBits, scratch, counts);
    launch_tile_ranges(stream, keys, countDev, capacity, tileBits, ranges);
  } else if (tiles <= kTileSortTiles / 2) {
    digit_pass<10, 8192, 8192>(stream, tmpKeys, tmpValues, keys, values, countDev, capacity, 0, tileBits, tiles, scratch, ranges);
  } else {
    digit_pass<11, 16384, 8192>(stream, tmpKeys, tmpValues, keys, values, countDev, capacity, 0, tileBits, tiles, scratch, ranges);
  }
}

size_t radix_count_words(uint64_t capacity, uint32_t bits) {
  if (capacity > kCountedSortKeys) return 0;
  return static_cast<size_t>(div_up(bits, 8)) * div_up(capacity, kCountedTile) * kCountedStride;
}
uint32_t radix_first_mask(uint32_t bits) { return (1u << div_up(bits, div_up(bits, 8))) - 1u; }

bool radix_sort_from_tmp(uint32_t bits) { return div_up(bits, 8) % 2 != 0; }

// Sorts (keys, values) stably by the low `bits` bits of the keys (1 <= bits <=
// 32), in ceil(bits / 8) passes of equal width. The result ends in keys/values;
// tmpKeys/tmpValues are the other half of each pass, and hold the input when the
// number of passes is odd (radix_sort_from_tmp), so that nothing is copied.
// countDev, when given, holds the element count (at most capacity). counts: the
// first pass's digits as the keys' writer counted them, the other passes' words
// zero (radix_count_words of them; null where that is 0).
void launch_radix_sort(hipStream_t stream, uint32_t *keys, uint32_t *values, uint32_t *tmpKeys, uint32_t *tmpValues,
                       const uint32_t *countDev, uint32_t capacity, uint32_t bits, uint32_t *scratch, uint32_t *counts) {
  if (capacity == 0 || bits == 0) return;
  const uint32_t passes = div_up(bits, 8);
  const uint32_t digit = div_up(bits, passes); // even split, at most 8 bits a pass
  const bool odd = radix_sort_from_tmp(bits), counted = radix_count_words(capacity, bits) != 0;
  const size_t passCounts = static_cast<size_t>(div_up(capacity, kCountedTile)) * kCountedStride;
  uint32_t *srcK = odd ? tmpKeys : keys, *srcV = odd ? tmpValues : values, *dstK = odd ? keys : tmpKeys, *dstV = odd ? values : tmpValues;
  for (uint32_t p = 0; p < passes; ++p) {
    // The last pass takes the bits that are left, so that no bit above `bits`
    // (which may carry other data) takes part in the order.
    const uint32_t shift = p * digit, next = shift + digit;
    const uint32_t nextBits = next >= bits ? 0u : (digit < bits - next ? digit : bits - next);
    uint32_t *mine = counted ? counts + p * passCounts : nullptr;
#define VSPLAT_SORT_PASS(BITS)                                                                                                     \
  case BITS:                                                                                                                       \
    if (counted) {                                                                                                                 \
      counted_pass<BITS>(stream, srcK, srcV, dstK, dstV, countDev, capacity, shift, mine, next, (1u << nextBits) - 1u, mine + passCounts); \
    } else {                                                                                                                       \
      sort_pass<BITS>(stream, srcK, srcV, dstK, dstV, countDev, capacity, shift, scratch);                                         \
    }                                                                                                                              \
    break;
    switch (digit < bits - shift ? digit : bits - shift) {
      VSPLAT_SORT_PASS(1)
      VSPLAT_SORT_PASS(2)
      VSPLAT_SORT_PASS(3)
      VSPLAT_SORT_PASS(4)
      VSPLAT_SORT_PASS(5)
      VSPLAT_SORT_PASS(6)
      VSPLAT_SORT_PASS(7)
      VSPLAT_SORT_PASS(8)
    }
#undef VSPLAT_SORT_PASS
    std::swap(srcK, dstK);
    std::swap(srcV, dstV);
  }
}

bool depth_sort_three_pass(uint64_t count) { return count > kCountedSortKeys; }

size_t depth_sort_scratch_words(uint64_t count) {
  if (!depth_sort_three_pass(count)) return radix_sort_scratch_words(count);
  return size_t{2048} * (1 + div_up(count, kDepthChunk));
}

void launch_depth_sort(hipStream_t stream, uint32_t *keys, uint32_t *values, uint32_t *tmpKeys, uint32_t *tmpValues, uint32_t count,
                       bool signs, uint32_t *scratch, uint32_t *counts) {
  if (!depth_sort_three_pass(count)) {
    launch_radix_sort(stream, keys, values, tmpKeys, tmpValues, nullptr, count, 32, scratch, counts);
    return;
  }
  // A key is all ones less the depth's bits: without a sign its highest bit is set,
  // as an invisible splat's is, and takes no part.
  const uint32_t low = signs ? 11 : 10, digits = 1u << low;
  const auto pass = signs ? digit_pass<11, kDepthChunk, kDepthChunk> : digit_pass<10, kDepthChunk, kDepthChunk>;
  pass(stream, tmpKeys, nullptr, keys, values, nullptr, count, 0, low, digits, scratch, nullptr);
  pass(stream, keys, values, tmpKeys, tmpValues, nullptr, count, low, low, digits, scratch, nullptr);
  digit_pass<11, kDepthChunk, kDepthChunk>(stream, tmpKeys, tmpValues, keys, values, nullptr, count, 2 * low, signs ? 10 : 11,
                                           signs ? 1024 : 2048, scratch, nullptr);
}

__global__ void fill_u32_kernel(uint32_t *__restrict__ dst, uint64_t count, uint32_t value) {
  for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < count; i += static_cast<uint64_t>(gridDim.x) * blockDim.x)
    dst[i] = value;
}

// Clears with a kernel rather than hipMemsetAsync, so that the whole step can
// be captured into a graph.
void launch_fill_u32(hipStream_t stream, uint32_t *dst, uint64_t count, uint32_t value) {
  if (count == 0) return;
  const uint64_t blocks64 = (count + 255) / 256;
  const uint32_t blocks = blocks64 < 8192 ? static_cast<uint32_t>(blocks64) : 8192;
  hipLaunchKernelGGL(fill_u32_kernel, dim3(blocks), dim3(256), 0, stream, dst, count, value);
}

// blockIdx.y is the run; a run whose ends are 16-byte aligned goes four words at a time.
__global__ __launch_bounds__(256) void copy_words_kernel(WordCopies c) {
  const uint32_t *from = c.from[blockIdx.y];
  uint32_t *to = c.to[blockIdx.y];
  const uint32_t words = c.words[blockIdx.y], t = blockIdx.x * 256u + threadIdx.x, stride = gridDim.x * 256u;
  const bool wide = ((reinterpret_cast<uintptr_t>(from) | reinterpret_cast<uintptr_t>(to)) & 15u) == 0u;
  const uint32_t vec4 = wide ? words / 4u : 0u;
  for (uint32_t i = t; i < vec4; i += stride) reinterpret_cast<uint4 *>(to)[i] = reinterpret_cast<const uint4 *>(from)[i];
  for (uint32_t i = vec4 * 4u + t; i < words; i += stride) to[i] = from[i];
}

void launch_copy_words(hipStream_t stream, const WordCopies &copies) {
  uint32_t most = 0;
  for (uint32_t k = 0; k < copies.count; ++k) most = copies.words[k] > most ? copies.words[k] : most;
  if (most == 0) return;
  const uint32_t blocks = div_up(most, 1024) < 256 ? div_up(most, 1024) : 256;
  hipLaunchKernelGGL(copy_words_kernel, dim3(blocks, copies.count), dim3(256), 0, stream, copies);
}

// blockIdx.y is the run.
__global__ __launch_bounds__(256) void clear_words_kernel(WordClears c) {
  uint32_t *to = c.to[blockIdx.y];
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < c.words[blockIdx.y]; i += gridDim.x * 256u) to[i] = 0u;
}

void launch_clear_words(hipStream_t stream, const WordClears &clears) {
  uint32_t most = 0;
  for (uint32_t k = 0; k < clears.count; ++k) most = clears.words[k] > most ? clears.words[k] : most;
  if (most == 0) return;
  const uint32_t blocks = div_up(most, 1024) < 256 ? div_up(most, 1024) : 256;
  hipLaunchKernelGGL(clear_words_kernel, dim3(blocks, clears.count), dim3(256), 0, stream, clears);
}

} // namespace vsplat
