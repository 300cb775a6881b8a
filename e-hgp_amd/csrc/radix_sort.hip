// Stable LSD radix sort of (uint64 key, uint32 value) pairs, 8-bit digits.
//
// Pass structure (one pass per digit), on tiles of 1 024 or 4 096 keys:
//   1. tile histograms: 64-key groups of equal digits are found with eight
//      ballots and counted with one LDS atomic per group;
//   2. base offsets of (digit, tile), digit-major, so equal digits keep tile
//      order: up to kDirectTiles tiles each scatter workgroup sums the counts
//      it needs itself; beyond that a multi-block inclusive scan over
//      [digit][tile] leaves them;
//   3. scatter: each of the four waves of a tile ranks its keys in order
//      (64-key chunks, eight ballots, a per-digit running count in LDS), the
//      tile is reordered by digit in LDS, and the reordered tile is written
//      out in index order, so the stores of a digit run are contiguous.  Key
//      order inside a digit is (wave, chunk, lane), the input order: the pass
//      is stable.
// Passes whose digit is the same for every key copy instead of scattering, so
// ping-pong buffers stay consistent.  Up to kSmallSort keys are placed by
// counting the keys before each (rs_rank).
//
// Below a few hundred thousand keys a pass is bound by its launches and by the
// few workgroups it has: tiles of 1 024 and the two-launch pass took the sorts
// of a 50 000-point build from four launches and 13 workgroups a pass to two
// and 49, the sort by counting those of a 256-point build from 128 launches to
// four (index of 256 points: 0.91 -> 0.26 ms with the rest of the build).
#include "radix_sort.hpp"

namespace mhgp {

namespace {

constexpr int kDirectTiles = 128;
constexpr int kSmallSort = 8192;
constexpr int kSmallBlock = 1024;
constexpr int kDigits = 256;
constexpr int kSortBlock = 256;
constexpr int kWaves = kSortBlock / 64;

__device__ inline uint64_t lanes_below() {
  const int lane = (int)(threadIdx.x & 63u);
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// Lanes of the wave holding a valid key with the same digit as this lane.
__device__ inline uint64_t digit_match(bool valid, uint32_t dig) {
  uint64_t match = __ballot(valid);
#pragma unroll
  for (int bit = 0; bit < 8; ++bit) {
    const uint64_t bal = __ballot(valid && ((dig >> bit) & 1u));
    match &= ((dig >> bit) & 1u) ? bal : ~bal;
  }
  return match;
}

// counts: [digit][tile], or [tile][digit] when the scatter sums them itself
template <int kTile, bool DIRECT>
__global__ void __launch_bounds__(kSortBlock) rs_histogram(const uint64_t *__restrict__ keys, int64_t n, int shift,
                                                           uint32_t *__restrict__ counts, int tiles) {
  __shared__ uint32_t h[kDigits];
  const int t = threadIdx.x;
  h[t] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * kTile;
  const uint64_t below = lanes_below();
  for (int i = t; i < kTile; i += kSortBlock) {
    const int64_t g = base + i;
    const bool valid = g < n;
    const uint32_t dig = valid ? (uint32_t)((keys[g] >> shift) & 0xff) : 0u;
    const uint64_t match = digit_match(valid, dig);
    // the lowest lane of each group adds the group
    if (valid && (match & below) == 0) atomicAdd(&h[dig], (uint32_t)__popcll(match));
  }
  __syncthreads();
  counts[DIRECT ? (size_t)blockIdx.x * kDigits + t : (size_t)t * tiles + blockIdx.x] = h[t];
}

template <int kTile, bool DIRECT>
__global__ void __launch_bounds__(kSortBlock) rs_scatter(const uint64_t *__restrict__ kin,
                                                         const uint32_t *__restrict__ vin,
                                                         uint64_t *__restrict__ kout,
                                                         uint32_t *__restrict__ vout, int64_t n, int shift,
                                                         const uint32_t *__restrict__ counts, int tiles) {
  constexpr int kChunks = kTile / kSortBlock;  // 64-key chunks per wave
  __shared__ uint64_t skey[kTile];
  __shared__ uint32_t sval[kTile];
  __shared__ uint32_t wrun[kWaves][kDigits];  // per wave: running count, then the wave's base
  __shared__ uint32_t lbase[kDigits];         // tile-local start of each digit
  __shared__ uint32_t gbase[kDigits];         // global start of the tile's keys of each digit
  __shared__ uint32_t wtot[kWaves], dtot[kWaves];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t base = (int64_t)blockIdx.x * kTile;
  // digit t: keys of the digit in earlier tiles and in all tiles (DIRECT), or
  // the scanned bounds of its keys
  uint32_t in_before = 0, in_all = 0;
  if (DIRECT) {
    // sixteen rows in flight: one at a time the loop was the pass (60 000 keys,
    // 59 tiles: 17.9 -> 8.5 us; 200 000 keys, 49 tiles of 4 096: 22.3 -> 14.5 us)
    for (int i0 = 0; i0 < tiles; i0 += 16) {
      uint32_t c[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) c[k] = counts[(size_t)min(i0 + k, tiles - 1) * kDigits + t];
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const uint32_t v = i0 + k < tiles ? c[k] : 0u;
        in_before += i0 + k < (int)blockIdx.x ? v : 0u;
        in_all += v;
      }
    }
  } else {
    const uint32_t lo = t == 0 ? 0u : counts[(size_t)t * tiles - 1];
    in_all = counts[(size_t)(t + 1) * tiles - 1] - lo;
  }
  if (__syncthreads_or(in_all == (uint32_t)n)) {  // one digit holds every key: identity pass
    for (int i = t; i < kTile; i += kSortBlock) {
      const int64_t g = base + i;
      if (g < n) {
        kout[g] = kin[g];
        vout[g] = vin[g];
      }
    }
    return;
  }
#pragma unroll
  for (int w = 0; w < kWaves; ++w) wrun[w][t] = 0;
  __syncthreads();
  uint64_t key[kChunks];
  uint32_t val[kChunks], pos[kChunks];
  const int64_t wbase = base + (int64_t)wave * (kChunks * 64) + lane;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int64_t g = wbase + c * 64;
    key[c] = g < n ? kin[g] : 0ull;
    val[c] = g < n ? vin[g] : 0u;
  }
  const uint64_t below = lanes_below();
  // rank inside the wave's keys of the same digit, in input order; the
  // running counts are per wave, and one wave's LDS operations take effect
  // in program order, so each chunk reads the counts the previous one left
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const bool valid = wbase + c * 64 < n;
    const uint32_t dig = (uint32_t)((key[c] >> shift) & 0xff);
    const uint64_t match = digit_match(valid, dig);
    const uint32_t rank = (uint32_t)__popcll(match & below);
    const uint32_t cnt = (uint32_t)__popcll(match);
    const uint32_t r0 = valid ? wrun[wave][dig] : 0u;
    pos[c] = r0 + rank;
    if (valid && rank + 1 == cnt) wrun[wave][dig] = r0 + cnt;
  }
  __syncthreads();
  // digit t: wave bases, tile-local start (exclusive scan over the digits)
  // and global start
  uint32_t tot = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const uint32_t c = wrun[w][t];
    wrun[w][t] = tot;
    tot += c;
  }
  uint32_t x = tot;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, (unsigned)d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) wtot[wave] = x;
  if (DIRECT) {
    // exclusive scan of the digits' totals
    uint32_t y = in_all;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t z = __shfl_up(y, (unsigned)d, 64);
      if (lane >= d) y += z;
    }
    if (lane == 63) dtot[wave] = y;
    __syncthreads();
    uint32_t digits_before = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) digits_before += w < wave ? dtot[w] : 0u;
    gbase[t] = digits_before + y - in_all + in_before;
  } else {
    const size_t e = (size_t)t * tiles + blockIdx.x;
    gbase[t] = e ? counts[e - 1] : 0u;
    __syncthreads();
  }
  uint32_t before = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) before += w < wave ? wtot[w] : 0u;
  lbase[t] = before + x - tot;
  __syncthreads();
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    if (wbase + c * 64 >= n) continue;
    const uint32_t dig = (uint32_t)((key[c] >> shift) & 0xff);
    const uint32_t lp = lbase[dig] + wrun[wave][dig] + pos[c];
    skey[lp] = key[c];
    sval[lp] = val[c];
  }
  __syncthreads();
  const int valid_n = (int)min((int64_t)kTile, n - base);
  for (int i = t; i < valid_n; i += kSortBlock) {
    const uint64_t k = skey[i];
    const uint32_t dig = (uint32_t)((k >> shift) & 0xff);
    const uint32_t gp = gbase[dig] + (uint32_t)i - lbase[dig];
    kout[gp] = k;
    vout[gp] = sval[i];
  }
}

// Up to kSmallSort keys: a key's place is the number of keys before it, counted
// by all 16 waves of a workgroup for 64 keys (a lane each), every wave over its
// share of the keys, which it reads with uniform addresses.  n^2 comparisons
// spread over the chip cost less than the 91 barriers of one workgroup's
// bitonic sort of 8 192 keys: the three sorts of a 256-point catalogue (256,
// 256 and 4 790 keys) 126 -> 44 us.  Against the passes, by builds of uniform
// clouds (two sorts each): 2 048 points 194 and 314 us, 4 096 227 and 330,
// 8 192 271 and 339, 12 000 314 and 345, 16 384 356 and 347; the line leaves
// what a chip shared with other streams costs the counting.
__global__ void __launch_bounds__(kSmallBlock) rs_rank(const uint64_t *__restrict__ keys, const uint32_t *__restrict__ vals,
                                                       int n, int shift, uint64_t mask, uint64_t *__restrict__ kout,
                                                       uint32_t *__restrict__ vout) {
  constexpr int kWaves = kSmallBlock / 64;
  __shared__ uint32_t part[kWaves][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int first = blockIdx.x * 64, i = first + lane;
  const uint64_t key = i < n ? keys[i] : 0, mine = (key >> shift) & mask;
  const int share = (n + kWaves - 1) / kWaves, j0 = wave * share, j1 = min(j0 + share, n);
  // equal keys keep their order: those at smaller positions come before
  uint32_t before = 0;
  const int lo = min(max(first, j0), j1), hi = min(max(first + 64, j0), j1);
  for (int j = j0; j < lo; ++j) before += ((keys[j] >> shift) & mask) <= mine;
  for (int j = lo; j < hi; ++j) {
    const uint64_t k = (keys[j] >> shift) & mask;
    before += k < mine || (k == mine && j < i);
  }
  for (int j = hi; j < j1; ++j) before += ((keys[j] >> shift) & mask) < mine;
  part[wave][lane] = before;
  __syncthreads();
  if (wave != 0 || i >= n) return;
  uint32_t place = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) place += part[w][lane];
  kout[place] = key;
  vout[place] = vals[i];
}

__global__ void rs_copy(const uint64_t *__restrict__ kin, const uint32_t *__restrict__ vin, int n, uint64_t *kout,
                        uint32_t *vout) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  kout[i] = kin[i];
  vout[i] = vin[i];
}

template <int kTile, bool DIRECT>
void sort_pass(RadixSorter &S, const uint64_t *ka, const uint32_t *va, uint64_t *kb, uint32_t *vb, int64_t n, int shift,
               int tiles, hipStream_t stream) {
  hipLaunchKernelGGL((rs_histogram<kTile, DIRECT>), dim3(tiles), dim3(kSortBlock), 0, stream, ka, n, shift, S.counts.p,
                     tiles);
  if (!DIRECT) S.scanner.inclusive(S.counts.p, (int64_t)kDigits * tiles, stream);
  hipLaunchKernelGGL((rs_scatter<kTile, DIRECT>), dim3(tiles), dim3(kSortBlock), 0, stream, ka, va, kb, vb, n, shift,
                     S.counts.p, tiles);
}

}  // namespace

void RadixSorter::sort(uint64_t *keys, uint32_t *vals, int64_t n, int begin_bit, int end_bit,
                       hipStream_t stream) {
  if (n <= 1) return;
  if (n <= kSmallSort) {
    const uint64_t mask = end_bit - begin_bit >= 64 ? ~0ull : (1ull << (end_bit - begin_bit)) - 1ull;
    tmp_keys.ensure(n);
    tmp_vals.ensure(n);
    hipLaunchKernelGGL(rs_rank, dim3(blocks_for(n, 64)), dim3(kSmallBlock), 0, stream, keys, vals, (int)n, begin_bit, mask,
                       tmp_keys.p, tmp_vals.p);
    hipLaunchKernelGGL(rs_copy, dim3(blocks_for(n, 256)), dim3(256), 0, stream, tmp_keys.p, tmp_vals.p, (int)n, keys, vals);
    MHGP_LAUNCH_CHECK();
    return;
  }
  // tiles of 1 024 keys while each scatter can sum their counts, then of 4 096
  const bool fine = n <= 1024 * kDirectTiles;
  const int tiles = blocks_for(n, fine ? 1024 : 4096);
  tmp_keys.ensure(n);
  tmp_vals.ensure(n);
  counts.ensure((size_t)kDigits * tiles);
  uint64_t *ka = keys, *kb = tmp_keys.p;
  uint32_t *va = vals, *vb = tmp_vals.p;
  int passes = 0;
  for (int shift = begin_bit; shift < end_bit; shift += 8) {
    if (fine) sort_pass<1024, true>(*this, ka, va, kb, vb, n, shift, tiles, stream);
    else if (tiles <= kDirectTiles) sort_pass<4096, true>(*this, ka, va, kb, vb, n, shift, tiles, stream);
    else sort_pass<4096, false>(*this, ka, va, kb, vb, n, shift, tiles, stream);
    MHGP_LAUNCH_CHECK();
    std::swap(ka, kb);
    std::swap(va, vb);
    passes++;
  }
  if (passes & 1) {
    MHGP_HIP(hipMemcpyAsync(keys, ka, n * sizeof(uint64_t), hipMemcpyDeviceToDevice, stream));
    MHGP_HIP(hipMemcpyAsync(vals, va, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, stream));
  }
}

}  // namespace mhgp
