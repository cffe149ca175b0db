// Stable LSD radix sort of 64-bit keys with 32-bit payloads.
//
// Replaces the std::sort of Subtree::buildTree (src/Subtree.h:281) and
// Reader::localSort (src/Reader.C:237-241).  The reference's std::sort is
// unstable; this sort is stable, so equal keys keep ascending original index,
// which is the order the oracle defines.
//
// Per 8-bit digit pass:
//   1. count_kernel   -- LDS histogram of each tile of 512 to 2048 keys;
//   2. with many tiles, the counts digit-major and one device-wide exclusive
//      scan of the 256 x tiles table, which yields every (digit, tile) output
//      offset; with few, the counts tile-major and summed by step 3;
//   3. scatter_kernel -- each wave ranks its quarter of the tile in rounds of
//                        64 with an 8-ballot digit match and per-wave LDS
//                        counters; ranks become tile-local positions, keys are
//                        staged through LDS and written out in digit runs so
//                        the HBM writes are contiguous.
#include "pt_common.h"
#include "pt_kernels.h"

#include <algorithm>

namespace {

constexpr int kSortThreads = 256;
constexpr int kSortWaves = kSortThreads / PT_WAVE;
constexpr int kSortItems = 8;
constexpr int kSortTile = kSortThreads * kSortItems;  // 2048 keys per block
constexpr int kRadix = 256;
// Up to this many tiles the scatter kernel sums the digit counts before its
// tile itself, 2 launches a pass instead of 5, and small sets take smaller
// tiles, whose rounds are fewer (the passes are a chain of latencies: launches,
// loads, rounds of ranking).  Sort of 4 digits, us, scan launches / own sums
// with 2, 4, 8 keys per thread: 30k keys 84 / 41, 46, -; 64k 86 / 51, 47, 54;
// 100k 87 / -, 54, 58; 8 digits of 200k 185 / -, -, 142.
constexpr int kOwnTiles = 128;
constexpr int64_t kOwnMax2 = 32768;
constexpr int64_t kOwnMax4 = (int64_t)kOwnTiles * kSortThreads * 4;
constexpr int64_t kOwnMax8 = (int64_t)kOwnTiles * kSortTile;

// OWN: the counts are written tile-major, else digit-major.
template <int ITEMS, bool OWN>
__global__ void __launch_bounds__(kSortThreads)
count_kernel(const uint64_t* __restrict__ keys, int64_t n, int shift, int ntiles,
             uint32_t* __restrict__ counts) {
  __shared__ uint32_t hist[kRadix];
  hist[threadIdx.x] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * (kSortThreads * ITEMS);
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    const int64_t i = base + (int64_t)j * kSortThreads + threadIdx.x;
    if (i < n) atomicAdd(&hist[(unsigned)(keys[i] >> shift) & (kRadix - 1)], 1u);
  }
  __syncthreads();
  counts[OWN ? (int64_t)blockIdx.x * kRadix + threadIdx.x
             : (int64_t)threadIdx.x * ntiles + blockIdx.x] = hist[threadIdx.x];
}

// Exclusive prefix of v over the work-group's threads.
__device__ __forceinline__ uint32_t sort_block_excl(uint32_t v, uint32_t* s_wsum) {
  const int lane = threadIdx.x & (PT_WAVE - 1), wave = threadIdx.x / PT_WAVE;
  uint32_t t = v;
#pragma unroll
  for (int d = 1; d < PT_WAVE; d <<= 1) {
    const uint32_t o = __shfl_up(t, d, PT_WAVE);
    if (lane >= d) t += o;
  }
  if (lane == PT_WAVE - 1) s_wsum[wave] = t;
  __syncthreads();
  for (int w = 0; w < wave; w++) t += s_wsum[w];
  __syncthreads();
  return t - v;
}

// FIRST: the payload is the key's input index (vals_in unused).  OWN: offsets
// holds the tile-major counts, else their digit-major exclusive scan.
template <bool FIRST, int ITEMS, bool OWN>
__global__ void __launch_bounds__(kSortThreads)
scatter_kernel(const uint64_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
               int64_t n, int shift, int ntiles, const uint32_t* __restrict__ offsets,
               uint64_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out) {
  __shared__ uint32_t wave_run[kSortWaves][kRadix];
  __shared__ uint32_t tile_off[kRadix];
  constexpr int kTile = kSortThreads * ITEMS;
  __shared__ uint64_t s_keys[kTile];
  __shared__ uint32_t s_vals[kTile];
  __shared__ uint32_t s_dst[kRadix];  // output slot of each digit's first key, less its tile slot
  __shared__ uint32_t s_wsum[kSortWaves];

  const int lane = threadIdx.x & (PT_WAVE - 1);
  const int wave = threadIdx.x / PT_WAVE;
  for (int i = threadIdx.x; i < kSortWaves * kRadix; i += kSortThreads)
    (&wave_run[0][0])[i] = 0;
  __syncthreads();

  // the thread's digit: its keys in all tiles and in the tiles before this one
  uint32_t all = 0, before_tile = 0;
  if (OWN) {
#pragma unroll 8
    for (int t = 0; t < ntiles; t++) {
      const uint32_t c = offsets[t * kRadix + threadIdx.x];
      all += c;
      before_tile += t < (int)blockIdx.x ? c : 0u;
    }
  }

  const int64_t tile_base = (int64_t)blockIdx.x * kTile;
  const int64_t wave_base = tile_base + (int64_t)wave * (ITEMS * PT_WAVE);
  uint64_t k[ITEMS];
  uint32_t v[ITEMS];
  uint32_t rank[ITEMS];
  const unsigned long long lt_mask = (1ull << lane) - 1ull;

#pragma unroll
  for (int r = 0; r < ITEMS; r++) {
    const int64_t i = wave_base + (int64_t)r * PT_WAVE + lane;
    const bool valid = i < n;
    k[r] = valid ? keys_in[i] : ~0ull;
    v[r] = valid ? (FIRST ? (uint32_t)i : vals_in[i]) : 0u;
    const uint32_t d = (uint32_t)(k[r] >> shift) & (kRadix - 1);
    // lanes holding the same digit (invalid lanes never match a valid one:
    // they are excluded from the initial mask)
    unsigned long long peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      const bool bit = (d >> b) & 1u;
      const unsigned long long bal = __ballot(bit);
      peers &= bit ? bal : ~bal;
    }
    const uint32_t before = wave_run[wave][d];
    const uint32_t rk = (uint32_t)__popcll(peers & lt_mask);
    rank[r] = before + rk;
    // the lowest peer lane publishes the new running count for this digit
    if (valid && rk == 0) wave_run[wave][d] = before + (uint32_t)__popcll(peers);
  }
  __syncthreads();

  // per-digit prefix over waves and tile-local digit offsets
  {
    const int d = threadIdx.x;  // kSortThreads == kRadix
    uint32_t acc = 0;
#pragma unroll
    for (int w = 0; w < kSortWaves; w++) {
      const uint32_t c = wave_run[w][d];
      wave_run[w][d] = acc;
      acc += c;
    }
    const uint32_t off = sort_block_excl(acc, s_wsum);
    tile_off[d] = off;
    const uint32_t out = OWN ? sort_block_excl(all, s_wsum) + before_tile
                             : offsets[(int64_t)d * ntiles + blockIdx.x];
    s_dst[d] = out - off;
  }
  __syncthreads();

#pragma unroll
  for (int r = 0; r < ITEMS; r++) {
    const int64_t i = wave_base + (int64_t)r * PT_WAVE + lane;
    if (i < n) {
      const uint32_t d = (uint32_t)(k[r] >> shift) & (kRadix - 1);
      const uint32_t pos = tile_off[d] + wave_run[wave][d] + rank[r];
      s_keys[pos] = k[r];
      s_vals[pos] = v[r];
    }
  }
  __syncthreads();

  const int64_t tile_n = (n - tile_base) < kTile ? (n - tile_base) : kTile;
  for (int j = threadIdx.x; j < tile_n; j += kSortThreads) {
    const uint64_t kk = s_keys[j];
    const uint32_t d = (uint32_t)(kk >> shift) & (kRadix - 1);
    const uint32_t dst = s_dst[d] + (uint32_t)j;  // modulo 2^32, below n
    keys_out[dst] = kk;
    vals_out[dst] = s_vals[j];
  }
}

__global__ void __launch_bounds__(256)
iota_kernel(uint32_t* __restrict__ v, int64_t n) {
  const int64_t i = blockIdx.x * 256ll + threadIdx.x;
  if (i < n) v[i] = (uint32_t)i;
}

// One digit pass; the first has no payload to read (vin null).
template <int ITEMS, bool OWN>
int sort_pass(const uint64_t* kin, const uint32_t* vin, int64_t n, int shift, int ntiles,
              uint32_t* counts, void* scan_scratch, uint64_t* kout, uint32_t* vout,
              hipStream_t s) {
  count_kernel<ITEMS, OWN><<<ntiles, kSortThreads, 0, s>>>(kin, n, shift, ntiles, counts);
  if (!OWN && pt_exclusive_scan_u32(counts, counts, (int64_t)ntiles * kRadix, scan_scratch,
                                    nullptr, s) != 0)
    return -1;
  if (!vin)
    scatter_kernel<true, ITEMS, OWN><<<ntiles, kSortThreads, 0, s>>>(kin, vin, n, shift, ntiles,
                                                                     counts, kout, vout);
  else
    scatter_kernel<false, ITEMS, OWN><<<ntiles, kSortThreads, 0, s>>>(kin, vin, n, shift, ntiles,
                                                                      counts, kout, vout);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

int64_t pt_sort_scratch_bytes(int64_t n) {
  const int64_t ntiles = (n + kSortTile - 1) / kSortTile;
  const int64_t table = std::max<int64_t>(ntiles, kOwnTiles) * kRadix;
  // counts table + scan scratch + ping-pong key/value buffers
  return table * 4 + pt_scan_scratch_bytes(table) + n * 8 + n * 4 + 1024;
}

// Sorts src (n keys, read only) into (keys, vals): vals = input index of
// each sorted key.  Scratch: pt_sort_scratch_bytes(n) bytes; begin_bit /
// end_bit bound the digit passes.
int pt_radix_sort(const uint64_t* src, uint64_t* keys, uint32_t* vals, int64_t n, int begin_bit,
                  int end_bit, void* scratch, hipStream_t s) {
  if (n <= 0) return 0;
  if (n == 1 || end_bit <= begin_bit) {
    if (n > 1) return -1;
    if (hipMemcpyAsync(keys, src, 8, hipMemcpyDeviceToDevice, s) != hipSuccess) return -1;
    iota_kernel<<<1, 256, 0, s>>>(vals, 1);
    return hipGetLastError() == hipSuccess ? 0 : -1;
  }
  if (n > 0x7fffffffll) return -1;
  const int tile = n <= kOwnMax2 ? kSortThreads * 2 : (n <= kOwnMax4 ? kSortThreads * 4 : kSortTile);
  const int ntiles = (int)((n + tile - 1) / tile);
  const int64_t table = (int64_t)ntiles * kRadix;
  char* p = (char*)scratch;
  uint32_t* counts = (uint32_t*)p;
  p += ((table * 4 + 255) / 256) * 256;
  void* scan_scratch = p;
  p += ((pt_scan_scratch_bytes(table) + 255) / 256) * 256;
  uint64_t* k2 = (uint64_t*)p;
  p += ((n * 8 + 255) / 256) * 256;
  uint32_t* v2 = (uint32_t*)p;

  // pass p writes (keys, vals) when an even number of passes follow it, the
  // scratch pair otherwise, so the last pass lands in (keys, vals)
  const int passes = (end_bit - begin_bit + 7) / 8;
  const uint64_t* kin = src;
  const uint32_t* vin = nullptr;
  for (int p = 0; p < passes; p++) {
    const int shift = begin_bit + 8 * p;
    const bool to_final = ((passes - 1 - p) % 2) == 0;
    uint64_t* kout = to_final ? keys : k2;
    uint32_t* vout = to_final ? vals : v2;
    int st = 0;
    if (n <= kOwnMax2)
      st = sort_pass<2, true>(kin, vin, n, shift, ntiles, counts, scan_scratch, kout, vout, s);
    else if (n <= kOwnMax4)
      st = sort_pass<4, true>(kin, vin, n, shift, ntiles, counts, scan_scratch, kout, vout, s);
    else if (n <= kOwnMax8)
      st = sort_pass<8, true>(kin, vin, n, shift, ntiles, counts, scan_scratch, kout, vout, s);
    else
      st = sort_pass<8, false>(kin, vin, n, shift, ntiles, counts, scan_scratch, kout, vout, s);
    if (st != 0) return st;
    kin = kout;
    vin = vout;
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int pt_launch_iota(uint32_t* v, int64_t n, hipStream_t s) {
  if (n <= 0) return 0;
  iota_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(v, n);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}
