// sort.hip -- device-wide exclusive scan and stable LSD radix sort.
//
// The sort orders (64-bit key, 32-bit value) pairs.  Each pass handles one
// digit of up to 8 bits in three kernels: per-block digit histogram, one
// exclusive scan of the digit-major histogram table, and a stable scatter.
// The scatter ranks equal digits inside a wavefront with ballots (one ballot
// per digit bit gives every lane the mask of lanes holding its digit) and
// keeps per-wave running counts in LDS, so ranks follow input order and the
// sort is stable.  Particle keys need 60 bits (the placeholder bit 60 is the
// same for every key): seven 8-bit passes and one 4-bit pass.
//
// Arrays of up to 524,288 keys are sorted by merging instead (see below).
//
// Replaces the single-rank presort of slsort_keys (sl_pepc mpi_pepckeys.c:167,
// sort_radix.c:33-151): for distinct keys both give the same permutation.
#include "kernels.h"

#include <utility>

namespace pepc {

namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr int kScanTile = kScanThreads * kScanItems;   // 4096

// ---------------------------------------------------------------- scan
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* total) {
  __shared__ uint32_t wsum[kScanThreads / kWave];
  const int w = threadIdx.x / kWave;
  uint32_t inc = wave_inclusive_scan(v);
  if (lane_id() == kWave - 1) wsum[w] = inc;
  __syncthreads();
  uint32_t off = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < kScanThreads / kWave; ++k) {
    uint32_t t = wsum[k];
    off += (k < w) ? t : 0u;
    tot += t;
  }
  __syncthreads();
  *total = tot;
  return off + inc - v;
}

__global__ __launch_bounds__(kScanThreads) void scan_reduce_kernel(const uint32_t* __restrict__ in,
                                                                    int64_t n,
                                                                    uint32_t* __restrict__ bsum,
                                                                    bool flags) {
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  uint32_t s = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    int64_t e = base + j * kScanThreads + threadIdx.x;
    if (e < n) s += flags ? (in[e] != 0u ? 1u : 0u) : in[e];
  }
  uint32_t tot;
  (void)block_exclusive_scan(s, &tot);
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// Exclusive scan of up to kScanTile * 4 block sums in one block; writes the
// grand total to *total when total != nullptr.
__global__ __launch_bounds__(kScanThreads) void scan_small_kernel(uint32_t* __restrict__ v, int nb,
                                                                   uint32_t* __restrict__ total) {
  const int per = (nb + kScanThreads - 1) / kScanThreads;
  const int b0 = threadIdx.x * per;
  uint32_t s = 0;
  for (int k = 0; k < per; ++k)
    if (b0 + k < nb) s += v[b0 + k];
  uint32_t tot;
  uint32_t run = block_exclusive_scan(s, &tot);
  for (int k = 0; k < per; ++k) {
    if (b0 + k < nb) {
      uint32_t t = v[b0 + k];
      v[b0 + k] = run;
      run += t;
    }
  }
  if (threadIdx.x == 0 && total) *total = tot;
}

__global__ __launch_bounds__(kScanThreads) void scan_apply_kernel(const uint32_t* __restrict__ in,
                                                                   uint32_t* __restrict__ out,
                                                                   int64_t n,
                                                                   const uint32_t* __restrict__ bsum) {
  __shared__ uint32_t tile[kScanTile];
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  if (base >= n) return;   // uniform over the block
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    int64_t e = base + j * kScanThreads + threadIdx.x;
    tile[j * kScanThreads + threadIdx.x] = e < n ? in[e] : 0u;
  }
  __syncthreads();
  uint32_t loc[kScanItems];
  uint32_t s = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    loc[j] = s;
    s += tile[threadIdx.x * kScanItems + j];
  }
  uint32_t tot;
  uint32_t off = block_exclusive_scan(s, &tot) + bsum[blockIdx.x];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) tile[threadIdx.x * kScanItems + j] = off + loc[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    int64_t e = base + j * kScanThreads + threadIdx.x;
    if (e < n) out[e] = tile[j * kScanThreads + threadIdx.x];
  }
}

// The nonzero marks in order: the g-th, at particle a, gives gfirst[g] = a and
// gcount[g] = its value.  Takes one tile of marks per block; bsum holds the
// number of marks of every tile, or their exclusive scan.  The count, the
// ranks and the list were four launches with the ranks written and read again;
// now two read the marks: 18 us in place of 33 at 4,194,304 particles, and two
// launches of 2 us fewer in every grow.
__global__ __launch_bounds__(kScanThreads) void group_list_kernel(
    int64_t n, const uint32_t* __restrict__ gmark, const uint32_t* __restrict__ bsum, bool scanned,
    uint32_t* __restrict__ gfirst, uint32_t* __restrict__ gcount, uint32_t* __restrict__ ngroups,
    unsigned long long* __restrict__ clock) {
  __shared__ uint32_t tile[kScanTile];
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  uint32_t before = 0;
  if (!scanned)
    for (unsigned k = threadIdx.x; k < blockIdx.x; k += kScanThreads) before += bsum[k];
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    const int64_t e = base + j * kScanThreads + threadIdx.x;
    tile[j * kScanThreads + threadIdx.x] = e < n ? gmark[e] : 0u;
  }
  uint32_t start;
  (void)block_exclusive_scan(before, &start);   // and the tile is complete
  if (scanned) start = bsum[blockIdx.x];
  uint32_t c[kScanItems], s = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    c[j] = tile[threadIdx.x * kScanItems + j];
    s += c[j] ? 1u : 0u;
  }
  uint32_t tot;
  uint32_t g = start + block_exclusive_scan(s, &tot);
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    if (!c[j]) continue;
    gfirst[g] = (uint32_t)(base + threadIdx.x * kScanItems + j);
    gcount[g] = c[j];
    ++g;
  }
  if (blockIdx.x + 1 == gridDim.x && threadIdx.x == 0) {
    *ngroups = start + tot;
    clock[kClockGrown] = wall_clock64();
  }
}

// ---------------------------------------------------------------- radix sort
constexpr int kSortThreads = 256;
constexpr int kSortItems = 8;
constexpr int kSortWaves = kSortThreads / kWave;
constexpr int kSortTile = kSortThreads * kSortItems;   // 2048
constexpr int kRadix = 256;
constexpr int kScanHereBlocks = 64;   // up to 131,072 elements: no separate digit scan

// The digit of element e is bits [shift, shift+nbits) of its key, or, when
// dsrc is given, of dsrc[value] (used to order by system after the keys).
__device__ __forceinline__ uint32_t radix_digit(unsigned long long key, uint32_t val,
                                                const uint32_t* dsrc, int shift, uint32_t mask) {
  return dsrc ? (dsrc[val] >> shift) & mask : (uint32_t)(key >> shift) & mask;
}

__global__ __launch_bounds__(kSortThreads) void radix_hist_kernel(
    const unsigned long long* __restrict__ keys, const uint32_t* __restrict__ vals,
    const uint32_t* __restrict__ dsrc, int64_t n, int shift, uint32_t mask,
    uint32_t* __restrict__ hist, int nblocks) {
  __shared__ uint32_t cnt[kRadix];
  cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
#pragma unroll 4
  for (int j = 0; j < kSortItems; ++j) {
    int64_t e = base + j * kSortThreads + threadIdx.x;
    if (e < n) atomicAdd(&cnt[radix_digit(keys[e], dsrc ? vals[e] : 0u, dsrc, shift, mask)], 1u);
  }
  __syncthreads();
  hist[(int64_t)threadIdx.x * nblocks + blockIdx.x] = cnt[threadIdx.x];
}

// Ranks each element within its block (stable), stages the block's elements
// in LDS in digit order, then writes them out so that consecutive threads
// store consecutive positions of one digit's run (coalesced stores).
// hscan is the digit-major table of per-block counts: exclusive-scanned along
// each digit's row by digit_scan_kernel, with the row totals in dtot, or,
// with scan_here, the histogram itself (dtot unused).
__global__ __launch_bounds__(kSortThreads) void radix_scatter_kernel(
    const unsigned long long* __restrict__ kin, const uint32_t* __restrict__ vin,
    unsigned long long* __restrict__ kout, uint32_t* __restrict__ vout,
    const uint32_t* __restrict__ dsrc, int64_t n, int shift, int nbits,
    const uint32_t* __restrict__ hscan, const uint32_t* __restrict__ dtot, int nblocks,
    bool scan_here) {
  const int64_t tile0 = (int64_t)blockIdx.x * kSortTile;
  __shared__ uint32_t wcnt[kSortWaves][kRadix];
  __shared__ uint32_t lbase[kRadix];
  __shared__ uint32_t gbase[kRadix];
  __shared__ uint32_t bbase[kRadix];   // digit d's elements in the blocks before this one
  __shared__ unsigned long long skey[kSortTile];
  __shared__ uint32_t sval[kSortTile];
  __shared__ uint8_t sdig[kSortTile];
  const int w = threadIdx.x / kWave;
  const uint32_t mask = (1u << nbits) - 1u;
#pragma unroll
  for (int k = 0; k < kSortWaves; ++k) wcnt[k][threadIdx.x] = 0;
  __syncthreads();

  const int64_t base = tile0 + (int64_t)w * (kSortItems * kWave);
  unsigned long long kk[kSortItems];
  uint32_t vv[kSortItems];
  uint32_t dig[kSortItems];
  uint32_t loc[kSortItems];
  const unsigned long long lt = lanemask_lt();
#pragma unroll
  for (int j = 0; j < kSortItems; ++j) {
    const int64_t e = base + j * kWave + lane_id();
    const bool valid = e < n;
    kk[j] = valid ? kin[e] : 0ull;
    vv[j] = valid ? vin[e] : 0u;
    const uint32_t d = valid ? radix_digit(kk[j], vv[j], dsrc, shift, mask) : 0u;
    dig[j] = d;
    unsigned long long peers = __ballot(valid);
    for (int b = 0; b < nbits; ++b) {
      const bool bit = (d >> b) & 1u;
      const unsigned long long m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    const uint32_t rank = (uint32_t)popc64(peers & lt);
    uint32_t c = 0;
    if (valid) c = wcnt[w][d];
    __builtin_amdgcn_wave_barrier();
    if (valid && rank == 0) wcnt[w][d] = c + (uint32_t)popc64(peers);
    __builtin_amdgcn_wave_barrier();
    loc[j] = c + rank;
  }
  __syncthreads();
  {
    // thread d: offsets of digit d per wave, and the block-local start of d
    const uint32_t d = threadIdx.x;
    uint32_t run = 0;
#pragma unroll
    for (int k = 0; k < kSortWaves; ++k) {
      const uint32_t t = wcnt[k][d];
      wcnt[k][d] = run;
      run += t;
    }
    uint32_t tot;
    lbase[d] = block_exclusive_scan(run, &tot);
    // digit d's total and its count in earlier blocks: from the digit scan,
    // or, for a few blocks (scan_here), from the histogram row of digit d
    uint32_t all, before;
    if (scan_here) {
      const uint32_t* row = hscan + (int64_t)d * nblocks;
      all = 0;
      before = 0;
      for (int b = 0; b < nblocks; ++b) {
        const uint32_t v = row[b];
        before += b < (int)blockIdx.x ? v : 0u;
        all += v;
      }
    } else {
      all = dtot[d];
      before = hscan[(int64_t)d * nblocks + blockIdx.x];
    }
    bbase[d] = before;
    // global start of digit d: digits below d over all blocks
    gbase[d] = block_exclusive_scan(all, &tot);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kSortItems; ++j) {
    const int64_t e = base + j * kWave + lane_id();
    if (e < n) {
      const uint32_t lp = lbase[dig[j]] + wcnt[w][dig[j]] + loc[j];
      skey[lp] = kk[j];
      sval[lp] = vv[j];
      sdig[lp] = (uint8_t)dig[j];
    }
  }
  __syncthreads();
  const int64_t rem = n - tile0;
  const int cnt = rem < kSortTile ? (int)rem : kSortTile;
  for (int i = threadIdx.x; i < cnt; i += kSortThreads) {
    const uint32_t d = sdig[i];
    const uint32_t pos = gbase[d] + bbase[d] + ((uint32_t)i - lbase[d]);
    kout[pos] = skey[i];
    vout[pos] = sval[i];
  }
}

// Exclusive scan of one digit's row of the block histogram (block b's count
// of digit d -> number of digit-d elements in blocks before b), row total to
// dtot[d].  One block per digit.
__global__ __launch_bounds__(kSortThreads) void digit_scan_kernel(uint32_t* __restrict__ hist,
                                                                 int nblocks,
                                                                 uint32_t* __restrict__ dtot) {
  uint32_t* row = hist + (int64_t)blockIdx.x * nblocks;
  const int per = (nblocks + kSortThreads - 1) / kSortThreads;
  const int b0 = threadIdx.x * per;
  uint32_t sum = 0;
  for (int k = 0; k < per; ++k)
    if (b0 + k < nblocks) sum += row[b0 + k];
  uint32_t tot;
  uint32_t run = block_exclusive_scan(sum, &tot);
  for (int k = 0; k < per; ++k) {
    if (b0 + k < nblocks) {
      const uint32_t t = row[b0 + k];
      row[b0 + k] = run;
      run += t;
    }
  }
  if (threadIdx.x == 0) dtot[blockIdx.x] = tot;
}

// ---------------------------------------------------------------- merge sort
// Smaller arrays: blocks of 2,048 pairs sorted in LDS (bitonic; values grow
// with the position, so ordering by (key, value) is the stable order), then
// four runs merged per launch, every element finding its place by binary
// searches in the three other runs.  A radix pass costs two dependent
// launches of 4 and 8 to 10 us whatever the size, eight times; here it is one
// launch per factor of four above 2,048.  Whole grow, radix against merging:
// 184 and 130 us for 1,777 particles, 254 and 186 for 32,768, 359 and 254 for
// 131,072, 412 and 368 for 524,288; 532 and 553 for 1,048,576, where the
// searches' scattered reads cost more than the passes.
constexpr int kMergeT = 1024;
constexpr int kMergeN = 2 * kMergeT;

// Orders this wave's LDS accesses for the compiler (LDS instructions of one
// wave execute in order).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__global__ __launch_bounds__(kMergeT) void merge_block_kernel(
    const unsigned long long* kin, const uint32_t* vin, unsigned long long* kout, uint32_t* vout,
    int64_t n) {
  __shared__ unsigned long long sk[kMergeN];
  __shared__ uint32_t sv[kMergeN];
  const int64_t base = (int64_t)blockIdx.x * kMergeN;
  const int cnt = n - base < kMergeN ? (int)(n - base) : kMergeN;
  int size = 2;
  while (size < cnt) size *= 2;
  const int t = threadIdx.x;
  for (int e = t; e < size; e += kMergeT) {
    sk[e] = e < cnt ? kin[base + e] : ~0ull;
    sv[e] = e < cnt ? vin[base + e] : ~0u;
  }
  __syncthreads();
  // A pair of distance j <= 64 lies in the 128 elements of one wave: those
  // stages need no barrier among themselves.
  for (int k = 2; k <= size; k *= 2) {
    for (int j = k / 2; j > 0; j /= 2) {
      if (t < size / 2) {
        const int a = 2 * t - (t & (j - 1)), b = a + j;
        const unsigned long long ka = sk[a], kb = sk[b];
        const uint32_t va = sv[a], vb = sv[b];
        const bool greater = ka > kb || (ka == kb && va > vb);
        if (greater == ((a & k) == 0)) {
          sk[a] = kb; sk[b] = ka;
          sv[a] = vb; sv[b] = va;
        }
      }
      const int next = j > 1 ? j / 2 : k;   // distance of the following stage
      if (j > kWave || next > kWave) __syncthreads();
      else wave_lds_order();
    }
  }
  __syncthreads();
  for (int e = t; e < cnt; e += kMergeT) {
    kout[base + e] = sk[e];
    vout[base + e] = sv[e];
  }
}

// The same blocks by counting: an element's place is the number of its block's
// elements that are smaller, or equal and before it.  A workgroup places 64 of
// the block's elements, one per lane, and each of its 16 waves counts over 128
// of the 2,048, so a block of keys keeps 32 CUs busy where the bitonic network
// runs its 66 dependent stages on one: 23 -> 9 us for 32,768 elements, 6 for
// 1,777.  The work grows with the number of blocks while the network's time
// does not.
constexpr int kRankT = 1024;
constexpr int kRankSpan = kMergeN / (kRankT / kWave);
static_assert(kRankSpan % kWave == 0, "a wave counts over whole runs of 64");

__global__ __launch_bounds__(kRankT) void rank_block_kernel(
    const unsigned long long* __restrict__ kin, const uint32_t* __restrict__ vin,
    unsigned long long* __restrict__ kout, uint32_t* __restrict__ vout, int64_t n) {
  __shared__ unsigned long long sk[kMergeN];
  __shared__ uint32_t part[kRankT / kWave][kWave];
  constexpr int kChunks = kMergeN / kWave;
  const int64_t base = blockIdx.x / kChunks * (int64_t)kMergeN;
  const int own = (int)(blockIdx.x % kChunks);
  const int cnt = n - base < kMergeN ? (int)(n - base) : kMergeN;
  const int t = threadIdx.x, lane = lane_id(), w = t / kWave;
  for (int e = t; e < kMergeN; e += kRankT) sk[e] = e < cnt ? kin[base + e] : ~0ull;
  __syncthreads();
  const int mine = own * kWave + lane;
  const unsigned long long key = sk[mine];   // keys are below 2^61, the padding above
  uint32_t c = 0;
#pragma unroll
  for (int g = 0; g < kRankSpan / kWave; ++g) {
    const int run = w * (kRankSpan / kWave) + g;
    const unsigned long long* r = sk + run * kWave;
    if (run == own) {
#pragma unroll 8
      for (int e = 0; e < kWave; ++e) c += r[e] < key + (e < lane ? 1ull : 0ull) ? 1u : 0u;
    } else {
      const unsigned long long bound = key + (run < own ? 1ull : 0ull);
#pragma unroll 8
      for (int e = 0; e < kWave; ++e) c += r[e] < bound ? 1u : 0u;
    }
  }
  part[w][lane] = c;
  __syncthreads();
  if (w != 0 || mine >= cnt) return;
  uint32_t rank = 0;
#pragma unroll
  for (int k = 0; k < kRankT / kWave; ++k) rank += part[k][lane];
  kout[base + rank] = key;
  vout[base + rank] = vin[base + mine];
}

// Runs of `run` elements (the last may be shorter), four to a group: element
// i of a run moves behind the elements of the group's earlier runs that are
// not greater and of its later runs that are smaller.  The searches are a
// chain of loads, so PAIR takes two steps at a time, for half as many loads
// again; that is the shorter way until the loads themselves fill the chip.
template <bool PAIR>
__global__ __launch_bounds__(256) void merge4_kernel(const unsigned long long* __restrict__ kin,
                                                     const uint32_t* __restrict__ vin,
                                                     unsigned long long* __restrict__ kout,
                                                     uint32_t* __restrict__ vout, int n, int run) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const unsigned long long key = kin[i];
  const int r = i / run, first = r & ~3;
  int pos[3] = {0, 0, 0}, begin[3], len[3];
  unsigned long long bound[3];   // elements below it come first (keys are below 2^61)
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int other = first + q + (first + q >= r ? 1 : 0);
    const int64_t b = (int64_t)other * run;
    // an empty run reads element 0 and takes nothing from it
    begin[q] = b < n ? (int)b : 1;
    len[q] = b < n ? (n - begin[q] < run ? n - begin[q] : run) : 0;
    bound[q] = other < r ? key + 1ull : key;
  }
  if constexpr (PAIR) {
    // two binary steps at a time (run is 2^11 times a power of four: 12, 14, ...
    // steps): their three pivots are loaded together
    for (int s = run; s > 1; s >>= 2) {
      const int h = s >> 1;
      unsigned long long a[3], b[3], c[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const unsigned long long* p = kin + begin[q];
        const int last = len[q] - 1;
        const int ia = pos[q] + h - 1, ib = pos[q] + s - 1, ic = pos[q] + s + h - 1;
        a[q] = p[ia < last ? ia : last];
        b[q] = p[ib < last ? ib : last];
        c[q] = p[ic < last ? ic : last];
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const bool up = pos[q] + s <= len[q] && b[q] < bound[q];
        pos[q] += up ? s : 0;
        if (pos[q] + h <= len[q] && (up ? c[q] : a[q]) < bound[q]) pos[q] += h;
      }
    }
  } else {
    for (int s = run; s > 0; s >>= 1) {
#pragma unroll
      for (int q = 0; q < 3; ++q)
        if (pos[q] + s <= len[q] && kin[begin[q] + pos[q] + s - 1] < bound[q]) pos[q] += s;
    }
  }
  const int64_t out = (int64_t)first * run + (i - r * run) + pos[0] + pos[1] + pos[2];
  kout[out] = key;
  vout[out] = vin[i];
}

__global__ __launch_bounds__(256) void gather4_kernel(int64_t n, const uint32_t* __restrict__ perm,
                                                      const double* __restrict__ x,
                                                      const double* __restrict__ y,
                                                      const double* __restrict__ z,
                                                      const double* __restrict__ q,
                                                      double* __restrict__ xs, double* __restrict__ ys,
                                                      double* __restrict__ zs, double* __restrict__ qs) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t p = perm[i];
  xs[i] = x[p];
  ys[i] = y[p];
  zs[i] = z[p];
  qs[i] = q[p];
}

__global__ __launch_bounds__(256) void copy_pairs_kernel(int64_t n,
                                                         const unsigned long long* __restrict__ kin,
                                                         const uint32_t* __restrict__ vin,
                                                         unsigned long long* __restrict__ kout,
                                                         uint32_t* __restrict__ vout) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  kout[i] = kin[i];
  vout[i] = vin[i];
}

void launch_copy_pairs(hipStream_t s, const unsigned long long* kin, const uint32_t* vin,
                       unsigned long long* kout, uint32_t* vout, int64_t n) {
  copy_pairs_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, kin, vin, kout, vout);
}

__global__ __launch_bounds__(256) void gather_rec_kernel(int64_t n, const uint32_t* __restrict__ perm,
                                                        const double4* __restrict__ rec,
                                                        double* __restrict__ xs, double* __restrict__ ys,
                                                        double* __restrict__ zs, double* __restrict__ qs) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double4 r = rec[perm[i]];
  xs[i] = r.x;
  ys[i] = r.y;
  zs[i] = r.z;
  qs[i] = r.w;
}

// Inverse of the grow permutation: out[perm[i]] = in[i].
__global__ __launch_bounds__(256) void scatter_back_kernel(int64_t n, const uint32_t* __restrict__ perm,
                                                          const double* __restrict__ in,
                                                          double* __restrict__ out) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[perm[i]] = in[i];
}

// Memory bound: 32 bytes read and 32 written per particle, one side of them
// scattered by the permutation in runs of 24 and 8 bytes. They take the place
// of a permutation that went to the host and back and of four indexed torch
// operations each way: a differentiable solve with its backward pass over
// 262,144 particles went from 5.1 to 4.0 ms.
__global__ __launch_bounds__(256) void restore_fields_kernel(
    int64_t n, const uint32_t* __restrict__ perm, const double* __restrict__ ex,
    const double* __restrict__ ey, const double* __restrict__ ez, const double* __restrict__ pot,
    double* __restrict__ e, double* __restrict__ phi) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t p = perm[i];
  e[3 * p] = ex[i];
  e[3 * p + 1] = ey[i];
  e[3 * p + 2] = ez[i];
  phi[p] = pot[i];
}

__global__ __launch_bounds__(256) void sort_fields_kernel(
    int64_t n, const uint32_t* __restrict__ perm, const double* __restrict__ e,
    const double* __restrict__ phi, double* __restrict__ ex, double* __restrict__ ey,
    double* __restrict__ ez, double* __restrict__ pot) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t p = perm[i];
  ex[i] = e[3 * p];
  ey[i] = e[3 * p + 1];
  ez[i] = e[3 * p + 2];
  pot[i] = phi[p];
}

// ---------------------------------------------------------------- tie order
// Order of equal keys as the reference's local presort leaves it.
//
// sort_radix_ip / rs_rec_ip (sl_pepc sort_radix.c:33-151) is an in-place MSD
// radix over 10-bit digits from bit 63 down.  A pass over a segment moves
// every element whose digit class k differs from the class of the region it
// sits in along permutation cycles; buckets above 256 elements recurse on
// the next digit, smaller ones get a stable insertion sort (sort_insert.c:
// 14-37).  Equal keys share every bucket, so their final order is the order
// in which the passes over the buckets that contain them leave them.
//
// In one pass an element already in its class's region stays where it is;
// the other slots of region k are filled, in increasing position, by the
// class-k elements in the order the cycles carry them there; and the cycles
// of the pass visit regions as a rotor walk: leaving region r always takes
// r's next not-yet-taken foreign slot (positions in increasing order), and
// the cycles started from region i (phase i, i = 0, 1, ...) end on their
// first return to i.  The walk is replayed here literally.  It is serial by
// nature (every step depends on the class read by the previous one), so the
// block prepares in parallel what the walk reads: the classes, the region
// bounds, and each region's foreign slots in increasing position as a list
// of (position, element, class) entries; one thread then walks, taking one
// list entry per step.
//
// Buckets without equal keys need nothing: for distinct keys the stable LSD
// order is the only sorted order.  So the replay descends only into buckets
// that hold a tie, and writes the final order of each such bucket into the
// permutation.  Runs only when the sort left equal adjacent keys (dup_count
// from dup_detect); one block per system.
//
// The equal keys are then moved apart in the same launch (fix_duplicates), so
// a system without any pays for one launch that returns at once; with the
// fix-up in seven more launches a solve of 32,768 particles took 411 us in
// place of 388, one of 1,777 particles 326 in place of 311.  With equal keys
// the steps are a chain of memory accesses, so a wave looks for the gaps: a
// third of 1,777 particles at one point took 62 ms with one thread, 8 with it.
constexpr int kTieThreads = 256;
constexpr int kTieWidth = 10;           // sl_tune_intern.h:22 (sort_radix_width_default)
constexpr int kTieThreshold = 256;      // sl_tune_intern.h:30 (sort_radix_threshold_rec)
constexpr int kTieClasses = 1 << kTieWidth;
constexpr int kTieDepth = 8;            // 64 bits in 10-bit digits: at most 7 passes

// key_to_intcoord_hilbert / key_to_coord, module_spacefilling.f90:445-565.
constexpr int kC3[8] = {0, 1, 3, 2, 6, 7, 5, 4};
constexpr int kGX[8] = {5, 6, 0, 5, 5, 0, 6, 5};
constexpr int kGR[8] = {0, 0, 0, 5, 0, 0, 6, 5};

__device__ void key_to_intcoord(unsigned long long key, long long ic[3]) {
  const int lev = level_of_key(key);
  ic[0] = ic[1] = ic[2] = 0;
  for (int i = 0; i < lev; ++i) {
    const int h = (int)((key >> (3 * i)) & 7ull);
    const int cval = kC3[h], rev = kGR[h], ex = kGX[h];
    if (i > 0) {
      for (int j = 0; j < 3; ++j)
        if ((rev >> j) & 1) ic[j] = (~ic[j]) & ((1ll << i) - 1);
      for (int j = 0; j < 2; ++j) {
        if (!((ex >> j) & 1)) continue;
        for (int k = j + 1; k < 3; ++k)
          if ((ex >> k) & 1) { long long t = ic[j]; ic[j] = ic[k]; ic[k] = t; }
      }
    }
    for (int j = 0; j < 3; ++j) ic[j] |= (long long)((cval >> j) & 1) << i;
  }
  for (int j = 0; j < 3; ++j) ic[j] <<= (kMaxLevel - lev);
}

// module_domains.f90:248-297 for one system of n particles (keys ks[0..n)),
// in the reference's loop order, by one wave: it visits the nd positions of
// list, those that start with a successor of the same key.  Only they are
// ever modified to a smaller key difference, so this equals visiting every
// position.  The reference's table of key differences kd(i) always equals
// ks[i] - ks[i - 1] (1-based i; 1 at the last position, which no step reads),
// so the keys stand for it.  A step's search for the nearest gap and its
// shift take 64 positions at a time; the steps themselves are a chain.
// lo/hi[r] keep the positions that step r moved.
constexpr int kDupNear = 4;

__device__ void dup_serial(long long n, unsigned long long* ks, const uint32_t* list, uint32_t nd,
                           uint32_t* lo, uint32_t* hi, DevScalars* sc) {
  const int lane = lane_id();
  const bool full = (long long)(ks[n - 1] - ks[0]) + 1 < n;   // :254-262
  if (full && lane == 0) atomicOr(&sc->flags, kFlagDupKeys);
  uint32_t pos = 0, mylo = 1, myhi = 0;   // lane l: of step l of 64
  for (uint32_t r = 0; r < nd; ++r) {
    const int l = (int)(r % kWave);
    if (l == 0) pos = r + lane < nd ? list[r + lane] : 0u;
    long long from = 1, to = 0;   // positions moved (0-based)
    const long long i1 = (long long)__builtin_amdgcn_readlane((int)pos, l) + 1;   // 1-based as in the source
    if (!full) {
      const long long jmax = (n - i1) > i1 ? (n - i1) : i1;
      // the step's own difference, loaded with the first gaps
      const bool equal = (long long)(ks[i1] - ks[i1 - 1]) < 1;
      // first a few gaps, which one or two cache lines hold
      for (long long j0 = 1, w = kDupNear; j0 <= jmax; j0 += w, w = kWave) {
        const long long j = j0 + (lane < w ? lane : 0);
        const bool has_dn = i1 - j >= 1, has_up = i1 + j <= n - 1;
        const long long dn = has_dn ? i1 - j : 1, up = has_up ? i1 + j : 1;
        const unsigned long long kd1 = ks[dn], kd0 = ks[dn - 1], ku1 = ks[up], ku0 = ks[up - 1];
        if (!equal) break;
        const bool down = has_dn && (long long)(kd1 - kd0) > 1;
        const bool hit = down || (has_up && (long long)(ku1 - ku0) > 1);
        const unsigned long long m = __ballot(hit);
        if (m) {
          const int first = __ffsll(m) - 1;
          const bool d = (__ballot(down) >> first) & 1ull;
          from = d ? i1 - (j0 + first) : i1;
          to = d ? i1 - 1 : i1 + (j0 + first) - 1;
          const unsigned long long by = d ? ~0ull : 1ull;   // -1 or +1
          for (long long t = from + lane; t <= to; t += kWave) ks[t] += by;
          break;
        }
      }
      // the next step's loads in every lane see this step's stores
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    if (lane == l) { mylo = (uint32_t)from; myhi = (uint32_t)to; }
    if (l == kWave - 1 || r + 1 == nd) {
      const uint32_t at = r - l + lane;
      if (at < nd) { lo[at] = mylo; hi[at] = myhi; }
    }
  }
}

// The system's particles [b, e): moves equal keys apart and puts every
// particle whose key changed (kin holds the keys in input order) at its new
// key's cell centre, in the records that the sorted particles are taken from.
// list[0..nd): the duplicates' positions in [b, e), increasing.  The steps'
// ranges are usually a position or two, so each thread replays whole steps.
__device__ void fix_duplicates(int64_t b, int64_t e, unsigned long long* ks, const uint32_t* perm,
                               const unsigned long long* kin, const uint32_t* list, uint32_t nd,
                               uint32_t* lo, uint32_t* hi, const DevBox* box, double4* rec,
                               DevScalars* sc) {
  __syncthreads();
  if (threadIdx.x < kWave) dup_serial(e - b, ks + b, list, nd, lo, hi, sc);
  __syncthreads();
  for (uint32_t r = threadIdx.x; r < nd; r += blockDim.x) {
    for (int64_t t = lo[r]; t <= (int64_t)hi[r]; ++t) {
      const unsigned long long key = ks[b + t];
      const uint32_t p = perm[b + t];
      if (key == kin[p]) continue;
      long long ic[3];
      key_to_intcoord(key, ic);
      rec[p].x = ((double)ic[0] + 0.5) * box->cell[0] + box->boxmin[0];
      rec[p].y = ((double)ic[1] + 0.5) * box->cell[1] + box->boxmin[1];
      rec[p].z = ((double)ic[2] + 0.5) * box->cell[2] + box->boxmin[2];
    }
  }
}

__global__ __launch_bounds__(kTieThreads) void tie_order_kernel(
    int64_t n, const int64_t* __restrict__ soff, unsigned long long* ks, uint32_t* perm,
    unsigned long long* kin, uint32_t* ord, uint32_t* ord2, uint16_t* __restrict__ cls,
    uint32_t* __restrict__ fp, unsigned long long* __restrict__ fec, uint32_t* list,
    const DevBox* __restrict__ boxes, double4* rec, DevScalars* __restrict__ sc) {
  if (sc->dup_count == 0) return;
  const int tid = threadIdx.x;
  const int64_t b = soff ? soff[blockIdx.x] : 0;
  const int64_t e = soff ? soff[blockIdx.x + 1] : n;
  if (e - b < 2) return;

  __shared__ uint32_t reg[kTieClasses + 1];   // region starts of the current pass
  __shared__ uint32_t nxt[kTieClasses];       // next unused entry of each region's slot list
  __shared__ uint32_t run_base;
  __shared__ unsigned long long skey[kTieThreshold];
  __shared__ int64_t fs[kTieDepth], fe[kTieDepth], fcur[kTieDepth];
  __shared__ int frh[kTieDepth], fnext[kTieDepth];
  __shared__ int depth;
  __shared__ int64_t found;

  // the positions with a successor of the same key, in increasing order
  list += b;
  if (tid == 0) run_base = 0;
  __syncthreads();
  {
    constexpr int kPer = 8;   // consecutive positions per thread per chunk
    for (int64_t base = b; base + 1 < e; base += (int64_t)kTieThreads * kPer) {
      const int64_t i0 = base + (int64_t)tid * kPer;
      unsigned long long k[kPer + 1];
#pragma unroll
      for (int j = 0; j <= kPer; ++j) k[j] = i0 + j < e ? ks[i0 + j] : 0ull;
      uint32_t nf = 0;
#pragma unroll
      for (int j = 0; j < kPer; ++j) nf += i0 + j + 1 < e && k[j + 1] == k[j] ? 1u : 0u;
      uint32_t tot;
      uint32_t off = run_base + block_exclusive_scan(nf, &tot);
#pragma unroll
      for (int j = 0; j < kPer; ++j)
        if (i0 + j + 1 < e && k[j + 1] == k[j]) list[off++] = (uint32_t)(i0 + j - b);
      __syncthreads();
      if (tid == 0) run_base += tot;
      __syncthreads();
    }
  }
  const uint32_t nd = run_base;   // replaced by the passes below
  __syncthreads();
  if (nd == 0) return;

  // keys in input order (the sort's input of this system is [b, e) too) and
  // the initial order of the top segment
  for (int64_t i = b + tid; i < e; i += kTieThreads) {
    kin[perm[i]] = ks[i];
    ord[i] = (uint32_t)i;
  }
  if (tid == 0) {
    depth = 1;
    fs[0] = b;
    fe[0] = e;
    frh[0] = 63;
    fnext[0] = -2;   // pass not run yet
  }
  __syncthreads();

  while (depth > 0) {
    const int d = depth - 1;
    const int64_t s0 = fs[d], e0 = fe[d];
    const int64_t m = e0 - s0;
    if (fnext[d] == -2) {
      // ---- one pass of rs_rec_ip over [s0, e0) on bits rhigh..sh
      const int rhigh = frh[d];
      const int cw = rhigh + 1 < kTieWidth ? rhigh + 1 : kTieWidth;
      const int sh = rhigh - cw + 1;
      const int K = 1 << cw;
      const unsigned long long mask = (unsigned long long)(K - 1);
      for (int c = tid; c <= K; c += kTieThreads) reg[c] = 0;
      for (int c = tid; c < K; c += kTieThreads) nxt[c] = 0;
      __syncthreads();
      for (int64_t t = tid; t < m; t += kTieThreads) {
        const uint32_t el = ord[s0 + t];
        const int c = (int)((kin[el] >> sh) & mask);
        cls[s0 + t] = (uint16_t)c;
        ord2[s0 + t] = el;
        atomicAdd(&reg[c + 1], 1u);
      }
      __syncthreads();
      if (tid == 0)
        for (int c = 0; c < K; ++c) reg[c + 1] += reg[c];
      __syncthreads();
      // elements already inside their class's region stay; count them
      for (int64_t t = tid; t < m; t += kTieThreads) {
        const int c = cls[s0 + t];
        if ((uint32_t)t >= reg[c] && (uint32_t)t < reg[c + 1]) atomicAdd(&nxt[c], 1u);
      }
      __syncthreads();
      // region r's foreign slots, in increasing position, become entries
      // [start_r, start_r+1) of the slot list (fp: position, fec: element and
      // its class); nxt[r] = start_r, and reg[r] is reused for start_r+1
      if (tid == 0) {
        uint32_t acc = 0;
        for (int c = 0; c < K; ++c) {
          const uint32_t f = reg[c + 1] - reg[c] - nxt[c];
          nxt[c] = acc;
          acc += f;
        }
        run_base = 0;
      }
      __syncthreads();
      {
        constexpr int kPer = 4;   // consecutive positions per thread per chunk
        for (int64_t base = 0; base < m; base += (int64_t)kTieThreads * kPer) {
          const int64_t t0 = base + (int64_t)tid * kPer;
          uint32_t flag[kPer], nf = 0;
#pragma unroll
          for (int j = 0; j < kPer; ++j) {
            const int64_t t = t0 + j;
            flag[j] = 0u;
            if (t < m) {
              const int c = cls[s0 + t];
              flag[j] = ((uint32_t)t >= reg[c] && (uint32_t)t < reg[c + 1]) ? 0u : 1u;
            }
            nf += flag[j];
          }
          uint32_t tot;
          uint32_t off = run_base + block_exclusive_scan(nf, &tot);
#pragma unroll
          for (int j = 0; j < kPer; ++j) {
            if (flag[j]) {
              const int64_t t = t0 + j;
              fp[s0 + off] = (uint32_t)t;
              fec[s0 + off] = (unsigned long long)ord[s0 + t] |
                              ((unsigned long long)cls[s0 + t] << 32);
              ++off;
            }
          }
          __syncthreads();
          if (tid == 0) run_base += tot;
          __syncthreads();
        }
      }
      if (tid == 0) {
        for (int c = 0; c < K; ++c) reg[c] = c + 1 < K ? nxt[c + 1] : run_base;
        // The walk: phase i starts a cycle at each of region i's remaining
        // foreign slots (increasing); the carried element goes to the next
        // unused foreign slot of its class's region, whose element is
        // carried on, until an element of class i closes the cycle in the
        // starting slot.  One list entry per step.
        const uint32_t* fpp = fp + s0;
        const unsigned long long* fe = fec + s0;
        uint32_t* o2 = ord2 + s0;
        for (int i = 0; i < K; ++i) {
          while (nxt[i] < reg[i]) {
            const uint32_t k0 = nxt[i]++;
            const uint32_t p0 = fpp[k0];
            const unsigned long long e0 = fe[k0];
            uint32_t el = (uint32_t)e0;
            int c = (int)(e0 >> 32);
            for (;;) {
              if (nxt[c] >= reg[c]) {   // cannot happen: every region receives what it sends
                atomicOr(&sc->flags, kFlagDupKeys);
                break;
              }
              const uint32_t k = nxt[c]++;
              const uint32_t p = fpp[k];
              const unsigned long long e2 = fe[k];
              o2[p] = el;
              el = (uint32_t)e2;
              const int c2 = (int)(e2 >> 32);
              if (c2 == i) {
                o2[p0] = el;
                break;
              }
              c = c2;
            }
          }
        }
        fnext[d] = sh - 1;
        fcur[d] = s0;
      }
      __syncthreads();
      for (int64_t t = tid; t < m; t += kTieThreads) ord[s0 + t] = ord2[s0 + t];
      __syncthreads();
      if (fnext[d] < 0) {
        // all 64 bits consumed: the segment holds one key, its order is final
        for (int64_t t = tid; t < m; t += kTieThreads) perm[s0 + t] = ord[s0 + t];
        __syncthreads();
        if (tid == 0) depth = d;
        __syncthreads();
        continue;
      }
    }
    // ---- next bucket of this pass that holds a tie
    const int sh = fnext[d] + 1;   // low bit of this pass's digit
    if (tid == 0) found = -1;
    __syncthreads();
    for (int64_t base = fcur[d]; base + 1 < e0; base += kTieThreads) {
      const int64_t i = base + tid;
      if (i + 1 < e0 && ks[i + 1] == ks[i]) atomicMin((unsigned long long*)&found, (unsigned long long)i);
      __syncthreads();
      if (found >= 0) break;
      __syncthreads();
    }
    __syncthreads();
    const int64_t t0 = found;
    if (t0 < 0) {
      if (tid == 0) depth = d;
      __syncthreads();
      continue;
    }
    // bucket = positions of [s0, e0) whose key shares ks[t0]'s bits above sh
    __shared__ int64_t cs, ce;
    if (tid == 0) {
      const unsigned long long pre = ks[t0] >> sh;
      int64_t lo = s0, hi = t0;   // first position with the prefix
      while (lo < hi) {
        const int64_t mid = lo + (hi - lo) / 2;
        if ((ks[mid] >> sh) < pre) lo = mid + 1; else hi = mid;
      }
      cs = lo;
      lo = t0 + 1;
      hi = e0;                    // first position past the prefix
      while (lo < hi) {
        const int64_t mid = lo + (hi - lo) / 2;
        if ((ks[mid] >> sh) <= pre) lo = mid + 1; else hi = mid;
      }
      ce = lo;
      fcur[d] = ce;
    }
    __syncthreads();
    const int64_t c0 = cs, c1 = ce, cm = c1 - c0;
    if (cm > kTieThreshold) {
      __syncthreads();
      if (tid == 0) {
        fs[d + 1] = c0;
        fe[d + 1] = c1;
        frh[d + 1] = fnext[d];
        fnext[d + 1] = -2;
        depth = d + 2;
      }
      __syncthreads();
      continue;
    }
    // stable insertion sort of a small bucket (sort_insert.c:14-37): rank
    // by key, equal keys in their current order
    uint32_t el = 0;
    unsigned long long k = 0;
    if (tid < cm) {
      el = ord[c0 + tid];
      k = kin[el];
      skey[tid] = k;
    }
    __syncthreads();
    if (tid < cm) {
      int r = 0;
      for (int u = 0; u < (int)cm; ++u) {
        const unsigned long long ku = skey[u];
        r += (ku < k || (ku == k && u < tid)) ? 1 : 0;
      }
      perm[c0 + r] = el;
    }
    __syncthreads();
  }
  fix_duplicates(b, e, ks, perm, kin, list, nd, ord + b, ord2 + b, boxes + (soff ? blockIdx.x : 0),
                 rec, sc);
}

}  // namespace

void launch_tie_order(hipStream_t s, int64_t n, int64_t nsys, const int64_t* soff,
                      unsigned long long* ks, uint32_t* perm, unsigned long long* kin,
                      uint32_t* ord, uint32_t* ord2, uint16_t* cls, uint32_t* fp,
                      unsigned long long* fec, uint32_t* list, const DevBox* boxes, double4* rec,
                      DevScalars* sc) {
  if (n < 2) return;
  tie_order_kernel<<<(unsigned)(nsys > 1 ? nsys : 1), kTieThreads, 0, s>>>(
      n, nsys > 1 ? soff : nullptr, ks, perm, kin, ord, ord2, cls, fp, fec, list, boxes,
      rec, sc);
}

int64_t scan_blocks(int64_t n) { return (n + kScanTile - 1) / kScanTile; }
int64_t sort_blocks(int64_t n) { return (n + kSortTile - 1) / kSortTile; }

void launch_scan(hipStream_t s, const uint32_t* in, uint32_t* out, int64_t n, uint32_t* bsum,
                 uint32_t* total) {
  if (n <= 0) return;
  const int64_t nb = scan_blocks(n);
  scan_reduce_kernel<<<(unsigned)nb, kScanThreads, 0, s>>>(in, n, bsum, false);
  scan_small_kernel<<<1, kScanThreads, 0, s>>>(bsum, (int)nb, total);
  scan_apply_kernel<<<(unsigned)nb, kScanThreads, 0, s>>>(in, out, n, bsum);
}

// Blocks of marks up to which each block of group_list_kernel adds the counts
// of the blocks before it itself, which saves the launch that scans them:
// they are 8 KB at most, four loads of 16 bytes a thread.
constexpr int64_t kGroupSumBlocks = 2048;

void launch_group_list(hipStream_t s, int64_t n, const uint32_t* gmark, uint32_t* bsum,
                       uint32_t* gfirst, uint32_t* gcount, uint32_t* ngroups,
                       unsigned long long* clock) {
  const int64_t nb = scan_blocks(n);
  const bool scanned = nb > kGroupSumBlocks;
  scan_reduce_kernel<<<(unsigned)nb, kScanThreads, 0, s>>>(gmark, n, bsum, true);
  if (scanned) scan_small_kernel<<<1, kScanThreads, 0, s>>>(bsum, (int)nb, nullptr);
  group_list_kernel<<<(unsigned)nb, kScanThreads, 0, s>>>(n, gmark, bsum, scanned, gfirst, gcount,
                                                          ngroups, clock);
}

// One stable pass over bits [shift, shift + nbits) of the keys (or, with dsrc,
// of dsrc[value]), output in (kout, vout).
static void launch_radix_pass(hipStream_t s, const unsigned long long* kin, const uint32_t* vin,
                              unsigned long long* kout, uint32_t* vout, int64_t n, int shift,
                              int nbits, uint32_t* hist, uint32_t* bsum, const uint32_t* dsrc) {
  const int nb = (int)sort_blocks(n);
  radix_hist_kernel<<<nb, kSortThreads, 0, s>>>(kin, vin, dsrc, n, shift, (1u << nbits) - 1u, hist,
                                                nb);
  // Few blocks: each scatter block sums its digits' rows itself, one launch
  // fewer per pass.  Otherwise bsum[0..255] holds the digit totals.
  const bool scan_here = nb <= kScanHereBlocks;
  if (!scan_here) digit_scan_kernel<<<kRadix, kSortThreads, 0, s>>>(hist, nb, bsum);
  radix_scatter_kernel<<<nb, kSortThreads, 0, s>>>(kin, vin, kout, vout, dsrc, n, shift, nbits, hist,
                                                   bsum, nb, scan_here);
}

// Largest array sorted by merging.
constexpr int64_t kMergeMax = 524288;

// Largest array whose blocks are sorted by counting: a whole grow of 65,536
// particles takes 182 us with it and 190 with the network, of 131,072 the
// same 234 and of 262,144 306 and 283.
constexpr int64_t kRankMax = 65536;

// Largest array merged with two search steps at a time (grow of 32,768
// particles 155 -> 145 us, 131,072 232 -> 222, but 524,288 346 -> 356).
constexpr int64_t kMergePairMax = 131072;

static int merge_launches(int64_t n) {
  int merges = 0;
  for (int64_t run = kMergeN; run < n; run *= 4) ++merges;
  return merges;
}

bool sort_input_second(int64_t n, bool batched) {
  return !batched && n <= kRankMax && merge_launches(n) % 2 == 0;
}

static void launch_merge_sort(hipStream_t s, unsigned long long* k0, uint32_t* v0,
                              unsigned long long* k1, uint32_t* v1, int64_t n) {
  const int merges = merge_launches(n);
  unsigned long long *ka = k0, *kb = k1;
  uint32_t *va = v0, *vb = v1;
  if (merges % 2) { std::swap(ka, kb); std::swap(va, vb); }   // so the result ends in (k0, v0)
  if (n <= kRankMax)   // not in place: the input is in the other pair
    rank_block_kernel<<<(unsigned)((n + kWave - 1) / kWave), kRankT, 0, s>>>(kb, vb, ka, va, n);
  else
    merge_block_kernel<<<(unsigned)((n + kMergeN - 1) / kMergeN), kMergeT, 0, s>>>(k0, v0, ka, va, n);
  int run = kMergeN;
  for (int m = 0; m < merges; ++m, run *= 4) {
    auto* merge = n <= kMergePairMax ? merge4_kernel<true> : merge4_kernel<false>;
    merge<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(ka, va, kb, vb, (int)n, run);
    std::swap(ka, kb);
    std::swap(va, vb);
  }
}

// Full sort of particle keys over bits [0, 60), values ascending on input.
// Input in (k0, v0), or in (k1, v1) where sort_input_second says so; the
// sorted result ends in (k0, v0).  With a system
// index per input particle (sysid != nullptr, values < nsys <= 65536), two more
// stable passes over its 16 bits order the particles by (system, key); the
// upper pass only runs when there are more than 256 systems, and then the
// lower one goes to (k1, v1) and the upper one back.
void launch_sort_keys(hipStream_t s, unsigned long long* k0, uint32_t* v0, unsigned long long* k1,
                      uint32_t* v1, int64_t n, uint32_t* hist, uint32_t* bsum,
                      const uint32_t* sysid, int64_t nsys) {
  if (!sysid && n <= kMergeMax) {
    launch_merge_sort(s, k0, v0, k1, v1, n);
    return;
  }
  static const int shifts[8] = {0, 8, 16, 24, 32, 40, 48, 56};
  static const int widths[8] = {8, 8, 8, 8, 8, 8, 8, 4};
  for (int p = 0; p < 8; ++p) {
    if (p % 2 == 0)
      launch_radix_pass(s, k0, v0, k1, v1, n, shifts[p], widths[p], hist, bsum, nullptr);
    else
      launch_radix_pass(s, k1, v1, k0, v0, n, shifts[p], widths[p], hist, bsum, nullptr);
  }
  if (sysid) {
    launch_radix_pass(s, k0, v0, k1, v1, n, 0, 8, hist, bsum, sysid);
    if (nsys > 256) {
      launch_radix_pass(s, k1, v1, k0, v0, n, 8, 8, hist, bsum, sysid);
    } else {
      launch_copy_pairs(s, k1, v1, k0, v0, n);
    }
  }
}

void launch_scatter_back(hipStream_t s, int64_t n, const uint32_t* perm, const double* in,
                         double* out) {
  scatter_back_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, perm, in, out);
}

void launch_restore_fields(hipStream_t s, int64_t n, const uint32_t* perm, const double* ex,
                           const double* ey, const double* ez, const double* pot, double* e,
                           double* phi) {
  restore_fields_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, perm, ex, ey, ez, pot, e, phi);
}

void launch_sort_fields(hipStream_t s, int64_t n, const uint32_t* perm, const double* e,
                        const double* phi, double* ex, double* ey, double* ez, double* pot) {
  sort_fields_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, perm, e, phi, ex, ey, ez, pot);
}

void launch_gather_rec(hipStream_t s, int64_t n, const uint32_t* perm, const double4* rec,
                       double* xs, double* ys, double* zs, double* qs) {
  gather_rec_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, perm, rec, xs, ys, zs, qs);
}

void launch_gather4(hipStream_t s, int64_t n, const uint32_t* perm, const double* x, const double* y,
                    const double* z, const double* q, double* xs, double* ys, double* zs,
                    double* qs) {
  gather4_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(n, perm, x, y, z, q, xs, ys, zs, qs);
}

}  // namespace pepc
