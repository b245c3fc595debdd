// common.h -- shared device helpers and data layouts of the MI355X tree solve.
//
// Wave64 primitives (ballot, lane masks, butterfly reductions), the device
// box record and the per-node records the walk reads.  Everything here is
// written for gfx950 (CDNA4): 64-lane wavefronts, 160 KiB LDS per CU.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pepc {

constexpr int kWave = 64;
constexpr int kMaxLevel = 20;          // (64 - 2) / 3, treevars.f90:371

// Status bits raised by kernels (read back by the host after a phase).
enum : uint32_t {
  kFlagDupKeys = 1u << 0,       // equal adjacent keys after the sort
  kFlagNodeOverflow = 1u << 1,  // node pool too small
  kFlagStackOverflow = 1u << 2, // walk stack overflow (never expected)
  kFlagDepth = 1u << 3,         // more than 20 levels needed
  kFlagBadBox = 1u << 4,        // non-finite or degenerate bounding box
  kFlagGroupOverflow = 1u << 5, // group larger than a wavefront
};

// Bounding box and derived per-level tables, module_box.f90:33-37 plus
// module_tree.f90:196-201 (boxlength2).
struct DevBox {
  double boxmin[3];
  double boxmax[3];
  double boxsize[3];
  double cell[3];               // boxsize / 2^20, the refinement length
  double b2[kMaxLevel + 1];     // maxval(boxsize)^2 / 4^l
  uint32_t qsign;               // kQPositive | kQNegative: signs among the charges
  uint32_t mixed;               // both signs at the grow: FP32 walk records in the second form below
};

// A system whose charges all have one sign has no dipole moments: a node's
// expansion centre is the |charge|-weighted mean of its particles.
enum : uint32_t { kQPositive = 1u, kQNegative = 2u };

// Device-wide scalars the host reads once per solve (one small copy).
struct DevScalars {
  uint32_t flags;
  uint32_t nnodes;
  uint32_t ntwig;
  uint32_t ngroups;
  uint32_t pad0;
  uint32_t maxlevel_used;
  uint32_t level_offset[kMaxLevel + 2];   // first node of every level; [kMaxLevel + 1] = nnodes
  uint32_t twig_offset[kMaxLevel + 2];    // first twig rank of every level; [kMaxLevel + 1] = ntwig
  unsigned long long interactions;
  unsigned long long mac_evals;
  unsigned long long p2p;
  unsigned long long m2p;
  unsigned long long amb_nodes;   // twigs the group box could not decide
  unsigned long long walk_steps;  // traversal steps (batches of up to 64 nodes)
  uint32_t dup_count;
  uint32_t pad;
};

// Node record read by the walk for the acceptance test: centre of charge
// and the squared box length of the node's level (for a leaf, whose centre
// is its particle, the last slot holds the particle's charge instead).
struct __align__(32) NodeGeom {
  double cx, cy, cz, b2;
};

// Topology: first child (twig) or particle index (leaf), child count
// (0 for a leaf), and the number of particles below the node.
struct __align__(16) NodeLink {
  uint32_t first;
  uint32_t nchild;
  uint32_t count;
  uint32_t level;
};

// Moments in the form the M2P kernel evaluates (see walk.hip): -3 times the
// quadrupole matrix A2 = {2 quad, off-diagonals}, twice the trace of quad, the
// dipole and the charge.
// Slots: 0..2 -3 A2 xx yy zz | 3 xy | 4 yz | 5 zx | 6 2 tr | 7..9 p | 10 q
// FP32 records of a system with charges of both signs (DevBox::mixed), the
// reference's terms: 0 q | 1..3 p | 4..6 2 quad | 7 xy | 8 yz | 9 zx | 10 tr
template <typename R>
struct __align__(16) NodeMoments {
  R v[16];
};

__device__ __forceinline__ int lane_id() { return __lane_id(); }

__device__ __forceinline__ unsigned long long lanemask_lt() {
  const int l = __lane_id();
  return l == 0 ? 0ull : (~0ull >> (64 - l));
}

__device__ __forceinline__ int popc64(unsigned long long m) { return __popcll(m); }

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}

__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, kWave));
  return v;
}

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, kWave));
  return v;
}

// Maximum over the wave (every lane active), uniform: each row of 16 lanes by
// DPP, then the four rows through scalar reads, so no LDS round trips.
__device__ __forceinline__ int wave_max_i32(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false));    // quad_perm [1,0,3,2]
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false));    // quad_perm [2,3,0,1]
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x124, 0xF, 0xF, false));   // row_ror:4
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, false));   // row_ror:8
  return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// Inclusive prefix sum across the wave (Hillis-Steele over 6 steps).
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
  const int l = __lane_id();
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    uint32_t t = __shfl_up(v, o, kWave);
    if (l >= o) v += t;
  }
  return v;
}

// Number of set bits of m in the lanes below this one (v_mbcnt_lo/hi).
__device__ __forceinline__ uint32_t mask_rank(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Exclusive prefix sum across the wave of values below 16, built from four
// ballots (bit planes) instead of lane shuffles; *total gets the wave's sum.
__device__ __forceinline__ uint32_t wave_exclusive_scan16(uint32_t v, uint32_t* total) {
  uint32_t ex = 0, tot = 0;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const unsigned long long m = __ballot((v >> b) & 1u);
    ex += mask_rank(m) << b;
    tot += (uint32_t)__popcll(m) << b;
  }
  *total = tot;
  return ex;
}

// Level of a key: position of the placeholder bit, module_spacefilling.f90:47-57.
__device__ __forceinline__ int level_of_key(unsigned long long k) {
  return (63 - __clzll((long long)k)) / 3;
}

// First level at which two distinct particle keys fall into different cells.
__device__ __forceinline__ int split_level(unsigned long long a, unsigned long long b) {
  unsigned long long x = a ^ b;
  int msb = 63 - __clzll((long long)x);
  return kMaxLevel - msb / 3;
}

// Device clock at the ends of a grow and of a walk, written by their own
// first and last kernels: four events on the stream took 14 us of every solve.
enum { kClockGrow = 0, kClockGrown, kClockWalk, kClockWalked, kClocks };

// Work queues of the persistent kernels, one per XCD: the items (in key
// order) are cut into nq contiguous ranges and workgroup b, which the
// dispatcher places on XCD b mod nq, takes items from range b mod nq first, so
// the waves sharing an XCD's L2 work on neighbouring items and reuse the same
// nodes.  A used-up range sends the wave on to the next one.
// The first items of a range belong to its workgroups by number, only the
// others are counted out by the range's head, and the first wave that finds a
// range used up says so in the last word, which a wave reads once, when its
// own range has ended.  Atomics on one address are served one after another
// (15 ns each), and every wave used to ask all eight heads at its end: 4,096
// waves spent 60 us of every walk that way (487 groups: 92 -> 28 us; 8,400:
// 198 -> 146; 134,000: 1.63 -> 1.59 ms).  Reading a head before asking it is
// worse (98 ns per item), and so is handing out several items at once, whose
// nodes the neighbouring waves then no longer share (4 at a time, 4,194,304
// particles: 5.13 -> 5.45 ms).
constexpr int kMaxQueues = 8;
constexpr int kQueueStride = 16;   // words: a 64-byte line for each head
constexpr int kQueueWords = (kMaxQueues + 1) * kQueueStride;   // zero at a kernel's start

struct GroupQueue {
  uint32_t nq, q, todo;   // queues, position, ranges to look at
  uint32_t mine;          // the item by number, then ~0
  bool looked;

  __device__ __forceinline__ void init(uint32_t queues) {
    nq = queues;
    q = blockIdx.x % nq;
    todo = (1u << nq) - 1u;
    mine = blockIdx.x / nq;
    looked = false;
  }
  // One lane of the workgroup: the next of n items, or n when there is none.
  __device__ __forceinline__ uint32_t next(uint32_t* heads, uint32_t n) {
    while (todo) {
      if ((todo >> q) & 1u) {
        const uint32_t lo = (uint32_t)((uint64_t)n * q / nq);
        const uint32_t size = (uint32_t)((uint64_t)n * (q + 1) / nq) - lo;
        const uint32_t given = (gridDim.x - q + nq - 1u) / nq;   // workgroups of this range
        uint32_t r = mine;
        mine = ~0u;
        if (r >= size && size > given) {
          r = given + atomicAdd(heads + kQueueStride * q, 1u);
          if (r == size) atomicOr(heads + kQueueStride * kMaxQueues, 1u << q);
        }
        if (r < size) return lo + r;
        todo &= ~(1u << q);
        if (!looked) {
          todo &= ~__hip_atomic_load(heads + kQueueStride * kMaxQueues, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
          looked = true;
        }
      }
      q = q + 1 == nq ? 0u : q + 1;
    }
    return n;
  }
};

}  // namespace pepc
