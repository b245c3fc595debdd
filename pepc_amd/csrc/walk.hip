// walk.hip -- persistent group walk with P2P/M2P force and potential kernels.
//
// Semantics (module_tree_walk_simple.f90:256-384): a group of target
// particles (a walk tile) descends the tree from the root; a leaf interacts
// with every target (P2P, self excluded); a twig is accepted for M2P only if
// every target passes the Barnes-Hut test theta2*d^2 > b^2(level)
// (coulomb/module_interaction_specific.f90:256-275), otherwise it is opened.
// Interaction counts per target and MAC-evaluation counts per group equal the
// reference's at the same group rule.
//
// Mapping to CDNA4.  One 64-lane wavefront owns one group at a time and pulls
// the next group from a device queue (persistent kernel).  A lane holds one
// or two of the group's targets (NT); the W lanes that hold them all form a
// slice, and the S = 64/W slices split every interaction list between them,
// so small groups still fill the wave.  Traversal is breadth-parallel: each step pops up to 64 nodes from an
// LDS stack, one node per lane, and decides it against the group's bounding
// box; only nodes whose decision the box cannot settle run the exact
// per-target FP64 test (all lanes, one ballot).  Accepted nodes and leaves are
// appended to M2P / P2P lists staged in LDS and evaluated in batches: every
// lane reads the same entry (LDS broadcast) and evaluates it for its target.
//
// Precision.  FP32 path (of systems whose charges have one sign; the others
// keep an evaluation of their own, see walk_group_mixed): coordinates relative to the group's first particle
// (differences taken in FP64 once per node, then rounded), FP32 kernels with
// fused multiply-add, FP32 partial sums per batch added to FP64 running sums
// (more exact than the compensated FP32 sums they replace, with half the
// instructions).  FP64 path: absolute coordinates, FP64 kernels, plain FP64
// accumulation, as the reference.
//
// What bounds it: vector-ALU issue.  With four waves per SIMD this chip
// issues an FP32 instruction every 3 clocks per SIMD and every other kind
// (FP64, integer, compares, any with a scalar operand) every 4.3 to 4.8; the
// 4.2M-particle explosion at theta 0.6 issued 4.36e9 VALU instructions at
// 3.0 clocks each.  So the design counts instructions: no dipole
// terms for one-signed charges (41 -> 36 per pair), list remainders kept so
// that passes are full, one ballot transposition for the exact tests and one
// for the pushes.  Now 3.87e9 instructions at 3.0 clocks, FP64 4.97e9 at 4.8
// (walk 5.13 and 10.2 ms).
//
// Periodic systems (PER): the group walks the tree once per lattice vector
// vbox of the mirror boxes, with its targets shifted to x - vbox
// (module_libpepc_main.f90:184-187, module_tree_walk_simple.f90:328,345);
// sums run on across the boxes.  Self is excluded in the central box only.
// FP64 keeps separations as (x - vbox) - coc and flushes its lists at the end
// of each box; FP32 puts the shift into the node frame instead (node entries
// relative to first particle - vbox), so its lists carry over.
//
// Sinks (SINK): targets other than the grown particles (the reference's
// traversal of another particle array, module_pepc.f90:394-433).  Targets
// come from their own arrays, one per group (the reference's rule for
// particles without keys, module_tree_walk_simple.f90:155-159) or in given
// runs; self is the reference's test, a zero separation from the leaf's
// particle (:331-340), checked exactly in FP64 against the source
// coordinates; lists are flushed at the end of each box.
//
// The M2P evaluation regroups the reference's expression
// (module_coulomb_kernels.f90:60-145) around the quadratic form
// S = d.A.d of the quadrupole tensor; it is the same polynomial in d and the
// moments (phi = q/r - d.p/r^3 + 3 S/r^5 - tr(A)/r^3 and E = -grad phi with
// r^2 = d^2 + eps^2), evaluated with fewer operations (see m2p).
#include "kernels.h"

#include <type_traits>

namespace pepc {

namespace {

constexpr int kStackCap = 512;      // entries the pop policy keeps below (FP64)
constexpr int kStackCap32 = 768;    // the same for FP32, whose lists leave LDS for it
constexpr int kStackSlack = 192;    // >= 7 * 21 + 8: depth-first overrun bound
constexpr int kListP = 64;
// Stack entries carry the node's kind in their top bit (set for a twig, and
// for a root whatever it is), so a leaf's step skips the walk-moment loads.
constexpr uint32_t kTwigBit = 0x80000000u;

template <typename R> struct Prec;
template <> struct Prec<float> {
  using V4 = float __attribute__((ext_vector_type(4)));
  // v_rsq_f32 (1 ulp).  Its argument is r^2 = d^2 + eps^2 of an interaction
  // that is not a self term; the input guard of rsqrtf() only matters for
  // denormal arguments, which would need |d| and eps below 1e-19.
  static __device__ __forceinline__ float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
  static __device__ __forceinline__ float fm(float a, float b, float c) { return fmaf(a, b, c); }
};
template <> struct Prec<double> {
  using V4 = double __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ double rsq(double x) { return rsqrt(x); }
  static __device__ __forceinline__ double fm(double a, double b, double c) { return fma(a, b, c); }
};

template <typename R>
struct Acc {
  double s[4];  // running sums   ex, ey, ez, pot
  R p[4];       // partial sums of the current batch
};

// M2P.  With w = 1/r^2, A2 = 2 Qt, tr = trace Qt, h = -3 w A2 d, y = d.h + 2 tr
// and p = the dipole:
//   phi = (1/r) (q - w (d.p + 0.5 y))
//   E   = (w/r) (c d + p + h),   c = q - w (3 d.p + 2.5 y - 2 tr)
// which is phi and -grad phi of module_coulomb_kernels.f90:60-145.  The
// separation d is target minus centre of charge.
// Every factor lies between r^-3 and the moments times r, so for charges near
// one FP32 holds separations and softenings from 1e-11 to 1e12.  E summed as
// r^-3 c d + r^-5 B d with a traceless B is an instruction shorter (solve of
// 4,194,304 particles 6.66 ms against 6.76, clustered 1,048,576 3.49 against
// 3.53), but r^-5 leaves FP32 below a separation of 2e-8 and above 4e7.
// Entry: {cx,cy,cz,q | -3 A2: xx,yy,zz,xy | yz,zx, 2 tr,px | py,pz,-,-}.
// Without a dipole (DIP = false) its terms and its words are left out.
template <typename R, bool DIP>
__device__ __forceinline__ void m2p(R dx, R dy, R dz, R q, const typename Prec<R>::V4& b,
                                    const typename Prec<R>::V4& c, R py, R pz, R eps2, R* p) {
  using P = Prec<R>;
  const R r2 = P::fm(dz, dz, P::fm(dy, dy, P::fm(dx, dx, eps2)));
  const R rd = P::rsq(r2);
  const R w = rd * rd;
  const R rd3 = rd * w;
  const R hx = w * P::fm(b.x, dx, P::fm(b.w, dy, c.y * dz));
  const R hy = w * P::fm(b.y, dy, P::fm(b.w, dx, c.x * dz));
  const R hz = w * P::fm(b.z, dz, P::fm(c.x, dy, c.y * dx));
  const R y = P::fm(dz, hz, P::fm(dy, hy, P::fm(dx, hx, c.z)));
  R vx = hx, vy = hy, vz = hz, cc;
  if constexpr (DIP) {
    const R px = c.w;
    const R av = P::fm(dz, pz, P::fm(dy, py, dx * px));
    p[3] = P::fm(rd, P::fm(-w, P::fm(R(0.5), y, av), q), p[3]);
    cc = P::fm(-w, P::fm(R(2.5), y, P::fm(R(3), av, -c.z)), q);
    vx += px; vy += py; vz += pz;
  } else {
    const R y2 = w * y;
    p[3] = P::fm(rd, P::fm(R(-0.5), y2, q), p[3]);
    cc = P::fm(w, c.z, P::fm(R(-2.5), y2, q));
  }
  p[0] = P::fm(rd3, P::fm(cc, dx, vx), p[0]);
  p[1] = P::fm(rd3, P::fm(cc, dy, vy), p[1]);
  p[2] = P::fm(rd3, P::fm(cc, dz, vz), p[2]);
}

// P2P (module_coulomb_kernels.f90:242-257): phi = q/r, E = q d / r^3.
template <typename R>
__device__ __forceinline__ void p2p(R dx, R dy, R dz, R q, R eps2, bool self, R* p) {
  using P = Prec<R>;
  R r2 = P::fm(dz, dz, P::fm(dy, dy, P::fm(dx, dx, eps2)));
  r2 = self ? R(1) : r2;
  const R qe = self ? R(0) : q;
  const R rd = P::rsq(r2);
  const R qrd = qe * rd;
  const R qrd3 = qrd * (rd * rd);
  p[3] += qrd;
  p[0] = P::fm(qrd3, dx, p[0]);
  p[1] = P::fm(qrd3, dy, p[1]);
  p[2] = P::fm(qrd3, dz, p[2]);
}

// Adds a batch's partial sums to the running sums, which are FP64 in both
// precisions.
template <typename R>
__device__ __forceinline__ void fold(Acc<R>& a) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    a.s[k] += (double)a.p[k];
    a.p[k] = R(0);
  }
}

// Exact reference MAC for one target, FP64 without contraction.
__device__ __forceinline__ bool mac_fails(double xt, double yt, double zt, double cx, double cy,
                                          double cz, double b2, double theta2) {
#pragma clang fp contract(off)
  const double dx = xt - cx, dy = yt - cy, dz = zt - cz;
  const double d2 = dx * dx + dy * dy + dz * dz;
  return !(theta2 * d2 > b2);
}

// Orders this wave's LDS accesses for the compiler.  A workgroup is one wave,
// whose LDS instructions execute in order, so no wait or barrier instruction
// is needed between one lane's write and another lane's read.
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// A value that is the same in every lane, moved to scalar registers.
__device__ __forceinline__ uint32_t uniform(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}
__device__ __forceinline__ double uniform(double v) {
  const int lo = __builtin_amdgcn_readfirstlane(__double2loint(v));
  const int hi = __builtin_amdgcn_readfirstlane(__double2hiint(v));
  return __hiloint2double(hi, lo);
}

template <int kCtrl>
__device__ __forceinline__ double dpp_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), kCtrl, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), kCtrl, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_value(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}
// Minimum over the wave (every lane active), uniform: each row of 16 lanes by
// DPP, then the four rows through scalar reads; no LDS round trips.
__device__ __forceinline__ double uniform_min(double v) {
  v = fmin(v, dpp_move<0xB1>(v));    // quad_perm [1,0,3,2]
  v = fmin(v, dpp_move<0x4E>(v));    // quad_perm [2,3,0,1]
  v = fmin(v, dpp_move<0x124>(v));   // row_ror:4
  v = fmin(v, dpp_move<0x128>(v));   // row_ror:8
  return uniform(fmin(fmin(lane_value(v, 0), lane_value(v, 16)),
                      fmin(lane_value(v, 32), lane_value(v, 48))));
}

// Centre and half width of the interval [lo, hi], the half width rounded up so
// that lo and hi lie within it of the (rounded) centre.
struct Span { double c, h; };
__device__ __forceinline__ Span span_of(double lo, double hi) {
  Span r;
  r.c = uniform(0.5 * (lo + hi));
  r.h = uniform(fmax(hi - r.c, r.c - lo) * (1.0 + 4e-15));
  return r;
}

// ---- FP32 groups of systems with charges of both signs
// Close pairs of opposite charges make a trajectory of such a system amplify
// any change of rounding, so its FP32 forces keep one fixed evaluation: the
// reference's grouping of the terms, one target per lane, lists emptied whole,
// Kahan sums, slices added in order.  With the form used for one-signed
// systems, 20 steps of 8,192 to 262,144 thermal particles differed from this
// one by 1e-5 in the velocities (their own FP32 error is 3e-5), and some pairs
// and their order by far more; a single solve by 1e-7.
// That form is the faster one (256 systems: 5.34 against 5.53 ms per solve;
// 65,536 particles: 392 against 409 us); the sums of many slices by lane
// instead of by shuffles took 65,536 sinks from 904 to 662 us.  The children
// are pushed by their parent's lane: eight lanes per parent, as in
// walk_kernel, spill here (256 systems 5.53 -> 5.67 ms).
struct MixedAcc {
  float s[4];  // running sums   ex, ey, ez, pot
  float c[4];  // compensation
  float p[4];  // partial sums of the current batch
};

// Entry {cx,cy,cz,q | px,py,pz,2qx | 2qy,2qz,xy,yz | zx,tr,-,-}.  With w = 1/r^2,
// A2 = [[2qx,xy,zx],[xy,2qy,yz],[zx,yz,2qz]], g = A2 d, S2 = d.g, a = d.p + tr:
//   phi = (1/r) (q - w (a - 1.5 w S2))
//   E   = (w/r) (c d + p - 3 w g),   c = q - 3 w (a - 2.5 w S2)
__device__ __forceinline__ void m2p_mixed(float dx, float dy, float dz, const Prec<float>::V4& b,
                                          const Prec<float>::V4& c, const Prec<float>::V4& d, float q,
                                          float eps2, float* p) {
  using R = float;
  using P = Prec<R>;
  const R r2 = P::fm(dz, dz, P::fm(dy, dy, P::fm(dx, dx, eps2)));
  const R rd = P::rsq(r2);
  const R w = rd * rd;
  const R rd3 = rd * w;
  const R px = b.x, py = b.y, pz = b.z, qx2 = b.w;
  const R qy2 = c.x, qz2 = c.y, xy = c.z, yz = c.w;
  const R zx = d.x, tr = d.y;
  const R gx = P::fm(qx2, dx, P::fm(xy, dy, zx * dz));
  const R gy = P::fm(qy2, dy, P::fm(xy, dx, yz * dz));
  const R gz = P::fm(qz2, dz, P::fm(yz, dy, zx * dx));
  const R s2 = P::fm(dz, gz, P::fm(dy, gy, dx * gx));
  const R av = P::fm(dz, pz, P::fm(dy, py, P::fm(dx, px, tr)));
  const R bv = w * s2;
  p[3] = P::fm(rd, P::fm(-w, P::fm(R(-1.5), bv, av), q), p[3]);
  const R w3 = R(3) * w;
  const R cc = P::fm(-w3, P::fm(R(-2.5), bv, av), q);
  p[0] = P::fm(rd3, P::fm(cc, dx, P::fm(-w3, gx, px)), p[0]);
  p[1] = P::fm(rd3, P::fm(cc, dy, P::fm(-w3, gy, py)), p[1]);
  p[2] = P::fm(rd3, P::fm(cc, dz, P::fm(-w3, gz, pz)), p[2]);
}

// Kahan step on the batch's partial sums.
__device__ __forceinline__ void fold_mixed(MixedAcc& a) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float y = a.p[k] - a.c[k];
    const float t = a.s[k] + y;
    a.c[k] = (t - a.s[k]) - y;
    a.s[k] = t;
    a.p[k] = 0.0f;
  }
}

// One group (targets a0 .. a0 + cnt - 1) of walk_kernel<float>, whose LDS
// arrays it uses; traversal, decisions, counts and records are the same.
template <int LM, bool PER, bool SINK>
__device__ __forceinline__ void walk_group_mixed(const WalkArgs& a, uint32_t g, uint32_t a0,
                                                 uint32_t cnt, uint32_t* stack,
                                                 Prec<float>::V4 (*lm)[4], Prec<float>::V4* lp,
                                                 uint32_t* lpi) {
  using R = float;
  using V4 = Prec<float>::V4;
  constexpr int kCap = kStackCap32;
  const int lane = threadIdx.x;
  const R eps2 = (R)a.eps2;
  const double theta2 = a.theta2;
  const double t_acc = theta2 * (1.0 - 1e-12), t_rej = theta2 * (1.0 + 1e-12);
  const double* __restrict__ TX = SINK ? a.tx : a.x;
  const double* __restrict__ TY = SINK ? a.ty : a.y;
  const double* __restrict__ TZ = SINK ? a.tz : a.z;
  // Lanes s*cnt .. s*cnt+cnt-1 form slice s (s < S = 64/cnt) and hold the
  // group's targets in order; the 64 - S*cnt remaining lanes hold copies
  // of targets for the box and take no part in the sums.
  const uint32_t T = cnt;
  const uint32_t S = kWave / T;
  const uint32_t s = (uint32_t)lane / T;
  const uint32_t t = (uint32_t)lane - s * T;
  const bool valid = s < S;
  const uint32_t tid = a0 + t;
  const double xt = TX[tid], yt = TY[tid], zt = TZ[tid];
  const double ox = uniform(xt), oy = uniform(yt), oz = uniform(zt);   // lane 0: target a0
  const double lox = uniform_min(xt), loy = uniform_min(yt), loz = uniform_min(zt);
  const double hix = -uniform_min(-xt), hiy = -uniform_min(-yt), hiz = -uniform_min(-zt);
  // target position relative to the group's first particle
  const R tx = (R)(xt - ox), ty = (R)(yt - oy), tz = (R)(zt - oz);

  MixedAcc acc;
#pragma unroll
  for (int k = 0; k < 4; ++k) { acc.s[k] = R(0); acc.c[k] = R(0); acc.p[k] = R(0); }

  uint32_t sp = 0, nm = 0, np = 0, cnt_p2p = 0, cnt_m2p = 0, namb = 0, nsteps = 0;
  uint32_t mac_lane = 0;   // this lane's MAC evaluations, summed over the wave at the end
  bool overflow = false;
  const uint32_t root = (!SINK && a.sys) ? a.sysroot[a.sys[a0]] : 0u;   // the group's own root
  double sx = xt, sy = yt, sz = zt;    // targets of the current box: x - vbox

  // Batches: entry k goes to slice k mod S; the loop count is uniform.
  // Two entries per pass (their LDS reads issued together), then the tail.
  auto flush_m2p = [&]() {
    uint32_t kk = 0;
    const uint32_t n2 = nm >= 2 * S ? nm - 2 * S + 1 : 0;
    if (valid) {
      for (; kk < n2; kk += 2 * S) {
        const uint32_t k = kk + s, k2 = k + S;
        const V4 e0 = lm[k][0], e1 = lm[k][1], e2 = lm[k][2], e3 = lm[k][3];
        const V4 f0 = lm[k2][0], f1 = lm[k2][1], f2 = lm[k2][2], f3 = lm[k2][3];
        m2p_mixed(tx - (R)e0.x, ty - (R)e0.y, tz - (R)e0.z, e1, e2, e3, (R)e0.w, eps2, acc.p);
        m2p_mixed(tx - (R)f0.x, ty - (R)f0.y, tz - (R)f0.z, f1, f2, f3, (R)f0.w, eps2, acc.p);
      }
    }
    kk = n2 ? ((n2 - 1) / (2 * S) + 1) * 2 * S : 0;
    for (; kk < nm; kk += S) {
      const uint32_t k = kk + s;
      if (valid && k < nm) {
        const V4 e0 = lm[k][0], e1 = lm[k][1], e2 = lm[k][2], e3 = lm[k][3];
        m2p_mixed(tx - (R)e0.x, ty - (R)e0.y, tz - (R)e0.z, e1, e2, e3, (R)e0.w, eps2, acc.p);
      }
    }
    fold_mixed(acc);
  };
  // self term: the reference's rule (a zero separation from the leaf's
  // particle) for sinks, the particle index for the grown particles
  auto p2p_self = [&](uint32_t k) -> bool {
    if constexpr (SINK) {
      const uint32_t j = lpi[k];
      return sx == a.x[j] && sy == a.y[j] && sz == a.z[j];
    } else {
      return lpi[k] == tid;   // mirror-box entries hold ~0u
    }
  };
  // Two entries per pass as for M2P (same per-lane order of terms).
  auto flush_p2p = [&]() {
    uint32_t kk = 0;
    const uint32_t n2 = np >= 2 * S ? np - 2 * S + 1 : 0;
    if (valid) {
      for (; kk < n2; kk += 2 * S) {
        const uint32_t k = kk + s, k2 = k + S;
        const V4 e = lp[k], f = lp[k2];
        const bool self1 = p2p_self(k), self2 = p2p_self(k2);
        p2p<R>(tx - (R)e.x, ty - (R)e.y, tz - (R)e.z, (R)e.w, eps2, self1, acc.p);
        p2p<R>(tx - (R)f.x, ty - (R)f.y, tz - (R)f.z, (R)f.w, eps2, self2, acc.p);
      }
    }
    kk = n2 ? ((n2 - 1) / (2 * S) + 1) * 2 * S : 0;
    for (; kk < np; kk += S) {
      const uint32_t k = kk + s;
      if (valid && k < np) {
        const V4 e = lp[k];
        p2p<R>(tx - (R)e.x, ty - (R)e.y, tz - (R)e.z, (R)e.w, eps2, p2p_self(k), acc.p);
      }
    }
    fold_mixed(acc);
  };

  const int nbox = PER ? a.nbox : 1;
  for (int box = 0; box < nbox && !overflow; ++box) {
  double vx = 0.0, vy = 0.0, vz = 0.0;
  if constexpr (PER) { vx = a.vbox[3 * box]; vy = a.vbox[3 * box + 1]; vz = a.vbox[3 * box + 2]; }
  const bool central = !PER || (vx == 0.0 && vy == 0.0 && vz == 0.0);
  // targets of this box: x - vbox; group box likewise (rounding is monotone,
  // so the shifted extremes are the extremes of the shifted targets)
  sx = xt - vx; sy = yt - vy; sz = zt - vz;
  const Span bx = span_of(lox - vx, hix - vx), by = span_of(loy - vy, hiy - vy),
             bz = span_of(loz - vz, hiz - vz);
  const double fox = ox - vx, foy = oy - vy, foz = oz - vz;   // node frame
  if (lane == 0) stack[0] = root | kTwigBit;
  sp = 1;
  wave_order();
  while (sp > 0) {
    // Up to min(64, LM) nodes are read from the top of the stack (so one
    // step's appends always fit an emptied list, positions nm + rank < LM);
    // after the box test only the longest run of them whose pushes fit
    // below the cap is visited, the rest stay on the stack.
    constexpr uint32_t kPop = (uint32_t)(LM < kWave ? LM : kWave);
    static_assert(kListP >= kWave, "P2P list must hold one full step");
    const uint32_t m = sp < kPop ? sp : kPop;
    if (nm + m > (uint32_t)LM) { wave_order(); flush_m2p(); nm = 0; }
    if (np + m > (uint32_t)kListP) { wave_order(); flush_p2p(); np = 0; }
    const bool has = (uint32_t)lane < m;
    const uint32_t entry = has ? stack[sp - 1 - lane] : 0u;
    const uint32_t node = entry & ~kTwigBit;
    const bool twig_entry = (entry & kTwigBit) != 0u;
    wave_order();
    ++nsteps;

    // All of a node's data is requested at once, before any decision, so a
    // traversal step waits for one memory round trip.  A twig also brings
    // its walk moments and its children's kinds; a leaf has neither.
    NodeGeom gm = {0.0, 0.0, 0.0, 0.0};
    NodeLink lk = {0u, 0u, 0u, 0u};
    V4 w0, w1, w2;
    uint32_t kids = 0u;
    if (has) {
      gm = a.geom[node];
      lk = a.link[node];
    }
    if (has && twig_entry) {
      kids = a.kidtwig[node];
      const V4* src = reinterpret_cast<const V4*>(&a.wm32[node]);
      w0 = src[0]; w1 = src[1]; w2 = src[2];
    }
    // Decide from the group's bounding box when possible (margins cover
    // every rounding of the exact per-target test below).
    bool acc_ok = false, rej = false;
    uint32_t macc = 0;
    if (has && lk.nchild != 0u) {
#pragma clang fp contract(fast)
      const double dx = fabs(gm.cx - bx.c), dy = fabs(gm.cy - by.c), dz = fabs(gm.cz - bz.c);
      const double ex = fmax(dx - bx.h, 0.0), ey = fmax(dy - by.h, 0.0), ez = fmax(dz - bz.h, 0.0);
      const double fx = dx + bx.h, fy = dy + by.h, fz = dz + bz.h;
      const double dmin2 = ex * ex + ey * ey + ez * ez;
      const double dmax2 = fx * fx + fy * fy + fz * fz;
      acc_ok = t_acc * dmin2 > gm.b2;
      rej = !acc_ok && t_rej * dmax2 <= gm.b2;
      macc = acc_ok ? cnt : (rej ? 1u : 0u);
    }
    // Visit lanes 0 .. k-1 for the largest k whose step leaves at most kCap
    // entries: sp - k + (children of lanes < k, counted for every twig the
    // box did not accept) <= kCap.  k >= 1 always, so the stack passes the
    // cap only by the one-node steps of a depth-first descent (within
    // kStackSlack), and k is never below the worst-case count
    // (kCap - sp) / 7.  Nodes k .. m-1 stay on the stack unvisited: none of
    // their decisions is counted.
    // While the worst case fits (7 net pushes per node), all m are visited
    // without the search.
    uint32_t k = m;
    if ((int)(7u * m) > (int)kCap - (int)sp) {
      const uint32_t pmax = (has && lk.nchild != 0u && !acc_ok) ? lk.nchild : 0u;
      uint32_t ptot;
      const uint32_t pex = wave_exclusive_scan16(pmax, &ptot);
      const bool fits = has && (int)(pex + pmax) - (lane + 1) <= (int)kCap - (int)sp;
      const unsigned long long fm = __ballot(fits);
      k = fm ? 64u - (uint32_t)__clzll((long long)fm) : 1u;
    }
    const bool keep = (uint32_t)lane < k;
    sp -= k;
    const bool leaf = keep && lk.nchild == 0u;
    const bool twig = keep && lk.nchild != 0u;
    // Undecided nodes: exact per-target test.  Every slice holds all the
    // targets, so slice s tests the s-th undecided node of the batch and S
    // nodes are settled per pass.  The nodes' centres and b^2 are staged in
    // the free tail of the M2P list (entries nm .. nm + m - 1, which this
    // step's appends overwrite only after the tests), so each slice reads
    // its node with one broadcast load per pass.
    const bool amb_me = twig && !acc_ok && !rej;
    const unsigned long long amb = __ballot(amb_me);
    const uint32_t na = (uint32_t)popc64(amb);
    namb += na;
    if (na) {
      const uint32_t my_rank = mask_rank(amb);
      if (amb_me) {
        double2* st = reinterpret_cast<double2*>(&lm[nm + my_rank][0]);
        st[0] = make_double2(gm.cx, gm.cy);
        st[1] = make_double2(gm.cz, gm.b2);
      }
      wave_order();
      for (uint32_t base = 0; base < na; base += S) {
        const uint32_t r = base + s;
        const bool active = valid && r < na;
        double2 c0 = make_double2(0.0, 0.0), c1 = c0;
        if (active) {
          const double2* st = reinterpret_cast<const double2*>(&lm[nm + r][0]);
          c0 = st[0];
          c1 = st[1];
        }
        const bool fail = active && mac_fails(sx, sy, sz, c0.x, c0.y, c1.x, c1.y, theta2);
        const unsigned long long ball = __ballot(fail);
        if (amb_me && my_rank >= base && my_rank < base + S) {
          const uint32_t rr = my_rank - base;
          const unsigned long long fm =
              (ball >> (rr * T)) & (T == 64 ? ~0ull : ((1ull << T) - 1ull));
          if (fm == 0ull) { acc_ok = true; macc = cnt; }
          else { rej = true; macc = (uint32_t)__ffsll((long long)fm); }
        }
      }
      wave_order();
    }
    mac_lane += twig ? macc : 0u;

    const bool take_m = twig && acc_ok;
    const unsigned long long am = __ballot(take_m);
    const unsigned long long pm = __ballot(leaf);
    if (take_m) {
      const uint32_t pos = nm + mask_rank(am);
      // w0 = {q, px, py, pz}, w1 = {2qx, 2qy, 2qz, xy}, w2 = {yz, zx, tr, -}
      const V4 e0 = V4{(float)(gm.cx - fox), (float)(gm.cy - foy), (float)(gm.cz - foz), w0.x};
      V4 e1, e2, e3;
      e1.x = w0.y; e1.y = w0.z; e1.z = w0.w; e1.w = w1.x;
      e2.x = w1.y; e2.y = w1.z; e2.z = w1.w; e2.w = w2.x;
      e3.x = w2.y; e3.y = w2.z; e3.z = 0; e3.w = 0;
      lm[pos][0] = e0; lm[pos][1] = e1; lm[pos][2] = e2; lm[pos][3] = e3;
    }
    if (leaf) {
      const uint32_t pos = np + mask_rank(pm);
      const V4 e = V4{(float)(gm.cx - fox), (float)(gm.cy - foy), (float)(gm.cz - foz), (float)gm.b2};
      lp[pos] = e;
      lpi[pos] = (SINK || central) ? lk.first : ~0u;
    }
    const uint32_t nma = (uint32_t)popc64(am), npa = (uint32_t)popc64(pm);
    nm += nma; np += npa; cnt_m2p += nma; cnt_p2p += npa;

    const uint32_t nc = (twig && !acc_ok) ? lk.nchild : 0u;   // at most 8
    uint32_t tot;
    const uint32_t excl = wave_exclusive_scan16(nc, &tot);
    if (sp + tot > (uint32_t)(kCap + kStackSlack)) { overflow = true; break; }
    for (uint32_t k = 0; k < nc; ++k)
      stack[sp + excl + k] = (lk.first + k) | (((kids >> k) & 1u) ? kTwigBit : 0u);
    sp += tot;
    wave_order();
  }
  if constexpr (PER && SINK) {   // next box shifts the targets
    wave_order();
    if (nm) flush_m2p();
    if (np) flush_p2p();
    nm = 0; np = 0;
  }
  }   // boxes
  wave_order();
  if (nm) flush_m2p();
  if (np) flush_p2p();

  // Combine the slices in FP64, in order (target t lives in lanes t, t+T, ...):
  // many slices through the list's LDS, one lane per sum, few by shuffles.
  double out[4];
  const bool by_lane = S > 4u;   // then 4 T sums fit the wave
#pragma unroll
  for (int k = 0; k < 4; ++k) out[k] = (double)acc.s[k] - (double)acc.c[k];
  if (by_lane) {
    double* sums = reinterpret_cast<double*>(&lm[0][0]);   // 4 x 64: 2 KB of the list
    static_assert(sizeof(V4) * 4 * LM >= 4 * kWave * sizeof(double), "the list holds the sums");
    wave_order();
#pragma unroll
    for (int k = 0; k < 4; ++k) sums[k * kWave + lane] = out[k];
    wave_order();
    const uint32_t k = s < 4u ? s : 3u;   // lane k T + t: component k of target t
    double v = sums[k * kWave + t];
    for (uint32_t o = 1; o < S; ++o) v += sums[k * kWave + t + o * T];
    double* dst = k == 0u ? a.ex : k == 1u ? a.ey : k == 2u ? a.ez : a.pot;
    if (s < 4u) dst[tid] = v * a.sign;
    wave_order();
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double v0 = out[k];
      double v = v0;
      for (uint32_t o = 1; o < S; ++o) v += __shfl(v0, (int)(t + o * T));
      out[k] = v * a.sign;
    }
  }
  if (overflow) {
    if (lane == 0) atomicOr(&a.sc->flags, kFlagStackOverflow);
  }
  if (s == 0 && valid) {
    if (!by_lane) {
      a.ex[tid] = out[0];
      a.ey[tid] = out[1];
      a.ez[tid] = out[2];
      a.pot[tid] = out[3];
    }
    a.work[tid] = (SINK ? 0.0 : 1.0) + (double)(cnt_p2p + cnt_m2p);
    a.np2p[tid] = cnt_p2p;
    a.nm2p[tid] = cnt_m2p;
  }
  const unsigned long long nmac = SINK ? 0ull : wave_sum((unsigned long long)mac_lane);
  if (!SINK && lane == 0) {   // per-group record, summed by walk_stats_kernel
    uint4* gs = reinterpret_cast<uint4*>(a.gstat + 8 * (size_t)g);
    gs[0] = make_uint4((uint32_t)nmac, cnt_p2p, cnt_m2p, namb);
    gs[1] = make_uint4(nsteps, cnt, 0u, 0u);
  }
  wave_order();
}

// LM: capacity of the M2P list staged in LDS (the list tile); the P2P list
// holds kListP entries.  The default tiles (LM * sizeof(R) = 256 bytes per
// float component: FP32 64, FP64 32) leave LDS for four one-wave workgroups
// per SIMD; the register budget is held to the same four (at most 128 VGPRs).
// The larger tiles are LDS-limited to three.
// NT: targets per lane.  Two halve the LDS reads per pair and fill groups of
// 17 to 64 targets better (1,000,003 particles, G = 64: 1.40 -> 1.19 ms), one
// fills groups up to 16 better (G = 16 unpacked: 1.76 against 1.64 ms) and
// then takes two list entries per pass; FP64 has no registers for two.
template <typename R, int LM, int NT, bool PER, bool SINK>
__global__ __launch_bounds__(kWave)
__attribute__((amdgpu_waves_per_eu(LM * sizeof(R) <= 256 ? 4 : 3)))
void walk_kernel(WalkArgs a) {
  using P = Prec<R>;
  using V4 = typename P::V4;
  // A step pops at most (cap - sp) / 7 nodes (each may push 8 children), so a
  // deep stack means small steps; wide near fields (small theta) fill it.
  // Four one-wave workgroups per SIMD leave 10 KB of LDS each: FP32 lists
  // take 5.4 KB, FP64 lists 6.4 KB, so only FP32 has room for the larger cap.
  constexpr int kCap = sizeof(R) == 4 ? kStackCap32 : kStackCap;
  __shared__ uint32_t stack[kCap + kStackSlack];
  __shared__ V4 lm[LM][4];
  __shared__ V4 lp[kListP];
  __shared__ uint32_t lpi[kListP];
  __shared__ uint2 opened[kWave];   // {first child, child count | kinds << 8} of a step's opened nodes

  const int lane = threadIdx.x;
  constexpr bool kPair = sizeof(R) == 4 && NT == 1;
  const R eps2 = (R)a.eps2;
  const double theta2 = a.theta2;
  const double t_acc = theta2 * (1.0 - 1e-12), t_rej = theta2 * (1.0 + 1e-12);
  const uint32_t ngroups = SINK ? a.nsink_groups : a.sc->ngroups;
  if (!SINK && blockIdx.x == 0 && lane == 0) {   // the sums of walk_stats_kernel
    a.sc->interactions = 0;
    a.sc->mac_evals = 0;
    a.sc->p2p = 0;
    a.sc->m2p = 0;
    a.sc->amb_nodes = 0;
    a.sc->walk_steps = 0;
    a.clock[kClockWalk] = wall_clock64();
  }
  const double* __restrict__ TX = SINK ? a.tx : a.x;
  const double* __restrict__ TY = SINK ? a.ty : a.y;
  const double* __restrict__ TZ = SINK ? a.tz : a.z;

  GroupQueue work;
  work.init((uint32_t)a.nqueue);
  for (;;) {
    uint32_t gg = ngroups;
    if (lane == 0) gg = work.next(a.queue, ngroups);
    const uint32_t g = uniform(gg);
    if (g >= ngroups) break;

    // Every lane holds NT of the group's T targets, u and (NT = 2) u + W with
    // W = ceil(T / NT), and lanes s*W .. s*W+W-1 form slice s (s < S = 64/W).
    // A lane without a second target repeats its first; the 64 - S*W lanes
    // past the slices repeat the last slice's entries; both are left out of
    // the sums.
    uint32_t a0, cnt;
    if (!SINK || a.gfirst) { a0 = uniform(a.gfirst[g]); cnt = uniform(a.gcount[g]); }
    else { a0 = g; cnt = 1u; }
    const DevBox& sbox = a.boxes[(!SINK && a.sys) ? a.sys[a0] : 0u];   // the group's system
    if constexpr (sizeof(R) == 4) {
      if (uniform(sbox.mixed)) {
        walk_group_mixed<LM, PER, SINK>(a, g, a0, cnt, stack, lm, lp, lpi);
        continue;
      }
    }
    const uint32_t T = cnt;
    const uint32_t W = (T + (uint32_t)NT - 1u) / (uint32_t)NT;
    const bool two = NT == 2 && T > 1u;
    const uint32_t S = uniform(kWave / W);
    const uint32_t divS = uniform((4096u + S - 1u) / S);   // r / S = (r * divS) >> 12 for r < 64
    const uint32_t s = (uint32_t)lane / W;
    const uint32_t u = (uint32_t)lane - s * W;
    const uint32_t se = s < S ? s : S - 1u;   // the slice whose entries this lane evaluates
    bool has1 = false;
    uint32_t tid[NT];
    double xt[NT], yt[NT], zt[NT];
    tid[0] = a0 + u;
    if constexpr (NT == 2) { has1 = u + W < T; tid[1] = has1 ? tid[0] + W : tid[0]; }
#pragma unroll
    for (int j = 0; j < NT; ++j) { xt[j] = TX[tid[j]]; yt[j] = TY[tid[j]]; zt[j] = TZ[tid[j]]; }
    const double ox = uniform(xt[0]), oy = uniform(yt[0]), oz = uniform(zt[0]);   // lane 0: target a0
    const double lox = uniform_min(fmin(xt[0], xt[NT - 1])), loy = uniform_min(fmin(yt[0], yt[NT - 1])),
                 loz = uniform_min(fmin(zt[0], zt[NT - 1]));
    const double hix = -uniform_min(-fmax(xt[0], xt[NT - 1])), hiy = -uniform_min(-fmax(yt[0], yt[NT - 1])),
                 hiz = -uniform_min(-fmax(zt[0], zt[NT - 1]));
    // target positions in the kernel's frame (FP64: set per box below)
    R tx[NT], ty[NT], tz[NT];
    Acc<R> acc[NT];
    double sx[NT], sy[NT], sz[NT];    // targets of the current box: x - vbox
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      tx[j] = (R)(xt[j] - ox); ty[j] = (R)(yt[j] - oy); tz[j] = (R)(zt[j] - oz);
      sx[j] = xt[j]; sy[j] = yt[j]; sz[j] = zt[j];
#pragma unroll
      for (int k = 0; k < 4; ++k) { acc[j].s[k] = 0.0; acc[j].p[k] = R(0); }
    }

    // Kept remainders (fewer than S entries) shorten the next steps' lists;
    // above 16 slices, where a list is a few passes at most, lists are emptied.
    const bool keep_rest = S <= 16u;
    const bool dipoles = uniform(sbox.qsign) == 3u;
    uint32_t sp = 0, nm = 0, np = 0, cnt_p2p = 0, cnt_m2p = 0, namb = 0, nsteps = 0;
    uint32_t mac_lane = 0;   // this lane's MAC evaluations, summed over the wave at the end
    bool overflow = false;
    const uint32_t root = (!SINK && a.sys) ? uniform(a.sysroot[a.sys[a0]]) : 0u;   // the group's own root

    // Batches: entry k goes to slice k mod S; the passes in which every slice
    // has an entry run without a mask, the last one with it.
    auto m2p_pair = [&](auto dip, const V4& e0, const V4& e1, const V4& e2, const V4& e3) __attribute__((always_inline)) {
      constexpr bool D = decltype(dip)::value;
      m2p<R, D>(tx[0] - e0.x, ty[0] - e0.y, tz[0] - e0.z, e0.w, e1, e2, e3.x, e3.y, eps2, acc[0].p);
      if constexpr (NT == 2)
        if (two)
          m2p<R, D>(tx[1] - e0.x, ty[1] - e0.y, tz[1] - e0.z, e0.w, e1, e2, e3.x, e3.y, eps2,
                    acc[1].p);
    };
    auto m2p_entry = [&](auto dip, uint32_t k) __attribute__((always_inline)) {
      const V4 e0 = lm[k][0], e1 = lm[k][1], e2 = lm[k][2], e3 = lm[k][3];
      m2p_pair(dip, e0, e1, e2, e3);
    };
    auto m2p_list = [&](auto dip, uint32_t r) __attribute__((always_inline)) {
      uint32_t k = r + se, kk = r + S;
      if constexpr (kPair) {
        for (; kk + S <= nm; kk += 2 * S, k += 2 * S) {
          const V4 e0 = lm[k][0], e1 = lm[k][1], e2 = lm[k][2], e3 = lm[k][3];
          const uint32_t k2 = k + S;
          const V4 f0 = lm[k2][0], f1 = lm[k2][1], f2 = lm[k2][2], f3 = lm[k2][3];
          m2p_pair(dip, e0, e1, e2, e3);
          m2p_pair(dip, f0, f1, f2, f3);
        }
      }
      for (; kk <= nm; kk += S, k += S) m2p_entry(dip, k);
      if (k < nm) m2p_entry(dip, k);
    };
    auto fold_all = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < NT; ++j) fold(acc[j]);
    };
    // Leaves the first nm mod S entries in the list when they still leave
    // room for `more` (so every pass is a full one), else empties it.
    auto flush_m2p = [&](uint32_t more) __attribute__((always_inline)) {
      const uint32_t rest = nm - ((nm * divS) >> 12) * S;
      const uint32_t r = keep_rest && rest + more <= (uint32_t)LM ? rest : 0u;
      if (dipoles) m2p_list(std::true_type{}, r);
      else m2p_list(std::false_type{}, r);
      fold_all();
      nm = r;
    };
    // self term: the reference's rule (a zero separation from the leaf's
    // particle) for sinks, the particle index for the grown particles
    auto p2p_entry = [&](uint32_t k) __attribute__((always_inline)) {
      const V4 e = lp[k];
      const uint32_t i = lpi[k];   // mirror-box entries hold ~0u
      bool self[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if constexpr (SINK) self[j] = sx[j] == a.x[i] && sy[j] == a.y[i] && sz[j] == a.z[i];
        else self[j] = i == tid[j];
      }
      p2p<R>(tx[0] - e.x, ty[0] - e.y, tz[0] - e.z, e.w, eps2, self[0], acc[0].p);
      if constexpr (NT == 2)
        if (two) p2p<R>(tx[1] - e.x, ty[1] - e.y, tz[1] - e.z, e.w, eps2, self[1], acc[1].p);
    };
    auto flush_p2p = [&](uint32_t more) __attribute__((always_inline)) {
      const uint32_t rest = np - ((np * divS) >> 12) * S;
      const uint32_t r = keep_rest && rest + more <= (uint32_t)kListP ? rest : 0u;
      uint32_t k = r + se, kk = r + S;
      for (; kk <= np; kk += S, k += S) p2p_entry(k);
      if (k < np) p2p_entry(k);
      fold_all();
      np = r;
    };

    const int nbox = PER ? a.nbox : 1;
    for (int box = 0; box < nbox && !overflow; ++box) {
    double vx = 0.0, vy = 0.0, vz = 0.0;
    if constexpr (PER) { vx = a.vbox[3 * box]; vy = a.vbox[3 * box + 1]; vz = a.vbox[3 * box + 2]; }
    const bool central = !PER || (vx == 0.0 && vy == 0.0 && vz == 0.0);
    // targets of this box: x - vbox; group box likewise (rounding is monotone,
    // so the shifted extremes are the extremes of the shifted targets)
    if constexpr (PER) {
#pragma unroll
      for (int j = 0; j < NT; ++j) { sx[j] = xt[j] - vx; sy[j] = yt[j] - vy; sz[j] = zt[j] - vz; }
    }
    const Span bx = span_of(lox - vx, hix - vx), by = span_of(loy - vy, hiy - vy),
               bz = span_of(loz - vz, hiz - vz);
    const double fox = PER ? uniform(ox - vx) : ox, foy = PER ? uniform(oy - vy) : oy,
                 foz = PER ? uniform(oz - vz) : oz;   // FP32 node frame
    if constexpr (sizeof(R) == 8) {
#pragma unroll
      for (int j = 0; j < NT; ++j) { tx[j] = sx[j]; ty[j] = sy[j]; tz[j] = sz[j]; }
    }
    if (lane == 0) stack[0] = root | kTwigBit;
    sp = 1;
    wave_order();
    while (sp > 0) {
      // Up to min(64, LM) nodes are read from the top of the stack (so one
      // step's appends always fit an emptied list, positions nm + rank < LM);
      // after the box test only the longest run of them whose pushes fit
      // below the cap is visited, the rest stay on the stack.
      constexpr uint32_t kPop = (uint32_t)(LM < kWave ? LM : kWave);
      static_assert(kListP >= kWave, "P2P list must hold one full step");
      const uint32_t m = sp < kPop ? sp : kPop;
      const bool has = (uint32_t)lane < m;
      const uint32_t entry = has ? stack[sp - 1 - lane] : 0u;
      const uint32_t node = entry & ~kTwigBit;
      const bool twig_entry = (entry & kTwigBit) != 0u;
      // at most one append per twig and one per leaf (a root counts as a twig
      // and may be a leaf)
      const uint32_t nt = (uint32_t)popc64(__ballot(twig_entry)), nl = m - nt + 1u;
      if (nm + nt > (uint32_t)LM) flush_m2p(nt);
      if (np + nl > (uint32_t)kListP) flush_p2p(nl);
      wave_order();
      ++nsteps;

      // All of a node's data is requested at once, before any decision, so a
      // traversal step waits for one memory round trip.  A twig also brings
      // its walk moments and its children's kinds; a leaf has neither.
      NodeGeom gm = {0.0, 0.0, 0.0, 0.0};
      NodeLink lk = {0u, 0u, 0u, 0u};
      V4 w0 = {}, w1 = {}, w2 = {};
      uint32_t kids = 0u;
      if (has) {
        gm = a.geom[node];
        lk = a.link[node];
      }
      if (has && twig_entry) {
        kids = a.kidtwig[node];
        const V4* src;
        if constexpr (sizeof(R) == 4) src = reinterpret_cast<const V4*>(&a.wm32[node]);
        else src = reinterpret_cast<const V4*>(&a.wm64[node]);
        w0 = src[0]; w1 = src[1]; w2 = src[2];
      }
      // Decide from the group's bounding box when possible.  The margins
      // cover every rounding here and in the exact per-target test below: a
      // distance to the box is either at least the half width, and then has
      // a relative error of a few ulps, or its error is below the part that
      // was added to the half width.
      bool acc_ok = false, rej = false;
      uint32_t macc = 0;
      if (has && lk.nchild != 0u) {
#pragma clang fp contract(fast)
        const double dx = fabs(gm.cx - bx.c), dy = fabs(gm.cy - by.c), dz = fabs(gm.cz - bz.c);
        const double ex = fmax(dx - bx.h, 0.0), ey = fmax(dy - by.h, 0.0), ez = fmax(dz - bz.h, 0.0);
        const double fx = dx + bx.h, fy = dy + by.h, fz = dz + bz.h;
        const double dmin2 = ex * ex + ey * ey + ez * ez;
        const double dmax2 = fx * fx + fy * fy + fz * fz;
        acc_ok = t_acc * dmin2 > gm.b2;
        rej = !acc_ok && t_rej * dmax2 <= gm.b2;
        macc = acc_ok ? cnt : (rej ? 1u : 0u);
      }
      // Visit lanes 0 .. k-1 for the largest k whose step leaves at most kCap
      // entries: sp - k + (children of lanes < k, counted for every twig the
      // box did not accept) <= kCap.  k >= 1 always, so the stack passes the
      // cap only by the one-node steps of a depth-first descent (within
      // kStackSlack), and k is never below the worst-case count
      // (kCap - sp) / 7.  Nodes k .. m-1 stay on the stack unvisited: none of
      // their decisions is counted.
      // While the worst case fits (7 net pushes per node), all m are visited
      // without the search.
      uint32_t k = m;
      if ((int)(7u * m) > (int)kCap - (int)sp) {
        const uint32_t pmax = (has && lk.nchild != 0u && !acc_ok) ? lk.nchild : 0u;
        uint32_t ptot;
        const uint32_t pex = wave_exclusive_scan16(pmax, &ptot);
        const bool fits = has && (int)(pex + pmax) - (lane + 1) <= (int)kCap - (int)sp;
        const unsigned long long fm = __ballot(fits);
        k = fm ? 64u - (uint32_t)__clzll((long long)fm) : 1u;
      }
      const bool keep = (uint32_t)lane < k;
      sp -= k;
      const bool leaf = keep && lk.nchild == 0u;
      const bool twig = keep && lk.nchild != 0u;
      // Undecided nodes: exact per-target test.  Every slice holds all the
      // targets, so slice s tests the s-th undecided node of the batch and S
      // nodes are settled per pass.  The nodes' centres and b^2 are staged in
      // the free tail of the M2P list (entries nm .. nm + m - 1, which this
      // step's appends overwrite only after the tests), so each slice reads
      // its node with one broadcast load per pass.  Pass p's failure ballots
      // are kept in lane p; afterwards each undecided node's lane fetches the
      // ballots of its pass and cuts out its slice.
      const bool amb_me = twig && !acc_ok && !rej;
      const unsigned long long amb = __ballot(amb_me);
      if (amb) {
        const uint32_t na = (uint32_t)popc64(amb);
        namb += na;
        const uint32_t my_rank = mask_rank(amb);
        if (amb_me) {
          double2* st = reinterpret_cast<double2*>(&lm[nm + my_rank][0]);
          st[0] = make_double2(gm.cx, gm.cy);
          st[1] = make_double2(gm.cz, gm.b2);
        }
        wave_order();
        int blo[NT], bhi[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) { blo[j] = 0; bhi[j] = 0; }
        uint32_t pass = 0;
        for (uint32_t base = 0; base < na; base += S, ++pass) {
          // slices past the last node repeat it
          const uint32_t r = base + s < na ? base + s : na - 1u;
          const double2* st = reinterpret_cast<const double2*>(&lm[nm + r][0]);
          const double2 c0 = st[0], c1 = st[1];
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            const bool f = mac_fails(sx[j], sy[j], sz[j], c0.x, c0.y, c1.x, c1.y, theta2);
            const unsigned long long ball = __ballot(f);
            blo[j] = (uint32_t)lane == pass ? (int)(uint32_t)ball : blo[j];
            bhi[j] = (uint32_t)lane == pass ? (int)(uint32_t)(ball >> 32) : bhi[j];
          }
        }
        const uint32_t mp = (my_rank * divS) >> 12;
        const uint32_t sh = (my_rank - mp * S) * W;
        unsigned long long f[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(mp << 2), blo[j]);
          const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(mp << 2), bhi[j]);
          // the node's W bits at the top, the others shifted out
          f[j] = ((((unsigned long long)hi << 32) | lo) >> sh) << (64u - W);
        }
        if (amb_me) {
          bool any = f[0] != 0ull;
          if constexpr (NT == 2) any = any || f[1] != 0ull;
          if (!any) { acc_ok = true; macc = cnt; }
          else {   // the first failing target, in order
            rej = true;
            uint32_t first = (uint32_t)__ffsll((long long)f[0]);
            if constexpr (NT == 2) first = f[0] ? first : W + (uint32_t)__ffsll((long long)f[1]);
            macc = first - (64u - W);
          }
        }
        wave_order();
      }
      mac_lane += twig ? macc : 0u;

      const bool take_m = twig && acc_ok;
      const unsigned long long am = __ballot(take_m);
      const unsigned long long pm = __ballot(leaf);
      if (take_m) {
        const uint32_t pos = nm + mask_rank(am);
        // the record is the entry's words in order, with q behind pz
        V4 e0;
        if constexpr (sizeof(R) == 4)
          e0 = V4{(float)(gm.cx - fox), (float)(gm.cy - foy), (float)(gm.cz - foz), w2.z};
        else
          e0 = V4{gm.cx, gm.cy, gm.cz, w2.z};
        lm[pos][0] = e0; lm[pos][1] = w0; lm[pos][2] = w1; lm[pos][3] = w2;
      }
      if (leaf) {
        const uint32_t pos = np + mask_rank(pm);
        V4 e;
        if constexpr (sizeof(R) == 4) {
          e = V4{(float)(gm.cx - fox), (float)(gm.cy - foy), (float)(gm.cz - foz), (float)gm.b2};
        } else {
          e = V4{gm.cx, gm.cy, gm.cz, gm.b2};
        }
        lp[pos] = e;
        lpi[pos] = (SINK || central) ? lk.first : ~0u;
      }
      const uint32_t nma = (uint32_t)popc64(am), npa = (uint32_t)popc64(pm);
      nm += nma; np += npa; cnt_m2p += nma; cnt_p2p += npa;

      // Children of the opened nodes, eight lanes per node: the nodes' child
      // runs are compacted in LDS, lane 8 j + c takes child c of the j-th,
      // and one ballot gives every child its place on the stack.
      const bool open = twig && !acc_ok;
      const unsigned long long om = __ballot(open);
      if (open) opened[mask_rank(om)] = make_uint2(lk.first, lk.nchild | (kids << 8));
      wave_order();
      const int no = (int)popc64(om);
      for (int o = 0; o < no; o += 8) {
        const int j = o + (lane >> 3);
        const uint32_t c = (uint32_t)lane & 7u;
        const uint2 rec = opened[j & (kWave - 1)];
        const bool child = j < no && c < (rec.y & 0xFFu);
        const unsigned long long cm = __ballot(child);
        const uint32_t nc = (uint32_t)popc64(cm);
        if (sp + nc > (uint32_t)(kCap + kStackSlack)) { overflow = true; break; }
        if (child)
          stack[sp + mask_rank(cm)] = (rec.x + c) | (((rec.y >> (8u + c)) & 1u) << 31);
        sp += nc;
      }
      if (overflow) break;
      wave_order();
    }
    if constexpr (PER && (sizeof(R) == 8 || SINK)) {   // next box shifts the targets
      if (nm) flush_m2p(LM + 1u);
      if (np) flush_p2p(kListP + 1u);
      wave_order();
    }
    }   // boxes
    if (nm) flush_m2p(LM + 1u);
    if (np) flush_p2p(kListP + 1u);
    wave_order();

    // combine the slices in FP64, halving their number per step (slice s adds
    // slice s + ceil(n/2)): a fixed order
    for (uint32_t rem = S; rem > 1;) {
      const uint32_t h = (rem + 1u) >> 1;
      const int src = (lane + (int)(h * W)) & (kWave - 1);
      const bool add = s + h < rem;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const double v = __shfl(acc[j].s[k], src);
          acc[j].s[k] += add ? v : 0.0;
        }
      }
      rem = h;
    }
    if (overflow) {
      if (lane == 0) atomicOr(&a.sc->flags, kFlagStackOverflow);
    }
    const double wk = (SINK ? 0.0 : 1.0) + (double)(cnt_p2p + cnt_m2p);
    if (s == 0) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (j == 0 || has1) {
          const uint32_t t = tid[j];
          a.ex[t] = acc[j].s[0] * a.sign;
          a.ey[t] = acc[j].s[1] * a.sign;
          a.ez[t] = acc[j].s[2] * a.sign;
          a.pot[t] = acc[j].s[3] * a.sign;
          a.work[t] = wk;
          a.np2p[t] = cnt_p2p;
          a.nm2p[t] = cnt_m2p;
        }
      }
    }
    const unsigned long long nmac = SINK ? 0ull : wave_sum((unsigned long long)mac_lane);
    if (!SINK && lane == 0) {   // per-group record, summed by walk_stats_kernel
      uint4* gs = reinterpret_cast<uint4*>(a.gstat + 8 * (size_t)g);
      gs[0] = make_uint4((uint32_t)nmac, cnt_p2p, cnt_m2p, namb);
      gs[1] = make_uint4(nsteps, cnt, 0u, 0u);
    }
  }
}

// Sums the per-group records into the device scalars (walk statistics of
// tree_walk_statistics, module_tree_walk_simple.f90:63-115).
// Also leaves the work-queue heads at zero for the next walk; the walk itself
// clears the sums, which saves a launch before it.
__global__ __launch_bounds__(256) void walk_stats_kernel(const uint32_t* __restrict__ gstat,
                                                        DevScalars* __restrict__ sc,
                                                        uint32_t* __restrict__ queue,
                                                        unsigned long long* __restrict__ clock) {
  if (blockIdx.x == 0 && threadIdx.x == 0) clock[kClockWalked] = wall_clock64();   // walk over
  const int64_t ng = sc->ngroups;
  if (blockIdx.x == 0 && threadIdx.x <= kMaxQueues) queue[kQueueStride * threadIdx.x] = 0;
  unsigned long long v[6] = {0, 0, 0, 0, 0, 0};
  for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < ng;
       g += (int64_t)gridDim.x * blockDim.x) {
    const uint4 r0 = reinterpret_cast<const uint4*>(gstat + 8 * g)[0];
    const uint4 r1 = reinterpret_cast<const uint4*>(gstat + 8 * g)[1];
    const unsigned long long c = r1.y;
    v[0] += c * (r0.y + r0.z);
    v[1] += r0.x;
    v[2] += c * r0.y;
    v[3] += c * r0.z;
    v[4] += r0.w;
    v[5] += r1.x;
  }
  __shared__ unsigned long long red[6][4];
  const int w = threadIdx.x / kWave;
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const unsigned long long s = wave_sum(v[k]);
    if (lane_id() == 0) red[k][w] = s;
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    const unsigned long long s = red[k][0] + red[k][1] + red[k][2] + red[k][3];
    if (s) {
      unsigned long long* dst[6] = {&sc->interactions, &sc->mac_evals, &sc->p2p, &sc->m2p,
                                    &sc->amb_nodes, &sc->walk_steps};
      atomicAdd(dst[k], s);
    }
  }
}

__global__ __launch_bounds__(256) void zero_words_kernel(uint32_t* words, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) words[i] = 0;
}

__global__ void publish_kernel(const DevScalars* __restrict__ src, DevScalars* __restrict__ dst) {
  for (unsigned k = threadIdx.x; k < sizeof(DevScalars) / 4; k += blockDim.x)
    reinterpret_cast<uint32_t*>(dst)[k] = reinterpret_cast<const uint32_t*>(src)[k];
}

// FP64 direct sum (src/utils/module_directsum.f90:34-172): all sources
// against a list of targets, self excluded by index, reference P2P form; with
// nbox > 1 every source in every mirror box (the target shifted by -v), self
// only in the central box (module_directsum.f90:80-93).
//
// Bound by FP64 issue (about 20 instructions and one v_rsq_f64 per pair), so
// the work is cut until the chip is full: a block holds `span` targets in
// 256/span slices, slice s taking every (256/span)-th source of the block's
// range of sources (blockIdx.y of gridDim.y ranges), and every (range, slice)
// writes its own partial sums, which direct_reduce_kernel adds in a fixed
// order.  4096 targets against 1,048,576 sources: 4.2 ms; 178 ms with one
// block per 256 targets (16 blocks) and a square root and a division per pair.
__global__ __launch_bounds__(kDirectT) void direct_kernel(
    int64_t n, const double* __restrict__ x, const double* __restrict__ y,
    const double* __restrict__ z, const double* __restrict__ q, int64_t ntest,
    const int64_t* __restrict__ testidx, double eps2, double sign, double* __restrict__ ex,
    double* __restrict__ ey, double* __restrict__ ez, double* __restrict__ pot, int nbox,
    const double* __restrict__ vbox, int span, int64_t range, double* __restrict__ partial) {
#pragma clang fp contract(fast)
  __shared__ double4 src[kDirectT];
  const int slices = kDirectT / span;
  const int s = threadIdx.x / span, t = threadIdx.x - s * span;
  const int64_t j = (int64_t)blockIdx.x * span + t;
  const int64_t tj = j < ntest ? testidx[j] : -1;
  const double xt = tj >= 0 ? x[tj] : 0.0, yt = tj >= 0 ? y[tj] : 0.0, zt = tj >= 0 ? z[tj] : 0.0;
  const int64_t begin = (int64_t)blockIdx.y * range;
  const int64_t end = begin + range < n ? begin + range : n;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int64_t base = begin; base < end; base += kDirectT) {
    const int64_t i = base + threadIdx.x;
    __syncthreads();
    if (i < end) src[threadIdx.x] = make_double4(x[i], y[i], z[i], q[i]);
    __syncthreads();
    const int lim = (end - base) < kDirectT ? (int)(end - base) : kDirectT;
    const int self = tj >= base && tj < base + lim ? (int)(tj - base) : -1;
    double part[4] = {0.0, 0.0, 0.0, 0.0};
    auto term = [&](const double4& c, double px, double py, double pz, bool skip) {
      const double dx = px - c.x, dy = py - c.y, dz = pz - c.z;
      const double r2 = dx * dx + dy * dy + dz * dz + eps2;
      const double rd = rsqrt(skip ? 1.0 : r2);
      const double qr = (skip ? 0.0 : c.w) * rd;
      const double qr3 = qr * (rd * rd);
      part[3] += qr;
      part[0] += qr3 * dx;
      part[1] += qr3 * dy;
      part[2] += qr3 * dz;
    };
    for (int b = 0; b < nbox; ++b) {
      double vx = 0.0, vy = 0.0, vz = 0.0;
      if (vbox) { vx = vbox[3 * b]; vy = vbox[3 * b + 1]; vz = vbox[3 * b + 2]; }
      const double px = xt - vx, py = yt - vy, pz = zt - vz;
      // only a wave with a target among these sources tests for it
      const int me = vx == 0.0 && vy == 0.0 && vz == 0.0 ? self : -1;
      if (__ballot(me >= 0)) {
        for (int k = s; k < lim; k += slices) term(src[k], px, py, pz, k == me);
      } else {
#pragma unroll 2
        for (int k = s; k < lim; k += slices) term(src[k], px, py, pz, false);
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] += part[c];
  }
  if (j >= ntest) return;
  if (partial) {
    const int64_t np = (int64_t)gridDim.y * slices, p = (int64_t)blockIdx.y * slices + s;
#pragma unroll
    for (int c = 0; c < 4; ++c) partial[(c * ntest + j) * np + p] = acc[c];
  } else {
    ex[j] = sign * acc[0];
    ey[j] = sign * acc[1];
    ez[j] = sign * acc[2];
    pot[j] = sign * acc[3];
  }
}

// One wave per target and component: lane l adds partials l, l + 64, ..., then
// the wave's fixed-shape sum.
__global__ __launch_bounds__(kDirectT) void direct_reduce_kernel(
    int64_t ntest, int np, const double* __restrict__ partial, double sign, double* __restrict__ ex,
    double* __restrict__ ey, double* __restrict__ ez, double* __restrict__ pot) {
  const int64_t row = blockIdx.x * (int64_t)(kDirectT / kWave) + threadIdx.x / kWave;
  if (row >= 4 * ntest) return;
  double v = 0.0;
  for (int p = lane_id(); p < np; p += kWave) v += partial[row * np + p];
  v = wave_sum(v);
  if (lane_id() == 0) {
    const int c = (int)(row / ntest);
    double* out = c == 0 ? ex : c == 1 ? ey : c == 2 ? ez : pot;
    out[row - c * ntest] = sign * v;
  }
}

}  // namespace

// Persistent grid: every wavefront the device can hold for this instance
// (both targets-per-lane forms have the same LDS and register budget).
int walk_default_blocks(int precision, int list_tile) {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) {
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, dev) == hipSuccess) cus = p.multiProcessorCount;
  }
  int per = 0;
  hipError_t e;
  if (precision == kWalkFP64)
    e = list_tile == 64
            ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, walk_kernel<double, 64, 1, false, false>, kWave, 0)
            : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, walk_kernel<double, 32, 1, false, false>, kWave, 0);
  else
    e = list_tile == 128
            ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, walk_kernel<float, 128, 1, false, false>, kWave, 0)
            : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, walk_kernel<float, 64, 1, false, false>, kWave, 0);
  if (e != hipSuccess || per < 1) per = 8;
  return cus * per;
}

void launch_zero_words(hipStream_t s, uint32_t* words, int n) {
  zero_words_kernel<<<(n + 255) / 256, 256, 0, s>>>(words, n);
}

void launch_publish(hipStream_t s, const DevScalars* src, DevScalars* dst) {
  publish_kernel<<<1, 64, 0, s>>>(src, dst);
}

bool walk_list_tile_ok(int precision, int list_tile) {
  if (list_tile == 0) return true;
  return precision == kWalkFP64 ? (list_tile == 32 || list_tile == 64)
                                : (list_tile == 64 || list_tile == 128);
}

// default list tile (0): the smaller of each precision, whose lower LDS use
// lets one more wavefront per SIMD resident (measured faster on MI355X)
template <bool PER, bool SINK>
static void launch_walk_t(hipStream_t s, const WalkArgs& a, int precision, int blocks,
                          int list_tile, int max_group) {
  if (precision == kWalkFP64) {
    if (list_tile == 64)
      walk_kernel<double, 64, 1, PER, SINK><<<blocks, kWave, 0, s>>>(a);
    else
      walk_kernel<double, 32, 1, PER, SINK><<<blocks, kWave, 0, s>>>(a);
  } else if (max_group > 16) {   // two targets per lane, see walk_kernel
    if (list_tile == 128)
      walk_kernel<float, 128, 2, PER, SINK><<<blocks, kWave, 0, s>>>(a);
    else
      walk_kernel<float, 64, 2, PER, SINK><<<blocks, kWave, 0, s>>>(a);
  } else {
    if (list_tile == 128)
      walk_kernel<float, 128, 1, PER, SINK><<<blocks, kWave, 0, s>>>(a);
    else
      walk_kernel<float, 64, 1, PER, SINK><<<blocks, kWave, 0, s>>>(a);
  }
}

void launch_walk(hipStream_t s, const WalkArgs& a, int precision, int blocks, int list_tile,
                 int max_group) {
  const bool sink = a.tx != nullptr;
  if (a.nbox > 1)
    sink ? launch_walk_t<true, true>(s, a, precision, blocks, list_tile, max_group)
         : launch_walk_t<true, false>(s, a, precision, blocks, list_tile, max_group);
  else
    sink ? launch_walk_t<false, true>(s, a, precision, blocks, list_tile, max_group)
         : launch_walk_t<false, false>(s, a, precision, blocks, list_tile, max_group);
}

void launch_walk_stats(hipStream_t s, const WalkArgs& a) {
  walk_stats_kernel<<<256, 256, 0, s>>>(a.gstat, a.sc, a.queue, a.clock);
}

// About kDirectBlocks blocks: eight of four waves for each of the 256 CUs.  A
// block never has fewer than 512 sources, and at most 65,535 ranges are used
// (the grid's second dimension).  Without a workspace: whole targets.
DirectPlan direct_plan(int64_t n, int64_t ntest) {
  DirectPlan p;
  p.span = kDirectT;
  while (p.span > 1 && p.span / 2 >= ntest) p.span /= 2;
  p.tblocks = (ntest + p.span - 1) / p.span;
  int64_t ranges = (kDirectBlocks + p.tblocks - 1) / p.tblocks;
  const int64_t most = n / 512 < 1 ? 1 : n / 512;
  if (ranges > most) ranges = most;
  if (ranges > 65535) ranges = 65535;
  // whole tiles of sources per range
  p.range = ((n + ranges - 1) / ranges + kDirectT - 1) / kDirectT * kDirectT;
  p.ranges = (n + p.range - 1) / p.range;
  p.partials = p.ranges * (kDirectT / p.span);
  return p;
}

void launch_direct(hipStream_t s, int64_t n, const double* x, const double* y, const double* z,
                   const double* q, int64_t ntest, const int64_t* testidx, double eps2, double sign,
                   double* ex, double* ey, double* ez, double* pot, double* work, int nbox,
                   const double* vbox) {
  if (ntest <= 0) return;
  DirectPlan p = direct_plan(n, ntest);
  if (!work || p.partials == 1) {
    p.span = kDirectT;
    p.tblocks = (ntest + kDirectT - 1) / kDirectT;
    p.range = n;
    p.ranges = 1;
    work = nullptr;
  }
  // A skipped pair adds zero times its separation, which is NaN for a target
  // that is not at a finite position.  Any other source makes that component NaN
  // too; a particle alone has no other, and its sums are empty.
  const int64_t sources = n == 1 && !vbox ? 0 : n;
  direct_kernel<<<dim3((unsigned)p.tblocks, (unsigned)p.ranges), kDirectT, 0, s>>>(
      sources, x, y, z, q, ntest, testidx, eps2, sign, ex, ey, ez, pot, nbox, vbox, p.span, p.range, work);
  if (work)
    direct_reduce_kernel<<<(unsigned)((4 * ntest + kDirectT / kWave - 1) / (kDirectT / kWave)),
                           kDirectT, 0, s>>>(ntest, (int)p.partials, work, sign, ex, ey, ez, pot);
}

}  // namespace pepc
