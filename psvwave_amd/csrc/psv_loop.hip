// psv_loop.hip -- resident time loops.
//
// A launch per time step reads and writes the whole state and reads the
// materials every step (104 B per point) and pays the launch latency.  On
// this device the state fits on chip: 256 compute units hold 128 MB of
// registers and 40 MB of LDS.  A resident loop therefore runs all time steps
// in one launch.  Each block owns one tile for the whole loop; stresses and
// material factors of its points stay in registers and LDS, velocities in
// LDS, and per step only the velocities on the three-point rim of each tile
// move, from block to block through memory.
//
// What bounds a step is FP64 issue (about 111 FP64 instructions per point and
// 40 others, at 1.8 ns per wave and instruction) plus one exchange, about 2 us
// from the last store to the first value read.  The exchange is hidden only
// where two blocks share a compute unit.  us per step of a forward (19
// receivers, no snapshots): 250 x 150 points 3.1 (a launch per step: 8.6),
// 680 x 380 4.8 to 5.1, 960 x 448 on one block per compute unit 5.9 and two
// such loops on two 8.0 (108e9 points per second), 1800 x 450 7.6 (a launch
// per step: 27).
//
// Tile.  Lane l of every wave is column x0 - 2 + l, wave w holds the rows
// q = w P .. w P + P - 1 of the tile, row q being z0 - 2 + q.  The velocity
// update of the own points needs stresses two points beyond them: the two
// outer lanes on either side and the two outer rows at either end compute
// those ring stresses redundantly from exchanged velocities, so one exchange
// per step suffices and every lane runs the same code.  Own points: up to 60
// columns and waves * P - 4 rows.
//
// Exchange.  A velocity on a tile's rim is sent as one 16-byte cell {low word, tag,
// high word, tag}: each 8-byte half carries its own tag (the step's number),
// so a receiver polls the cells themselves and needs no separate flag, no
// fence and no ordering between stores.  Cells are written and read at
// device scope (past the XCD's own L2).  Two cell sets alternate: a block
// overwrites the cells of step k at step k + 2, after it has received every
// neighbour's step k + 1, which that neighbour sends after consuming step k
// (neighbours read each other's rims on all sides, so this holds for each
// pair of tiles that exchange anything; tiles are at least 3 points wide and
// high, so only adjacent tiles do).
//
// All blocks of a launch must be resident at once.  The gate below admits no
// more blocks than the device holds; should other work in another process
// keep some of them out, the blocks notice at the start (bounded wait), all
// of them leave without having written anything, and the host runs the loop
// with one launch per step instead.
#include "psv_loop.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <type_traits>

#include "psv_model.h"

namespace psv {

namespace {

typedef const LoopArgs __attribute__((address_space(4))) ConstArgs;
// Device memory behind a generic pointer that was itself read from memory.
template <class T>
using Global = __attribute__((address_space(1))) T;
template <class T>
__device__ __forceinline__ Global<T> *gp(T *p) {
  return (Global<T> *)p;
}

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int kVW = 67;  // velocity columns -2 .. 64 around the 64 lanes; column
                         // 65, which no value in use depends on, is the next
                         // row's column -2, always zero
constexpr int kDeviceScope = 16;  // buffer cache policy: device scope (sc1)

// A value the compiler cannot see through: what is computed from it in a
// time step is not kept in registers across all of them.
__device__ __forceinline__ int fresh(int v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ __forceinline__ unsigned fresh(unsigned v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ __forceinline__ double fresh(double v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ __forceinline__ int fresh_uniform(int v) {  // of a scalar register
  asm volatile("" : "+s"(v));
  return v;
}
__device__ __forceinline__ int fresh_scalar(int v) {
  v = __builtin_amdgcn_readfirstlane(v);
  asm volatile("" : "+s"(v));
  return v;
}
__device__ __forceinline__ const ConstArgs *fresh(const ConstArgs *v) {
  asm volatile("" : "+s"(v));
  return v;
}

// Quotients x / d by a grid spacing d in [2^-40, 2^40], correctly rounded.
// FastDiv's operations (psv_kernels.hip) serve x = 0 and 2^-960 <= |x| <=
// 2^980.  In lanes `scaled` x was scaled by 2^128 before (exactly) and the
// last operation, a fused multiply-add that scales its result by 2^-128
// before its one rounding, undoes it; in the others it is a plain one, at
// the same rate.
struct Spacing {
  double d, y, zh, zl;
  __device__ double quotient(double x, unsigned long long scaled) const {
    const double q0 = __builtin_fma(x, zl, x * zh);
    const double r = __builtin_fma(q0, d, -x);
    return __builtin_amdgcn_div_fmas(-r, y, q0, __builtin_amdgcn_inverse_ballot_w64(scaled));
  }
};
// The lanes whose dividends have to be scaled: those where the difference
// they are formed from is below 2^-500 (with material factors of exponents in
// [-300, 100], a dividend is below 2^-400 there and above 2^-800 or zero
// elsewhere).
__device__ __forceinline__ unsigned long long small_lanes(double difference) {
  return __ballot(__builtin_fabs(difference) < 0x1p-500);
}
__device__ __forceinline__ int scale_of(unsigned long long lanes) {
  return fresh(__builtin_amdgcn_inverse_ballot_w64(lanes) ? 128 : 0);
}
__device__ __forceinline__ void scale(double &x, int exponent) {
  x = __builtin_amdgcn_ldexp(x, exponent);
}

// How the next pass over some values divides (one code for all three, the
// wave branches around what a mode adds: separate passes cost registers, and
// spilled factors, read back behind the other block's polls, made a pass
// three times as long): kNormal if each is zero or of a binary exponent (frexp) in [elimit, 600]; kSmall if only the
// lower bound fails, as in the numerical precursor ahead of a wavefront;
// kIeee otherwise (a plain IEEE division for every value: runs that
// overflow).  Two roundings of differences can cancel to 2^-109 of the
// smallest value, so with material factors of exponents e_f in [-300, 100] a
// dividend is zero or at least 2^(elimit - 110 + min(e_f, 0)); elimit =
// -849 - min(e_f, 0) keeps that above 2^-960.  The upper bound leaves room
// for one step's growth, so a value that is not finite is never the first
// one out of range.
enum : int { kNormal = 0, kSmall = 1, kIeee = 2 };
constexpr int kExpMax = 600;
struct Range {
  int emin = 0, emax = 0;  // of zeros and of values that are not finite: 0
  __device__ void values(double a, double b) {
    const int ea = __builtin_amdgcn_frexp_exp(a), eb = __builtin_amdgcn_frexp_exp(b);
    emin = min(emin, min(ea, eb));
    emax = max(emax, max(ea, eb));
  }
  // also for values that may be infinite or no numbers
  __device__ void any_values(double a, double b) {
    values(a, b);
    finite(a, b);
  }
  __device__ void finite(double a, double b) {
    if (!(__builtin_fabs(a) + __builtin_fabs(b) < 0x1p800)) emax = 4096;
  }
  // adds the wave's need to *word (in LDS): one lane's atomic per wave, not
  // one per lane, which all hit one bank
  __device__ void report(int *word, int elimit) const {
    const unsigned long long small = __ballot(emin < elimit), large = __ballot(emax > kExpMax);
    if (small | large) {
      const int m = (small ? kSmall : 0) | (large ? kIeee : 0);
      if ((int)__ffsll((unsigned long long)__ballot(1)) - 1 == (int)(threadIdx.x & 63))
        atomicOr(word, m);
    }
  }
};

// The terms of one point's strain rates (stress_point's expression trees), in
// place: from the differences x_* and z_* of vx and vz along x and z to
// txx's, tzz's and txz's rates, lambda and mu of txx and tzz included.
template <bool IEEE>
__device__ __forceinline__ void stress_rates(double dvx_x, double dvz_z, double dvx_z,
                                             double dvz_x, double lm, double mu, bool small,
                                             const Spacing &dx, const Spacing &dz, double &xx_rate,
                                             double &zz_rate, double &xz_rate) {
  // one operation instead of two, the same value where 2 mu does not overflow
  const double la = IEEE ? lm - 2 * mu : __builtin_fma(-2.0, mu, lm);
  double xx_x = lm * dvx_x, xx_z = la * dvz_z, zz_x = la * dvx_x, zz_z = lm * dvz_z;
  if (IEEE) {
    xx_x /= dx.d, xx_z /= dz.d, zz_x /= dx.d, zz_z /= dz.d, dvx_z /= dz.d, dvz_x /= dx.d;
  } else {
    unsigned long long sx = 0, sz = 0, sxx = 0, sxz = 0;
    if (small) {
      sx = small_lanes(dvx_x), sz = small_lanes(dvz_z);
      sxx = small_lanes(dvx_z), sxz = small_lanes(dvz_x);
      const int ex = scale_of(sx), ez = scale_of(sz);
      scale(xx_x, ex), scale(zz_x, ex), scale(xx_z, ez), scale(zz_z, ez);
      scale(dvx_z, scale_of(sxx)), scale(dvz_x, scale_of(sxz));
    }
    xx_x = dx.quotient(xx_x, sx), zz_x = dx.quotient(zz_x, sx);
    xx_z = dz.quotient(xx_z, sz), zz_z = dz.quotient(zz_z, sz);
    dvx_z = dz.quotient(dvx_z, sxx), dvz_x = dx.quotient(dvz_x, sxz);
  }
  xx_rate = xx_x + xx_z, zz_rate = zz_x + zz_z, xz_rate = dvx_z + dvz_x;
}

// The stress divergences of one point (velocity_point's expression trees)
// from the differences of txx and txz along x and z for vx, of txz and tzz
// for vz.
template <bool IEEE>
__device__ __forceinline__ void velocity_rates(double vx_x, double vx_z, double vz_x, double vz_z,
                                               bool small, const Spacing &dx, const Spacing &dz,
                                               double &vx_rate, double &vz_rate) {
  if (IEEE) {
    vx_x /= dx.d, vx_z /= dz.d, vz_x /= dx.d, vz_z /= dz.d;
  } else {
    unsigned long long a = 0, b = 0, c = 0, d = 0;
    if (small) {
      a = small_lanes(vx_x), b = small_lanes(vx_z), c = small_lanes(vz_x), d = small_lanes(vz_z);
      scale(vx_x, scale_of(a)), scale(vx_z, scale_of(b));
      scale(vz_x, scale_of(c)), scale(vz_z, scale_of(d));
    }
    vx_x = dx.quotient(vx_x, a), vx_z = dz.quotient(vx_z, b);
    vz_x = dx.quotient(vz_x, c), vz_z = dz.quotient(vz_z, d);
  }
  vx_rate = vx_x + vx_z, vz_rate = vz_x + vz_z;
}

// Keeps the scheduler from interleaving the stencils of several rows (whose
// operands would then all be live at once).
__device__ __forceinline__ void row_fence() { __builtin_amdgcn_sched_barrier(0); }

// min(a, b) of factors that are no NaN (one instruction; fmin adds a quieting
// one per operand).
__device__ __forceinline__ double min_factor(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// The blocks of a launch meet before any of them writes anything: true when
// all are resident.  state: 0 waiting, 1 go, 2 leave; exactly one of go and
// leave is ever decided.
__device__ bool loop_meet(const LoopLaunch &l) {
  unsigned *const state = l.sync + 1;
  if (l.poison && __hip_atomic_load(l.poison, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
    unsigned want = 0;
    __hip_atomic_compare_exchange_strong(state, &want, 2u, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
  } else if (__hip_atomic_fetch_add(l.sync, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) +
                 1 ==
             (unsigned)l.nblocks) {
    unsigned want = 0;
    if (__hip_atomic_compare_exchange_strong(state, &want, 1u, __ATOMIC_RELAXED,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      __hip_atomic_store(l.status, (unsigned)kLoopRan, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
  }
  // 0.1 s of the 100 MHz constant clock: the gate lets no other launch of this
  // process wait here meanwhile
  const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
  for (;;) {
    const unsigned s = __hip_atomic_load(state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (s) {
      if (s == 2 && l.poison)
        __hip_atomic_store(l.poison, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return s == 1;
    }
    if (__builtin_amdgcn_s_memrealtime() - t0 > 10000000ull) {
      unsigned want = 0;
      __hip_atomic_compare_exchange_strong(state, &want, 2u, __ATOMIC_RELAXED,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_s_sleep(2);
  }
}

template <int KIND, bool ADJ>
__global__ void __launch_bounds__(64 * kLoopKinds[KIND].waves)
    __attribute__((amdgpu_waves_per_eu(4, 4)))
resident_loop(LoopLaunch l) {
  constexpr int P = kLoopKinds[KIND].rows, NW = kLoopKinds[KIND].waves;
  constexpr int NT = 64 * NW, SR = NW * P;
  constexpr int VROWS = SR + 4;  // velocity rows q = -2 .. SR + 1
  constexpr int NV = VROWS * kVW + 1;
  // rim and frame cells per thread (own at most 60 x (SR - 4))
  constexpr int NSEND = (60 * (SR - 4) - 54 * (SR - 10) + NT - 1) / NT;
  constexpr int NRECV = (66 * (SR + 2) - 60 * (SR - 4) + NT - 1) / NT;
  constexpr int RIM = loop_rim_cells(KIND);
  static_assert(NSEND * NT <= RIM, "a tile's rim fits its cells");
  // Velocities; taper factors of the rows; txx of the own rows 2 .. SR - 3,
  // txz of all rows, and of tzz the rows other waves read, each wave's rows 0,
  // 1 and P - 1.  In one array in this order, so that a strip's neighbour rows
  // lie at fixed offsets from its own: those of the first and last wave that
  // do not exist, which no own point uses, are read from the array beside.
  constexpr int ZR = P < 3 ? P : 3;
  constexpr int NXX = (SR - 4) * 64, NXZ = SR * 64, NZZ = NW * ZR * 64;
  __shared__ double s_mem[NV + NXX + NXZ + NZZ + NV + SR];
  double *const s_vx = s_mem, *const s_xx = s_vx + NV, *const s_xz = s_xx + NXX;
  double *const s_zz = s_xz + NXZ, *const s_vz = s_zz + NZZ, *const s_tz = s_vz + NV;
  // what the next pass over the velocities (by step parity) and over the
  // stresses needs, kNormal | kSmall | kIeee
  __shared__ int s_vmode[2], s_smode, s_factor;
  __shared__ int s_go, s_stall;

  const Global<const int> *const bp = gp((const int *)(l.blocks + blockIdx.x));
  const struct { int x, y, z; } bt = {bp[0], bp[1], bp[2]};
  // the arguments do not change while the launch runs: read through the
  // constant address space, uniform values stay in scalar registers
  const ConstArgs &A0 = ((const ConstArgs *)l.loops)[bt.x], &A = A0;
  if (threadIdx.x == 0) {
    s_go = loop_meet(l);
    s_stall = 0;
    s_smode = s_factor = 0;
  }
  __syncthreads();
  if (!s_go) return;

  // The passes over the rows need nearly all of a wave's 128 registers: what
  // they do not use is packed, derived again from the thread's number, or
  // read back from memory where it is used.
  const int tid = threadIdx.x, lane = tid & 63;
  auto lane_of = [&]() { return fresh(tid) & 63; };
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nx = A.nx, nz = A.nz, nt = A.nt;
  // first column of tile column i and first row of tile row i (uniform, but
  // divided in vector registers)
  auto tile_x0 = [&](int i) {
    return __builtin_amdgcn_readfirstlane((int)((long long)i * nx / A.ntx));
  };
  auto tile_z0 = [&](int i) {
    return __builtin_amdgcn_readfirstlane((int)((long long)i * nz / A.ntz));
  };
  const int tile = __builtin_amdgcn_readfirstlane(bt.z * A.ntx + bt.y);
  const int x0 = tile_x0(bt.y), wt = tile_x0(bt.y + 1) - x0;  // own columns
  const int z0 = tile_z0(bt.z), ht = tile_z0(bt.z + 1) - z0;  // own rows
  const int q0 = w * P;         // first row of the strip
  const int zs = z0 - 2 + q0;   // its grid row
  const int x = x0 - 2 + lane;
  const bool own_x = lane >= 2 && lane < 2 + wt;
  // strip rows with a stress / velocity stencil, and own rows
  // the strip's rows with a stress stencil (bit j), with a velocity stencil
  // (bit 4 + j), its own rows (8 + j) and the rows s_xx has (12 + j)
  int rows = 0;
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int q = q0 + j, z = zs + j;
    const bool stencil = z >= 2 && z < nz - 2, own = q >= 2 && q < ht + 2;
    rows |= (stencil && q < ht + 4) << j | (stencil && own) << (4 + j) | own << (8 + j) |
            (q >= 2 && q < SR - 2) << (12 + j);
  }
  rows = __builtin_amdgcn_readfirstlane(rows);
  // (tested anew in each pass: a scalar register, not one per row and test)
  auto has = [&](int test, int j) { return (fresh_uniform(rows) >> (test + j) & 1) != 0; };
  enum : int { kStressRow = 0, kVelocityRow = 4, kOwnRow = 8, kXxRow = 12 };
  const bool xs = x >= 2 && x < nx - 2 && lane < wt + 4;
  const bool xv = own_x && xs;
  const double dts = A.dts;

  // ---- the tile's constants and initial state ----
  double lm[P], mu[P], bd[P];
  // Stresses: tzz and, of the first XK rows, txx stay in registers; txz and the
  // other rows' txx (of own rows; the ring's is not used) in LDS, where the
  // velocity pass reads them anyway.
  constexpr int XK = P == 4 ? 0 : P;
  double xx[P], zz[P];
  int factor_exp = 0;  // smallest of the material factors; -4096: one is too large
  const double tx = gp(A.taper_x)[min(x, nx + 1)];
  {
    const int xc = min(x, nx + 1);
#pragma unroll
    for (int j = 0; j < P; ++j) {
      const int zc = min(zs + j, nz + 1);
      const long long g = A.origin + (long long)zc * A.pitch + xc;
      mu[j] = gp(A.mu)[g];
      lm[j] = gp(A.lm)[g];
      bd[j] = gp(A.b)[g] * dts;
      for (double f : {lm[j], lm[j] - 2 * mu[j]})
        if (f != 0.0) factor_exp = min(factor_exp, __builtin_amdgcn_frexp_exp(f));
      for (double f : {lm[j], lm[j] - 2 * mu[j], mu[j], dts * mu[j], bd[j], dts})
        if (!(__builtin_fabs(f) <= 0x1p100)) factor_exp = -4096;
      xx[j] = zz[j] = 0.0;
      double xz = 0.0;
      if (A.in[0] && x >= 0 && x < nx && zs + j >= 0 && zs + j < nz) {
        const long long s = A.in_origin + (long long)(zs + j) * A.in_pitch + x;
        xx[j] = gp(A.in[2])[s];
        zz[j] = gp(A.in[3])[s];
        xz = gp(A.in[4])[s];
      }
      s_xz[(q0 + j) * 64 + lane] = xz;
      if (has(kXxRow, j)) s_xx[(q0 + j - 2) * 64 + lane] = xx[j];
      if (j < 2 || j == P - 1) s_zz[(w * ZR + min(j, 2)) * 64 + lane] = zz[j];
    }
  }
  for (int i = threadIdx.x; i < SR; i += NT) s_tz[i] = gp(A.taper_z)[min(z0 - 2 + i, nz + 1)];
  // a tile with factors out of range divides by the IEEE sequence throughout,
  // and so does the first step from a given state, whose values are not tested
  if (factor_exp < 0) atomicMin(&s_factor, factor_exp);
  if (threadIdx.x == 0) {
    s_vmode[A.k0 & 1] = kNormal;
    s_vmode[(A.k0 + 1) & 1] = A.in[0] ? kIeee : kNormal;
  }
  for (int i = threadIdx.x; i < NV; i += NT) {
    const int r = i / kVW, c = i - r * kVW;
    const int zi = z0 - 2 + r - 2, xi = x0 - 2 + c - 2;
    double a = 0.0, b = 0.0;
    if (A.in[0] && xi >= x0 - 3 && xi < x0 + wt + 3 && zi >= z0 - 3 && zi < z0 + ht + 3 &&
        xi >= 0 && xi < nx && zi >= 0 && zi < nz) {
      const long long s = A.in_origin + (long long)zi * A.in_pitch + xi;
      a = gp(A.in[0])[s];
      b = gp(A.in[1])[s];
    }
    s_vx[i] = a;
    s_vz[i] = b;
  }

  // ---- this thread's cells ----
  // A tile's rim cells are numbered along its first three and last three
  // rows, then the first three columns of the rows between, then the last
  // three, so that what a neighbour reads lies together;
  // cell i of component c and set p lies at ((tile * 2 + p) * 2 + c) * RIM +
  // i.  So a line of cells has one writer, and no tile reads lines that it
  // writes: with cells of several tiles in one line, a read waited for the
  // reader's own write to reach memory first (1.7 us instead of 0.7).
  auto vidx = [](int r, int c) { return (r + 4) * kVW + c + 4; };
  auto rim_cell = [](int wt, int ht, int r, int c) {
    if (wt <= 6 || ht <= 6) return r * wt + c;
    if (r < 3) return r * wt + c;
    if (r >= ht - 3) return (r - ht + 6) * wt + c;
    return 6 * wt + (c < 3 ? (r - 3) * 3 + c : (ht + r - 9) * 3 + c - wt + 3);
  };
  // LDS indices of the rim cell it sends (low half; kNoCell: none) and of its
  // receiver (high half), and of the frame cells it receives
  constexpr unsigned kNoCell = 0xffffu;
  static_assert(NSEND == 1 && NRECV <= 2 && NV < (int)kNoCell, "cells are packed in halves");
  unsigned send_rec = kNoCell << 16, recv_pack = 0;
  unsigned recv_g[NRECV];
  {
    const int i = tid;
    int r, c;
    bool on;
    if (wt > 6 && ht > 6) {
      on = i < 6 * wt + 6 * (ht - 6);
      if (i < 6 * wt) {
        const int k = i / wt;
        r = k < 3 ? k : ht - 6 + k;
        c = i - k * wt;
      } else {
        const int k = (i - 6 * wt) / 3, m = i - 6 * wt - 3 * k;
        r = 3 + (k < ht - 6 ? k : k - (ht - 6));
        c = k < ht - 6 ? m : wt - 3 + m;
      }
    } else {
      on = i < wt * ht;
      r = i / wt;
      c = i - r * wt;
    }
    send_rec |= on ? (unsigned)vidx(r, c) : kNoCell;
  }
#pragma unroll
  for (int s = 0; s < NRECV; ++s) {
    const int i = threadIdx.x + s * NT;
    const int fw = wt + 6, rows = 3 * fw;
    int r, c;
    bool on = i < 2 * rows + 6 * ht;
    if (i < 2 * rows) {
      const int k = i / fw;
      r = k < 3 ? k - 3 : ht - 3 + k;
      c = i - k * fw - 3;
    } else {
      const int k = (i - 2 * rows) / 3, m = i - 2 * rows - 3 * k;
      r = k < ht ? k : k - ht;
      c = k < ht ? m - 3 : wt + m;
    }
    const int xi = x0 + c, zi = z0 + r;
    on = on && xi >= 0 && xi < nx && zi >= 0 && zi < nz;
    recv_pack |= (on ? (unsigned)vidx(r, c) : kNoCell) << (16 * s);
    recv_g[s] = 0;
    if (on) {  // the adjacent tile that owns the point
      const int ox = bt.y + (c < 0 ? -1 : c >= wt ? 1 : 0);
      const int oz = bt.z + (r < 0 ? -1 : r >= ht ? 1 : 0);
      const int ox0 = (int)((long long)ox * nx / A.ntx), oz0 = (int)((long long)oz * nz / A.ntz);
      const int ow = (int)((long long)(ox + 1) * nx / A.ntx) - ox0;
      const int oh = (int)((long long)(oz + 1) * nz / A.ntz) - oz0;
      recv_g[s] = (unsigned)((oz * A.ntx + ox) * 4 * RIM +
                             rim_cell(ow, oh, zi - oz0, xi - ox0)) * 16u;
    }
  }
  const auto cells =
      __builtin_amdgcn_make_buffer_rsrc(A.cells, 0, A.cells_bytes, 0x00020000);

  // ---- this wave's injection targets: target t in lane t ----
  const int tg0 = __builtin_amdgcn_readfirstlane(gp(A.inj_off)[tile * NW + w]);
  const int ntg = __builtin_amdgcn_readfirstlane(gp(A.inj_off)[tile * NW + w + 1]) - tg0;
  auto inj_entry = [](const ConstArgs &A, int e) {
    const Global<const InjEntry> *const p = gp(A.inj) + e;
    return InjEntry{p->local, p->comp, p->src, p->pad, p->coef};
  };
  auto inj_sample = [&](const ConstArgs &A, const InjEntry &E, int it) {
    const double *const s = ADJ ? (E.comp ? A.adj_z : A.adj_x) : A.stf;
    return gp(s)[(long long)E.src * nt + it];
  };
  auto inj_term = [](const ConstArgs &A, int comp, double coef, double b, double val) {
    return ADJ ? A.dt * b * val / A.dxdz : coef * val * A.dt * b / (comp ? A.d4z : A.d4x);
  };
  // ---- this thread's receiver ----
  int rec_k = 0;
  double rec_sx = 0.0, rec_sz = 0.0;  // (read back where registers are short)
  if (!ADJ && A.rec_off) {
    const int r0 = gp(A.rec_off)[tile], nr = gp(A.rec_off)[tile + 1] - r0;
    if (tid < nr) {
      send_rec = (send_rec & 0xffffu) | (unsigned)gp(A.rec)[r0 + tid].local << 16;
      rec_k = gp(A.rec)[r0 + tid].src;
    }
  }
  __syncthreads();

  const int tile_exp = __builtin_amdgcn_readfirstlane(s_factor);
  const int floor_mode = tile_exp < -300 ? kIeee : kNormal;
  const int elimit = -849 - tile_exp;
  auto mode_of = [&](int needs) {  // needs: kSmall and kIeee bits
    return min(max(floor_mode, __builtin_amdgcn_readfirstlane(needs)), (int)kIeee);
  };
  // LDS indices of the strip's first velocity and stress row, each to be added
  // to the lane
  const int vrow = (q0 + 2) * kVW + 2, srow = q0 * 64;
  unsigned tag = l.tag0;

  // The velocity that the lane's first injection target adds to (2 LDS index +
  // component; -1: none; bit 30: several terms) and its next term.
  int inj_at = -1;
  double inj_value = 0.0;
  constexpr int kInjMore = 1 << 30;
  auto inj_fetch = [&](int base, int it) {
    const ConstArgs &A = *fresh(&A0);
    const int t = base + lane_of();
    inj_at = -1;
    if (t < ntg) {
      const Global<const InjEntry> *const p = gp(A.inj_head) + tg0 + t;
      const InjEntry E = {p->local, p->comp, p->src, p->pad, p->coef};
      const int r = E.local >> 6, c = E.local & 63;
      inj_at = ((vrow + r * kVW + c) << 1) | E.comp | (E.pad ? kInjMore : 0);
      inj_value = inj_term(A, E.comp, E.coef,
                           gp(A.b)[A.origin + (long long)(zs + r) * A.pitch + x0 - 2 + c],
                           inj_sample(A, E, it));
    }
  };

  // What a step does with the state at its start: receivers, snapshot store,
  // correlation; and its injection terms.  Called between sending the rims and
  // the first poll for the neighbours' (the state then is the next step's),
  // which hides it.
  int phase = (ADJ ? nt - 1 - A0.k0 : A0.k0) % A0.si;  // of the next step's time index
  auto begin_step = [&](int k) {
    const ConstArgs &A = *fresh(&A0);
    const int it = ADJ ? nt - 1 - k : k;
    const bool snap_step = phase == 0;
    phase = ADJ ? (phase == 0 ? A.si : phase) - 1 : (phase + 1 == A.si ? 0 : phase + 1);
    const unsigned rec_l = fresh(send_rec) >> 16;
    if (!ADJ && rec_l != kNoCell) {
      // receiver record at the start of the step (src/fdModel.cpp:576-596),
      // which continues the previous step's
      const long long at = (long long)fresh(rec_k) * nt + it;
      const double ax = A.dt * s_vx[rec_l] / A.dxdz, az = A.dt * s_vz[rec_l] / A.dxdz;
      double sx = rec_sx, sz = rec_sz;
      if (P == 4 && k > 0) sx = gp(A.rtf_x)[at - 1], sz = gp(A.rtf_z)[at - 1];
      sx = k == 0 ? ax : sx + ax;
      sz = k == 0 ? az : sz + az;
      gp(A.rtf_x)[at] = sx;
      gp(A.rtf_z)[at] = sz;
      if (P < 4) rec_sx = sx, rec_sz = sz;
    }
    if (ntg > 0) inj_fetch(0, it);
    if (snap_step && A.snap[0] && it / A.si % A.slot_every == 0) {
      const int ln = lane_of(), va0 = vrow + ln, xk = x0 - 2 + ln;
      const int slot = it / A.si;
      const long long so = (long long)(slot / A.slot_every - A.slot0) * A.slot_stride;
      if (!ADJ) {
        if (own_x)
#pragma unroll
          for (int j = 0; j < P; ++j)
            if (has(kOwnRow, j)) {
              const long long ci = so + (long long)(zs + j) * nx + xk;
              __builtin_nontemporal_store(s_vx[va0 + j * kVW], gp(A.snap[0]) + ci);
              __builtin_nontemporal_store(s_vz[va0 + j * kVW], gp(A.snap[1]) + ci);
              __builtin_nontemporal_store(s_xx[srow + ln + (j - 2) * 64], gp(A.snap[2]) + ci);
              __builtin_nontemporal_store(zz[j], gp(A.snap[3]) + ci);
              __builtin_nontemporal_store(s_xz[srow + ln + j * 64], gp(A.snap[4]) + ci);
            }
      } else {
        const long long ko = A.defer_stride * slot;
        if (own_x && xk >= A.kx0 && xk < A.kx1)
#pragma unroll
          for (int j = 0; j < P; ++j) {
            const int z = zs + j;
            if (has(kOwnRow, j) && z >= A.kz0 && z < A.kz1) {
              const long long c = (long long)z * nx + xk, ci = so + c, ck = ko + c;
              double r = 0.0, la_k = 0.0, m = 0.0, s[5];
#pragma unroll
              for (int f = 0; f < 5; ++f) s[f] = __builtin_nontemporal_load(gp(A.snap[f]) + ci);
              if (!A.defer_stride) {
                r = __builtin_nontemporal_load(gp(A.rho_k) + ck);
                la_k = __builtin_nontemporal_load(gp(A.lam_k) + ck);
                m = __builtin_nontemporal_load(gp(A.mu_k) + ck);
              }
              correlate_point(A.wcorr, lm[j], mu[j], s_vx[va0 + j * kVW], s_vz[va0 + j * kVW],
                              s_xx[srow + ln + (j - 2) * 64], zz[j], s_xz[srow + ln + j * 64], s[0],
                              s[1], s[2], s[3], s[4], r, la_k, m);
              __builtin_nontemporal_store(r, gp(A.rho_k) + ck);
              __builtin_nontemporal_store(la_k, gp(A.lam_k) + ck);
              __builtin_nontemporal_store(m, gp(A.mu_k) + ck);
            }
            row_fence();
          }
      }
    }
  };
  begin_step(A.k0);

  for (int k = A.k0; k < A.k1; ++k, ++tag) {
    const int it = ADJ ? nt - 1 - k : k;
    // ---- stresses ----
    const int vmode = mode_of(s_vmode[(k + 1) & 1]);
    if (xs) {
      const Spacing dx{A.dx, A.rdx, A.zhx, A.zlx}, dz{A.dz, A.rdz, A.zhz, A.zlz};
      const int ln = lane_of(), va = vrow + ln, sa = srow + ln, ta = fresh(q0);
      const int za = fresh_scalar(w) * ZR * 64 + ln;
      Range range;
      // vx rows -1 .. P + 1 and vz rows -2 .. P of the lane's column
      double cx[P + 3], cz[P + 3];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        cx[j] = s_vx[va + (j - 1) * kVW];
        cz[j] = s_vz[va + (j - 2) * kVW];
      }
#pragma unroll
      for (int j = 0; j < P; ++j) {
        const int v = va + j * kVW;
        cx[j + 3] = s_vx[v + 2 * kVW];
        cz[j + 3] = s_vz[v + kVW];
        if (has(kStressRow, j)) {
          const double dvx_x = kC1 * (s_vx[v + 1] - cx[j + 1]) + kC2 * (s_vx[v - 1] - s_vx[v + 2]);
          const double dvz_z = kC1 * (cz[j + 2] - cz[j + 1]) + kC2 * (cz[j] - cz[j + 3]);
          const double dvx_z = kC1 * (cx[j + 2] - cx[j + 1]) + kC2 * (cx[j] - cx[j + 3]);
          const double dvz_x = kC1 * (cz[j + 2] - s_vz[v - 1]) + kC2 * (s_vz[v - 2] - s_vz[v + 1]);
          // read while the rates are computed, not before: the neighbours'
          // registers are free by now
          if (P == 4) row_fence();
          double tz;
          if (P < 4) tz = s_tz[ta + j];
          double xz = s_xz[sa + j * 64];
          if (j >= XK) xx[j] = has(kXxRow, j) ? s_xx[sa + (j - 2) * 64] : 0.0;
          mu[j] = fresh(mu[j]);  // 2 mu, dts mu: computed here, not kept (and spilled)
          double xx_rate, zz_rate, xz_rate;
          if (__builtin_expect(vmode == kIeee, 0))
            stress_rates<true>(dvx_x, dvz_z, dvx_z, dvz_x, lm[j], mu[j], false, dx, dz, xx_rate,
                               zz_rate, xz_rate);
          else
            stress_rates<false>(dvx_x, dvz_z, dvx_z, dvz_x, lm[j], mu[j], vmode == kSmall, dx, dz,
                                xx_rate, zz_rate, xz_rate);
          if (P == 4) tz = s_tz[ta + j];
          const double taper = min_factor(tx, tz);
          xx[j] = taper * (xx[j] + dts * xx_rate);
          zz[j] = taper * (zz[j] + dts * zz_rate);
          xz = taper * (xz + dts * mu[j] * xz_rate);
          range.values(xx[j], zz[j]);
          range.values(xz, xz);
          if (vmode == kIeee) {
            asm volatile("");  // a branch, no selects for the other modes to run
            range.finite(xx[j], zz[j]);
            range.finite(xz, xz);
          }
          s_xz[sa + j * 64] = xz;
          if (has(kXxRow, j)) s_xx[sa + (j - 2) * 64] = xx[j];
          if (j < 2 || j == P - 1) s_zz[za + min(j, 2) * 64] = zz[j];
        }
        row_fence();
      }
      range.report(&s_smode, elimit);
    }
    __syncthreads();

    // ---- velocities ----
    if (threadIdx.x == 0) s_vmode[(k + 1) & 1] = 0;  // read by all before the barrier
    const int smode = mode_of(s_smode);
    if (xv) {
      const Spacing dx{A.dx, A.rdx, A.zhx, A.zlx}, dz{A.dz, A.rdz, A.zhz, A.zlz};
      const int ln = lane_of(), va = vrow + ln, sa = srow + ln, ta = fresh(q0);
      const int za = fresh_scalar(w) * ZR * 64 + ln;
      Range range;
      // txz rows -2 .. P and tzz rows -1 .. P + 1 of the lane's column
      double xz[P + 3] = {s_xz[sa - 128], s_xz[sa - 64], s_xz[sa]};
      double cz[P + 3] = {s_zz[za - 64], zz[0], P > 1 ? zz[P > 1 ? 1 : 0] : s_zz[za + ZR * 64]};
#pragma unroll
      for (int j = 0; j < P; ++j) {
        xz[j + 3] = s_xz[sa + (j + 1) * 64];
        cz[j + 3] = j + 2 < P ? zz[j + 2 < P ? j + 2 : 0] : s_zz[za + (ZR + j + 2 - P) * 64];
        if (has(kVelocityRow, j)) {
          const int s = sa + j * 64, x2 = s - 2 * 64;
          const double xx0 = j < XK ? xx[j] : s_xx[x2];
          const double vx_x = kC1 * (xx0 - s_xx[x2 - 1]) + kC2 * (s_xx[x2 - 2] - s_xx[x2 + 1]);
          const double vx_z = kC1 * (xz[j + 2] - xz[j + 1]) + kC2 * (xz[j] - xz[j + 3]);
          const double vz_x = kC1 * (s_xz[s + 1] - xz[j + 2]) + kC2 * (s_xz[s - 1] - s_xz[s + 2]);
          const double vz_z = kC1 * (cz[j + 2] - cz[j + 1]) + kC2 * (cz[j] - cz[j + 3]);
          if (P == 4) row_fence();
          const double tz = s_tz[ta + j], vx0 = s_vx[va + j * kVW], vz0 = s_vz[va + j * kVW];
          double vx_rate, vz_rate;
          if (__builtin_expect(smode == kIeee, 0))
            velocity_rates<true>(vx_x, vx_z, vz_x, vz_z, false, dx, dz, vx_rate, vz_rate);
          else
            velocity_rates<false>(vx_x, vx_z, vz_x, vz_z, smode == kSmall, dx, dz, vx_rate,
                                  vz_rate);
          const double taper = min_factor(tx, tz);
          const double vx = taper * (vx0 + bd[j] * vx_rate);
          const double vz = taper * (vz0 + bd[j] * vz_rate);
          range.values(vx, vz);
          if (smode == kIeee) {
            asm volatile("");
            range.finite(vx, vz);
          }
          s_vx[va + j * kVW] = vx;
          s_vz[va + j * kVW] = vz;
        }
        row_fence();
      }
      range.report(&s_vmode[k & 1], elimit);
    }
    // injection: lane t adds the terms of target t in list order
    for (int base = 0; base < ntg; base += 64) {
      const ConstArgs &A = *fresh(&A0);
      if (base) inj_fetch(base, it);
      if (inj_at >= 0) {
        const int vi = (inj_at & ~kInjMore) >> 1;
        double *const v = (inj_at & 1 ? s_vz : s_vx) + vi;
        double a = *v + inj_value;
        if (inj_at & kInjMore) {  // several terms at one point
          const int t = tg0 + base + lane_of();
          int e = gp(A.inj_first)[t];
          const int e1 = gp(A.inj_first)[t + 1];
          const int r = vi / kVW - 2, c = vi % kVW - 2;
          const double bv = gp(A.b)[A.origin + (long long)(z0 - 2 + r) * A.pitch + x0 - 2 + c];
          for (++e; e < e1; ++e) {
            const InjEntry F = inj_entry(A, e);
            a += inj_term(A, F.comp, F.coef, bv, inj_sample(A, F, it));
          }
        }
        *v = a;
        Range range;
        range.any_values(a, a);
        range.report(&s_vmode[k & 1], elimit);
      }
    }
    __syncthreads();

    // ---- exchange ----
    if (threadIdx.x == 0) s_smode = 0;  // read by all before the barrier
    if (k + 1 < A.k1) {
      const unsigned set = (k & 1) ? 2u * RIM * 16u : 0u;
      const unsigned send_l = fresh(send_rec) & 0xffffu;
      if (send_l != kNoCell) {
        const double a = s_vx[send_l], b = s_vz[send_l];
        const u32x4 ca = {(unsigned)__double2loint(a), tag, (unsigned)__double2hiint(a), tag};
        const u32x4 cb = {(unsigned)__double2loint(b), tag, (unsigned)__double2hiint(b), tag};
        const int to = fresh(tid) * 16, base = (int)(tile * 4u * RIM * 16u + set);
        __builtin_amdgcn_raw_buffer_store_b128(ca, cells, to, base, kDeviceScope);
        __builtin_amdgcn_raw_buffer_store_b128(cb, cells, to, base + RIM * 16, kDeviceScope);
      }
      u32x4 ra[NRECV], rb[NRECV];
      unsigned recv_l[NRECV];
#pragma unroll
      for (int s = 0; s < NRECV; ++s) recv_l[s] = fresh(recv_pack) >> (16 * s) & 0xffffu;
      auto poll = [&]() {
#pragma unroll
        for (int s = 0; s < NRECV; ++s)
          if (recv_l[s] != kNoCell) {
            ra[s] = __builtin_amdgcn_raw_buffer_load_b128(cells, (int)recv_g[s], (int)set,
                                                          kDeviceScope);
            rb[s] = __builtin_amdgcn_raw_buffer_load_b128(cells, (int)recv_g[s],
                                                          (int)(set + RIM * 16u), kDeviceScope);
          }
        asm volatile("" ::: "memory");
      };
      begin_step(k + 1);
      // polls share the fabric with the cells they wait for: asking at once
      // and without pause cost 960 x 448 points 6.8 us per step against 6.0 with
      // these pauses (of 64 cycles each; both measured together), longer ones no
      // less
      __builtin_amdgcn_s_sleep(P == 4 ? 8 : 4);
      poll();
      for (unsigned spin = 0;;) {
        bool ready = true;
#pragma unroll
        for (int s = 0; s < NRECV; ++s)
          if (recv_l[s] != kNoCell)
            ready = ready && ra[s].y == tag && ra[s].w == tag && rb[s].y == tag && rb[s].w == tag;
        if (ready) break;
        // all blocks run, so a neighbour answers within microseconds; a wait
        // of some seconds means that the device is broken
        if (++spin > (1u << 23)) {
          s_stall = 1;
          break;
        }
        __builtin_amdgcn_s_sleep(2);
        poll();
      }
      Range range;
#pragma unroll
      for (int s = 0; s < NRECV; ++s)
        if (recv_l[s] != kNoCell) {
          const unsigned at = recv_l[s];
          const double a = __hiloint2double((int)ra[s].z, (int)ra[s].x);
          const double b = __hiloint2double((int)rb[s].z, (int)rb[s].x);
          s_vx[at] = a;
          s_vz[at] = b;
          range.any_values(a, b);
        }
      range.report(&s_vmode[k & 1], elimit);
      __syncthreads();
      if (s_stall) {
        if (threadIdx.x == 0)
          __hip_atomic_store(l.status, (unsigned)kLoopStalled, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_SYSTEM);
        return;
      }
    } else if (A.out[0] && own_x) {
#pragma unroll
      for (int j = 0; j < P; ++j)
        if (has(kOwnRow, j)) {
          const long long g = A.origin + (long long)(zs + j) * A.pitch + x0 - 2 + lane;
          gp(A.out[0])[g] = s_vx[vrow + lane + j * kVW];
          gp(A.out[1])[g] = s_vz[vrow + lane + j * kVW];
          gp(A.out[2])[g] = s_xx[srow + lane + (j - 2) * 64];
          gp(A.out[3])[g] = zz[j];
          gp(A.out[4])[g] = s_xz[srow + lane + j * 64];
        }
    }
  }
}

}  // namespace

namespace {

// Puts a launch's arguments and its zeroed meeting words in place, in stream
// order before it.
__global__ void prepare_loop_kernel(LoopArgs *dst, LoopArgs a, unsigned *sync) {
  const int n = (int)(sizeof(LoopArgs) / 8);
  const unsigned long long *const src = (const unsigned long long *)&a;
  for (int i = threadIdx.x; i < n; i += blockDim.x) ((unsigned long long *)dst)[i] = src[i];
  if (threadIdx.x < 2) sync[threadIdx.x] = 0;
}
static_assert(sizeof(LoopArgs) % 8 == 0, "LoopArgs is copied in 8-byte words");

// Blocks of a loop kernel that a compute unit holds, at most two.
template <int KIND>
int loop_blocks_per_cu() {
  int n = 2;
  for (const void *kernel :
       {(const void *)resident_loop<KIND, false>, (const void *)resident_loop<KIND, true>}) {
    int k = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&k, kernel, 64 * kLoopKinds[KIND].waves,
                                                     0) != hipSuccess)
      k = 0;
    n = std::min(n, k);
  }
  return n;
}

constexpr int kMaxDevices = 64;
constexpr int kXcdCus = 32;  // compute units per XCD

// XCDs of a device and blocks per compute unit of the loop kernels;
// xcds = 0 where the loops cannot run.
struct LoopDevice {
  int xcds = -1;
  int per_cu[kNumLoopKinds] = {};
};
const LoopDevice &loop_device(int dev) {
  static std::mutex m;
  static LoopDevice known[kMaxDevices];
  std::lock_guard<std::mutex> lock(m);
  LoopDevice &d = known[dev];
  if (d.xcds < 0) {
    int cus = 0;
    d.xcds = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess
                 ? cus / kXcdCus
                 : 0;
    d.per_cu[0] = loop_blocks_per_cu<0>();
    d.per_cu[1] = loop_blocks_per_cu<1>();
    d.per_cu[2] = loop_blocks_per_cu<2>();
    d.per_cu[3] = loop_blocks_per_cu<3>();
    d.per_cu[4] = loop_blocks_per_cu<4>();
    for (int n : d.per_cu)
      if (n < 1) d.xcds = 0;
    (void)hipGetLastError();
  }
  return d;
}
// Loop launches of one device in generations: the launches of a generation
// fit the device together, and each of them starts after every launch of the
// generation before, so at no time does the sum of running blocks exceed
// what can be resident.  One object per device for the whole process (all
// models, streams and threads launch through it); it holds a few events, no
// device memory.  An event belongs to the stream it is recorded on and goes
// when that stream goes (forget), under the same lock as every use of it.
class LoopGate {
 public:
  void launch(int kind, bool adjoint, const LoopLaunch &l, hipStream_t s,
              const LoopDevice &device) {
    std::lock_guard<std::mutex> lock(m_);
    // blocks on one XCD (they go to the XCDs in turn), and whether two share a
    // compute unit
    const int blocks = (l.nblocks + device.xcds - 1) / device.xcds;
    const bool half = device.per_cu[kind] == 2;
    retire(old_);
    retire(before_);
    retire(now_);
    // launches of one stream follow each other: each stream counts once, with
    // its largest.  Beside blocks that need a whole compute unit every block
    // counts as one, since those that could share a unit may have one each.
    std::map<hipStream_t, int> most;
    bool halves = half;
    for (const Entry &e : now_) {
      most[e.stream] = std::max(most[e.stream], e.blocks);
      halves = halves && e.half;
    }
    most[s] = std::max(most[s], blocks);
    int sum = 0;
    for (const auto &m : most) sum += m.second;
    if (sum > (halves ? 2 : 1) * kXcdCus && !now_.empty()) {
      // the launches of now_ themselves wait for those of before_
      old_.insert(old_.end(), before_.begin(), before_.end());
      before_.swap(now_);
      now_.clear();
    }
    for (const Entry &e : before_)
      if (e.stream != s) check(hipStreamWaitEvent(s, e.end, 0), "hipStreamWaitEvent");
    hipEvent_t end;
    std::vector<hipEvent_t> &spare = spare_[s];
    if (spare.empty()) {
      check(hipEventCreateWithFlags(&end, hipEventDisableTiming), "hipEventCreate");
    } else {
      end = spare.back();
      spare.pop_back();
    }
    const hipError_t le = launch_loop(kind, adjoint, l, s);
    const hipError_t re = hipEventRecord(end, s);
    now_.push_back({end, s, blocks, half});
    check(le, "resident time loop");
    check(re, "hipEventRecord");
  }
  // Stream s has been synchronised and is about to be destroyed.
  void forget(hipStream_t s) {
    std::lock_guard<std::mutex> lock(m_);
    for (std::vector<Entry> *list : {&now_, &before_, &old_}) {
      size_t kept = 0;
      for (const Entry &e : *list) {
        if (e.stream == s)
          (void)hipEventDestroy(e.end);
        else
          (*list)[kept++] = e;
      }
      list->resize(kept);
    }
    auto it = spare_.find(s);
    if (it == spare_.end()) return;
    for (hipEvent_t e : it->second) (void)hipEventDestroy(e);
    spare_.erase(it);
  }

 private:
  struct Entry {
    hipEvent_t end;
    hipStream_t stream;
    int blocks;
    bool half;
  };
  static void check(hipError_t e, const char *what) {
    if (e != hipSuccess) throw RuntimeError(std::string(what) + ": " + hipGetErrorString(e));
  }
  void retire(std::vector<Entry> &list) {
    size_t kept = 0;
    for (const Entry &e : list) {
      if (hipEventQuery(e.end) == hipSuccess) {
        spare_[e.stream].push_back(e.end);
      } else {
        (void)hipGetLastError();  // not ready is no error of a later call
        list[kept++] = e;
      }
    }
    list.resize(kept);
  }
  std::mutex m_;
  std::vector<Entry> now_, before_, old_;  // old_: events not yet reusable
  std::map<hipStream_t, std::vector<hipEvent_t>> spare_;
};

LoopGate *loop_gates() {
  static LoopGate *const gates = new LoopGate[kMaxDevices];  // lives until the process ends
  return gates;
}

}  // namespace

hipError_t launch_loop_prepare(LoopArgs *dst, const LoopArgs &a, unsigned *sync,
                               hipStream_t s) {
  hipLaunchKernelGGL(prepare_loop_kernel, dim3(1), dim3(64), 0, s, dst, a, sync);
  return hipGetLastError();
}

int loop_capacity(int kind, int per_unit) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev >= kMaxDevices) return 0;
  const LoopDevice &d = loop_device(dev);
  return d.xcds * kXcdCus * std::min(d.per_cu[kind], per_unit);
}

void loop_gate_forget(hipStream_t s) {
  for (int i = 0; i < kMaxDevices; ++i) loop_gates()[i].forget(s);
}

void gated_launch_loop(int kind, bool adjoint, const LoopLaunch &l, hipStream_t s) {
  int dev = 0;
  if (l.nblocks > loop_capacity(kind) || hipGetDevice(&dev) != hipSuccess || dev >= kMaxDevices)
    throw RuntimeError("resident time loop: the device cannot hold its blocks");
  loop_gates()[dev].launch(kind, adjoint, l, s, loop_device(dev));
}

hipError_t launch_loop(int kind, bool adjoint, const LoopLaunch &l, hipStream_t s) {
  const dim3 grid((unsigned)l.nblocks), block(64 * kLoopKinds[kind].waves);
  auto launch = [&](auto forward, auto backward) {
    hipLaunchKernelGGL(adjoint ? backward : forward, grid, block, 0, s, l);
  };
  switch (kind) {
    case 0: launch(resident_loop<0, false>, resident_loop<0, true>); break;
    case 1: launch(resident_loop<1, false>, resident_loop<1, true>); break;
    case 2: launch(resident_loop<2, false>, resident_loop<2, true>); break;
    case 3: launch(resident_loop<3, false>, resident_loop<3, true>); break;
    case 4: launch(resident_loop<4, false>, resident_loop<4, true>); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace psv
