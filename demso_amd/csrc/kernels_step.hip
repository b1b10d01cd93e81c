// kernels_step.hip -- HIP kernels for hash, cell fill, reorder/cellStart,
// collide and integrate on gfx950.
//
// One lane per particle throughout.  Arithmetic follows the reference kernel
// bodies operation by operation (no FMA contraction in this file: the pragma
// below and -ffp-contract=off), so FP32 results equal the IEEE sequence of
// src/particles_kernel.cuh.  Terms the reference writes with the double
// literals M_PI / 2*M_PI / 1.2 are evaluated in double as C++ promotes them.
#include "contact_math.h"
#include "dem_internal.h"

#include <math.h>

#include <type_traits>

#pragma clang fp contract(off)

namespace dem {
namespace {

__device__ __forceinline__ uint32_t clamp_idx(uint32_t t, uint32_t count) {
  return t < count ? t : count - 1u;
}

__device__ __forceinline__ void clamp_cell(const Instance& in, int& gx, int& gy) {
  gx = min(max(gx, 0), (int)in.grid[0] - 1);
  gy = min(max(gy, 0), (int)in.grid[1] - 1);
}

// seriesAssociation (src/particles_kernel.cuh:36-41).
__device__ __forceinline__ float series(float a, float b) {
  if (a == 0.0f || b == 0.0f) return 0.0f;
  return (a * b) / (a + b);
}

// Radius, mass, inertia of particle i: from its type row, or from the
// per-particle radius with m = (areal*r)*r and I = 2*m*r*r/5 (src/main.cu:193).
template <bool kRadius>
__device__ __forceinline__ void body(const Material& m, const float* __restrict__ radius,
                                     uint32_t i, float& r, float& mass, float& inertia) {
  if (kRadius) {
    r = radius[i];
    mass = (m.areal * r) * r;
    // t / 5 rounded to float: 0.2 is within 2^-53 of 1/5 and t / 5 at least
    // 2^-28 from every midpoint of two floats (and never one), so the
    // product in double rounds to the same float
    inertia = (float)((double)(((2.0f * mass) * r) * r) * 0.2);
  } else {
    r = m.radius;
    mass = m.mass;
    inertia = m.inertia;
  }
}

// pressure += len/(4*M_PI*r*r) in double (src/particles_kernel.cuh:284, 339, 433);
// den is 4*M_PI*r*r evaluated once per particle in the same order.
__device__ __forceinline__ float add_pressure(float p, float len, double den) {
  return (float)((double)p + (double)len / den);
}

// RN(sqrt(x)) < m, the Coulomb test of the shear law (length(Ftrial) < Ftmax,
// src/particles_kernel.cuh:295), for x a sum of two
// float squares (+0 or more, or NaN).  RN is monotone and the root of a
// float is never a rounding midpoint, so the test is x < (m-)^2, m- the
// midpoint below m, which lies in [m^2 (1 - 2^-23), m^2).  For m in
// [2^-63, 2^63] t = RN(m m) is a normal float within 2^-24 of m^2, so
// x < RN(t (1 - 2^-20)) proves the test true and x > RN(t (1 + 2^-20))
// proves it false; only between the two (or for other m, or NaN) is the
// correctly rounded root taken.
__device__ __forceinline__ bool sqrt_below(float x, float m) {
  if (m >= 0x1p-63f && m <= 0x1p63f) {
    const float t = m * m;
    if (x < t * (1.0f - 0x1p-20f)) return true;
    if (x > t * (1.0f + 0x1p-20f)) return false;
  }
  return sqrtf(x) < m;
}

__device__ __forceinline__ double pressure_den(float r) {
  return 4 * M_PI * (double)r * (double)r;
}

// ---------------------------------------------------------------- calcHash --
// Cell key of one particle: calcGridHash (src/particles_kernel.cuh:123-130)
// with the instance's key base; clamped or wrapped as the flags say.
__device__ __forceinline__ uint32_t cell_key_in(const StepConst& c, const Instance& in, float2 p) {
  int gx, gy;
  grid_pos(in, p, gx, gy);
  uint32_t cx, cy;
  if (c.flags & DEM_GRID_CLAMP) {
    clamp_cell(in, gx, gy);
    cx = (uint32_t)gx;
    cy = (uint32_t)gy;
  } else {
    cx = (uint32_t)gx & (in.grid[0] - 1u);
    cy = (uint32_t)gy & (in.grid[1] - 1u);
  }
  return in.cell_base + cy * in.grid[0] + cx;
}

template <bool kMulti>
__device__ __forceinline__ uint32_t cell_key(const StepConst& c, float2 p, const uint32_t* __restrict__ type,
                                             uint32_t i) {
  const Instance in =
      kMulti ? c.inst[clamp_idx(c.mat[clamp_idx(type[i], c.num_types)].inst, c.num_instances)] : c.inst0;
  return cell_key_in(c, in, p);
}

// calcHashD (src/particles_kernel.cuh:133-151).  kPer particles a lane: a
// block covers kPer * blockDim consecutive particles, lane t taking t,
// t + blockDim, ... (each pass over the block's lanes stays coalesced).
template <bool kMulti, int kPer>
__global__ __launch_bounds__(256) void k_hash(StepConst c, const float2* __restrict__ pos,
                                              const uint32_t* __restrict__ type,
                                              uint32_t* __restrict__ hash,
                                              uint32_t* __restrict__ index, uint32_t n) {
  const uint32_t base = blockIdx.x * c.block * kPer + threadIdx.x;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const uint32_t i = base + (uint32_t)k * c.block;
    if (i < n) {
      hash[i] = cell_key<kMulti>(c, pos[i], type, i);
      index[i] = i;
    }
  }
}

// -------------------------------------------------------------- cell fill --
// cudaMemset(cellStart, 0xff) of src/functions.cu:371 as a kernel (a memset
// node in a captured graph is avoided on purpose).
__global__ __launch_bounds__(256) void k_fill(uint32_t* __restrict__ p, uint32_t v, uint32_t n, int vec) {
  const uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) * 4u;
  if (i >= n) return;
  if (vec && i + 3u < n) {
    *reinterpret_cast<uint4*>(p + i) = make_uint4(v, v, v, v);
  } else {
    for (uint32_t k = i; k < n && k < i + 4u; ++k) p[k] = v;
  }
}

// --------------------------------------------------------------- reorder --
// reorderDataAndFindCellStartD (src/particles_kernel.cuh:156-233).  The
// previous key is read from global memory (it is in the same cache line for
// all lanes but lane 0).  Keys >= num_cells, indices >= n and IDs >= n are
// skipped instead of being written out of bounds.  kFull = false gathers the
// positions and the per-particle constants only: the owned simulation's step
// reads velocity, angle and spin through the sorted index instead (collide
// for its own particle and its contacts, integrate for every particle).
template <bool kRadius, bool kFull, int kPer>
__global__ __launch_bounds__(256) void k_reorder(
    uint32_t* __restrict__ cell_start, uint32_t* __restrict__ cell_end, float2* __restrict__ s_pos,
    float2* __restrict__ s_vel, float* __restrict__ s_theta, float* __restrict__ s_omega,
    uint32_t* __restrict__ s_id, uint32_t* __restrict__ s_loc, uint32_t* __restrict__ s_type,
    float* __restrict__ s_radius, const uint32_t* __restrict__ hash,
    const uint32_t* __restrict__ index, const float2* __restrict__ o_pos,
    const float2* __restrict__ o_vel, const float* __restrict__ o_theta,
    const float* __restrict__ o_omega, const uint32_t* __restrict__ o_id,
    const uint32_t* __restrict__ o_type, const float* __restrict__ o_radius, uint32_t n,
    uint32_t num_cells) {
  // kPer particles a lane, as k_hash
  const uint32_t base = blockIdx.x * blockDim.x * kPer + threadIdx.x;
#pragma unroll
  for (int kk = 0; kk < kPer; ++kk) {
    const uint32_t i = base + (uint32_t)kk * blockDim.x;
    if (i >= n) continue;
    const uint32_t h = hash[i];
    if (i == 0) {
      if (h < num_cells) cell_start[h] = 0;
    } else {
      const uint32_t hp = hash[i - 1];
      if (h != hp) {
        if (h < num_cells) cell_start[h] = i;
        if (hp < num_cells) cell_end[hp] = i;
      }
    }
    if (i == n - 1 && h < num_cells) cell_end[h] = n;

    const uint32_t k = index[i];
    if (k >= n) continue;
    s_pos[i] = o_pos[k];
    if (kFull) {
      s_vel[i] = o_vel[k];
      s_theta[i] = o_theta[k];
      s_omega[i] = o_omega[k];
    }
    const uint32_t id = o_id[k];
    s_id[i] = id;
    if (id < n) s_loc[id] = i;
    s_type[i] = o_type[k];
    if (kRadius) s_radius[i] = o_radius[k];
  }
}

// --------------------------------------------------------------- collide --
// collideD (src/particles_kernel.cuh:459-549) with collideCell (:345-385),
// collideSpheres (:235-307) and attractSpheres (:310-342) inlined.
//
// The kernel's cost is per candidate (instructions and the latency of the
// dependent loads), so the candidate loop is kept lean:
//  * the three cells of a row are consecutive keys, so their candidates are
//    one contiguous range of the sorted arrays; collideCell returns one
//    partial float2 per cell that collideD adds up, so the running partial
//    sum is flushed into the total when a candidate that may exert a force
//    lies in a later cell (RowSum; flushing only there changes nothing, as
//    candidates without force add +0 and the sums start at +0 and never
//    become -0).  Where a wrapping grid makes the row non-contiguous (edge
//    columns), the row's three cells are walked one by one in the reference
//    order;
//  * most candidates are not in contact: d2 = rx*rx+ry*ry is the float the
//    reference takes sqrtf of, and if d2 > fl(R*R)*(1+2^-20) then
//    sqrtf(d2) >= R for certain (fl(R*R)*(1+2^-20) exceeds the square of
//    the midpoint between R and its predecessor while R*R is a normal float,
//    i.e. R >= 2^-63; smaller R always takes the exact path), so the correctly rounded
//    sqrt and the contact law run only for candidates that may touch; the
//    contact decision itself is the reference's dist < R;
//  * the neighbour's velocity, spin and material are loaded only for actual
//    contacts, except in the plain mode, which loads them with the position
//    (the reference loads them for every candidate; the values used are the
//    same).
constexpr uint32_t kNoBoundary = 0xFFFFFFFFu;

struct PairCtx {
  float2 p, v;
  float w, rA, dt;
  double den;
  double rden;  // RN(1/den), for the contact-list mode's pressure terms
  float attract;  // the particle's material's coefficient
  uint32_t tA;
};

// The pressure term with the particle's rounded reciprocal y = RN(1/den) and
// two fused corrections: q1 = RN(a y) (off by more than an ulp for about 1%
// of inputs), q2 = RN(q1 + RN(a - q1 den) y) (within a tiny fraction of an
// ulp of a/den, so faithful), q3 = RN(q2 + (a - q2 den) y), where the
// remainder of the faithful q2 is exact.  q3 is the correctly rounded a/den
// (Markstein's theorem for y = RN(1/den) and a faithful quotient: the
// remainder and den * ulp/2 lie on the grid ulp(den) ulp/2 and differ from
// ulp/(2y) by less than one step of it, so q2 + r y and a/den lie on the same
// side of every rounding midpoint, and a/den is never one).  a is a float
// length and den = 4 pi r^2 of a float r, so no step overflows or underflows
// in double.  The remainder is not finite only where the length is not or den
// is zero or infinite, and there a y already is a / den.  Five FP64
// operations per contact instead of a division sequence.
__device__ __forceinline__ double pressure_quotient(float len, double den, double rden) {
  const double a = (double)len;
  double qd = a * rden;
  const double rem = fma(-qd, den, a);
  if (__builtin_expect(__builtin_isfinite(rem), 1)) {
    qd = fma(rem, rden, qd);
    qd = fma(fma(-qd, den, a), rden, qd);
  }
  return qd;
}

__device__ __forceinline__ float add_pressure_recip(float p, float len, double den, double rden) {
  return (float)((double)p + pressure_quotient(len, den, rden));
}

// A distance's root and the unit vector (rx, ry) / dist, with kFast by root
// and quotients (the same floats).
template <bool kFast>
__device__ __forceinline__ float length_of(float d2, float& y) {
  if constexpr (kFast) return root(d2, y);
  else return sqrtf(d2);
}
template <bool kFast>
__device__ __forceinline__ void unit(float rx, float ry, float dist, float y, float& nx, float& ny) {
  if constexpr (kFast) {
    quotients(rx, ry, dist, y, nx, ny);
  } else {
    nx = rx / dist;
    ny = ry / dist;
  }
}

// collideSpheres' contact law (src/particles_kernel.cuh:255-303) for a
// partner B of material tB at the direction (nx, ny) and distance dist < R:
// the force on A as collideSpheres returns it (ffx, ffy), the length of its
// normal part (the pressure term's numerator) as the return value, and the
// friction moment term mterm (+0 without friction; the moment is a sum that
// starts at +0 and is never -0, so adding +0 leaves it unchanged).
template <bool kFast>
__device__ __forceinline__ float contact_terms(const StepConst& c, const PairCtx& q, float nx, float ny, float dist,
                                               float R, float rB, uint32_t tB, float2 vB, float wB, float& ffx,
                                               float& ffy, float& mterm) {
  const float4 pr = c.pair[q.tA * c.num_types + tB];
  const float kn = pr.x, kt = pr.y, cn = pr.z, mu = pr.w;
  const float tx = -ny, ty = nx;
  const float rvx = vB.x - q.v.x, rvy = vB.y - q.v.y;
  const float vn = rvx * nx + rvy * ny;
  const float vtx = rvx - vn * nx, vty = rvy - vn * ny;
  const float s = -kn * (R - dist);
  ffx = s * nx;
  ffy = s * ny;
  if (vn < 0.0f) {
    const float s2 = cn * vn;
    ffx += s2 * nx;
    ffy += s2 * ny;
  }
  float y;
  const float flen = length_of<kFast>(ffx * ffx + ffy * ffy, y);
  mterm = 0.0f;
  if (mu != 0.0f) {
    const float sr = q.rA * q.w + rB * wB;
    const float cvx = vtx - sr * tx, cvy = vty - sr * ty;
    float ftx = (kt * cvx) * q.dt, fty = (kt * cvy) * q.dt;
    const float ftmax = mu * flen;
    if (!sqrt_below(ftx * ftx + fty * fty, ftmax)) {
      const float cl = length_of<kFast>(cvx * cvx + cvy * cvy, y);
      unit<kFast>(ftmax * cvx, ftmax * cvy, cl, y, ftx, fty);
    }
    ffx += ftx;
    ffy += fty;
    mterm = q.rA * (ftx * tx + fty * ty);
  }
  return flen;
}

// The contact law with its pressure term added to pres and its moment term
// to moment.
template <bool kFast = false>
__device__ __forceinline__ void contact_force(const StepConst& c, const PairCtx& q, float nx, float ny, float dist,
                                              float R, float rB, uint32_t tB, float2 vB, float wB, float& ffx,
                                              float& ffy, float& moment, float& pres) {
  float mterm;
  const float flen = contact_terms<kFast>(c, q, nx, ny, dist, R, rB, tB, vB, wB, ffx, ffy, mterm);
  pres = kFast ? add_pressure_recip(pres, flen, q.den, q.rden) : add_pressure(pres, flen, q.den);
  moment += mterm;
}

// attractSpheres (src/particles_kernel.cuh:310-342) for a partner with
// attraction coefficient aB: the force on A and its pressure term.
template <bool kFast = false>
__device__ __forceinline__ void attract_force(const PairCtx& q, float nx, float ny, float dist, float rB, float aB,
                                              float& afx, float& afy, float& pres) {
  const float aA = q.attract;
  const float adA = (float)((double)(q.rA * 2.0f) * 1.2);
  const float adB = (float)((double)(rB * 2.0f) * 1.2);
  afx = 0.0f;
  afy = 0.0f;
  if (dist < adA) {
    const float s = aA * (adA - dist);
    afx += s * nx;
    afy += s * ny;
  }
  if (dist < adB) {
    const float s = aB * (adB - dist);
    afx += s * nx;
    afy += s * ny;
  }
  float y;
  const float len = length_of<kFast>(afx * afx + afy * afy, y);
  pres = kFast ? add_pressure_recip(pres, len, q.den, q.rden) : add_pressure(pres, len, q.den);
}

// Velocity and spin of the sorted particles: vel[j], omega[j], or with a
// gather index vel[gat[j]], omega[gat[j]] (the previous step's arrays,
// before the sort).
// Element i of an array.  kOff32: addressed by a 32-bit byte offset from the
// array's base, which the loads take as a scalar base plus one 32-bit lane
// register (64-bit address arithmetic per load otherwise); only for arrays
// of at most 4 GiB, which the launcher checks.
template <bool kOff32, class T>
__device__ __forceinline__ const T& ld(const T* __restrict__ base, uint32_t i) {
  if constexpr (kOff32)
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + i * (uint32_t)sizeof(T));
  else
    return base[i];
}

struct Dyn {
  const float2* __restrict__ vel;
  const float* __restrict__ omega;
  const uint32_t* __restrict__ gat;
  template <bool kOff32>
  __device__ __forceinline__ uint32_t at(uint32_t j) const { return gat ? ld<kOff32>(gat, j) : j; }
};

// A neighbour candidate as the pair law reads it.  With kDyn its velocity,
// spin and material row are loaded together with its position and radius
// (one dependent load fewer for every contact, three more registers);
// without, they are loaded only for candidates that touch.
struct Cand {
  float2 p;
  float r;
  uint32_t t;
  float2 v;
  float w;
};

// The row's per-cell partial sum: collideCell's sums start at +0 for every
// cell and collideD adds them in cell order.  Candidates that exert no force
// add +0, which leaves a partial sum unchanged (a sum that starts at +0 is
// never -0), so the partial sum is flushed into the total only where a
// candidate that may exert a force lies in a later cell of the row than the
// sum's (cell index (j >= b0) + (j >= b1), the row's cell ends), and at the
// row's end: the same additions in the same order as flushing at every cell
// end.
struct RowSum {
  float cfx = 0.0f, cfy = 0.0f;
  uint32_t cell = 0, b0, b1;
  __device__ __forceinline__ void at(uint32_t j, float& fx, float& fy) {
    const uint32_t k = (uint32_t)(j >= b0) + (uint32_t)(j >= b1);
    if (k != cell) {
      fx += cfx;
      fy += cfy;
      cfx = 0.0f;
      cfy = 0.0f;
      cell = k;
    }
  }
};

template <bool kRadius, bool kOne, bool kDyn, bool kO>
__device__ __forceinline__ void candidate_at(const StepConst& c, const PairCtx& q, uint32_t j, bool self,
                                             const Cand& b, const Dyn& d, const uint32_t* __restrict__ type,
                                             RowSum& rsum, float& fx, float& fy, float& moment, float& pres) {
  const float rx = b.p.x - q.p.x, ry = b.p.y - q.p.y;
  const float d2 = rx * rx + ry * ry;
  const float R = q.rA + b.r;
  const bool maybe = !(d2 > (R * R) * 1.00000095367431640625f) || R < 1.0842022e-19f;
  // the particle itself is skipped (collideCell's j != index test)
  if (self || !(maybe || c.attract)) return;
  rsum.at(j, fx, fy);
  float& cfx = rsum.cfx;
  float& cfy = rsum.cfy;
  const float dist = sqrtf(d2);
  const float rB = b.r;
  uint32_t tB = b.t;
  if (kRadius && !kOne && !kDyn) tB = clamp_idx(ld<kO>(type, j), c.num_types);
  if (dist < R) {
    float ffx, ffy;
    float2 vB;
    float wB;
    if (kDyn) {
      vB = b.v;
      wB = b.w;
    } else {
      const uint32_t jv = d.at<kO>(j);
      vB = ld<kO>(d.vel, jv);
      wB = ld<kO>(d.omega, jv);
    }
    contact_force(c, q, rx / dist, ry / dist, dist, R, rB, tB, vB, wB, ffx, ffy, moment, pres);
    cfx += ffx;
    cfy += ffy;
  }
  if (c.attract) {
    float afx, afy;
    attract_force(q, rx / dist, ry / dist, dist, rB, c.mat[tB].attract, afx, afy, pres);
    cfx += afx;
    cfy += afy;
  }
}

// A candidate that the contact-list walk marked (its velocity, spin and
// material row loaded): the same sums, without the test that the mark was.
__device__ __forceinline__ void listed_pair(const StepConst& c, const PairCtx& q, const Cand& b, float& cfx,
                                            float& cfy, float& moment, float& pres) {
  const float rx = b.p.x - q.p.x, ry = b.p.y - q.p.y;
  const float R = q.rA + b.r;
  float y, nx, ny;
  const float dist = root(rx * rx + ry * ry, y);
  if (!(dist < R || c.attract)) return;
  quotients(rx, ry, dist, y, nx, ny);
  if (dist < R) {
    float ffx, ffy;
    contact_force<true>(c, q, nx, ny, dist, R, b.r, b.t, b.v, b.w, ffx, ffy, moment, pres);
    cfx += ffx;
    cfy += ffy;
  }
  if (c.attract) {
    float afx, afy;
    attract_force<true>(q, nx, ny, dist, b.r, c.mat[b.t].attract, afx, afy, pres);
    cfx += afx;
    cfy += afy;
  }
}

// The pair with the controlled particle (src/particles_kernel.cuh:527-541,
// USE_ATOMIC 0): f = collideSpheres + attractSpheres, summed on its own and
// then added to the particle's force and moment; the reaction on the
// controlled particle, -f and -m / rA * rC, goes to per-particle vectors.
__device__ __forceinline__ void control_pair(const StepConst& c, const PairCtx& q, const dem_controlled& C,
                                             float& fx, float& fy, float& moment, float& pres, float& react_x,
                                             float& react_y, float& react_m) {
  const uint32_t tC = clamp_idx(C.type, c.num_types);
  const float rC = c.mat[tC].radius;
  const float rx = C.pos[0] - q.p.x, ry = C.pos[1] - q.p.y;
  const float dist = sqrtf(rx * rx + ry * ry);
  const float R = q.rA + rC;
  float m = 0.0f, f_x = 0.0f, f_y = 0.0f;
  if (dist < R) {
    float mterm = 0.0f;
    contact_force(c, q, rx / dist, ry / dist, dist, R, rC, tC, make_float2(C.vel[0], C.vel[1]), C.omega, f_x, f_y,
                  mterm, pres);
    m = m + mterm;  // collideSpheres adds into the caller's m (0)
  }
  if (c.attract) {
    float afx, afy;
    attract_force(q, rx / dist, ry / dist, dist, rC, c.mat[tC].attract, afx, afy, pres);
    f_x += afx;
    f_y += afy;
  }
  fx += f_x;
  fy += f_y;
  moment += m;
  react_x = -f_x;
  react_y = -f_y;
  react_m = -m / q.rA * rC;
}

// Candidate j's position and radius (and, without a radius array, its
// material row), plus with kDyn its velocity, spin and material row.
// (kOne: every particle has material row 0, so no type is read.)
template <bool kRadius, bool kOne, bool kDyn, bool kO>
__device__ __forceinline__ void candidate_load(const StepConst& c, uint32_t j, const float2* __restrict__ pos,
                                               const uint32_t* __restrict__ type, const float* __restrict__ radius,
                                               const Dyn& d, Cand& b) {
  b.p = ld<kO>(pos, j);
  if (kRadius) {
    b.r = ld<kO>(radius, j);
    b.t = kDyn && !kOne ? clamp_idx(ld<kO>(type, j), c.num_types) : 0u;
  } else {
    b.t = kOne ? 0u : clamp_idx(ld<kO>(type, j), c.num_types);
    b.r = c.mat[b.t].radius;
  }
  if (kDyn) {
    const uint32_t jv = d.at<kO>(j);
    b.v = ld<kO>(d.vel, jv);
    b.w = ld<kO>(d.omega, jv);
  }
}

template <bool kRadius, bool kOne, bool kDyn, bool kO>
__device__ __forceinline__ void candidate(const StepConst& c, const PairCtx& q, uint32_t j, bool self,
                                          const float2* __restrict__ pos, const Dyn& d,
                                          const uint32_t* __restrict__ type, const float* __restrict__ radius,
                                          RowSum& rsum, float& fx, float& fy, float& moment, float& pres) {
  Cand b;
  candidate_load<kRadius, kOne, kDyn, kO>(c, j, pos, type, radius, d, b);
  candidate_at<kRadius, kOne, kDyn, kO>(c, q, j, self, b, d, type, rsum, fx, fy, moment, pres);
}

// Forces on sorted particle i from its 3x3 cell neighbourhood (the body of
// collideD, src/particles_kernel.cuh:459-549): sum of the pair forces fx,
// fy, the moment and the pressure, plus the particle's own radius, mass,
// inertia and material (for integrate).
struct Own {
  float r, mass, inertia;
  uint32_t t;
  float2 p, v;
  float w;
  uint32_t cell;  // the key of the particle's cell
};

// Candidate modes of the collide kernels: kPlain walks each row's candidates
// one load at a time (each candidate's velocity and spin loaded with its
// position); kPrefetch loads each one iteration ahead; kBatch loads the first
// candidate of all three rows at once before walking them (three loads in
// flight); kList first walks the rows testing only position and radius and
// sets a bit per candidate that may touch, then runs the contact law over the
// set bits of all three rows, so a wave executes the contact law as often as
// its busiest lane has contacts instead of at every candidate where some lane
// has one.  The order of the sums is the same in every mode.  Preloading
// two or three candidates a row needs 73 or 81 VGPRs (6 waves per SIMD
// instead of 8) and was slower.
constexpr int kPlain = 0, kPrefetch = 1, kBatch = 2, kList = 3;
constexpr int kBatchN = 1;

// Material layouts of the kernels: one material row (no type is read), one
// instance with several rows, or an ensemble of instances.
constexpr int kOneMat = 0, kManyMat = 1, kInstances = 2;

// The radii of the contact-list walk's marks are taken this much longer.
constexpr float kReach = 1.0f + 0x1p-18f;

// w[y] = 2 w[y] + !(x[y] > limit) for the three rows: each comparison's carry
// is added with the shift (the compiler takes a select and a shift-or).  A
// lane mask that a vector instruction wrote may be read by another only two
// instructions later on gfx950, so the three comparisons come first.
__device__ __forceinline__ void shift_in(uint32_t (&w)[3], const float (&x)[3], float limit) {
  uint64_t m0, m1, m2;
  asm("v_cmp_ngt_f32_e64 %3, %6, %9\n\t"
      "v_cmp_ngt_f32_e64 %4, %7, %9\n\t"
      "v_cmp_ngt_f32_e64 %5, %8, %9\n\t"
      "v_addc_co_u32_e64 %0, vcc, %0, %0, %3\n\t"
      "v_addc_co_u32_e64 %1, vcc, %1, %1, %4\n\t"
      "v_addc_co_u32_e64 %2, vcc, %2, %2, %5"
      : "+&v"(w[0]), "+&v"(w[1]), "+&v"(w[2]), "=&s"(m0), "=&s"(m1), "=&s"(m2)
      : "v"(x[0]), "v"(x[1]), "v"(x[2]), "s"(limit)
      : "vcc");
}

// The contact-list walk's windows, one set a wave in LDS: the positions and
// radii of the sorted particles [w0, w1) that hold the candidates of all the
// wave's lanes in a neighbour row (the lanes' ranges follow each other in
// sorted order, so a row's window is a little longer than a wave).  Loaded
// once, coalesced; each lane then walks its candidates in LDS.  The vector
// cache looks up one line a cycle, and walking the candidates through it
// (585 lookups a wave at 4M settling discs, where it was busy 93% of the
// kernel's time) bound the kernel: with the windows it took 50 us there
// (59), 150 us on the 4M dense pack (172), 136 us on the 8.2M-disc ensemble
// (149).  Now vector instructions bound it: with one word of marks, the rows'
// ranges by minimum and maximum and the short roots, quotients and cells, 53
// us there (54 before, on the same machine) with 381 instructions a wave, 128
// us on the dense pack (151) with 1,435, 143 us on the ensemble (152) with 478.
// Three rows of kWindow entries, then kWindowSlack more, as a lane with few
// candidates reads on past its row's.
// An entry's three words lie together, so a lane's walk has one address a row
// (and no bank conflict, a wave's lanes being 3 words apart).  Eight waves a
// SIMD fit (32 x 5,120 bytes of 160 KB).
constexpr uint32_t kWindow = 128, kWindowSlack = 32;
struct WindowEntry {
  float x, y, r;
};
struct WaveWindow {
  WindowEntry at[3 * kWindow + kWindowSlack];
};
static_assert(sizeof(WaveWindow) <= 5120, "eight waves a SIMD");

// This wave's windows in the block's dynamic LDS (window_bytes(block)).
extern __shared__ __attribute__((aligned(16))) unsigned char dem_windows[];
__device__ __forceinline__ WaveWindow* wave_window() {
  return reinterpret_cast<WaveWindow*>(dem_windows) + __builtin_amdgcn_readfirstlane(threadIdx.x / (uint32_t)kWave);
}
inline size_t window_bytes(int mode, int block) {
  return mode == kList ? sizeof(WaveWindow) * (size_t)((block + kWave - 1) / kWave) : 0;
}

// kUni: every lane of the call has material row t_uni (a wave-uniform value,
// so the material row and the instance geometry are scalar loads and the
// grid arithmetic scalar).
template <bool kRadius, int kMat, int kMode, bool kControl, bool kO, bool kUni = false, bool kEarly = false>
__device__ __forceinline__ void collide_particle(const StepConst& c, uint32_t i, const float2* __restrict__ pos,
                                                 const Dyn& d, const uint32_t* __restrict__ type,
                                                 const float* __restrict__ radius,
                                                 const uint32_t* __restrict__ cell_start,
                                                 const uint32_t* __restrict__ cell_end, uint32_t n, Own& own,
                                                 const ControlOut& ctl, float& fx_out, float& fy_out,
                                                 float& moment_out, float& pres_out, uint32_t t_uni = 0,
                                                 WaveWindow* win = nullptr) {
  constexpr bool kMulti = kMat == kInstances, kOne = kMat == kOneMat;
  PairCtx q;
  own.t = kOne ? 0u : (kUni ? t_uni : clamp_idx(type[i], c.num_types));
  q.tA = own.t;
  const Material mA = c.mat[own.t];
  q.attract = mA.attract;
  const Instance in = kMulti ? c.inst[clamp_idx(mA.inst, c.num_instances)] : c.inst0;
  const float r_i = kRadius ? ld<kO>(radius, i) : 0.0f;
  body<kRadius>(mA, &r_i, 0u, q.rA, own.mass, own.inertia);
  own.r = q.rA;
  q.p = ld<kO>(pos, i);
  // The particle's own velocity and spin feed only the contact law (and the
  // fused kernel's integrate): the contact-list walk loads them once it has
  // marked a candidate (or at the end, where a caller uses them), the other
  // modes, and with kEarly the list too, up front.
  bool have_dyn = false;
  auto load_own_dyn = [&]() {
    const uint32_t iv = d.at<kO>(i);
    q.v = ld<kO>(d.vel, iv);
    q.w = ld<kO>(d.omega, iv);
    q.den = pressure_den(q.rA);
    have_dyn = true;
  };
  if (kMode != kList || kControl || kEarly) load_own_dyn();
  own.p = q.p;
  q.dt = c.dt;
  const bool clamp = c.flags & DEM_GRID_CLAMP;
  const int G0 = (int)in.grid[0], G1 = (int)in.grid[1];
  float fx = 0.0f, fy = 0.0f, moment = 0.0f, pres = 0.0f;
  int gx, gy;
  grid_pos(in, q.p, gx, gy);
  if (clamp) clamp_cell(in, gx, gy);
  // x columns of a row: clamp -> out-of-range skipped; wrap -> & (G-1)
  const bool vx0 = !clamp || gx > 0, vx2 = !clamp || gx < G0 - 1;
  const uint32_t x0 = ((uint32_t)gx - 1u) & (clamp ? 0xFFFFFFFFu : (uint32_t)G0 - 1u);
  const uint32_t x1 = clamp ? (uint32_t)gx : ((uint32_t)gx & ((uint32_t)G0 - 1u));
  const uint32_t x2 = ((uint32_t)gx + 1u) & (clamp ? 0xFFFFFFFFu : (uint32_t)G0 - 1u);
  own.cell = in.cell_base + (clamp ? (uint32_t)gy : (uint32_t)gy & ((uint32_t)G1 - 1u)) * (uint32_t)G0 + x1;
  // a wrap that moves a column to the other edge breaks key contiguity
  bool by_cell = !(clamp || (x0 + 1u == x1 && x1 + 1u == x2));
  if (!by_cell) {
    // The usual case: every row's three cells are consecutive keys, so a row
    // is one candidate range [rs, re) with the cell ends b0, b1 inside it.
    // The ranges of all three rows are loaded first (their loads overlap),
    // and each candidate's position and radius are fetched one iteration
    // ahead; the summation order is unchanged.
    // The cells' starts are increasing, an empty cell's is the largest word
    // and its end is taken as 0, so the range is the least start and the
    // largest end.  b0 and b1, where the second and third cell begin, are the
    // range's start for empty cells before them (a flush of an empty sum
    // changes nothing).  A column or row outside a clamped grid stands in as
    // the centre one: a cell read twice changes neither the range nor what
    // lies in which of two cells, a row's range is emptied.
    uint32_t rs[3], re[3], b0[3], b1[3];
    const uint32_t cyc = clamp ? (uint32_t)gy : (uint32_t)gy & ((uint32_t)G1 - 1u);
    const bool top = cyc == 0u, bottom = cyc == (uint32_t)G1 - 1u;
    const uint32_t around = clamp ? 0u : ((uint32_t)G1 - 1u) * (uint32_t)G0;
    const uint32_t row1 = in.cell_base + cyc * (uint32_t)G0;
    const uint32_t rows[3] = {top ? row1 + around : row1 - (uint32_t)G0, row1,
                              bottom ? row1 - around : row1 + (uint32_t)G0};
    const uint32_t xl = vx0 ? x0 : x1, xr = vx2 ? x2 : x1;
#pragma unroll
    for (int y = 0; y < 3; ++y) {
      const uint32_t s0 = ld<kO>(cell_start, rows[y] + xl), s1 = ld<kO>(cell_start, rows[y] + x1),
                     s2 = ld<kO>(cell_start, rows[y] + xr);
      const uint32_t e0r = ld<kO>(cell_end, rows[y] + xl), e1r = ld<kO>(cell_end, rows[y] + x1),
                     e2r = ld<kO>(cell_end, rows[y] + xr);
      const uint32_t e0 = s0 != kEmpty ? e0r : 0u, e1 = s1 != kEmpty ? e1r : 0u, e2 = s2 != kEmpty ? e2r : 0u;
      re[y] = min(max(max(e0, e1), e2), n);
      if (y == 0) re[y] = clamp && top ? 0u : re[y];
      if (y == 2) re[y] = clamp && bottom ? 0u : re[y];
      rs[y] = min(min(min(s0, s1), s2), re[y]);
      b0[y] = max(e0, rs[y]);
      b1[y] = max(e1, b0[y]);
    }
    Cand cb[3][kBatchN];
    if (kMode == kBatch) {
      // index 0 stands in for a candidate past the row's end (never used)
#pragma unroll
      for (int y = 0; y < 3; ++y)
#pragma unroll
        for (int k = 0; k < kBatchN; ++k) {
          const uint32_t j = rs[y] + (uint32_t)k;
          candidate_load<kRadius, kOne, false, kO>(c, j < re[y] ? j : 0u, pos, type, radius, d, cb[y][k]);
        }
    }
    const uint32_t len[3] = {re[0] - rs[0], re[1] - rs[1], re[2] - rs[2]};
    if (kMode == kList && (!c.attract || fabsf(q.rA) > 0.0f) && max(len[0], max(len[1], len[2])) <= 0xFFFFu) {
      // First one bit per candidate that may exert a force (from position and
      // radius), then the law over the set bits in the rows' order, so a wave
      // runs the law as often as its busiest lane has contacts.  Candidates
      // that exert no force add +0, so skipping them leaves every sum
      // unchanged; a cell's partial sum is flushed when the walk moves on to a
      // later cell.  (An attracting candidate out of reach adds +0 / den to
      // the pressure: +0 for a radius; the 16,290-disc pile's fused step takes
      // 15.7 us this way, 42 one candidate at a time.)
      // The three rows are walked together, from the wave's windows in LDS
      // (WaveWindow) or from global memory.  The walk is most of the kernel's
      // instructions on sparse states, so each candidate costs as few as
      // possible: a mark is one comparison shifted into the row's word
      // (candidate k at bit 31 - k), and the particle itself and the places
      // past the row's end are cleared afterwards.  A mark may be set without
      // a contact, never the other way round: where a contact is, the law's
      // d2 < R^2; d2 here (one rounding less) is within 2^-22 of it, and R
      // here is R (1 + 2^-18) within 2^-23, so d2 - R^2 rounds to a negative
      // number, or to at most 2^-125 where the squares underflow; NaN is
      // marked.
      // where a row's second and third cells begin, 16 bits each
      uint32_t cut[3];
#pragma unroll
      for (int y = 0; y < 3; ++y) cut[y] = (b0[y] - rs[y]) | (b1[y] - rs[y]) << 16;
      // At most 2^-125 where a candidate at p with radius r may exert a force.
      const float reach = q.rA * kReach;
      auto beyond = [&](auto attract, float x, float y, float r) {
        const float rx = x - q.p.x, ry = y - q.p.y;
        const float d2 = __builtin_fmaf(ry, ry, rx * rx);
        float R = __builtin_fmaf(r, kReach, reach);
        // (attractSpheres reaches 2.4 times either radius)
        if constexpr (attract) R = fmaxf(R, (2.4f * kReach) * fmaxf(q.rA, r));
        return __builtin_fmaf(-R, R, d2);
      };
      // The windows, where the whole wave is here and every lane's ranges
      // lie in them (rows far apart, as around wide empty spaces, do not fit
      // and are walked in global memory).
      uint32_t w0[3], w1[3];
      uint64_t outside = ~__ballot(win != nullptr);
#pragma unroll
      for (int y = 0; y < 3; ++y) {
        // (rows that are empty in the whole wave: any lane's range is empty)
        const uint64_t some = __ballot(len[y] != 0u);
        w0[y] = (uint32_t)__builtin_amdgcn_readlane((int)rs[y], __builtin_ctzll(some | 1ull << 63));
        w1[y] = (uint32_t)__builtin_amdgcn_readlane((int)re[y], 63 - __builtin_clzll(some | 1ull));
        w1[y] = some ? w1[y] : w0[y];
        outside |= (__ballot(rs[y] < w0[y]) | __ballot(re[y] > w1[y])) & some;
        outside |= w1[y] - w0[y] > kWindow ? ~0ull : 0ull;
      }
      const bool in_win = outside == 0;
      if (in_win) {
        const uint32_t lane = __lane_id();
        auto put = [&](uint32_t e, const Cand& b) {
          win->at[e].x = b.p.x;
          win->at[e].y = b.p.y;
          win->at[e].r = b.r;
        };
        auto stage = [&](uint32_t e) {
          Cand b[3];
#pragma unroll
          for (int y = 0; y < 3; ++y)
            if (w0[y] + e < w1[y]) candidate_load<kRadius, kOne, false, kO>(c, w0[y] + e, pos, type, radius, d, b[y]);
#pragma unroll
          for (int y = 0; y < 3; ++y)
            if (w0[y] + e < w1[y]) put((uint32_t)y * kWindow + e, b[y]);
        };
        stage(lane);
        // what is left of the three windows: usually a few places each, taken
        // by a quarter of the wave a row
        constexpr uint32_t kQuarter = (uint32_t)kWave / 4u;
        auto longer = [&](uint32_t k) { return (w1[0] - w0[0] > k) | (w1[1] - w0[1] > k) | (w1[2] - w0[2] > k); };
        if (longer((uint32_t)kWave + kQuarter)) {
          stage((uint32_t)kWave + lane);
        } else if (longer((uint32_t)kWave)) {
          const uint32_t y = lane / kQuarter, e = (uint32_t)kWave + lane % kQuarter;
          const uint32_t a = y == 0u ? w0[0] : (y == 1u ? w0[1] : w0[2]), z = y == 0u ? w1[0] : (y == 1u ? w1[1] : w1[2]);
          if (y < 3u && a + e < z) {
            Cand b;
            candidate_load<kRadius, kOne, false, kO>(c, a + e, pos, type, radius, d, b);
            put(y * kWindow + e, b);
          }
        }
        // (one wave's LDS instructions execute in order; this keeps the
        // compiler's order)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
      // candidate j of row y has the window entry j - base[y]
      const uint32_t base[3] = {w0[0], w0[1] - kWindow, w0[2] - 2u * kWindow};
      // The candidates of three parts of rows (m of them from f, with
      // window entries from f - b0, at most 31 each) marked into w, left-aligned: the first one at bit 31.
      // Lanes with shorter parts walk on (WaveWindow's slack) as long as any
      // has candidates: the loop is the wave's.
      auto mark = [&](auto attract, const uint32_t (&f)[3], const uint32_t (&m)[3], const uint32_t (&b0)[3],
                      uint32_t (&w)[3]) {
        const uint32_t L = max(m[0], max(m[1], m[2]));
        uint32_t k = 0;
        if (in_win) {
          const WindowEntry* e[3];
#pragma unroll
          for (int y = 0; y < 3; ++y) e[y] = win->at + (m[y] ? f[y] - b0[y] : 0u);
          // two candidates a row at a time
          for (; __ballot(k < L); k += 2u) {
            WindowEntry b[3][2];
#pragma unroll
            for (int y = 0; y < 3; ++y) {
              b[y][0] = e[y][0];
              b[y][1] = e[y][1];
              e[y] += 2;
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              const float x[3] = {beyond(attract, b[0][u].x, b[0][u].y, b[0][u].r),
                                  beyond(attract, b[1][u].x, b[1][u].y, b[1][u].r),
                                  beyond(attract, b[2][u].x, b[2][u].y, b[2][u].r)};
              shift_in(w, x, 0x1p-125f);
            }
          }
        } else {
          // a part already walked re-reads its last candidate
          for (; __ballot(k < L); ++k) {
            Cand b[3];
#pragma unroll
            for (int y = 0; y < 3; ++y)
              candidate_load<kRadius, kOne, false, kO>(c, m[y] ? f[y] + min(k, m[y] - 1u) : 0u, pos, type, radius, d,
                                                       b[y]);
            const float x[3] = {beyond(attract, b[0].p.x, b[0].p.y, b[0].r), beyond(attract, b[1].p.x, b[1].p.y, b[1].r),
                                beyond(attract, b[2].p.x, b[2].p.y, b[2].r)};
            shift_in(w, x, 0x1p-125f);
          }
        }
#pragma unroll
        for (int y = 0; y < 3; ++y) w[y] = k ? w[y] << (32u - k) : 0u;
      };
      auto clear_marks = [&](const uint32_t (&f)[3], const uint32_t (&m)[3], uint32_t (&w)[3]) {
#pragma unroll
        for (int y = 0; y < 3; ++y) {
          w[y] &= ~(~0u >> m[y]);                         // past the part's end
          w[y] &= ~(0x80000000u >> min(i - f[y], 31u));  // the particle itself (there is no 32nd candidate)
        }
      };
      // candidate j (entry e of the windows), as the law reads it
      auto listed = [&](uint32_t j, uint32_t e) {
        Cand b;
        if (in_win) {
          b.p = make_float2(win->at[e].x, win->at[e].y);
          b.r = win->at[e].r;
          b.t = kOne ? 0u : clamp_idx(ld<kO>(type, j), c.num_types);
          const uint32_t jv = d.at<kO>(j);
          b.v = ld<kO>(d.vel, jv);
          b.w = ld<kO>(d.omega, jv);
        } else {
          candidate_load<kRadius, kOne, true, kO>(c, j, pos, type, radius, d, b);
        }
        return b;
      };
      // The three rows' marks follow each other in one word, and a second word
      // has a bit where a cell begins, so a step of the contact loop is a
      // count of zeros and a count of cells (14 instructions with 32 bits, 21
      // with 64; rows with words of their own took 30, and registers that cost
      // a wave a SIMD).
      float cfx = 0.0f, cfy = 0.0f;  // the cell's partial sum
      auto flush = [&]() {
        fx += cfx;
        fy += cfy;
        cfx = 0.0f;
        cfy = 0.0f;
      };
      auto marks = [&](auto word, const uint32_t (&f)[3], const uint32_t (&m)[3]) {
        using W = decltype(word);
        constexpr uint32_t kUp = 8u * sizeof(W) - 32u;
        uint32_t w[3] = {0u, 0u, 0u};
        if (c.attract) mark(std::true_type{}, f, m, base, w);
        else mark(std::false_type{}, f, m, base, w);
        clear_marks(f, m, w);
        return (W)w[0] << kUp | (W)w[1] << kUp >> m[0] | (W)w[2] << kUp >> (m[0] + m[1]);
      };
      // The law over the marked candidates of the rows, which are the parts.
      auto contacts = [&](auto h, decltype(h) cells, const uint32_t (&f)[3], const uint32_t (&m)[3]) {
        using W = decltype(h);
        const uint32_t l1 = m[0], l2 = m[0] + m[1], f1 = f[1] - l1, f2 = f[2] - l2;
        uint32_t cell = 0u;
        while (h) {
          uint32_t k, in_cell;
          if constexpr (sizeof(W) == 8) k = (uint32_t)__builtin_clzll(h);
          else k = (uint32_t)__builtin_clz(h);
          const W after = (W)(~(W)0 >> 1) >> k;
          h &= after;
          if constexpr (sizeof(W) == 8) in_cell = (uint32_t)__popcll(cells & ~after);
          else in_cell = (uint32_t)__popc(cells & ~after);
          const bool in0 = k < l1, in1 = k < l2;
          const uint32_t j = k + (in0 ? f[0] : (in1 ? f1 : f2));
          const uint32_t e = j - (in0 ? w0[0] : (in1 ? w0[1] - kWindow : w0[2] - 2u * kWindow));
          if (in_cell != cell) {
            flush();
            cell = in_cell;
          }
          listed_pair(c, q, listed(j, e), cfx, cfy, moment, pres);
        }
      };
      // every row in one pass
      auto whole = [&](auto word) {
        using W = decltype(word);
        const W h = marks(word, rs, len);
        if (h) {
          // the particle's velocity, spin and the pressure terms' reciprocal,
          // only where a candidate may touch
          if (!have_dyn) load_own_dyn();
          q.rden = 1.0 / q.den;
          // (a row outside the grid is empty, and its boundaries lie anywhere)
          W cells = 0;
          uint32_t at = 0;
#pragma unroll
          for (int y = 0; y < 3; ++y) {
            const W b = ((W)1 << (8u * sizeof(W) - 1u)) >> at;
            cells |= len[y] ? b | b >> (cut[y] & 0xFFFFu) | b >> (cut[y] >> 16) : (W)0;
            at += len[y];
          }
          contacts(h, cells, rs, len);
          flush();
        }
      };
      const uint32_t total = len[0] + len[1] + len[2], L = max(len[0], max(len[1], len[2]));
      if (__builtin_expect_with_probability(__ballot(total > 31u) == 0, 1, 0.9)) {
        whole(0u);
      } else if (__builtin_expect_with_probability(__ballot(total > 63u || L > 31u) == 0, 1, 0.9999)) {
        whole((uint64_t)0);
      } else {
        // Crowded neighbourhoods: a row's candidates up to 93 at a time, as
        // three parts of equal length walked together: 300,304 dense discs
        // with 72, 144, 324 and 900 candidates take 31, 37, 92 and 205 us a
        // collide (38, 59, 205 and 539 in passes over 31 candidates of which
        // two rows waited, 56, 73, 129 and 260 one at a time).  In a loop over
        // the rows, whose ranges are found again: a rare path, kept from
        // deciding how many registers the kernels take.
        if (!have_dyn) load_own_dyn();
        q.rden = 1.0 / q.den;
        float2 pc = q.p;
        asm("" : "+v"(pc.x), "+v"(pc.y));
        uint32_t tc = own.t;
        if constexpr (kMulti && !kUni) asm("" : "+v"(tc));
        const Instance in = kMulti ? c.inst[clamp_idx(c.mat[tc].inst, c.num_instances)] : c.inst0;
        const int G0 = (int)in.grid[0], G1 = (int)in.grid[1];
        int gx, gy;
        grid_pos(in, pc, gx, gy);
        if (clamp) clamp_cell(in, gx, gy);
#pragma unroll 1
        for (uint32_t y = 0; y < 3u; ++y) {
          const int iy = gy + (int)y - 1;
          const bool ok = !clamp || (iy >= 0 && iy < G1);
          const uint32_t at1 = in.cell_base + (clamp ? (uint32_t)(ok ? iy : gy) : (uint32_t)iy & ((uint32_t)G1 - 1u)) * (uint32_t)G0 +
                               (clamp ? (uint32_t)gx : (uint32_t)gx & ((uint32_t)G0 - 1u));
          const uint32_t at0 = clamp && gx == 0 ? at1 : at1 - 1u, at2 = clamp && gx == G0 - 1 ? at1 : at1 + 1u;
          const uint32_t s0 = ld<kO>(cell_start, at0), s1 = ld<kO>(cell_start, at1), s2 = ld<kO>(cell_start, at2);
          const uint32_t e0 = s0 != kEmpty ? ld<kO>(cell_end, at0) : 0u, e1 = s1 != kEmpty ? ld<kO>(cell_end, at1) : 0u,
                         e2 = s2 != kEmpty ? ld<kO>(cell_end, at2) : 0u;
          const uint32_t last = ok ? min(max(max(e0, e1), e2), n) : 0u, first = min(min(min(s0, s1), s2), last);
          const uint32_t count = last - first, c1 = max(e0, first) - first, c2 = max(e1 - first, c1);
          const uint32_t wy = y == 0u ? w0[0] : (y == 1u ? w0[1] - kWindow : w0[2] - 2u * kWindow);
          const uint32_t rows[3] = {wy, wy, wy};
          uint32_t cell = 0u;
          for (uint32_t done = 0; __ballot(done < count); done += 93u) {
            const uint32_t left = done < count ? min(count - done, 93u) : 0u, part = (left + 2u) / 3u;
            uint32_t f[3], m[3], w[3] = {0u, 0u, 0u};
#pragma unroll
            for (uint32_t s = 0; s < 3u; ++s) {
              f[s] = first + done + s * part;
              m[s] = left > s * part ? min(part, left - s * part) : 0u;
            }
            if (c.attract) mark(std::true_type{}, f, m, rows, w);
            else mark(std::false_type{}, f, m, rows, w);
            clear_marks(f, m, w);
            uint32_t h0 = w[0], h1 = w[1], h2 = w[2];
            while (h0 | h1 | h2) {
              const bool in0 = h0 != 0u, in1 = h1 != 0u;
              const uint32_t k = (uint32_t)__builtin_clz(in0 ? h0 : (in1 ? h1 : h2)), rest = ~(0x80000000u >> k);
              h2 = in0 || in1 ? h2 : h2 & rest;
              h1 = in0 ? h1 : h1 & rest;
              h0 &= rest;
              const uint32_t at = done + k + (in0 ? 0u : (in1 ? part : 2u * part));
              const uint32_t in_cell = (at >= c1 ? 1u : 0u) + (at >= c2 ? 1u : 0u);
              if (in_cell != cell) {
                flush();
                cell = in_cell;
              }
              listed_pair(c, q, listed(first + at, first + at - rows[0]), cfx, cfy, moment, pres);
            }
          }
          flush();
        }
      }
    } else if (kMode == kList) {
      by_cell = true;
    } else {
#pragma unroll
      for (int y = 0; y < 3; ++y) {
        RowSum rsum;
        rsum.b0 = b0[y];
        rsum.b1 = b1[y];
        const uint32_t end = re[y];
        if (kMode == kPrefetch) {
          // each candidate's position and radius fetched one iteration ahead
          // (pays off with many candidates per row, costs registers)
          uint32_t j = rs[y];
          Cand nx{};
          if (j < end) candidate_load<kRadius, kOne, false, kO>(c, j, pos, type, radius, d, nx);
          for (; j < end; ++j) {
            const Cand b = nx;
            if (j + 1u < end) candidate_load<kRadius, kOne, false, kO>(c, j + 1u, pos, type, radius, d, nx);
            candidate_at<kRadius, kOne, false, kO>(c, q, j, j == i, b, d, type, rsum, fx, fy, moment, pres);
          }
        } else {
          uint32_t j = rs[y];
          if (kMode == kBatch) {
#pragma unroll
            for (int k = 0; k < kBatchN; ++k, ++j)
              if (j < end)
                candidate_at<kRadius, kOne, false, kO>(c, q, j, j == i, cb[y][k], d, type, rsum, fx, fy, moment, pres);
          }
          for (; j < end; ++j)
            candidate<kRadius, kOne, kMode == kPlain, kO>(c, q, j, j == i, pos, d, type, radius, rsum, fx, fy, moment,
                                                       pres);
        }
        fx += rsum.cfx;
        fy += rsum.cfy;
      }
    }
  }
  if (by_cell) {
    // A wrapping grid's x edge, and rows too long for the contact list: the
    // cells one by one, in the reference order (the list kernels' rare path:
    // in loops, and from a cell computed again, as unrolled or with the cell
    // kept over the list walk it decided how many registers they take).
    if (!have_dyn) load_own_dyn();
    float2 pc = q.p;
    asm("" : "+v"(pc.x), "+v"(pc.y));
    uint32_t tc = own.t;
    if constexpr (kMulti && !kUni) asm("" : "+v"(tc));
    const Instance in = kMulti ? c.inst[clamp_idx(c.mat[tc].inst, c.num_instances)] : c.inst0;
    const int G0 = (int)in.grid[0], G1 = (int)in.grid[1];
    int gx, gy;
    grid_pos(in, pc, gx, gy);
    if (clamp) clamp_cell(in, gx, gy);
#pragma unroll 1
    for (int y = -1; y <= 1; ++y) {
      const int iy = gy + y;
      if (clamp && (iy < 0 || iy >= G1)) continue;
      const uint32_t row = in.cell_base + (clamp ? (uint32_t)iy : (uint32_t)iy & ((uint32_t)G1 - 1u)) * (uint32_t)G0;
#pragma unroll 1
      for (int sg = 0; sg < 3; ++sg) {
        const int ix = gx + sg - 1;
        if (clamp && (ix < 0 || ix >= G0)) continue;
        const uint32_t cell = row + (clamp ? (uint32_t)ix : (uint32_t)ix & ((uint32_t)G0 - 1u));
        const uint32_t st = cell_start[cell];
        if (st == kEmpty) continue;
        const uint32_t en = min(cell_end[cell], n);
        RowSum rsum;  // one cell: no boundary inside
        rsum.b0 = kNoBoundary;
        rsum.b1 = kNoBoundary;
        for (uint32_t j = st; j < en; ++j)
          candidate<kRadius, kOne, false, kO>(c, q, j, j == i, pos, d, type, radius, rsum, fx, fy, moment, pres);
        fx += rsum.cfx;
        fy += rsum.cfy;
      }
    }
  }
  if (kControl) {
    float rx, ry, rm;
    control_pair(c, q, *ctl.state, fx, fy, moment, pres, rx, ry, rm);
    ctl.react_x[i] = rx;
    ctl.react_y[i] = ry;
    ctl.react_m[i] = rm;
  }
  if (!have_dyn) load_own_dyn();  // (dead, and dropped, where the caller does not use them)
  own.v = q.v;
  own.w = q.w;
  fx_out = fx;
  fy_out = fy;
  moment_out = moment;
  pres_out = pres;
}

#define DEM_COLLIDE_PARAMS                                                                    \
  StepConst c, const float2* __restrict__ pos, const float2* __restrict__ vel,              \
      float2* __restrict__ acc, const float* __restrict__ omega, float* __restrict__ alpha, \
      const uint32_t* __restrict__ type, const float* __restrict__ radius,                  \
      const uint32_t* __restrict__ cell_start, const uint32_t* __restrict__ cell_end,       \
      float* __restrict__ pressure, ControlOut ctl, const uint32_t* __restrict__ gat,                \
      uint32_t* __restrict__ quiet, uint32_t n

// A wave whose discs all feel no force stores zeros without the three
// divisions: the sums start at +0 and are never -0, so fx, fy and moment
// are +0 exactly when nothing acted, and +0 over a positive finite mass or
// inertia is +0.  With a quiet array (the owned simulation's in-place
// step, whose integrate reads it) the wave records that instead of
// storing the zeros: quiet[i / 64] = 1 when acc and alpha of the wave's 64
// slots are +0 and were not written, else 0.
// (with a radius array the inertia is t / 5, t = ((2 mass) r) r, and t / 5
// rounds to a positive finite value exactly when 3 * 2^-149 <= t <= FLT_MAX:
// the check needs no division, which only a wave with a force then does)
template <bool kRadius>
__device__ __forceinline__ void store_acc(const Own& own, float fx, float fy, float moment, uint32_t i,
                                          float2* __restrict__ acc, float* __restrict__ alpha,
                                          uint32_t* __restrict__ quiet, float2& a, float& al) {
  bool inertia_ok;
  if constexpr (kRadius) {
    const float t = ((2.0f * own.mass) * own.r) * own.r;
    inertia_ok = t >= __uint_as_float(3u) && t <= 3.402823466e38f;
  } else {
    inertia_ok = own.inertia > 0.0f && own.inertia <= 3.402823466e38f;
  }
  const bool still = fx == 0.0f && fy == 0.0f && moment == 0.0f && own.mass > 0.0f &&
                     own.mass <= 3.402823466e38f && inertia_ok;
  const bool wave_still = __ballot(!still) == 0;
  if (quiet && __lane_id() == 0) quiet[i / (uint32_t)kWave] = wave_still ? 1u : 0u;
  a = make_float2(0.0f, 0.0f);
  al = 0.0f;
  if (!wave_still) {
    a = make_float2(fx / own.mass, fy / own.mass);
    al = moment / own.inertia;
  }
  if (!wave_still || !quiet) {
    acc[i] = a;
    alpha[i] = al;
  }
}

template <bool kRadius, int kMat, int kMode, bool kControl, bool kO>
__device__ __forceinline__ void collide_kernel_body(DEM_COLLIDE_PARAMS) {
  const uint32_t i = xcd_block() * blockDim.x + threadIdx.x;
  if (i >= n) return;
  Own own;
  float fx, fy, moment, pres;
  const Dyn d{vel, omega, gat};
  WaveWindow* win = kMode == kList ? wave_window() : nullptr;
  bool done = false;
  if constexpr (kMat == kInstances) {
    // waves inside one instance (all but the few that straddle a boundary)
    const uint32_t t = clamp_idx(type[i], c.num_types);
    const uint32_t t0 = __builtin_amdgcn_readfirstlane(t);
    if (__ballot(t != t0) == 0) {
      collide_particle<kRadius, kMat, kMode, kControl, kO, true>(c, i, pos, d, type, radius, cell_start, cell_end, n,
                                                                 own, ctl, fx, fy, moment, pres, t0, win);
      done = true;
    }
  }
  if (!done)
    collide_particle<kRadius, kMat, kMode, kControl, kO>(c, i, pos, d, type, radius, cell_start, cell_end, n, own,
                                                         ctl, fx, fy, moment, pres, 0u,
                                                         kMat == kInstances ? nullptr : win);
  float2 a;
  float al;
  store_acc<kRadius>(own, fx, fy, moment, i, acc, alpha, quiet, a, al);
  pressure[i] = pres;
}

template <bool kRadius, int kMat, int kMode, bool kControl, bool kO>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kMode == kList ? 7 : 1))) void k_collide(DEM_COLLIDE_PARAMS) {
  collide_kernel_body<kRadius, kMat, kMode, kControl, kO>(c, pos, vel, acc, omega, alpha, type, radius, cell_start,
                                                          cell_end, pressure, ctl, gat, quiet, n);
}

// The list mode is held to 72 VGPRs, 7 waves a SIMD: what spills then is the
// walk of crowded neighbourhoods.  (8 waves, 64 VGPRs and 78 SGPRs,
// spill on the common path: 131 us against 128 on the 4M dense pack, 159
// against 143 on the 8.2M-disc ensemble.)
// The one-material batched mode needed 65 VGPRs with 64-bit addresses; held to 64 (8
// waves per SIMD) it does not spill.  The other batched layouts would spill
// 12-19 registers under the same bound, so they keep k_collide.
template <bool kRadius>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_collide_batch(DEM_COLLIDE_PARAMS) {
  collide_kernel_body<kRadius, kOneMat, kBatch, false, true>(c, pos, vel, acc, omega, alpha, type, radius,
                                                             cell_start, cell_end, pressure, ctl, gat, quiet, n);
}
#undef DEM_COLLIDE_PARAMS

// kO (32-bit offsets) for states whose arrays stay under 4 GiB; larger ones
// (or DEM_STEP_WIDE) run the plain mode with 64-bit addresses.
template <bool kRadius, int kMat, int kMode, bool kControl, bool kO>
constexpr auto collide_kernel() {
  if constexpr (!kO)
    return &k_collide<kRadius, kMat, kPlain, kControl, false>;
  else if constexpr (kMat == kOneMat && kMode == kBatch && !kControl)
    return &k_collide_batch<kRadius>;
  else
    return &k_collide<kRadius, kMat, kMode, kControl, true>;
}

// ------------------------------------------------------------- integrate --
__device__ __forceinline__ float wrap_theta(float th) {
  const double twopi = 2 * M_PI;
  if ((double)th > twopi) th = (float)((double)th - twopi * floor((double)th / twopi));
  if (th < 0.0f) th = (float)((double)th - twopi * floor((double)th / twopi));
  return th;
}

// integrateSystemD (src/particles_kernel.cuh:580-627) with collideBoundary
// (:388-456) inlined for the bottom wall, on one particle: p, v, w, th are
// updated in place; pres gains the bottom wall's term when it is hit (the
// return value says whether the bottom-wall law ran).  With pres_src, pres
// is first loaded from it, and only on that branch.
__device__ __forceinline__ bool integrate_particle(const StepConst& c, const Material& m, const Instance& in, float r,
                                                   float mass, float inertia, float2 a, float alpha_i, float2& p,
                                                   float2& v, float& w, float& th, float& pres,
                                                   const float* pres_src) {
  const float dt = c.dt;
  v.x = v.x + (c.gx + a.x) * dt;
  v.y = v.y + (c.gy + a.y) * dt;
  p.x = p.x + v.x * dt;
  p.y = p.y + v.y * dt;
  w = w + alpha_i * dt;
  th = th + w * dt;
  th = wrap_theta(th);

  const float bd = -m.bdamp;
  const float Lx = in.box[0], Ly = in.box[1];
  if (p.x > Lx - r) {
    p.x = Lx - r;
    v.x = v.x * bd;
  }
  if (p.x < r) {
    p.x = r;
    v.x = v.x * bd;
  }
  if (!(c.flags & DEM_OPEN_TOP) && p.y > Ly - r) {
    p.y = Ly - r;
    v.y = v.y * bd;
  }
  if (p.y < r) {
    // collideBoundary(pos, vel, omega, type, (pos.x, 0), wallAlpha, pressure)
    float wallAlpha = 0.0f;
    float pr = pres_src ? *pres_src : pres;
    const float rx = p.x - p.x, ry = 0.0f - p.y;
    const float dist = sqrtf(rx * rx + ry * ry);
    float wfx = 0.0f, wfy = 0.0f;
    if (dist < r) {
      const float nx = rx / dist, ny = ry / dist;
      const float tx = -ny, ty = nx;
      const float rvx = -v.x, rvy = -v.y;
      const float vn = rvx * nx + rvy * ny;
      const float vtx = rvx - vn * nx, vty = rvy - vn * ny;
      const float kt = series(m.kt, c.bkt);
      const float s = -mass;
      wfx = s * c.gx;
      wfy = s * c.gy;
      if (vn < 0.0f) {
        const float s2 = m.cn * vn;
        wfx += s2 * nx;
        wfy += s2 * ny;
      }
      const float flen = sqrtf(wfx * wfx + wfy * wfy);
      pr = add_pressure(pr, flen, pressure_den(r));
      if (m.mu != 0.0f) {
        const float sr = r * w;
        const float cvx = vtx - sr * tx, cvy = vty - sr * ty;
        float ftx = (kt * cvx) * dt, fty = (kt * cvy) * dt;
        const float ftmax = m.mu * flen;
        if (!sqrt_below(ftx * ftx + fty * fty, ftmax)) {
          const float cl = sqrtf(cvx * cvx + cvy * cvy);
          ftx = (ftmax * cvx) / cl;
          fty = (ftmax * cvy) / cl;
        }
        wfx = ftx;
        wfy = fty;
        wallAlpha = wallAlpha + (r * (ftx * tx + fty * ty)) / inertia;
      }
    }
    const float ax = wfx / mass, ay = wfy / mass;
    v.x = v.x + ax * dt;
    v.y = v.y + ay * dt;
    p.x = p.x + (ax * dt) * dt;
    p.y = p.y + (ay * dt) * dt;
    w = w + wallAlpha * dt;
    th = th + (wallAlpha * dt) * dt;
    p.y = r;
    v.y = v.y * bd;
    pres = pr;
    return true;
  }
  return false;
}

// The next step's hash of an integrated particle (NextKeys): the cell key of
// its new position p and whether it left the cell of its sorted slot, whose
// key is old (the state stays in this order until the next sort).  kWhole:
// for launch_resort_whole.  Every lane of the wave that holds a particle
// calls this.
template <bool kWhole>
__device__ __forceinline__ void next_key(const StepConst& c, const NextKeys& nk, float2 p, uint32_t old,
                                         const Instance& in, uint32_t i, uint32_t n) {
  const uint32_t k = cell_key_in(c, in, p);
  const bool mover = k != old;
  if (mover) nk.key[i] = k;  // a stayer's key is its sorted key
  const uint64_t moved = __ballot(mover);
  const uint32_t list = kWhole ? i / (uint32_t)kWave % kMoverLists : 0u;
  uint32_t at = 0;
  if (__lane_id() == 0) {  // lane 0 holds the wave's first index, a multiple of 64
    const uint32_t w0 = i / 32u, nwords = (n + 31u) / 32u;
    nk.bits[w0] = (uint32_t)moved;
    if (w0 + 1u < nwords) nk.bits[w0 + 1u] = (uint32_t)(moved >> 32);
    const uint32_t cnt = (uint32_t)__popcll(moved);
    if (cnt) {
      if constexpr (kWhole) at = atomicAdd(nk.list_count + list * kMoverStride, cnt);
      else atomicAdd(&nk.tile_count[i / kResortTile], cnt);
    }
  }
  if (kWhole && moved) {
    const uint32_t cap = mover_list_cap(n);
    at = __builtin_amdgcn_readfirstlane(at) + (uint32_t)__popcll(moved & ((1ull << __lane_id()) - 1ull));
    if (mover && at < cap) nk.list[list * cap + at] = ((uint64_t)k << 32) | i;
  }
}

// NextKeys' other outputs, particle i's share (the launchers refuse a clear_n
// for which cell + n could pass 2^32 and the loop start again).
__device__ __forceinline__ void next_clear(const NextKeys& nk, uint32_t i, uint32_t n) {
  for (uint32_t cell = i; cell < nk.clear_n; cell += n) nk.clear[cell] = kEmpty;
  if (i == 0u && nk.listed) *nk.host_listed = *nk.listed;
}

// integrateSystemD over all particles, with the next step's keys (kNext 1:
// NextKeys; 2: for launch_resort_whole; 0: none).  The input and output arrays may be
// the same (in place, as the reference) or different (the owned
// simulation writes the integrated state back to its home buffer); each
// lane reads and writes only its own slot.
template <bool kRadius, int kMat, int kNext, int kPer>
__global__ __launch_bounds__(256) void k_integrate(
    StepConst c, const float2* pos_in, const float2* vel_in, const float* theta_in, const float* omega_in,
    float2* pos_out, float2* vel_out, float* theta_out, float* omega_out, const float2* __restrict__ acc,
    const float* __restrict__ alpha, const uint32_t* __restrict__ type, const float* __restrict__ radius,
    float* __restrict__ pressure, NextKeys nk, const uint32_t* __restrict__ gat,
    const uint32_t* __restrict__ quiet, uint32_t n) {
  constexpr bool kMulti = kMat == kInstances;
  const bool in_place = !gat && omega_out == omega_in && theta_out == theta_in;
  // kPer particles a lane, as k_hash.  The inputs of all kPer particles are
  // loaded before any output is stored (the in and out arrays may be the
  // same, so the compiler could not move a later particle's loads above an
  // earlier one's stores); each lane reads and writes only its own slots.
  const uint32_t base = blockIdx.x * c.block * kPer + threadIdx.x;
  uint32_t t[kPer];
  float2 p_old[kPer], v[kPer], a[kPer];
  float w[kPer], th[kPer], al[kPer], rad[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const uint32_t i = base + (uint32_t)k * c.block;
    if (i >= n) continue;
    if (kNext == 2) next_clear(nk, i, n);
    t[k] = kMat == kOneMat ? 0u : clamp_idx(type[i], c.num_types);
    // velocity, spin and angle through the gather index when one is given
    const uint32_t g = gat ? gat[i] : i;
    p_old[k] = pos_in[i];
    v[k] = vel_in[g];
    w[k] = omega_in[g];
    th[k] = theta_in[g];
    // a run of 64 slots that collide marked quiet has acc = alpha = +0 (not
    // stored); the wave's 64 slots are one such run (one scalar load)
    const bool still = quiet && quiet[__builtin_amdgcn_readfirstlane(i) / (uint32_t)kWave] != 0u;
    a[k] = still ? make_float2(0.0f, 0.0f) : acc[i];
    al[k] = still ? 0.0f : alpha[i];
    rad[k] = kRadius ? radius[i] : 0.0f;
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const uint32_t i = base + (uint32_t)k * c.block;
    if (i >= n) continue;
    auto run = [&](const Material& m, const Instance& in) {
      float r, mass, inertia;
      body<kRadius>(m, rad + k, 0u, r, mass, inertia);
      float2 p = p_old[k], vv = v[k];
      float ww = w[k], tt = th[k];
      float pres = 0.0f;
      if (integrate_particle(c, m, in, r, mass, inertia, a[k], al[k], p, vv, ww, tt, pres, pressure + i))
        pressure[i] = pres;
      pos_out[i] = p;
      vel_out[i] = vv;
      // in place, a spin or angle whose bits did not change is not stored
      // again (a disc at rest: no spin, no moment)
      if (!in_place || __float_as_uint(ww) != __float_as_uint(w[k])) omega_out[i] = ww;
      if (!in_place || __float_as_uint(tt) != __float_as_uint(th[k])) theta_out[i] = tt;
      // (the key the particle is sorted by is the hash of its position before
      // integrate, recomputed here rather than read)
      if (kNext) next_key<kNext == 2>(c, nk, p, cell_key_in(c, in, p_old[k]), in, i, n);
    };
    if constexpr (kMulti) {
      // a wave inside one instance reads its material row and geometry as
      // scalars
      const uint32_t t0 = __builtin_amdgcn_readfirstlane(t[k]);
      if (__ballot(t[k] != t0) == 0) {
        const Material m = c.mat[t0];
        run(m, c.inst[clamp_idx(m.inst, c.num_instances)]);
        continue;
      }
    }
    const Material m = c.mat[t[k]];
    run(m, kMulti ? c.inst[clamp_idx(m.inst, c.num_instances)] : c.inst0);
  }
}

// collide + integrate + the next step's hash in one pass over the sorted
// particles: forces from the sorted state (pos, vel, omega in the *_in
// arrays), accelerations and pressure written as collide writes them, and the
// integrated state written to the *_out arrays, other ones, so no lane
// overwrites a neighbour's input (an angle feeds no neighbour: theta_out may
// be theta_in).  The arithmetic is that of k_collide followed by k_integrate.
// One pass instead of two reads positions, radii and cell ranges once, writes
// no accelerations to read back, and streams while collide's instructions,
// which bound it, issue: 67 us against 53 + 29 for 4M settling discs, 145
// against 128 + 42 on the 4M dense pack, 199 against 143 + 82 on the
// 8.2M-disc ensemble (208 with material rows and geometries loaded per lane
// in every wave; an ensemble of 300 discs an instance, where a fifth of the
// waves straddle two, takes 30.5 us a step either way).
template <bool kRadius, int kMat, bool kWhole, int kMode, bool kControl, bool kO>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kWhole ? 4 : 7))) void k_collide_integrate(
    StepConst c, const float2* __restrict__ pos_in, const float2* __restrict__ vel_in,
    const float* __restrict__ omega_in, const float* theta_in, const uint32_t* __restrict__ type,
    const float* __restrict__ radius, const uint32_t* __restrict__ cell_start,
    const uint32_t* __restrict__ cell_end, float2* __restrict__ acc, float* __restrict__ alpha,
    float* __restrict__ pressure, float2* __restrict__ pos_out, float2* __restrict__ vel_out,
    float* __restrict__ omega_out, float* theta_out, NextKeys nk, ControlOut ctl, uint32_t* __restrict__ quiet,
    uint32_t n) {
  const uint32_t i = xcd_block() * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if constexpr (kWhole) next_clear(nk, i, n);
  const Dyn d{vel_in, omega_in, nullptr};
  WaveWindow* win = kMode == kList ? wave_window() : nullptr;
  Own own;
  float fx, fy, moment, pres;
  // (small states do not fill the chip, so latency counts, not registers:
  // every load that can go out first does)
  const float th_first = kWhole ? theta_in[i] : 0.0f;
  bool uniform = false;
  uint32_t t0 = 0;
  if constexpr (kMat == kInstances && !kWhole) {
    // a wave inside one instance (all but the few that straddle a boundary)
    // reads its material row and geometry as scalars
    const uint32_t t = clamp_idx(type[i], c.num_types);
    t0 = __builtin_amdgcn_readfirstlane(t);
    uniform = __ballot(t != t0) == 0;
    if (__builtin_expect(uniform, 1))
      collide_particle<kRadius, kMat, kMode, kControl, kO, true, kWhole>(c, i, pos_in, d, type, radius, cell_start,
                                                                         cell_end, n, own, ctl, fx, fy, moment, pres,
                                                                         t0, win);
  }
  if (!uniform)
    collide_particle<kRadius, kMat, kMode, kControl, kO, false, kWhole>(c, i, pos_in, d, type, radius, cell_start,
                                                                        cell_end, n, own, ctl, fx, fy, moment, pres,
                                                                        0u, win);
  const Material m = uniform ? c.mat[t0] : c.mat[own.t];
  const Instance in = kMat == kInstances ? c.inst[clamp_idx(m.inst, c.num_instances)] : c.inst0;
  body<kRadius>(m, &own.r, 0u, own.r, own.mass, own.inertia);  // (again, rather than kept)
  float2 a;
  float al;
  store_acc<kRadius>(own, fx, fy, moment, i, acc, alpha, quiet, a, al);
  float2 p = own.p, v = own.v;
  float w = own.w;
  const float th_in = kWhole ? th_first : theta_in[i];
  float th = th_in;
  (void)integrate_particle(c, m, in, own.r, own.mass, own.inertia, a, al, p, v, w, th, pres, nullptr);
  pressure[i] = pres;
  pos_out[i] = p;
  vel_out[i] = v;
  omega_out[i] = w;
  if (theta_out != theta_in || __float_as_uint(th) != __float_as_uint(th_in)) theta_out[i] = th;
  next_key<kWhole>(c, nk, p, own.cell, in, i, n);
}

// Whether next_clear's index stays below 2^32.
inline bool clear_ends(const NextKeys& nk, uint32_t n) { return nk.clear_n <= 0xFFFFFFFFu - n; }

inline dim3 grid_for(uint32_t n, int block) { return dim3((n + (uint32_t)block - 1u) / (uint32_t)block); }

}  // namespace

// Particles a lane of the streaming kernels (hash, reorder, integrate): 1, 2
// or 4 (the autotuner's choice); anything else runs as 1.
inline int per_of(int per) { return per == 2 || per == 4 ? per : 1; }
#define DEM_PER(MACRO, PER) \
  do {                      \
    if ((PER) == 4) MACRO(4); \
    else if ((PER) == 2) MACRO(2); \
    else MACRO(1);          \
  } while (0)

hipError_t launch_hash(const StepConst& c, hipStream_t s, int block, const float2* pos,
                       const uint32_t* type, uint32_t* hash, uint32_t* index, uint32_t n, int per) {
  if (n == 0) return hipSuccess;
  StepConst cb = c;
  cb.block = (uint32_t)block;
  per = per_of(per);
  const dim3 grid = grid_for((n + (uint32_t)per - 1u) / (uint32_t)per, block);
#define DEM_HASH(P)                                                                                        \
  do {                                                                                                    \
    if (type && c.num_instances > 1)                                                                      \
      hipLaunchKernelGGL((k_hash<true, P>), grid, dim3(block), 0, s, cb, pos, type, hash, index, n);       \
    else                                                                                                  \
      hipLaunchKernelGGL((k_hash<false, P>), grid, dim3(block), 0, s, cb, pos, type, hash, index, n);      \
  } while (0)
  DEM_PER(DEM_HASH, per);
#undef DEM_HASH
  return hipGetLastError();
}

hipError_t launch_fill(hipStream_t s, uint32_t* p, uint32_t value, uint32_t count) {
  if (count == 0) return hipSuccess;
  const int vec = (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
  const uint32_t threads = (count + 3u) / 4u;
  hipLaunchKernelGGL(k_fill, grid_for(threads, 256), dim3(256), 0, s, p, value, count, vec);
  return hipGetLastError();
}

hipError_t launch_reorder(hipStream_t s, int block, uint32_t* cell_start, uint32_t* cell_end,
                          float2* s_pos, float2* s_vel, float* s_theta, float* s_omega,
                          uint32_t* s_id, uint32_t* s_loc, uint32_t* s_type, float* s_radius,
                          const uint32_t* hash, const uint32_t* index, const float2* o_pos,
                          const float2* o_vel, const float* o_theta, const float* o_omega,
                          const uint32_t* o_id, const uint32_t* o_type, const float* o_radius,
                          uint32_t n, uint32_t num_cells, bool full, int per) {
  if (n == 0) return hipSuccess;
  per = per_of(per);
  const dim3 grid = grid_for((n + (uint32_t)per - 1u) / (uint32_t)per, block);
#define DEM_REORDER(R, F, P)                                                                                 \
  hipLaunchKernelGGL((k_reorder<R, F, P>), grid, dim3(block), 0, s, cell_start, cell_end, s_pos, s_vel,       \
                     s_theta, s_omega, s_id, s_loc, s_type, s_radius, hash, index, o_pos, o_vel, o_theta,     \
                     o_omega, o_id, o_type, o_radius, n, num_cells)
#define DEM_REORDER_P(P)                                                     \
  do {                                                                       \
    if (s_radius) {                                                          \
      if (full) DEM_REORDER(true, true, P); else DEM_REORDER(true, false, P); \
    } else {                                                                 \
      if (full) DEM_REORDER(false, true, P); else DEM_REORDER(false, false, P); \
    }                                                                        \
  } while (0)
  DEM_PER(DEM_REORDER_P, per);
#undef DEM_REORDER_P
#undef DEM_REORDER
  return hipGetLastError();
}

// Kernel variant dispatch: kRadius x material layout x (candidate mode,
// control), where the controlled particle uses the plain or the list mode.
inline int mat_kind(const StepConst& c) {
  return c.num_instances > 1 ? kInstances : (c.num_types == 1 ? kOneMat : kManyMat);
}
#define DEM_DISPATCH_RM(MACRO, MODE, X)                                  \
  do {                                                                   \
    const int mk_ = mat_kind(c);                                         \
    if (radius) {                                                        \
      if (mk_ == kInstances) MACRO(true, kInstances, MODE, X);           \
      else if (mk_ == kOneMat) MACRO(true, kOneMat, MODE, X);            \
      else MACRO(true, kManyMat, MODE, X);                               \
    } else {                                                             \
      if (mk_ == kInstances) MACRO(false, kInstances, MODE, X);          \
      else if (mk_ == kOneMat) MACRO(false, kOneMat, MODE, X);           \
      else MACRO(false, kManyMat, MODE, X);                              \
    }                                                                    \
  } while (0)
// (a controlled particle is set for a single instance; an ensemble that the
// context is given afterwards meets it in every instance, one candidate at a
// time)
#define DEM_DISPATCH_CTL(MACRO, MODE)                                    \
  do {                                                                   \
    const int mk_ = mat_kind(c);                                         \
    if (radius) {                                                        \
      if (mk_ == kInstances) MACRO(true, kInstances, kPlain, true);      \
      else if (mk_ == kOneMat) MACRO(true, kOneMat, MODE, true);         \
      else MACRO(true, kManyMat, MODE, true);                            \
    } else {                                                             \
      if (mk_ == kInstances) MACRO(false, kInstances, kPlain, true);     \
      else if (mk_ == kOneMat) MACRO(false, kOneMat, MODE, true);        \
      else MACRO(false, kManyMat, MODE, true);                           \
    }                                                                    \
  } while (0)
#define DEM_DISPATCH(MACRO)                                              \
  do {                                                                   \
    if (ctl && mode == kList) DEM_DISPATCH_CTL(MACRO, kList);            \
    else if (ctl) DEM_DISPATCH_CTL(MACRO, kPlain);                       \
    else if (mode == kPrefetch) DEM_DISPATCH_RM(MACRO, kPrefetch, false);\
    else if (mode == kBatch) DEM_DISPATCH_RM(MACRO, kBatch, false);      \
    else if (mode == kList) DEM_DISPATCH_RM(MACRO, kList, false);        \
    else DEM_DISPATCH_RM(MACRO, kPlain, false);                          \
  } while (0)

hipError_t launch_collide(const StepConst& c, hipStream_t s, int block, const float2* pos,
                          const float2* vel, float2* acc, const float* omega, float* alpha,
                          const uint32_t* type, const float* radius, const uint32_t* cell_start,
                          const uint32_t* cell_end, float* pressure, uint32_t n, int mode,
                          const ControlOut* ctl, const uint32_t* gat, uint32_t* quiet) {
  if (n == 0) return hipSuccess;
  StepConst cb = c;
  cb.block = (uint32_t)block;
  if (quiet && block % kWave) return hipErrorInvalidValue;  // the flags cover aligned 64-particle runs
  const ControlOut co = ctl ? *ctl : ControlOut{};
  // 32-bit byte offsets reach every element while n * 8 B and cells * 4 B
  // stay within 4 GiB
  const bool o32 = !(mode & kWideMode) && n <= (1u << 29) && c.cells <= (1u << 30);
  mode &= ~kWideMode;
#define DEM_COLLIDE(R, M, P, X)                                                                             \
  do {                                                                                                      \
    if (o32)                                                                                                \
      hipLaunchKernelGGL((collide_kernel<R, M, P, X, true>()), grid_for(n, block), dim3(block),                 \
                         window_bytes(P, block), s, cb, pos,                                                      \
                         vel, acc, omega, alpha, type, radius, cell_start, cell_end, pressure, co, gat, quiet, n); \
    else                                                                                                    \
      hipLaunchKernelGGL((collide_kernel<R, M, P, X, false>()), grid_for(n, block), dim3(block), 0, s, cb,     \
                         pos, vel, acc, omega, alpha, type, radius, cell_start, cell_end, pressure, co, gat, quiet, \
                         n);                                                                                \
  } while (0)
  DEM_DISPATCH(DEM_COLLIDE);
#undef DEM_COLLIDE
  return hipGetLastError();
}

hipError_t launch_collide_integrate(const StepConst& c, hipStream_t s, int block, const float2* pos_in,
                                    const float2* vel_in, const float* omega_in, const float* theta_in,
                                    const uint32_t* type, const float* radius, const uint32_t* cell_start,
                                    const uint32_t* cell_end, float2* acc, float* alpha, float* pressure,
                                    float2* pos_out, float2* vel_out, float* omega_out, float* theta_out,
                                    const NextKeys& next, uint32_t n, int mode, const ControlOut* ctl,
                                    uint32_t* quiet) {
  if (n == 0) return hipSuccess;
  StepConst cb = c;
  cb.block = (uint32_t)block;
  if (block % kWave) return hipErrorInvalidValue;  // waves must cover aligned 64-particle runs
  if (!clear_ends(next, n)) return hipErrorInvalidValue;
  const ControlOut co = ctl ? *ctl : ControlOut{};
  const bool o32 = !(mode & kWideMode) && n <= (1u << 29) && c.cells <= (1u << 30);  // (launch_collide)
#define DEM_CI_W(R, M, W, P, X)                                                                                    \
  hipLaunchKernelGGL((k_collide_integrate<R, M, W, P, X, P == kList>), grid_for(n, block), dim3(block),            \
                     window_bytes(P, block), s, cb, pos_in, vel_in, omega_in, theta_in, type, radius, cell_start,   \
                     cell_end, acc, alpha, pressure, pos_out, vel_out, omega_out, theta_out, next, co, quiet, n)
#define DEM_CI(R, M, P, X)                   \
  do {                                       \
    if (next.list) DEM_CI_W(R, M, true, P, X); \
    else DEM_CI_W(R, M, false, P, X);        \
  } while (0)
  // contact lists (from 4,096 discs, 6.3 us against 6.0 one candidate ahead,
  // and 65,536, 6.8 against 7.0, to 4M dense ones, where walking candidates one
  // at a time runs the contact law at every candidate some lane touches), or
  // one candidate at a time with 64-bit addresses
  if (o32 && ctl) DEM_DISPATCH_CTL(DEM_CI, kList);
  else if (o32) DEM_DISPATCH_RM(DEM_CI, kList, false);
  else if (ctl) DEM_DISPATCH_CTL(DEM_CI, kPlain);
  else DEM_DISPATCH_RM(DEM_CI, kPlain, false);
#undef DEM_CI
#undef DEM_CI_W
  return hipGetLastError();
}
#undef DEM_DISPATCH
#undef DEM_DISPATCH_CTL
#undef DEM_DISPATCH_RM

// ---- controlled particle: reaction sum and move ------------------------------
// reduceVecD (src/particles_kernel.cuh:552-578) on the three reaction
// vectors: block b sums values [512 b, 512 b + 512) (zeros past n) by the
// same pairwise tree.  The last block to finish (it takes the last of the
// tickets, which it resets) adds the block sums in order
// (src/functions.cu:505-513, there on the host), one lane per quantity, then
// makes the kinematic move of the controlled particle (src/main.cu:510-514)
// when `move` is set.  No block waits for another; a second launch for the
// sum took 4.3 us after the first's 4.5.
__global__ __launch_bounds__(kReactBlock) void k_reduce_reaction(
    const float* __restrict__ rx, const float* __restrict__ ry, const float* __restrict__ rm, float* __restrict__ bx,
    float* __restrict__ by, float* __restrict__ bm, uint32_t n, uint32_t blocks, float* __restrict__ reaction,
    dem_controlled* state, int move, uint32_t* __restrict__ ticket) {
  __shared__ float cx[kReactBlock], cy[kReactBlock], cm[kReactBlock];
  __shared__ uint32_t s_last;
  const uint32_t t = threadIdx.x, i = blockIdx.x * kReactBlock + t;
  cx[t] = i < n ? rx[i] : 0.0f;
  cy[t] = i < n ? ry[i] : 0.0f;
  cm[t] = i < n ? rm[i] : 0.0f;
  __syncthreads();
  for (uint32_t h = kReactBlock / 2; h != 0; h /= 2) {
    if (t < h) {
      cx[t] += cx[t + h];
      cy[t] += cy[t + h];
      cm[t] += cm[t + h];
    }
    __syncthreads();
  }
  if (t == 0) {
    if (blockIdx.x < blocks) {
      bx[blockIdx.x] = cx[0];
      by[blockIdx.x] = cy[0];
      bm[blockIdx.x] = cm[0];
    }
    __threadfence();
    s_last = atomicAdd(ticket, 1u) + 1u == gridDim.x;
  }
  __syncthreads();
  if (!s_last) return;
  __threadfence();
  // the block sums to LDS (512 at a time), from where one lane a quantity adds them
  float acc = 0.0f;
  for (uint32_t b0 = 0; b0 < blocks; b0 += kReactBlock) {
    __syncthreads();
    if (b0 + t < blocks) {
      cx[t] = bx[b0 + t];
      cy[t] = by[b0 + t];
      cm[t] = bm[b0 + t];
    }
    __syncthreads();
    if (t < 3) {
      const float* v = t == 0 ? cx : (t == 1 ? cy : cm);
      for (uint32_t k = 0; k < min(blocks - b0, kReactBlock); ++k) acc += v[k];
    }
  }
  if (t < 3) reaction[t] = acc;
  if (t == 0) {
    *ticket = 0u;
    if (move) {
      dem_controlled& C = *state;
      C.pos[0] = (float)((double)C.pos[0] + C.move[0]);
      C.pos[1] = (float)((double)C.pos[1] + C.move[1]);
      if ((double)C.pos[1] < C.wrap_below_y) C.pos[1] = C.reset_y;
      if ((double)C.pos[0] > C.wrap_above_x) C.pos[0] = C.reset_x;
    }
  }
}

hipError_t launch_control_finish(hipStream_t s, const ControlOut& ctl, float* bx, float* by, float* bm, uint32_t n,
                                 float* reaction, dem_controlled* state, bool move) {
  const uint32_t blocks = (n + kReactBlock - 1u) / kReactBlock;
  uint32_t* ticket = reinterpret_cast<uint32_t*>(reaction + 3);
  hipLaunchKernelGGL(k_reduce_reaction, dim3(blocks ? blocks : 1u), dim3(kReactBlock), 0, s, ctl.react_x, ctl.react_y,
                     ctl.react_m, bx, by, bm, n, blocks, reaction, state, move ? 1 : 0, ticket);
  return hipGetLastError();
}

hipError_t launch_integrate(const StepConst& c, hipStream_t s, int block, float2* pos, float2* vel,
                            const float2* acc, float* theta, float* omega, const float* alpha,
                            const uint32_t* type, const float* radius, float* pressure, uint32_t n,
                            const NextKeys* next, int per) {
  return launch_integrate_to(c, s, block, pos, vel, theta, omega, pos, vel, theta, omega, acc, alpha, type, radius,
                             pressure, n, next, nullptr, per);
}

hipError_t launch_integrate_to(const StepConst& c, hipStream_t s, int block, const float2* pos_in,
                               const float2* vel_in, const float* theta_in, const float* omega_in, float2* pos_out,
                               float2* vel_out, float* theta_out, float* omega_out, const float2* acc,
                               const float* alpha, const uint32_t* type, const float* radius, float* pressure,
                               uint32_t n, const NextKeys* next, const uint32_t* gat, int per,
                               const uint32_t* quiet) {
  if (n == 0) return hipSuccess;
  StepConst cb = c;
  cb.block = (uint32_t)block;
  if (block % kWave) return hipErrorInvalidValue;  // waves must cover aligned 64-particle runs
  if (next && !clear_ends(*next, n)) return hipErrorInvalidValue;
  per = per_of(per);
  const dim3 grid = grid_for((n + (uint32_t)per - 1u) / (uint32_t)per, block);
  const NextKeys nk = next ? *next : NextKeys{};
#define DEM_INTEGRATE(R, M, X, P)                                                                         \
  hipLaunchKernelGGL((k_integrate<R, M, X, P>), grid, dim3(block), 0, s, cb, pos_in, vel_in, theta_in,    \
                     omega_in, pos_out, vel_out, theta_out, omega_out, acc, alpha, type, radius, pressure, nk, \
                     gat, quiet, n)
#define DEM_INTEGRATE_X(R, M, P)            \
  do {                                      \
    if (next && next->list) DEM_INTEGRATE(R, M, 2, P); \
    else if (next) DEM_INTEGRATE(R, M, 1, P);          \
    else DEM_INTEGRATE(R, M, 0, P);                    \
  } while (0)
#define DEM_INTEGRATE_P(P)                                                \
  do {                                                                    \
    const int mk = mat_kind(c);                                           \
    if (radius) {                                                         \
      if (mk == kInstances) DEM_INTEGRATE_X(true, kInstances, P);         \
      else if (mk == kOneMat) DEM_INTEGRATE_X(true, kOneMat, P);          \
      else DEM_INTEGRATE_X(true, kManyMat, P);                            \
    } else {                                                              \
      if (mk == kInstances) DEM_INTEGRATE_X(false, kInstances, P);        \
      else if (mk == kOneMat) DEM_INTEGRATE_X(false, kOneMat, P);         \
      else DEM_INTEGRATE_X(false, kManyMat, P);                           \
    }                                                                     \
  } while (0)
  DEM_PER(DEM_INTEGRATE_P, per);
#undef DEM_INTEGRATE_P
#undef DEM_INTEGRATE_X
#undef DEM_INTEGRATE
  return hipGetLastError();
}

}  // namespace dem
