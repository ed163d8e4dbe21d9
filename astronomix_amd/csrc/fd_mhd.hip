// MI355X (gfx950) kernels and C ABI of the finite-difference MHD step:
// characteristic WENO-5 fluxes, HOW-MHD constrained transport and SSPRK(5,4)
// (astronomix/_finite_difference/**, leo1200/astronomix v0.5.1).
//
// Passes of one right-hand-side evaluation (all direction-specific; the
// reference's transposes become index arithmetic):
//   k_first    conserved rows of the state as the first stage's input
//   k_weno     interface fluxes along x, y and z in one launch: the cells of a
//              tile are staged in LDS with their flux and wave speeds; each
//              thread builds the interface eigen-system once and runs the 7
//              characteristic WENO-5 reconstructions (_weno.py:111-324,
//              _eigen.py:116-911); also emits the CT modified fluxes
//              (_constrained_transport.py:81-102)
//   k_ct_edge  edge EMFs by 4th-order interpolation (_constrained_transport.py:107-131)
//   k_ct_avg   point values to averages (_interpolate.py:38-62)
//   k_face     6th-order curl of the EMFs + SSPRK combine of the face fields
//   k_combine  flux divergence + SSPRK combine of the conserved state
//              (_ssprk.py:224-228, 300-311), then the next stage's input:
//              positivity floors and the face-to-centre B with its energy
//              correction (_enforce_positivity.py:21-59,
//              _constrained_transport.py:160-198); after the last stage the
//              primitive state
// Boundaries are periodic.

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <new>
#include <vector>

#include "amx.h"
#include "common.h"
#include "snapshots.h"

namespace amx {
namespace fd {

constexpr int TBZ = 32;  // columns of a WENO block of the x and y directions
constexpr int TP = 16;   // its interfaces along the direction
constexpr int NTH = TP * TBZ;

struct Phys {
  float gamma, gm1, inv_gm1, rhomin, pgmin, inv_rhomin;
  int positivity;
};

struct Grid {
  int nx, ny, nz;
  long sx, sy;  // strides of x and y (z contiguous)
  long nc;
};

// Byte offset of a cell in a field, with its coordinates: one division per
// cell in 32-bit arithmetic (grids have < 2^30 cells), none for its stencil
// neighbours, and loads with a scalar base and a 32-bit offset.
struct Pos {
  unsigned o;
  int x, y, z;
};

__device__ __forceinline__ float ld(const float* p, unsigned o) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + o);
}

__device__ __forceinline__ void st(float* p, unsigned o, float v) {
  *reinterpret_cast<float*>(reinterpret_cast<char*>(p) + o) = v;
}

__device__ __forceinline__ Pos pos_of(const Grid& g, unsigned c) {
  Pos p;
  p.o = 4u * c;
  const unsigned t = c / (unsigned)g.nz;
  p.z = (int)(c - t * (unsigned)g.nz);
  p.x = (int)(t / (unsigned)g.ny);
  p.y = (int)(t - (unsigned)p.x * (unsigned)g.ny);
  return p;
}

// neighbour of p along axis by s (periodic, |s| <= the axis's cells)
__device__ __forceinline__ unsigned nb(const Grid& g, const Pos& p, int axis, int s) {
  const int i = axis == 0 ? p.x : (axis == 1 ? p.y : p.z), n = axis == 0 ? g.nx : (axis == 1 ? g.ny : g.nz);
  const unsigned step = 4u * (axis == 0 ? (unsigned)g.sx : (axis == 1 ? (unsigned)g.sy : 1u));
  const bool out = s < 0 ? i + s < 0 : i + s >= n;
  const unsigned in = (unsigned)s * step, wrapped = (unsigned)(s < 0 ? s + n : s - n) * step;
  return p.o + (out ? wrapped : in);
}

// step control of the FD loop: dt, t and the slotted CFL partial maxima
struct Ctl {
  float dt;
  float t;
  int steps;
  int run;  // the current step is taken (a step queued past the loop's end is not)
  unsigned cflp[3][NSLOT];
};

__device__ __forceinline__ float dss(float x) { return fsqrt(fmaxf(x, 1e-12f)); }

// Rows of a direction's frame in the state's numbering (the reference's swaps
// of (m_x, m_d) and (B_x, B_d)); an involution.
constexpr int FRAME[3][8] = {{0, 1, 2, 3, 4, 5, 6, 7}, {0, 2, 1, 3, 4, 6, 5, 7}, {0, 3, 2, 1, 4, 7, 6, 5}};

__device__ __forceinline__ int perm(int dir, int v) { return FRAME[dir][v]; }

// cell floors of the building-block routines (_eigen.py:62-74 / 148-160)
struct Cell {
  float rho, vx, vy, vz, v2, b2, p, E;
};

__device__ __forceinline__ Cell floored(const float* q, const Phys& ph) {
  Cell c;
  c.rho = q[0];
  const float ri = frcp(c.rho);
  c.vx = q[1] * ri;
  c.vy = q[2] * ri;
  c.vz = q[3] * ri;
  c.v2 = (c.vx * c.vx + c.vy * c.vy) + c.vz * c.vz;
  c.b2 = (q[5] * q[5] + q[6] * q[6]) + q[7] * q[7];
  c.E = q[4];
  c.p = ph.gm1 * (c.E - 0.5f * (c.rho * c.v2 + c.b2));
  if (c.rho < ph.rhomin || c.p < ph.pgmin) c.rho = fmaxf(c.rho, ph.rhomin);
  if (c.rho < ph.rhomin || c.p < ph.pgmin) c.p = fmaxf(c.p, ph.pgmin);
  if (c.rho < ph.rhomin || c.p < ph.pgmin) c.E = c.p * ph.inv_gm1 + 0.5f * (c.rho * c.v2 + c.b2);
  return c;
}

// (vx, c_fast, c_alfven, c_slow) of one cell (_eigenvalue_building_blocks,
// _eigen.py:27-114); the 7 eigenvalues are vx -/+ these and vx itself
__device__ __forceinline__ void cell_speeds(const float* q, float* sp, const Phys& ph) {
  const Cell c = floored(q, ph);
  const float Bx = q[5];
  const float rinv = frcp(c.rho);
  const float cs2 = fmaxf(0.f, ph.gamma * fabsf(c.p * rinv));
  const float s = c.b2 * rinv + cs2;
  const float droot = dss(fmaxf(0.f, s * s - ((4.f * (Bx * Bx)) * rinv) * cs2));
  sp[0] = c.vx;
  sp[1] = dss(fmaxf(0.f, 0.5f * (s + droot)));
  sp[2] = dss(fmaxf(0.f, (Bx * Bx) * rinv));
  sp[3] = dss(fmaxf(0.f, 0.5f * (s - droot)));
}

// _cfl_time_step_fd (_timestep_estimator.py(FD):25-87): mx[d] = max of itself and
// |lambda| of the 7 modes along d of the conserved state of the primitive row values w
__device__ __forceinline__ void cfl_speeds(const float* w, const Phys& ph, float* mx) {
  const float rho = w[0];
  const float vx = w[1], vy = w[2], vz = w[3];
  const float Bx = w[5], By = w[6], Bz = w[7];
  const float u2 = (vx * vx + vy * vy) + vz * vz;
  const float b2 = (Bx * Bx + By * By) + Bz * Bz;
  const float u[8] = {rho, rho * vx, rho * vy, rho * vz, (w[4] * ph.inv_gm1 + (0.5f * rho) * u2) + 0.5f * b2, Bx, By, Bz};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    float r[8], sp[4];
#pragma unroll
    for (int v = 0; v < 8; ++v) r[v] = u[perm(d, v)];
    cell_speeds(r, sp, ph);
    const float l[7] = {sp[0] - sp[1], sp[0] - sp[2], sp[0] - sp[3], sp[0], sp[0] + sp[3], sp[0] + sp[2], sp[0] + sp[1]};
#pragma unroll
    for (int s = 0; s < 7; ++s) {
      const float m = fabsf(l[s]);
      mx[d] = (m != m || m > mx[d]) ? m : mx[d];
    }
  }
}

// A block's maxima into its slot: an atomic only where the slot is still
// below (an L2 round trip each; at one block per 256 cells of a 256^3 grid the
// unconditional ones took longer than the pass over the state).
__device__ __forceinline__ void cfl_reduce(const float* mx, Ctl* ctl, unsigned (*sred)[4]) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const unsigned m = block_max_u<4>(canon_bits(mx[d]), sred[d]);
    if (threadIdx.x == 0) {
      unsigned* slot = &ctl->cflp[d][blockIdx.x & (NSLOT - 1)];
      if (m > __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(slot, m);
    }
  }
}

// LDS fields of a staged cell, in the direction's frame.
enum { C_Q = 0, C_F = 8, C_VX = 15, C_CF = 16, C_CA = 17, C_CS = 18, C_VY = 19, C_VZ = 20, C_H = 21, NFIELD = 22 };

// One cell of the window: conserved rows u, its flux (_fluxes.py:20-69; rows
// 0-4, 6, 7 -- the normal field's flux is 0), v_x and the fast, Alfven and slow
// speeds (_eigen.py:27-114; the 7 eigenvalues are v_x -/+ these and v_x), and
// what the interface averages need of it (_eigen.py:148-190).
__device__ __forceinline__ void stage_cell(const float* u, const Phys& ph, float* o) {
  const float rho = u[0], ri = frcp(rho);
  const float vx = u[1] * ri, vy = u[2] * ri, vz = u[3] * ri;
  const float Bx = u[5], By = u[6], Bz = u[7];
  const float u2 = (vx * vx + vy * vy) + vz * vz;
  const float b2 = (Bx * Bx + By * By) + Bz * Bz;
  const float pc = ph.gm1 * ((u[4] - (0.5f * rho) * u2) - 0.5f * b2);
  float fr = rho, fp = pc;
  if (ph.positivity) {
    fr = fmaxf(rho, ph.rhomin);
    fp = fmaxf(pc, ph.pgmin);
  }
  const float Pt = fp + 0.5f * b2;
  const float vB = (vx * Bx + vy * By) + vz * Bz;
  const float E = (fp * ph.inv_gm1 + (0.5f * fr) * u2) + 0.5f * b2;
#pragma unroll
  for (int v = 0; v < 8; ++v) o[C_Q + v] = u[v];
  o[C_F + 0] = fr * vx;
  o[C_F + 1] = ((fr * (vx * vx)) + Pt) - Bx * Bx;
  o[C_F + 2] = ((fr * vx) * vy) - Bx * By;
  o[C_F + 3] = ((fr * vx) * vz) - Bx * Bz;
  o[C_F + 4] = (E + Pt) * vx - vB * Bx;
  o[C_F + 5] = By * vx - Bx * vy;
  o[C_F + 6] = Bz * vx - Bx * vz;
  // the eigen-system's own floors (_eigen.py:62-74, 148-160)
  const bool low = rho < ph.rhomin;
  const float rinv = low ? ph.inv_rhomin : ri;
  const float pe = pc < ph.pgmin ? ph.pgmin : pc;
  const float cs2 = fmaxf(0.f, ph.gamma * fabsf(pe * rinv));
  const float s = b2 * rinv + cs2;
  const float bx2 = (Bx * Bx) * rinv;
  const float droot = dss(s * s - (4.f * bx2) * cs2);
  o[C_VX] = vx;
  o[C_CF] = dss(0.5f * (s + droot));
  o[C_CA] = dss(bx2);
  o[C_CS] = dss(0.5f * (s - droot));
  o[C_VY] = vy;
  o[C_VZ] = vz;
  o[C_H] = (u[4] + pe) * rinv;
}

// Coefficients of the characteristic fields at one interface
// (_eigen.py:116-337), the projections and the columns taken apart into the
// combinations that the fast, slow, Alfven and entropy fields share. The
// degeneracy signs of the reference (multiplying a field's row and column
// alike) drop out of row, odd WENO function and column together.
struct EB {
  float vx, vy, vz, hv2, by, bz, bty, btz, btv;
  float a1, a2, b1, b2;  // fast / slow weight of W and of T
  float c1, c2;          // fast (slow) weight of N and slow (fast) weight of S, sign of B_x apart
  float sgn, al, k3, e0;
  float af, as, cf, csl, p1, p2, z1, z2, rsr;
};

__device__ __forceinline__ float frsq(float x) { return __builtin_amdgcn_rsqf(x); }

__device__ __forceinline__ EB interface_blocks(const float* A, const float* B, const Phys& ph) {
  EB e;
  const float ra = A[0] < ph.rhomin ? ph.rhomin : A[0], rb = B[0] < ph.rhomin ? ph.rhomin : B[0];
  const float rho = 0.5f * (ra + rb);
  e.vx = 0.5f * (A[1] + B[1]);
  e.vy = 0.5f * (A[2] + B[2]);
  e.vz = 0.5f * (A[3] + B[3]);
  const float H = 0.5f * (A[4] + B[4]);
  const float bx = 0.5f * (A[5] + B[5]);
  e.by = 0.5f * (A[6] + B[6]);
  e.bz = 0.5f * (A[7] + B[7]);
  const float v2 = (e.vx * e.vx + e.vy * e.vy) + e.vz * e.vz;
  e.hv2 = 0.5f * v2;
  const float bt2 = e.by * e.by + e.bz * e.bz;
  const float ri = frcp(rho);
  const float b2r = (bx * bx + bt2) * ri;
  const float bx2r = (bx * bx) * ri;
  const float cs2 = ph.gm1 * (H - 0.5f * (v2 + b2r));
  const float cs = dss(cs2);
  const float s = b2r + cs2;
  const float droot = dss(s * s - (4.f * bx2r) * cs2);
  const float cf2 = fmaxf(0.5f * (s + droot), 1e-12f), cl2 = fmaxf(0.5f * (s - droot), 1e-12f);
  e.cf = fsqrt(cf2);
  e.csl = fsqrt(cl2);
  e.sgn = bx >= 0.f ? 1.f : -1.f;
  const float rbt = frsq(fmaxf(bt2, 1e-12f));
  e.bty = e.by * rbt;
  e.btz = e.bz * rbt;
  const float rd = frsq(fmaxf(cf2 - cl2, 1e-12f));
  e.af = dss(cs2 - cl2) * rd;
  e.as = dss(cf2 - cs2) * rd;
  const float rc = fmaxf(rho, 1e-12f);
  e.rsr = frsq(rc);
  const float sqrt_rho = rc * e.rsr;
  const float ci = cs2 > 0.f ? frcp(cs2) : 0.f;
  // rows carry 1/2 of the eigenvectors' normalisation and 1/2 of the flux splitting
  const float k = 0.25f * ci, g0 = -ph.gm1;
  const float gk = g0 * k, tk = (cs * sqrt_rho) * k;
  e.a1 = e.af * gk;
  e.a2 = e.as * gk;
  e.b1 = e.as * tk;
  e.b2 = -(e.af * tk);
  e.c1 = (e.af * e.cf) * k;
  e.c2 = (e.as * e.csl) * k;
  e.al = (0.25f * e.sgn) * sqrt_rho;
  e.k3 = (-0.5f * g0) * ci;
  e.e0 = cs2 > 0.f ? 0.5f : 0.f;
  e.btv = e.bty * e.vy + e.btz * e.vz;
  const float gam2 = (ph.gamma - 2.f) * ph.inv_gm1;
  e.p1 = e.af * (cf2 - gam2 * cs2);
  e.p2 = e.as * (cl2 - gam2 * cs2);
  const float cr = cs * e.rsr;
  e.z1 = cr * e.as;
  e.z2 = cr * e.af;
  return e;
}

// u (rows 0, 1, 2, 3, 4, 6, 7 of the conserved vector) on the 7 characteristic
// fields, order of _eigen.py: fast-, Alfven-, slow-, entropy, slow+, Alfven+, fast+
// (_eigen_L_row, _eigen.py:625-911), times 1/2.
__device__ __forceinline__ void project(const EB& e, const float* u, float* m) {
  float W = -(e.hv2 * u[0]) - u[4];
  W = e.vx * u[1] + W;
  W = e.vy * u[2] + W;
  W = e.vz * u[3] + W;
  W = e.by * u[5] + W;
  W = e.bz * u[6] + W;
  const float T = e.bty * u[5] + e.btz * u[6];
  const float A2 = e.bty * u[6] - e.btz * u[5];
  const float N = e.vx * u[0] - u[1];
  const float p2 = e.vy * u[0] - u[2], p3 = e.vz * u[0] - u[3];
  const float S = e.sgn * (e.bty * p2 + e.btz * p3);
  const float A1 = 0.25f * (e.btz * p2 - e.bty * p3);
  const float fs = e.a1 * W + e.b1 * T, fa = e.c1 * N - e.c2 * S;
  const float ss = e.a2 * W + e.b2 * T, sa = e.c2 * N + e.c1 * S;
  m[0] = fs + fa;
  m[6] = fs - fa;
  m[2] = ss + sa;
  m[4] = ss - sa;
  m[3] = e.k3 * W + e.e0 * u[0];
  m[1] = e.al * A2 + A1;
  m[5] = A1 - e.al * A2;
}

// 3 times the WENO interpolant with Jiang-Shu weights (_weno.py:185-205). The
// indicators are taken over 13 (the weights do not change, the floor of their
// sum does by 169). SAFE: one reciprocal per weight, for any finite indicator.
// Otherwise the weights share one reciprocal of their common denominator: the
// sum of products of two squared indicators, or its floor, a product of three,
// which grows faster and is the larger from differences of about 1e3 on. `den`
// returns the value that is inverted, and the caller repeats the interface the
// SAFE way above PHI_MAX, where the reciprocal would lose digits. (Looking at
// the sum alone let the floor overflow below it: weights of 0, an interpolant off
// by up to a tenth of the differences where these are 3e3 to 1e5; now within 6e-7
// of float64 from 1 to 1e8, as the SAFE form.)
constexpr float PHI_MAX = 1e37f;

template <bool SAFE>
__device__ __forceinline__ float weno_phi3(float a, float b, float c, float d, float& den) {
  const float eps = 1e-8f / 13.f, r3 = 3.f / 13.f, lim = 169e-14f;
  const float x = a - b, y = b - c, z = c - d;
  const float t0 = x - 2.f * b, t1 = b + c, t2 = 2.f * c + z;
  const float e0 = x * x + ((r3 * t0) * t0 + eps);
  const float e1 = y * y + ((r3 * t1) * t1 + eps);
  const float e2 = z * z + ((r3 * t2) * t2 + eps);
  if (SAFE) {
    const float a0 = frcp(e0 * e0) * (1.f / 169.f), a1 = frcp(e1 * e1) * (6.f / 169.f), a2 = frcp(e2 * e2) * (3.f / 169.f);
    const float rs = frcp(fmaxf((a0 + a1) + a2, 1e-14f));
    den = 0.f;
    return (a0 * rs) * (x - y) + (0.5f * (a2 * rs) - 0.25f) * (y - z);
  } else {
    const float s0 = e0 * e0, s1 = e1 * e1, s2 = e2 * e2;
    const float n0 = s1 * s2, q = 1.5f * s0;
    const float n2 = q * s1, n1 = q * s2;  // half and a quarter of them
    den = fmaxf(4.f * n1 + (2.f * n2 + n0), (lim * s0) * n0);
    const float r = frcp(den);
    return (n0 * r) * (x - y) + (n2 * r - 0.25f) * (y - z);
  }
}

struct WenoDir {
  const float* u[8];  // frame rows of the stage state: density and momenta after the
                      // floors, E and B after update_cell_center_fields
  float* F[7];        // interface flux (cell i -> face i+1/2), frame rows 0-4, 6, 7
  float* mod[2];      // CT modified fluxes of frame rows 6 and 7
};

struct WenoArgs {
  const Ctl* ctl;
  WenoDir d[3];
  unsigned first[4];  // first block of each direction, and the number of blocks
  int zin;            // interfaces of a z block
  unsigned mzp, mz;   // ceil(2^20 / (nz + 5)), ceil(2^20 / nz): quotients below 1024
  unsigned ntx, nty;  // tiles of TP positions along x and y
  Grid g;
  Phys ph;
};

constexpr int NSTAGE = (TP + 5) * TBZ;           // staged cells of a block
constexpr int NCELL = (NSTAGE + 63) / 64 * 64;  // an LDS field: whole units of ds_read2st64

__device__ __forceinline__ unsigned small_div(unsigned x, unsigned m) { return (x * m) >> 20; }

// The 7 characteristic WENO-5 fluxes of one interface added to the linear part
// (_weno.py:134-235). s: the staged cells, c: LDS index of cell i-2, ws: index
// step between window cells (known to the compiler: WS, else 0). Returns the
// largest denominator of weno_phi3.
template <bool SAFE, int WS>
__device__ __forceinline__ float interface_flux(const float (*s)[NCELL], int c, int ws, const Phys& ph, float* out) {
  // Field v of window cell k. Single reads: the compiler would pair reads, whose
  // offsets have 8 bits, and sum up addresses for them (71 to 85 of 1312
  // instructions); a single read has 16 bits, enough for every field.
  auto rd = [&](int v, int k) -> float {
    return __hip_atomic_load(&s[v][c + k * (WS ? WS : ws)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  };
  float A[8], B[8];
  {
    constexpr int f[8] = {C_Q, C_VX, C_VY, C_VZ, C_H, C_Q + 5, C_Q + 6, C_Q + 7};
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      A[v] = rd(f[v], 2);
      B[v] = rd(f[v], 3);
    }
  }
  const EB e = interface_blocks(A, B, ph);
  float df[5][7], dq[5][7];  // characteristic differences of the flux and of the state
  {
    float t[5][7];
#pragma unroll
    for (int v = 0; v < 7; ++v) {
      float w[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) w[k] = rd(C_F + v, k);
#pragma unroll
      for (int k = 0; k < 5; ++k) t[k][v] = w[k + 1] - w[k];
      out[v] = (1.0f / 12.0f) * (((-w[1] + 7.f * w[2]) + 7.f * w[3]) - w[4]);
    }
#pragma unroll
    for (int k = 0; k < 5; ++k) project(e, t[k], df[k]);
#pragma unroll
    for (int v = 0; v < 7; ++v) {
      float w[6];
      const int row = v < 5 ? v : v + 1;
#pragma unroll
      for (int k = 0; k < 6; ++k) w[k] = rd(C_Q + row, k);
#pragma unroll
      for (int k = 0; k < 5; ++k) t[k][v] = w[k + 1] - w[k];
    }
#pragma unroll
    for (int k = 0; k < 5; ++k) project(e, t[k], dq[k]);
  }
  // largest |eigenvalue| of each field over the window
  float am[7];
#pragma unroll
  for (int m = 0; m < 7; ++m) am[m] = 0.f;
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const float vx = rd(C_VX, k);
    am[3] = fmaxf(am[3], fabsf(vx));
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const float sp = rd(C_CF + m, k);
      am[m] = fmaxf(am[m], fabsf(vx - sp));
      am[6 - m] = fmaxf(am[6 - m], fabsf(vx + sp));
    }
  }
  // C_CF, C_CA, C_CS are the speeds of fields (0, 6), (1, 5), (2, 4)
  float fs[7], top = 0.f;
#pragma unroll
  for (int m = 0; m < 7; ++m) {
    const float x = am[m];
    float su, sd;
    const float up = weno_phi3<SAFE>(df[0][m] + x * dq[0][m], df[1][m] + x * dq[1][m], df[2][m] + x * dq[2][m],
                                     df[3][m] + x * dq[3][m], su);
    const float dn = weno_phi3<SAFE>(df[4][m] - x * dq[4][m], df[3][m] - x * dq[3][m], df[2][m] - x * dq[2][m],
                                     df[1][m] - x * dq[1][m], sd);
    top = fmaxf(fmaxf(top, su), sd);
    fs[m] = (dn - up) * (1.f / 3.f);
  }
  // the columns (_eigen_R_col, _eigen.py:340-622) on the shared combinations
  const float p = fs[0] + fs[6], q = fs[6] - fs[0], ps = fs[2] + fs[4], qs = fs[4] - fs[2];
  const float pa = fs[1] + fs[5], qa = (fs[1] - fs[5]) * (e.sgn * e.rsr);
  const float G = (e.af * p + e.as * ps) + fs[3];
  const float afq = e.af * e.cf, asq = e.as * e.csl;
  const float X = afq * q + asq * qs;
  const float Y = e.sgn * (afq * qs - asq * q);
  const float T2 = e.bty * Y - e.btz * pa, T3 = e.btz * Y + e.bty * pa;
  const float Z = e.z1 * p - e.z2 * ps;
  out[0] += G;
  out[1] += e.vx * G + X;
  out[2] += e.vy * G + T2;
  out[3] += e.vz * G + T3;
  out[4] += (((e.hv2 * G + e.vx * X) + e.vy * T2) + e.vz * T3) + (e.p1 * p + e.p2 * ps);
  out[5] += e.bty * Z - e.btz * qa;
  out[6] += e.btz * Z + e.bty * qa;
  return top;
}

// Interface fluxes along the three directions (_weno_flux_x/_y/_z), one
// interface per thread. A block stages the cells of its window in LDS with
// their flux, speeds and enthalpy (each thread's own work), then every thread
// computes one interface from 6 staged cells.
//   x, y: 16 positions along the direction (+ 5 halo cells) times 32 lanes that
//         run along the flattened plane of the other two axes, so that no lane
//         is idle whatever nz is (8 times 64 stages 13 cells for 8 interfaces
//         instead of 21 for 16);
//   z:    a range of `zin` interfaces in linear order; each row piece in it is
//         staged with its own 5 halo cells (wrapped in its row).
//
// Bound by VALU issue: 1190 instructions an interface, 14 WENO functions of 36
// among them. What keeps them few: differences of the window are projected
// rather than its cells (10 vectors, not 12, and the flux's cancellation happens
// before the products); the rows and columns of the seven fields share their
// sums (34 operations a vector instead of 45, and no row is ever formed); the
// three weights of a WENO function share one quarter-rate reciprocal; LDS
// offsets are immediates. LDS holds 22 fields of a cell (62 KB a block, two
// blocks of 8 waves on a CU), each read once per interface; 119 VGPRs, 4 waves a
// SIMD.
// 256^3, three directions: 3554 -> 1794 us; 101^3: 305 -> 128 us, where 64
// lanes along z of 101 cells had also left a fifth of the lanes idle; 32^3:
// 32 -> 10.7 us, three launches in one.
__global__ __launch_bounds__(NTH) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_weno(const WenoArgs a) {
  __shared__ float s[NFIELD][NCELL];
  if (!a.ctl->run) return;
  const Grid g = a.g;
  const Phys ph = a.ph;
  const int tid = threadIdx.x, w = tid / TBZ, l = tid % TBZ;
  unsigned bid = blockIdx.x;
  const int dir = bid < a.first[1] ? 0 : (bid < a.first[2] ? 1 : 2);
  bid -= a.first[dir];
  const WenoDir& D = a.d[dir];
  int ws, c0;            // window: LDS index of cell i-2 and the step to the next
  unsigned gc;           // this thread's interface (its left cell)
  bool live;
  if (dir < 2) {
    const unsigned nt = dir == 0 ? a.ntx : a.nty;
    const unsigned tile = bid % nt, pb = bid / nt;
    const unsigned np = dir == 0 ? (unsigned)g.sx : (unsigned)g.nx * (unsigned)g.nz;
    const int n = dir == 0 ? g.nx : g.ny;
    const unsigned st = dir == 0 ? (unsigned)g.sx : (unsigned)g.nz;
    const unsigned pl = pb * TBZ + l, p = pl < np ? pl : np - 1;
    unsigned base = p;
    if (dir == 1) {
      const unsigned x = p / (unsigned)g.nz;
      base = x * (unsigned)g.sx + (p - x * (unsigned)g.nz);
    }
    const int i0 = (int)tile * TP;
    for (int r = w; r < TP + 5; r += TP) {
      const unsigned gi = base + (unsigned)wrapi(i0 - 2 + r, n) * st;
      float u[8], o[NFIELD];
#pragma unroll
      for (int v = 0; v < 8; ++v) u[v] = ld(D.u[v], 4u * gi);
      stage_cell(u, ph, o);
#pragma unroll
      for (int v = 0; v < NFIELD; ++v) s[v][r * TBZ + l] = o[v];
    }
    ws = TBZ;
    c0 = w * TBZ + l;
    gc = base + (unsigned)(i0 + w) * st;
    live = pl < np && i0 + w < n;
  } else {
    const unsigned nz = (unsigned)g.nz, nc = (unsigned)g.nc, nrow = nc / nz;
    const unsigned start = bid * (unsigned)a.zin;
    const unsigned row0 = start / nz, z0 = start - row0 * nz, len0 = nz - z0;
    const unsigned left = nc - start < (unsigned)a.zin ? nc - start : (unsigned)a.zin;
    // pieces: the rest of row0, then whole rows, the last one cut
    const unsigned pieces = left <= len0 ? 1 : 1 + (left - len0 + nz - 1) / nz;
    const unsigned ncell = left + 5 * pieces;
    for (unsigned c = tid; c < ncell; c += NTH) {
      const unsigned c1 = c - (len0 + 5);
      const unsigned j = c < len0 + 5 ? 0 : 1 + small_div(c1, a.mzp);
      const unsigned at = j == 0 ? c : c1 - (j - 1) * (nz + 5);
      const int z = wrapi((int)((j == 0 ? z0 : 0) + at) - 2, (int)nz);
      const unsigned r = row0 + j < nrow ? row0 + j : nrow - 1;
      const unsigned gi = r * nz + (unsigned)z;
      float u[8], o[NFIELD];
#pragma unroll
      for (int v = 0; v < 8; ++v) u[v] = ld(D.u[v], 4u * gi);
      stage_cell(u, ph, o);
#pragma unroll
      for (int v = 0; v < NFIELD; ++v) s[v][c] = o[v];
    }
    const unsigned t = (unsigned)tid;
    const unsigned j = t < len0 ? 0 : 1 + small_div(t - len0, a.mz);
    ws = 1;
    c0 = (int)(t + 5 * j);
    gc = start + t;
    live = t < left;
  }
  __syncthreads();
  if (!live) return;
  float out[7];
  float top;
  if (dir < 2) {
    top = interface_flux<false, TBZ>(s, c0, ws, ph, out);
    // the two forms kept apart: joined at their weights (as the compiler would,
    // the code being the same) they spill 31 registers, 1.9 times the time
    asm volatile("; x, y" : "+v"(top), "+v"(out[0]), "+v"(out[1]), "+v"(out[2]), "+v"(out[3]), "+v"(out[4]), "+v"(out[5]), "+v"(out[6]));
  } else {
    top = interface_flux<false, 1>(s, c0, ws, ph, out);
    asm volatile("; z" : "+v"(top), "+v"(out[0]), "+v"(out[1]), "+v"(out[2]), "+v"(out[3]), "+v"(out[4]), "+v"(out[5]), "+v"(out[6]));
  }
  if (!(top < PHI_MAX)) {
    // opaque to the compiler, which otherwise keeps the first pass's 70
    // projections in registers for this one
    asm volatile("" : "+v"(c0));
    interface_flux<true, 0>(s, c0, ws, ph, out);
  }
#pragma unroll
  for (int v = 0; v < 7; ++v) st(D.F[v], 4u * gc, out[v]);
  // CT modified fluxes: frame rows 6 / 7 plus c2f(B_d) c2f(v_t) (_constrained_transport.py:81-102)
  float bn[4], v2[4], v3[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int c = c0 + (k + 1) * ws;
    bn[k] = s[C_Q + 5][c];
    v2[k] = s[C_VY][c];
    v3[k] = s[C_VZ][c];
  }
  const float bf = (((-bn[0] + 9.f * bn[1]) + 9.f * bn[2]) - bn[3]) * (1.f / 16.f);
  const float v2f = (((-v2[0] + 9.f * v2[1]) + 9.f * v2[2]) - v2[3]) * (1.f / 16.f);
  const float v3f = (((-v3[0] + 9.f * v3[1]) + 9.f * v3[2]) - v3[3]) * (1.f / 16.f);
  st(D.mod[0], 4u * gc, out[5] + bf * v2f);
  st(D.mod[1], 4u * gc, out[6] + bf * v3f);
}

// ---------------------------------------------------------------- stencils
__device__ __forceinline__ float c2f(const Grid& g, const float* a, const Pos& p, int ax) {
  return (((-ld(a, nb(g, p, ax, -1)) + 9.f * ld(a, p.o)) + 9.f * ld(a, nb(g, p, ax, 1))) - ld(a, nb(g, p, ax, 2))) * (1.f / 16.f);
}

// of the faces at offsets -3 .. 2
__device__ __forceinline__ float f2c_of(const float* f) {
  return (((((3.f * f[0] - 25.f * f[1]) + 150.f * f[2]) + 150.f * f[3]) - 25.f * f[4]) + 3.f * f[5]) * (1.f / 256.f);
}

__device__ __forceinline__ float f2c(const Grid& g, const float* f, const Pos& p, int ax) {
  float v[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) v[k] = ld(f, k == 3 ? p.o : nb(g, p, ax, k - 3));
  return f2c_of(v);
}

__device__ __forceinline__ float d6(const Grid& g, const float* f, const Pos& p, int ax) {
  const float c1 = 75.f / 64.f, c2 = -25.f / 384.f, c3 = 3.f / 640.f;
  return (c1 * (ld(f, p.o) - ld(f, nb(g, p, ax, -1))) + c2 * (ld(f, nb(g, p, ax, 1)) - ld(f, nb(g, p, ax, -2)))) +
         c3 * (ld(f, nb(g, p, ax, 2)) - ld(f, nb(g, p, ax, -3)));
}

__device__ __forceinline__ float p2a(const Grid& g, const float* q, const Pos& p, int A, int B) {
  const float sa = ((ld(q, nb(g, p, A, -1)) - 2.f * ld(q, p.o)) + ld(q, nb(g, p, A, 1))) * (1.f / 24.f);
  const float sb = ((ld(q, nb(g, p, B, -1)) - 2.f * ld(q, p.o)) + ld(q, nb(g, p, B, 1))) * (1.f / 24.f);
  return (ld(q, p.o) + sa) + sb;
}

#define FD_LOOP(g)                                                                     \
  for (unsigned c = blockIdx.x * blockDim.x + threadIdx.x; c < (unsigned)(g).nc; \
       c += gridDim.x * blockDim.x)

// Conserved rows of the primitive ones (rho, v, p, B), in place (_equations.py:65-101).
__device__ __forceinline__ void conserved(float* q, const Phys& ph) {
  const float rho = q[0], vx = q[1], vy = q[2], vz = q[3];
  const float u2 = (vx * vx + vy * vy) + vz * vz;
  const float b2 = (q[5] * q[5] + q[6] * q[6]) + q[7] * q[7];
  q[1] = rho * vx;
  q[2] = rho * vy;
  q[3] = rho * vz;
  q[4] = (q[4] * ph.inv_gm1 + (0.5f * rho) * u2) + 0.5f * b2;
}

// _enforce_positivity of conserved rows with the field energy b2/2 (_enforce_positivity.py:21-59)
__device__ __forceinline__ void floor_state(float& rho, float& E, const float* m, float b2, const Phys& ph) {
  rho = fmaxf(rho, ph.rhomin);
  const float ri = frcp(rho);
  const float vx = m[0] * ri, vy = m[1] * ri, vz = m[2] * ri;
  const float v2 = (vx * vx + vy * vy) + vz * vz;
  const float p = fmaxf(ph.gm1 * ((E - (0.5f * rho) * v2) - 0.5f * b2), ph.pgmin);
  E = (p * ph.inv_gm1 + (0.5f * rho) * v2) + 0.5f * b2;
}

// cell-centred B of the faces (update_cell_center_fields)
__device__ __forceinline__ void centre_field(const Grid& g, const float* const* b, const Pos& P, float* B) {
#pragma unroll
  for (int i = 0; i < 3; ++i) B[i] = f2c(g, b[i], P, i);
}

// The first stage's input: the primitive state (11 rows) as conserved rows with
// the floors, and update_cell_center_fields into qt = (E, B_x, B_y, B_z).
// Only what k_weno reads is written: the stage combines take q0 and b0 from the
// state itself, which stays as it is until the last of them. Bound by memory
// (R11 W8): with the copies of q0 in three buffers and a pass of its own for
// the floors it moved 49 fields.
struct FirstArgs {
  const Ctl* ctl;
  const float* w[11];
  float* q[4];
  float* qt[4];
  Grid g;
  Phys ph;
};

__global__ void k_first(const FirstArgs a) {
  if (!a.ctl->run) return;
  const Grid g = a.g;
  const Phys ph = a.ph;
  FD_LOOP(g) {
    const Pos P = pos_of(g, c);
    float q[8], B[3];
#pragma unroll
    for (int v = 0; v < 8; ++v) q[v] = ld(a.w[v], P.o);
    conserved(q, ph);
    const float b2 = (q[5] * q[5] + q[6] * q[6]) + q[7] * q[7];
    if (ph.positivity) floor_state(q[0], q[4], q + 1, b2, ph);
    centre_field(g, a.w + 8, P, B);
    const float nb2 = (B[0] * B[0] + B[1] * B[1]) + B[2] * B[2];
#pragma unroll
    for (int v = 0; v < 4; ++v) st(a.q[v], P.o, q[v]);
    st(a.qt[0], P.o, q[4] + 0.5f * (nb2 - b2));
#pragma unroll
    for (int i = 0; i < 3; ++i) st(a.qt[1 + i], P.o, B[i]);
  }
}

// edge EMFs (_constrained_transport.py:104-131)
struct EdgeArgs {
  const Ctl* ctl;
  const float* fyx;  // B_y flux at x-faces (modified)
  const float* fzx;  // B_z flux at x-faces
  const float* fxy;  // B_x flux at y-faces
  const float* fzy;  // B_z flux at y-faces
  const float* fyz;  // B_y flux at z-faces
  const float* fxz;  // B_x flux at z-faces
  float* O[3];       // Omega_x, Omega_y, Omega_z
  Grid g;
};

__global__ void k_ct_edge(const EdgeArgs a) {
  if (!a.ctl->run) return;
  const Grid g = a.g;
  FD_LOOP(g) {
    const Pos P = pos_of(g, c);
    const float oz = c2f(g, a.fxy, P, 0) - c2f(g, a.fyx, P, 1);
    const float ox = c2f(g, a.fyz, P, 1) - c2f(g, a.fzy, P, 2);
    const float oy = c2f(g, a.fzx, P, 2) - c2f(g, a.fxz, P, 0);
    st(a.O[2], P.o, oz);
    st(a.O[0], P.o, ox);
    st(a.O[1], P.o, oy);
  }
}

struct AvgArgs {
  const Ctl* ctl;
  const float* O[3];
  float* Ob[3];
  Grid g;
};

__global__ void k_ct_avg(const AvgArgs a) {
  if (!a.ctl->run) return;
  const Grid g = a.g;
  FD_LOOP(g) {
    const Pos P = pos_of(g, c);
    const float oz = p2a(g, a.O[2], P, 0, 1), ox = p2a(g, a.O[0], P, 1, 2), oy = p2a(g, a.O[1], P, 0, 2);
    st(a.Ob[2], P.o, oz);
    st(a.Ob[0], P.o, ox);
    st(a.Ob[1], P.o, oy);
  }
}

// SSPRK(5,4) coefficients (_ssprk.py:247-272)
struct Coef {
  float k1, k2, k3, ff;  // q0 weight, dt weight, current weight, final-state weight
};

// What a stage reads and writes of the carried buffers: the first stage has
// k3 = ff = 0; the second is the first to accumulate into the final state
// (seeded with ff0 q0, _ssprk.py:321-324); the last adds to it only.
enum { ST_FIRST = 0, ST_SECOND = 1, ST_MID = 2, ST_LAST = 3 };

struct FaceArgs {
  const float* Ob[3];
  const float* b0[3];
  float* bc[3];
  float* bf[3];
  const Ctl* ctl;
  float inv_dx, ff0;
  Coef k;
  Grid g;
};

// 6th-order curl of the averaged EMFs and the stage combine of the faces
template <int ST>
__global__ void k_face(const FaceArgs a) {
  if (!a.ctl->run) return;
  const Grid g = a.g;
  const float dtdx = (a.k.k2 * a.ctl->dt) * a.inv_dx;
  FD_LOOP(g) {
    const Pos P = pos_of(g, c);
    const float r[3] = {(-dtdx) * d6(g, a.Ob[2], P, 1) + dtdx * d6(g, a.Ob[1], P, 2),
                        (-dtdx) * d6(g, a.Ob[0], P, 2) + dtdx * d6(g, a.Ob[2], P, 0),
                        (-dtdx) * d6(g, a.Ob[1], P, 0) + dtdx * d6(g, a.Ob[0], P, 1)};
    // every load before the first store, which the compiler may not move them past
    float bn[3], bf[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      bf[i] = ST >= ST_MID ? ld(a.bf[i], P.o) : 0.f;
      if (ST == ST_LAST) {
        bf[i] = bf[i] + r[i];
        continue;
      }
      const float b0 = ld(a.b0[i], P.o);
      bn[i] = ST == ST_FIRST ? __fmul_rn(a.k.k1, b0) + r[i] : (a.k.k1 * b0 + a.k.k3 * ld(a.bc[i], P.o)) + r[i];
      if (ST == ST_SECOND) bf[i] = __fmul_rn(a.ff0, b0);
      bf[i] = bf[i] + bn[i] * a.k.ff;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (ST != ST_LAST) st(a.bc[i], P.o, bn[i]);
      if (ST != ST_FIRST) st(a.bf[i], P.o, bf[i]);
    }
  }
}

struct CombineArgs {
  const float* F[3][8];  // interface fluxes of the state's rows (none for the normal field)
  float* w[11];          // the state at the step's start; the last stage writes it
  float* qc[8];
  float* qf[8];
  const float* b[3];     // the stage's new faces
  float* qt[4];
  Ctl* ctl;
  float inv_dx, ff0;
  int want_cfl;          // last stage: the CFL maxima of the new state
  int floors;            // of the next stage's input
  Coef k;
  Grid g;
  Phys ph;
};

// Flux divergence (_ssprk.py:224-228), the stage combine (_ssprk.py:300-311) and
// the next stage's input in one pass: floors and update_cell_center_fields; after
// the last stage the final field update, floors (_ssprk.py:336-347) and the
// conserved -> primitive map with the faces appended (_evolve_state.py:63-71).
// Bound by memory: R21 fluxes + 3 faces + 8 to 24 carried rows, W12 to 20 (last
// stage R32 W11). As a pass of its own each, the combine, the floors with the
// field update, the start and the end of a step moved 461 fields a step instead
// of 302.
template <int ST>
__global__ void k_combine(const CombineArgs a) {
  __shared__ unsigned sred[3][4];
  if (!a.ctl->run) return;
  float mx[3] = {0.f, 0.f, 0.f};
  const Grid g = a.g;
  const Phys ph = a.ph;
  const float dtdx = (a.k.k2 * a.ctl->dt) * a.inv_dx;
  FD_LOOP(g) {
    const Pos P = pos_of(g, c);
    const unsigned xm = nb(g, P, 0, -1), ym = nb(g, P, 1, -1), zm = nb(g, P, 2, -1);
    // Every load first, and kept there by the scheduling barrier: left to
    // itself the compiler paired them with their uses, two in flight at a time
    // (1119 instead of 882 us in the stages that carry all rows).
    float q0[8], q[8], qf[8], qc[8], B[3], f0[3][8], f1[3][8], bf[3][6];
#pragma unroll
    for (int v = 0; v < 8; ++v) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        if (v == 5 + d) continue;
        f0[d][v] = ld(a.F[d][v], P.o);
        f1[d][v] = ld(a.F[d][v], d == 0 ? xm : (d == 1 ? ym : zm));
      }
      if (ST != ST_LAST) q0[v] = ld(a.w[v], P.o);
      if (ST >= ST_MID) qf[v] = ld(a.qf[v], P.o);
      if (ST == ST_SECOND || ST == ST_MID) qc[v] = ld(a.qc[v], P.o);
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
      for (int k = 0; k < 6; ++k) bf[i][k] = ld(a.b[i], k == 3 ? P.o : nb(g, P, i, k - 3));
    }
    __builtin_amdgcn_sched_barrier(0);
    if (ST != ST_LAST) conserved(q0, ph);
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      float div = v == 5 ? 0.f : f0[0][v] - f1[0][v];
      if (v != 6) div += f0[1][v] - f1[1][v];
      if (v != 7) div += f0[2][v] - f1[2][v];
      const float rhs = (-dtdx) * div;
      if (ST == ST_LAST) {
        q[v] = qf[v] + rhs;
        continue;
      }
      q[v] = ST == ST_FIRST ? __fmul_rn(a.k.k1, q0[v]) + rhs : (a.k.k1 * q0[v] + a.k.k3 * qc[v]) + rhs;
      if (ST == ST_SECOND) qf[v] = __fmul_rn(a.ff0, q0[v]);
      if (ST != ST_FIRST) qf[v] = qf[v] + q[v] * a.k.ff;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) B[i] = f2c_of(bf[i]);
    const float ob2 = (q[5] * q[5] + q[6] * q[6]) + q[7] * q[7];
    const float nb2 = (B[0] * B[0] + B[1] * B[1]) + B[2] * B[2];
    if (ST != ST_LAST) {
      if (a.floors) floor_state(q[0], q[4], q + 1, ob2, ph);
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        st(a.qc[v], P.o, q[v]);
        if (ST != ST_FIRST) st(a.qf[v], P.o, qf[v]);
      }
      st(a.qt[0], P.o, q[4] + 0.5f * (nb2 - ob2));
#pragma unroll
      for (int i = 0; i < 3; ++i) st(a.qt[1 + i], P.o, B[i]);
    } else {
      float rho = q[0], E = q[4] + 0.5f * (nb2 - ob2);
      if (ph.positivity) floor_state(rho, E, q + 1, nb2, ph);
      const float ri = frcp(rho);
      const float ux = q[1] * ri, uy = q[2] * ri, uz = q[3] * ri;
      const float u2 = (ux * ux + uy * uy) + uz * uz;
      float p = ph.gm1 * ((E - (0.5f * rho) * u2) - 0.5f * nb2);
      if (ph.positivity) {
        rho = fmaxf(rho, ph.rhomin);
        p = fmaxf(p, ph.pgmin);
      }
      st(a.w[0], P.o, rho);
      st(a.w[1], P.o, ux);
      st(a.w[2], P.o, uy);
      st(a.w[3], P.o, uz);
      st(a.w[4], P.o, p);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        st(a.w[5 + i], P.o, B[i]);
        st(a.w[8 + i], P.o, bf[i][3]);
      }
      if (a.want_cfl) {
        const float wn[8] = {rho, ux, uy, uz, p, B[0], B[1], B[2]};
        cfl_speeds(wn, ph, mx);
      }
    }
  }
  if (ST == ST_LAST && a.want_cfl) cfl_reduce(mx, a.ctl, sred);
}

struct StepParams {
  float t_end, C, dx, dt_max;
  int fixed, num_timesteps, exact_end;
  int any_time;      // no loop: the step size of a state by itself
  int clamp_tp = 0;  // clamp dt to tp - t (snapshot time points, time_integration.py:671-674)
  float tp = 0.f;
};

// One wavefront, a lane per partial slot; the scalars are the same in every
// lane, and everything read is loaded before the first store.
//
// END: the end of a step. BEGIN: the next step's dt = min(C dx / (lx + ly + lz),
// dt_max) (_timestep_estimator.py(FD):89-90), or t_end / num_timesteps; clamp to
// t_end - t (time_integration.py:667-678); and whether there is one.
template <bool END, bool BEGIN>
__device__ __forceinline__ void step_control(Ctl* c, const StepParams& p) {
  const int run = c->run;
  const float dt0 = c->dt;
  float t = c->t;
  int steps = c->steps;
  unsigned m[3] = {0u, 0u, 0u};
  if (BEGIN) {
#pragma unroll
    for (int d = 0; d < 3; ++d) m[d] = c->cflp[d][threadIdx.x];
  }
  if (END && run) {
    t = t + dt0;
    steps += 1;
    c->t = t;
    c->steps = steps;
  }
  if (!BEGIN) return;
  const int go = p.fixed ? steps < p.num_timesteps : (p.any_time || t < p.t_end);
  c->run = go;
  if (!go) return;
  float dt;
  if (p.fixed) {
    dt = p.t_end / (float)p.num_timesteps;
  } else {
    float l[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) l[d] = __uint_as_float(wave_max_u(m[d]));
    dt = (p.C * p.dx) / ((l[0] + l[1]) + l[2]);
    dt = p.dt_max < dt ? p.dt_max : dt;
  }
  if (p.clamp_tp) {
    const float rem = p.tp - t;
    dt = rem < dt ? rem : dt;
  }
  if (p.exact_end) {
    const float rem = p.t_end - t;
    dt = rem < dt ? rem : dt;
  }
  c->dt = dt;
#pragma unroll
  for (int d = 0; d < 3; ++d) c->cflp[d][threadIdx.x] = 0u;
}

__global__ void k_step_begin(Ctl* c, StepParams p) { step_control<false, true>(c, p); }
__global__ void k_step_end(Ctl* c) { step_control<true, false>(c, StepParams()); }
__global__ void k_step_end_begin(Ctl* c, StepParams p) { step_control<true, true>(c, p); }

__global__ void k_set_dt(Ctl* c, const float* dtp) {
  c->dt = *dtp;
  c->run = 1;
}

__global__ void k_reset(Ctl* c) {
  c->dt = 0.f;
  c->t = 0.f;
  c->steps = 0;
  c->run = 0;
  for (int d = 0; d < 3; ++d) c->cflp[d][threadIdx.x] = 0u;
}

__global__ void k_dt_out(const Ctl* c, float* out) { *out = c->dt; }

}  // namespace fd
}  // namespace amx

// ============================================================================
// C ABI
// ============================================================================

using namespace amx;
using namespace amx::fd;

struct amx_fd_ctx {
  amx_fd_config cfg;
  Grid g;
  Phys ph;
  float dx, inv_dx;
  float* ws;
  // buffer offsets (fields of nc floats)
  float *QC[8], *QF[8], *QT[4], *F[3][7], *MOD[6], *OM[3], *OMB[3], *BC[3], *BF[3];
  Ctl* ctl;
  Ctl* hctl;
  int timing;
  std::vector<hipEvent_t> ev;
  std::vector<int> pend;  // pairs of event indices of WENO launches
  int ev_used;
  double weno_ms;
  long weno_launches;
  void* snapwork;  // snapshot diagnostics partials (allocated on first use)
  amx_step_hook hook;  // between-step hook of the step loop (forcing), or null
  void* hook_user;
};

namespace {

constexpr int FD_FIELDS = 8 * 2 + 4 + 7 * 3 + 6 + 3 + 3 + 3 + 3;  // 59

amx_status fd_validate(const amx_fd_config* c) {
  if (!c) return amx_fail(AMX_ERR_INVALID, "null config%s");
  if (c->nx < 6 || c->ny < 6 || c->nz < 6) return amx_fail(AMX_ERR_INVALID, "FD grid needs >= 6 cells per axis%s");
  if (!(c->grid_spacing > 0)) return amx_fail(AMX_ERR_INVALID, "grid_spacing must be positive%s");
  if ((long)c->nx * c->ny * c->nz >= (1L << 30))
    return amx_fail(AMX_ERR_INVALID, "a grid of 2^30 cells or more is not supported (32-bit cell indices)%s");
  return AMX_OK;
}

dim3 fd_grid(const amx_fd_ctx* c) {
  long b = (c->g.nc + 255) / 256;
  return dim3((unsigned)b);
}

int fd_tbegin(amx_fd_ctx* c, hipStream_t st) {
  if (!c->timing) return -1;
  if (c->ev_used + 2 > (int)c->ev.size()) {
    for (int i = 0; i < 2; ++i) {
      hipEvent_t e;
      if (hipEventCreate(&e) != hipSuccess) return -1;
      c->ev.push_back(e);
    }
  }
  const int i = c->ev_used;
  c->ev_used += 2;
  (void)hipEventRecord(c->ev[i], st);
  return i;
}

void fd_tend(amx_fd_ctx* c, hipStream_t st, int i) {
  if (i < 0) return;
  (void)hipEventRecord(c->ev[i + 1], st);
  c->pend.push_back(i);
}

void fd_tresolve(amx_fd_ctx* c) {
  for (int i : c->pend) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, c->ev[i], c->ev[i + 1]) == hipSuccess) {
      c->weno_ms += ms;
      c->weno_launches += 1;
    }
  }
  c->pend.clear();
  c->ev_used = 0;
}

// All three directions in one launch: a small grid's blocks share the chip.
hipError_t launch_weno(amx_fd_ctx* c, hipStream_t st) {
  const Grid& g = c->g;
  WenoArgs a;
  a.ctl = c->ctl;
  for (int d = 0; d < 3; ++d) {
    for (int v = 0; v < 8; ++v) {
      const int r = FRAME[d][v];
      a.d[d].u[v] = r < 4 ? c->QC[r] : c->QT[r - 4];
    }
    for (int v = 0; v < 7; ++v) a.d[d].F[v] = c->F[d][v];
    a.d[d].mod[0] = c->MOD[2 * d];
    a.d[d].mod[1] = c->MOD[2 * d + 1];
  }
  auto up = [](long n, long m) { return (unsigned)((n + m - 1) / m); };
  a.ntx = up(g.nx, TP);
  a.nty = up(g.ny, TP);
  // short rows: fewer interfaces per z block, so that their halo cells fit
  // (512 interfaces meet up to 1 + ceil(511 / nz) rows, 5 halo cells each)
  static_assert(NTH + 5 * (1 + (NTH - 1 + 16) / 17) <= NCELL && NTH / 2 + 5 * (1 + (NTH / 2 - 1 + 5) / 6) <= NCELL,
                "z blocks do not fit");
  a.zin = g.nz >= 17 ? NTH : NTH / 2;
  a.mz = up(1 << 20, g.nz);
  a.mzp = up(1 << 20, g.nz + 5);
  a.first[0] = 0;
  a.first[1] = up(g.sx, TBZ) * a.ntx;
  a.first[2] = a.first[1] + up((long)g.nx * g.nz, TBZ) * a.nty;
  a.first[3] = a.first[2] + up(g.nc, a.zin);
  a.g = g;
  a.ph = c->ph;
  const int e = fd_tbegin(c, st);
  hipLaunchKernelGGL(k_weno, dim3(a.first[3]), dim3(NTH), 0, st, a);
  fd_tend(c, st, e);
  return hipGetLastError();
}

// SSPRK(5,4) coefficients (_ssprk.py:319-343)
const float K1[5] = {1.0f, 0.44437049406734f, 0.62010185138540f, 0.17807995410773f, -2.081261929715610e-02f};
const float K2[5] = {0.39175222700392f, 0.36841059262959f, 0.25189177424738f, 0.54497475021237f, 0.22600748319395f};
const float K3[5] = {0.0f, 0.55562950593266f, 0.37989814861460f, 0.82192004589227f, 5.03580947213895e-01f};
const float FF[5] = {-2.081261929715610e-02f, 0.0f, 0.51723167208978f, -6.518979800418380e-12f, 5.03580947213895e-01f};

// one _evolve_state_fd on the (11, nx, ny, nz) state with dt in ctl->dt
amx_status fd_step(amx_fd_ctx* c, float* state, hipStream_t st, int want_cfl) {
  const long nc = c->g.nc;
  float* w[11];
  for (int v = 0; v < 11; ++v) w[v] = state + (long)v * nc;
  const dim3 grid = fd_grid(c), blk(256);
  FirstArgs ia;
  ia.ctl = c->ctl;
  for (int v = 0; v < 11; ++v) ia.w[v] = w[v];
  for (int v = 0; v < 4; ++v) {
    ia.q[v] = c->QC[v];
    ia.qt[v] = c->QT[v];
  }
  ia.g = c->g;
  ia.ph = c->ph;
  hipLaunchKernelGGL(k_first, grid, blk, 0, st, ia);
  AMX_HIPCHK(hipGetLastError());
  for (int s = 0; s < 5; ++s) {
    Coef k;
    k.k1 = K1[s];
    k.k2 = K2[s];
    k.k3 = K3[s];
    k.ff = s < 4 ? FF[s + 1] : 0.f;
    AMX_HIPCHK(launch_weno(c, st));
    EdgeArgs ea;
    ea.ctl = c->ctl;
    ea.fyx = c->MOD[0];
    ea.fzx = c->MOD[1];
    ea.fxy = c->MOD[2];
    ea.fzy = c->MOD[3];
    ea.fyz = c->MOD[4];
    ea.fxz = c->MOD[5];
    for (int i = 0; i < 3; ++i) ea.O[i] = c->OM[i];
    ea.g = c->g;
    hipLaunchKernelGGL(k_ct_edge, grid, blk, 0, st, ea);
    AMX_HIPCHK(hipGetLastError());
    AvgArgs av;
    av.ctl = c->ctl;
    for (int i = 0; i < 3; ++i) {
      av.O[i] = c->OM[i];
      av.Ob[i] = c->OMB[i];
    }
    av.g = c->g;
    hipLaunchKernelGGL(k_ct_avg, grid, blk, 0, st, av);
    AMX_HIPCHK(hipGetLastError());
    FaceArgs fa;
    for (int i = 0; i < 3; ++i) {
      fa.Ob[i] = c->OMB[i];
      fa.b0[i] = w[8 + i];
      fa.bc[i] = c->BC[i];
      fa.bf[i] = c->BF[i];
    }
    fa.ctl = c->ctl;
    fa.inv_dx = c->inv_dx;
    fa.ff0 = FF[0];
    fa.k = k;
    fa.g = c->g;
    CombineArgs qa;
    for (int v = 0; v < 8; ++v) {
      for (int d = 0; d < 3; ++d) {
        const int f = FRAME[d][v];  // frame rows 0-4, 6, 7 are stored
        qa.F[d][v] = f == 5 ? nullptr : c->F[d][f < 5 ? f : f - 1];
      }
      qa.qc[v] = c->QC[v];
      qa.qf[v] = c->QF[v];
    }
    for (int v = 0; v < 11; ++v) qa.w[v] = w[v];
    for (int v = 0; v < 4; ++v) qa.qt[v] = c->QT[v];
    for (int i = 0; i < 3; ++i) qa.b[i] = s == 4 ? c->BF[i] : c->BC[i];
    qa.ctl = c->ctl;
    qa.want_cfl = want_cfl;
    qa.inv_dx = c->inv_dx;
    qa.ff0 = FF[0];
    qa.floors = s + 1 < 4 && c->ph.positivity;  // the last stage's input has none (_ssprk.py:333-335)
    qa.k = k;
    qa.g = c->g;
    qa.ph = c->ph;
    const int kind = s == 0 ? ST_FIRST : (s == 1 ? ST_SECOND : (s < 4 ? ST_MID : ST_LAST));
    static void (*const face[])(FaceArgs) = {k_face<ST_FIRST>, k_face<ST_SECOND>, k_face<ST_MID>, k_face<ST_LAST>};
    static void (*const combine[])(CombineArgs) = {k_combine<ST_FIRST>, k_combine<ST_SECOND>, k_combine<ST_MID>,
                                                   k_combine<ST_LAST>};
    hipLaunchKernelGGL(face[kind], grid, blk, 0, st, fa);
    AMX_HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(combine[kind], grid, blk, 0, st, qa);
    AMX_HIPCHK(hipGetLastError());
  }
  return AMX_OK;
}

}  // namespace

extern "C" amx_status amx_fd_workspace_bytes(const amx_fd_config* cfg, size_t* bytes) {
  amx_status s = fd_validate(cfg);
  if (s != AMX_OK) return s;
  if (!bytes) return amx_fail(AMX_ERR_INVALID, "null output%s");
  *bytes = sizeof(float) * (size_t)FD_FIELDS * cfg->nx * cfg->ny * cfg->nz + sizeof(Ctl);
  return AMX_OK;
}

extern "C" amx_status amx_fd_create(const amx_fd_config* cfg, amx_fd_ctx** out) {
  amx_status s = fd_validate(cfg);
  if (s != AMX_OK) return s;
  if (!out) return amx_fail(AMX_ERR_INVALID, "null output%s");
  amx_fd_ctx* c = new (std::nothrow) amx_fd_ctx();
  if (!c) return amx_fail(AMX_ERR_NOMEM, "host allocation failed%s");
  c->cfg = *cfg;
  c->g.nx = cfg->nx;
  c->g.ny = cfg->ny;
  c->g.nz = cfg->nz;
  c->g.sy = cfg->nz;
  c->g.sx = (long)cfg->ny * cfg->nz;
  c->g.nc = (long)cfg->nx * cfg->ny * cfg->nz;
  c->ph.gamma = cfg->gamma;
  c->ph.gm1 = cfg->gamma - 1.0f;
  c->ph.inv_gm1 = 1.0f / c->ph.gm1;
  c->ph.rhomin = cfg->minimum_density;
  c->ph.pgmin = cfg->minimum_pressure;
  c->ph.inv_rhomin = 1.0f / cfg->minimum_density;
  c->ph.positivity = cfg->enforce_positivity ? 1 : 0;
  c->dx = (float)cfg->grid_spacing;
  c->inv_dx = (float)(1.0 / cfg->grid_spacing);
  const long nc = c->g.nc;
  if (hipMalloc((void**)&c->ws, sizeof(float) * (size_t)FD_FIELDS * nc) != hipSuccess) {
    delete c;
    return amx_fail(AMX_ERR_NOMEM, "device workspace allocation failed%s");
  }
  float* p = c->ws;
  auto take = [&](float** dst, int n) {
    for (int i = 0; i < n; ++i) {
      dst[i] = p;
      p += nc;
    }
  };
  take(c->QC, 8);
  take(c->QF, 8);
  take(c->QT, 4);
  for (int d = 0; d < 3; ++d) take(c->F[d], 7);
  take(c->MOD, 6);
  take(c->OM, 3);
  take(c->OMB, 3);
  take(c->BC, 3);
  take(c->BF, 3);
  if (hipMalloc((void**)&c->ctl, sizeof(Ctl)) != hipSuccess ||
      hipHostMalloc((void**)&c->hctl, sizeof(Ctl), hipHostMallocDefault) != hipSuccess) {
    (void)hipFree(c->ws);
    delete c;
    return amx_fail(AMX_ERR_NOMEM, "control allocation failed%s");
  }
  hipLaunchKernelGGL(k_reset, dim3(1), dim3(NSLOT), 0, 0, c->ctl);
  if (hipDeviceSynchronize() != hipSuccess) return amx_fail(AMX_ERR_HIP, "init sync failed%s");
  *out = c;
  return AMX_OK;
}

extern "C" amx_status amx_fd_destroy(amx_fd_ctx* c) {
  if (!c) return AMX_OK;
  (void)hipDeviceSynchronize();
  (void)hipFree(c->ws);
  (void)hipFree(c->ctl);
  (void)hipHostFree(c->hctl);
  if (c->snapwork) (void)hipFree(c->snapwork);
  for (auto e : c->ev) (void)hipEventDestroy(e);
  delete c;
  return AMX_OK;
}

namespace amx {
namespace fd {

struct CflArgs {
  const float* w[8];
  Grid g;
  Phys ph;
  Ctl* ctl;
};

// the CFL maxima of a state (the step loop takes them in its last k_combine)
__global__ void k_cfl(const CflArgs a) {
  __shared__ unsigned sred[3][4];
  const Grid g = a.g;
  float mx[3] = {0.f, 0.f, 0.f};
  FD_LOOP(g) {
    float w[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) w[v] = ld(a.w[v], 4u * c);
    cfl_speeds(w, a.ph, mx);
  }
  cfl_reduce(mx, a.ctl, sred);
}

}  // namespace fd
}  // namespace amx

namespace {

hipError_t fd_cfl(amx_fd_ctx* c, const float* state, hipStream_t st) {
  CflArgs a;
  for (int v = 0; v < 8; ++v) a.w[v] = state + (long)v * c->g.nc;
  a.g = c->g;
  a.ph = c->ph;
  a.ctl = c->ctl;
  const dim3 grid = fd_grid(c);  // fewer blocks, each with one atomic per direction
  hipLaunchKernelGGL(k_cfl, dim3(grid.x < 4096 ? grid.x : 4096), dim3(256), 0, st, a);
  return hipGetLastError();
}

StepParams fd_params(const amx_fd_ctx* c, const amx_fv_run* run) {
  StepParams p;
  p.t_end = run ? run->t_end : 0.f;
  p.C = c->cfg.C_cfl;
  p.dx = c->dx;
  p.dt_max = c->cfg.dt_max;
  p.fixed = run ? run->fixed_timestep : 0;
  p.num_timesteps = run ? run->num_timesteps : 1;
  p.exact_end = run ? run->exact_end_time : 0;
  p.any_time = !run;
  return p;
}

}  // namespace

extern "C" amx_status amx_fd_cfl_dt(amx_fd_ctx* c, const float* state, float* d_dt, void* stream) {
  if (!c || !state || !d_dt) return amx_fail(AMX_ERR_INVALID, "null argument%s");
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_reset, dim3(1), dim3(NSLOT), 0, st, c->ctl);
  AMX_HIPCHK(hipGetLastError());
  AMX_HIPCHK(fd_cfl(c, state, st));
  hipLaunchKernelGGL(k_step_begin, dim3(1), dim3(NSLOT), 0, st, c->ctl, fd_params(c, nullptr));
  hipLaunchKernelGGL(k_dt_out, dim3(1), dim3(1), 0, st, (const Ctl*)c->ctl, d_dt);
  AMX_HIPCHK(hipGetLastError());
  return AMX_OK;
}

extern "C" amx_status amx_fd_evolve_state(amx_fd_ctx* c, float* state, const float* d_dt, void* stream) {
  if (!c || !state || !d_dt) return amx_fail(AMX_ERR_INVALID, "null argument%s");
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_set_dt, dim3(1), dim3(1), 0, st, c->ctl, d_dt);
  AMX_HIPCHK(hipGetLastError());
  return fd_step(c, state, st, 0);
}

namespace {

// Layout of an FD state (registered_variables.py:188-198) for the snapshot
// diagnostics: max |div B| is taken over the face fields.
amx_diag_desc fd_diag_desc(const amx_fd_ctx* c, double box_size) {
  amx_diag_desc d;
  d.num_vars = 11;
  d.dim = 3;
  d.nx = c->cfg.nx;
  d.ny = c->cfg.ny;
  d.nz = c->cfg.nz;
  d.rho_row = 0;
  d.vel_row = 1;
  d.p_row = 4;
  d.mag_row = 8;
  d.div_mode = AMX_DIV_FACES;
  d.gamma = c->cfg.gamma;
  d.grid_spacing = c->cfg.grid_spacing;
  d.box_size = box_size;
  return d;
}

// The FD branch of the step loop (time_integration.py:629-801), with the
// snapshot rows of time_integration.py:539-610, 736-745 when snp is given.
amx_status fd_loop(amx_fd_ctx* c, float* state, const amx_fv_run* run, amx::snap::Driver* snp, amx_fv_stats* stats,
                   hipStream_t st) {
  hipLaunchKernelGGL(k_reset, dim3(1), dim3(NSLOT), 0, st, c->ctl);
  AMX_HIPCHK(hipGetLastError());
  StepParams sp = fd_params(c, run);
  // the end-time clamp is off with snapshot time points (time_integration.py:677)
  if (snp && snp->spec->use_timepoints) sp.exact_end = 0;
  long steps = 0;
  float t = 0.f, dt = 0.f;
  // Without snapshot rows or a hook nothing is needed from the host between
  // steps: they are queued in batches, one readback each, as many as the last
  // dt says are left (16 at most; one at first). Steps queued past the end do
  // nothing (ctl.run). The CFL maxima of a new state come from its last stage.
  const bool batch = !snp && !c->hook;
  const int want_cfl = !run->fixed_timestep;
  if (want_cfl) AMX_HIPCHK(fd_cfl(c, state, st));
  for (;;) {
    if (run->fixed_timestep) {
      if (steps >= run->num_timesteps) break;
    } else if (!(t < run->t_end)) {
      break;
    }
    if (run->max_steps >= 0 && steps >= run->max_steps) break;
    if (snp) {
      amx_status s = snp->begin(t, state, st);
      if (s != AMX_OK) return s;
      sp.clamp_tp = snp->clamp();
      if (sp.clamp_tp) sp.tp = snp->clamp_target();
    }
    long n = 1;
    if (batch) {
      long left = run->fixed_timestep ? run->num_timesteps - steps : 1;
      if (!run->fixed_timestep && dt > 0.f) {
        const float rest = (run->t_end - t) / dt;
        left = rest < 16.f ? (long)ceilf(rest) : 16;
      }
      if (run->max_steps >= 0 && run->max_steps - steps < left) left = run->max_steps - steps;
      n = left < 1 ? 1 : (left > 16 ? 16 : left);
    }
    hipLaunchKernelGGL(k_step_begin, dim3(1), dim3(NSLOT), 0, st, c->ctl, sp);
    AMX_HIPCHK(hipGetLastError());
    if (c->hook && c->hook(c->hook_user, state, &c->ctl->dt, steps, st) != 0)
      return amx_fail(AMX_ERR_INVALID, "the step hook stopped the run%s");
    for (long i = 0; i < n; ++i) {
      amx_status s = fd_step(c, state, st, want_cfl);
      if (s != AMX_OK) return s;
      if (i + 1 < n)
        hipLaunchKernelGGL(k_step_end_begin, dim3(1), dim3(NSLOT), 0, st, c->ctl, sp);
      else
        hipLaunchKernelGGL(k_step_end, dim3(1), dim3(NSLOT), 0, st, c->ctl);
      AMX_HIPCHK(hipGetLastError());
    }
    AMX_HIPCHK(hipMemcpyAsync(c->hctl, c->ctl, offsetof(Ctl, cflp), hipMemcpyDeviceToHost, st));
    AMX_HIPCHK(hipStreamSynchronize(st));
    fd_tresolve(c);
    t = c->hctl->t;
    dt = c->hctl->dt;
    steps = c->hctl->steps;
    if (snp) {
      amx_status s = snp->end(t, state, st);
      if (s != AMX_OK) return s;
    }
  }
  if (snp) snp->finish(steps);
  if (stats) {
    stats->steps = steps;
    stats->t = t;
    stats->fixed_point_iterations = 0;
    stats->max_fixed_point_iterations = 0;
  }
  return AMX_OK;
}

}  // namespace

extern "C" amx_status amx_fd_time_integration(amx_fd_ctx* c, float* state, const amx_fv_run* run, amx_fv_stats* stats,
                                              void* stream) {
  if (!c || !state || !run) return amx_fail(AMX_ERR_INVALID, "null argument%s");
  if (run->fixed_timestep && run->num_timesteps <= 0) return amx_fail(AMX_ERR_INVALID, "num_timesteps must be positive%s");
  return fd_loop(c, state, run, nullptr, stats, (hipStream_t)stream);
}

extern "C" amx_status amx_fd_time_integration_snapshots(amx_fd_ctx* c, float* state, const amx_fv_run* run,
                                                        const amx_snapshot_spec* spec, amx_snapshot_out* out,
                                                        amx_fv_stats* stats, void* stream) {
  if (!c || !state || !run || !spec) return amx_fail(AMX_ERR_INVALID, "null argument%s");
  if (run->fixed_timestep && run->num_timesteps <= 0) return amx_fail(AMX_ERR_INVALID, "num_timesteps must be positive%s");
  amx::snap::Driver d;
  d.spec = spec;
  d.out = out;
  d.desc = fd_diag_desc(c, spec->box_size);
  d.t_end = run->t_end;
  d.work = nullptr;
  amx_status s = amx::snap::validate(spec, out, d.desc);
  if (s != AMX_OK) return s;
  if (!spec->callback) {
    if (!c->snapwork && hipMalloc(&c->snapwork, amx::snap::work_bytes()) != hipSuccess) {
      c->snapwork = nullptr;
      return amx_fail(AMX_ERR_NOMEM, "snapshot workspace allocation failed%s");
    }
    d.work = c->snapwork;
  }
  return fd_loop(c, state, run, &d, stats, (hipStream_t)stream);
}

extern "C" amx_status amx_fd_set_step_hook(amx_fd_ctx* c, amx_step_hook hook, void* user) {
  if (!c) return amx_fail(AMX_ERR_INVALID, "null context%s");
  c->hook = hook;
  c->hook_user = user;
  return AMX_OK;
}

extern "C" amx_status amx_fd_set_timing(amx_fd_ctx* c, int enable) {
  if (!c) return amx_fail(AMX_ERR_INVALID, "null context%s");
  AMX_HIPCHK(hipDeviceSynchronize());
  c->pend.clear();
  c->ev_used = 0;
  c->timing = enable ? 1 : 0;
  c->weno_ms = 0.0;
  c->weno_launches = 0;
  return AMX_OK;
}

extern "C" amx_status amx_fd_get_timing(amx_fd_ctx* c, double* weno_ms, long* weno_launches) {
  if (!c || !weno_ms || !weno_launches) return amx_fail(AMX_ERR_INVALID, "null argument%s");
  AMX_HIPCHK(hipDeviceSynchronize());
  fd_tresolve(c);
  *weno_ms = c->weno_ms;
  *weno_launches = c->weno_launches;
  return AMX_OK;
}

namespace amx {
namespace fd {

// b_d = 4th-order centre-to-face interpolation of B_d along d
// (initialize_interface_fields, _constrained_transport.py:201-213)
struct C2fArgs {
  const float* B[3];
  float* b[3];
  Grid g;
};

// Cell indices here, not byte offsets: this entry point takes grids of 2^30
// cells and more, whose byte offsets do not fit in 32 bits.
__global__ void k_interface_fields(const C2fArgs a) {
  const Grid g = a.g;
  FD_LOOP(g) {
    const Pos P = pos_of(g, c);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const float* B = a.B[d];
      const int i = d == 0 ? P.x : (d == 1 ? P.y : P.z), n = d == 0 ? g.nx : (d == 1 ? g.ny : g.nz);
      const unsigned sd = d == 0 ? (unsigned)g.sx : (d == 1 ? (unsigned)g.sy : 1u);
      auto at = [&](int s) { return B[c + (unsigned)(wrapi(i + s, n) - i) * sd]; };
      a.b[d][c] = (((-at(-1) + 9.f * B[c]) + 9.f * at(1)) - at(2)) * (1.f / 16.f);
    }
  }
}

}  // namespace fd
}  // namespace amx

extern "C" amx_status amx_fd_interface_fields(const float* B, float* b, int nx, int ny, int nz, void* stream) {
  if (!B || !b) return amx_fail(AMX_ERR_INVALID, "null argument%s");
  if (nx < 3 || ny < 3 || nz < 3) return amx_fail(AMX_ERR_INVALID, "grid needs >= 3 cells per axis%s");
  if (B == b) return amx_fail(AMX_ERR_INVALID, "B and b must not alias%s");
  C2fArgs a;
  a.g.nx = nx;
  a.g.ny = ny;
  a.g.nz = nz;
  a.g.sy = nz;
  a.g.sx = (long)ny * nz;
  a.g.nc = (long)nx * ny * nz;
  for (int d = 0; d < 3; ++d) {
    a.B[d] = B + d * a.g.nc;
    a.b[d] = b + d * a.g.nc;
  }
  long nb = (a.g.nc + 255) / 256;
  if (nb > 256L * 64) nb = 256L * 64;
  hipLaunchKernelGGL(k_interface_fields, dim3((unsigned)nb), dim3(256), 0, (hipStream_t)stream, a);
  AMX_HIPCHK(hipGetLastError());
  return AMX_OK;
}
