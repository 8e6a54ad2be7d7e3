// tsm_stage.hip -- the stage kernel: one workgroup per vertex tile.
//
// One launch per Runge-Kutta stage does everything of the stage for a tile
// (src/fv.cc:699-1059, :1066-1192, :1197-1312, :1635-1707): states of the
// tile's slots into LDS, entropy-variable gradients of the owned vertices and
// the first halo ring (so that both ends of every local face have theirs),
// every local face's flux, the gather per owned vertex in reference face order,
// periodic set sums, viscous terms, boundary fluxes and the update.  The last
// stage also forms the residual-norm partials (src/fv.cc:1801-1879) and the
// next step's local time step (src/fv.cc:1499-1621) from the new state, so a
// step needs no separate time-step pass.  No atomics on floating-point values.
// Every sum that a state depends on has one order, whatever the tile size; the
// residual norm is a sum over tiles and has one order for each number of tiles.
//
// What bounds it: at 1025^2 (KEPES-TeCNO Rusanov, minmod) a stage's FP64
// issue (0.60 of the rate), LDS (0.36) and HBM traffic (2.8 of 4.9 TB/s) are within
// a factor of two of each other, and a tile's phases depend on one another through
// barriers, so the layout is chosen to keep four tiles per CU in different phases.
// Under a kernel trace a stage takes 95 us, the last 117 and the launch that ends the
// step 10 (with gradients in launches of their own: 98, the last 124, and 58 more a
// stage); a step by itself 301 us (492).  On small meshes a stage is one tile's chain,
// 10 to 13 us.
//  - gradients never go through memory.  A second launch and a 64-byte record
//    per vertex written and read back by every neighbouring tile cost more than
//    forming the first ring's gradients twice;
//  - the gradient of a vertex v is the sum over its cells (v, b, d) of
//    N_b (V_b - V_v) + N_d (V_d - V_v) with the coordinates taken relative to
//    v: a cell's three normals sum to zero.  Walked in ring order each
//    neighbour is read once, 16 multiply-adds a cell;
//  - the one entropy variable that needs logarithms is kept per vertex beside
//    the state (V_in/V_out) by the stage that forms the state: two logarithms
//    per owned vertex instead of four per slot.  The others are multiples of
//    beta = 1/(2RT), formed where they are used;
//  - slot and face records are contiguous in LDS (48, 80 and 48 bytes) and
//    read 16 bytes at a time: addresses are one multiply with immediate
//    offsets, and 16 successive records fall on 16 different bank groups.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "tsm_device.h"
#include "tsm_physics.h"

namespace tsm {
namespace {

// XCD-aware tile order.  Workgroups go to the chip's 8 XCDs in turn (block b
// to XCD b mod 8), each XCD with its own L2.  Block b of a row of n tiles
// takes tile start(x) + b/8 of the contiguous range of XCD x = b mod 8, so
// every XCD walks a compact run of neighbouring tiles and the halo records
// it reads are mostly the owned records of tiles it has just staged (a
// bijection of [0, n): XCD x gets n/8 tiles, one more for the first n mod 8).
__device__ __forceinline__ int xcd_tile(int b, int n) {
  const int x = b % 8, j = b / 8;
  const int q = n / 8, rem = n % 8;
  return x * q + min(x, rem) + j;
}

__device__ __forceinline__ Prim ld_prim(const double* W, size_t i) {
  const double4 q = reinterpret_cast<const double4*>(W)[i];
  return Prim{q.x, q.y, q.z, q.w};
}
__device__ __forceinline__ double2 lds2(const double* p) { return *reinterpret_cast<const double2*>(p); }
__device__ __forceinline__ void sts2(double* p, double a, double b) {
  *reinterpret_cast<double2*>(p) = make_double2(a, b);
}

template <int FLUX, int REC>
struct Layout {
  static constexpr bool TEC = FLUX == F_ROE || FLUX == F_RUS;
  static constexpr bool GRAD = TEC && REC != R_FIRST;
  static constexpr bool PT = !TEC && FLUX != F_KEPEC;  // fluxes of (T, p)
  // record A per slot: u v | beta V0 | x y (KEPEC: rho for V0; PT: unused)
  static constexpr int NA = 6;
  // record B per gradient slot: dE x8 | rho c (without gradients: rho c, or T p)
  static constexpr int NB = GRAD ? 10 : (FLUX == F_KEPEC ? 0 : 2);
};
constexpr int NFR = 6;   // record per local face: flux x4 | normal
constexpr int NBT = 6;   // record per boundary term: normal | dq x4
constexpr int NWT = 12;  // record per wall term: flux of the three corners, wall flux
constexpr int NVC = 6;   // record per viscous cell: its flux to the first two corners
constexpr int FPT = 2;   // faces per thread
constexpr int SR_VERTS = 64;  // owned vertices of a tile with periodic sets: at most a quarter of 256

// Cell viscous flux: stress and energy flux per unit normal from the mean
// entropy variables (vx, vy, l) and their gradients (x, y each)
// (src/material.cc:158-230).  F.n = -(t n); e1 = without the conducted heat.
struct ViscTensor { double xx, xy, yy, ex, ey, qx, qy; };
__device__ __forceinline__ ViscTensor visc_tensor(const Gas& gas, const ViscParams& vp, double vx,
                                                  double vy, double l, const double* d) {
#pragma clang fp contract(fast)
  const double il = frcp(l);
  const double u = -vx * il, v = -vy * il;
  double mu;
  if (vp.mu_model == 0) {
    mu = vp.mu_ref;
  } else {
    const double T = fdiv(-1.0, gas.R * l);
    mu = vp.mu_model == 1 ? fdiv(vp.mu_ref * pow(T, 1.5), T + vp.T_0)
                          : vp.mu_ref * pow(fdiv(T, vp.T_ref), vp.omega);
  }
  // kappa / R = mu gamma / ((gamma - 1) Pr)
  const double kr = vp.heat_active ? mu * (gas.gamma * gas.ig1) * vp.iprandtl : 0.0;
  if (!vp.visc_active) mu = 0.0;
  const double ux = -il * (d[0] + u * d[4]), uy = -il * (d[1] + u * d[5]);
  const double wx = -il * (d[2] + v * d[4]), wy = -il * (d[3] + v * d[5]);
  const double m23 = mu * (2.0 / 3.0);
  ViscTensor t;
  t.xx = m23 * (2.0 * ux - wy);
  t.yy = m23 * (2.0 * wy - ux);
  t.xy = mu * (uy + wx);
  const double q = kr * il * il;
  t.qx = q * d[4];
  t.qy = q * d[5];
  t.ex = u * t.xx + v * t.xy + t.qx;
  t.ey = u * t.xy + v * t.yy + t.qy;
  return t;
}

// Half the boundary correction of one bface to its cell's gradient
// (src/fv.cc:926-966): the mean of the boundary states' entropy variables minus
// the mean of the vertices' own, at both ends.
__device__ __forceinline__ void flux_vars(const Gas& gas, const Prim& w, double* V) {
  V[3] = -fdiv(1.0, gas.R * w.T);
  V[0] = entropy_var0(gas, w);
  V[1] = -w.u * V[3];
  V[2] = -w.v * V[3];
}
// This is end e's share of it; V0: its own first entropy variable where that is
// kept, else null.
__device__ __forceinline__ void boundary_dq(const DevGeo& G, const StageArgs& A, const Gas& gas,
                                            int s, size_t off, int b, int e, int v,
                                            const double* V0, double* dq) {
  const Prim w = ld_prim(A.W_in, off + v);
  Prim x = w;
  bc_apply1(G.btype[b], bc_values(G, s, b, e), G.bn[2 * b], G.bn[2 * b + 1], x);
  double V[4], Vb[4];
  V[3] = -fdiv(1.0, gas.R * w.T);
  V[0] = V0 ? V0[off + v] : entropy_var0(gas, w);
  V[1] = -w.u * V[3];
  V[2] = -w.v * V[3];
  flux_vars(gas, x, Vb);
#pragma unroll
  for (int q = 0; q < 4; ++q) dq[q] = 0.5 * (Vb[q] - V[q]);
}

// The state of a wall cell (wall_cell_state) from its term's wall faces: vertices,
// bface with the vertices' ends of it in the top bits, face.
__device__ __forceinline__ Ent wall_state(const DevGeo& G, const double* W, size_t off, int s,
                                          const Gas& gas, const uint4* faces) {
  Ent e{0.0, 0.0, 0.0, 0.0};
  int n = 0;
  for (int t = 0; t < 2; ++t) {
    const uint4 q = faces[t];
    const int f = (int)q.w, b = (int)(q.z & 0x3fffffffu);
    if (f < 0) break;
    const int type = G.btype[b];
    const double nx = G.fn[2 * f], ny = G.fn[2 * f + 1];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      Prim st = ld_prim(W, off + (k ? q.y : q.x));
      bc_apply1(type, bc_values(G, s, b, (q.z >> (30 + k)) & 1), nx, ny, st);
      const Ent x = prim2ent(gas, st);
      e.vx += x.vx; e.vy += x.vy; e.l += x.l;
    }
    ++n;
  }
  const double sc = 0.5 * 1.0 / n;
  e.vx *= sc; e.vy *= sc; e.l *= sc;
  return e;
}

template <int FLUX, int REC>
__device__ __forceinline__ Cons pair_flux(const Gas& gas, const FluxOpts& fo, double rx, double ry,
                                          const Side& L, const Side& R, const double* gdl,
                                          const double* gdr, double unx, double uny, double ssw) {
  if (FLUX == F_ROE || FLUX == F_RUS)
    return tecno_flux<FLUX == F_ROE, REC>(gas, fo, rx, ry, L, R, gdl, gdr, unx, uny, ssw);
  if (FLUX == F_KEPEC) return kepec_flux_s(gas, L, R, unx, uny);
  if (FLUX == F_KEP) return kep_flux(gas, L.w, R.w, unx, uny);
  if (FLUX == F_ROEEC) return roe_ec_flux(gas, L.w, R.w, unx, uny);
  return avg_flux(gas, L.w, R.w, unx, uny);
}

// Boundary flux of bface b, normal (nx, ny), at its end e with state wm
// (src/fv.cc:1100-1189)
template <int FLUX, int REC>
__device__ __forceinline__ Cons bflux(const DevGeo& G, const FluxOpts& fo, const Gas& gas, int b,
                                   int s, int e, double nx, double ny, const Prim& wm) {
  const int type = G.btype[b];
  Prim s0 = wm, s1 = wm;
  bc_apply2(type, bc_values(G, s, b, e), nx, ny, s0, s1);
  if (type == TSM_BC_FARFIELD) {
    double area = fsqrt(nx * nx + ny * ny);
    double ia = fdiv(1.0, area);
    const double z[4] = {0, 0, 0, 0};
    constexpr bool TEC = FLUX == F_ROE || FLUX == F_RUS;
    Side L = make_side<TEC, FLUX == F_ROE>(gas, s0), R = make_side<TEC, FLUX == F_ROE>(gas, s1);
    Cons F = pair_flux<FLUX, REC>(gas, fo, 0.0, 0.0, L, R, z, z, nx * ia, ny * ia, 0.0);
    F.m *= area; F.mx *= area; F.my *= area; F.e *= area;
    return F;
  }
  return inviscid_bflux(gas, s0, s1, nx, ny);
}

// Walk around a gradient slot, neighbour by neighbour in ring order.  acc: the
// sum over the cells of G_c = 2 A_c grad V with V and the coordinates relative to
// the centre.  A neighbour w between a and b belongs to the cells (centre, a, w)
// and (centre, w, b), so its share of acc is V_w times the rotated b - a: eight
// multiply-adds a neighbour.  Where the chain ends the missing neighbour is the
// centre itself (zero), and a closed chain's ends are each other's neighbours.
struct Rel { double x, y, q0, q1, q2, q3; };
struct Fan {
  double cx, cy, c0, c1, c2, c3;  // centre
  Rel p, first;                   // previous neighbour, first of the chain
  double ax, ay;                  // the one before the previous
  bool closed;
};
// entropy variables of a slot record
__device__ __forceinline__ void slot_vars(const double2& uv, const double2& bV, double& v0, double& v1,
                                          double& v2, double& v3) {
  const double b2 = 2.0 * bV.x;
  v0 = bV.y;
  v1 = uv.x * b2;
  v2 = uv.y * b2;
  v3 = -b2;
}
__device__ __forceinline__ Rel fan_rel(const Fan& f, const double* SA, unsigned e) {
  const double* a = SA + 6 * (e & SI_MASK);
  const double2 uv = lds2(a), bV = lds2(a + 2), xy = lds2(a + 4);
  Rel r;
  slot_vars(uv, bV, r.q0, r.q1, r.q2, r.q3);
  r.q0 -= f.c0; r.q1 -= f.c1; r.q2 -= f.c2; r.q3 -= f.c3;
  r.x = xy.x - f.cx;
  r.y = xy.y - f.cy;
  return r;
}
__device__ __forceinline__ void fan_share(double ex, double ey, const Rel& w, double* acc) {
  acc[0] = __builtin_fma(ey, w.q0, acc[0]); acc[1] = __builtin_fma(-ex, w.q0, acc[1]);
  acc[2] = __builtin_fma(ey, w.q1, acc[2]); acc[3] = __builtin_fma(-ex, w.q1, acc[3]);
  acc[4] = __builtin_fma(ey, w.q2, acc[4]); acc[5] = __builtin_fma(-ex, w.q2, acc[5]);
  acc[6] = __builtin_fma(ey, w.q3, acc[6]); acc[7] = __builtin_fma(-ex, w.q3, acc[7]);
}
__device__ __forceinline__ void fan_centre(Fan& f, const double* SA, int slot) {
  const double* a = SA + 6 * slot;
  const double2 uv = lds2(a), bV = lds2(a + 2), xy = lds2(a + 4);
  slot_vars(uv, bV, f.c0, f.c1, f.c2, f.c3);
  f.cx = xy.x; f.cy = xy.y;
}
__device__ __forceinline__ void fan_first(Fan& f, const Rel& w, unsigned e) {
  f.first = f.p = w;
  f.ax = f.ay = 0.0;
  f.closed = (e & SI_CLOSED) != 0;
}
__device__ __forceinline__ void fan_next(Fan& f, const Rel& w, double* acc) {
  fan_share(w.x - f.ax, w.y - f.ay, f.p, acc);
  f.ax = f.p.x; f.ay = f.p.y;
  f.p = w;
}
__device__ __forceinline__ void fan_end(Fan& f, double* acc) {
  const double ex = f.closed ? f.first.x : 0.0, ey = f.closed ? f.first.y : 0.0;
  fan_share(ex - f.ax, ey - f.ay, f.p, acc);
  if (f.closed) fan_share(-f.p.x, -f.p.y, f.first, acc);
}
__device__ __forceinline__ unsigned item_at(const uint4& it, int u) {
  const unsigned w[4] = {it.x, it.y, it.z, it.w};
  return (w[u >> 1] >> (16 * (u & 1))) & 0xffffu;
}
// the first chain, up to eight neighbours
__device__ __forceinline__ void walk_chain(Fan& f, const uint4& it, const double* SA, double* acc) {
  fan_first(f, fan_rel(f, SA, item_at(it, 0)), item_at(it, 0));
#pragma unroll
  for (int u = 1; u < 8; ++u) {
    const unsigned e = item_at(it, u);
    if (e < SI_CENTRE) fan_next(f, fan_rel(f, SA, e), acc);
  }
  fan_end(f, acc);
}
// One group of a slot's extras: a further chain around its own or another centre
// (periodic sets) or boundary terms.  Few slots of a tile have any, and those of a
// tile are mostly alike, so a group is unrolled like the first chain: entry by
// entry in a loop, a tile with periodic vertices took 18,600 cycles for its
// gradients instead of 3,000.
__device__ __forceinline__ void walk_group(Fan& f, const uint4& g, const double* SA, const double* SBT,
                                           double* acc) {
  const unsigned head = item_at(g, 0);
  if (head < SI_TERM) {
    unsigned e = item_at(g, 1);
    if (!(head & SI_FLAG)) {
      fan_centre(f, SA, head & SI_MASK);
      fan_first(f, fan_rel(f, SA, e), e);
    } else {
      fan_next(f, fan_rel(f, SA, e), acc);
    }
#pragma unroll
    for (int u = 2; u < 8; ++u) {
      e = item_at(g, u);
      if (e < SI_CENTRE) fan_next(f, fan_rel(f, SA, e), acc);
    }
    if (!(head & SI_CLOSED)) fan_end(f, acc);
  } else {
#pragma unroll
    for (int u = 1; u < 8; ++u) {
      const unsigned e = item_at(g, u);
      if (e >= SI_END) continue;
      const double* b = SBT + NBT * (e & SI_MASK);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        acc[2 * q] = __builtin_fma(b[0], b[2 + q], acc[2 * q]);
        acc[2 * q + 1] = __builtin_fma(b[1], b[2 + q], acc[2 * q + 1]);
      }
    }
  }
}

// One viscous cell from its corners' records: the flux to its first two corners
// (half of -t n with n the corner's cell normal, that is the rotated opposite
// side).  The third corner's is minus their sum: the normals sum to zero.
__device__ __forceinline__ void viscous_cell(unsigned x, const double* SA, const Gas& gas,
                                             const ViscParams& vp, double* out) {
#pragma clang fp contract(fast)
  Fan f;
  fan_centre(f, SA, x & 1023u);
  const Rel b = fan_rel(f, SA, (x >> 10) & 1023u), d = fan_rel(f, SA, (x >> 20) & 1023u);
  const double ia = frcp(b.x * d.y - b.y * d.x);
  const double g[6] = {(d.y * b.q1 - b.y * d.q1) * ia, (b.x * d.q1 - d.x * b.q1) * ia,
                       (d.y * b.q2 - b.y * d.q2) * ia, (b.x * d.q2 - d.x * b.q2) * ia,
                       (d.y * b.q3 - b.y * d.q3) * ia, (b.x * d.q3 - d.x * b.q3) * ia};
  const double th = 1.0 / 3.0;
  const ViscTensor t = visc_tensor(gas, vp, f.c1 + (b.q1 + d.q1) * th, f.c2 + (b.q2 + d.q2) * th,
                                   f.c3 + (b.q3 + d.q3) * th, g);
  const double nx0 = 0.5 * (b.y - d.y), ny0 = 0.5 * (d.x - b.x), nx1 = 0.5 * d.y, ny1 = -0.5 * d.x;
  sts2(out, t.xx * nx0 + t.xy * ny0, t.xy * nx0 + t.yy * ny0);
  sts2(out + 2, t.ex * nx0 + t.ey * ny0, t.xx * nx1 + t.xy * ny1);
  sts2(out + 4, t.xy * nx1 + t.yy * ny1, t.ex * nx1 + t.ey * ny1);
}
__device__ __forceinline__ void viscous_add(unsigned e, const double* SVC, double* visc) {
  const double* o = SVC + NVC * (e & 0x1fffu);
  const unsigned z = e >> 13;
  const double2 a = lds2(o), b = lds2(o + 2), c = lds2(o + 4);
  if (z == 0) { visc[0] += a.x; visc[1] += a.y; visc[2] += b.x; }
  else if (z == 1) { visc[0] += b.y; visc[1] += c.x; visc[2] += c.y; }
  else { visc[0] -= a.x + b.y; visc[1] -= a.y + c.x; visc[2] -= b.x + c.y; }
}

// Residual norm, time advance, loop test and the next step's global dt
// (src/fv.cc:1591-1618, :1801-1879, :2273-2316) from the step's sums; c: the
// sample's control block as the step found it.
__device__ __forceinline__ void step_ctl(const StageArgs& A, const StepParams& P, Ctl c, int nv,
                                         const double* part, double x, int log_slot, int s) {
  double n[4];
  for (int k = 0; k < 4; ++k) {
    n[k] = sqrt(part[k]) / nv;
    c.rn[k] = n[k];
  }
  const double tot = sqrt((n[0] * n[0]) + (n[1] * n[1] + n[2] * n[2]) + (n[3] * n[3]));
  if (c.iter == 0) {
    c.res0 = tot;
    if (c.res0 == 0.0) c.res0 = 1.0;
  }
  c.res_total = tot / c.res0;
  c.iter += 1;
  c.t += c.dt;
  if (c.reached && P.unsteady) { c.counter += 1; c.reached = 0; }
  if (A.log && log_slot >= 0) {
    double* Lg = A.log + ((size_t)s * A.log_cap + log_slot) * 4;
    Lg[0] = (double)c.iter; Lg[1] = c.dt; Lg[2] = c.t; Lg[3] = c.res_total;
  }
  const bool go = c.res_total > P.min_residue && (P.unsteady ? true : c.iter < P.max_iter) &&
                  c.t < P.final_time;
  if (!go) {
    c.done = 1;
  } else {
    double dt = x;
    if (P.unsteady && !(P.time_step > 0.0)) {
      const double target = A.tstamps[min(c.counter, P.n_stamps)];
      if (c.t + dt > target) { dt = target - c.t; c.reached = 1; }
    }
    c.dt = dt;
  }
  A.ctl[s] = c;
}

// A wave's sum or minimum in its lane 63 by data-parallel primitives: shifts within
// rows of 16 lanes, then a row's last lane to the next row and the first half's to the
// second.  Lanes without a source take the neutral element z.
template <int CTRL, int ROWS, class F>
__device__ __forceinline__ double dpp_step(double x, double z, F f) {
  const long long xb = __double_as_longlong(x), zb = __double_as_longlong(z);
  const int lo = __builtin_amdgcn_update_dpp((int)zb, (int)xb, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(zb >> 32), (int)(xb >> 32), CTRL, ROWS, 0xf, false);
  return f(x, __longlong_as_double(((long long)hi << 32) | (unsigned)lo));
}
template <class F>
__device__ __forceinline__ double wave_fold(double x, double z, F f) {
  x = dpp_step<0x111, 0xf>(x, z, f);
  x = dpp_step<0x112, 0xf>(x, z, f);
  x = dpp_step<0x114, 0xf>(x, z, f);
  x = dpp_step<0x118, 0xf>(x, z, f);
  x = dpp_step<0x142, 0xa>(x, z, f);
  return dpp_step<0x143, 0xc>(x, z, f);
}
__device__ __forceinline__ double wave_sum(double x) {
  return wave_fold(x, 0.0, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ double wave_min(double x) {  // of values up to 1e20
  return wave_fold(x, 1.0e20, [](double a, double b) { return fmin(a, b); });
}

// The end of a step by one wave, from the partials of nblk blocks: lane i takes
// those of blocks i, i + 64, ... in that order, then the wave's tree.  Every mesh of
// up to FOLD_TILES tiles ends its steps so, in the last stage or in a launch of its
// own: which of the two it is depends on the samples beside this one, its norm does
// not.  LAUNCH: in the last stage's own launch, where the partials were written
// through to memory before their blocks counted themselves in and are read past the
// caches.
__device__ __forceinline__ double agent_load(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_store(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool LAUNCH>
__device__ __forceinline__ void final_wave(const StageArgs& A, const StepParams& P, int nblk, int nv,
                                           const double* dtpart, int log_slot, int s) {
  const int lane = threadIdx.x & 63;
  const Ctl c = A.ctl[s];
  if (!LAUNCH && c.done) return;
  auto load = [](const double* p) { return LAUNCH ? agent_load(p) : *p; };
  const double* q = A.partial + (size_t)s * nblk * 4;
  const double* dq = dtpart + (size_t)s * nblk;
  double part[4] = {0, 0, 0, 0}, x = 1.0e20;
  for (int i0 = 0; i0 < nblk; i0 += 8 * 64) {
    double a[8][5];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + 64 * u + lane;
#pragma unroll
      for (int k = 0; k < 4; ++k) a[u][k] = i < nblk ? load(q + 4 * (size_t)i + k) : 0.0;
      a[u][4] = i < nblk ? load(dq + i) : 1.0e20;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
#pragma unroll
      for (int k = 0; k < 4; ++k) part[k] += a[u][k];
      x = fmin(x, a[u][4]);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) part[k] = wave_sum(part[k]);
  x = wave_min(x);
  if (lane == 63) step_ctl(A, P, c, nv, part, x, log_slot, s);
}

// Per-block partials of the last stage without a block barrier: every wave with
// owned vertices reduces its residual-norm sums and smallest local dt, its lane 63
// leaves them in LDS and counts itself in with an LDS integer atomic; the
// last wave to arrive adds the waves' values in wave order and writes the
// block's slot.  Waves that finish early leave at once.  Where the sample's
// blocks are counted (A.arrive), the last block's wave ends the step.
__device__ __forceinline__ void block_partials(const StageArgs& A, const StepParams& P, double* part,
                                               double dtv, double* wred, int* arrive, double* dtpart,
                                               int s, int t, int nt, int nv, int nw, int log_slot) {
  const int w = threadIdx.x >> 6;
  if (w >= nw) return;
#pragma unroll
  for (int k = 0; k < 4; ++k) part[k] = wave_sum(part[k]);
  dtv = wave_min(dtv);
  int ends = 0;
  if ((threadIdx.x & 63) == 63) {
#pragma unroll
    for (int k = 0; k < 4; ++k) wred[5 * w + k] = part[k];
    wred[5 * w + 4] = dtv;
    __threadfence_block();
    if (atomicAdd(arrive, 1) == nw - 1) {
      __threadfence_block();
      double sum[4] = {wred[0], wred[1], wred[2], wred[3]};
      double m = wred[4];
      for (int u = 1; u < nw; ++u) {
#pragma unroll
        for (int k = 0; k < 4; ++k) sum[k] += wred[5 * u + k];
        m = fmin(m, wred[5 * u + 4]);
      }
      const size_t slot = (size_t)s * nt + t;
      if (A.arrive) {
#pragma unroll
        for (int k = 0; k < 4; ++k) agent_store(A.partial + slot * 4 + k, sum[k]);
        agent_store(dtpart + slot, m);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // written before the block is counted
        ends = __hip_atomic_fetch_add(A.arrive + s, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nt - 1;
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) A.partial[slot * 4 + k] = sum[k];
        dtpart[slot] = m;
      }
    }
  }
  if (!__builtin_amdgcn_readlane(ends, 63)) return;
  asm volatile("" ::: "memory");
  final_wave<true>(A, P, nt, nv, dtpart, log_slot, s);
  if ((threadIdx.x & 63) == 0)
    __hip_atomic_store(A.arrive + s, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

// One tile of one sample.  NS: 0 Euler; 1 Navier-Stokes; 2 Navier-Stokes on a
// mesh with wall cells.
template <int FLUX, int REC, int LAST, int NS>
__device__ __forceinline__ void stage_body(const DevGeo& G, const StageTab& T, const StageArgs& A,
                                           const StepParams& P, const double* Wn, double* dtpart,
                                           int r, int t, int s, int nbx, int log_slot) {
  using L = Layout<FLUX, REC>;
  extern __shared__ __attribute__((aligned(16))) double lds[];
  __shared__ double wred[8 * 5];
  __shared__ int arrive;
  const int finished = A.ctl[s].done;
  const int tid = threadIdx.x, nth = blockDim.x;
  const int4 D = T.desc[t];
  const int b0 = D.x, nown = D.y, n1 = D.z, nfl = D.w & 0x3fffffff;
  const bool simple = (D.w >> 30) == 0;
  double* SA = lds;
  double* SB = SA + L::NA * T.ms;
  double* SF = lds;                  // over SA/SB once every face flux is formed
  double* SAR = SF + NFR * T.mf;     // last stage: face areas
  double* SDL = SAR + T.mf;          // ... and distances of their ends (viscous)
  double* SVC = SB + L::NB * T.ms1;  // viscous cells, consumed before the fluxes
  double* SBF = lds + NFR * T.bf0;   // boundary entries as faces bf0 + k, kept from phase 2 on
  double* SBA = SBF + NFR * T.mb;    // ... and their areas
  double* SBT = SBA + ((T.mb + 1) & ~1);  // boundary terms
  double* SWT = SBT + NBT * T.mbt;   // wall terms
  double* SR = SWT + NWT * T.mwt;    // periodic exchange
  const size_t off = (size_t)s * G.nv;
  const Gas gas = load_gas(A, s);
  if (LAST && tid == 0) arrive = 0;  // read after the phase barriers

  // ---- requests: slot ids, this thread's faces, its gradient slot's items ----
  const int* sid = T.sid + (size_t)t * T.ms;
  const int ga = tid < T.ms ? sid[tid] : -1;
  const int gb = tid + nth < T.ms ? sid[tid + nth] : -1;
  unsigned flr[FPT];
  double2 fnn[FPT];
#pragma unroll
  for (int q = 0; q < FPT; ++q) {
    const int j = tid + q * nth;
    flr[q] = 0;
    fnn[q] = make_double2(1.0, 0.0);
    if (j < T.mf) {
      flr[q] = T.f_lr[(size_t)t * T.mf + j];
      fnn[q] = T.f_n[(size_t)t * T.mf + j];
    }
  }
  uint4 it = make_uint4(0, 0, 0, 0), it2 = make_uint4(0, 0, 0, 0);
  int2 ix = make_int2(0, 0);
  double fact = 0.0;
  if (L::GRAD && tid < n1) {
    it = T.items[(size_t)t * T.ms1 + tid];
    if (!simple) {
      it2 = T.items2[(size_t)t * T.ms1 + tid];
      ix = T.item_x[(size_t)t * T.ms1 + tid];
    }
    fact = G.gfact[ga];
  }
  // boundary terms and viscous cells go from the last thread down: its wave has
  // no gradient slots.  Boundary entries start at the first wave, wall terms at the
  // second: the waves of a tile at a wall then end this phase together
  const int back = nth - 1 - tid;
  int e0 = 0, nbe = 0;
  int2 be = make_int2(0, 0);
  if (T.mb) {
    e0 = T.vbp[b0];
    nbe = T.vbp[b0 + nown] - e0;
    if (tid < nbe) be = T.be[e0 + tid];
  }
  unsigned vcell = ~0u;
  uint4 vc = make_uint4(0, 0, 0, 0);
  if (NS) {
    if (back < T.mc) vcell = T.vcells[(size_t)t * T.mc + back];
    if (tid < nown) vc = T.vc8[b0 + tid];
  }

  // ---- phase 1: slot records, boundary terms ---------------------------------
  // the part of record B beside the gradients
  auto slot_b = [&](int gid, const Prim& w, double rho) -> double2 {
    if (L::PT) return make_double2(w.T, w.p);
    // Roe: the sound speed, negated where the vertex's Liou sensor is set
    // (liou_fix; c > 0, so the sign carries the flag)
    double c = 0.0;
    if (FLUX == F_ROE) {
      c = sound_speed(gas, w);
      if (A.ssw && A.ssw[off + gid] > 0.0) c = -c;
    }
    return make_double2(rho, c);
  };
  auto put_slot = [&](int i, int gid, const Prim& w, double V0, const double2& xy) {
    const double beta = 0.5 * frcp(gas.R * w.T);
    const double rho = (2.0 * beta) * w.p;
    double* a = SA + L::NA * i;
    sts2(a, w.u, w.v);
    sts2(a + 2, beta, L::TEC ? V0 : rho);
    sts2(a + 4, xy.x, xy.y);
    if (L::NB && i < n1) {
      const double2 q = slot_b(gid, w, rho);
      sts2(SB + L::NB * i + (L::GRAD ? 8 : 0), q.x, q.y);
    }
  };
  if (finished) return;  // here, so that the requests do not wait for the answer
  {
    Prim wa{1, 0, 0, 1}, wb{1, 0, 0, 1};
    double va = 0.0, vb = 0.0;
    double2 xa = make_double2(0, 0), xb = make_double2(0, 0);
    if (ga >= 0) {
      wa = ld_prim(A.W_in, off + ga);
      if (L::TEC) va = A.V_in[off + ga];
      xa = T.xy[ga];
    }
    if (gb >= 0) {
      wb = ld_prim(A.W_in, off + gb);
      if (L::TEC) vb = A.V_in[off + gb];
      xb = T.xy[gb];
    }
    if (ga >= 0) put_slot(tid, ga, wa, va, xa);
    if (gb >= 0) put_slot(tid + nth, gb, wb, vb, xb);
    for (int i = tid + 2 * nth; i < T.ms; i += nth) {
      const int g = sid[i];
      if (g < 0) break;
      put_slot(i, g, ld_prim(A.W_in, off + g), L::TEC ? A.V_in[off + g] : 0.0, T.xy[g]);
    }
  }
  if (L::GRAD && !simple) {
    const int k0 = T.btbeg[t], nbt = T.btbeg[t + 1] - k0;
    for (int j = back; j < 2 * nbt; j += nth) {  // two lanes a term, one for each end
      const int4 bt = T.bt[k0 + (j >> 1)];
      const int b = bt.x;
      double dq[4];
      boundary_dq(G, A, gas, s, off, b, j & 1, (j & 1) ? bt.z : bt.y, A.V_in, dq);
#pragma unroll
      for (int q = 0; q < 4; ++q) dq[q] += __shfl_xor(dq[q], 1, 64);
      if (j & 1) continue;
      double* o = SBT + NBT * (j >> 1);
      sts2(o, G.bn[2 * b], G.bn[2 * b + 1]);
      sts2(o + 2, dq[0], dq[1]);
      sts2(o + 4, dq[2], dq[3]);
    }
  }
  __syncthreads();

  // ---- phase 2: gradients, viscous cell fluxes, wall terms ---------------------
  double visc[3] = {0.0, 0.0, 0.0};  // of this thread's owned vertex
  if (L::GRAD) {
    for (int k = tid; k < n1; k += nth) {
      if (k != tid) {
        it = T.items[(size_t)t * T.ms1 + k];
        if (!simple) {
          it2 = T.items2[(size_t)t * T.ms1 + k];
          ix = T.item_x[(size_t)t * T.ms1 + k];
        }
        fact = G.gfact[sid[k]];
      }
      double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      Fan f;
      if (simple) {
        fan_centre(f, SA, k);
        walk_chain(f, it, SA, acc);
      } else {
        int more = ix.x >> 12;
        uint4 g2 = make_uint4(0, 0, 0, 0);
        if (more > 0) g2 = T.ov[ix.y];
        fan_centre(f, SA, ix.x & SI_MASK);
        if (item_at(it, 0) < SI_CENTRE) walk_chain(f, it, SA, acc);
        int at = ix.y;
        while (item_at(it2, 0) < SI_END) {
          walk_group(f, it2, SA, SBT, acc);
          if (more-- == 0) break;
          it2 = g2;
          if (more > 0) g2 = T.ov[++at];
        }
      }
      double* d = SB + L::NB * k;
#pragma unroll
      for (int q = 0; q < 8; q += 2) sts2(d + q, acc[q] * fact, acc[q + 1] * fact);
    }
  }
  for (int j = tid; j < nbe; j += nth) {  // boundary fluxes, half a bface per end
    if (j != tid) be = T.be[e0 + j];
    const int b = be.x;
    const Prim wm = ld_prim(A.W_in, off + b0 + (be.y & 0xffff));
    const double nx = G.bn[2 * b], ny = G.bn[2 * b + 1];
    const Cons F = bflux<FLUX, REC>(G, A.fo, gas, b, s, be.y >> 16, nx, ny, wm);
    double* o = SBF + NFR * j;
    sts2(o, F.m * 0.5, F.mx * 0.5);
    sts2(o + 2, F.my * 0.5, F.e * 0.5);
    if (LAST) {
      sts2(o + 4, 0.5 * nx, 0.5 * ny);
      SBA[j] = 0.5 * fsqrt(nx * nx + ny * ny);
    }
  }
  if (NS) {
    // every cell of the owned vertices once, then summed per vertex in cell order
    for (int j = back; j < T.mc; j += nth) {
      const unsigned x = j == back ? vcell : T.vcells[(size_t)t * T.mc + j];
      if (x != ~0u) viscous_cell(x, SA, gas, A.vp, SVC + NVC * j);
    }
    if (NS == 2) {
      // wall cells (src/fv.cc:1236-1312): one thread per bface forms its cell's
      // flux to the three corners and the wall flux through the bface
      const int k0 = T.wtbeg[t], nwt = T.wtbeg[t + 1] - k0;
      for (int j = tid >= 64 ? tid - 64 : tid + nth - 64; j < nwt; j += nth) {
        const uint4 wc = T.wcell[3 * (size_t)(k0 + j)];
        const int b = (int)wc.x;
        Fan f;
        fan_centre(f, SA, wc.y & 0xffffu);
        double q[2][4], x[2], y[2];
        for (int e = 0; e < 2; ++e) {
          const double* a = SA + L::NA * (e ? wc.z : (wc.y >> 16));
          const double2 uv = lds2(a), bV = lds2(a + 2), xy = lds2(a + 4);
          slot_vars(uv, bV, q[e][0], q[e][1], q[e][2], q[e][3]);
          x[e] = xy.x - f.cx; y[e] = xy.y - f.cy;
          q[e][1] -= f.c1; q[e][2] -= f.c2; q[e][3] -= f.c3;
        }
        double d[6];
        for (int z = 0; z < 3; ++z) {
          d[2 * z] = y[1] * q[0][z + 1] - y[0] * q[1][z + 1];
          d[2 * z + 1] = x[0] * q[1][z + 1] - x[1] * q[0][z + 1];
        }
        for (int z = 0; z < 2; ++z) {
          const unsigned jt = z ? wc.w >> 16 : wc.w & 0xffffu;
          if (jt == 0xffffu) continue;
          double bx, by, dq[4];
          if (L::GRAD) {
            const double* q4 = SBT + NBT * jt;
            bx = q4[0]; by = q4[1];
            dq[1] = q4[3]; dq[2] = q4[4]; dq[3] = q4[5];
          } else {  // no gradient pass: jt is the bface's place in its cell's list
            const int bf = G.cbf[2 * (size_t)G.blc[b] + jt];
            bx = G.bn[2 * bf]; by = G.bn[2 * bf + 1];
            double de[4];
            boundary_dq(G, A, gas, s, off, bf, 0, G.bv[2 * bf], nullptr, dq);
            boundary_dq(G, A, gas, s, off, bf, 1, G.bv[2 * bf + 1], nullptr, de);
            for (int w = 0; w < 4; ++w) dq[w] += de[w];
          }
          for (int w = 0; w < 3; ++w) { d[2 * w] += bx * dq[w + 1]; d[2 * w + 1] += by * dq[w + 1]; }
        }
        const double ia = fdiv(1.0, x[0] * y[1] - y[0] * x[1]);
        for (int z = 0; z < 6; ++z) d[z] *= ia;
        const Ent sw = wall_state(G, A.W_in, off, s, gas, T.wcell + 3 * (size_t)(k0 + j) + 1);
        const ViscTensor v = visc_tensor(gas, A.vp, sw.vx, sw.vy, sw.l, d);
        double* o = SWT + NWT * j;
        const double nx[3] = {y[0] - y[1], y[1], -y[0]}, ny[3] = {x[1] - x[0], -x[1], x[0]};
        for (int z = 0; z < 3; ++z) {
          const double hx = 0.5 * nx[z], hy = 0.5 * ny[z];
          o[3 * z] = v.xx * hx + v.xy * hy;
          o[3 * z + 1] = v.xy * hx + v.yy * hy;
          o[3 * z + 2] = v.ex * hx + v.ey * hy;
        }
        const double hx = -0.5 * G.bn[2 * b], hy = -0.5 * G.bn[2 * b + 1];
        const bool ad = bc_adiabatic(G.btype[b]);
        o[9] = v.xx * hx + v.xy * hy;
        o[10] = v.xy * hx + v.yy * hy;
        o[11] = (v.ex - (ad ? v.qx : 0.0)) * hx + (v.ey - (ad ? v.qy : 0.0)) * hy;
      }
    }
  }
  if (L::GRAD || NS) __syncthreads();
  if (NS && tid < nown) {
    const unsigned w[4] = {vc.x, vc.y, vc.z, vc.w};
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const unsigned e = (w[u >> 1] >> (16 * (u & 1))) & 0xffffu;
      if (e != GE_END) viscous_add(e, SVC, visc);
    }
    if ((w[3] >> 16) != GE_END) {  // more than eight, maybe
      const int k0 = G.vc_ptr[b0 + tid], n = T.vccnt[b0 + tid];
      for (int k = 8; k < n; ++k) viscous_add(T.vcent[k0 + k], SVC, visc);
    }
  }

  // ---- phase 3: local face fluxes (registers, then LDS) ------------------------
  double fl[FPT][4], fdl[FPT];
#pragma unroll
  for (int q = 0; q < FPT; ++q) {
    const int j = tid + q * nth;
    if (j >= nfl) continue;
    const int l = flr[q] & 0xffff, rr = flr[q] >> 16;
    double ia;
    const double area = face_area(fnn[q].x, fnn[q].y, &ia);
    const double *al = SA + L::NA * l, *ar = SA + L::NA * rr;
    const double *bl = SB + L::NB * l, *br = SB + L::NB * rr;
    Side Ls, Rs;
    const double2 uvl = lds2(al), uvr = lds2(ar), bVl = lds2(al + 2), bVr = lds2(ar + 2);
    Ls.w = Prim{1, uvl.x, uvl.y, 1};
    Rs.w = Prim{1, uvr.x, uvr.y, 1};
    Ls.beta = bVl.x; Rs.beta = bVr.x;
    double ssw = 0.0;
    if (L::TEC) {
      const double2 rcl = lds2(bl + (L::GRAD ? 8 : 0)), rcr = lds2(br + (L::GRAD ? 8 : 0));
      slot_vars(uvl, bVl, Ls.V[0], Ls.V[1], Ls.V[2], Ls.V[3]);
      slot_vars(uvr, bVr, Rs.V[0], Rs.V[1], Rs.V[2], Rs.V[3]);
      Ls.rho = rcl.x; Rs.rho = rcr.x;
      Ls.c = fabs(rcl.y); Rs.c = fabs(rcr.y);
      ssw = (rcl.y < 0.0 || rcr.y < 0.0) ? 1.0 : 0.0;
    } else if (L::PT) {
      const double2 tl = lds2(bl), tr = lds2(br);
      Ls.w.T = tl.x; Ls.w.p = tl.y;
      Rs.w.T = tr.x; Rs.w.p = tr.y;
    } else {
      Ls.rho = bVl.y; Rs.rho = bVr.y;
    }
    double gdl[4] = {0, 0, 0, 0}, gdr[4] = {0, 0, 0, 0}, rx = 0.0, ry = 0.0;
    if (L::GRAD) {
#pragma clang fp contract(fast)
      const double2 xl = lds2(al + 4), xr = lds2(ar + 4);
      rx = xr.x - xl.x;
      ry = xr.y - xl.y;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const double2 dl = lds2(bl + 2 * k), dr = lds2(br + 2 * k);
        gdl[k] = dl.x * rx + dl.y * ry;
        gdr[k] = dr.x * rx + dr.y * ry;
      }
    }
    if (NS && LAST) {
      const double2 xl = lds2(al + 4), xr = lds2(ar + 4);
      const double dx = xr.x * 1.0 + xl.x * -1.0, dy = xr.y * 1.0 + xl.y * -1.0;
      fdl[q] = fsqrt(dx * dx + dy * dy);
    }
    const Cons F = pair_flux<FLUX, REC>(gas, A.fo, rx, ry, Ls, Rs, gdl, gdr, fnn[q].x * ia, fnn[q].y * ia, ssw);
    fl[q][0] = F.m * area; fl[q][1] = F.mx * area; fl[q][2] = F.my * area; fl[q][3] = F.e * area;
  }
  // the update's operands, requested here so that their latency overlaps the
  // barriers and the flux records' way through LDS
  const bool own = tid < nown;
  const int v = b0 + tid;
  Prim w0{1, 0, 0, 1};
  double4 wn4 = make_double4(1.0, 0.0, 0.0, 1.0);
  double area_v = 1.0;
  uint4 ge = make_uint4(0, 0, 0, 0);
  if (own) {
    ge = T.ge8[v];
    w0 = ld_prim(A.W_in, off + v);
    if (r != 0 || A.scheme == 1) wn4 = reinterpret_cast<const double4*>(Wn)[off + v];
    area_v = G.dcarea[v];
  }
  __syncthreads();  // every slot record read: their space takes the face records
#pragma unroll
  for (int q = 0; q < FPT; ++q) {
    const int j = tid + q * nth;
    if (j >= nfl) continue;
    double* o = SF + NFR * j;
    sts2(o, fl[q][0], fl[q][1]);
    sts2(o + 2, fl[q][2], fl[q][3]);
    if (LAST) {
      double ia;
      sts2(o + 4, fnn[q].x, fnn[q].y);
      SAR[j] = face_area(fnn[q].x, fnn[q].y, &ia);
      if (NS) SDL[j] = fdl[q];
    }
  }
  __syncthreads();

  // ---- phase 4: gather, periodic sums, update ----------------------------------
  // A vertex's entries are its faces, then its boundary entries, which have face
  // records of their own; the first eight arrive packed, longer lists follow from
  // memory, so every sum keeps the reference order (+F at a face's left end, -F at
  // its right).
  double acc[4] = {0, 0, 0, 0};
  if (LAST && own && A.W_keep)  // the last stage's input state, kept for the caller
    reinterpret_cast<double4*>(A.W_keep)[off + v] = make_double4(w0.T, w0.u, w0.v, w0.p);
  const unsigned gw[4] = {ge.x, ge.y, ge.z, ge.w};
  int rest = -1;  // position in the vertex's list where the packed entries stop
  auto add_face = [&](unsigned e) {
    const double* f = SF + NFR * (e & 0x3fffu);
    const double2 a = lds2(f), b = lds2(f + 2);
    const double sg = (e & 0x8000u) ? -1.0 : 1.0;
    acc[0] = __builtin_fma(sg, a.x, acc[0]);
    acc[1] = __builtin_fma(sg, a.y, acc[1]);
    acc[2] = __builtin_fma(sg, b.x, acc[2]);
    acc[3] = __builtin_fma(sg, b.y, acc[3]);
  };
  int gk0 = 0, gne = 0, gnf = 0, gnb = 0;  // longer lists: start, length, faces, first boundary entry
  auto entry = [&](int k) -> unsigned {
    return k < gnf ? (unsigned)T.gent[gk0 + k] : (unsigned)(T.bf0 + gnb + k - gnf);
  };
  if (own) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const unsigned e = (gw[u >> 1] >> (16 * (u & 1))) & 0xffffu;
      if (!(e & 0x4000u)) add_face(e);
      else if (e == GE_MORE) rest = u;
    }
    if (rest >= 0) {
      gk0 = T.gptr[v];
      gne = T.gptr[v + 1] - gk0;
      if (T.mb) {
        gnb = T.vbp[v] - e0;
        gnf = gne - (T.vbp[v + 1] - e0 - gnb);
      } else {
        gnf = gne;
      }
      for (int k = rest; k < gne; ++k) add_face(entry(k));
    }
    if (NS) {  // viscous fluxes after the faces (src/fv.cc:1197-1232), then the wall terms
      acc[1] += visc[0]; acc[2] += visc[1]; acc[3] += visc[2];
      if (NS == 2)
        for (int q = G.vbe_ptr[v]; q < G.vbe_ptr[v + 1]; ++q) {
          const unsigned e = T.wvent[q];
          const double* o = SWT + NWT * (e & SI_MASK);
          const double* c = o + 3 * ((e >> 13) & 3u);
          acc[1] += c[0]; acc[2] += c[1]; acc[3] += c[2];
          if (e & 0x8000u) { acc[1] += o[9]; acc[2] += o[10]; acc[3] += o[11]; }
        }
    }
  }
  const bool per = T.tper[t] != 0;
  const int TB = SR_VERTS;
  if (per) {
    if (own)
#pragma unroll
      for (int k = 0; k < 4; ++k) SR[k * TB + tid] = acc[k];
    __syncthreads();
    if (own) {
      const int pi = T.pinfo[v];
      if (pi >= 0) {
        const int first = pi >> 8, cnt = pi & 255;
        double tot[4] = {0, 0, 0, 0};
        for (int m = 0; m < cnt; ++m)
#pragma unroll
          for (int k = 0; k < 4; ++k) tot[k] += SR[k * TB + first + m];
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[k] = tot[k];
      }
    }
  }
  double part[4] = {0, 0, 0, 0};
  double lam = 0.0;
  if (own) {
    if (LAST) {
      const double wt = G.weight[v];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const double q = fdiv(acc[k], area_v);
        part[k] = (q * q) * wt;
      }
    }
    const double factor = fdiv(A.dtl ? A.dtl[off + v] : A.ctl[s].dt, area_v);
    Cons U;
    const Prim wn{wn4.x, wn4.y, wn4.z, wn4.w};
    if (A.scheme == 1) {  // RK4 (src/fv.cc:1661-1673): U_old plus a multiple of R, or of
                          // the stages' weighted sum R2 in the last stage
      const double rks[4] = {1.0, 1.0 / 2.0, 1.0 / 2.0, 1.0};
      double* R2 = A.R2 + 4 * (off + v);
      const double ir = 1.0 / rks[r];
      double q[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const double r2 = (r == 0 ? 0.0 : R2[k]) + acc[k] * ir;
        R2[k] = r2;
        q[k] = (r < 3) ? acc[k] : r2;
      }
      const double c = (r < 3) ? -factor * rks[r < 3 ? r + 1 : 3] : -factor / 6.0;
      const Cons Uo = prim2con(gas, wn);
      U.m = Uo.m * 1.0 + q[0] * c; U.mx = Uo.mx * 1.0 + q[1] * c;
      U.my = Uo.my * 1.0 + q[2] * c; U.e = Uo.e * 1.0 + q[3] * c;
    } else {  // SSP-RK3, or Heun's two-stage SSP form (src/fv.cc:1640-1651, :1675-1686)
      const double a_rk[3] = {0.0, 3.0 / 4.0, 1.0 / 3.0};
      const double b_rk[3] = {1.0, 1.0 / 4.0, 2.0 / 3.0};
      const bool heun = A.scheme == 2;
      const double b = heun ? (1.0 - r * 0.5) : b_rk[r], a = heun ? r * 0.5 : a_rk[r];
      const double c = -factor * b;
      U = prim2con(gas, w0);
      U.m *= b; U.mx *= b; U.my *= b; U.e *= b;
      if (r == 0) {  // a = 0: U_old * 0 contributes an exact zero
        U.m += 0.0 + acc[0] * c; U.mx += 0.0 + acc[1] * c;
        U.my += 0.0 + acc[2] * c; U.e += 0.0 + acc[3] * c;
      } else {
        const Cons Uo = prim2con(gas, wn);
        U.m += Uo.m * a + acc[0] * c; U.mx += Uo.mx * a + acc[1] * c;
        U.my += Uo.my * a + acc[2] * c; U.e += Uo.e * a + acc[3] * c;
      }
    }
    const Prim w1 = con2prim(gas, U);
    reinterpret_cast<double4*>(A.W_out)[off + v] = make_double4(w1.T, w1.u, w1.v, w1.p);
    if (L::TEC) A.V_out[off + v] = entropy_var0(gas, w1);
    if (LAST) {  // spectral radius for the next step's dt, src/fv.cc:1511-1553
      const double cm = sound_speed(gas, w1);
      auto add_lam = [&](unsigned e) {
        const int j = e & 0x3fffu;
        const double2 n = lds2(SF + NFR * j + 4);
        const double vn = w1.u * n.x + w1.v * n.y;
        lam += fabs(vn) + cm * (j < T.bf0 ? SAR[j] : SBA[j - T.bf0]);
      };
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const unsigned e = (gw[u >> 1] >> (16 * (u & 1))) & 0xffffu;
        if (!(e & 0x4000u)) add_lam(e);
      }
      if (rest >= 0)
        for (int k = rest; k < gne; ++k) add_lam(entry(k));
      if (NS) {  // viscous share, after every inviscid term (src/fv.cc:1555-1580)
        double mu;
        const double Tm = w1.T;
        if (A.vp.mu_model == 0) mu = A.vp.mu_ref;
        else if (A.vp.mu_model == 1) mu = A.vp.mu_ref * pow(Tm, 1.5) / (Tm + A.vp.T_0);
        else mu = A.vp.mu_ref * pow(Tm / A.vp.T_ref, A.vp.omega);
        const double rho = density(gas, w1);
        auto add_visc = [&](unsigned e) {
          const int j = e & 0x3fffu;
          if (j >= T.bf0) return;
          lam += fdiv(fdiv(mu * SAR[j], SDL[j]), rho);
        };
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const unsigned e = (gw[u >> 1] >> (16 * (u & 1))) & 0xffffu;
          if (!(e & 0x4000u)) add_visc(e);
        }
        if (rest >= 0)
          for (int k = rest; k < gnf; ++k) add_visc(entry(k));
      }
    }
  }
  if (LAST) {
    if (per) {
      __syncthreads();  // SR reads of the residual exchange are complete
      if (own) SR[tid] = lam;
      __syncthreads();
      if (own) {
        const int pi = T.pinfo[v];
        if (pi >= 0) {
          const int first = pi >> 8, cnt = pi & 255;
          double tot = 0.0;
          for (int m = 0; m < cnt; ++m) tot = tot + SR[first + m];
          lam = tot;
        }
      }
    }
    double dtv = 1.0e20;
    if (own) {
      dtv = (P.time_step > 0.0) ? P.time_step : fdiv(P.cfl * area_v, lam);
      if (A.dtl) A.dtl[off + v] = dtv;  // steady mode: read by this vertex only, next step
    }
    block_partials(A, P, part, dtv, wred, &arrive, dtpart, s, t, nbx, G.nv, (nown + 63) >> 6, log_slot);
  }
}

// Four waves per SIMD (128 VGPRs): the LDS of a 128-vertex tile (36 KB) allows
// four tiles of four waves per CU.  Viscous terms with gradients need 50 KB at 112
// vertices, three tiles.
template <int FLUX, int REC, int LAST, int NS>
__global__ __launch_bounds__(512, (NS && Layout<FLUX, REC>::GRAD ? 3 : 4)) void k_stage(
    DevGeo G, StageTab T, StageArgs A, StepParams P, const double* Wn, double* dtpart, int r,
    int log_slot) {
  stage_body<FLUX, REC, LAST, NS>(G, T, A, P, Wn, dtpart, r, xcd_tile(blockIdx.x, gridDim.x),
                                  blockIdx.y, gridDim.x, log_slot);
}
// The same over the tiles and samples of several contexts (the levels of a
// multilevel run): block b belongs to the level whose range [base_fu, ...)
// holds it, tile (b - base) mod ntiles, sample (b - base) / ntiles.
template <int FLUX, int REC, int LAST>
__global__ __launch_bounds__(512, 4) void k_stage_packed(const PackLevel* __restrict__ pk,
                                                                    int nl, int r) {
  const int b = blockIdx.x;
  int l = 0;
  while (l + 1 < nl && b >= pk[l + 1].base_fu) ++l;
  const PackLevel& L = pk[l];
  const int nt = L.T.ntiles, local = b - L.base_fu;
  stage_body<FLUX, REC, LAST, 0>(L.G, L.T, L.A, L.P, L.Wn, L.dtpart, r, local % nt, local / nt, nt, -1);
}

// ---------------------------------------------------------------------------
// end of a step of contexts with more tiles than the stage kernel folds
// ---------------------------------------------------------------------------
namespace {
// The last stage ends the steps of a context with up to this many tiles over all its
// samples, which run at once: eight partials a lane of the wave that does it.  A step
// of the vortex (Roe, minmod) against a launch of its own: 129^2 (150 tiles) 37.7 us
// against 41.8, 200^2 43.0 / 45.7, 257^2 (541) 53.9 / 54.3, 350^2 63.2 / 62.7.  Where
// tiles queue for a CU each is held up by the wait for its partials: 32 samples of
// 257^2 took 1.15 times as long.
constexpr int FOLD_TILES = 512;

template <int NV>
__device__ __forceinline__ void bsum(double* v, double* red) {
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 63)
#pragma unroll
    for (int k = 0; k < NV; ++k) red[wid * NV + k] = v[k];
  __syncthreads();
  if (threadIdx.x == 0) {
    const int nw = blockDim.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double s = red[k];
      for (int w = 1; w < nw; ++w) s += red[w * NV + k];
      v[k] = s;
    }
  }
}
__device__ __forceinline__ double bmin(double x, double* red) {
  x = wave_min(x);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 63) red[wid] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int nw = blockDim.x >> 6;
    x = red[0];
    for (int w = 1; w < nw; ++w) x = fmin(x, red[w]);
  }
  return x;
}
__device__ __forceinline__ void step_final_body(const StageArgs& A, const StepParams& P, int nblk,
                                                int nv, const double* dtpart, int log_slot,
                                                int s) {
  __shared__ double red[64];
  const Ctl c = A.ctl[s];
  if (c.done) return;
  double part[4] = {0, 0, 0, 0};
  double x = 1.0e20;
  const double4* q4 = reinterpret_cast<const double4*>(A.partial) + (size_t)s * nblk;
  const double* dq = dtpart + (size_t)s * nblk;
  int i = threadIdx.x;
  for (; i + 3 * (int)blockDim.x < nblk; i += 4 * blockDim.x) {  // four independent loads in flight
    double4 a[4];
    double d[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) { a[u] = q4[i + u * blockDim.x]; d[u] = dq[i + u * blockDim.x]; }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      part[0] += a[u].x; part[1] += a[u].y; part[2] += a[u].z; part[3] += a[u].w;
      x = fmin(x, d[u]);
    }
  }
  for (; i < nblk; i += blockDim.x) {
    const double4 a = q4[i];
    part[0] += a.x; part[1] += a.y; part[2] += a.z; part[3] += a.w;
    x = fmin(x, dq[i]);
  }
  bsum<4>(part, red);
  __syncthreads();
  x = bmin(x, red);
  if (threadIdx.x == 0) step_ctl(A, P, c, nv, part, x, log_slot, s);
}
}  // namespace
__global__ __launch_bounds__(1024) void k_step_final_tiled(StageArgs A, StepParams P, int nblk,
                                                          int nv, const double* dtpart,
                                                          int log_slot) {
  step_final_body(A, P, nblk, nv, dtpart, log_slot, blockIdx.x);
}
// ... with up to FOLD_TILES tiles
__global__ __launch_bounds__(64) void k_step_final_wave(StageArgs A, StepParams P, int nblk, int nv,
                                                        const double* dtpart, int log_slot) {
  final_wave<false>(A, P, nblk, nv, dtpart, log_slot, blockIdx.x);
}
__global__ __launch_bounds__(1024) void k_step_final_packed(const PackLevel* __restrict__ pk, int nl) {
  const int b = blockIdx.x;
  int l = 0;
  while (l + 1 < nl && b >= pk[l + 1].base_final) ++l;
  const PackLevel& L = pk[l];
  if (L.T.ntiles > FOLD_TILES) step_final_body(L.A, L.P, L.T.ntiles, L.G.nv, L.dtpart, -1, b - L.base_final);
  else if (threadIdx.x < 64) final_wave<false>(L.A, L.P, L.T.ntiles, L.G.nv, L.dtpart, -1, b - L.base_final);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
int stage_block(const StageTab& T) {
  int b = std::max(T.tb, (T.mf + FPT - 1) / FPT);
  b = ((b + 63) / 64) * 64;
  return std::max(b, T.fu_block);
}
int stage_block_max() { return 512; }
bool stage_ends_step(int ntiles, int samples) { return (long)ntiles * samples <= FOLD_TILES; }

namespace {
size_t lds_of(const StageTab& T) {
  return sizeof(double) * ((size_t)NFR * (T.bf0 + T.mb) + ((T.mb + 1) & ~1) + (size_t)NBT * T.mbt +
                           (size_t)NWT * T.mwt + (T.n_periodic_tiles > 0 ? 4 * SR_VERTS : 0) + 2);
}
template <int FLUX, int REC>
void go(const DevGeo& G, const StageTab& T, const StageArgs& A, const StepParams& P, const double* Wn,
        double* dtpart, int S, int r, bool last, int log_slot, hipStream_t st) {
  const size_t lds = lds_of(T);
  const dim3 grid(T.ntiles, S), blk(stage_block(T));
  auto run = [&](auto kern) {
    if (lds > 48 * 1024)
      (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kern, grid, blk, lds, st, G, T, A, P, Wn, dtpart, r, log_slot);
  };
  if (A.ns && A.ns_walls) {
    if (last) run(k_stage<FLUX, REC, 1, 2>); else run(k_stage<FLUX, REC, 0, 2>);
  } else if (A.ns) {
    if (last) run(k_stage<FLUX, REC, 1, 1>); else run(k_stage<FLUX, REC, 0, 1>);
  } else {
    if (last) run(k_stage<FLUX, REC, 1, 0>); else run(k_stage<FLUX, REC, 0, 0>);
  }
}
template <int FLUX, int REC>
void go_packed(const PackLevel* d, const PackPlan& p, int r, bool last, hipStream_t st) {
  auto run = [&](auto kern) {
    if (p.fu_lds > 48 * 1024)
      (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.fu_lds);
    hipLaunchKernelGGL(kern, dim3(p.fu_blocks), dim3(p.fu_block), p.fu_lds, st, d, p.nl, r);
  };
  if (last) run(k_stage_packed<FLUX, REC, 1>); else run(k_stage_packed<FLUX, REC, 0>);
}
// f(flux, reconstruction) as compile-time constants
template <int FLUX, class F>
void with_rec(int rec, F&& f) {
  switch (rec) {
    case R_FIRST: f.template operator()<FLUX, R_FIRST>(); break;
    case R_SECOND: f.template operator()<FLUX, R_SECOND>(); break;
    case R_MUSCL: f.template operator()<FLUX, R_MUSCL>(); break;
    case R_ALBADA: f.template operator()<FLUX, R_ALBADA>(); break;
    case R_MINMOD: f.template operator()<FLUX, R_MINMOD>(); break;
    case R_TVB: f.template operator()<FLUX, R_TVB>(); break;
    default: f.template operator()<FLUX, R_ENO2>(); break;
  }
}
template <class F>
void with_scheme(int flux, int rec, F&& f) {
  switch (flux) {
    case F_ROE: with_rec<F_ROE>(rec, f); break;
    case F_RUS: with_rec<F_RUS>(rec, f); break;
    case F_KEPEC: f.template operator()<F_KEPEC, R_FIRST>(); break;
    case F_ROEEC: f.template operator()<F_ROEEC, R_FIRST>(); break;
    case F_KEP: f.template operator()<F_KEP, R_FIRST>(); break;
    default: f.template operator()<F_AVG, R_FIRST>(); break;
  }
}
struct Launch {
  const DevGeo& G; const StageTab& T; const StageArgs& A; const StepParams& P;
  const double* Wn; double* dtpart; int S, r; bool last; int log_slot; hipStream_t st;
  template <int FLUX, int REC> void operator()() { go<FLUX, REC>(G, T, A, P, Wn, dtpart, S, r, last, log_slot, st); }
};
struct LaunchPacked {
  const PackLevel* d; const PackPlan& p; int r; bool last; hipStream_t st;
  template <int FLUX, int REC> void operator()() { go_packed<FLUX, REC>(d, p, r, last, st); }
};
}  // namespace

size_t stage_lds(const StageTab& T) { return lds_of(T); }
// records of the main part: the widest layout of the slots, or the faces
int stage_main_records(const StageTab& T, bool grad, bool ns) {
  using L = Layout<F_ROE, R_MINMOD>;
  using L1 = Layout<F_ROE, R_FIRST>;
  const int slots = L::NA * T.ms + (grad ? L::NB : L1::NB) * T.ms1 + (ns ? NVC * T.mc : 0);
  return (std::max(slots, (NFR + (ns ? 2 : 1)) * T.mf) + NFR - 1) / NFR;
}
bool stage_has_gradients(int flux, int rec) { return (flux == F_ROE || flux == F_RUS) && rec != R_FIRST; }
bool stage_keeps_var0(int flux) { return flux == F_ROE || flux == F_RUS; }

void launch_stage(int flux, int rec, const DevGeo& G, const StageTab& T, const StageArgs& A,
                  const StepParams& P, const double* Wn, double* dtpart, int S, int r, bool last,
                  int log_slot, hipStream_t st) {
  Launch f{G, T, A, P, Wn, dtpart, S, r, last, log_slot, st};
  with_scheme(flux, rec, f);
}

void launch_step_final_tiled(const DevGeo& G, const StageArgs& A, const StepParams& P, int S,
                             int nblk, const double* dtpart, int log_slot, hipStream_t st) {
  if (A.arrive) return;  // ended by the last stage
  if (nblk <= FOLD_TILES)
    hipLaunchKernelGGL(k_step_final_wave, dim3(S), dim3(64), 0, st, A, P, nblk, G.nv, dtpart, log_slot);
  else
    hipLaunchKernelGGL(k_step_final_tiled, dim3(S), dim3(1024), 0, st, A, P, nblk, G.nv, dtpart, log_slot);
}

// ---------------------------------------------------------------------------
// packed launches: every kernel of a step runs once over the tiles and
// samples of all levels (contexts with the same scheme), each block doing
// exactly what it does in its own context's launch
// ---------------------------------------------------------------------------
void pack_plan(PackLevel* lv, int nl, int flux, int rec, PackPlan& p) {
  p = PackPlan{};
  p.nl = nl;
  for (int l = 0; l < nl; ++l) {
    PackLevel& L = lv[l];
    L.base_fu = p.fu_blocks;         p.fu_blocks += L.T.ntiles * L.S;
    L.base_final = p.final_blocks;   p.final_blocks += L.A.arrive ? 0 : L.S;
    p.fu_block = std::max(p.fu_block, stage_block(L.T));
    p.fu_lds = std::max(p.fu_lds, stage_lds(L.T));
  }
}

void launch_packed_stage(int flux, int rec, const PackLevel* d, const PackPlan& p, int r,
                         bool last, hipStream_t st) {
  LaunchPacked f{d, p, r, last, st};
  with_scheme(flux, rec, f);
}

void launch_packed_final(const PackLevel* d, const PackPlan& p, hipStream_t st) {
  if (p.final_blocks == 0) return;
  hipLaunchKernelGGL(k_step_final_packed, dim3(p.final_blocks), dim3(1024), 0, st, d, p.nl);
}

}  // namespace tsm
