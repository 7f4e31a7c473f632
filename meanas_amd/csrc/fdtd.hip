// Time-domain Yee updates (FDTD) on real fields.
//
// maxwell_h: h -= dt curl_forward(e) / mu   (meanas/fdtd/base.py:67-125)
// maxwell_e: e += dt curl_back(h) / epsilon (meanas/fdtd/base.py:13-64)
// with curl_forward / curl_back as in meanas/fdmath/functional.py: periodic forward
// differences (f[n+1] - f[n]) / dx_e[n] and backward differences (f[n] - f[n-1]) / dx_h[n],
// unit widths when the grid gives none.  Materials divide, as the reference does.
//
// The updates, the CPML and the divergence march along x, a thread per (y, z) column, or have a
// thread per cell, as energy and flux do (see Column); runs of several steps pipeline two steps
// per pass (k_fdtd_steps).
#include <algorithm>
#include <cstdlib>
#include <string>
#include <type_traits>

#include "common.hpp"
#include "../../include/meanas_fdfd.h"

namespace mx {

int set_error(const std::string& msg);

namespace {

constexpr int kFB = 256;

struct RGrid {
  int nx, ny, nz;
  const double* dxe[3];
  const double* dxh[3];
};

__device__ __forceinline__ double width(const double* w, int n) { return w ? w[n] : 1.0; }
// width n of a table with n uniform over the block: a scalar load (constant address
// space) into SGPRs
__device__ __forceinline__ double width_u(const double* w, int n) {
  return w ? ((const MX_CONST double*)w)[n] : 1.0;
}

// A thread's part of a column kernel: cell t = j nz + k of the (y, z) plane and the planes
// [ib, ie).  The work items (kFB threads each) are dealt so that each XCD -- workgroups go
// round the 8 of them -- has a contiguous run, whose neighbouring rows and planes meet in
// its L2.  Two forms, by the type of the byte offsets (column_grid chooses):
//   32 bits: a column each, marching along x through one slab.  Consecutive threads take
//     consecutive cells of the flattened plane (no lanes lost on short or odd rows), and a
//     block stays in one slab, so the plane and what belongs to it are uniform;
//   64 bits: a cell each, consecutive threads consecutive cells of the grid (`slab`: nonzero,
//     or 0 to take the items in the order of the blocks).
template <typename OFF> constexpr bool kMarches = sizeof(OFF) == 4;
struct Column {
  int j, k, t, ib, ie;
  bool ok;
};
template <typename OFF> __device__ __forceinline__ Column column(const RGrid& g, int slab) {
  const int plane = g.ny * g.nz, run = kMarches<OFF> ? plane : g.nx * plane;
  const int pieces = (run + kFB - 1) / kFB;
  const int nwork = kMarches<OFF> ? pieces * ((g.nx + slab - 1) / slab) : pieces, per = (nwork + 7) / 8;
  const bool plain = !kMarches<OFF> && slab == 0;
  const int w = plain ? (int)blockIdx.x : (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  const int s = kMarches<OFF> ? w / pieces : 0, piece = w - s * pieces;
  Column c;
  c.t = piece * kFB + (int)threadIdx.x;
  c.ok = (plain || (int)(blockIdx.x / 8) < per) && w < nwork && c.t < run;
  if constexpr (kMarches<OFF>) {
    c.ib = s * slab;
    c.ie = min(c.ib + slab, g.nx);
  } else {
    c.ib = c.t / plane;
    c.ie = c.ib + 1;
    c.t -= c.ib * plane;
  }
  c.j = c.t / g.nz;
  c.k = c.t - c.j * g.nz;
  return c;
}
// width n of the x axis, n a plane of the thread's column
template <typename OFF> __device__ __forceinline__ double width_x(const double* w, int n) {
  if constexpr (kMarches<OFF>) return width_u(w, n);
  else return width(w, n);
}
// element of `f` at a uniform element offset plus a thread's byte offset: with a 32-bit OFF
// one load from an SGPR base and a VGPR offset
template <typename T, typename OFF>
__device__ __forceinline__ T at(const T* f, size_t base, OFF off) {
  return *(const MX_GLOBAL T*)((const MX_GLOBAL char*)(f + base) + off);
}
// A thread offset that does not change in a loop, as if it did: otherwise its extension to
// 64 bits is hoisted, and the loads take per-thread 64-bit addresses (two registers and an
// addition each) instead of an SGPR base and the offset.
template <typename OFF> __device__ __forceinline__ OFF in_loop(OFF off) {
  asm volatile("" : "+v"(off));
  return off;
}
template <typename T, typename OFF>
__device__ __forceinline__ void put(T* f, size_t base, OFF off, T v) {
  *(MX_GLOBAL T*)((MX_GLOBAL char*)(f + base) + off) = v;
}

// x / d given rd = 1 / d: one product, its exact residual and one correction, then the
// divide fix-up instruction for zeros, infinities and NaN; it also makes an infinity of a
// quotient that overflows, where the correction is inf - inf.  4 instructions at full rate;
// the compiler's divide takes 9 (float32) or 13 (float64) of that issue time.
// Where the residual is exact (dividends above 2^-102 in float32, 2^-969 in float64) the
// value rounded at the end is within 2^-20 ulp of the quotient (2^-50 in float64), so the
// result is the correctly rounded quotient in all but about one of 10^6 (10^15) near-ties;
// smaller dividends give a quotient within an ulp (float32, 1e-37: 2.3 % of them an ulp off).
// Divisors that recip() takes: magnitudes from 2^-126 to 2^126 in float32, from 2^-1022 in
// float64, zero and infinity.  A larger float32 one counts as infinite (the hardware flushes
// its reciprocal), a subnormal one as zero.  Looking for them in each cell, to divide by the
// compiler's code there, cost 3 to 7 % (registers: up to 1.6 times in float64 runs with mu).
__device__ __forceinline__ double div_by(double x, double d, double rd) {
  const double q = x * rd;
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-q, d, x), rd, q), d, x);
}
__device__ __forceinline__ float div_by(float x, float d, float rd) {
  const float q = x * rd;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-q, d, x), rd, q), d, x);
}

// 1 / d to within an ulp, for div_by: the hardware's reciprocal and Newton steps
__device__ __forceinline__ double recip(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
}
__device__ __forceinline__ float recip(float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
}

// value of the next / previous lane of the wave (DPP wave shifts; the end lanes get 0)
template <int CTRL> __device__ __forceinline__ float lane_shift(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int CTRL> __device__ __forceinline__ double lane_shift(double v) {
  typedef int __attribute__((ext_vector_type(2))) I2;
  const I2 w = __builtin_bit_cast(I2, v);
  I2 r;
  r.x = __builtin_amdgcn_update_dpp(0, w.x, CTRL, 0xf, 0xf, true);
  r.y = __builtin_amdgcn_update_dpp(0, w.y, CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, r);
}
// a value that is the same in every lane, as a scalar (SGPRs)
__device__ __forceinline__ float wave_value(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double wave_value(double v) {
  typedef int __attribute__((ext_vector_type(2))) I2;
  I2 w = __builtin_bit_cast(I2, v);
  w.x = __builtin_amdgcn_readfirstlane(w.x);
  w.y = __builtin_amdgcn_readfirstlane(w.y);
  return __builtin_bit_cast(double, w);
}
template <typename T> __device__ __forceinline__ T lane_next(T v) { return lane_shift<0x130>(v); }
template <typename T> __device__ __forceinline__ T lane_prev(T v) { return lane_shift<0x138>(v); }

// One leapfrog half step, HBM-bound: 36 (H) and 48 (E) bytes a cell in float32.  Marching
// with the x neighbour in registers, no index division per cell and each XCD on its own
// run of the grid reads each value about once (a thread per cell read 1.3 times as much).
// E / H update: 256^3 float32 152 / 119 us (177 / 167 before), 5.3 / 5.1 TB/s, a large copy's
// rate; float64 303 / 240 us (313 / 249); 150 x 141 x 130, in cache, float32 21 / 17 us (28 / 24),
// float64 39 / 31 us (47 / 37).  Where columns lose: column_grid, launch_update.
// H' = H - dt curl_f(E) / mu (EUPD false) or E' = E + dt curl_b(H) / eps (EUPD true), in
// place: f is the field differenced, out the one updated.
template <typename T, bool EUPD, typename OFF>
__global__ __launch_bounds__(kFB) void k_fdtd_update(RGrid g, T dt, const T* __restrict__ f, T* __restrict__ out,
                                                     const T* __restrict__ mat, T mat_s, int slab) {
  const Column c = column<OFF>(g, slab);
  if (!c.ok) return;
  const int nx = g.nx, ny = g.ny, nz = g.nz, plane = ny * nz;
  const size_t nc = (size_t)nx * plane;
  // neighbours of the difference: the cell before (E update) or after (H update)
  const int jn = EUPD ? (c.j == 0 ? ny - 1 : c.j - 1) : (c.j + 1 == ny ? 0 : c.j + 1);
  const int kn = EUPD ? (c.k == 0 ? nz - 1 : c.k - 1) : (c.k + 1 == nz ? 0 : c.k + 1);
  const OFF own0 = (OFF)c.t * (OFF)sizeof(T);
  const OFF oy0 = ((OFF)jn * (OFF)nz + (OFF)c.k) * (OFF)sizeof(T), oz0 = ((OFF)c.j * (OFF)nz + (OFF)kn) * (OFF)sizeof(T);
  const double* const* wd = EUPD ? g.dxh : g.dxe;
  const T dy = (T)width(wd[1], c.j), dz = (T)width(wd[2], c.k);
  const T ry = T(1) / dy, rz = T(1) / dz;
  const T rs = recip(mat_s);
  // x: the plane carried along is i - 1 (E update) or i (H update)
  T car[3];
  {
    const int ip = EUPD ? (c.ib == 0 ? nx - 1 : c.ib - 1) : c.ib;
#pragma unroll
    for (int q = 0; q < 3; ++q) car[q] = at(f, q * nc + (size_t)ip * plane, own0);
  }
#pragma unroll 1
  for (int i = c.ib; i < c.ie; ++i) {
    const OFF own = in_loop(own0), oy = in_loop(oy0), oz = in_loop(oz0);
    const size_t pi = (size_t)i * plane;
    const size_t pl = EUPD ? pi : (size_t)(i + 1 == nx ? 0 : i + 1) * plane;
    T ld[3], o[3], m[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) ld[q] = at(f, q * nc + pl, own);
    const T y0 = at(f, pi, oy), y2 = at(f, 2 * nc + pi, oy), z0 = at(f, pi, oz), z1 = at(f, nc + pi, oz);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      o[q] = at((const T*)out, q * nc + pi, own);
      m[q] = mat ? at(mat, q * nc + pi, own) : mat_s;
    }
    const T dx = (T)width_x<OFF>(wd[0], i), rx = recip(dx);
    const T (&here)[3] = EUPD ? ld : car;
    const T (&xn)[3] = EUPD ? car : ld;
    auto dif = [](T a, T b, T w, T r) { return div_by(EUPD ? a - b : b - a, w, r); };
    const T cc[3] = {dif(here[2], y2, dy, ry) - dif(here[1], z1, dz, rz),
                     dif(here[0], z0, dz, rz) - dif(here[2], xn[2], dx, rx),
                     dif(here[1], xn[1], dx, rx) - dif(here[0], y0, dy, ry)};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const T up = div_by(dt * cc[q], m[q], mat ? recip(m[q]) : rs);
      put(out, q * nc + pi, own, EUPD ? o[q] + up : o[q] - up);
      car[q] = ld[q];
    }
  }
}

__device__ __forceinline__ int wrap(int v, int n) {
  const int r = v % n;
  return r < 0 ? r + n : r;
}

// ---- leapfrog steps (mx_fdtd_run) ----------------------------------------------------
// One pass does S steps (1 or 2): E_0, H_0 and the materials are read once, E_S and H_S
// written once into a second buffer pair (the pairs alternate between passes, so no block
// ever reads a half-updated field).  Two steps a pass halve the bytes per step.
//
// A block is W waves; its lanes are 64 consecutive z cells and its rows W consecutive y
// cells, S of each on every side being halo that the neighbouring blocks compute as well
// (all indices wrap, so every lane holds a cell of the periodic grid).  It marches along x
// over `slab` planes: in iteration i, stage s (1..S) forms H_s and E_s, the fields after s
// steps, of plane i - 2 (s - 1):
//   phase 1:  H_s = H_{s-1} - dt curl_f(E_{s-1}) / mu     (all stages)
//   phase 2:  E_s = E_{s-1} + dt curl_b(H_s) / eps        (all stages)
// z neighbours come from the next lane, y neighbours through LDS (two components of E and
// of H per stage, one barrier per phase); x neighbours and the planes on their way from
// one stage to the next stay in the thread's registers.  E_0, H_0 and the materials are
// loaded one iteration ahead into alternating register sets, so nothing waits for a load
// in the iteration that issues it.  Only the last stage is stored, by the lanes and rows
// that are not halo: each stage's fields are valid one cell further in than those of the
// stage before.  The expressions are those of k_fdtd_update without contraction,
// so a run equals the step-by-step updates bit for bit.
//
// Bound by the divisions' issue (58% of the time at 256^3 in float64) together with the
// reads, 1.36 times the algorithmic ones with the halos.  In float32 the rows that a stage
// does not need are left out (a row is a wave: 38 of 48 row stages remain, 2 to 4 %; float64
// spills with it).  Per step of a run (in brackets with passes of one step and compiler
// divides): 256^3 float64 275 us (435), 256^3 float32 148 us (266), 190 x 160 x 201 float32
// 56 us (129).  12 or 14 rows (step_shape): 8 rows recompute half of theirs (330 / 170 us at
// 256^3), 16 rows leave float64 128 VGPRs of the 142 it needs (396 / 155 us).  Three steps a
// pass spill in float64 and gain nothing in float32 (159 us), since the halo grows with each.
// Two rows per thread measured 285 / 161 us.
constexpr int kStepRows = 12, kStepRowsMore = 14;   // (14 in float32 only)
constexpr int kStepMaxSlab = 128, kStepMinSlab = 4;
constexpr int kStepTab = 136;    // planes of the x table: the slab and the pipeline's run-in
enum : int { MU_ONE = 0, MU_SCALAR = 1, MU_FIELD = 2 };

// OFF: byte offsets within one component
template <typename T, typename OFF, int W, int S, bool EPS, int MU>
__global__ __launch_bounds__(64 * W) void k_fdtd_steps(RGrid g, T dt, const T* __restrict__ e0,
                                                               const T* __restrict__ h0, T* __restrict__ e1,
                                                               T* __restrict__ h1, const T* __restrict__ eps,
                                                               T eps_s, const T* __restrict__ mu, T mu_s, int slab) {
#pragma clang fp contract(off)
  constexpr int OY = W - 2 * S, OZ = 64 - 2 * S;
  constexpr bool kSkip = sizeof(T) == 4;
  __shared__ T sE[S][2][W + 1][64];   // E_{s-1} x, z by row
  __shared__ T sH[S][2][W + 1][64];   // H_s x, z by row + 1
  __shared__ T sX[kStepTab][4];       // dx_e, 1 / dx_e, dx_h, 1 / dx_h by plane
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const int nc = nx * ny * nz, plane = ny * nz;
  const int ntj = (ny + OY - 1) / OY, ntk = (nz + OZ - 1) / OZ, tiles = ntj * ntk;
  const int nwork = ((nx + slab - 1) / slab) * tiles;
  // workgroups are dealt round-robin to the 8 XCDs: XCD x takes a contiguous run of work
  // items, neighbouring tiles of one slab, so that the halos they share are in its own L2
  const int per = (nwork + 7) / 8;
  const int w = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (w >= nwork) return;
  const int slab_id = w / tiles, tile = w - slab_id * tiles;
  const int j0 = (tile / ntk) * OY, k0 = (tile % ntk) * OZ;
  const int ib = slab_id * slab, ie = min(ib + slab, nx);
  const int tz = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int j = j0 + ty - S, k = k0 + tz - S;
  const bool valid = ty >= S && ty < W - S && tz >= S && tz < 64 - S && j < ny && k < nz;
  const int jw = wrap(j, ny), kw = wrap(k, nz);
  // with 32-bit offsets an SGPR base per component and one VGPR offset per plane
  const OFF own = (OFF)(jw * nz + kw) * (OFF)sizeof(T);
  const OFF pbytes = (OFF)plane * (OFF)sizeof(T);
  auto ld = [&](const T* f, int c, OFF off) -> T {
    return *(const MX_GLOBAL T*)((const MX_GLOBAL char*)(f + (size_t)c * nc) + off);
  };
  auto st = [&](T* f, int c, OFF off, T v) {
    *(MX_GLOBAL T*)((MX_GLOBAL char*)(f + (size_t)c * nc) + off) = v;
  };

  // iterations t = 0..nt-1 hold plane first + t in stage 1; stage s trails by 2 (s - 1)
  const int first = ib - S, nt = (ie - ib) + 3 * S - 2;
  constexpr int kLag = 2 * (S - 1);
  for (int t = ty * 64 + tz; t < nt + kLag; t += 64 * W) {
    const int n = wrap(first - kLag + t, nx);
    const T de = (T)width(g.dxe[0], n), dh = (T)width(g.dxh[0], n);
    sX[t][0] = de;
    sX[t][1] = T(1) / de;
    sX[t][2] = dh;
    sX[t][3] = T(1) / dh;
  }
  const T dye = (T)width_u(g.dxe[1], jw), dyh = (T)width_u(g.dxh[1], jw);
  const T rye = wave_value(T(1) / dye), ryh = wave_value(T(1) / dyh);
  const T dze = (T)width(g.dxe[2], kw), dzh = (T)width(g.dxh[2], kw);
  const T rze = T(1) / dze, rzh = T(1) / dzh;
  const T rmu = wave_value(recip(mu_s)), reps = wave_value(recip(eps_s));

  struct In { T e[3], h[3], ep[3], m[3]; };   // E_0 of plane i+1; H_0, eps, mu of plane i
  In A, B;
  T Ec[S][3];                  // E_{s-1} of the stage's plane
  T En[S][3];                  // and of the next one (stage 1 has it in the In)
  T H1[S][3], H2[S][3];        // H_s of the plane before, and of the one before that
  T ep[2 * S - 1][3], er[2 * S - 1][3];   // eps of plane i, i-1, ... and its reciprocal
  T mm[2 * S - 1][3], mr[2 * S - 1][3];   // mu likewise
#pragma unroll
  for (int c = 0; c < 3; ++c) {
#pragma unroll
    for (int s = 0; s < S; ++s) Ec[s][c] = En[s][c] = H1[s][c] = H2[s][c] = T(0);
#pragma unroll
    for (int q = 0; q < 2 * S - 1; ++q) ep[q][c] = er[q][c] = mm[q][c] = mr[q][c] = T(1);
  }
  int pn = wrap(first, nx);    // the plane of H_0 and the materials in the next fetch
  auto fetch = [&](In& I) {
    const int p1 = pn + 1 == nx ? 0 : pn + 1;
    const OFF o1 = (OFF)p1 * pbytes + own, o0 = (OFF)pn * pbytes + own;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      I.e[c] = ld(e0, c, o1);
      I.h[c] = ld(h0, c, o0);
      if constexpr (EPS) I.ep[c] = ld(eps, c, o0);
      if constexpr (MU == MU_FIELD) I.m[c] = ld(mu, c, o0);
    }
    pn = p1;
  };
#pragma unroll
  for (int c = 0; c < 3; ++c) Ec[0][c] = ld(e0, c, (OFF)pn * pbytes + own);
  fetch(A);
  auto put_e = [&]() {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      sE[s][0][ty][tz] = Ec[s][0];
      sE[s][1][ty][tz] = Ec[s][2];
    }
  };
  // rows that no wave writes, read only for halo values that are never used
  if (ty == 0) {
#pragma unroll
    for (int s = 0; s < S; ++s) sE[s][0][W][tz] = sE[s][1][W][tz] = sH[s][0][0][tz] = sH[s][1][0][tz] = T(0);
  }
  put_e();
  __syncthreads();

  auto step = [&](const int t, In& cur, In& nxt) {
    fetch(nxt);
    // phase 1
    T hs[S][3] = {};
    if constexpr (MU == MU_FIELD) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        mm[0][c] = cur.m[c];
        mr[0][c] = recip(cur.m[c]);
      }
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (kSkip && (ty < s || ty > W - 2 - s)) continue;   // (uniform in a wave)
      const T* xt = sX[t + kLag - 2 * s];
      const T dx = xt[0], rx = xt[1];
      const T (&ec)[3] = Ec[s];
      const T (&en)[3] = s == 0 ? cur.e : En[s];
      const T ex_y = sE[s][0][ty + 1][tz], ez_y = sE[s][1][ty + 1][tz];
      const T ex_z = lane_next(ec[0]), ey_z = lane_next(ec[1]);
      const T cc[3] = {div_by(ez_y - ec[2], dye, rye) - div_by(ey_z - ec[1], dze, rze),
                       div_by(ex_z - ec[0], dze, rze) - div_by(en[2] - ec[2], dx, rx),
                       div_by(en[1] - ec[1], dx, rx) - div_by(ex_y - ec[0], dye, rye)};
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const T hb = s == 0 ? cur.h[c] : H2[s > 0 ? s - 1 : 0][c];
        T up = dt * cc[c];   // mu = 1: the quotient is the dividend
        if constexpr (MU == MU_FIELD) up = div_by(up, mm[2 * s][c], mr[2 * s][c]);
        if constexpr (MU == MU_SCALAR) up = div_by(up, mu_s, rmu);
        hs[s][c] = hb - up;
      }
      sH[s][0][ty + 1][tz] = hs[s][0];
      sH[s][1][ty + 1][tz] = hs[s][2];
    }
    __syncthreads();
    // phase 2
    T es[S][3] = {};
    if constexpr (EPS) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        ep[0][c] = cur.ep[c];
        er[0][c] = recip(cur.ep[c]);
      }
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (kSkip && (ty < s + 1 || ty > W - 2 - s)) continue;
      const T* xt = sX[t + kLag - 2 * s];
      const T dx = xt[2], rx = xt[3];
      const T hx = hs[s][0], hy = hs[s][1], hz = hs[s][2];
      const T hx_y = sH[s][0][ty][tz], hz_y = sH[s][1][ty][tz];
      const T hx_z = lane_prev(hx), hy_z = lane_prev(hy);
      const T cc[3] = {div_by(hz - hz_y, dyh, ryh) - div_by(hy - hy_z, dzh, rzh),
                       div_by(hx - hx_z, dzh, rzh) - div_by(hz - H1[s][2], dx, rx),
                       div_by(hy - H1[s][1], dx, rx) - div_by(hx - hx_y, dyh, ryh)};
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const T up = EPS ? div_by(dt * cc[c], ep[2 * s][c], er[2 * s][c]) : div_by(dt * cc[c], eps_s, reps);
        es[s][c] = Ec[s][c] + up;
      }
    }
    const int out = first + t - kLag;   // plane of the last stage
    if (valid && out >= ib && out < ie) {
      const OFF o = (OFF)out * pbytes + own;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        st(e1, c, o, es[S - 1][c]);
        st(h1, c, o, hs[S - 1][c]);
      }
    }
    // hand the planes on
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        H2[s][c] = H1[s][c];
        H1[s][c] = hs[s][c];
        Ec[s][c] = s == 0 ? cur.e[c] : En[s][c];
        if (s > 0) En[s][c] = es[s > 0 ? s - 1 : 0][c];
      }
#pragma unroll
      for (int q = 2 * S - 2; q > 0; --q) {
        ep[q][c] = ep[q - 1][c];
        er[q][c] = er[q - 1][c];
        mm[q][c] = mm[q - 1][c];
        mr[q][c] = mr[q - 1][c];
      }
    }
    put_e();
    // the barrier ends the step, in straight line with the LDS writes before it.  A form of this
    // kernel with the barrier as the loop's first instruction was compiled without the wait for
    // the writes on the back edge (seen in its assembly), and a row's old values were read now
    // and then; in the present build every barrier of the library comes after its wait
    __syncthreads();
  };
  int t = 0;
#pragma unroll 1
  for (; t + 1 < nt; t += 2) {
    step(t, A, B);
    step(t + 1, B, A);
  }
  if (t < nt) step(t, A, B);
}

// ---- convolutional PML (fdtd/pml.py:96-230) ---------------------------------------
// The six derivatives d_a f_c (a != c) use dx_h along every axis.
// Each layer the cell lies in (in the table's order: axis 0..2, polarity -1 then +1)
// scales the two derivatives along its axis by p2, advances the cell's psi_u, psi_v
// (u < v the components other than the axis) with p0 and p1, stores them in the psi
// precision, and adds s psi_u to the auxiliary term of u and -s psi_v to v's, in the psi
// precision, s = (-1, 1, -1)[axis].  Precisions follow the reference's array code with
// float64 widths: differences of field values in the field precision, divided by the
// float64 width, so derivatives, psi updates and the final sum are double; dt / material
// is taken in the material's (field) precision, dt / scalar in double.
//
// A thread owns one (y, z) column and marches along x over `slab` planes (see Column): the
// index divisions, the neighbour offsets, the y and z widths and the layer positions are
// per thread, the plane's are uniform, and the x neighbour comes from the thread's own
// registers.  Every array index of the derivatives is a constant (the layers are visited
// by face; a layer loop with run-time indexes put them into LDS), and the psi values and
// profiles a thread needs are loaded with the fields, not one dependent load after another
// in the layer's branch.  The widths divide through their reciprocals.
// Bound by latency at 4-5 waves per SIMD and by the traffic (48 and 36 B a cell in float32
// for the E and H updates, psi aside).  E + H update, 8-cell layers on all faces, per step:
// 150 x 141 x 130 float32 63 us (106 with a thread per cell), float64 85 us (120); 256^3
// float32 364 us (506), float64 622 us (666).
struct CpmlFace {
  int start, thickness;   // thickness 0: no layer on this face
  const double* p;        // p0, p1, p2, `thickness` values each
  void* psi;
};
struct CpmlTable { CpmlFace f[MX_CPML_MAX_LAYERS]; };   // by 2 axis + (polarity > 0)

// One layer along axis A at its cell, with profiles p and psi values (u, v) in q.
template <int A, typename TP>
__device__ __forceinline__ void cpml_layer(const double (&p)[3], TP (&q)[2], double (&d)[3][3], TP (&aux)[3]) {
  constexpr int u = A == 0 ? 1 : 0, v = A == 2 ? 1 : 2;
  d[A][u] *= p[2];
  d[A][v] *= p[2];
  q[0] = (TP)((double)q[0] * p[0]);
  q[1] = (TP)((double)q[1] * p[0]);
  q[0] = (TP)((double)q[0] + p[1] * d[A][v]);
  q[1] = (TP)((double)q[1] + p[1] * d[A][u]);
  const TP sg = A == 1 ? TP(1) : TP(-1);
  aux[u] = aux[u] + sg * q[0];
  aux[v] = aux[v] + (-sg) * q[1];
}

template <typename T, typename TP, bool EUPD, typename OFF>
__global__ __launch_bounds__(kFB) void k_cpml(RGrid g, T dt, const T* __restrict__ f, T* __restrict__ out,
                                              const T* __restrict__ mat, double const_scale, CpmlTable tab, int slab) {
  const Column c = column<OFF>(g, slab);
  if (!c.ok) return;
  const int nx = g.nx, ny = g.ny, nz = g.nz, plane = ny * nz;
  const size_t nc = (size_t)nx * plane;
  // neighbours of the difference: the cell before (E update) or after (H update)
  const int jn = EUPD ? (c.j == 0 ? ny - 1 : c.j - 1) : (c.j + 1 == ny ? 0 : c.j + 1);
  const int kn = EUPD ? (c.k == 0 ? nz - 1 : c.k - 1) : (c.k + 1 == nz ? 0 : c.k + 1);
  const OFF own0 = (OFF)c.t * (OFF)sizeof(T);
  const OFF oy0 = ((OFF)jn * (OFF)nz + (OFF)c.k) * (OFF)sizeof(T), oz0 = ((OFF)c.j * (OFF)nz + (OFF)kn) * (OFF)sizeof(T);
  const double wy = width(g.dxh[1], c.j), wz = width(g.dxh[2], c.k);
  const double ry = 1.0 / wy, rz = 1.0 / wz;
  // the thread's place in the y and z layers: whether it lies in one, its profiles, its
  // byte offset in a plane of the layer's psi
  bool in_y[2], in_z[2];
  OFF fy0[2], fz0[2];
  double ly[2][3], lz[2][3];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const CpmlFace &Y = tab.f[2 + q], &Z = tab.f[4 + q];
    const int py = c.j - Y.start, pz = c.k - Z.start;
    in_y[q] = (unsigned)py < (unsigned)Y.thickness;
    in_z[q] = (unsigned)pz < (unsigned)Z.thickness;
    fy0[q] = ((OFF)py * (OFF)nz + (OFF)c.k) * (OFF)sizeof(TP);
    fz0[q] = ((OFF)c.j * (OFF)Z.thickness + (OFF)pz) * (OFF)sizeof(TP);
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      ly[q][n] = in_y[q] ? Y.p[n * Y.thickness + py] : 0.0;
      lz[q][n] = in_z[q] ? Z.p[n * Z.thickness + pz] : 0.0;
    }
  }

  // x: the plane carried along is i - 1 of y, z (E update) or i of all (H update)
  T car[3];
  {
    const int ip = EUPD ? (c.ib == 0 ? nx - 1 : c.ib - 1) : c.ib;
#pragma unroll
    for (int q = 0; q < 3; ++q) car[q] = at(f, q * nc + (size_t)ip * plane, own0);
  }
#pragma unroll 1
  for (int i = c.ib; i < c.ie; ++i) {
    const OFF own = in_loop(own0), oy = in_loop(oy0), oz = in_loop(oz0), op = in_loop((OFF)c.t * (OFF)sizeof(TP));
    const OFF fy[2] = {in_loop(fy0[0]), in_loop(fy0[1])}, fz[2] = {in_loop(fz0[0]), in_loop(fz0[1])};
    const size_t pi = (size_t)i * plane;
    const size_t pl = EUPD ? pi : (size_t)(i + 1 == nx ? 0 : i + 1) * plane;
    T ld[3], o[3], m[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) ld[q] = at(f, q * nc + pl, own);
    const T y0 = at(f, pi, oy), y2 = at(f, 2 * nc + pi, oy), z0 = at(f, pi, oz), z1 = at(f, nc + pi, oz);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      o[q] = at((const T*)out, q * nc + pi, own);
      m[q] = mat ? at(mat, q * nc + pi, own) : T(1);
    }
    // psi of the layers the cell lies in, loaded with the fields
    TP sx[2][2], sy[2][2], sz[2][2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const CpmlFace &X = tab.f[q], &Y = tab.f[2 + q], &Z = tab.f[4 + q];
      if ((unsigned)(i - X.start) < (unsigned)X.thickness) {
        const size_t r = (size_t)(i - X.start) * plane;
        sx[q][0] = at((const TP*)X.psi, r, op);
        sx[q][1] = at((const TP*)X.psi, r + (size_t)X.thickness * plane, op);
      }
      if (in_y[q]) {
        sy[q][0] = at((const TP*)Y.psi, (size_t)i * Y.thickness * nz, fy[q]);
        sy[q][1] = at((const TP*)Y.psi, (size_t)(nx + i) * Y.thickness * nz, fy[q]);
      }
      if (in_z[q]) {
        sz[q][0] = at((const TP*)Z.psi, (size_t)i * ny * Z.thickness, fz[q]);
        sz[q][1] = at((const TP*)Z.psi, (size_t)(nx + i) * ny * Z.thickness, fz[q]);
      }
    }
    const double wx = width_x<OFF>(g.dxh[0], i), rx = recip(wx);
    const T (&here)[3] = EUPD ? ld : car;
    const T (&xn)[3] = EUPD ? car : ld;
    auto dif = [](T a, T b, double w, double r) { return div_by((double)(EUPD ? a - b : b - a), w, r); };
    double d[3][3];
    d[0][1] = dif(here[1], xn[1], wx, rx);
    d[0][2] = dif(here[2], xn[2], wx, rx);
    d[1][0] = dif(here[0], y0, wy, ry);
    d[1][2] = dif(here[2], y2, wy, ry);
    d[2][0] = dif(here[0], z0, wz, rz);
    d[2][1] = dif(here[1], z1, wz, rz);
#pragma unroll
    for (int q = 0; q < 3; ++q) car[q] = ld[q];
    TP aux[3] = {TP(0), TP(0), TP(0)};
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const CpmlFace& X = tab.f[q];
      const int pos = i - X.start;
      if ((unsigned)pos < (unsigned)X.thickness) {
        const double p[3] = {width_x<OFF>(X.p, pos), width_x<OFF>(X.p, X.thickness + pos), width_x<OFF>(X.p, 2 * X.thickness + pos)};
        cpml_layer<0, TP>(p, sx[q], d, aux);
        const size_t r = (size_t)pos * plane;
        put((TP*)X.psi, r, op, sx[q][0]);
        put((TP*)X.psi, r + (size_t)X.thickness * plane, op, sx[q][1]);
      }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const CpmlFace& Y = tab.f[2 + q];
      if (in_y[q]) {
        cpml_layer<1, TP>(ly[q], sy[q], d, aux);
        put((TP*)Y.psi, (size_t)i * Y.thickness * nz, fy[q], sy[q][0]);
        put((TP*)Y.psi, (size_t)(nx + i) * Y.thickness * nz, fy[q], sy[q][1]);
      }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const CpmlFace& Z = tab.f[4 + q];
      if (in_z[q]) {
        cpml_layer<2, TP>(lz[q], sz[q], d, aux);
        put((TP*)Z.psi, (size_t)i * ny * Z.thickness, fz[q], sz[q][0]);
        put((TP*)Z.psi, (size_t)(nx + i) * ny * Z.thickness, fz[q], sz[q][1]);
      }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int c1 = (q + 1) % 3, c2 = (q + 2) % 3;
      const double curl = (d[c1][c2] - d[c2][c1]) + (double)aux[q];
      const double scale = mat ? (double)div_by(dt, m[q], recip(m[q])) : const_scale;
      put(out, q * nc + pi, own, (T)(EUPD ? (double)o[q] + scale * curl : (double)o[q] - scale * curl));
    }
  }
}

// ---- conducting boundary (fdtd/boundaries.py:12-78) ---------------------------------
// One face's planes along `dir` are rewritten in place, one thread per (u, v) position
// of the face (u < v the other two axes).  A thread reads its column before it writes
// it and touches no other column, so threads need no ordering.
//   polarity -1, planes 0 and 1:
//     E: f_d[0] = 0, f_u[0] = f_u[1], f_v[0] = f_v[1]
//     H: f_d[0] = f_d[1], f_u[0] = f_v[0] = 0
//   polarity +1, planes L = n - 1, L - 1, L - 2:
//     E: f_d[L] = -f_d[L-2], f_d[L-1] = 0, f_u[L] = f_u[L-1], f_v[L] = f_v[L-1]
//     H: f_d[L] = f_d[L-1], f_u[L] = -f_u[L-2], f_u[L-1] = 0, and the same for v
// These are the image values of a mirror plane at 1/2 (polarity -1) or n - 3/2 (+1)
// across which tangential E and normal H are even, normal E and tangential H odd.
template <typename T>
__global__ __launch_bounds__(kFB) void k_conducting(int nx, int ny, int nz, int dir, int pol, int is_h,
                                                    T* __restrict__ f) {
  const int dims[3] = {nx, ny, nz};
  const long long strides[3] = {(long long)ny * nz, nz, 1};
  const int u = dir == 0 ? 1 : 0, v = dir == 2 ? 1 : 2;
  const long long nc = (long long)nx * ny * nz;
  const int nplane = dims[u] * dims[v];
  const int last = dims[dir] - 1;
  for (int t = blockIdx.x * kFB + threadIdx.x; t < nplane; t += gridDim.x * kFB) {
    const long long base = (t / dims[v]) * strides[u] + (t % dims[v]) * strides[v];
    auto at = [&](int comp, int plane) -> T& { return f[comp * nc + base + plane * strides[dir]]; };
    if (pol < 0) {
      if (!is_h) {
        const T fu = at(u, 1), fv = at(v, 1);
        at(dir, 0) = T(0);
        at(u, 0) = fu;
        at(v, 0) = fv;
      } else {
        const T fd = at(dir, 1);
        at(dir, 0) = fd;
        at(u, 0) = T(0);
        at(v, 0) = T(0);
      }
    } else {
      if (!is_h) {
        const T fd = at(dir, last - 2), fu = at(u, last - 1), fv = at(v, last - 1);
        at(dir, last) = -fd;
        at(dir, last - 1) = T(0);
        at(u, last) = fu;
        at(v, last) = fv;
      } else {
        const T fd = at(dir, last - 1), fu = at(u, last - 2), fv = at(v, last - 2);
        at(dir, last) = fd;
        at(u, last) = -fu;
        at(u, last - 1) = T(0);
        at(v, last) = -fv;
        at(v, last - 1) = T(0);
      }
    }
  }
}

// ---- energy and Poynting flux (fdtd/energy.py) ------------------------------------
// Rounding follows the reference's array expressions: the field products and the
// component sum in the field precision (in component order, starting from the x term),
// the widths in double (the float64 width arrays promote) multiplied one axis at a time,
// and nothing contracted into fused multiply-adds.  `form` is one of MX_ENERGY_*.

// HBM-bound, a thread per cell, every load of a cell before any is used.  256^3: energy_hstep
// with widths float64 314 us, float32 163 us (358 / 208 with each component's loads behind the
// one before; columns marching along x 345 / 189), without widths 303 / 162 us (327 / 177; 343 / 188).

template <typename T>
__global__ __launch_bounds__(kFB) void k_energy(RGrid g, int form, T dt, const T* __restrict__ f0,
                                                const T* __restrict__ f1, const T* __restrict__ f2,
                                                const T* __restrict__ f3, const T* __restrict__ eps, T eps_s,
                                                const T* __restrict__ mu, T mu_s, double* __restrict__ out, int order) {
#pragma clang fp contract(off)
  const Column col = column<size_t>(g, order);
  if (!col.ok) return;
  const int i = col.ib, nc = g.nx * g.ny * g.nz, cell = i * g.ny * g.nz + col.t;
  const double wex = width(g.dxe[0], i), wey = width(g.dxe[1], col.j), wez = width(g.dxe[2], col.k);
  const double whx = width(g.dxh[0], i), why = width(g.dxh[1], col.j), whz = width(g.dxh[2], col.k);
  // every load of the cell before any is used (f2, f3 and the materials only if given)
  T a0[3], a1[3], a2[3], a3[3], me[3], mh[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const int q = c * nc + cell;
    a0[c] = f0[q];
    a1[c] = f1[q];
    a2[c] = f2 ? f2[q] : T(0);
    a3[c] = f3 ? f3[q] : T(0);
    me[c] = eps ? eps[q] : eps_s;
    mh[c] = mu ? mu[q] : mu_s;
  }
  T se = T(0), sh = T(0);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    T ee, hh = T(0);
    switch (form) {
      case MX_ENERGY_DXMUL: ee = a0[c]; hh = a1[c]; break;
      case MX_ENERGY_HSTEP: ee = a0[c] * a2[c]; hh = a1[c] * a1[c]; break;
      case MX_ENERGY_ESTEP: ee = a1[c] * a1[c]; hh = a0[c] * a2[c]; break;
      case MX_ENERGY_H2E: ee = a2[c] * (a2[c] - a0[c]) / dt; hh = a1[c] * (a3[c] - a1[c]) / dt; break;
      case MX_ENERGY_E2H: ee = a1[c] * (a3[c] - a1[c]) / dt; hh = a2[c] * (a2[c] - a0[c]) / dt; break;
      default: ee = a0[c] * a1[c]; break;   // j0 . e1, no material
    }
    const T we = form == MX_ENERGY_J ? ee : ee * me[c];
    const T wh = hh * mh[c];
    se = c == 0 ? we : se + we;
    sh = c == 0 ? wh : sh + wh;
  }
  const double ue = (double)se * wex * wey * wez;
  out[cell] = form == MX_ENERGY_J ? ue : ue + (double)sh * whx * why * whz;
}

// s = E(+1) x H with both width-weighted (fdtd/energy.py:10-87): s_x = ey(i+1) hz - ez(i+1) hy
// and cyclically, E taken at the next cell along the component's axis (periodic), in
// double, stored in the field precision.
// HBM-bound.  With widths in columns, which load the y and z ones once: 256^3 float64 235 us,
// float32 120 us (256 / 134 before; a thread per cell 254 / 127); without, a thread per cell:
// 211 / 104 us (224 / 113; columns 231 / 118).
template <typename T, typename OFF>
__global__ __launch_bounds__(kFB) void k_poynting(RGrid g, const T* __restrict__ e, const T* __restrict__ h,
                                                  T* __restrict__ s, int slab) {
#pragma clang fp contract(off)
  const Column col = column<OFF>(g, slab);
  if (!col.ok) return;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const size_t plane = (size_t)ny * nz, nc = nx * plane;
  const int jn = col.j + 1 == ny ? 0 : col.j + 1, kn = col.k + 1 == nz ? 0 : col.k + 1;
  const OFF own0 = (OFF)col.t * (OFF)sizeof(T);
  const OFF oy0 = ((OFF)jn * (OFF)nz + (OFF)col.k) * (OFF)sizeof(T);
  const OFF oz0 = ((OFF)col.j * (OFF)nz + (OFF)kn) * (OFF)sizeof(T);
  const double wey = width(g.dxe[1], col.j), wez = width(g.dxe[2], col.k);
  const double why = width(g.dxh[1], col.j), whz = width(g.dxh[2], col.k);
#pragma unroll 1
  for (int i = col.ib; i < col.ie; ++i) {
    const OFF own = in_loop(own0), oy = in_loop(oy0), oz = in_loop(oz0);
    const size_t pi = i * plane, pn = (size_t)(i + 1 == nx ? 0 : i + 1) * plane;
    const T h0 = at(h, pi, own), h1 = at(h, nc + pi, own), h2 = at(h, 2 * nc + pi, own);
    const T eyx = at(e, nc + pn, own), ezx = at(e, 2 * nc + pn, own), ezy = at(e, 2 * nc + pi, oy), exy = at(e, pi, oy);
    const T exz = at(e, pi, oz), eyz = at(e, nc + pi, oz);
    const double wex = width_x<OFF>(g.dxe[0], i);
    const double hx = (double)h0 * width_x<OFF>(g.dxh[0], i), hy = (double)h1 * why, hz = (double)h2 * whz;
    const double s0 = ((double)eyx * wey) * hz - ((double)ezx * wez) * hy;
    const double s1 = ((double)ezy * wez) * hx - ((double)exy * wex) * hz;
    const double s2 = ((double)exz * wex) * hy - ((double)eyz * wey) * hx;
    put(s, pi, own, (T)s0);
    put(s, nc + pi, own, (T)s1);
    put(s, 2 * nc + pi, own, (T)s2);
  }
}

// ds = sum_a (s_a - s_a(previous cell along a)), unit spacing (deriv_back() without
// widths, fdtd/energy.py:90-125), in the field precision.
template <typename T, typename OFF>
__global__ __launch_bounds__(kFB) void k_poynting_div(RGrid g, const T* __restrict__ s, T* __restrict__ ds, int slab) {
#pragma clang fp contract(off)
  const Column col = column<OFF>(g, slab);
  if (!col.ok) return;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const size_t plane = (size_t)ny * nz, nc = nx * plane;
  const int jp = col.j == 0 ? ny - 1 : col.j - 1, kp = col.k == 0 ? nz - 1 : col.k - 1;
  const OFF own0 = (OFF)col.t * (OFF)sizeof(T);
  const OFF oy0 = ((OFF)jp * (OFF)nz + (OFF)col.k) * (OFF)sizeof(T);
  const OFF oz0 = ((OFF)col.j * (OFF)nz + (OFF)kp) * (OFF)sizeof(T);
  T sx = at(s, (size_t)(col.ib == 0 ? nx - 1 : col.ib - 1) * plane, own0);
#pragma unroll 1
  for (int i = col.ib; i < col.ie; ++i) {
    const OFF own = in_loop(own0), oy = in_loop(oy0), oz = in_loop(oz0);
    const size_t pi = i * plane;
    const T s0 = at(s, pi, own);
    const T dx = s0 - sx;
    const T dy = at(s, nc + pi, own) - at(s, nc + pi, oy);
    const T dz = at(s, 2 * nc + pi, own) - at(s, 2 * nc + pi, oz);
    put(ds, pi, own, dx + dy + dz);
    sx = s0;
  }
}

bool rgrid(const mx_fdtd_grid* g, RGrid* v, std::string* why) {
  if (!g || g->nx < 1 || g->ny < 1 || g->nz < 1) { *why = "bad grid"; return false; }
  if (3LL * g->nx * g->ny * g->nz >= (1LL << 31)) { *why = "grid too large (3N must be < 2^31)"; return false; }
  v->nx = g->nx; v->ny = g->ny; v->nz = g->nz;
  for (int a = 0; a < 3; ++a) {
    v->dxe[a] = g->dxe[a];
    v->dxh[a] = g->dxh[a];
  }
  return true;
}

// Launch of a kernel with a thread per cell (the 64-bit form of `column`).  Work goes by XCD
// where nine values a cell stay in the 256 MB cache, else in the order of the blocks, as the
// memory channels like it better: Poynting flux without widths of 100 x 110 x 120 in float64
// 15.3 us by XCD, 20.7 plain; 256^3 float64 237 / 211 us, float32 114 / 104; energy of 256^3 float64
// 330 / 303 us.
struct ColumnGrid { bool marches; int slab; unsigned blocks; };
ColumnGrid cell_grid(const RGrid& v, int prec) {
  const long long cells = (long long)v.nx * v.ny * v.nz, bytes = 9 * cells * (prec == MX_REAL64 ? 8 : 4);
  const long long nwork = (cells + kFB - 1) / kFB;
  return {false, bytes <= (256ll << 20) ? 1 : 0, (unsigned)((nwork + 7) / 8 * 8)};
}

// Launch of a column kernel: slabs of at most `deepest` planes (6, 4 or 2), shallower while
// the chip has fewer than 8 blocks per CU.  Slabs of 2/4/6/10/16 planes, H then E update of
// float64: 200 x 181 x 190 232.6, 233.8, 236.8, 239.0, 242.2 us, 256^3 559, 560, 554, 576, 564;
// float32: 200 x 181 x 190 85.0, 84.2, 86.7, 89.0, 93.2, 256^3 275, 273, 278, 285, 281.  With
// CPML, float32, slabs of 2/4/6/8: 228 x 100 x 180 50.2, 43.2, 42.8, 43.5 us.
// A plane of fewer than kThinPlane cells leaves too much of a block without columns, and the
// byte offsets of one, in the widest type that the kernel holds a value per cell of
// (`prec`), may not fit 32 bits: then a thread per cell.  Columns / cells, E update of float64:
// 2000000 x 1 x 1 887 / 30 us, 40000 x 8 x 10 50 / 43, 4000 x 16 x 15 15.4 / 14.7, 3000 x 20 x 20
// 19.1 / 17.9, 5000 x 32 x 32 89 / 91; with CPML, float32: 8000 x 25 x 25 69 / 80, 3000 x 300 x 1 18 / 12.
constexpr long long kThinPlane = 512;
ColumnGrid column_grid(const RGrid& v, int prec, int deepest) {
  const long long plane = (long long)v.ny * v.nz;
  if (plane < kThinPlane || plane * (prec == MX_REAL64 ? 8 : 4) >= (1ll << 32)) return cell_grid(v, prec);
  const long long pieces = (plane + kFB - 1) / kFB;
  int slab = 0;
  for (int want : {6, 4, 2}) {
    if (want > deepest) continue;
    slab = std::min(want, v.nx);
    if (pieces * ((v.nx + slab - 1) / slab) >= 2048) break;
  }
  return {true, slab, (unsigned)((pieces * ((v.nx + slab - 1) / slab) + 7) / 8 * 8)};
}

template <bool EUPD>
hipError_t launch_update(const RGrid& v, int prec, double dt, const void* f, void* out, const void* mat, double mat_s,
                         hipStream_t s) {
  // float64 with a material field, from twice the cache on: a thread per cell.  E update,
  // columns / cells: 170 x 171 x 172 88 / 92 us, 180^3 107 / 106, 210 x 200 x 170 139 / 129,
  // 256^3 318 / 303, 150 x 400 x 400 462 / 426; without a material (H) 80 / 86 at 180^3, 240 / 243 at 256^3
  // (float32 E update 152 / 150 at 256^3, 47 / 64 at 200 x 181 x 190: columns).
  const bool cells = prec == MX_REAL64 && mat && 96ll * v.nx * v.ny * v.nz > (512ll << 20);
  const ColumnGrid cg = cells ? cell_grid(v, prec) : column_grid(v, prec, 4);
#define MX_UPDATE_CASE(T, OFF)                                                                                      \
  hipLaunchKernelGGL((k_fdtd_update<T, EUPD, OFF>), dim3(cg.blocks), dim3(kFB), 0, s, v, (T)dt, (const T*)f, (T*)out, \
                     (const T*)mat, (T)mat_s, cg.slab)
  if (prec == MX_REAL64) { if (cg.marches) MX_UPDATE_CASE(double, unsigned); else MX_UPDATE_CASE(double, size_t); }
  else { if (cg.marches) MX_UPDATE_CASE(float, unsigned); else MX_UPDATE_CASE(float, size_t); }
#undef MX_UPDATE_CASE
  return hipGetLastError();
}
hipError_t launch_h(const RGrid& v, int prec, double dt, const void* e, void* h, const void* mu, double mu_s,
                    hipStream_t s) {
  return launch_update<false>(v, prec, dt, e, h, mu, mu_s, s);
}
hipError_t launch_e(const RGrid& v, int prec, double dt, void* e, const void* h, const void* eps, double eps_s,
                    hipStream_t s) {
  return launch_update<true>(v, prec, dt, h, e, eps, eps_s, s);
}

hipError_t launch_conducting(const RGrid& v, int prec, int dir, int pol, int is_h, void* f, hipStream_t s) {
  const int dims[3] = {v.nx, v.ny, v.nz};
  const long long nplane = (long long)dims[dir == 0 ? 1 : 0] * dims[dir == 2 ? 1 : 2];
  const long long nb = (nplane + kFB - 1) / kFB;
  const unsigned grid = (unsigned)(nb > 16384 ? 16384 : nb);
  if (prec == MX_REAL64)
    hipLaunchKernelGGL(k_conducting<double>, dim3(grid), dim3(kFB), 0, s, v.nx, v.ny, v.nz, dir, pol, is_h,
                       (double*)f);
  else
    hipLaunchKernelGGL(k_conducting<float>, dim3(grid), dim3(kFB), 0, s, v.nx, v.ny, v.nz, dir, pol, is_h,
                       (float*)f);
  return hipGetLastError();
}

hipError_t launch_energy(const RGrid& v, int prec, int form, double dt, const void* const* f, const void* eps,
                         double eps_s, const void* mu, double mu_s, double* out, hipStream_t s) {
  const ColumnGrid cg = cell_grid(v, prec);
#define MX_ENERGY_CASE(T)                                                                                          \
  hipLaunchKernelGGL(k_energy<T>, dim3(cg.blocks), dim3(kFB), 0, s, v, form, (T)dt, (const T*)f[0], (const T*)f[1], \
                     (const T*)f[2], (const T*)f[3], (const T*)eps, (T)eps_s, (const T*)mu, (T)mu_s, out, cg.slab)
  if (prec == MX_REAL64) MX_ENERGY_CASE(double);
  else MX_ENERGY_CASE(float);
#undef MX_ENERGY_CASE
  return hipGetLastError();
}

hipError_t launch_poynting(const RGrid& v, int prec, const void* e, const void* h, void* out, hipStream_t s) {
  bool widths = false;
  for (int a = 0; a < 3; ++a) widths = widths || v.dxe[a] || v.dxh[a];
  const ColumnGrid cg = widths ? column_grid(v, prec, 6) : cell_grid(v, prec);
#define MX_POYNTING_CASE(T, OFF)                                                                                        \
  hipLaunchKernelGGL((k_poynting<T, OFF>), dim3(cg.blocks), dim3(kFB), 0, s, v, (const T*)e, (const T*)h, (T*)out, cg.slab)
  if (prec == MX_REAL64) { if (cg.marches) MX_POYNTING_CASE(double, unsigned); else MX_POYNTING_CASE(double, size_t); }
  else { if (cg.marches) MX_POYNTING_CASE(float, unsigned); else MX_POYNTING_CASE(float, size_t); }
#undef MX_POYNTING_CASE
  return hipGetLastError();
}

hipError_t launch_poynting_div(const RGrid& v, int prec, const void* sv, void* ds, hipStream_t s) {
  const ColumnGrid cg = column_grid(v, prec, 6);
#define MX_DIV_CASE(T, OFF) \
  hipLaunchKernelGGL((k_poynting_div<T, OFF>), dim3(cg.blocks), dim3(kFB), 0, s, v, (const T*)sv, (T*)ds, cg.slab)
  if (prec == MX_REAL64) { if (cg.marches) MX_DIV_CASE(double, unsigned); else MX_DIV_CASE(double, size_t); }
  else { if (cg.marches) MX_DIV_CASE(float, unsigned); else MX_DIV_CASE(float, size_t); }
#undef MX_DIV_CASE
  return hipGetLastError();
}

// Layer table of a CPML update: faces in increasing (axis, polarity) order (the order
// the reference accumulates in), each inside the grid, with its arrays.
bool cpml_table(const RGrid& v, const mx_cpml_layer* layers, int n, bool eupd, CpmlTable* tab, std::string* why) {
  if (n < 0 || n > MX_CPML_MAX_LAYERS) { *why = "nlayers must be 0..6"; return false; }
  if (n > 0 && !layers) { *why = "null layer table"; return false; }
  const int dims[3] = {v.nx, v.ny, v.nz};
  for (CpmlFace& f : tab->f) f = CpmlFace{0, 0, nullptr, nullptr};
  int prev = -1;
  for (int q = 0; q < n; ++q) {
    const mx_cpml_layer& L = layers[q];
    if (L.axis < 0 || L.axis > 2) { *why = "layer axis must be 0, 1 or 2"; return false; }
    if (L.polarity != -1 && L.polarity != 1) { *why = "layer polarity must be -1 or +1"; return false; }
    if (L.thickness < 1 || L.thickness > dims[L.axis]) { *why = "layer thickness must be 1..n along its axis"; return false; }
    const int key = 2 * L.axis + (L.polarity > 0);
    if (key <= prev) { *why = "layers must be in increasing (axis, polarity) order, one per face"; return false; }
    prev = key;
    if (!L.p_e || !L.p_h || !L.psi_e || !L.psi_h) { *why = "null layer array"; return false; }
    tab->f[key] = CpmlFace{L.polarity < 0 ? 0 : dims[L.axis] - L.thickness, L.thickness, eupd ? L.p_e : L.p_h,
                           eupd ? L.psi_e : L.psi_h};
  }
  return true;
}

template <bool EUPD>
hipError_t launch_cpml(const RGrid& v, int prec, int psi_prec, double dt, const void* f, void* out,
                       const void* mat, double mat_s, const CpmlTable& tab, hipStream_t s) {
  // a layer's plane has at most the grid plane's cells, in the psi precision
  const ColumnGrid cg = column_grid(v, prec == MX_REAL64 ? prec : psi_prec, 6);
#define MX_CPML_CASE(T, TP, OFF)                                                                              \
  hipLaunchKernelGGL((k_cpml<T, TP, EUPD, OFF>), dim3(cg.blocks), dim3(kFB), 0, s, v, (T)dt, (const T*)f, (T*)out, \
                     (const T*)mat, dt / mat_s, tab, cg.slab)
  if (prec == MX_REAL64) {
    if (psi_prec == MX_REAL64) { if (cg.marches) MX_CPML_CASE(double, double, unsigned); else MX_CPML_CASE(double, double, size_t); }
    else { if (cg.marches) MX_CPML_CASE(double, float, unsigned); else MX_CPML_CASE(double, float, size_t); }
  } else {
    if (psi_prec == MX_REAL64) { if (cg.marches) MX_CPML_CASE(float, double, unsigned); else MX_CPML_CASE(float, double, size_t); }
    else { if (cg.marches) MX_CPML_CASE(float, float, unsigned); else MX_CPML_CASE(float, float, size_t); }
  }
#undef MX_CPML_CASE
  return hipGetLastError();
}

struct StepShape { int rows, slab; double cost; };
long long step_tiles(const RGrid& v, int rows, int steps) {
  const int oy = rows - 2 * steps, oz = 64 - 2 * steps;
  return (long long)((v.ny + oy - 1) / oy) * ((v.nz + oz - 1) / oz);
}

// Rows and slab depth of a pass: those with the least modelled time, over all equal divisions
// of x (at most 125 depths a row count, 0.5 us, once per run).  A block takes slab + 3 S - 2 iterations, each as long as its rows are many; the n
// blocks that a CU gets (256 CUs) cost n, plus a fifth of one in float32, where two blocks
// share a CU.  Measured at 256^3 float64, two steps: slabs 16/24/32/48/64/128 model
// 200/196/180/208/204/264, time 611/576/542/595/572/696 us.  Float32 with 14 rows instead of
// 12, model / time: 100^3 1.17 / 1.13, 150x141x130 0.82 / 0.85, 320^3 0.94 / 0.88, 256^3 1.15 /
// 1.02 (float64 has no registers for 14).  Against 12 rows and slabs of powers of two and
// three halves of them, us per step: float32 150x141x130 with mu 45 / 39, 320^3 309 / 256,
// 64x150x250 with mu 38 / 31, float64 150x141x130 with mu 114 / 89, 190x160x201 123 / 111;
// 256^3, 60^3 and 100^3 alike.
StepShape step_shape(const RGrid& v, int steps, size_t elem) {
  static const int forced = [] {   // MEANAS_AMD_FDTD_SLAB overrides the slab depth (tuning runs)
    const char* env = getenv("MEANAS_AMD_FDTD_SLAB");
    return env ? atoi(env) : 0;
  }();
  const int deepest = forced > 0 ? std::min(forced, kStepMaxSlab) : kStepMaxSlab;
  const int shallowest = forced > 0 ? deepest : kStepMinSlab;
  StepShape best{0, 0, 0.0};
  for (int rows : {kStepRows, kStepRowsMore}) {
    if (rows > kStepRows && elem != 4) continue;
    const long long tiles = step_tiles(v, rows, steps);
    // the equal divisions: every slab depth that is the ceiling of nx over some count
    for (int depth = std::min(deepest, v.nx); depth >= std::min(shallowest, v.nx); --depth) {
      const int count = (v.nx + depth - 1) / depth, slab = (v.nx + count - 1) / count;
      if (slab != depth && forced <= 0) continue;
      const double n = (double)((tiles * count + 255) / 256) + (elem == 4 ? 0.2 : 0.0);
      const double cost = n * (depth + 3 * steps - 2) * rows;
      if (best.slab == 0 || cost < best.cost) best = {rows, depth, cost};
    }
  }
  return best;
}

template <typename T, typename OFF, int S>
hipError_t launch_pass(const RGrid& v, const StepShape& shape, T dt, const void* ei, const void* hi, void* eo, void* ho, const void* eps,
                       double eps_s, const void* mu, double mu_s, hipStream_t s) {
  static_assert(kStepMaxSlab + 5 * S - 4 <= kStepTab, "x table");
  const int slab = shape.slab;
  const long long nwork = step_tiles(v, shape.rows, S) * ((v.nx + slab - 1) / slab);
  const unsigned nb = (unsigned)(((nwork + 7) / 8) * 8);
#define MX_STEP_CASE(EPS, MU)                                                                                   \
  hipLaunchKernelGGL((k_fdtd_steps<T, OFF, W, S, EPS, MU>), dim3(nb), dim3(64, W), 0, s, v, dt, (const T*)ei,        \
                     (const T*)hi, (T*)eo, (T*)ho, (const T*)eps, (T)eps_s, (const T*)mu, (T)mu_s, slab)
  auto go = [&](auto rows) {
    constexpr int W = decltype(rows)::value;
    if constexpr (S == 1 || sizeof(OFF) == 4) {   // (single_steps)
      if (mu) {
        if (eps) MX_STEP_CASE(true, MU_FIELD); else MX_STEP_CASE(false, MU_FIELD);
        return;
      }
    }
    if (mu_s == 1.0) { if (eps) MX_STEP_CASE(true, MU_ONE); else MX_STEP_CASE(false, MU_ONE); }
    else { if (eps) MX_STEP_CASE(true, MU_SCALAR); else MX_STEP_CASE(false, MU_SCALAR); }
  };
  if constexpr (sizeof(T) == 4) {
    if (shape.rows == kStepRowsMore) go(std::integral_constant<int, kStepRowsMore>());
    else go(std::integral_constant<int, kStepRows>());
  } else {
    go(std::integral_constant<int, kStepRows>());
  }
#undef MX_STEP_CASE
  return hipGetLastError();
}

// Grids of few x planes, where a pass's run-in (3 S - 2 planes a slab) is most of its work.
// Separate updates on one plane, and on two while the fields and materials stay in the cache;
// passes of one step on two, and in float64 with a mu field (whose two-step pass spills) on up
// to four.  us per step, two steps a pass / one / separate: float64 1 x 1000 x 1000 55 / 47 / 35, with mu
// 70 / 55 / 37, 1 x 4000 x 4000 698 / 640 / 539; 2 x 1000 x 1000 69 / 65 / 57, 2 x 2000 x 2000 254 / 251 / 272, with
// mu 382 / 301 / 322; 4 x 500 x 500 33 / 33 / 36, with mu 46 / 38 / 38; 5 x 1000 x 1000 with mu 159 / 190 / 231;
// float32 1 x 1000 x 1000 37 / 30 / 24, 2 x 1000 x 1000 43 / 34 / 34, 3 x 1000 x 1000 50 / 48 / 46.
bool separate_updates(const RGrid& v, int prec, bool mu_field) {
  const long long bytes = (mu_field ? 12ll : 9ll) * v.nx * v.ny * v.nz * (prec == MX_REAL64 ? 8 : 4);
  return v.nx == 1 || (v.nx == 2 && bytes <= (256ll << 20));
}
// `wide`: 64-bit offsets (components of 4 GiB and more), which spill more with a mu field:
// 840 x 805 x 800 with mu 34 ms a step in passes of two, 13.6 of one (without mu 7.8 of two).
bool single_steps(const RGrid& v, int prec, bool mu_field, bool wide) {
  return v.nx <= 2 || (prec == MX_REAL64 && mu_field && (v.nx <= 4 || wide));
}

// `steps` steps by passes of two, a last single one if their number is odd (or of one each):
// (e, h) -> (e2, h2) -> (e, h) -> ...; *passes: how many
template <typename T, typename OFF>
hipError_t launch_steps(const RGrid& v, T dt, void* e, void* h, void* e2, void* h2, const void* eps, double eps_s,
                        const void* mu, double mu_s, int steps, int* passes, hipStream_t s) {
  const bool single = single_steps(v, sizeof(T) == 8 ? MX_REAL64 : MX_REAL32, mu != nullptr, sizeof(OFF) == 8);
  *passes = single ? steps : steps / 2 + steps % 2;
  const StepShape two = step_shape(v, 2, sizeof(T)), one = step_shape(v, 1, sizeof(T));
  for (int t = 0; t < *passes; ++t) {
    void* ei = (t & 1) ? e2 : e;
    void* hi = (t & 1) ? h2 : h;
    void* eo = (t & 1) ? e : e2;
    void* ho = (t & 1) ? h : h2;
    const hipError_t err = !single && 2 * t + 2 <= steps
                               ? launch_pass<T, OFF, 2>(v, two, dt, ei, hi, eo, ho, eps, eps_s, mu, mu_s, s)
                               : launch_pass<T, OFF, 1>(v, one, dt, ei, hi, eo, ho, eps, eps_s, mu, mu_s, s);
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

int check_args(const mx_fdtd_grid* g, int prec, const void* a, const void* b, RGrid* v, const char* who) {
  std::string why;
  if (!rgrid(g, v, &why)) return set_error(std::string(who) + ": " + why);
  if (prec != MX_REAL32 && prec != MX_REAL64) return set_error(std::string(who) + ": prec must be MX_REAL32 or MX_REAL64");
  if (!a || !b) return set_error(std::string(who) + ": null field");
  return 0;
}

}  // namespace
}  // namespace mx

extern "C" {

int mx_fdtd_h(const mx_fdtd_grid* g, int32_t prec, double dt, const void* e, void* h, const void* mu,
              double mu_scalar, void* stream) {
  mx::RGrid v;
  if (mx::check_args(g, prec, e, h, &v, "mx_fdtd_h")) return -1;
  const hipError_t err = mx::launch_h(v, prec, dt, e, h, mu, mu_scalar, reinterpret_cast<hipStream_t>(stream));
  return err == hipSuccess ? 0 : mx::set_error(std::string("mx_fdtd_h: ") + hipGetErrorString(err));
}

int mx_fdtd_e(const mx_fdtd_grid* g, int32_t prec, double dt, void* e, const void* h, const void* eps,
              double eps_scalar, void* stream) {
  mx::RGrid v;
  if (mx::check_args(g, prec, e, h, &v, "mx_fdtd_e")) return -1;
  const hipError_t err = mx::launch_e(v, prec, dt, e, h, eps, eps_scalar, reinterpret_cast<hipStream_t>(stream));
  return err == hipSuccess ? 0 : mx::set_error(std::string("mx_fdtd_e: ") + hipGetErrorString(err));
}

int mx_fdtd_run(const mx_fdtd_grid* g, int32_t prec, double dt, void* e, void* h, const void* eps,
                double eps_scalar, const void* mu, double mu_scalar, int32_t steps, void* stream) {
  mx::RGrid v;
  if (mx::check_args(g, prec, e, h, &v, "mx_fdtd_run")) return -1;
  if (steps < 0) return mx::set_error("mx_fdtd_run: steps < 0");
  if (steps == 0) return 0;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const size_t comp = (size_t)v.nx * v.ny * v.nz * (prec == MX_REAL64 ? 8 : 4), bytes = 3 * comp;
  if (mx::separate_updates(v, prec, mu != nullptr)) {
    for (int t = 0; t < steps; ++t) {
      hipError_t err = mx::launch_h(v, prec, dt, e, h, mu, mu_scalar, s);
      if (err == hipSuccess) err = mx::launch_e(v, prec, dt, e, h, eps, eps_scalar, s);
      if (err != hipSuccess) return mx::set_error(std::string("mx_fdtd_run: ") + hipGetErrorString(err));
    }
    return 0;
  }
  // passes alternate between (e, h) and a second pair, allocated in stream order
  void* e2 = nullptr;
  void* h2 = nullptr;
  int passes = 0;
  hipError_t err = hipMallocAsync(&e2, bytes, s);
  if (err == hipSuccess) err = hipMallocAsync(&h2, bytes, s);
  if (err == hipSuccess)
    err = prec == MX_REAL32
              ? mx::launch_steps<float, unsigned>(v, (float)dt, e, h, e2, h2, eps, eps_scalar, mu, mu_scalar, steps, &passes, s)
          : comp < (size_t)1 << 32
              ? mx::launch_steps<double, unsigned>(v, dt, e, h, e2, h2, eps, eps_scalar, mu, mu_scalar, steps, &passes, s)
              : mx::launch_steps<double, size_t>(v, dt, e, h, e2, h2, eps, eps_scalar, mu, mu_scalar, steps, &passes, s);
  if (err == hipSuccess && (passes & 1)) {   // the last pass wrote the second pair
    err = hipMemcpyAsync(e, e2, bytes, hipMemcpyDeviceToDevice, s);
    if (err == hipSuccess) err = hipMemcpyAsync(h, h2, bytes, hipMemcpyDeviceToDevice, s);
  }
  if (e2) (void)hipFreeAsync(e2, s);
  if (h2) (void)hipFreeAsync(h2, s);
  return err == hipSuccess ? 0 : mx::set_error(std::string("mx_fdtd_run: ") + hipGetErrorString(err));
}

int mx_fdtd_cpml_e(const mx_fdtd_grid* g, int32_t prec, int32_t psi_prec, double dt, void* e, const void* h,
                   const void* eps, double eps_scalar, const mx_cpml_layer* layers, int32_t nlayers, void* stream) {
  mx::RGrid v;
  if (mx::check_args(g, prec, e, h, &v, "mx_fdtd_cpml_e")) return -1;
  if (psi_prec != MX_REAL32 && psi_prec != MX_REAL64) return mx::set_error("mx_fdtd_cpml_e: psi_prec must be MX_REAL32 or MX_REAL64");
  mx::CpmlTable tab;
  std::string why;
  if (!mx::cpml_table(v, layers, nlayers, true, &tab, &why)) return mx::set_error("mx_fdtd_cpml_e: " + why);
  const hipError_t err = mx::launch_cpml<true>(v, prec, psi_prec, dt, h, e, eps, eps_scalar, tab,
                                               reinterpret_cast<hipStream_t>(stream));
  return err == hipSuccess ? 0 : mx::set_error(std::string("mx_fdtd_cpml_e: ") + hipGetErrorString(err));
}

int mx_fdtd_cpml_h(const mx_fdtd_grid* g, int32_t prec, int32_t psi_prec, double dt, const void* e, void* h,
                   const void* mu, double mu_scalar, const mx_cpml_layer* layers, int32_t nlayers, void* stream) {
  mx::RGrid v;
  if (mx::check_args(g, prec, e, h, &v, "mx_fdtd_cpml_h")) return -1;
  if (psi_prec != MX_REAL32 && psi_prec != MX_REAL64) return mx::set_error("mx_fdtd_cpml_h: psi_prec must be MX_REAL32 or MX_REAL64");
  mx::CpmlTable tab;
  std::string why;
  if (!mx::cpml_table(v, layers, nlayers, false, &tab, &why)) return mx::set_error("mx_fdtd_cpml_h: " + why);
  const hipError_t err = mx::launch_cpml<false>(v, prec, psi_prec, dt, e, h, mu, mu_scalar, tab,
                                                reinterpret_cast<hipStream_t>(stream));
  return err == hipSuccess ? 0 : mx::set_error(std::string("mx_fdtd_cpml_h: ") + hipGetErrorString(err));
}

int mx_fdtd_conducting_boundary(const mx_fdtd_grid* g, int32_t prec, int32_t direction, int32_t polarity,
                                int32_t field, void* f, void* stream) {
  mx::RGrid v;
  if (mx::check_args(g, prec, f, f, &v, "mx_fdtd_conducting_boundary")) return -1;
  if (direction < 0 || direction > 2) return mx::set_error("mx_fdtd_conducting_boundary: direction must be 0, 1 or 2");
  if (polarity != -1 && polarity != 1) return mx::set_error("mx_fdtd_conducting_boundary: polarity must be -1 or +1");
  if (field != MX_FIELD_E && field != MX_FIELD_H)
    return mx::set_error("mx_fdtd_conducting_boundary: field must be MX_FIELD_E or MX_FIELD_H");
  const int dims[3] = {v.nx, v.ny, v.nz};
  if (dims[direction] < (polarity < 0 ? 2 : 3))
    return mx::set_error("mx_fdtd_conducting_boundary: the axis needs at least 2 cells (polarity -1) or 3 (+1)");
  const hipError_t err = mx::launch_conducting(v, prec, direction, polarity, field == MX_FIELD_H, f,
                                               reinterpret_cast<hipStream_t>(stream));
  return err == hipSuccess ? 0 : mx::set_error(std::string("mx_fdtd_conducting_boundary: ") + hipGetErrorString(err));
}

int mx_fdtd_energy(const mx_fdtd_grid* g, int32_t prec, int32_t form, double dt, const void* const* f,
                   const void* eps, double eps_scalar, const void* mu, double mu_scalar, double* out, void* stream) {
  static const int kNeeds[6] = {2, 3, 3, 4, 4, 2};   // fields each form reads
  mx::RGrid v;
  if (!f) return mx::set_error("mx_fdtd_energy: null field table");
  if (mx::check_args(g, prec, f[0], out, &v, "mx_fdtd_energy")) return -1;
  if (form < MX_ENERGY_DXMUL || form > MX_ENERGY_J) return mx::set_error("mx_fdtd_energy: unknown form");
  for (int q = 0; q < kNeeds[form]; ++q)
    if (!f[q]) return mx::set_error("mx_fdtd_energy: null field for this form");
  if ((form == MX_ENERGY_H2E || form == MX_ENERGY_E2H) && !(dt != 0.0)) return mx::set_error("mx_fdtd_energy: dt must be nonzero");
  const void* fs[4] = {f[0], f[1], kNeeds[form] > 2 ? f[2] : nullptr, kNeeds[form] > 3 ? f[3] : nullptr};
  const hipError_t err = mx::launch_energy(v, prec, form, dt, fs, eps, eps_scalar, mu, mu_scalar, out,
                                           reinterpret_cast<hipStream_t>(stream));
  return err == hipSuccess ? 0 : mx::set_error(std::string("mx_fdtd_energy: ") + hipGetErrorString(err));
}

int mx_fdtd_poynting(const mx_fdtd_grid* g, int32_t prec, const void* e, const void* h, void* s, void* stream) {
  mx::RGrid v;
  if (mx::check_args(g, prec, e, h, &v, "mx_fdtd_poynting")) return -1;
  if (!s) return mx::set_error("mx_fdtd_poynting: null output");
  const hipError_t err = mx::launch_poynting(v, prec, e, h, s, reinterpret_cast<hipStream_t>(stream));
  return err == hipSuccess ? 0 : mx::set_error(std::string("mx_fdtd_poynting: ") + hipGetErrorString(err));
}

int mx_fdtd_poynting_divergence(const mx_fdtd_grid* g, int32_t prec, const void* s, void* ds, void* stream) {
  mx::RGrid v;
  if (mx::check_args(g, prec, s, ds, &v, "mx_fdtd_poynting_divergence")) return -1;
  const hipError_t err = mx::launch_poynting_div(v, prec, s, ds, reinterpret_cast<hipStream_t>(stream));
  return err == hipSuccess ? 0 : mx::set_error(std::string("mx_fdtd_poynting_divergence: ") + hipGetErrorString(err));
}

}  // extern "C"
