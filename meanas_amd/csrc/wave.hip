// The unscaled wave operators as single passes over a field (complex128):
//
//   e_full (meanas/fdfd/operators.py:40-96):   y = pe (curl_b(pm / mu curl_f(pe x)) - w^2 eps pe x)
//   h_full (operators.py:126-180) through its reversed dual: with every cell index of x and
//     y reversed, h_full is e_full of the reversed grid with eps and mu, E and H widths and
//     the masks exchanged (the operator passed in is that dual one)
//   TFSF and boundary sources (operators.py:366-450):  y = c k (A0 (q x) - q (A0 x)), A0 =
//     e_full, q a real field (the region), k a real field or absent (the kept cells)
//
// The solver's symmetrised operator is A = P A0 P^-1; here the differences divide by the
// widths themselves, so no diagonal passes surround the product.
//
// A block is kRows waves: lanes are 64 consecutive z cells, rows consecutive y cells, one
// of each on every side being halo that the neighbouring blocks compute as well (indices
// wrap, so every lane holds a cell of the periodic grid).  It marches along x; per plane:
//   phase 1: H = pm / mu curl_f(E)     (E of plane i+1 from the thread's own loads)
//   phase 2: y = pe (curl_b(H) - w^2 eps E)
// with z neighbours from the next lane, y neighbours through LDS, x neighbours in
// registers, and the loads of a plane issued one plane ahead.
//
// HBM-bound (104 B a cell with real isotropic eps), in cache bound by the latency of a
// plane's two phases.  Through the symmetrised apply, A0 was two diagonal passes around it
// and a table upload, an allocation and two synchronisations per call.  112 x 98 x 121
// with permeability and metal: 57 us a call (152 through the apply); isotropic 30 us, 4.6
// TB/s; 160 x 150 x 160 isotropic 89 us.  A 96 x 80 x 90 boundary source 38 us (273 as two
// products with A0 and five array passes).  Rows (waves) per block, calls in us: 6/8/10/12
// rows isotropic 32/30/31/33, with permeability (154 VGPRs) 80/61/57/63, sources (180-232
// VGPRs) 48/38/57/54.
#include <algorithm>
#include <string>

#include "common.hpp"
#include "../../include/meanas_fdfd.h"

namespace mx {

int set_error(const std::string& msg);
bool wave_op(const mx_operator& op, OpView<double>* v, std::string* why);   // solver.hip

namespace {

constexpr int kMaxSlab = 64;

// complex value of the next / previous lane of the wave (DPP wave shifts; ends get 0)
template <int CTRL> __device__ __forceinline__ double lane_shift(double v) {
  typedef int __attribute__((ext_vector_type(2))) I2;
  const I2 w = __builtin_bit_cast(I2, v);
  I2 r;
  r.x = __builtin_amdgcn_update_dpp(0, w.x, CTRL, 0xf, 0xf, true);
  r.y = __builtin_amdgcn_update_dpp(0, w.y, CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, r);
}
typedef cplx<double> C;
__device__ __forceinline__ C lane_next(C v) { return C{lane_shift<0x130>(v.re), lane_shift<0x130>(v.im)}; }
__device__ __forceinline__ C lane_prev(C v) { return C{lane_shift<0x138>(v.re), lane_shift<0x138>(v.im)}; }

__device__ __forceinline__ int wrapw(int v, int n) {
  const int r = v % n;
  return r < 0 ? r + n : r;
}
__device__ __forceinline__ C inverse(C d) { return cdiv(C{1.0, 0.0}, d); }

struct Widths {
  const C* e[3];   // dxes[0], dxes[1]
  const C* h[3];
};

// F = 1: y = A0 x; F = 2: y = c k (A0 (q x) - q (A0 x)).  ROWS waves per block.
template <int F, int MK, int ROWS>
__global__ __launch_bounds__(64 * ROWS) void k_wave(OpView<double> op, Widths wd, const C* __restrict__ x,
                                                    C* __restrict__ y, const double* __restrict__ qf,
                                                    const double* __restrict__ kf, C cc, int rev, int slab) {
  constexpr int OY = ROWS - 2, OZ = 62;
  __shared__ C sE[F][2][ROWS + 1][64];   // E x, z by row
  __shared__ C sH[F][2][ROWS + 1][64];   // H x, z by row + 1
  __shared__ C sX[kMaxSlab + 2][2];      // 1 / dx_e, 1 / dx_h by plane
  const int nx = op.nx, ny = op.ny, nz = op.nz;
  const int plane = ny * nz, nc = nx * plane;
  const int ntj = (ny + OY - 1) / OY, ntk = (nz + OZ - 1) / OZ, tiles = ntj * ntk;
  const int nwork = ((nx + slab - 1) / slab) * tiles;
  // XCD w % 8 takes a contiguous run of work items (neighbouring tiles of a slab)
  const int per = (nwork + 7) / 8;
  const int w = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (w >= nwork) return;
  const int slab_id = w / tiles, tile = w - slab_id * tiles;
  const int j0 = (tile / ntk) * OY, k0 = (tile % ntk) * OZ;
  const int ib = slab_id * slab, ie = min(ib + slab, nx);
  const int tz = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int j = j0 + ty - 1, k = k0 + tz - 1;
  const bool valid = ty >= 1 && ty < ROWS - 1 && tz >= 1 && tz < 63 && j < ny && k < nz;
  const int jw = wrapw(j, ny), kw = wrapw(k, nz);
  const int own = jw * nz + kw;                                            // materials
  const int fown = rev ? (ny - 1 - jw) * nz + (nz - 1 - kw) : own;        // fields

  constexpr bool ISO = MK == MK_SIMPLE || MK == MK_MASK;
  const bool has_mask = MK == MK_MASK || (MK == MK_GENERAL && (op.flags & OPF_MASK) != 0);
  const bool has_mu = MK == MK_GENERAL && (op.flags & OPF_MU) != 0;

  const int first = ib - 1, nt = (ie - ib) + 1;   // planes first .. ie - 1
  for (int t = ty * 64 + tz; t < nt; t += 64 * ROWS) {
    const int n = wrapw(first + t, nx);
    sX[t][0] = inverse(wd.e[0][n]);
    sX[t][1] = inverse(wd.h[0][n]);
  }
  const C rye = inverse(wd.e[1][jw]), ryh = inverse(wd.h[1][jw]);
  const C rze = inverse(wd.e[2][kw]), rzh = inverse(wd.h[2][kw]);

  struct In { C e[3]; double q[3]; uint8_t m; };   // field, region and mask of a plane
  struct Mat { C eps[3], mu[3]; };                  // w^2 eps and 1 / mu of a plane
  auto fetch = [&](In& I, int p) {
    const int fp = (rev ? nx - 1 - p : p) * plane + fown, mp = p * plane + own;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      I.e[c] = gload<double>(x, c * nc + fp);
      if constexpr (F == 2) I.q[c] = gload1<double>(qf, c * nc + mp);
    }
    I.m = has_mask ? gload1<uint8_t>(op.mask, mp) : 0;
  };
  auto material = [&](const double* base, bool is_complex, bool aniso, int c, int cell) -> C {
    const int idx = aniso ? c * nc + cell : cell;
    return is_complex ? gload<double>(base, idx) : C{gload1<double>(base, idx), 0.0};
  };
  auto fetch_mat = [&](Mat& M, int p) {
    const int cell = p * plane + own;
    if constexpr (ISO) {
      M.eps[0] = material(op.eps, false, false, 0, cell);
    } else {
#pragma unroll
      for (int c = 0; c < 3; ++c)
        M.eps[c] = MK == MK_ANISO ? material(op.eps, false, true, c, cell)
                                  : material(op.eps, op.flags & OPF_EPS_COMPLEX, op.flags & OPF_EPS_ANISO, c, cell);
    }
    if (has_mu) {
#pragma unroll
      for (int c = 0; c < 3; ++c)
        M.mu[c] = material(op.inv_mu, op.flags & OPF_MU_COMPLEX, op.flags & OPF_MU_ANISO, c, cell);
    }
  };
  // the unknown: the field (times q), zero on PEC components
  auto unknown = [&](const In& I, int f, int c) -> C {
    if ((I.m >> c) & 1) return zero<double>();
    return F == 2 && f == 0 ? I.q[c] * I.e[c] : I.e[c];
  };

  In A, B;
  Mat M;
  C Ec[F][3], H1[F][3];   // E of plane i; H of plane i - 1
  uint8_t mc;             // mask and region of plane i
  double qc[3];
  auto take = [&](const In& I) {
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
      for (int c = 0; c < 3; ++c) Ec[f][c] = unknown(I, f, c);
    mc = I.m;
    if constexpr (F == 2) {
#pragma unroll
      for (int c = 0; c < 3; ++c) qc[c] = I.q[c];
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
      sE[f][0][ty][tz] = Ec[f][0];
      sE[f][1][ty][tz] = Ec[f][2];
    }
  };
  int p = wrapw(first, nx);
  auto next = [&](int v) { return v + 1 == nx ? 0 : v + 1; };
  fetch(A, p);
  fetch_mat(M, p);
  // rows that no wave writes, read only for halo values that are never used
  if (ty == 0) {
#pragma unroll
    for (int f = 0; f < F; ++f)
      sE[f][0][ROWS][tz] = sE[f][1][ROWS][tz] = sH[f][0][0][tz] = sH[f][1][0][tz] = zero<double>();
  }
#pragma unroll
  for (int f = 0; f < F; ++f)
#pragma unroll
    for (int c = 0; c < 3; ++c) H1[f][c] = zero<double>();
  take(A);
  fetch(A, next(p));
  __syncthreads();

  auto step = [&](const int t, In& cur, In& nxt) {
    const int p1 = next(p);
    Mat Mn;
    fetch(nxt, next(p1));
    fetch_mat(Mn, p1);
    const C rx = sX[t][0], rxh = sX[t][1];
    C hs[F][3];
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const C (&ec)[3] = Ec[f];
      const C en1 = unknown(cur, f, 1), en2 = unknown(cur, f, 2);
      const C ex_y = sE[f][0][ty + 1][tz], ez_y = sE[f][1][ty + 1][tz];
      const C ex_z = lane_next(ec[0]), ey_z = lane_next(ec[1]);
      hs[f][0] = rye * (ez_y - ec[2]) - rze * (ey_z - ec[1]);
      hs[f][1] = rze * (ex_z - ec[0]) - rx * (en2 - ec[2]);
      hs[f][2] = rx * (en1 - ec[1]) - rye * (ex_y - ec[0]);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if (has_mu) hs[f][c] = M.mu[c] * hs[f][c];
        if ((mc >> (3 + c)) & 1) hs[f][c] = zero<double>();
      }
      sH[f][0][ty + 1][tz] = hs[f][0];
      sH[f][1][ty + 1][tz] = hs[f][2];
    }
    __syncthreads();
    C o[F][3];
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const C hx = hs[f][0], hy = hs[f][1], hz = hs[f][2];
      const C hx_y = sH[f][0][ty][tz], hz_y = sH[f][1][ty][tz];
      const C hx_z = lane_prev(hx), hy_z = lane_prev(hy);
      o[f][0] = ryh * (hz - hz_y) - rzh * (hy - hy_z);
      o[f][1] = rzh * (hx - hx_z) - rxh * (hz - H1[f][2]);
      o[f][2] = rxh * (hy - H1[f][1]) - ryh * (hx - hx_y);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        o[f][c] = o[f][c] - op.w2 * (M.eps[ISO ? 0 : c] * Ec[f][c]);
        if ((mc >> c) & 1) o[f][c] = zero<double>();
        H1[f][c] = hs[f][c];
      }
    }
    if (valid && t > 0) {
      const int fp = (rev ? nx - 1 - p : p) * plane + fown, mp = p * plane + own;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if constexpr (F == 2) {
          C v = cc * (o[0][c] - qc[c] * o[1][c]);
          if (kf) v = gload1<double>(kf, c * nc + mp) * v;
          gstore<double>(y, c * nc + fp, v);
        } else {
          gstore<double>(y, c * nc + fp, o[0][c]);
        }
      }
    }
    take(cur);
    M = Mn;
    p = p1;
    // the barrier ends the step, in straight line with the LDS writes (k_fdtd_steps, fdtd.hip,
    // says why)
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

// Slab depth with the least modelled time: a block takes slab + 1 planes, and a CU's n
// blocks share it.
int wave_slab(const OpView<double>& v, int rows) {
  const long long tiles = (long long)((v.ny + rows - 3) / (rows - 2)) * ((v.nz + 61) / 62);
  int best = 1;
  double best_cost = 0.0;
  for (int want : {2, 3, 4, 6, 8, 12, 16, 24, 32, kMaxSlab}) {
    const int slab = std::min(want, v.nx);
    const long long blocks = tiles * ((v.nx + slab - 1) / slab);
    const double cost = ((double)((blocks + 255) / 256) + 0.3) * (slab + 2);
    if (best_cost == 0.0 || cost < best_cost) {
      best_cost = cost;
      best = slab;
    }
  }
  return best;
}

template <int F>
hipError_t launch_wave(const OpView<double>& v, const Widths& wd, const void* x, void* y, const double* q, const double* k,
                       C c, int rev, hipStream_t s) {
  const int kind = mat_kind(v.flags);
  const int rows = F == 1 && kind == MK_GENERAL ? 10 : 8;
  const int slab = wave_slab(v, rows);
  const long long tiles = (long long)((v.ny + rows - 3) / (rows - 2)) * ((v.nz + 61) / 62);
  const long long nwork = tiles * ((v.nx + slab - 1) / slab);
  const unsigned nb = (unsigned)((nwork + 7) / 8 * 8);
#define MX_WAVE_CASE(MK)                                                                                              \
  case MK: {                                                                                                          \
    constexpr int R = F == 1 && MK == MK_GENERAL ? 10 : 8;                                                            \
    hipLaunchKernelGGL((k_wave<F, MK, R>), dim3(nb), dim3(64, R), 0, s, v, wd, (const C*)x, (C*)y, q, k, c, rev, slab); \
    break;                                                                                                            \
  }
  switch (kind) {
    MX_WAVE_CASE(MK_SIMPLE)
    MX_WAVE_CASE(MK_ANISO)
    MX_WAVE_CASE(MK_MASK)
    MX_WAVE_CASE(MK_GENERAL)
  }
#undef MX_WAVE_CASE
  return hipGetLastError();
}

}  // namespace
}  // namespace mx

extern "C" {

int mx_wave(const mx_operator* op, const mx_grid* g, int32_t reversed, const void* x, void* y, void* stream) {
  using namespace mx;
  OpView<double> v;
  std::string why;
  if (!op || !g || !x || !y) return set_error("mx_wave: null argument");
  if (!wave_op(*op, &v, &why)) return set_error("mx_wave: " + why);
  if (g->nx != op->nx || g->ny != op->ny || g->nz != op->nz) return set_error("mx_wave: grid and operator differ");
  Widths wd;
  for (int a = 0; a < 3; ++a) {
    if (!g->dxe[a] || !g->dxh[a]) return set_error("mx_wave: missing cell widths");
    wd.e[a] = (const C*)g->dxe[a];
    wd.h[a] = (const C*)g->dxh[a];
  }
  const hipError_t e = launch_wave<1>(v, wd, x, y, nullptr, nullptr, C{1.0, 0.0}, reversed ? 1 : 0,
                                          reinterpret_cast<hipStream_t>(stream));
  return e == hipSuccess ? 0 : set_error(std::string("mx_wave: ") + hipGetErrorString(e));
}

int mx_wave_source(const mx_operator* op, const mx_grid* g, const double* region, const double* keep, double c_re,
                   double c_im, const void* x, void* y, void* stream) {
  using namespace mx;
  OpView<double> v;
  std::string why;
  if (!op || !g || !region || !x || !y) return set_error("mx_wave_source: null argument");
  if (!wave_op(*op, &v, &why)) return set_error("mx_wave_source: " + why);
  if (g->nx != op->nx || g->ny != op->ny || g->nz != op->nz) return set_error("mx_wave_source: grid and operator differ");
  Widths wd;
  for (int a = 0; a < 3; ++a) {
    if (!g->dxe[a] || !g->dxh[a]) return set_error("mx_wave_source: missing cell widths");
    wd.e[a] = (const C*)g->dxe[a];
    wd.h[a] = (const C*)g->dxh[a];
  }
  const hipError_t e = launch_wave<2>(v, wd, x, y, region, keep, C{c_re, c_im}, 0,
                                         reinterpret_cast<hipStream_t>(stream));
  return e == hipSuccess ? 0 : set_error(std::string("mx_wave_source: ") + hipGetErrorString(e));
}

}  // extern "C"
