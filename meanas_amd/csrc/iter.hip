// One-launch COCG iteration for small systems (fused form, complex128).
//
// The fused iteration of vector.hip is three launches (apply, one finishing block per
// system, update); on a small grid each is a few microseconds of latency -- launch, table
// and state loads, one pass in cache -- whatever the size.  Here one launch does all of it:
//   k_iter : every block sums the partials of the launch before and advances a private copy
//            of the scalar state (alpha, beta, checks: fin_update_state, fin_apply_state);
//            r' = r - alpha q, p' = r' + beta p on its tile and a one-cell halo, x_lo on its
//            tile; q' = A p' on its tile; partials of p'^T q', q'^T q', r'^T r', ||r'||^2.
// The halo's r' and p' are computed again by every block that needs them, from the same
// values by the same expressions, so nothing has to be exchanged inside the launch.  No
// block may read what another of the same launch writes, so r, p, q, the state and the
// partials alternate between two copies from launch to launch (`par`: the copy read).  A
// run of launches starts with everything in the first copies.  A system that pauses stays
// where it is (SF_ALT: its r and p are in the second buffers) and later launches only copy
// its state forward; its residual replacement brings r and p back to the first.
//   k_iter<INIT> : q = A p and its partials at the start of a run of launches, for systems
//                  whose q does not belong to their p (SF_QVALID clear: the first run, after a
//                  residual replacement);
//   k_iter_fin   : after the run, the last update's checks; the state returns to its first
//                  copy, where replacements and the host find it (after an odd number of
//                  launches k_iter_back copies r and p back as well).
// What bounds it: below about 100 tiles the chain of latencies inside the launch (state and
// partials, sums, scalars, fields, three barriers); above, issue (about 800 vector
// instructions a wave) and LDS at the four waves a SIMD that the 120 registers allow, and
// the cache traffic of r, p, q with their halos (64^3: 390 B a cell through L2, 5.6 TB/s).
// Microseconds per iteration of one system, against the three launches: 16^3 10.7 / 22.7,
// 28x24x33 12.8 / 23.5, 44x40x36 with PEC 13.6 / 26.9, 48^3 14.4 / 29.8.  What was tried:
// H = curl p kept in LDS instead of evaluated at each neighbour (9 to 3.75 evaluations a
// cell) and sums taken by one wave each through LDS instead of seven wave sums in every wave
// gave 15 %; several tiles per block 35 % slower (the loads of a tile wait for the tile
// before), nontemporal stores 10 to 20 % slower (the next launch finds the lines in L2).
// The scalar state evolves as with the three launches; the sums are taken in another
// order (by these tiles), so the two forms agree to rounding, not bit for bit.  Which form a
// system uses depends on its own grid alone.
#include <string>

#include "cocg_state.hpp"
#include "common.hpp"

namespace mx {

namespace {

constexpr int kT = 8;                       // tile edge: 8 x 8 x 8 cells, one per thread
constexpr int kH = kT + 2;                  // with its halo
constexpr int kH1 = kT + 1;
constexpr int kHalo = kH * kH * kH;
constexpr int kThreads = kT * kT * kT;
constexpr int kShell = kHalo - kThreads;    // halo cells: one each for the first 488 threads
static_assert(kShell <= kThreads, "a thread takes at most one halo cell");
constexpr int kSums = 7;                    // r'r' re, im, ||r||^2; p'q re, im; q'q re, im
constexpr int kWords = (int)(sizeof(SysState) / 8);
static_assert(kWords <= 64, "state words: one per lane of a wave");

typedef cplx<double> C;

// What a block needs to know about its system: from the kernel's arguments if the launch
// has one system, else from the tables.  (Each dependent load costs about a microsecond
// here: a kernel starts with cold L1 and L2 lines of what the launch before wrote.)
struct IterDesc {
  OpView<double> op;
  C *ra, *rb, *pa, *pb, *qa, *qb, *xl;   // first and second copies
  SysState *sa, *sb;
  double *ta, *tb;
  int nblk;
};
__host__ __device__ __forceinline__ IterDesc iter_desc(const SysDesc& S, const OpView<double>& op) {
  return IterDesc{op, (C*)S.vec[VS_R], (C*)S.vec[VS_R2], (C*)S.vec[VS_P], (C*)S.vec[VS_P2], (C*)S.vec[VS_Q],
                  (C*)S.vec[VS_Q2], (C*)S.vec[VS_XLO], S.st, S.st2, S.part_it[0], S.part_it[1], S.nblk_iter};
}

// Sum over the wave with DPP: shifts within rows of 16 lanes, then the two row broadcasts.
template <int CTRL, int ROWS> __device__ __forceinline__ double dpp_add(double v) {
  typedef int __attribute__((ext_vector_type(2))) I2;
  const I2 w = __builtin_bit_cast(I2, v);
  I2 r;
  r.x = __builtin_amdgcn_update_dpp(0, w.x, CTRL, ROWS, 0xf, false);
  r.y = __builtin_amdgcn_update_dpp(0, w.y, CTRL, ROWS, 0xf, false);
  return v + __builtin_bit_cast(double, r);
}
__device__ __forceinline__ double wave_total(double v) {   // valid in lane 63
  v = dpp_add<0x111, 0xf>(v);   // row_shr:1
  v = dpp_add<0x112, 0xf>(v);   // row_shr:2
  v = dpp_add<0x114, 0xf>(v);   // row_shr:4
  v = dpp_add<0x118, 0xf>(v);   // row_shr:8
  v = dpp_add<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
  return dpp_add<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
}
// This lane's share of the sum of `n` values, lane 0 to 63 in turn.  Eight loads are in
// flight together, those past the end at the last value and not counted.
__device__ __forceinline__ double lane_share(const double* v, int n, int lane) {
  double t = 0.0;
  for (int b = lane; b < n; b += 512) {
    double w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = gload1<double>(v, min(b + 64 * k, n - 1));
#pragma unroll
    for (int k = 0; k < 8; ++k) t += b + 64 * k < n ? w[k] : 0.0;
  }
  return t;
}

// coordinate base - 1 + h of a periodic axis of n cells (0 <= base < n, 0 <= h < kH)
__device__ __forceinline__ int halo_coord(int base, int h, int n) {
  int v = base - 1 + h;
  if (n >= kH) {
    v += v < 0 ? n : 0;
    return v >= n ? v - n : v;
  }
  v %= n;
  return v < 0 ? v + n : v;
}

template <int MK, bool INIT, bool ONE>
__global__ __launch_bounds__(kThreads, 4) void k_iter(IterDesc one, const OpView<double>* __restrict__ ops,
                                                      const SysDesc* __restrict__ systems,
                                                      const BlockMap* __restrict__ bmap, int par) {
  __shared__ C sP[3][kHalo];                 // p' of the tile and its halo, zero on PEC
  __shared__ C sH[3][kT * kH1 * kH1];        // curl p' on the tile and the cells before it
  __shared__ uint8_t sM[kHalo];              // mask bits
  __shared__ FaFb<double> sC[3][kH];         // forward-difference coefficients by axis
  __shared__ double s_red[kSums];
  __shared__ SysState s_st;
  const int tid = threadIdx.x;
  IterDesc D;
  int local;
  if constexpr (ONE) {
    D = one;
    // XCD x (block % 8) takes a contiguous run of tiles
    const int n = D.nblk, x = blockIdx.x % 8;
    local = n / 8 * x + min(x, n % 8) + (int)(blockIdx.x / 8);
  } else {
    const BlockMap bm = bmap[blockIdx.x];
    const SysDesc& S = systems[bm.sys];
    D = iter_desc(S, ops[S.op]);
    local = bm.local;
  }
  const int nblk = D.nblk;
  const SysState* const gst = par ? D.sb : D.sa;
  SysState* const gst_to = par ? D.sa : D.sb;
  const double* const part = par ? D.tb : D.ta;
  unsigned long long word = 0;
  if (tid < kWords) word = reinterpret_cast<const unsigned long long*>(gst)[tid];
  const int f0 = gload1<int>(&gst->flags, 0);
  // partial sums of the launch before: loaded ahead of the fields, so that waiting for them
  // does not wait for those
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double share = 0.0;   // wave q takes sum q
  if constexpr (!INIT) {
    if (wave < kSums) share = lane_share(part + wave * nblk, nblk, lane);
  }

  const OpView<double>& op = D.op;
  const int nx = op.nx, ny = op.ny, nz = op.nz;
  const int nc = nx * ny * nz;
  const int nty = (ny + kT - 1) / kT, ntz = (nz + kT - 1) / kT;
  const int x0 = local / (nty * ntz) * kT, tile = local % (nty * ntz);
  const int y0 = tile / ntz * kT, z0 = tile % ntz * kT;
  constexpr bool ISO = MK == MK_SIMPLE || MK == MK_MASK;
  const bool has_mask = MK == MK_MASK || (MK == MK_GENERAL && (op.flags & OPF_MASK) != 0);
  const bool has_mu = MK == MK_GENERAL && (op.flags & OPF_MU) != 0;

  const int to = INIT ? par : 1 - par;       // the copies this launch writes
  const C* __restrict__ r0 = par ? D.rb : D.ra;
  const C* __restrict__ p0 = par ? D.pb : D.pa;
  const C* __restrict__ q0 = par ? D.qb : D.qa;
  C* __restrict__ r1 = to ? D.rb : D.ra;
  C* __restrict__ p1 = to ? D.pb : D.pa;
  C* __restrict__ q1 = to ? D.qb : D.qa;
  C* __restrict__ xl = D.xl;

  // this thread's own cell and its halo cell: the x faces, then the y faces and the z faces
  // of the remaining block
  const int lx = tid / (kT * kT), ly = tid / kT % kT, lz = tid % kT;
  const bool own = x0 + lx < nx && y0 + ly < ny && z0 + lz < nz;
  const int ocell = (halo_coord(x0, lx + 1, nx) * ny + halo_coord(y0, ly + 1, ny)) * nz + halo_coord(z0, lz + 1, nz);
  constexpr int DX = kH * kH, DY = kH, DZ = 1;
  const int on = (lx + 1) * DX + (ly + 1) * DY + lz + 1;
  int sx, sy, sz;
  if (tid < 2 * DX) {
    sx = tid < DX ? 0 : kH - 1;
    const int v = tid < DX ? tid : tid - DX;
    sy = v / kH;
    sz = v % kH;
  } else if (tid < 2 * DX + 2 * kT * kH) {
    const int v = tid - 2 * DX, w = v % (kT * kH);
    sy = v < kT * kH ? 0 : kH - 1;
    sx = 1 + w / kH;
    sz = w % kH;
  } else {
    const int v = tid - 2 * DX - 2 * kT * kH, w = v % (kT * kT);
    sz = v < kT * kT ? 0 : kH - 1;
    sx = 1 + w / kT;
    sy = 1 + w % kT;
  }
  const bool shell = tid < kShell;
  const int scell = shell ? (halo_coord(x0, sx, nx) * ny + halo_coord(y0, sy, ny)) * nz + halo_coord(z0, sz, nz) : ocell;
  const int sn = shell ? sx * DX + sy * DY + sz : 0;
  C ro[3], po[3], qo[3], rs[3], ps[3], qs[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    po[c] = gload<double>(p0, c * nc + ocell);
    if constexpr (!INIT) {
      ro[c] = gload<double>(r0, c * nc + ocell);
      qo[c] = gload<double>(q0, c * nc + ocell);
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    ps[c] = gload<double>(p0, c * nc + scell);
    if constexpr (!INIT) {
      rs[c] = gload<double>(r0, c * nc + scell);
      qs[c] = gload<double>(q0, c * nc + scell);
    }
  }
  const uint8_t mo = has_mask ? gload1<uint8_t>(op.mask, ocell) : 0, ms = has_mask ? gload1<uint8_t>(op.mask, scell) : 0;
  // eps of the own cell; coefficients of the tile's planes
  auto material = [&](const double* base, bool is_complex, bool aniso, int c, int at) -> C {
    const int idx = aniso ? c * nc + at : at;
    return is_complex ? gload<double>(base, idx) : C{gload1<double>(base, idx), 0.0};
  };
  if (tid < 3 * kH) {
    const int a = tid / kH, h = tid % kH;
    const int base = a == 0 ? x0 : a == 1 ? y0 : z0, n = a == 0 ? nx : a == 1 ? ny : nz;
    const AxisCoef<double>* tab = op.coef + (a == 0 ? 0 : a == 1 ? nx : nx + ny);
    sC[a][h] = coef_at(tab, halo_coord(base, h, n));
  }

  // systems that are not running: carry the state over
  const bool runnable = !(f0 & (SF_PAUSE | SF_DONE | SF_INACTIVE));
  if (INIT && (!runnable || (f0 & SF_QVALID))) return;
  if (!runnable) {
    if (local == 0 && tid < kWords) reinterpret_cast<unsigned long long*>(gst_to)[tid] = word;
    return;
  }
  // the scalar state: every block forms the same one
  if (tid < kWords) reinterpret_cast<unsigned long long*>(&s_st)[tid] = word;
  if constexpr (!INIT) {
    if (wave < kSums) {
      share = wave_total(share);
      if (lane == 63) s_red[wave] = share;
    }
    __syncthreads();
    if (tid == 0) {
      int f = f0;
      const double tu[3] = {s_red[0], s_red[1], s_red[2]};
      const double ta[4] = {s_red[3], s_red[4], s_red[5], s_red[6]};
      if (f & SF_UPD_PENDING) fin_update_state(&s_st, f, tu, true);
      if (!(f & SF_PAUSE)) fin_apply_state(&s_st, f, ta, true);
      if (!(f & SF_PAUSE)) f |= SF_QVALID;
      else if (par) f |= SF_ALT;
      s_st.flags = f;
    }
  }
  __syncthreads();
  const int f = s_st.flags;
  if constexpr (!INIT) {
    if (local == 0 && tid < kWords)
      reinterpret_cast<unsigned long long*>(gst_to)[tid] = reinterpret_cast<unsigned long long*>(&s_st)[tid];
    if (f & SF_PAUSE) return;
  }

  // ---- r' = r - alpha q, p' = r' + beta p; x_lo += xc1 p + xc2 r
  const C alpha = s_st.alpha, beta = s_st.beta;
  double acc[kSums] = {};
  if constexpr (!INIT) {
    if (own && !(f & SF_XSKIP)) {
      const C xc1 = s_st.xc1, xc2 = s_st.xc2;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int e = c * nc + ocell;
        gstore<double>(xl, e, gload<double>(xl, e) + xc1 * po[c] + xc2 * ro[c]);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    C pn = po[c];
    if constexpr (!INIT) {
      const C rn = ro[c] - alpha * qo[c];
      pn = rn + beta * po[c];
      if (own) {
        const int e = c * nc + ocell;
        gstore<double>(r1, e, rn);
        gstore<double>(p1, e, pn);
        acc[0] += rn.re * rn.re - rn.im * rn.im;
        acc[1] += 2.0 * rn.re * rn.im;
        acc[2] += rn.re * rn.re + rn.im * rn.im;
      }
    }
    po[c] = (mo >> c) & 1 ? zero<double>() : pn;   // the unknown is zero on PEC components
    sP[c][on] = po[c];
  }
  if (has_mask) sM[on] = mo;
  if (shell) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      C pn = ps[c];
      if constexpr (!INIT) pn = rs[c] - alpha * qs[c] + beta * ps[c];
      sP[c][sn] = (ms >> c) & 1 ? zero<double>() : pn;
    }
    if (has_mask) sM[sn] = ms;
  }
  C eps[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (ISO) eps[c] = c == 0 ? material(op.eps, false, false, 0, ocell) : eps[0];
    else if (MK == MK_ANISO) eps[c] = material(op.eps, false, true, c, ocell);
    else eps[c] = material(op.eps, op.flags & OPF_EPS_COMPLEX, op.flags & OPF_EPS_ANISO, c, ocell);
  }
  __syncthreads();

  // ---- H = curl p' / mu at the own cell, and by the first three waves at the cells before
  // the tile's x, y and z faces
  const FaFb<double> cx = sC[0][lx + 1], cy = sC[1][ly + 1], cz = sC[2][lz + 1];
  // component c of the H at halo position `at` = (hx, hy, hz)
  auto h_at = [&](int c, int at, const FaFb<double>& x, const FaFb<double>& y, const FaFb<double>& z, int px, int py,
                  int pz) -> C {
    auto e = [&](int k, int i) { return sP[k][i]; };
    C h = c == 0   ? dif(y.fa, e(2, at + DY), y.fb, e(2, at)) - dif(z.fa, e(1, at + DZ), z.fb, e(1, at))
          : c == 1 ? dif(z.fa, e(0, at + DZ), z.fb, e(0, at)) - dif(x.fa, e(2, at + DX), x.fb, e(2, at))
                   : dif(x.fa, e(1, at + DX), x.fb, e(1, at)) - dif(y.fa, e(0, at + DY), y.fb, e(0, at));
    if (has_mu) {
      const int g = (halo_coord(x0, px, nx) * ny + halo_coord(y0, py, ny)) * nz + halo_coord(z0, pz, nz);
      h = material(op.inv_mu, op.flags & OPF_MU_COMPLEX, op.flags & OPF_MU_ANISO, c, g) * h;
    }
    return has_mask && ((sM[at] >> (3 + c)) & 1) ? zero<double>() : h;
  };
  // where H lives in sH: cell (ix, iy, iz) of the tile, -1 before a face
  const auto ix0 = [](int ix, int iy, int iz) { return (ix * kH1 + iy + 1) * kH1 + iz + 1; };
  const auto ix1 = [](int ix, int iy, int iz) { return ((ix + 1) * kT + iy) * kH1 + iz + 1; };
  const auto ix2 = [](int ix, int iy, int iz) { return ((ix + 1) * kH1 + iy + 1) * kT + iz; };
  C out[3];
  {
    const C h0 = h_at(0, on, cx, cy, cz, lx + 1, ly + 1, lz + 1);
    const C h1 = h_at(1, on, cx, cy, cz, lx + 1, ly + 1, lz + 1);
    const C h2 = h_at(2, on, cx, cy, cz, lx + 1, ly + 1, lz + 1);
    sH[0][ix0(lx, ly, lz)] = h0;
    sH[1][ix1(lx, ly, lz)] = h1;
    sH[2][ix2(lx, ly, lz)] = h2;
    out[0] = cy.fb * h2 - cz.fb * h1;
    out[1] = cz.fb * h0 - cx.fb * h2;
    out[2] = cx.fb * h1 - cy.fb * h0;
  }
  if (wave < 3) {
    const int a = lane / kT, b = lane % kT;
    if (wave == 0) {
      const int at = (a + 1) * DY + b + 1;
      sH[1][ix1(-1, a, b)] = h_at(1, at, sC[0][0], sC[1][a + 1], sC[2][b + 1], 0, a + 1, b + 1);
      sH[2][ix2(-1, a, b)] = h_at(2, at, sC[0][0], sC[1][a + 1], sC[2][b + 1], 0, a + 1, b + 1);
    } else if (wave == 1) {
      const int at = (a + 1) * DX + b + 1;
      sH[0][ix0(a, -1, b)] = h_at(0, at, sC[0][a + 1], sC[1][0], sC[2][b + 1], a + 1, 0, b + 1);
      sH[2][ix2(a, -1, b)] = h_at(2, at, sC[0][a + 1], sC[1][0], sC[2][b + 1], a + 1, 0, b + 1);
    } else {
      const int at = (a + 1) * DX + (b + 1) * DY;
      sH[0][ix0(a, b, -1)] = h_at(0, at, sC[0][a + 1], sC[1][b + 1], sC[2][0], a + 1, b + 1, 0);
      sH[1][ix1(a, b, -1)] = h_at(1, at, sC[0][a + 1], sC[1][b + 1], sC[2][0], a + 1, b + 1, 0);
    }
  }
  __syncthreads();

  // ---- q' = A p' at the own cell
  if (own) {
    const C mx = sC[0][lx].fa, my = sC[1][ly].fa, mz = sC[2][lz].fa;
    out[0] = out[0] - my * sH[2][ix2(lx, ly - 1, lz)] + mz * sH[1][ix1(lx, ly, lz - 1)];
    out[1] = out[1] + mx * sH[2][ix2(lx - 1, ly, lz)] - mz * sH[0][ix0(lx, ly, lz - 1)];
    out[2] = out[2] - mx * sH[1][ix1(lx - 1, ly, lz)] + my * sH[0][ix0(lx, ly - 1, lz)];
    const bool mr = INIT && (f & SF_MR) != 0;   // rescue step: ||q||^2 instead of p^T q, q^T q
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const C ec = po[c];
      out[c] = out[c] - op.w2 * (eps[c] * ec);
      if ((mo >> c) & 1) out[c] = zero<double>();
      gstore<double>(q1, c * nc + ocell, out[c]);
      if (mr) {
        acc[5] += norm2(out[c]);
      } else {
        const C pq = ec * out[c], qq = out[c] * out[c];
        acc[3] += pq.re;
        acc[4] += pq.im;
        acc[5] += qq.re;
        acc[6] += qq.im;
      }
    }
  }
  // the tile's sums, through LDS (over sP, which nobody reads any more): wave q takes sum q
  double* const s_acc = reinterpret_cast<double*>(&sP[0][0]);
#pragma unroll
  for (int q = 0; q < kSums; ++q) s_acc[q * kThreads + tid] = acc[q];
  __syncthreads();
  if (wave < kSums) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < kThreads / 64; ++k) t += s_acc[wave * kThreads + 64 * k + lane];
    t = wave_total(t);
    if (lane == 63) ((MX_GLOBAL double*)(to ? D.tb : D.ta))[wave * nblk + local] = t;
  }
}

// After a run of launches (the state and partials in copy `par`): the last update's checks;
// the state back to its first copy.
__global__ __launch_bounds__(kThreads) void k_iter_fin(const SysDesc* __restrict__ systems,
                                                       const int* __restrict__ syslist, int par) {
  __shared__ double s_red[3];
  __shared__ SysState s_st;
  const SysDesc& S = systems[syslist[blockIdx.x]];
  const int tid = threadIdx.x, nblk = S.nblk_iter;
  if (tid < kWords)
    reinterpret_cast<unsigned long long*>(&s_st)[tid] = reinterpret_cast<const unsigned long long*>(par ? S.st2 : S.st)[tid];
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (wave < 3) {
    const double t = wave_total(lane_share(S.part_it[par] + wave * nblk, nblk, lane));
    if (lane == 63) s_red[wave] = t;
  }
  __syncthreads();
  if (tid == 0) {
    SysState st = s_st;
    int f = st.flags;
    const double tu[3] = {s_red[0], s_red[1], s_red[2]};
    const bool running = !(f & (SF_PAUSE | SF_DONE | SF_INACTIVE));
    if (running && (f & SF_UPD_PENDING)) fin_update_state(&st, f, tu, true);
    if (par && running) {
      f &= ~SF_QVALID;                     // q and its sums are in the second copies
      if (f & SF_PAUSE) f |= SF_ALT;       // so are r and p (k_iter_back copies those of a running system)
    }
    st.flags = f;
    s_st = st;
  }
  __syncthreads();
  if (tid < kWords)
    reinterpret_cast<unsigned long long*>(S.st)[tid] = reinterpret_cast<unsigned long long*>(&s_st)[tid];
}

// r and p of the running systems from their second buffers to the first
__global__ __launch_bounds__(kThreads) void k_iter_back(const SysDesc* __restrict__ systems,
                                                        const BlockMap* __restrict__ bmap) {
  const BlockMap bm = bmap[blockIdx.x];
  const SysDesc& S = systems[bm.sys];
  if (gload1<int>(&S.st->flags, 0) & (SF_PAUSE | SF_DONE | SF_INACTIVE)) return;
  const long long stride = (long long)S.nblk_iter * kThreads;
  for (long long e = (long long)bm.local * kThreads + threadIdx.x; e < S.n3; e += stride) {
    gstore<double>(S.vec[VS_R], (int)e, gload<double>(S.vec[VS_R2], (int)e));
    gstore<double>(S.vec[VS_P], (int)e, gload<double>(S.vec[VS_P2], (int)e));
  }
}

template <bool INIT>
hipError_t launch(int kind, const IterDesc* one, const OpView<double>* ops, const SysDesc* sys, const BlockMap* bmap, int nb,
                  int par, hipStream_t s) {
  static const IterDesc none{};
#define MX_ITER_CASE(MK)                                                                                         \
  case MK:                                                                                                       \
    if (one) hipLaunchKernelGGL((k_iter<MK, INIT, true>), dim3(nb), dim3(kThreads), 0, s, *one, ops, sys, bmap, par); \
    else hipLaunchKernelGGL((k_iter<MK, INIT, false>), dim3(nb), dim3(kThreads), 0, s, none, ops, sys, bmap, par);   \
    break;
  switch (kind) {
    MX_ITER_CASE(MK_SIMPLE)
    MX_ITER_CASE(MK_ANISO)
    MX_ITER_CASE(MK_MASK)
    default: MX_ITER_CASE(MK_GENERAL)
  }
#undef MX_ITER_CASE
  return hipGetLastError();
}

}  // namespace

int iter_blocks(int nx, int ny, int nz) {
  return ((nx + kT - 1) / kT) * ((ny + kT - 1) / kT) * ((nz + kT - 1) / kT);
}

// `n` iterations of the systems in bmap and syslist, ready for a residual replacement;
// one_sys and one_op describe the system if there is only one (else null)
hipError_t launch_iterations(int kind, const SysDesc* one_sys, const OpView<double>* one_op, const OpView<double>* ops,
                             const SysDesc* sys, const BlockMap* bmap, int nb, const int* syslist, int nsys, int n,
                             hipStream_t s) {
  if (nb <= 0 || n <= 0) return hipSuccess;
  IterDesc d;
  const IterDesc* one = nullptr;
  if (one_sys && one_op && one_sys->nblk_iter == nb) {
    d = iter_desc(*one_sys, *one_op);
    one = &d;
  }
  hipError_t e = launch<true>(kind, one, ops, sys, bmap, nb, 0, s);
  for (int i = 0; i < n && e == hipSuccess; ++i) e = launch<false>(kind, one, ops, sys, bmap, nb, i & 1, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_iter_fin, dim3(nsys), dim3(kThreads), 0, s, sys, syslist, n & 1);
  if (n & 1) hipLaunchKernelGGL(k_iter_back, dim3(nb), dim3(kThreads), 0, s, sys, bmap);
  return hipGetLastError();
}

}  // namespace mx
