// cells.hip — one RK substep's right-hand side and update of a field without shocked faces or
// order-reduced boundaries, cell by cell.
//
// The difference of a cell's two KEEP face fluxes telescopes: with G(a, b) the symmetric pair
// term of the split form (kernels_gpu.F90:150-337),
//   F(c) - F(c-1) = sum_l c_l [ G(c, c+l) - G(c-l, c) ],
// so a cell needs its own six pairs per direction and no face flux of a neighbour.  The pair
// factors P = +-c_l/4 dxi (rho_c + rho_n)(un_c + un_n) do not depend on the advected variable:
// a species' convective term in all three directions is sum_n P_n (Y_c + Y_n) over 18
// neighbours.  Three kernels:
//   cell_momentum_kernel   momentum and the energy but for the enthalpy flux: KEEP pairs,
//     staggered viscous faces (visflx_{x,y,z}_cuf, :3658-4031) and reduced viscous terms
//     (visflx_reduced_cuf, :3539-3656) from one read of the 18 neighbours; momentum's update;
//   cell_species_kernel    the species' convection and diffusion, the enthalpy flux and the
//     energy's update;
//   finish_species_kernel  (finish.hip) the chemistry source and the species' update.
// In the general path three directional sweeps read and write fl and read w_aux once each,
// and wait for about 20 dependent staging rounds per tile; these kernels touch each plane of
// w_aux once or twice.  They are bound by the rate of vector loads: a wave's load costs 16-17
// cycles of its CU's L1 whether a lane takes 8 or 16 bytes (measured: 30 and 61 B/clk).  So
// the species, with 19 + 7 values per cell each, go through LDS.
#include <type_traits>

#include "finish.h"
#include "thermo_dev.h"

namespace streams {

struct CellArgs {
  const double *cd1, *met[3], *coord[3];
  const int *mask;
  Thermo th;
  double r_univ, rhodt, gamdt, rhodt_next;
  int init, fold;
};

// Tiles of TX x TY x TZ cells, one per thread, x fastest, then the y tiles of a band, then z, then the
// next band; one contiguous range of tiles per XCD.  Whole rows first, because a row of 38 cells
// touches up to twice the 128-byte lines of its 32: 256^3 8.51 -> 8.25 ms a call.
constexpr int TX = 32, TY = 4, TZ = 2, YBAND = 8;
struct CellTiles {
  int nxt, nzt, yb;           // tiles along x and z, y tiles of a band
  unsigned tiles;             // with the last band filled up
};
inline bool cell_tiles(const Box &b, CellTiles &r) {
  const int nyt = (b.ny + TY - 1) / TY;
  r.nxt = (b.nx + TX - 1) / TX;
  r.nzt = (b.nz + TZ - 1) / TZ;
  r.yb = nyt < YBAND ? nyt : YBAND;
  const long n = (long)r.nxt * r.nzt * r.yb * ((nyt + r.yb - 1) / r.yb);
  r.tiles = (unsigned)n;
  return n <= 0xffffff00l;
}
// First cell of this workgroup's tile (it may lie past ny in the last band).
__device__ inline void tile_origin(const CellTiles &r, unsigned tile, int &i0, int &j0, int &k0) {
  i0 = 1 + TX * (int)(tile % r.nxt);
  tile /= r.nxt;
  const int y = (int)(tile % r.yb);
  tile /= r.yb;
  k0 = 1 + TZ * (int)(tile % r.nzt);
  j0 = 1 + TY * ((int)(tile / r.nzt) * r.yb + y);
}

// A tile of one plane with its star of W cells on each side in LDS: [z][y][x] with the
// corners left unset.  Each thread copies its own cell and ROUNDS cells of the halo, whose
// places are worked out once (cells past the end of the padded plane, which only threads
// outside the box would use, are read at its end).
template <int W>
struct StarTile {
  static constexpr int SX = TX + 2 * W, SY = TY + 2 * W, SZ = TZ + 2 * W, SIZE = SX * SY * SZ;
  static constexpr int NZ = 2 * W * TX * TY, NY = 2 * W * TX * TZ, NXH = 2 * W * TY * TZ;
  static constexpr int HALO = NZ + NY + NXH, ROUNDS = (HALO + 255) / 256;
  static constexpr int DY = SX, DZ = SX * SY;
  unsigned own, src[ROUNDS];          // byte offsets in the plane
  int me, dst[ROUNDS];                // places in LDS
  bool last;                          // this thread takes part in the last round
  __device__ inline static int place(int x, int y, int z) { return (x + W) + SX * ((y + W) + SY * (z + W)); }
  __device__ inline void init(const Box &b, int i0, int j0, int k0, int tid) {
    auto off = [&](int x, int y, int z) {
      const int i = min(i0 + x, b.nx + b.ng), j = min(j0 + y, b.ny + b.ng), k = min(k0 + z, b.nz + b.ng);
      return (unsigned)b.p(i, j, k) * 8u;
    };
    const int tx = tid % TX, ty = tid / TX % TY, tz = tid / (TX * TY);
    own = off(tx, ty, tz);
    me = place(tx, ty, tz);
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      int e = tid + 256 * r, x, y, z;
      if (r == ROUNDS - 1) {
        last = e < HALO;
        e = last ? e : 0;
      }
      if (e < NZ) {
        x = e % TX;
        y = e / TX % TY;
        z = e / (TX * TY);
        z = z < W ? z - W : z - W + TZ;
      } else if (e < NZ + NY) {
        e -= NZ;
        x = e % TX;
        z = e / TX % TZ;
        y = e / (TX * TZ);
        y = y < W ? y - W : y - W + TY;
      } else {
        e -= NZ + NY;
        x = e % (2 * W);
        y = e / (2 * W) % TY;
        z = e / (2 * W * TY);
        x = x < W ? x - W : x - W + TX;
      }
      src[r] = off(x, y, z);
      dst[r] = place(x, y, z);
    }
  }
  struct Held {
    double v[ROUNDS + 1];
  };
  template <class Cell>
  __device__ inline void load(const double *plane, const Cell &cell, Held &h) const {
    h.v[ROUNDS] = cell(plane, own);
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) h.v[r] = cell(plane, src[r]);
  }
  __device__ inline void store(double *buf, const Held &h) const {
    buf[me] = h.v[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r)
      if (r < ROUNDS - 1 || last) buf[dst[r]] = h.v[r];
  }
};

// c1/2, ... T^5/5 polynomial of a cph row by Horner: h = a6 + T (a1 + T (a2/2 + ...))
__device__ inline double enthalpy_row(const double *c, double T) {
  double h = c[4];
  h = fma(h, T, c[3]);
  h = fma(h, T, c[2]);
  h = fma(h, T, c[1]);
  h = fma(h, T, c[0]);
  return fma(h, T, c[5]);
}

// Addressing and RK update of one cell.  Variable and neighbour are the same for all lanes, so
// they go into a scalar base address and one 32-bit byte offset addresses every load of a
// thread.
struct CellAccess {
  const double *wa;
  double *w, *fl, *fln;
  long ps, fs;
  unsigned pt, t;               // byte offsets in a padded and in an interior plane
  bool inside, fluid;
  template <class T>
  __device__ static inline auto &cell(T *base, unsigned off) {
    using C = std::conditional_t<std::is_const_v<T>, const char, char>;
    unsigned long u = (unsigned long)base;
    asm("" : "+s"(u));          // keep the scalar part apart: else it is added to off first
    return *(__attribute__((address_space(1))) T *)((__attribute__((address_space(1))) C *)u + off);
  }
  // variable m (reference index), o cells further; p: pt or an opaque copy of it, which keeps a
  // group of loads from being issued before the groups ahead of it (they would all be in
  // registers at once)
  __device__ inline double at(long o, int m, unsigned p) const { return cell(wa + (o + ps * (m - 1)), p); }
  // right-hand side of variable m (0-based): update_flux, update_field and, folded in, this
  // substep's (init: f0 is what fln holds before) or the next one's init_flux
  __device__ inline void update(const CellArgs &A, int m, double acc, int init) const {
    if (!inside) return;
    auto &flm = cell(fl + fs * m, t), &flnm = cell(fln + fs * m, t), &wm = cell(w + ps * m, pt);
    const double f0 = init == 1 ? -A.rhodt * flm : flnm;
    const double fn = f0 - A.gamdt * acc;
    if (A.fold) {
      flnm = -A.rhodt_next * acc;
    } else {
      flm = acc;
      flnm = fn;
    }
    if (fluid) wm = wm + fn;
  }
  // the same right-hand side left in fl for a later kernel's update
  __device__ inline void leave(const CellArgs &A, int m, double acc) const {
    if (!inside) return;
    auto &flm = cell(fl + fs * m, t);
    if (A.init == 1) cell(fln + fs * m, t) = -A.rhodt * flm;
    flm = acc;
  }
};

// Cell of this thread in the tile at (i0, j0, k0); threads past the end of the box work on its
// last cell and write nothing.
__device__ inline CellAccess cell_access(const Box &b, int i0, int j0, int k0, double *w, const double *wa, double *fl,
                                         double *fln, const int *mask, int &i, int &j, int &k) {
  i = i0 + (int)threadIdx.x % TX;
  j = j0 + (int)threadIdx.x / TX % TY;
  k = k0 + (int)threadIdx.x / (TX * TY);
  const bool inside = i <= b.nx && j <= b.ny && k <= b.nz;
  i = min(i, b.nx);
  j = min(j, b.ny);
  k = min(k, b.nz);
  const unsigned pt = (unsigned)b.p(i, j, k);
  return CellAccess{wa, w, fl, fln, b.pstride(), b.fstride(), pt * 8u, (unsigned)b.f(i, j, k) * 8u, inside,
                    mask == nullptr || mask[pt] == 0};
}

template <int NS, int LB>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5)))
cell_momentum_kernel(Box b, double *__restrict__ w, const double *__restrict__ wa, double *__restrict__ fl,
                     double *__restrict__ fln, CellArgs A, CellTiles BT) {
  using X = Idx<NS>;
  const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);
  if (tile >= BT.tiles) return;
  int i0, j0, k0, i, j, k;
  tile_origin(BT, tile, i0, j0, k0);
  if (j0 > b.ny) return;                       // a band's filling
  const CellAccess C = cell_access(b, i0, j0, k0, w, wa, fl, fln, A.mask, i, j, k);
  const unsigned pt = C.pt;
  auto at = [&](long o, int m, unsigned p) { return C.at(o, m, p); };
  const long st[3] = {1, b.px(), b.px() * b.py()};
  const int ijk[3] = {i, j, k};
  const double rc = at(0, X::J_R, pt), tc = at(0, X::J_T, pt), pc = at(0, X::J_P, pt);
  double eacc = 0.0;
  const double vc[3] = {at(0, X::J_U, pt), at(0, X::J_V, pt), at(0, X::J_W, pt)};
  const double qc = 0.5 * (vc[0] * vc[0] + vc[1] * vc[1] + vc[2] * vc[2]);
  const double hc = at(0, X::J_H, pt);
  const double muc = at(0, X::J_MU, pt), kc = at(0, X::J_K_COND, pt), dvc = at(0, X::J_DIV, pt);
  const double ec = hc - pc / rc - qc;
  double macc[3] = {0.0, 0.0, 0.0};
  double g[3][5];             // d/dx_d of u, v, w, mu, div/3
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double met = A.met[d][ijk[d] - 1];
    const double *xc = A.coord[d] + ijk[d] + b.ng - 1;
    const double dxhl = 2.0 / (xc[1] - xc[-1]);
#pragma unroll
    for (int q = 0; q < 5; ++q) g[d][q] = 0.0;
#pragma unroll
    for (int l = 1; l <= LB; ++l) {
      const double cl = A.cd1[(l - 1) + 4 * (LB - 1)] * met;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const long q = (s == 0 ? l : -l) * st[d];
        unsigned p = pt;
        opaque(p);
        const double sg = s == 0 ? 1.0 : -1.0;
        const double vn[3] = {at(q, X::J_U, p), at(q, X::J_V, p), at(q, X::J_W, p)};
        const double rn = at(q, X::J_R, p), hn = at(q, X::J_H, p), mun = at(q, X::J_MU, p), dvn = at(q, X::J_DIV, p);
        const double pn = at(q, X::J_P, p);
        g[d][0] += sg * cl * vn[0];
        g[d][1] += sg * cl * vn[1];
        g[d][2] += sg * cl * vn[2];
        g[d][3] += sg * cl * mun;
        g[d][4] += sg * cl * dvn;
        const double qn = 0.5 * (vn[0] * vn[0] + vn[1] * vn[1] + vn[2] * vn[2]);
        const double f = sg * 0.25 * cl * (rc + rn) * (vc[d] + vn[d]);
        macc[0] += f * (vc[0] + vn[0]);
        macc[1] += f * (vc[1] + vn[1]);
        macc[2] += f * (vc[2] + vn[2]);
        macc[d] += sg * cl * pn;
        const double en = hn - pn * rcp_nr(rn) - qn;
        eacc += f * (ec + en + (vc[0] * vn[0] + vc[1] * vn[1] + vc[2] * vn[2]));
        eacc += sg * cl * (vc[d] * pn + vn[d] * pc);
        if (l == 1) {
          const double dx = s == 0 ? xc[1] - xc[0] : xc[0] - xc[-1];
          const double muf = 0.5 * (muc + mun) / dx * dxhl;
          const double kf = 0.5 * (kc + at(q, X::J_K_COND, p)) / dx * dxhl;
          macc[0] -= muf * (vn[0] - vc[0]);
          macc[1] -= muf * (vn[1] - vc[1]);
          macc[2] -= muf * (vn[2] - vc[2]);
          eacc -= kf * (at(q, X::J_T, p) - tc) + muf * (qn - qc);
        }
        // the neighbour's terms are summed before the next one's loads
        opaque(eacc);
#pragma unroll
        for (int m = 0; m < 3; ++m) opaque(macc[m]);
#pragma unroll
        for (int m = 0; m < 5; ++m) opaque(g[d][m]);
      }
    }
  }
  // reduced viscous terms
  const double d2 = 2.0 * dvc;
  const double s11 = g[0][0] - d2, s12 = g[0][1], s13 = g[0][2];
  const double s21 = g[1][0], s22 = g[1][1] - d2, s23 = g[1][2];
  const double s31 = g[2][0], s32 = g[2][1], s33 = g[2][2] - d2;
  const double sigx = g[0][3] * s11 + g[1][3] * s12 + g[2][3] * s13 + muc * g[0][4];
  const double sigy = g[0][3] * s21 + g[1][3] * s22 + g[2][3] * s23 + muc * g[1][4];
  const double sigz = g[0][3] * s31 + g[1][3] * s32 + g[2][3] * s33 + muc * g[2][4];
  const double sigah = (s11 * g[0][0] + s12 * g[1][0] + s13 * g[2][0] + s21 * g[0][1] + s22 * g[1][1] +
                        s23 * g[2][1] + s31 * g[0][2] + s32 * g[1][2] + s33 * g[2][2]) * muc;
  eacc -= sigx * vc[0] + sigy * vc[1] + sigz * vc[2] + sigah;
C.update(A, NS + 0, macc[0] - sigx, A.init);
  C.update(A, NS + 1, macc[1] - sigy, A.init);
  C.update(A, NS + 2, macc[2] - sigz, A.init);
  C.leave(A, NS + 3, eacc);
}

template <int NS, int LB>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
cell_species_kernel(Box b, double *__restrict__ w, const double *__restrict__ wa, double *__restrict__ fl,
                    double *__restrict__ fln, CellArgs A, CellTiles BT) {
  using X = Idx<NS>;
  __shared__ double tlds[thermo_lds_doubles<NS>(TH_CPH)];
  __shared__ double ybuf[StarTile<LB>::SIZE], dbuf[StarTile<1>::SIZE], tbuf[StarTile<1>::SIZE], wbuf[StarTile<1>::SIZE];
  const ThermoLds TL = thermo_stage<NS, 0>(A.th, tlds, TH_CPH);
  const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);
  if (tile >= BT.tiles) return;
  int i0, j0, k0, i, j, k;
  tile_origin(BT, tile, i0, j0, k0);
  if (j0 > b.ny) return;                       // a band's filling
  const CellAccess C = cell_access(b, i0, j0, k0, w, wa, fl, fln, A.mask, i, j, k);
  const long ps = C.ps;
  const unsigned pt = C.pt;
  auto at = [&](long o, int m, unsigned p) { return C.at(o, m, p); };
  auto cell = [](const double *base, unsigned off) { return CellAccess::cell(base, off); };
  const long st[3] = {1, b.px(), b.px() * b.py()};
  const int ijk[3] = {i, j, k};
  StarTile<1> ST;
  ST.init(b, i0, j0, k0, threadIdx.x);
  typename StarTile<1>::Held yh1, dh;
  ST.load(wa, cell, yh1);
  ST.load(wa + ps * X::J_D_START, cell, dh);
  {
    // temperature and mixture weight W = R_univ rho T / p of the tile and its faces
    typename StarTile<1>::Held th, rh, ph;
    ST.load(wa + ps * (X::J_T - 1), cell, th);
    ST.load(wa + ps * (X::J_R - 1), cell, rh);
    ST.load(wa + ps * (X::J_P - 1), cell, ph);
    ST.store(tbuf, th);
#pragma unroll
    for (int r = 0; r <= StarTile<1>::ROUNDS; ++r) rh.v[r] = A.r_univ * rh.v[r] * th.v[r] / ph.v[r];
    ST.store(wbuf, rh);
  }
  __syncthreads();
  constexpr int yo[3] = {1, StarTile<LB>::DY, StarTile<LB>::DZ}, so[3] = {1, StarTile<1>::DY, StarTile<1>::DZ};
  const double *tl = tbuf + ST.me, *wl = wbuf + ST.me, *y1 = ybuf + ST.me, *dl = dbuf + ST.me;
  const double Wc = wl[0];
  // ---- the faces' sums over the species: F = a/2 sum_s t_s, t_s = (D_c + D_n)(y_n W_n - y_c W_c)
  double an[6], F[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    const double *xc = A.coord[q / 2] + ijk[q / 2] + b.ng - 1;
    const double dx = q % 2 == 0 ? xc[1] - xc[0] : xc[0] - xc[-1];
    const double Wn = wl[q % 2 == 0 ? so[q / 2] : -so[q / 2]];
    // half of mwmif times the half of the averaged diffusivity, times the divergence metric
    an[q] = 0.25 * (Wn + Wc) / (Wn * Wc) / dx * (2.0 / (xc[1] - xc[-1]));
    F[q] = 0.0;
    opaque(an[q]);
  }
#pragma unroll 1
  for (int s = 0; s < NS; ++s) {
    __syncthreads();                           // the buffers' last readers are done
    ST.store(ybuf, yh1);
    ST.store(dbuf, dh);
    __syncthreads();
    if (s + 1 < NS) {
      ST.load(wa + ps * (s + 1), cell, yh1);
      ST.load(wa + ps * (X::J_D_START + s + 1), cell, dh);
    }
    const double yw = y1[0] * Wc, rd = dl[0];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      const int o = q % 2 == 0 ? so[q / 2] : -so[q / 2];
      F[q] += (rd + dl[o]) * (y1[o] * wl[o] - yw);
    }
  }
  StarTile<LB> YT;
  YT.init(b, i0, j0, k0, threadIdx.x);
  typename StarTile<LB>::Held yh;
  YT.load(wa, cell, yh);
  ST.load(wa + ps * X::J_D_START, cell, dh);
#pragma unroll
  for (int q = 0; q < 6; ++q) F[q] *= 0.5 * an[q];
  // ---- pair factors of the neighbours +1, -1, +2, -2, ...
  double P[3][2 * LB], psum = 0.0;
  const double rc = at(0, X::J_R, pt);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double met = 0.25 * A.met[d][ijk[d] - 1], vc = at(0, X::J_U + d, pt);
    unsigned p = pt;
    opaque(p);
#pragma unroll
    for (int l = 1; l <= LB; ++l) {
      const double cl = A.cd1[(l - 1) + 4 * (LB - 1)] * met;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const long o = q == 0 ? l * st[d] : -l * st[d];
        const double f = (q == 0 ? cl : -cl) * (rc + at(o, X::J_R, p)) * (vc + at(o, X::J_U + d, p));
        P[d][2 * (l - 1) + q] = f;
        psum += f;
      }
    }
#pragma unroll
    for (int q = 0; q < 2 * LB; ++q) opaque(P[d][q]);
    opaque(psum);
  }
  // ---- species by species, the next one's planes on their way meanwhile; a face's flux is
  // F (y_c + y_n) - a t_s
  const double *yl = ybuf + YT.me;
  double he = 0.0;
#pragma unroll 1
  for (int s = 0; s < NS; ++s) {
    __syncthreads();
    YT.store(ybuf, yh);
    ST.store(dbuf, dh);
    __syncthreads();
    if (s + 1 < NS) {
      YT.load(wa + ps * (s + 1), cell, yh);
      ST.load(wa + ps * (X::J_D_START + s + 1), cell, dh);
    }
    const double yc = yl[0], yw = yc * Wc, rd = dl[0];
    const double *tr = TL.tr + s * (TMAXSET + 1);
    auto h_of = [&](double T) {
      int m = 0;
      for (int q = 1; q < TL.nsetcv; ++q) m = T >= tr[q] ? q : m;
      return enthalpy_row(TL.cph + (m * NS + s) * TSTRIDE, T);
    };
    double hc = h_of(tl[0]);
    double acc = psum * yc;
    opaque(hc);
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      const int sg = q % 2 == 0 ? 1 : -1;
      const int o = sg * so[q / 2];
      const double yn = yl[sg * yo[q / 2]];
      const double flux = F[q] * (yc + yn) - an[q] * ((rd + dl[o]) * (yn * wl[o] - yw));
      acc += flux;
      he += flux * (hc + h_of(tl[o]));
      acc += P[q / 2][q % 2] * yn;
#pragma unroll
      for (int l = 2; l <= LB; ++l) acc += P[q / 2][2 * (l - 1) + q % 2] * yl[sg * l * yo[q / 2]];
      opaque(acc);
      opaque(he);
    }
    C.leave(A, s, acc);
  }
  if (C.inside) C.update(A, NS + 3, CellAccess::cell(fl + C.fs * (NS + 3), C.t) + 0.5 * he, 2);
}

template <int NS, int LB>
void cells_launch(unsigned g, hipStream_t st, const Box &b, double *w, const double *wa, double *fl, double *fln,
                  const CellArgs &A, const CellTiles &BT) {
  cell_momentum_kernel<NS, LB><<<g, 256, 0, st>>>(b, w, wa, fl, fln, A, BT);
  cell_species_kernel<NS, LB><<<g, 256, 0, st>>>(b, w, wa, fl, fln, A, BT);
}

}  // namespace streams

using namespace streams;

// One RK substep from the auxiliaries on (the three sweeps of streams_rhs_sweep followed by
// streams_rhs_finish, or with fold by streams_rhs_finish_next) for a field in which every face
// takes the KEEP flux at the full order: no shocked face, no order-reduced boundary, no
// forced-zero face.
extern "C" int streams_rhs_cells(int n_s, int nx, int ny, int nz, int ng, int nv_aux, int lmax_base, double *w,
                                 const double *w_aux, double *fl, double *fln, const double *coeff_deriv1,
                                 const double *dcsidx, const double *detady, const double *dzitdz, const double *x,
                                 const double *y, const double *z, const double *cp_coeff, int nsetcv,
                                 const double *trange, int indx_cp_l, int indx_cp_r, double r_univ, int chem,
                                 int nreactions, const double *mw, const double *kin_pack, const double *kc_tab,
                                 int num_t_tab, double t_min_tab, double dt_tab, int init, double rhodt,
                                 double gamdt, int fold, double rhodt_next, const int *fluid_mask, void *stream) {
  if (nv_aux < 2 * n_s + 13 || nx < 2 || ny < 2 || nz < 2 || ng < lmax_base) return STREAMS_E_DIMS;
  if (lmax_base < 3 || lmax_base > 4 || init < 1 || init > 2) return STREAMS_E_OPTION;
  if (nsetcv < 1 || nsetcv > TMAXSET || indx_cp_l != 0 || indx_cp_r != 4) return STREAMS_E_OPTION;
  if (n_s > KTB) return STREAMS_E_NSPECIES;
  Box b{nx, ny, nz, ng};
  CellTiles BT;
  if (b.pstride() >= 1l << 29 || !cell_tiles(b, BT)) return STREAMS_E_DIMS;
  CellArgs A{coeff_deriv1, {dcsidx, detady, dzitdz}, {x, y, z}, fluid_mask,
             Thermo{nullptr, cp_coeff, trange, nsetcv, indx_cp_l, indx_cp_r}, r_univ, rhodt, gamdt, rhodt_next, init, fold};
  const unsigned g = xcd_grid(BT.tiles);
  hipStream_t st = as_stream(stream);
  STREAMS_DISPATCH_NS(n_s, (lmax_base == 3 ? cells_launch<NS, 3>(g, st, b, w, w_aux, fl, fln, A, BT)
                                           : cells_launch<NS, 4>(g, st, b, w, w_aux, fl, fln, A, BT)));
  FinishArgs F{};
  F.mask = fluid_mask;
  F.mw = mw;
  F.K = KinPacked{kin_pack, kc_tab, nreactions, num_t_tab, t_min_tab, dt_tab, r_univ};
  F.chem = chem && nreactions > 0;
  F.gamdt = gamdt;
  F.fold = fold;
  F.rhodt_next = rhodt_next;
  return finish_species_launch(n_s, b, w, w_aux, fl, fln, F, st);
}
