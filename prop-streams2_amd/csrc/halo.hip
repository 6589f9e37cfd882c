// halo.hip — ghost-cell fills: single-rank loopback exchange and physical boundaries.
//
// The reference exchanges ng-deep face slabs through pack -> MPI (or a device copy when
// the neighbour is the rank itself) -> unpack (base_gpu.F90:1132-1264).  On one GPU the
// periodic exchange is a direct copy from the opposite interior slab into the ghost slab,
// one launch for all axes, sides and variables.  When an axis is shorter than ng the source slab
// overlaps the ghost slab of the same axis; there a thread takes a whole line across both and reads its
// sources before it writes any of them.  Extrapolation fills any run of faces in one launch as well.

#include "common.h"

namespace streams {

// axis 0: (i in 1..ng, j in 1..ny, k in 1..nz); axis 1: (i 1..nx, j 1..ng, k 1..nz);
// axis 2: (i 1..nx, j 1..ny, k 1..ng).  The flat index covers slab, side, variable; on an axis
// shorter than ng it covers the lines across the slabs (extent 1 along the axis) and variables.
template <class I>
struct Slab {
  I n;                      // threads of this axis
  unsigned blocks;
  int e0, e1, e2;           // extents in i, j, k
  bool line;
};
template <class I>
struct SwapPlan {
  Slab<I> ax[3];
};

constexpr int NG_LINE = 8;  // deepest ghost layer a line keeps in registers

__device__ inline void slab_src_dst(const Box &b, int ax, int side, int a, int bq, int c, long &src,
                                    long &dst) {
  // side 0: left ghost <- right interior slab; side 1: right ghost <- left interior slab
  int i = a, j = bq, k = c;
  if (ax == 0) {
    if (side == 0) { src = b.p(b.nx - b.ng + i, j, k); dst = b.p(i - b.ng, j, k); }
    else { src = b.p(i, j, k); dst = b.p(b.nx + i, j, k); }
  } else if (ax == 1) {
    if (side == 0) { src = b.p(i, b.ny - b.ng + j, k); dst = b.p(i, j - b.ng, k); }
    else { src = b.p(i, j, k); dst = b.p(i, b.ny + j, k); }
  } else {
    if (side == 0) { src = b.p(i, j, b.nz - b.ng + k); dst = b.p(i, j, k - b.ng); }
    else { src = b.p(i, j, k); dst = b.p(i, j, b.nz + k); }
  }
}

// All periodic axes in one launch, a range of workgroups per axis: a launch takes about 4 us on
// this GPU, as long as its copies in a small box (19x14x11 cells: three launches 10.5 us -> one of
// 4).  On an axis shorter than ng the sources lie in ghosts that are written as well, but only in
// those of the same line: a thread reads its line's sources before it writes any, which takes the
// place of a staging buffer's allocation and two more launches.
template <class I>
__global__ void __launch_bounds__(256) swap_kernel(Box b, SwapPlan<I> plan, double *__restrict__ w) {
  unsigned blk = blockIdx.x;
  int ax = 0;
  if (blk >= plan.ax[0].blocks) { blk -= plan.ax[0].blocks; ax = 1; }
  if (ax == 1 && blk >= plan.ax[1].blocks) { blk -= plan.ax[1].blocks; ax = 2; }
  const Slab<I> s = plan.ax[ax];
  I t = (I)blk * 256 + threadIdx.x;
  if (t >= s.n) return;
  const int a = 1 + (int)(t % s.e0); t /= s.e0;
  const int bq = 1 + (int)(t % s.e1); t /= s.e1;
  const int c = 1 + (int)(t % s.e2); t /= s.e2;
  long src, dst;
  if (s.line && b.ng > NG_LINE) {
    // deeper: in place, each side from the end that its sources are written last
    double *v = w + b.pstride() * (long)t;
    for (int side = 0; side < 2; ++side)
      for (int q = 0; q < b.ng; ++q) {
        const int l = side == 0 ? 1 + q : b.ng - q;
        slab_src_dst(b, ax, side, ax == 0 ? l : a, ax == 1 ? l : bq, ax == 2 ? l : c, src, dst);
        v[dst] = v[src];
      }
  } else if (s.line) {
    double *v = w + b.pstride() * (long)t;
    double x[2][NG_LINE];
#pragma unroll
    for (int side = 0; side < 2; ++side)
#pragma unroll
      for (int l = 0; l < NG_LINE; ++l)
        if (l < b.ng) {
          slab_src_dst(b, ax, side, ax == 0 ? 1 + l : a, ax == 1 ? 1 + l : bq, ax == 2 ? 1 + l : c, src, dst);
          x[side][l] = v[src];
        }
#pragma unroll
    for (int side = 0; side < 2; ++side)
#pragma unroll
      for (int l = 0; l < NG_LINE; ++l)
        if (l < b.ng) {
          slab_src_dst(b, ax, side, ax == 0 ? 1 + l : a, ax == 1 ? 1 + l : bq, ax == 2 ? 1 + l : c, src, dst);
          v[dst] = x[side][l];
        }
  } else {
    slab_src_dst(b, ax, (int)(t & 1), a, bq, c, src, dst);
    const long ps = b.pstride() * (long)(t >> 1);
    w[dst + ps] = w[src + ps];
  }
}

// bcextr_var_cuf / bcextr_cuf: zero-order extrapolation of the faces first..last (1..6) of
// nv variables, a row of workgroups (blockIdx.y) per face; sources are interior points, so the
// faces are independent.
__global__ void __launch_bounds__(256) extr_kernel(Box b, int first, int nv, double *__restrict__ w) {
  const int ilat = first + (int)blockIdx.y;
  const int e0 = (ilat <= 2) ? b.ny : b.nx;
  const int e1 = (ilat <= 4) ? b.nz : b.ny;
  const long n = (long)b.ng * e0 * e1 * nv;
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  int l, a, c, m;
  // flat index: l fastest, then the two face coordinates, then the variable
  l = 1 + (int)(t % b.ng); long r = t / b.ng;
  a = 1 + (int)(r % e0); r /= e0;
  c = 1 + (int)(r % e1); r /= e1;
  m = (int)r;
  long src, dst;
  switch (ilat) {
    case 1: src = b.p(1, a, c); dst = b.p(1 - l, a, c); break;
    case 2: src = b.p(b.nx, a, c); dst = b.p(b.nx + l, a, c); break;
    case 3: src = b.p(a, 1, c); dst = b.p(a, 1 - l, c); break;
    case 4: src = b.p(a, b.ny, c); dst = b.p(a, b.ny + l, c); break;
    case 5: src = b.p(a, c, 1); dst = b.p(a, c, 1 - l); break;
    default: src = b.p(a, c, b.nz); dst = b.p(a, c, b.nz + l); break;
  }
  const long ps = b.pstride() * m;
  w[dst + ps] = w[src + ps];
}

// bcwall_ad_cuf: mirror with the three momenta reversed
__global__ void __launch_bounds__(256) wall_ad_kernel(Box b, int ilat, int ns, long n, double *__restrict__ w) {
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  int nv = ns + 4;
  int l = 1 + (int)(t % b.ng); long r = t / b.ng;
  int e0 = (ilat <= 2) ? b.ny : b.nx;
  int e1 = (ilat <= 4) ? b.nz : b.ny;
  int a = 1 + (int)(r % e0); r /= e0;
  int c = 1 + (int)(r % e1); r /= e1;
  int m = (int)r;  // 0-based variable
  long src, dst;
  switch (ilat) {
    case 1: src = b.p(l, a, c); dst = b.p(1 - l, a, c); break;
    case 2: src = b.p(b.nx + 1 - l, a, c); dst = b.p(b.nx + l, a, c); break;
    case 3: src = b.p(a, l, c); dst = b.p(a, 1 - l, c); break;
    case 4: src = b.p(a, b.ny + 1 - l, c); dst = b.p(a, b.ny + l, c); break;
    case 5: src = b.p(a, c, l); dst = b.p(a, c, 1 - l); break;
    default: src = b.p(a, c, b.nz + 1 - l); dst = b.p(a, c, b.nz + l); break;
  }
  const long ps = b.pstride() * m;
  double v = w[src + ps];
  w[dst + ps] = (m >= ns && m < ns + 3) ? -v : v;
  (void)nv;
}

int extr_faces(const Box &b, int first, int last, int nv, double *w, hipStream_t st) {
  long n = 0;                                        // points of the largest face
  for (int ilat = first; ilat <= last; ++ilat) {
    const long f = (long)b.ng * (ilat <= 2 ? b.ny : b.nx) * (ilat <= 4 ? b.nz : b.ny) * nv;
    n = f > n ? f : n;
  }
  if (n <= 0) return 0;
  extr_kernel<<<dim3(blocks_for(n, 256), last - first + 1), 256, 0, st>>>(b, first, nv, w);
  return hip_status();
}

// 64-bit point indices only where a slab holds more points than 32 bits count
template <class I>
int swap_launch(const Box &b, const int *periodic, int nv, double *w, hipStream_t st) {
  SwapPlan<I> plan{};
  unsigned g = 0;
  const int n[3] = {b.nx, b.ny, b.nz};
  for (int ax = 0; ax < 3; ++ax) {
    Slab<I> &s = plan.ax[ax];
    if (!periodic[ax]) continue;
    s.line = n[ax] < b.ng;
    const int depth = s.line ? 1 : b.ng;
    s.e0 = ax == 0 ? depth : b.nx;
    s.e1 = ax == 1 ? depth : b.ny;
    s.e2 = ax == 2 ? depth : b.nz;
    s.n = (I)s.e0 * s.e1 * s.e2 * nv * (s.line ? 1 : 2);
    s.blocks = blocks_for((long)s.n, 256);
    g += s.blocks;
  }
  if (g == 0) return 0;
  swap_kernel<I><<<g, 256, 0, st>>>(b, plan, w);
  return hip_status();
}

}  // namespace streams

using namespace streams;

extern "C" int streams_bcswap(int nx, int ny, int nz, int ng, int nv, double *w, const int *periodic,
                              void *stream) {
  if (nx < 1 || ny < 1 || nz < 1 || ng < 1 || nv < 1 || !periodic) return STREAMS_E_DIMS;
  Box b{nx, ny, nz, ng};
  hipStream_t st = as_stream(stream);
  // The reference packs all six slabs before unpacking any.  Sources of one axis never lie
  // in the ghost slabs of another axis (their tangential indices are interior), so the
  // axes are independent.
  const long most = 2L * ng * nv;
  const bool wide = most * ny * nz > 0xfff00000l || most * nx * nz > 0xfff00000l || most * nx * ny > 0xfff00000l;
  return wide ? swap_launch<unsigned long>(b, periodic, nv, w, st) : swap_launch<unsigned>(b, periodic, nv, w, st);
}

extern "C" int streams_bcextr_var(int nx, int ny, int nz, int ng, double *w_var, void *stream) {
  Box b{nx, ny, nz, ng};
  return extr_faces(b, 1, 6, 1, w_var, as_stream(stream));
}

extern "C" int streams_bcextr(int ilat, int nx, int ny, int nz, int ng, int nv, double *w, void *stream) {
  if (ilat < 1 || ilat > 6) return STREAMS_E_DIMS;
  Box b{nx, ny, nz, ng};
  return extr_faces(b, ilat, ilat, nv, w, as_stream(stream));
}

extern "C" int streams_bcwall_ad(int n_s, int ilat, int nx, int ny, int nz, int ng, double *w, void *stream) {
  if (ilat < 1 || ilat > 6 || n_s < 1) return STREAMS_E_DIMS;
  Box b{nx, ny, nz, ng};
  int e0 = (ilat <= 2) ? ny : nx;
  int e1 = (ilat <= 4) ? nz : ny;
  long n = (long)ng * e0 * e1 * (n_s + 4);
  if (n <= 0) return 0;
  wall_ad_kernel<<<blocks_for(n, 256), 256, 0, as_stream(stream)>>>(b, ilat, n_s, n, w);
  return hip_status();
}

extern "C" int streams_species_supported(int *list, int cap) {
  static const int compiled[] = {
#define STREAMS_LIST_ENTRY(n) n,
      STREAMS_NS_LIST(STREAMS_LIST_ENTRY)
#undef STREAMS_LIST_ENTRY
  };
  int n = (int)(sizeof(compiled) / sizeof(compiled[0]));
  for (int q = 0; q < n && q < cap; ++q) list[q] = compiled[q];
  return n;
}
