// ca_corner.h -- the eight grid_avg8 corners (utils.h:18-23) of an AFM cell in
// a Ca solve: the word that k_ca_corners keeps of each, and the ATP value that
// a fused launch's cells compute from it.  A corner is numbered in binary x, y,
// z (bit 0: the upper x).  The index arithmetic takes the grid's sizes from any
// record that has them, so that the same code runs in the kernels (k_field.hip)
// and in a CPU test.
#pragma once
#include "epi_dev.h"
#include "ca_laws.h"

namespace epi {

// A corner's word: x the point, wrapped in x and y; y its voxel word (Tis::vox);
// z the masks of its six stencil neighbours (bits 0-5: x-, x+, y-, y+, z-, z+)
// and the flags below; w the point as it lies (a periodic copy at x = NX or
// y = NY).  A grid's points may pass 2^32 (42 bytes a point of grid arrays:
// 180 GB), so z also holds bits 32-39 of both points (in bits 12-19 of x's, in
// bits 20-27 of w's); 2^40 points are more than any card holds.
constexpr unsigned CQ_XM = 1u << 6, CQ_XP = 1u << 7, CQ_YM = 1u << 8, CQ_YP = 1u << 9;   // x = 0, x = NX - 1, ...
constexpr unsigned CQ_ZM = 1u << 10, CQ_ZP = 1u << 11;   // z = 0 (mirror), z = NZ - 1 (self)
constexpr unsigned CQ_PLAIN = 1u << 30;   // not updated inside the solve: read as it is
constexpr unsigned CQ_SLOW = 1u << 31;    // a mask byte above 1: the masks come from the map

__device__ __forceinline__ uint4 corner_pack(long long v, unsigned word, unsigned bits, long long raw) {
  return make_uint4((unsigned)v, word, bits | (unsigned)(v >> 32) << 12 | (unsigned)(raw >> 32) << 20, (unsigned)raw);
}
__device__ __forceinline__ long long corner_at(uint4 q) { return (long long)(q.z >> 12 & 0xffu) << 32 | q.x; }
__device__ __forceinline__ long long corner_raw(uint4 q) { return (long long)(q.z >> 20 & 0xffu) << 32 | q.w; }
// of a cell that has no corners: point 0, as it lies
__device__ __forceinline__ uint4 corner_none() { return make_uint4(0u, 0u, CQ_PLAIN, 0u); }

// corner k of the cell at lattice point (x, y, z)
template <class G>
__device__ __forceinline__ uint4 corner_word(const G& t, int izb, int x, int y, int z, int k) {
  const int NX = t.NX, NY = t.NY, NZ = t.NZ;
  int j = x + (k & 1), kk = y + ((k >> 1) & 1);
  const int l = z + (k >> 2);
  const long long raw = gidx(t, j, kk, l);
  if (j == NX) j = 0;
  if (kk == NY) kk = 0;
  const long long v = gidx(t, j, kk, l);
  unsigned word = 0, bits = CQ_PLAIN;
  if (l < izb && izb <= NZ) {
    const int px = j == 0 ? NX - 1 : j - 1, nx = j == NX - 1 ? 0 : j + 1;
    const int py = kk == 0 ? NY - 1 : kk - 1, ny = kk == NY - 1 ? 0 : kk + 1;
    const int pz = l == 0 ? 1 : l - 1, nz = l + 1 == NZ ? NZ - 1 : l + 1;
    const uint8_t m[6] = {t.cmap2[gidx(t, px, kk, l)], t.cmap2[gidx(t, nx, kk, l)], t.cmap2[gidx(t, j, py, l)],
                          t.cmap2[gidx(t, j, ny, l)], t.cmap2[gidx(t, j, kk, pz)], t.cmap2[gidx(t, j, kk, nz)]};
    bits = (j == 0 ? CQ_XM : 0) | (j == NX - 1 ? CQ_XP : 0) | (kk == 0 ? CQ_YM : 0) | (kk == NY - 1 ? CQ_YP : 0) |
           (l == 0 ? CQ_ZM : 0) | (l + 1 == NZ ? CQ_ZP : 0);
    for (int q = 0; q < 6; q++) {
      if (m[q] > 1) bits |= CQ_SLOW;
      bits |= (unsigned)(m[q] & 1) << q;
    }
    word = t.vox[v];
  }
  return corner_pack(v, word, bits, raw);
}

// The ATP value of a cell's corner `k` after the ATP update that runs beside
// its launch, computed from the buffer before it (the grid kernel's expression,
// atp_new).  The corners of a cell are the points of a cube, so three of a
// corner's six stencil neighbours are the cube's other corners and come from
// their lanes (ix, iy, iz: across in x, y, z); the other three, the point
// itself and the owner's diff_u are loaded, without branches, so that the loads
// of the cell's entries can be issued behind them.  A corner that the update
// leaves alone takes its value from the buffer after it, in `ox`.
struct Corner { double c0, ox, oy, oz, diffu; };
template <class A>
__device__ __forceinline__ Corner corner_load(const A& a, int k, uint4 q) {
  const double* __restrict__ at = a.A0;
  const long long v = corner_at(q);
  const unsigned f = q.z;
  const bool hx = k & 1, hy = k & 2, hz = k & 4;
  const int dx = hx ? ((f & CQ_XP) ? 1 - a.NX : 1) : ((f & CQ_XM) ? a.NX - 1 : -1);
  const int wy = (a.NY - 1) * a.XP;   // only fused launches take corners so, and their planes are below 4 GB
  const int dy = hy ? ((f & CQ_YP) ? -wy : a.XP) : ((f & CQ_YM) ? wy : -a.XP);
  const long long dz = hz ? ((f & CQ_ZP) ? 0 : a.PL) : ((f & CQ_ZM) ? a.PL : -a.PL);
  const bool plain = f & CQ_PLAIN;
  const unsigned cell1 = q.y & 0x7fffffffu;
  Corner r;
  r.c0 = at[v];
  r.ox = *(plain ? a.A1 + v : at + v + dx);
  r.oy = at[plain ? v : v + dy];
  r.oz = at[plain ? v : v + dz];
  r.diffu = a.dfo[cell1 ? cell1 - 1 : 0];
  return r;
}
template <class A>
__device__ __forceinline__ double corner_new(const AtpK& ak, double inv_dx, const A& a, int k, uint4 q, const Corner& r,
                                             double ix, double iy, double iz) {
  const unsigned f = q.z;
  const bool hx = k & 1, hy = k & 2, hz = k & 4;
  const double c0 = r.c0;
  // next_z(NZ - 1) is the point itself (utils.cpp:32-72); such a point is the
  // upper corner (oz above) or, with its cell at the grid's top, the lower one
  const double izn = !hz && (f & CQ_ZP) ? c0 : iz;
  unsigned word = q.y;
  double diffu = (word & 0x7fffffffu) ? r.diffu : 0.0;
  double m[6];
#pragma unroll
  for (int b = 0; b < 6; b++) m[b] = (double)((f >> b) & 1);
  if (f & CQ_SLOW) {
    const uint8_t* __restrict__ cm2 = a.cm2;
    const long long v = corner_at(q), wy = (long long)(a.NY - 1) * a.XP;
    m[0] = cm2[v + ((f & CQ_XM) ? a.NX - 1 : -1)];
    m[1] = cm2[v + ((f & CQ_XP) ? 1 - a.NX : 1)];
    m[2] = cm2[v + ((f & CQ_YM) ? wy : -(long long)a.XP)];
    m[3] = cm2[v + ((f & CQ_YP) ? -wy : a.XP)];
    m[4] = cm2[v + ((f & CQ_ZM) ? a.PL : -a.PL)];
    m[5] = cm2[v + ((f & CQ_ZP) ? 0 : a.PL)];
  }
  const double nv = atp_new(ak, c0, hx ? ix : r.ox, hx ? r.ox : ix, hy ? iy : r.oy, hy ? r.oy : iy, hz ? iz : r.oz,
                            hz ? r.oz : izn, m[0], m[1], m[2], m[3], m[4], m[5], diffu, (double)(word >> 31), inv_dx);
  return (f & CQ_PLAIN) ? r.ox : nv;
}

}  // namespace epi
