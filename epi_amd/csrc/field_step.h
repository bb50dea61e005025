// field_step.h -- the two pieces of a step's field work that other launches
// may carry beside their own (k_field.hip, k_connect.hip): the stamping of
// the voxel maps (setup_map_lat, map.cpp:18-167) and the B stencil
// (calc_ext_stim, ext_stim.cpp:18-69).  Each is a function of a block's number
// and the number of blocks that share the work.
#pragma once
#include "epi_dev.h"

namespace epi {

__device__ __forceinline__ int lat_wrap(long v, int N, Status* st) {
  // precalc_lat_* hold i%N for i in [0, 3N) (utils.cpp:18-30)
  const long i = v + N;
  if (i < 0 || i >= 3L * N) { set_err(st, ERR_OUT_OF_GRID); return (int)(((i % N) + N) % N); }
  return (int)(i % N);
}
// the same for a box index that rarely leaves [0, N): no division there
__device__ __forceinline__ int lat_near(int v, int N, Status* st) {
  if (v >= 0 && v < N) return v;
  if (v < 0 && v >= -N) return v + N;
  if (v >= N && v < 2 * N) return v - N;
  return lat_wrap(v, N, st);
}

// set_lattice (:18-22), the sphere stamping (:39-155) and the periodic planes
// x = NX and y = NY (:156-166); the last writer of the serial loop is the
// highest cell index, hence atomicMax on cmap1.
//
// MS lanes per cell (1, 4 or 16, a launch shape) walk the stamp box x
// fastest, so a group's lanes write runs of consecutive x of one or two
// rows: a store or an atomic touches a few cache lines, where lanes a plane
// apart touched one line each (bound by those transactions and, on a small
// tissue, by the walk's length).  A voxel of row y = 0 or column x = 0 is
// written to its periodic copies too, which the clear has emptied, so no
// kernel copies the planes afterwards.  The result does not depend on MS (a
// max and idempotent stores).  16 lanes against the z-fastest walk with its
// default of one: 420 cells 39 -> 7.9 us, 36,000 cells 41 -> 16.5 us (23.9 with
// 16 lanes there), 32 uneven tissues of 290,000 cells 577 -> 175 us, and no
// copy kernel (5 to 23 us).
template <int MS>
__device__ __forceinline__ void map_stamp_part(const Tis& t, int pb, int bid, int nblk) {
  Status* st = t.st;
  const int zl = threadIdx.x & (MS - 1);
  const double FAC_MAP = t.prm.FAC_MAP;
  const int NX = t.NX, NY = t.NY, NZ = t.NZ, XP = t.XP;
  const long long PL = t.PL;
  const double dx = t.dx, dy = t.dy, dz = t.dz;
  int* __restrict__ cmap1 = t.cmap1;
  uint8_t* __restrict__ cmap2 = t.cmap2;
  int ztop = 0;
  const int cap = t.cap;
  int c = (bid * blockDim.x + threadIdx.x) / MS;
  // the first cell's words are loaded in one round trip with the cell count
  // (a cell past the count reads allocated, stale slots)
  const int c0 = c < cap ? c : cap - 1;
  P3 p = ld_pos(t, pb, c0);
  uint8_t s = t.state[c0];
  double r = t.radius[c0];
  const int n = st->n;
  const int step = nblk * blockDim.x / MS;
  for (; c < n; c += step) {
    const int lx = lat_wrap((long)(int)(p.x * t.inv_dx), NX, st);
    const int ly = lat_wrap((long)(int)(p.y * t.inv_dy), NY, st);
    const int lz = lat_wrap((long)(int)(p.z * t.inv_dz), NZ, st);
    if (zl == 0) { t.lat[3 * c] = lx; t.lat[3 * c + 1] = ly; t.lat[3 * c + 2] = lz; }
    const bool afm = is_afm(s);
    const int irx = afm ? 2 * t.irx : t.irx, iry = afm ? 2 * t.iry : t.iry, irz = afm ? 2 * t.irz : t.irz;
    const double normal_radSq = r * r;
    const double crad = FAC_MAP * r;
    const double cradSq = crad * crad;
    const int z_b = lz - irz, z_u = lz + irz;
    const int zmin = z_b >= 1 ? z_b : 1;
    const int zmax = z_u < NZ ? z_u : NZ - 1;
    ztop = max(ztop, zmax);
    const int nzr = zmax - zmin + 1;
    const int bx = 2 * irx + 1, by = 2 * iry + 1;
    if (nzr <= 0) {   // no plane to stamp: the box's x and y range is still checked
      if (zl == 0) {
        for (int k = lx - irx; k <= lx + irx; k++) lat_wrap(k, NX, st);
        for (int l = ly - iry; l <= ly + iry; l++) lat_wrap(l, NY, st);
      }
    } else {
      // the zl-th voxel of the box, then every MS-th: (ix, iy, iz) with ix
      // fastest, advanced by MS's own digits in that radix
      const int sx = MS % bx, sy = MS / bx % by, sz = MS / (bx * by);
      int ix = zl % bx, iy = zl / bx % by, iz = zl / (bx * by);
      while (iz < nzr) {
        const int k = lx - irx + ix, l = ly - iry + iy, m = zmin + iz;
        const double diffx = p_diff_x(t, k * dx, p.x);
        const double diffy = p_diff_y(t, l * dy, p.y);
        const double diffz = m * dz - p.z;
        const int ipx = lat_near(k, NX, st), ipy = lat_near(l, NY, st);
        const double distSq = diffx * diffx + diffy * diffy + diffz * diffz;
        const bool in1 = distSq < normal_radSq, in2 = afm && distSq < cradSq;
        const bool mark = afm ? in1 && in2 : in1;
        if (in2 || mark) {
          // a plane has fewer than 2^32 points (a grid of three such planes does
          // not fit the card), so the place within it is unsigned 32 bits
          const long long v = (long long)m * PL + ((unsigned)ipy * (unsigned)XP + (unsigned)ipx);
          // the voxel, and its copies in the planes x = NX, y = NY
          for (int copy = 0; copy < 4; copy++) {
            if (((copy & 1) && ipx != 0) || ((copy & 2) && ipy != 0)) continue;
            const long long w = v + ((copy & 1) ? NX : 0) + ((copy & 2) ? (long long)NY * XP : 0);
            if (in2) cmap2[w] = 1;
            if (mark) atomicMax(&cmap1[w], c);
            if (ipx != 0 && ipy != 0) break;
          }
        }
        ix += sx; iy += sy; iz += sz;
        if (ix >= bx) { ix -= bx; iy++; }
        if (iy >= by) { iy -= by; iz++; }
      }
    }
    const int cn = c + step;
    if (cn < n) { p = ld_pos(t, pb, cn); s = t.state[cn]; r = t.radius[cn]; }
  }
  for (int o = 32; o > 0; o >>= 1) ztop = max(ztop, __shfl_down(ztop, o, 64));
  if ((threadIdx.x & 63) == 0 && ztop > __hip_atomic_load(&st->stamp_z, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax(&st->stamp_z, ztop);
}

// ---- ext_stim B: calc_ext_stim (ext_stim.cpp:18-69) ------------------------
struct BK {   // fB's constants, copied out of the record before any store (see CaK)
  double THRESH_DEAD, DUR_ALIVE, DUR_DEAD, kb;
};
__device__ __forceinline__ BK b_k(const Params& pm) { return BK{pm.THRESH_DEAD, pm.DUR_ALIVE, pm.DUR_DEAD, pm.kb}; }
__device__ __forceinline__ double fB(const BK& k, double age, double B, bool cornif) {   // :9-16
  return (cornif && age > k.THRESH_DEAD - k.DUR_ALIVE && age <= k.THRESH_DEAD + k.DUR_DEAD ? 1 : 0) - k.kb * B;
}

// exclusive prefix sum of v over a block of blockDim.x (a multiple of 64,
// at most 1024) threads; returns the block total in *total
__device__ __forceinline__ int block_exclusive_scan(int v, int* total) {
  __shared__ int s_w[16];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) s_w[wv] = x;
  __syncthreads();
  int before = 0, all = 0;
  for (int i = 0; i < nw; i++) {
    const int w = s_w[i];
    if (i < wv) before += w;
    all += w;
  }
  __syncthreads();
  *total = all;
  return before + x - v;
}

// The B stencil's iz_bound = (int)((zzmax + FAC_MAP * R_max) * inv_dz)
// (ext_stim.cpp:22) from the device's zzmax.  One outside [0, NZ] sweeps
// nothing and is reported as ERR_OUT_OF_GRID; the sweep's NX NY iz_bound
// points are added to the tissue's count (both by the thread that counts).
__device__ __forceinline__ int b_iz_bound(const Tis& t, bool counts) {
  const double zzmax = __longlong_as_double((long long)t.st->zzmax_bits);
  int izb = (int)((zzmax + t.prm.iz_margin) * t.inv_dz);
  if (izb > t.NZ || izb < 0) {
    if (counts) set_err(t.st, ERR_OUT_OF_GRID);
    izb = 0;
  }
  if (counts) t.st->grid_b += (long long)t.NX * t.NY * izb;
  return izb;
}

// Tiles of a work list for this block: a grid-stride loop.  With `xcd` (and
// a grid that is a multiple of 8) the list is cut into 8 contiguous runs,
// one per XCD (workgroups go to the XCDs round-robin by id), so that tiles
// that share halo rows share an L2.
struct TileWalk {
  int w, end, stride;
  // block b of G walking the list (b = blockIdx.x, G = gridDim.x unless the
  // launch shares its grid with other work)
  __device__ TileWalk(int total, int xcd, int b, int G) {
    if (xcd && G >= 8 && (G & 7) == 0) {
      const int seg = (total + 7) / 8, x = b & 7;
      w = x * seg + (b >> 3);
      end = min(total, (x + 1) * seg);
      stride = G >> 3;
    } else {
      w = b;
      end = total;
      stride = G;
    }
  }
};

// One (x, y) column of a tile: planes l0 .. l1 - 1, at most ZB of them.
// Every load of the column is issued before any value is used: the column's
// own planes l0 - 1 .. l1 (mirror prev_z(0) = 1, self next_z(NZ - 1) =
// NZ - 1, utils.cpp:32-72), then each plane's four lateral neighbours, masks
// and voxel cell, then the cells' states and ages.  So a tile waits for three
// memory round trips, not three per plane.  The arithmetic is
// ext_stim.cpp:36-57's, in its order.
template <int ZB>
__device__ __forceinline__ void b_column(const Tis& t, int j, int k, int l0, int l1, int bp) {
  const int NX = t.NX, NY = t.NY, NZ = t.NZ;
  const BK bk = b_k(t.prm);
  const double DB = t.prm.DB, DT_Ca = t.prm.DT_Ca;
  const double* __restrict__ carr = t.bf[bp];
  double* __restrict__ narr = t.bf[1 - bp];
  const uint8_t* __restrict__ cm2 = t.cmap2;
  const int prev_x = j == 0 ? NX - 1 : j - 1, next_x = j == NX - 1 ? 0 : j + 1;
  const int prev_y = k == 0 ? NY - 1 : k - 1, next_y = k == NY - 1 ? 0 : k + 1;
  const long long PL = t.PL;
  const long long cxy = gidx(t, j, k, 0);
  const int nl = l1 - l0;
  double cz[ZB + 2];
  uint8_t mz[ZB + 2];
#pragma unroll
  for (int q = 0; q < ZB + 2; q++) {
    int l = q == 0 ? (l0 == 0 ? 1 : l0 - 1) : l0 + q - 1;
    if (l > NZ - 1) l = NZ - 1;
    cz[q] = 0;
    mz[q] = 0;
    if (q <= nl + 1) {
      cz[q] = carr[cxy + l * PL];
      mz[q] = cm2[cxy + l * PL];
    }
  }
  double xm[ZB], xp[ZB], ym[ZB], yp[ZB];
  uint8_t mxm[ZB], mxp[ZB], mym[ZB], myp[ZB];
  int cell[ZB];
#pragma unroll
  for (int q = 0; q < ZB; q++) {
    xm[q] = xp[q] = ym[q] = yp[q] = 0;
    mxm[q] = mxp[q] = mym[q] = myp[q] = 0;
    cell[q] = -1;
    if (q < nl) {
      const int l = l0 + q;
      const long long vxm = gidx(t, prev_x, k, l), vym = gidx(t, j, prev_y, l);
      const long long vyp = gidx(t, j, next_y, l), vxp = gidx(t, next_x, k, l);
      xm[q] = carr[vxm]; ym[q] = carr[vym]; yp[q] = carr[vyp]; xp[q] = carr[vxp];
      mxm[q] = cm2[vxm]; mym[q] = cm2[vym]; myp[q] = cm2[vyp]; mxp[q] = cm2[vxp];
      cell[q] = t.cmap1[cxy + l * PL];
    }
  }
  // a voxel's state and age are read together (the age of a cell that is
  // neither DEAD nor ALIVE is then dropped), one round trip after the map
  uint8_t cs[ZB];
  double age[ZB];
#pragma unroll
  for (int q = 0; q < ZB; q++) {
    cs[q] = MEMB;
    age[q] = 0.0;
    if (cell[q] >= 0) {
      cs[q] = t.state[cell[q]];
      age[q] = t.agek[cell[q]];
    }
  }
#pragma unroll
  for (int q = 0; q < ZB; q++) age[q] = (cs[q] == DEAD || cs[q] == ALIVE) ? age[q] : 0.0;
  const double inv_dz = t.inv_dz;
#pragma unroll
  for (int q = 0; q < ZB; q++) {
    if (q < nl) {
      const int l = l0 + q;
      const bool flg = cs[q] == DEAD || cs[q] == ALIVE;
      const double cext = cz[q + 1];
      const double nv = cext + DT_Ca * (DB *
          ((double)mxm[q] * (xm[q] - cext)
           + (double)mym[q] * (ym[q] - cext)
           + (double)mz[q] * (cz[q] - cext)
           + (double)mz[q + 2] * (cz[q + 2] - cext)
           + (double)myp[q] * (yp[q] - cext)
           + (double)mxp[q] * (xp[q] - cext))
          * inv_dz * inv_dz + fB(bk, age[q], cext, flg));
      narr[cxy + l * PL] = nv;
      // periodic copies (:63-66)
      if (k == 0) narr[gidx(t, j, NY, l)] = nv;
      if (j == 0) narr[gidx(t, NX, k, l)] = nv;
      if (j == 0 && k == 0) narr[gidx(t, NX, NY, l)] = nv;
    }
  }
}

// The same column with the z column rolling through registers, one plane
// after the other: three values and masks live at a time, so a tile of many
// planes keeps the registers (and occupancy) of one.  Large tiles, where the
// sweep is bandwidth- and not latency-bound, take this form.  The voxel's
// cell is read one plane ahead and its state and age together, so a plane
// waits for one memory round trip, not for the chain map -> state -> age.
__device__ __forceinline__ void b_column_roll(const Tis& t, int j, int k, int l0, int l1, int bp) {
  const int NX = t.NX, NY = t.NY, NZ = t.NZ;
  const BK bk = b_k(t.prm);
  const double DB = t.prm.DB, DT_Ca = t.prm.DT_Ca;
  const double* __restrict__ carr = t.bf[bp];
  double* __restrict__ narr = t.bf[1 - bp];
  const uint8_t* __restrict__ cm2 = t.cmap2;
  const int* __restrict__ cm1 = t.cmap1;
  const uint8_t* __restrict__ cst = t.state;
  const double* __restrict__ cage = t.agek;
  const int prev_x = j == 0 ? NX - 1 : j - 1, next_x = j == NX - 1 ? 0 : j + 1;
  const int prev_y = k == 0 ? NY - 1 : k - 1, next_y = k == NY - 1 ? 0 : k + 1;
  const double inv_dz = t.inv_dz;
  const long long PL = t.PL;
  const long long cxy = gidx(t, j, k, 0);
  const int pz = l0 == 0 ? 1 : l0 - 1;   // mirror z (utils.cpp:32-72)
  double czm = carr[cxy + pz * PL];
  int mzm = cm2[cxy + pz * PL];
  double cc = carr[cxy + l0 * PL];
  int mc = cm2[cxy + l0 * PL];
  int cell = l0 < l1 ? cm1[cxy + l0 * PL] : -1;
  for (int l = l0; l < l1; l++) {
    const int next_z = l + 1 == NZ ? NZ - 1 : l + 1;
    const long long v = cxy + l * PL;
    const long long vzp = cxy + next_z * PL;
    const double czp = carr[vzp];
    const int mzp = cm2[vzp];
    const int cell_next = l + 1 < l1 ? cm1[v + PL] : -1;
    uint8_t s = MEMB;
    double a = 0;
    if (cell >= 0) {
      s = cst[cell];
      a = cage[cell];
    }
    const bool flg = s == DEAD || s == ALIVE;
    const double dum_age = flg ? a : 0.0;
    const double cext = cc;
    const long long vxm = gidx(t, prev_x, k, l), vym = gidx(t, j, prev_y, l);
    const long long vyp = gidx(t, j, next_y, l), vxp = gidx(t, next_x, k, l);
    const double nv = cext + DT_Ca * (DB *
        ((double)cm2[vxm] * (carr[vxm] - cext)
         + (double)cm2[vym] * (carr[vym] - cext)
         + (double)mzm * (czm - cext)
         + (double)mzp * (czp - cext)
         + (double)cm2[vyp] * (carr[vyp] - cext)
         + (double)cm2[vxp] * (carr[vxp] - cext))
        * inv_dz * inv_dz + fB(bk, dum_age, cext, flg));
    narr[v] = nv;
    if (k == 0) narr[gidx(t, j, NY, l)] = nv;
    if (j == 0) narr[gidx(t, NX, k, l)] = nv;
    if (j == 0 && k == 0) narr[gidx(t, NX, NY, l)] = nv;
    czm = cc; mzm = mc;
    cc = czp; mc = mzp;
    cell = cell_next;
  }
}

// One tile of the B stencil: one thread per (x, y) point; tiles of up to 2
// planes load the column first (b_column), taller ones roll it
// (b_column_roll).
template <int ZB>
__device__ __forceinline__ void b_tile(const Tis& t, int local, int iz_bound, int bp) {
  const int bs = blockDim.x;
  const int NX = t.NX, plane = NX * t.NY;
  const int npt = (plane + bs - 1) / bs;
  const int p = (local % npt) * bs + (int)threadIdx.x;
  if (p >= plane) return;
  const int l0 = (local / npt) * ZB;
  const int l1 = min(l0 + ZB, iz_bound);
  if (ZB >= 4) b_column_roll(t, p % NX, p / NX, l0, l1, bp);
  else b_column<ZB>(t, p % NX, p / NX, l0, l1, bp);
}

// The B stencil of one tissue by nblk blocks: its tiles follow from its
// iz_bound, which every block takes from zzmax itself, so no list is built
// (k_wl_b, a launch of one block, 4 to 5 us) nor read.  The first block's first
// thread does k_wl_b's share.
template <int ZB>
__device__ __forceinline__ void ext_stim_part(const Tis& t, int bp, int xcd, int bid, int nblk) {
  const int iz_bound = __builtin_amdgcn_readfirstlane(b_iz_bound(t, bid == 0 && threadIdx.x == 0));
  const int total = ((t.NX * t.NY + (int)blockDim.x - 1) / (int)blockDim.x) * ((iz_bound + ZB - 1) / ZB);
  for (TileWalk tw(total, xcd, bid, nblk); tw.w < tw.end; tw.w += tw.stride) b_tile<ZB>(t, tw.w, iz_bound, bp);
}

}  // namespace epi
