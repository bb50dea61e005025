// k_field.hip -- setup_map_lat (map.cpp:18-167), calc_ext_stim
// (ext_stim.cpp:18-69) and calc_ca2p (ca2p.cpp:14-402) on CDNA4.
//
// Grids are z-major with x fastest (x pitch padded to 16 doubles), so a
// wavefront reads 64 consecutive x points of one (y, z) row.  The stencils
// map threads to (x, y) columns and march z in chunks of ZB planes (a
// template parameter; the y rows per block are a launch parameter, both set
// by the autotuner); the number of active planes (iz_bound) is derived on the
// device from zzmax and the z chunks are grid-strided, so no host round trip
// is needed.
#include <algorithm>
#include <type_traits>

#include "epi_dev.h"
#include "launch.h"
#include "epi_group.h"
#include "ca_laws.h"
#include "ca_corner.h"
#include "rd_dev.h"
#include "field_step.h"

namespace epi {

// ---- voxel maps ---------------------------------------------------------
// Only planes 0..stamp_z can hold stamps (stamp_z never decreases), so only
// they are cleared; the rest of the maps stays empty from the first build.
// In a step the bucket insertion's spare blocks do it (map_clear, epi_dev.h).
__global__ void __launch_bounds__(256) k_map_clear(const Tis* __restrict__ T) {
  map_clear(T[blockIdx.y], blockIdx.x, gridDim.x);
}

template <int MS>
__global__ void __launch_bounds__(128) k_map_stamp(const Tis* __restrict__ T, int pb) {
  map_stamp_part<MS>(T[blockIdx.y], pb, blockIdx.x, gridDim.x);
}

// ---- flattened work lists ------------------------------------------------
// A launch over tissues of different sizes numbers the tiles of all of them
// consecutively, tissue by tissue: off[i] is the first tile of the launch's
// i-th tissue and off[nt] the total.  A tile is a chunk of `bs` consecutive
// points of the tissue's (x, y) plane (x fastest, so a wave's lanes read
// consecutive x of one or two rows) times a chunk of ZB z planes, plane
// chunks fastest.  No lane covers a point outside its tissue except in the
// last plane chunk, and no block is launched for a tissue that has no work.

// The B stencil's list, once zzmax is on the device: per tissue iz_bound into
// izb[i], and ceil(NX NY / bs) ceil(iz_bound / zb) tiles.  One block.
__global__ void __launch_bounds__(256) k_wl_b(const Tis* __restrict__ T, int ntis, int bs, int zb,
                                              int* __restrict__ off, int* __restrict__ izb_out) {
  int carry = 0;
  for (int base = 0; base < ntis; base += blockDim.x) {
    const int i = base + threadIdx.x;
    int cnt = 0;
    if (i < ntis) {
      const Tis& t = T[i];
      const int izb = b_iz_bound(t, true);
      izb_out[i] = izb;
      cnt = ((t.NX * t.NY + bs - 1) / bs) * ((izb + zb - 1) / zb);
    }
    int tot;
    const int ex = block_exclusive_scan(cnt, &tot);
    if (i < ntis) off[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) off[ntis] = carry;
}

// the launch's tissue of tile w: the last i in [lo, nt) with off[i] <= w
template <class F>
__device__ __forceinline__ int wl_find(F off, int lo, int nt, int w) {
  int hi = nt - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off(mid) <= w) lo = mid; else hi = mid - 1;
  }
  return lo;
}

constexpr int WL_LDS_T = 1024;   // tissues whose list a block stages in LDS

// The B stencil over its tile list.
template <int ZB>
__global__ void __launch_bounds__(256) k_ext_stim(const Tis* __restrict__ T, const int* __restrict__ woff,
                                                  const int* __restrict__ wizb, int ntis, int bp, int xcd) {
  __shared__ int s_off[WL_LDS_T + 1];
  __shared__ int s_izb[WL_LDS_T];
  const bool lds = ntis <= WL_LDS_T;
  if (lds) {
    for (int i = threadIdx.x; i <= ntis; i += blockDim.x) {
      s_off[i] = woff[i];
      if (i < ntis) s_izb[i] = wizb[i];
    }
    __syncthreads();
  }
  auto off = [&](int i) { return lds ? s_off[i] : woff[i]; };
  int ti = 0;
  for (TileWalk tw(off(ntis), xcd, blockIdx.x, gridDim.x); tw.w < tw.end; tw.w += tw.stride) {
    // the tile, hence its tissue, is the block's: held in scalar registers,
    // so the tissue's record is read with scalar loads
    ti = __builtin_amdgcn_readfirstlane(wl_find(off, ti, ntis, tw.w));
    b_tile<ZB>(T[ti], tw.w - __builtin_amdgcn_readfirstlane(off(ti)),
               __builtin_amdgcn_readfirstlane(lds ? s_izb[ti] : wizb[ti]), bp);
  }
}

// The B stencil of one tissue (ext_stim_part)
template <int ZB>
__global__ void __launch_bounds__(256) k_ext_stim_one(const Tis* __restrict__ T, int bp, int xcd) {
  ext_stim_part<ZB>(T[0], bp, xcd, blockIdx.x, gridDim.x);
}

// ---- calc_ca2p ------------------------------------------------------------
// init_ca2p_avg (:20-27), the per-cell "touches AIR" flag used by
// init_ca2p_map (:262-268), the (ca2p, IP3) pairs, the packed coupled entries
// and the constants of the Ca laws.  BL lanes per cell take its list BL
// entries at a time: the neighbours' states in one gather, the coupled entries
// placed by a ballot (one lane walking the list waited for two round trips per
// entry: 27 us for lists of up to 40).
constexpr int BL = 16;
__global__ void __launch_bounds__(256) k_ca_begin(const Tis* __restrict__ T, const int* tlist, int cb, int zero_avg) {
  const Tis& t = T[tlist ? tlist[blockIdx.y] : blockIdx.y];
  const int n = t.st->n;
  const int start = t.nmemb + t.nder;
  const int lane = threadIdx.x & (BL - 1);
  // the constants are read before any store (see CaK)
  const Params& pm = t.prm;
  const double thgra = pm.thgra, thpri = pm.thpri, delta_th = pm.delta_th, TSP = pm.THRESH_SP;
  const double kpa = pm.kpa, Kpri = pm.Kpri, delta_K = pm.delta_K, delta_I = pm.delta_I, ik = pm.iage_kitei;
  for (int c = (blockIdx.x * blockDim.x + threadIdx.x) / BL; c < n; c += gridDim.x * blockDim.x / BL) {
    const int* row = t.col[cb] + (size_t)c * t.ns;
    const int len = t.nlen[cb][c];
    const uint8_t s = t.state[c];
    const bool afm = c >= start && is_afm(s), takes = afm || (c >= start && s == DEAD);
    const double* g = t.gj[cb] + (size_t)c * t.ns;
    const size_t at = (size_t)c * t.ns;
    bool air = false;
    int k = 0;
    for (int e0 = 0; e0 < len; e0 += BL) {
      const int e = e0 + lane;
      const int o = e < len ? row[e] : -1;
      const uint8_t so = o >= 0 ? t.state[o] : MEMB;
      const double gv = o >= 0 && takes ? g[e] : 0.0;
      air = air || so == AIR;
      // which entries take part in the gap-junction sums (supra_calc
      // :201-209; dead_IP3_calc :160-165 counts the ALIVE ones)
      const int kd = so == ALIVE ? 3 : (so == DEAD || so == FIX || so == MUSUME) ? 1 : 0;
      const unsigned m = (unsigned)(__ballot(takes && kd) >> (threadIdx.x & 48)) & 0xffffu;
      if (takes && kd) {
        const size_t i = at + k + __popc(m & ((1u << lane) - 1));
        t.ca_w[i] = (o << 2) | kd;
        t.ca_sl[i] = (unsigned short)e;
        t.ca_g[i] = gv;
      }
      k += __popc(m);
    }
    const bool any_air = ((__ballot(air) >> (threadIdx.x & 48)) & 0xffffu) != 0;
    if (lane != 0) continue;
    t.touch_air[c] = any_air;
    t.ca_cn[c] = k;
    t.ca_up[0][c] = make_double2(t.ca2p[0][c], t.ip3[0][c]);
    t.ca_up[1][c] = make_double2(t.ca2p[1][c], t.ip3[1][c]);
    if (!afm) continue;
    // calc_th, calc_Kpa, calc_IAG (ca2p.cpp:90-126): agek and state do
    // not change during a solve
    const bool is_alive = s == ALIVE;
    const double agek = t.agek[c];
    if (zero_avg) t.ca2p_avg[c] = 0;
    t.ca_th[c] = is_alive ? thgra + ((thpri - thgra) * 0.5) * (1.0 + tanh((TSP - agek) / delta_th)) : thpri;
    t.ca_kpa[c] = is_alive ? kpa + ((Kpri - kpa) * 0.5) * (1.0 + tanh((TSP - agek) / delta_K)) : Kpri;
    t.ca_iag[c] = is_alive ? 0.5 * (1.0 + tanh((agek - TSP) / delta_I)) : ik;
  }
}

// init_ca2p_map (:238-278): per voxel of the active box the AFM owner
// (+1, 0 = the dummy zero) and the air flag in bit 31; and the masks of its
// neighbours (ATP_refresh's, :302-338), which do not change during a solve
__global__ void __launch_bounds__(256) k_ca_vox(const Tis* __restrict__ T, const int* tlist) {
  const Tis& t = T[tlist ? tlist[blockIdx.y] : blockIdx.y];
  const int izb = ca_iz_bound(t);
  const int NX = t.NX, NY = t.NY, NZ = t.NZ;
  if (izb > NZ || izb < 0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) set_err(t.st, ERR_OUT_OF_GRID);
    return;
  }
  const unsigned plane = (unsigned)NX * NY;
  for (int l = blockIdx.z; l < izb; l += gridDim.z) {
    const int pz = l == 0 ? 1 : l - 1, nz = l + 1 == NZ ? NZ - 1 : l + 1;
    for (unsigned p = blockIdx.x * blockDim.x + threadIdx.x; p < plane; p += gridDim.x * blockDim.x) {
      const int k = (int)div_by(p, NX, t.mg_nx), j = (int)(p - (unsigned)k * NX);
      const long long v = gidx(t, j, k, l);
      const int c = t.cmap1[v];
      unsigned w = 0;
      if (c >= 0) w = (is_afm(t.state[c]) ? (unsigned)(c + 1) : 0u) | ((unsigned)t.touch_air[c] << 31);
      t.vox[v] = w;
      const uint8_t* __restrict__ m2 = t.cmap2;
      const uint8_t m[6] = {m2[gidx(t, j == 0 ? NX - 1 : j - 1, k, l)], m2[gidx(t, j == NX - 1 ? 0 : j + 1, k, l)],
                            m2[gidx(t, j, k == 0 ? NY - 1 : k - 1, l)], m2[gidx(t, j, k == NY - 1 ? 0 : k + 1, l)],
                            m2[gidx(t, j, k, pz)], m2[gidx(t, j, k, nz)]};
      unsigned bits = 0;
      for (int q = 0; q < 6; q++) bits |= m[q] > 1 ? VMK_SLOW : (unsigned)m[q] << q;
      t.vmk[v] = (uint8_t)bits;
    }
  }
}

// Workgroups go to the 8 XCDs round-robin by linear id.  With `on`, the
// linear id is renumbered so that each XCD runs one contiguous run of logical
// ids (a bijection for any grid size): neighbouring cells and grid rows then
// share an L2.  Results do not depend on it.
__device__ __forceinline__ unsigned xcd_order(unsigned L, unsigned G, int on) {
  if (!on) return L;
  const unsigned q = G >> 3, r = G & 7, x = L & 7;
  return x * q + min(x, r) + (L >> 3);
}

// diff_u of a sub-step by Ca parity: the sub-step at parity cp writes it and
// its ATP update reads it, so a fused launch (ATP of one sub-step beside the
// cells of the next) reads one buffer while it writes the other.

// What a launch of the Ca kernels reads and writes of one tissue, resolved from
// its descriptor and the parities.  A one-tissue launch carries it by value,
// as kernel arguments: its waves then start on the cells' words without first
// fetching pointers through the descriptor (a round trip of the five a
// sub-step's cells wait for).  The laws' constants stay in the descriptor: they
// are needed late, and by value they would be held in scalar registers from
// the start, more of them than a wave has.
struct CaArg {
  const Status* st;
  const uint8_t* state;
  const int* cn;
  const int* w;
  double* g;
  const double2* up;      // (ca2p, IP3) before the sub-step
  double2* upn;           // and after it
  const double* dfo;      // diff_u that the ATP update and the recomputed corners read
  double* dfn;            // diff_u that the cells write
  const uint4* cq;
  const double *th, *kpa, *iag, *bx;
  double *exi, *avg;
  const double* A0;       // ATP before the launch's ATP update
  double* A1;             // and after it
  const uint8_t* cm2;
  const unsigned* vox;
  const uint8_t* vmk;
  long long PL;
  int start, cap, ns, NX, NY, NZ, XP;
  unsigned mg_nx;
};
// cells at Ca parity cpc; the ATP update of the sub-step at Ca parity cpa from
// ATP buffer ap
__host__ __device__ __forceinline__ CaArg ca_arg(const Tis& t, int cpc, int cpa, int ap) {
  CaArg a;
  a.st = t.st; a.state = t.state; a.cn = t.ca_cn; a.w = t.ca_w; a.g = t.ca_g;
  a.up = t.ca_up[cpc]; a.upn = t.ca_up[1 - cpc];
  a.dfo = cpa ? t.ca_dfu : t.diff_u; a.dfn = cpc ? t.ca_dfu : t.diff_u;
  a.cq = t.ca_cq; a.th = t.ca_th; a.kpa = t.ca_kpa; a.iag = t.ca_iag; a.bx = t.ca_bx;
  a.exi = t.ex_inert; a.avg = t.ca2p_avg; a.A0 = t.atp[ap]; a.A1 = t.atp[1 - ap];
  a.cm2 = t.cmap2; a.vox = t.vox; a.vmk = t.vmk; a.PL = t.PL; a.mg_nx = t.mg_nx;
  a.start = t.nmemb + t.nder; a.cap = t.cap; a.ns = t.ns;
  a.NX = t.NX; a.NY = t.NY; a.NZ = t.NZ; a.XP = t.XP;
  return a;
}

// The voxel map, the masks, B and iz_bound do not change during a solve, so
// each AFM cell keeps, for all of its sub-steps, its ca2p_by_ext_stim and, of
// its eight grid_avg8 corners, the point, its voxel word, neighbour masks and
// where the stencil wraps.  One lane per (cell, corner), after k_ca_vox.
__global__ void __launch_bounds__(256) k_ca_corners(const Tis* __restrict__ T, const int* tlist, int bp) {
  const Tis& t = T[tlist ? tlist[blockIdx.y] : blockIdx.y];
  const int n = t.st->n;
  const int start = t.nmemb + t.nder;
  const int izb = ca_iz_bound(t);
  const CaK ck = ca_k(t.prm);
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < 8LL * n;
       i += (long long)gridDim.x * blockDim.x) {
    const int c = (int)(i >> 3), k = (int)(i & 7);
    if (c < start || !is_afm(t.state[c])) continue;
    const int x = t.lat[3 * c], y = t.lat[3 * c + 1], z = t.lat[3 * c + 2];
    const double b = t.bf[bp][gidx(t, x + (k & 1), y + ((k >> 1) & 1), z + (k >> 2))];
    t.ca_cq[i] = corner_word(t, izb, x, y, z, k);
    // grid_avg8 (utils.h:18-23) of B in its order: 000 100 010 001 110 101 011 111
    const double sum = __shfl(b, 0, 8) + __shfl(b, 1, 8) + __shfl(b, 2, 8) + __shfl(b, 4, 8) + __shfl(b, 3, 8) +
                       __shfl(b, 5, 8) + __shfl(b, 6, 8) + __shfl(b, 7, 8);
    if (k == 0) t.ca_bx[c] = ca2p_by_ext(ck, 0.125 * sum);
  }
}

// corner_new of the cell's corner `k` (its lane is k): the cube's other corners
// come from their lanes
__device__ __forceinline__ double corner_value(const Tis& t, const CaArg& a, int k, uint4 q, const Corner& r) {
  const double c0 = r.c0;
  return corner_new(atp_k(t.prm), t.inv_dx, a, k, q, r, __shfl_xor(c0, 1, 64), __shfl_xor(c0, 2, 64), __shfl_xor(c0, 4, 64));
}

// dead_IP3_calc (:156-173) and supra_calc (:182-222).  A group of CG lanes (8
// or 16) owns one cell: lanes evaluate the gap-junction terms of the packed
// coupled entries (and update gj toward ALIVE neighbours) 32 at a time, and the
// first eight take one grid_avg8 corner of ATP each; two lanes sum the
// terms in list order, one the Ca2+ and one the IP3 side.  Each group takes
// one cell, so the grid must cover every cell past the membrane and dermis (a
// launch that does not is reported as ERR_INVALID); a loop over cells would
// keep loop-invariant constants of the math in registers for the whole kernel
// and cost a wave per SIMD.
//
// What bounds it: the chain of round trips through the Infinity Cache (what
// the other XCDs wrote is in no local L2 after a launch) and, on a large
// tissue, the cache lines its gathers touch.  So everything that depends on
// the cell alone is loaded in the first round trip (a lane each for the six
// per-cell values), the entries' pairs and the corners' neighbours in the
// second, and nothing after them; gj sits beside the entries instead of in the
// list row's slots; the quotients of the reaction terms that depend on the
// cell alone are one division, a lane each, while the gathers fly, and the two
// that do not are another one.  Per fused sub-step, against the same split
// with the row's slots, B read anew, all corners read by every lane and a
// leader's own loads and divisions (8 lanes, one-plane tiles): 17,500 AFM
// cells 11.3 -> 10.2 us, 700 cells 7.1 -> 5.7 us (with 16 lanes 6.4 -> 5.6, and
// 11.3 on the large tissue, so 8 is the default).
//
// With REC, the ATP corners are computed from the buffer before the ATP update
// that runs beside this launch (corner_recomputed), else read.
// With SAVE (a reaction-diffusion window's reverse pass), the cell also
// writes what the reverse sub-step reads of the state before it into segment
// slot `slot`: ca2p and IP3 (AFM and DEAD cells), ex_inert, the ATP
// grid_avg8 and the gj of its coupled entries (AFM cells).
constexpr int C_BLOCK = 128;

template <int CG, bool REC, bool SAVE>
__device__ __forceinline__ void ca_cells_part(const Tis& t, const CaArg& a, unsigned bx, unsigned nbx,
                                              const RdTis* __restrict__ sv, int slot) {
  constexpr int C_GROUPS = C_BLOCK / CG;
  constexpr int CCAP = 32;          // entries per chunk: more than nearly every cell has
  constexpr int EPL = CCAP / CG;    // of them per lane
  static_assert(CG >= 8 && EPL * CG == CCAP && CCAP <= ROW_SLOTS_MIN, "eight corner lanes, whole chunks inside a row");
  // per-entry terms for the summing lanes, corners, and the per-cell values
  // and quotients; rows padded so that the groups of a wave read different banks
  __shared__ double2 s_a[C_GROUPS][CCAP + 1];
  __shared__ double s_g[C_GROUPS][9];
  __shared__ double s_v[C_GROUPS][11];
  const int lane = threadIdx.x & (CG - 1);
  const int grp = threadIdx.x / CG;
  const int c = a.start + bx * C_GROUPS + grp;
  if (c >= a.cap) return;
  // First round trip: the cell's own words, its first chunk's entries and its
  // corners' words, beside the cell count (a device value).  A cell past the
  // count reads allocated, stale slots and leaves once the count is in; a row
  // holds ns >= ROW_SLOTS_MIN slots, and entries past len are masked.
  const uint8_t s = a.state[c];
  const int len = a.cn[c];
  const double2 uc = a.up[c];
  const size_t row = (size_t)c * a.ns;
  int en[EPL];
  double gv[EPL];
#pragma unroll
  for (int i = 0; i < EPL; i++) { en[i] = a.w[row + lane + i * CG]; gv[i] = a.g[row + lane + i * CG]; }
  uint4 q = a.cq[8 * (size_t)c + (lane & 7)];
  const double* __restrict__ vp =
      lane == 0 ? a.th : lane == 1 ? a.kpa : lane == 2 ? a.iag : lane == 3 ? a.bx : lane == 4 ? a.exi : a.avg;
  const double val = vp[c];
  const int n = a.st->n;
  if (bx == 0 && threadIdx.x == 0 && a.start + (long long)nbx * C_GROUPS < n) set_err(t.st, ERR_INVALID);
  if (c >= n) return;
  const bool dead = s == DEAD;
  if (!dead && !is_afm(s)) return;
  // Second round trip: the corners' points and the entries' pairs.  A DEAD
  // cell has no corners (its words may never have been written): point 0, as
  // it lies.
  if (dead) q = corner_none();
  Corner cr;
  double raw = 0;
  if (REC) cr = corner_load(a, lane & 7, q);
  else raw = a.A0[corner_raw(q)];
  double2 w[EPL];
#pragma unroll
  for (int i = 0; i < EPL; i++) w[i] = a.up[lane + i * CG < len ? en[i] >> 2 : c];
  const CaK ck = ca_k(t.prm);
  const double ca_du = t.ca_du, ca_dp = t.ca_dp;
  const double u = uc.x, p = uc.y;
  // meanwhile, the quotients that depend on the cell alone (:36-87, :128-136),
  // a lane each
  const double k2 = ck.para_k2 * ck.para_k2;
  const double num = lane == 0 ? ck.mu1 * p : lane == 1 ? ck.para_bb * u : lane == 2 ? ck.gamma * u : k2;
  const double den = lane == 0 ? p + ck.kmu : lane == 1 ? ck.para_k1 + u : lane == 2 ? ck.kg + u : k2 + u * u;
  const double quo = num / den;
  if (lane < 6) s_v[grp][lane] = val;
  if (lane < 4) s_v[grp][6 + lane] = quo;
  const double cv = REC ? corner_value(t, a, lane & 7, q, cr) : raw;
  if (lane < 8) s_g[grp][lane] = cv;
  double acc = 0;   // lane 0: the Ca2+ sum, lane 1: the IP3 sum (DEAD: lane 1 IP3, lane 0 the ALIVE count)
  for (int e0 = 0; e0 < len; e0 += CCAP) {
    const int m = min(CCAP, len - e0);
    if (e0 > 0) {
#pragma unroll
      for (int i = 0; i < EPL; i++) {
        const int e = lane + i * CG;
        en[i] = e < m ? a.w[row + e0 + e] : 0;
        gv[i] = e < m ? a.g[row + e0 + e] : 0.0;
      }
#pragma unroll
      for (int i = 0; i < EPL; i++) w[i] = a.up[lane + i * CG < m ? en[i] >> 2 : c];
    }
#pragma unroll
    for (int i = 0; i < EPL; i++) {
      const int e = lane + i * CG;
      if (e < m) {
        const bool alive = (en[i] & 3) == 3;
        if (dead) {
          // adding the +0.0 of an entry that is not ALIVE leaves the sums as
          // they are (they start at +0.0, so neither is ever -0.0)
          s_a[grp][e] = alive ? make_double2(1.0, w[i].y) : make_double2(0.0, 0.0);
        } else {
          s_a[grp][e] = make_double2(gv[i] * (w[i].x - u), gv[i] * (w[i].y - p));
          if (SAVE) sv->sg[(size_t)slot * a.cap * a.ns + row + e0 + e] = gv[i];
          if (alive) a.g[row + e0 + e] = gv[i] + ck.DT_Ca * fw_term(ck.wd, fabs(w[i].x - u), gv[i]);
        }
      }
    }
    wave_sync();
    // in list order, four entries' LDS reads ahead of their adds
    if (lane < 2) {
      const double* v = reinterpret_cast<const double*>(s_a[grp]) + lane;
      int e = 0;
      for (; e + 4 <= m; e += 4) {
        double d[4];
#pragma unroll
        for (int j = 0; j < 4; j++) d[j] = v[2 * (e + j)];
#pragma unroll
        for (int j = 0; j < 4; j++) acc += d[j];
      }
      for (; e < m; e++) acc += v[2 * e];
    }
    wave_sync();
  }
  if (dead) {
    const double count = __shfl(acc, 0, CG);
    if (lane == 1) {
      if (SAVE) {
        sv->su[slot * (size_t)a.cap + c] = u;
        sv->sp[slot * (size_t)a.cap + c] = p;
      }
      // ca2p of a DEAD cell stays as it is
      reinterpret_cast<double*>(a.upn + c)[1] = p + ck.DT_Ca * (ca_dp * (acc - count * p) - ck.Kpp * p);
    }
    return;
  }
  wave_sync();
  if (lane >= 3) return;
  const double* g = s_g[grp];
  const double* v = s_v[grp];
  // grid_avg8 in its order: 000 100 010 001 110 101 011 111
  const double Aavg = 0.125 * (g[0] + g[1] + g[2] + g[4] + g[3] + g[5] + g[6] + g[7]);
  const double exi = v[4];
  const double late = (lane == 2 ? v[9] - exi : v[1] * Aavg) / (lane == 2 ? v[0] : ck.H0 + Aavg);
  if (lane == 0) {
    const double er1 = ck.mu0 + v[6], er2 = ck.para_b + v[7];
    const double diff_u = ck.k_flux * er1 * er2 * exi - v[8] + ck.leak_from_storage + v[3] + ca_du * v[2] * acc;
    a.dfn[c] = diff_u;
    const double cs = u + ck.DT_Ca * diff_u;
    a.upn[c].x = cs;
    a.avg[c] = v[5] + cs;
  } else if (lane == 1) {
    a.upn[c].y = p + ck.DT_Ca * ((late - ck.Kpp * p) + ca_dp * v[2] * acc);
  } else {
    a.exi[c] = exi + ck.DT_Ca * late;
    if (SAVE) {
      const size_t k = slot * (size_t)a.cap + c;
      sv->su[k] = u;
      sv->sp[k] = p;
      sv->sh[k] = exi;
      sv->sAv[k] = Aavg;
    }
  }
}

template <int CG, bool ONE, bool SAVE>
__global__ void __launch_bounds__(C_BLOCK) k_ca_cells(const Tis* __restrict__ T, CaList cl, CaArg one, int cp, int ap,
                                                      int xcd, const RdTis* __restrict__ sv, int slot) {
  const unsigned b = xcd_order(blockIdx.x, gridDim.x, xcd);
  if (ONE) {
    ca_cells_part<CG, false, SAVE>(T[cl.t0], one, b, cl.ncb, SAVE ? sv + cl.t0 : nullptr, slot);
  } else {
    const int4 e = cl.cmap[b];
    ca_cells_part<CG, false, SAVE>(T[e.x], ca_arg(T[e.x], cp, cp, ap), e.y, e.z, SAVE ? sv + e.x : nullptr, slot);
  }
}

// ATP_refresh (:302-338) with the periodic copies of planes 0..iz_bound.
//
// One (x, y) column of a tile, planes l0 .. l1 - 1 (at most ZB), atp_new per
// point.  What bounds it: the instructions of a point more than its bytes (a
// wave's FP64 and address work at four cycles each; 6,900 waves a sub-step on
// the large tissue).  So the six neighbours' masks come as one byte of the
// solve's vmk, every address is a plane's base, the same for the whole wave,
// plus an offset within the plane kept in bytes (type Off: 32 bits, or 64 for
// planes of 4 GB), and the divisions of the tile's index are multiplications
// (div_by): about 120 instructions a point instead of 400.
//
// Tiles of up to 2 planes load everything first: the column, the lateral
// neighbours, masks and voxel words, then the owners' diff_u.  Taller ones
// roll the column through registers, the voxel word read one plane ahead, so
// that a plane waits for one round trip and few values are live at a time.
template <class Off>
struct AtpAddr {   // byte offsets of a column's points within a plane of doubles
  Off c, xm, xp, ym, yp;
  __device__ AtpAddr(const CaArg& t, int j, int k) {
    const Off wx = (Off)(t.NX - 1) * 8, wy = (Off)(t.NY - 1) * t.XP * 8, row = (Off)t.XP * 8;
    c = ((Off)k * t.XP + j) * 8;
    xm = j == 0 ? c + wx : c - 8;
    xp = j == t.NX - 1 ? c - wx : c + 8;
    ym = k == 0 ? c + wy : c - row;
    yp = k == t.NY - 1 ? c - wy : c + row;
  }
};
template <class Off>
__device__ __forceinline__ double at_f64(const double* plane, Off o) {
  return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(plane) + o);
}
// atp_new of one point with its mask byte and voxel word; plane l of the maps
template <class Off>
__device__ __forceinline__ double atp_point(const AtpK& ak, const CaArg& t, const AtpAddr<Off>& o, int l, double c0,
                                            double xm, double xp, double ym, double yp, double zm, double zp,
                                            unsigned mk, unsigned w, double diffu, double inv_dx) {
  double m[6];
#pragma unroll
  for (int b = 0; b < 6; b++) m[b] = (double)((mk >> b) & 1);
  if (mk & VMK_SLOW) {
    const uint8_t* __restrict__ cm2 = t.cm2;
    const long long p = (long long)l * t.PL;
    m[0] = cm2[p + o.xm / 8]; m[1] = cm2[p + o.xp / 8]; m[2] = cm2[p + o.ym / 8]; m[3] = cm2[p + o.yp / 8];
    m[4] = cm2[(long long)(l == 0 ? 1 : l - 1) * t.PL + o.c / 8];
    m[5] = cm2[(long long)(l + 1 == t.NZ ? l : l + 1) * t.PL + o.c / 8];
  }
  return atp_new(ak, c0, xm, xp, ym, yp, zm, zp, m[0], m[1], m[2], m[3], m[4], m[5], diffu, (double)(w >> 31), inv_dx);
}
// a point's new value and its periodic copies (:334-337)
template <class Off>
__device__ __forceinline__ void atp_store(const CaArg& t, double* plane, Off c, int j, int k, double nv) {
  char* p = reinterpret_cast<char*>(plane);
  *reinterpret_cast<double*>(p + c) = nv;
  if (j == 0 || k == 0) {
    const Off wx = (Off)t.NX * 8, wy = (Off)t.NY * t.XP * 8;
    if (k == 0) *reinterpret_cast<double*>(p + c + wy) = nv;
    if (j == 0) *reinterpret_cast<double*>(p + c + wx) = nv;
    if (j == 0 && k == 0) *reinterpret_cast<double*>(p + wx + wy) = nv;
  }
}

template <int ZB, class Off>
__device__ __forceinline__ void atp_column(const Tis& ti, const CaArg& t, int j, int k, int l0, int l1) {
  const AtpK ak = atp_k(ti.prm);
  const double inv_dx = ti.inv_dx;
  const AtpAddr<Off> o(t, j, k);
  const int nl = l1 - l0;
  const double* __restrict__ A = t.A0;
  double cz[ZB + 2], xm[ZB], xp[ZB], ym[ZB], yp[ZB], diffu[ZB];
  unsigned mk[ZB], w[ZB];
#pragma unroll
  for (int q = 0; q < ZB + 2; q++) {
    int l = q == 0 ? (l0 == 0 ? 1 : l0 - 1) : l0 + q - 1;   // mirror z boundary (utils.cpp:32-72)
    if (l > t.NZ - 1) l = t.NZ - 1;
    cz[q] = q <= nl + 1 ? at_f64(A + l * t.PL, o.c) : 0.0;
  }
#pragma unroll
  for (int q = 0; q < ZB; q++) {
    xm[q] = xp[q] = ym[q] = yp[q] = 0;
    mk[q] = w[q] = 0;
    if (q < nl) {
      const long long pl = (l0 + q) * t.PL;
      w[q] = *reinterpret_cast<const unsigned*>(reinterpret_cast<const char*>(t.vox + pl) + o.c / 2);
      mk[q] = t.vmk[pl + o.c / 8];
      xm[q] = at_f64(A + pl, o.xm); xp[q] = at_f64(A + pl, o.xp);
      ym[q] = at_f64(A + pl, o.ym); yp[q] = at_f64(A + pl, o.yp);
    }
  }
#pragma unroll
  for (int q = 0; q < ZB; q++) {
    const unsigned cell1 = w[q] & 0x7fffffffu;
    diffu[q] = cell1 ? t.dfo[cell1 - 1] : 0.0;
  }
#pragma unroll
  for (int q = 0; q < ZB; q++)
    if (q < nl) {
      const double nv = atp_point(ak, t, o, l0 + q, cz[q + 1], xm[q], xp[q], ym[q], yp[q], cz[q], cz[q + 2], mk[q], w[q],
                                  diffu[q], inv_dx);
      atp_store(t, t.A1 + (l0 + q) * t.PL, o.c, j, k, nv);
    }
}

template <class Off>
__device__ __forceinline__ void atp_column_roll(const Tis& ti, const CaArg& t, int j, int k, int l0, int l1) {
  const AtpK ak = atp_k(ti.prm);
  const double inv_dx = ti.inv_dx;
  const AtpAddr<Off> o(t, j, k);
  const double* __restrict__ A = t.A0;
  const long long PL = t.PL;
  auto vox = [&](int l) {
    return *reinterpret_cast<const unsigned*>(reinterpret_cast<const char*>(t.vox + l * PL) + o.c / 2);
  };
  double zm = at_f64(A + (l0 == 0 ? 1 : l0 - 1) * PL, o.c);   // mirror z (utils.cpp:32-72)
  double c0 = at_f64(A + l0 * PL, o.c);
  unsigned w = l0 < l1 ? vox(l0) : 0u;
  for (int l = l0; l < l1; l++) {
    const long long pl = l * PL;
    const double zp = at_f64(A + (l + 1 == t.NZ ? pl : pl + PL), o.c);
    const unsigned wn = l + 1 < l1 ? vox(l + 1) : 0u;
    const unsigned mk = t.vmk[pl + o.c / 8];
    const unsigned cell1 = w & 0x7fffffffu;
    const double diffu = cell1 ? t.dfo[cell1 - 1] : 0.0;
    const double xm = at_f64(A + pl, o.xm), xp = at_f64(A + pl, o.xp), ym = at_f64(A + pl, o.ym),
                 yp = at_f64(A + pl, o.yp);
    atp_store(t, t.A1 + pl, o.c, j, k, atp_point(ak, t, o, l, c0, xm, xp, ym, yp, zm, zp, mk, w, diffu, inv_dx));
    zm = c0;
    c0 = zp;
    w = wn;
  }
}

// one tile of a solve's list: blockDim.x consecutive points of the (x, y)
// plane times ZB planes; mg_npt: div_by's magic for its tiles per plane
template <int ZB, class Off>
__device__ __forceinline__ void atp_tile(const Tis& ti, const CaArg& t, unsigned local, unsigned mg_npt, int izb) {
  const int NX = t.NX, NY = t.NY;
  const unsigned bs = blockDim.x, plane = (unsigned)NX * NY;
  const unsigned npt = (plane + bs - 1) / bs;
  const unsigned zt = div_by(local, npt, mg_npt);
  const unsigned p = (local - zt * npt) * bs + threadIdx.x;
  if (p >= plane) return;
  const int k = (int)div_by(p, NX, t.mg_nx), j = (int)(p - (unsigned)k * NX);
  const int l0 = (int)zt * ZB;
  if (ZB >= 4) atp_column_roll<Off>(ti, t, j, k, l0, min(l0 + ZB, izb));
  else atp_column<ZB, Off>(ti, t, j, k, l0, min(l0 + ZB, izb));
  // plane l = iz_bound: copies of values left in the next buffer (:334-337);
  // the corner (NX, NY) ends as a copy of (0, 0)
  if (l0 == 0 && (j == 0 || k == 0)) {
    double* __restrict__ narr = t.A1;
    if (k == 0) narr[gidx(t, j, NY, izb)] = narr[gidx(t, j, 0, izb)];
    if (j == 0) narr[gidx(t, NX, k, izb)] = narr[gidx(t, 0, k, izb)];
    if (j == 0 && k == 0) narr[gidx(t, NX, NY, izb)] = narr[gidx(t, 0, 0, izb)];
  }
}

// the ATP tiles of a solve's list, walked grid-stride by `nb` blocks of
// which this is block `b` (XCD runs with xcd): the tile offsets, iz_bound
// and tissue ids of up to CA_LDS_T tissues are staged in LDS (kept small: the
// fused kernel's cell blocks hold LDS of their own)
constexpr int CA_LDS_T = 256;
template <int ZB, bool ONE, class Off>
__device__ __forceinline__ void atp_walk(const Tis* __restrict__ T, const CaList& cl, int b, int nb, int xcd, int ap,
                                         int cp) {
  if (ONE) {   // one tissue: its id and iz_bound come with the list
    const Tis& t = T[cl.t0];
    const CaArg a = ca_arg(t, cp, cp, ap);
    for (TileWalk tw(cl.atiles, xcd, b, nb); tw.w < tw.end; tw.w += tw.stride) atp_tile<ZB, Off>(t, a, tw.w, cl.mg_npt, cl.izb0);
    return;
  }
  const int nt = cl.ntis;
  __shared__ int s_off[CA_LDS_T + 1];
  __shared__ int2 s_ti[CA_LDS_T];
  const bool lds = nt <= CA_LDS_T;
  if (lds) {
    for (int i = threadIdx.x; i <= nt; i += blockDim.x) {
      s_off[i] = cl.aoff[i];
      if (i < nt) s_ti[i] = make_int2(cl.atis[i], cl.aizb[i]);
    }
    __syncthreads();
  }
  auto off = [&](int i) { return lds ? s_off[i] : cl.aoff[i]; };
  int ti = 0;
  for (TileWalk tw(off(nt), xcd, b, nb); tw.w < tw.end; tw.w += tw.stride) {
    // uniform over the block (see k_ext_stim)
    ti = __builtin_amdgcn_readfirstlane(wl_find(off, ti, nt, tw.w));
    const int2 q = lds ? s_ti[ti] : make_int2(cl.atis[ti], cl.aizb[ti]);
    const Tis* t = T + __builtin_amdgcn_readfirstlane(q.x);
    atp_tile<ZB, Off>(*t, ca_arg(*t, cp, cp, ap), tw.w - __builtin_amdgcn_readfirstlane(off(ti)), 0u,
                      __builtin_amdgcn_readfirstlane(q.y));
  }
}

template <int ZB, bool ONE, class Off>
__global__ void __launch_bounds__(256) k_atp(const Tis* __restrict__ T, CaList cl, int ap, int cp, int xcd) {
  atp_walk<ZB, ONE, Off>(T, cl, blockIdx.x, gridDim.x, xcd, ap, cp);
}

// one launch for the ATP update of sub-step i (parities cp, ap) and the cells
// of sub-step i + 1: blocks [0, ncb) take the cells (one entry of the list's
// cell-block map each), the rest walk the ATP tiles.  With xcd (the grid then
// holds 8 ceil(ncb / 8) cell blocks, the last ones idle, and a multiple of 8
// ATP blocks) each XCD (block id mod 8) walks one contiguous run of the ATP
// tiles, so that the tiles above and below a tile, which read its plane,
// share its L2; the cell blocks stay dealt round-robin (contiguous runs of
// cells are runs of one layer, whose cells cost alike, and left the XCDs
// unevenly loaded).  Results do not depend on it.
constexpr int F_BLOCK = 128;

template <int CG, int ZB, bool ONE, bool SAVE>
__global__ void __launch_bounds__(F_BLOCK) k_ca_fused(const Tis* __restrict__ T, CaList cl, CaArg one, int cp, int ap,
                                                      int ncb, int xcd, const RdTis* __restrict__ sv, int slot) {
  int cbk = -1;   // this block's cell block, or -1 for an ATP block
  int ab = 0, an = 0;
  if (xcd) {
    const int cblocks = (ncb + 7) & ~7;   // a multiple of 8: ATP block ids keep their XCD
    if ((int)blockIdx.x < cblocks) {
      cbk = (int)blockIdx.x;
      if (cbk >= ncb) return;
    } else {
      ab = (int)blockIdx.x - cblocks;
      an = (int)gridDim.x - cblocks;
    }
  } else if ((int)blockIdx.x < ncb) {
    cbk = (int)blockIdx.x;
  } else {
    ab = (int)blockIdx.x - ncb;
    an = (int)gridDim.x - ncb;
  }
  if (cbk < 0) {
    atp_walk<ZB, ONE, unsigned>(T, cl, ab, an, xcd, ap, cp);
  } else if (ONE) {
    ca_cells_part<CG, true, SAVE>(T[cl.t0], one, cbk, ncb, SAVE ? sv + cl.t0 : nullptr, slot);
  } else {
    const int4 e = cl.cmap[cbk];
    ca_cells_part<CG, true, SAVE>(T[e.x], ca_arg(T[e.x], 1 - cp, cp, ap), e.y, e.z, SAVE ? sv + e.x : nullptr, slot);
  }
}

// The packed gj back into the list rows and the (ca2p, IP3) pairs into their
// arrays; at the end of a solve (ca2p.cpp:400-402) also the averages divided
// and the cells past the membrane and dermis that are not AFM cleared.
__global__ void __launch_bounds__(256) k_ca_end(const Tis* __restrict__ T, const int* tlist, int cb, int what) {
  const Tis& t = T[tlist ? tlist[blockIdx.y] : blockIdx.y];
  const int n = t.st->n;
  const int Ca_ITR = t.prm.Ca_ITR;
  const int lane = threadIdx.x & (BL - 1);
  for (int c = t.nmemb + t.nder + (blockIdx.x * blockDim.x + threadIdx.x) / BL; c < n;
       c += gridDim.x * blockDim.x / BL) {
    const size_t at = (size_t)c * t.ns;
    const uint8_t s = t.state[c];
    const int k = t.ca_cn[c];
    for (int e = lane; e < k; e += BL) t.gj[cb][at + t.ca_sl[at + e]] = t.ca_g[at + e];
    if (lane != 0) continue;
    const bool afm = is_afm(s);
    if (afm || s == DEAD) {
      for (int b = 0; b < 2; b++) {
        const double2 w = t.ca_up[b][c];
        t.ca2p[b][c] = w.x;
        t.ip3[b][c] = w.y;
      }
    }
    if (what == CA_END_SOLVE) {
      if (afm) {
        t.ca2p_avg[c] = t.ca2p_avg[c] / Ca_ITR;
      } else {
        t.ca2p_avg[c] = 0;
        t.ca2p[0][c] = 0;
        t.ca2p[1][c] = 0;
      }
    }
    if (what != CA_END_PUT) t.diff_u[c] = 0;
  }
}

__global__ void __launch_bounds__(256) k_ca_swap(const Tis* __restrict__ T, const int* __restrict__ tlist) {
  const Tis& t = T[tlist[blockIdx.y]];
  const long long stride = (long long)gridDim.x * blockDim.x;
  const long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  for (long long i = i0; i < t.gsize; i += stride) {
    const double a = t.atp[0][i];
    t.atp[0][i] = t.atp[1][i];
    t.atp[1][i] = a;
  }
  const int n = t.st->n;
  for (long long c = i0; c < n; c += stride) {
    const double u = t.ca2p[0][c], p = t.ip3[0][c];
    const double2 w = t.ca_up[0][c];
    t.ca2p[0][c] = t.ca2p[1][c];
    t.ca2p[1][c] = u;
    t.ip3[0][c] = t.ip3[1][c];
    t.ip3[1][c] = p;
    t.ca_up[0][c] = t.ca_up[1][c];
    t.ca_up[1][c] = w;
  }
}

__global__ void k_sw_reset(const Tis* __restrict__ T, const int* tlist) {
  const Tis& t = T[tlist ? tlist[blockIdx.x] : blockIdx.x];
  if (threadIdx.x == 0) t.st->sw = 0;
}

void launch_ca_swap(hipStream_t s, const Tis* dT, const int* tlist, int ntis, int max_n, long long max_gsize) {
  const long long items = std::max<long long>(max_gsize, max_n);
  const long long g = std::min<long long>((items + 255) / 256, 4096);
  EPI_LAUNCH(K_CA_SWAP, k_ca_swap, dim3((unsigned)g, ntis), dim3(256), 0, s, dT, tlist);
}

unsigned map_clear_blocks(long long max_gsize) {
  // four quads a thread, if every plane had been stamped: the stores of 32
  // uneven tissues (72 MB of maps) took 57 us with one quad a thread
  const long long q = (max_gsize / 16 + 255) / 256;
  return (unsigned)(q < 1 ? 1 : q < 65535 ? q : 65535);
}

void launch_map_clear(hipStream_t s, const Tis* dT, int ntis, long long max_gsize) {
  EPI_LAUNCH(K_MAP_CLEAR, k_map_clear, dim3(map_clear_blocks(max_gsize), ntis), dim3(256), 0, s, dT);
}

void launch_map_stamp(hipStream_t s, const Tis* dT, int ntis, int pb, int max_n, const Tuning& tu) {
  if (tu.map_lanes == 16)
    EPI_LAUNCH(K_MAP_STAMP, k_map_stamp<16>, dim3((16 * max_n + 127) / 128, ntis), dim3(128), 0, s, dT, pb);
  else if (tu.map_lanes == 4)
    EPI_LAUNCH(K_MAP_STAMP, k_map_stamp<4>, dim3((4 * max_n + 127) / 128, ntis), dim3(128), 0, s, dT, pb);
  else
    EPI_LAUNCH(K_MAP_STAMP, k_map_stamp<1>, dim3((max_n + 127) / 128, ntis), dim3(128), 0, s, dT, pb);
}

namespace {
// a grid-stride walk over the list: the grid is sized from the host's estimate
// (the last known zzmax), one block per tile (a cap at the blocks the CUs hold
// at once left a tail of blocks waiting: 376-383 against 328-338 us on the
// 256-tissue batch), and a multiple of 8 so that the XCD split applies
unsigned ext_stim_blocks(long long tiles_est) {
  return (unsigned)((std::min(std::max(tiles_est, 1LL), 1LL << 24) + 7) / 8 * 8);
}
}  // namespace

void launch_ext_stim_list(hipStream_t s, const Tis* dT, int ntis, int bp, long long tiles_est, const int* d_wl,
                          const Tuning& tu) {
  by_zb(tu.b_zb, [&](auto zbc) {
    EPI_LAUNCH(K_EXT_STIM, k_ext_stim<decltype(zbc)::value>, dim3(ext_stim_blocks(tiles_est)), dim3(64 * tu.b_rows), 0, s, dT,
               d_wl, d_wl + ntis + 1, ntis, bp, tu.b_xcd);
  });
}

void launch_ext_stim(hipStream_t s, const Tis* dT, int ntis, int bp, long long tiles_est, int* d_wl,
                     const Tuning& tu) {
  const int bs = 64 * tu.b_rows;
  if (ntis == 1) {
    by_zb(tu.b_zb, [&](auto zbc) {
      EPI_LAUNCH(K_EXT_STIM, k_ext_stim_one<decltype(zbc)::value>, dim3(ext_stim_blocks(tiles_est)), dim3(bs), 0, s, dT, bp,
                 tu.b_xcd);
    });
    return;
  }
  EPI_LAUNCH(K_WL, k_wl_b, dim3(1), dim3(256), 0, s, dT, ntis, bs, tu.b_zb, d_wl, d_wl + ntis + 1);
  launch_ext_stim_list(s, dT, ntis, bp, tiles_est, d_wl, tu);
}

static unsigned ca_lane_blocks(int max_n) { return ((unsigned)max_n * BL + 255) / 256; }

void launch_ca_corners(hipStream_t s, const Tis* dT, const int* tlist, int ntis, int bp, int max_n) {
  EPI_LAUNCH(K_CA_CORNERS, k_ca_corners, dim3((8 * max_n + 255) / 256, ntis), dim3(256), 0, s, dT, tlist, bp);
}

void launch_ca_begin(hipStream_t s, const Tis* dT, const int* tlist, int ntis, int cb, int bp, int max_n,
                     long long max_plane, int max_izb, int zero_avg) {
  EPI_LAUNCH(K_CA_BEGIN, k_ca_begin, dim3(ca_lane_blocks(max_n), ntis), dim3(256), 0, s, dT, tlist, cb, zero_avg);
  const unsigned gb = (unsigned)std::max<long long>(1, std::min<long long>((max_plane + 255) / 256, 65535));
  EPI_LAUNCH(K_CA_VOX, k_ca_vox, dim3(gb, ntis, (unsigned)std::max(1, std::min(max_izb, 65535))), dim3(256), 0, s, dT, tlist);
  launch_ca_corners(s, dT, tlist, ntis, bp, max_n);
}

void launch_ca_end(hipStream_t s, const Tis* dT, const int* tlist, int ntis, int cb, int max_n, int what) {
  EPI_LAUNCH(K_CA_END, k_ca_end, dim3(ca_lane_blocks(max_n), ntis), dim3(256), 0, s, dT, tlist, cb, what);
  if (what == CA_END_SOLVE) EPI_LAUNCH(K_SW_RESET, k_sw_reset, dim3(ntis), dim3(64), 0, s, dT, tlist);
}

namespace {
// the launch's by-value tissue: a one-tissue list's, or nothing that is read
CaArg one_arg(const CaList& cl, int cpc, int cpa, int ap) {
  return cl.ntis == 1 ? ca_arg(*cl.h0, cpc, cpa, ap) : CaArg{};
}

// f with true or false as a type, by b
template <class F>
void by_bool(bool b, F f) {
  if (b) f(std::true_type());
  else f(std::false_type());
}
// f with the lanes per cell, whether the list has one tissue and whether the
// launch saves, as types
template <class F>
void by_cells(const CaList& cl, const Tuning& tu, const RdTis* sv, F f) {
  by_bool(cl.ntis == 1, [&](auto one) {
    by_bool(sv != nullptr, [&](auto save) {
      if (ca_lanes(tu.ca_group) == 8) f(std::integral_constant<int, 8>(), one, save);
      else f(std::integral_constant<int, 16>(), one, save);
    });
  });
}

void launch_cells(hipStream_t s, const Tis* dT, const CaList& cl, int cp, int ap, const Tuning& tu, const RdTis* sv,
                  int slot) {
  by_cells(cl, tu, sv, [&](auto cg, auto one, auto save) {
    const auto kfn = k_ca_cells<decltype(cg)::value, decltype(one)::value, decltype(save)::value>;
    EPI_LAUNCH(K_CA_CELLS, kfn, dim3((unsigned)std::max(cl.ncb, 1)), dim3(C_BLOCK), 0, s, dT, cl,
               one_arg(cl, cp, cp, ap), cp, ap, tu.xcd, sv, slot);
  });
}

// blocks that walk a list of `tiles` tiles: one per tile (as launch_ext_stim),
// a multiple of 8 (the XCD split)
unsigned walk_blocks(long long tiles) {
  const long long cap = 1LL << 24;
  long long g = std::min(std::max(tiles, 1LL), cap);
  return (unsigned)((g + 7) / 8 * 8);
}

void launch_atp(hipStream_t s, const Tis* dT, const CaList& cl, int cp, int ap, const Tuning& tu) {
  const dim3 g(walk_blocks(cl.atiles));
  by_zb(tu.a_zb, [&](auto zbc) {
    constexpr int zb = decltype(zbc)::value;
    const auto k1 = k_atp<zb, true, unsigned>, kn = k_atp<zb, false, unsigned>,
               kw = k_atp<zb, false, unsigned long long>;
    EPI_LAUNCH(K_ATP, (cl.wide ? kw : cl.ntis == 1 ? k1 : kn), g, dim3(cl.abs), 0, s, dT, cl, ap, cp, tu.xcd);
  });
}

// the ATP update of the sub-step at (cp, ap) beside the cells of the next one
void launch_fused(hipStream_t s, const Tis* dT, const CaList& cl, int cp, int ap, const Tuning& tu, const RdTis* sv,
                  int slot) {
  const unsigned cblocks = tu.xcd ? (unsigned)(cl.ncb + 7) / 8 * 8 : (unsigned)cl.ncb;
  const dim3 g(cblocks + walk_blocks(cl.atiles));
  by_cells(cl, tu, sv, [&](auto cg, auto one, auto save) {
    constexpr int CG = decltype(cg)::value;
    constexpr bool ONE = decltype(one)::value, SAVE = decltype(save)::value;
    const auto k1 = k_ca_fused<CG, 1, ONE, SAVE>, k2 = k_ca_fused<CG, 2, ONE, SAVE>;
    EPI_LAUNCH(K_CA_FUSED, (tu.a_zb == 2 ? k2 : k1), g, dim3(F_BLOCK), 0, s, dT, cl, one_arg(cl, 1 - cp, cp, ap), cp, ap,
               cl.ncb, tu.xcd, sv, slot);
  });
}
}  // namespace

int ca_list_bs(const Tuning& tu, bool fused) { return fused ? F_BLOCK : 64 * tu.a_rows; }

void launch_ca_substeps(hipStream_t s, const Tis* dT, const CaList& cl, int& cp, int& ap, int n_sub, const Tuning& shape,
                        const RdTis* sv, int slot, bool last_cells_only) {
  // contiguous runs per XCD only where every CU gets several workgroups: a run
  // gathers the tiles of one height, and with few of them the XCDs are uneven
  // (1,200 workgroups 6 % slower, 4,700 1.3 % faster, 292,000 cells in 32 tissues
  // 4 % faster)
  constexpr long long XCD_BLOCKS = 2048;
  Tuning tu = shape;
  tu.xcd = shape.xcd && cl.ncb + cl.atiles >= XCD_BLOCKS;
  const bool fuse = tu.ca_fuse && n_sub >= 2;
  // fused: cells of sub-step 0; then (ATP of i, cells of i + 1); then ATP of the last
  for (int i = 0; i < n_sub; i++) {
    if (i == 0 || !fuse) launch_cells(s, dT, cl, cp, ap, tu, sv, slot + i);
    if (i + 1 < n_sub && fuse) {
      launch_fused(s, dT, cl, cp, ap, tu, sv, slot + i + 1);
    } else if (i + 1 < n_sub || !last_cells_only) {
      launch_atp(s, dT, cl, cp, ap, tu);
    }
    cp ^= 1;
    ap ^= 1;
  }
}

}  // namespace epi
