// epi_dev.h -- device-side data layout and the scalar laws of the epi5_MT hot
// path, for CDNA4 (gfx950).
//
// Layout: one Tis descriptor per tissue in device memory; kernels take the
// descriptor array and use blockIdx.y as the tissue index, so a single
// launch advances every tissue of a batch.  Cells are SoA, neighbour lists
// are fixed-stride rows (stride = ns entries per cell), grids are stored
// z-major / x-fastest with a padded x pitch.
//
// Every FP64 expression keeps the operand order of the reference so that a
// build without FP contraction (-ffp-contract=off) reproduces it.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "params.h"

namespace epi {

// cell states, epi5_MT/define.h:36-47
enum : uint8_t { ALIVE = 0, DEAD = 1, DISA = 2, UNUSED = 3, FIX = 4, BLANK = 5,
                 DER = 6, MUSUME = 7, AIR = 8, MEMB = 9 };

// status codes, mirrored in include/epi_amd.h
enum { OK = 0, ERR_CAPACITY = 1, ERR_STRONG_INTERACTION = 2, ERR_NO_DERMIS = 3,
       ERR_OUT_OF_GRID = 4, ERR_REMOVE_ALIAS = 5, ERR_RNG_EXHAUSTED = 6,
       ERR_INVALID = 7, ERR_HIP = 8, ERR_PAIR_REMOVED = 9 };

// ---- constants -----------------------------------------------------------
// The physics constants are runtime values, one record per tissue (Tis::prm,
// params.h).  What stays here fixes the shape of the build.
constexpr int MEMB_ADJ = 6;                // define.h:147-153 (TRI_MEMB)
constexpr int MAX_CONN = 400;              // define.h:80, cell_connection.cpp:30
constexpr int N3 = 200;                    // cell_connection.cpp:28
// the fewest slots of a list row: kernels read a row's first chunk before they
// know its length, and check that it fits
constexpr int ROW_SLOTS_MIN = 64;
// A bucket is a head of eight words, its count and its first seven cells (two
// 16-byte loads), and the rest of its slots elsewhere: the five heads that a
// sweep reads of a column lie in two or three cache lines.  Words between two
// buckets' further slots: a multiple of 4, for 16-byte loads of four cells.
constexpr int BUCKET_HEAD = 8;
__host__ __device__ constexpr int bucket_more(int bcap) { return bcap < BUCKET_HEAD ? 4 : (bcap - (BUCKET_HEAD - 1) + 3) & ~3; }
constexpr double AREA_GRID = 2.0 + 1e-7;   // cell_connection.cpp:16-19 (the bucket edge)

// force laws (cell_interaction.cpp:68-76)
enum : int { LAW_NONE = 0, LAW_OTHER, LAW_DER_DER, LAW_FIXMU, LAW_FIX_MEMB,
             LAW_MU_MEMB, LAW_ALAIRDE, LAW_MEMB_MEMB, LAW_PAIR };

// A pointer into device memory that a kernel reads from a descriptor.  The
// compiler cannot know where a pointer loaded from memory leads and would
// reach it with flat instructions, which also wait as LDS accesses do, cannot
// take a scalar base and return in no order; this one says that it is global.
// The layout is a pointer's; files without kernels see a plain one.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(EPI_NO_KERNELS)
template <class T>
struct GPtr {
  __attribute__((address_space(1))) T* p;
  __host__ __device__ __forceinline__ GPtr& operator=(T* q) {
    p = (__attribute__((address_space(1))) T*)q;
    return *this;
  }
  __host__ __device__ __forceinline__ operator T*() const { return (T*)p; }
  __host__ __device__ __forceinline__ T* operator->() const { return (T*)p; }
};
#else
template <class T>
using GPtr = T*;
#endif

// ---- per-tissue device status (changes on device) ---------------------
struct Status {
  int n;                  // live cells
  int n_old;              // cells before the last state renewal
  int err;                // first error code
  int sw;                 // cornifications since the last Ca solve (uint8 wrap)
  int ndiv;               // divisions in the last renewal
  int nrm;                // removals in the last renewal
  int maxlen;             // longest neighbour list of any build or epi_set_lists
  int stamp_z;            // highest z plane ever stamped into the voxel maps
  long long rng_pos;      // replay cursor
  long long next_uid;
  unsigned long long zzmax_bits;  // calc_zzmax result (non-negative double bits)
  double zzmax;
  long long timestep;     // CellManager::current_timestep; advanced once per renewal
  int nstat;              // records in cst_store
  int force_err;          // first error code of the force kernels, which run ahead of the status read-back
  long long grid_b;       // sum of nx*ny*iz_bound over the B sweeps (k_wl_b)
};

// ---- per-tissue descriptor (constant between allocations) ---------------
struct Tis {
  // geometry
  int nmemb, nder, cap, ns;   // ns = neighbour row stride
  int NX, NY, NZ, XP;         // XP = padded x pitch of grid rows
  long long PL;               // plane pitch (XP*(NY+1))
  long long gsize;            // XP*(NY+1)*(NZ+1)
  double LX, LY, LZ, dx, dy, dz, inv_dx, inv_dy, inv_dz;
  int ANX, ANY, ANZ, bcap;
  int irx, iry, irz;
  unsigned mg_nx;             // div_magic(NX, NX NY)
  // ca2p_du (ca2p.cpp:183), dp (ca2p.cpp:17), eps_m, K_TOTAL, Kspring and
  // KBEND (cell_interaction.cpp:21-28) as the kernels use them: prm's
  // values, or a window's while one is open
  double ca_du, ca_dp;
  double m_eps, m_kadh, m_kspring, m_kbend;
  GPtr<Status> st;
  // cells
  GPtr<uint8_t> state; GPtr<uint8_t> is_malignant; GPtr<uint8_t> touch_air;
  GPtr<int> fix_origin; GPtr<int> rest_div_times; GPtr<int> pair; GPtr<int> dermis; GPtr<int> lat;  // lat: 3/cell
  GPtr<double> pos[2][3];          // [buffer][axis]
  GPtr<double> radius, div_age_thresh;
  GPtr<double> ca2p[2]; GPtr<double> ip3[2];
  GPtr<double> ca2p_avg, ex_inert, agek, ageb, ex_fat, in_fat, spr_nat_len, diff_u;
  GPtr<double> ca_th, ca_kpa, ca_iag;   // per-solve constants of the Ca step (agek and state are frozen)
  // The coupled list entries of the AFM and DEAD cells during a solve or
  // window, packed to the front of a row of ns in list order: the word
  // neighbour << 2 | kind (1 coupled, 3 coupled ALIVE), the entry's slot in the
  // list row, and its gj, which lives here until k_ca_end puts it back; and
  // their number per cell (0 for the other cells)
  GPtr<int> ca_w;
  GPtr<unsigned short> ca_sl;
  GPtr<double> ca_g;
  GPtr<int> ca_cn;
  // (ca2p, IP3) of buffer b during a solve or window, so that a list entry
  // reads its neighbour's pair with one 16-byte gather; the arrays ca2p and
  // ip3 follow at its end (k_ca_end)
  GPtr<double2> ca_up[2];
  // diff_u of the Ca sub-steps at parity 1 (parity 0 writes diff_u itself)
  GPtr<double> ca_dfu;
  // per AFM cell and grid_avg8 corner (binary x, y, z), during a solve: the
  // corner's point, voxel word, masks and flags (ca_corner.h)
  GPtr<uint4> ca_cq;
  GPtr<double> ca_bx;   // ca2p_by_ext_stim per AFM cell (B does not change during a solve)
  GPtr<long long> uid; GPtr<long long> old_uid[2]; GPtr<int> src_row;
  // cell_stat (define.h:198-202): per cell k_aging_start, k_cornified,
  // k_disap (-1 = never set); cst_store (cellmanager.h:106): the records of
  // removed DEAD cells, up to cap of them, Status::nstat in use
  GPtr<long long> cst; GPtr<long long> cst_store;
  // neighbour rows (two buffers: current and previous build)
  GPtr<int> nlen[2]; GPtr<int> col[2]; GPtr<double> gj[2];
  GPtr<int> nlo;                   // entries of the row below the cell index
  GPtr<int> btmp; GPtr<int> bcnt;       // upper partners gathered during the sweep
  GPtr<int> memb6;                 // triangular adjacency, 6 per membrane cell
  // buckets
  GPtr<int> bucket_of; GPtr<int> bucket; GPtr<int> bucket_rest;
  // (x, y, z, radius) of every cell after the periodic fix, written by the
  // bucket insertion: the sweep and the row assembly gather a candidate's
  // position and radius with one 32-byte load instead of four
  GPtr<double4> pk[2]; GPtr<int4> fa;
  // state renewal
  GPtr<double> div_dir;   // per division: its direction
  GPtr<int> rm_list;
  // per block of 256 cells past the dermis: the cells that need a draw and
  // those that go, and how many
  GPtr<int> rd_list; GPtr<int> rm_pack; GPtr<int> rd_n; GPtr<int> rm_n;
  // grids
  GPtr<double> atp[2]; GPtr<double> bf[2];
  // vox, vmk: during a solve or window, per voxel of the active box, the AFM
  // owner and air flag (k_ca_vox) and the masks of its six neighbours in one
  // byte (bits 0-5: x-, x+, y-, y+, z-, z+; VMK_SLOW when one is above 1)
  GPtr<int> cmap1; GPtr<uint8_t> cmap2; GPtr<unsigned> vox; GPtr<uint8_t> vmk;
  // replay stream
  GPtr<const double> rng; long long rng_n;
  // the tissue's runtime parameters (epi_set_params)
  Params prm;
};

// the record of a cell's attributes that the force laws read (Tis::fa)
__device__ __forceinline__ int4 force_attr(int pair, int dermis, int rest_div_times, uint8_t state, bool strong) {
  return make_int4(pair, dermis, rest_div_times, state | (strong ? 256 : 0));
}
__device__ __forceinline__ void set_err(Status* st, int e) { atomicCAS(&st->err, 0, e); }
// of a force kernel: kept apart until the next renewal takes it over, so that
// a step's status never shows an error of the step after it
__device__ __forceinline__ void set_force_err(Status* st, int e) { atomicCAS(&st->force_err, 0, e); }

// ---- geometry helpers: utils.h:25-53 ----------------------------------
__device__ __forceinline__ double p_diff_x(const Tis& t, double x1, double x2) {
  const double diff = x1 - x2;
  if (diff > 0.5 * t.LX) return diff - t.LX;
  if (diff <= -0.5 * t.LX) return diff + t.LX;
  return diff;
}
__device__ __forceinline__ double p_diff_y(const Tis& t, double y1, double y2) {
  const double diff = y1 - y2;
  if (diff > 0.5 * t.LY) return diff - t.LY;
  if (diff <= -0.5 * t.LY) return diff + t.LY;
  return diff;
}
__device__ __forceinline__ double min0(double a) { return a > 0 ? a : 0; }

#define POW6(x) ((x) * (x) * (x) * (x) * (x) * (x))
#define POW3(x) ((x) * (x) * (x))

struct P3 { double x, y, z; };

__device__ __forceinline__ P3 ld_pos(const Tis& t, int pb, int c) {
  return P3{t.pos[pb][0][c], t.pos[pb][1][c], t.pos[pb][2][c]};
}

__device__ __forceinline__ double dist_sq(const Tis& t, P3 a, P3 b) {
  const double diffx = p_diff_x(t, a.x, b.x);
  const double diffy = p_diff_y(t, a.y, b.y);
  const double diffz = a.z - b.z;
  return diffx * diffx + diffy * diffy + diffz * diffz;
}

// grid index of (x, y, z) lattice point in the device layout
template <class G>   // a Tis, or what a launch carries of one (CaArg)
__device__ __forceinline__ long long gidx(const G& t, int j, int k, int l) {
  return (long long)l * t.PL + (long long)k * t.XP + j;
}

constexpr unsigned VMK_SLOW = 0x80u;

// n / d for n below the limit the magic was made for (0: none was)
__device__ __forceinline__ unsigned div_by(unsigned n, unsigned d, unsigned magic) {
  return magic ? __umulhi(n, magic) : n / d;
}
// ceil(2^32 / d) if n * that / 2^32 rounds down to n / d for every n < limit
// (the excess e = magic d - 2^32 < d adds n e / (d 2^32) < 1 / d), else 0
inline unsigned div_magic(unsigned d, unsigned long long limit) {
  const unsigned long long m = ((1ull << 32) + d - 1) / d, e = m * d - (1ull << 32);
  return d > 1 && limit * e < (1ull << 32) ? (unsigned)m : 0u;
}

// empties the voxel maps' planes 0..stamp_z, four voxels per thread, by block
// b of nb blocks (a plane holds PL = XP (NY + 1) voxels with XP a multiple of
// 16, and the maps start 256-byte aligned)
__device__ __forceinline__ void map_clear(const Tis& t, int b, int nb) {
  const int planes = min(t.st->stamp_z, t.NZ) + 1;
  const long long g4 = (long long)planes * t.PL / 4;
  int4* __restrict__ m1 = reinterpret_cast<int4*>(static_cast<int*>(t.cmap1));
  unsigned* __restrict__ m2 = reinterpret_cast<unsigned*>(static_cast<uint8_t*>(t.cmap2));
  for (long long q = (long long)b * blockDim.x + threadIdx.x; q < g4; q += (long long)nb * blockDim.x) {
    m1[q] = make_int4(-1, -1, -1, -1);
    m2[q] = 0u;
  }
}

__device__ __forceinline__ bool is_afm(uint8_t s) { return s == ALIVE || s == FIX || s == MUSUME; }

}  // namespace epi
