// k_connect.hip -- connect_cell (cell_connection.cpp:38-203) and calc_zzmax
// (proc.cpp:34-43) on CDNA4.
//
// Neighbour rows are rebuilt every step in the reference's canonical order:
//   [6 membrane neighbours if MEMB] ++ [partners o < X found by X's own
//   5x5x5 bucket sweep, in sweep order] ++ [partners c > X, ascending c].
// k_bucket_insert  places cells in fixed-capacity buckets (grid_init :38-62),
// k_sweep          runs connect_proc (:70-129) for every non-membrane cell:
//                  the lower part of its own row is written directly, the
//                  upper parts of its partners are appended with atomics,
// k_finish         sorts the upper parts, carries gap-junction
//                  values over from the previous rows by cell uid
//                  (gj_refresh :133-152), picks the dermis (:158-185) and
//                  leaves the buckets empty for the next build.
#include "epi_dev.h"
#include "launch.h"
#include "epi_group.h"
#include "gj_carry.h"
#include "field_step.h"

namespace epi {

// calc_zzmax (proc.cpp:34-43): z values that matter are positive, where the
// IEEE bit order is the numeric order
__device__ __forceinline__ bool counts_zzmax(uint8_t s) { return s == DEAD || s == ALIVE || s == MUSUME || s == FIX; }
// a lane's maximum into the tissue's, which was cleared before this launch
// and only grows during it
__device__ __forceinline__ void zzmax_add(Status* st, double m) {
  for (int o = 32; o > 0; o >>= 1) {
    const double v = __shfl_down(m, o, 64);
    if (m < v) m = v;
  }
  const unsigned long long mb = (unsigned long long)__double_as_longlong(m);
  if ((threadIdx.x & 63) == 0 && m > 0 &&
      mb > __hip_atomic_load(&st->zzmax_bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax(&st->zzmax_bits, mb);
}

// grid_init (:38-62); with fix != 0 it first applies cell_pos_periodic_fix
// (cellmanager.cpp:395-414) to the cell, which touches only that cell.
// In a step (STEP) the launch carries two more pieces of work that need only
// what it reads or nothing, and that would otherwise be three launches on the
// side stream before the stamping (zz_set, zzmax, clear: 12 us of a step of
// 420 cells with their gaps): calc_zzmax over the same cells (the maximum was
// cleared by the renewal), and, in the blocks from cell_blocks on, the emptying of
// the voxel maps, which nothing reads between the last step's B sweep or solve
// and this step's stamping.
__device__ __forceinline__ void insert_cells(const Tis& t, int pb, int fix, bool step, int nblocks) {
  Status* st = t.st;
  const int n = st->n, start = t.nmemb + t.nder;
  double zmax = 0;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += nblocks * blockDim.x) {
    double x = t.pos[pb][0][c], y = t.pos[pb][1][c];
    const double z = t.pos[pb][2][c];
    const double r = t.radius[c];
    if (step && c >= start && zmax < z && counts_zzmax(t.state[c])) zmax = z;
    if (fix) {
      if (x > t.LX) { x = x - t.LX; t.pos[pb][0][c] = x; }
      else if (x < 0) { x = x + t.LX; t.pos[pb][0][c] = x; }
      if (y > t.LY) { y = y - t.LY; t.pos[pb][1][c] = y; }
      else if (y < 0) { y = y + t.LY; t.pos[pb][1][c] = y; }
    }
    const long aix = (long)((0.5 * t.LX - p_diff_x(t, 0.5 * t.LX, x)) / AREA_GRID);
    const long aiy = (long)((0.5 * t.LY - p_diff_y(t, 0.5 * t.LY, y)) / AREA_GRID);
    const long aiz = (long)((min0(z)) / AREA_GRID);
    t.pk[pb][c] = make_double4(x, y, z, r);
    t.bcnt[c] = 0;
    t.nlo[c] = 0;
    if (aix >= t.ANX || aiy >= t.ANY || aiz >= t.ANZ || aix < 0 || aiy < 0 || aiz < 0) {
      set_err(st, ERR_OUT_OF_GRID);
      t.bucket_of[c] = -1;
      continue;
    }
    const int b = (int)((aix * t.ANY + aiy) * t.ANZ + aiz);
    t.bucket_of[c] = b;
    int* const head = t.bucket + (size_t)b * BUCKET_HEAD;
    const int slot = atomicAdd(head, 1);
    // the reference asserts fewer than N3 = 200 cells per bucket (:59)
    if (slot + 1 >= N3 || slot >= t.bcap) { set_err(st, ERR_CAPACITY); continue; }
    if (slot < BUCKET_HEAD - 1) head[1 + slot] = c;
    else t.bucket_rest[(size_t)b * bucket_more(t.bcap) + slot - (BUCKET_HEAD - 1)] = c;
  }
  if (step) zzmax_add(st, zmax);
}

template <bool STEP>
__global__ void __launch_bounds__(256) k_bucket_insert(const Tis* __restrict__ T, int pb, int fix, int cell_blocks) {
  const Tis& t = T[blockIdx.y];
  if (STEP && (int)blockIdx.x >= cell_blocks) map_clear(t, blockIdx.x - cell_blocks, gridDim.x - cell_blocks);
  else insert_cells(t, pb, fix, STEP, cell_blocks);
}

// connect_proc (:70-129): the 5x5x5 sweep, periodic in x, y and z, buckets
// in ascending (j, k, l) with cells in ascending index inside a bucket.
// A group of G = 32 lanes (64: a launch shape for few cells) takes one cell.
//
// What bounds it is the chain of memory round trips where the GPU is mostly
// idle and the instructions where it is full, so the group works on a flat
// list of candidates: a lane asks for the heads of 128 / G consecutive buckets
// of the 125 in sweep order at once (bucket q is (j, k, l) = (q / 25,
// q / 5 % 5, q % 5); a head is its count and seven cells), the cells below the group's own go to a list in LDS with their bucket, and
// the lanes take the list's entries in turn, so a position is read and tested
// only for a real candidate and no lane waits for a full column.  The hits
// are put in sweep order by rank of (bucket, cell), which needs no order in
// the buckets, and the lanes take them in turn again for the appends to the
// partners' rows (an atomic whose result the store needs).  More candidates
// or hits than the lists hold go through sweep_crowded.
// Measured against buckets sorted by a launch of their own and one column of
// five buckets per lane, walked one after the other, sort and sweep: 16.1 ->
// 9.5 us (a tissue of 420 cells), 26.7 -> 12.2 (4,300), 45.2 -> 35.8 (36,400),
// 290 -> 280 (32 tissues, 292,000 cells).
constexpr int SWEEP_C = 384;   // candidates of a cell
constexpr int SWEEP_H = 64;    // hits of a cell
constexpr int SWEEP_Q = 36;    // a hit's key: its bucket above the cell index

__device__ __forceinline__ bool sweep_hit(const Tis& t, const P3& pc, double rc, const double4& po) {
  const double diffx = p_diff_x(t, pc.x, po.x);
  const double diffy = p_diff_y(t, pc.y, po.y);
  const double diffz = pc.z - po.z;
  const double rad_sum = rc + po.w;
  const double lj = t.prm.LJ_THRESH;
  return diffx * diffx + diffy * diffy + diffz * diffz <= lj * lj * rad_sum * rad_sum;
}

// v mod A for the indices a sweep meets: 0 <= v < 2 A + 2, or any v where A = 1
__device__ __forceinline__ int wrap_index(int v, int A) {
  v -= v >= A ? A : 0;
  v -= v >= A ? A : 0;
  return A == 1 ? 0 : v;
}
struct SweepAt { int x, y, z; };   // the bucket a sweep is around
__device__ __forceinline__ int sweep_bucket(const Tis& t, const SweepAt& at, int q) {
  const int bx = wrap_index(at.x - 2 + q / 25 + t.ANX, t.ANX), by = wrap_index(at.y - 2 + q / 5 % 5 + t.ANY, t.ANY),
            bz = wrap_index(at.z - 2 + q % 5 + t.ANZ, t.ANZ);
  return (bx * t.ANY + by) * t.ANZ + bz;
}

__device__ __forceinline__ void sweep_append(const Tis& t, int c, int o) {
  const int slot = atomicAdd(&t.bcnt[o], 1);
  if (slot < t.ns) t.btmp[(size_t)o * t.ns + slot] = c;
}

// a sweep of any size, without lists: each lane counts its buckets' hits, and
// writes them in order, each time the least cell above the last one
template <int G>
__device__ __forceinline__ int sweep_crowded(const Tis& t, const double4* pk, int c, const P3& pc, double rc,
                                             const SweepAt& at, int lane, int* row) {
  constexpr int NB = 128 / G;
  const int q1 = min(NB * lane + NB, 125);
  auto cell = [&](int b, int m) -> int {
    return m < BUCKET_HEAD - 1 ? t.bucket[(size_t)b * BUCKET_HEAD + 1 + m]
                               : t.bucket_rest[(size_t)b * bucket_more(t.bcap) + m - (BUCKET_HEAD - 1)];
  };
  int cnt = 0;
  for (int q = NB * lane; q < q1; q++) {
    const int b = sweep_bucket(t, at, q);
    const int sz = min(t.bucket[(size_t)b * BUCKET_HEAD], t.bcap);
    for (int m = 0; m < sz; m++) {
      const int o = cell(b, m);
      cnt += o < c && sweep_hit(t, pc, rc, pk[o]);
    }
  }
  int total;
  int off = group_exclusive_scan<G>(cnt, lane, &total);
  if (cnt)
    for (int q = NB * lane; q < q1; q++) {
      const int b = sweep_bucket(t, at, q);
      const int sz = min(t.bucket[(size_t)b * BUCKET_HEAD], t.bcap);
      for (int last = -1;;) {
        int best = c;
        for (int m = 0; m < sz; m++) {
          const int o = cell(b, m);
          if (o > last && o < best && sweep_hit(t, pc, rc, pk[o])) best = o;
        }
        if (best == c) break;
        if (off < t.ns) row[off] = best;
        off++;
        sweep_append(t, c, best);
        last = best;
      }
    }
  return total;
}

template <int G>
__device__ __forceinline__ void sweep_part(const Tis& t, int pb, int nb, int nblk) {
  constexpr int NB = 128 / G;   // buckets of a lane
  Status* st = t.st;
  const int n = st->n;
  const int ANX = t.ANX, ANY = t.ANY, ANZ = t.ANZ, bcap = t.bcap, ns = t.ns;
  const int lane = threadIdx.x & (G - 1);
  const int groups = nblk * (blockDim.x / G);
  __shared__ int s_cand[256 / G][SWEEP_C];
  __shared__ uint8_t s_cq[256 / G][SWEEP_C];
  __shared__ unsigned long long s_hit[256 / G][SWEEP_H];
  int* const cand = s_cand[threadIdx.x / G];
  uint8_t* const cq = s_cq[threadIdx.x / G];
  unsigned long long* const hits = s_hit[threadIdx.x / G];
  const unsigned long long below = (1ull << lane) - 1;   // lanes of the group before this one
  // a ballot's bits of this group
  auto group_bits = [&](bool p) {
    const unsigned long long b = __ballot(p);
    return G == 64 ? b : b >> (threadIdx.x & 32) & 0xffffffffull;
  };
  int* const col = t.col[nb];
  const double4* const pk = t.pk[pb];
  for (int c = t.nmemb + blockIdx.x * (blockDim.x / G) + threadIdx.x / G; c < n; c += groups) {
    const double4 pq = pk[c];
    const P3 pc{pq.x, pq.y, pq.z};
    const double rc = pq.w;
    const long lx = (long)(pc.x / AREA_GRID);
    const long ly = (long)(pc.y / AREA_GRID);
    const long lz = (long)(pc.z / AREA_GRID);
    const bool bad = lx >= ANX || ly >= ANY || lz >= ANZ || lx < 0 || ly < 0 || lz < 0;
    if (bad) {
      if (lane == 0) set_err(st, ERR_OUT_OF_GRID);
      continue;
    }
    const SweepAt at{(int)lx, (int)ly, (int)lz};
    int bk[NB];
    int4 w4[NB][2];
#pragma unroll
    for (int u = 0; u < NB; u++) {
      bk[u] = sweep_bucket(t, at, min(NB * lane + u, 124));   // past the last: its head again, counted empty below
      const int4* const head = reinterpret_cast<const int4*>(t.bucket + (size_t)bk[u] * BUCKET_HEAD);
      w4[u][0] = head[0];
      w4[u][1] = head[1];
    }
    int sz[NB], cnt = 0, most = 0;
#pragma unroll
    for (int u = 0; u < NB; u++) {
      sz[u] = NB * lane + u < 125 ? min(w4[u][0].x, bcap) : 0;
      most = max(most, sz[u]);
      const int w[7] = {w4[u][0].y, w4[u][0].z, w4[u][0].w, w4[u][1].x, w4[u][1].y, w4[u][1].z, w4[u][1].w};
#pragma unroll
      for (int v = 0; v < 7; v++) cnt += v < sz[u] && w[v] < c;   // a slot past the count holds a past build's cell
    }
    int nc;
    int at_c = group_exclusive_scan<G>(cnt, lane, &nc);
    if (nc <= SWEEP_C) {
#pragma unroll
      for (int u = 0; u < NB; u++) {
        const int w[7] = {w4[u][0].y, w4[u][0].z, w4[u][0].w, w4[u][1].x, w4[u][1].y, w4[u][1].z, w4[u][1].w};
#pragma unroll
        for (int v = 0; v < 7; v++)
          if (v < sz[u] && w[v] < c) {
            cand[at_c] = w[v];
            cq[at_c++] = (uint8_t)(NB * lane + u);
          }
      }
    }
    // buckets of more than seven cells: four more of each at a time
    for (int m0 = BUCKET_HEAD - 1; nc <= SWEEP_C && group_bits(m0 < most); m0 += 4) {
#pragma unroll
      for (int u = 0; u < NB; u++)
        w4[u][0] = *reinterpret_cast<const int4*>(t.bucket_rest + (size_t)bk[u] * bucket_more(bcap) +
                                                  (m0 < sz[u] ? m0 - (BUCKET_HEAD - 1) : 0));
      int more = 0;
#pragma unroll
      for (int u = 0; u < NB; u++) {
        const int w[4] = {w4[u][0].x, w4[u][0].y, w4[u][0].z, w4[u][0].w};
#pragma unroll
        for (int v = 0; v < 4; v++) more += m0 + v < sz[u] && w[v] < c;
      }
      int add;
      int at_m = nc + group_exclusive_scan<G>(more, lane, &add);
      nc += add;
      if (nc > SWEEP_C) break;
#pragma unroll
      for (int u = 0; u < NB; u++) {
        const int w[4] = {w4[u][0].x, w4[u][0].y, w4[u][0].z, w4[u][0].w};
#pragma unroll
        for (int v = 0; v < 4; v++)
          if (m0 + v < sz[u] && w[v] < c) {
            cand[at_m] = w[v];
            cq[at_m++] = (uint8_t)(NB * lane + u);
          }
      }
    }
    int total = 0;
    if (nc <= SWEEP_C) {
      wave_sync();
      // 2 G candidates at a time, both positions asked for together
      for (int i0 = 0; i0 < nc; i0 += 2 * G) {
        int o[2], q[2];
        double4 po[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
          const int i = i0 + k * G + lane;
          o[k] = i < nc ? cand[i] : c;
          q[k] = i < nc ? cq[i] : 0;
          po[k] = pk[o[k]];
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {
          const bool hit = o[k] != c && sweep_hit(t, pc, rc, po[k]);
          const unsigned long long hb = group_bits(hit);
          const int i = total + __popcll(hb & below);
          if (hit && i < SWEEP_H) hits[i] = (unsigned long long)q[k] << SWEEP_Q | (unsigned)o[k];
          total += __popcll(hb);
        }
      }
    }
    int* const row = col + (size_t)c * ns;
    if (nc > SWEEP_C || total > SWEEP_H) {
      total = sweep_crowded<G>(t, pk, c, pc, rc, at, lane, row);
    } else {
      wave_sync();
      for (int i = lane; i < total; i += G) {
        const unsigned long long key = hits[i];
        const int o = (int)key;   // the key's low 32 bits
        int rk = 0;
        for (int k = 0; k < total; k++) rk += hits[k] < key;
        if (rk < ns) row[rk] = o;
        sweep_append(t, c, o);
      }
      wave_sync();   // the lists are the next cell's from here
    }
    if (lane == 0) t.nlo[c] = total;
  }
}

// Blocks [0, sweep_blocks) sweep; with MS lanes per cell the rest stamp the
// voxel maps (MS = 0: there is none), which like the sweep needs only what the
// insertion left.
template <int G, int MS>
__global__ void __launch_bounds__(256) k_sweep(const Tis* __restrict__ T, int pb, int nb, int sweep_blocks) {
  const Tis& t = T[blockIdx.y];
  if constexpr (MS > 0) {
    if ((int)blockIdx.x >= sweep_blocks) {
      map_stamp_part<MS>(t, pb, blockIdx.x - sweep_blocks, gridDim.x - sweep_blocks);
      return;
    }
  }
  sweep_part<G>(t, pb, nb, sweep_blocks);
}

// Row assembly, gj carry-over and dermis.  A group of KG lanes owns one
// cell.  Rows of at most KCAP entries are assembled in LDS: the lower part
// (written by k_sweep in sweep order) and the upper partners (gathered in
// k_sweep in arbitrary order, placed here by rank since they are distinct),
// each entry with its uid.  The previous row's uids and gj values are staged
// in LDS too and each lane resolves the gap junction of its entries there
// (gj_refresh :133-152: a directed edge keeps its value while it stays in the
// list, a new edge starts at gj_init).
// The dermis (find_dermis :158-172: the first MEMB entry of minimal distance
// in list order, strictly below LX^2) is a lexicographic (distance, entry)
// minimum over the group.  Longer rows take the same steps through global
// memory.
// The time is the chain of round trips: the cell's words; the rows' first
// KPRE entries (unconditional: a row has ROW_SLOTS_MIN slots) with the
// previous row's length and values; the uids of both.  The launch also does
// what the next build needs of this one (every cell's row is its own from
// here, the uids are kept beside the rows they number, the buckets are
// emptied): a launch of its own for that took 2.5 to 4.4 us and its gap.
constexpr int KG = 16;
constexpr int KCAP = 64;   // rows (and previous rows) longer than this take the global-memory path
constexpr int KPRE = 2;    // entries of each row a lane asks for before it knows the lengths
constexpr int K_BLOCK = 128;
constexpr int K_GROUPS = K_BLOCK / KG;
static_assert(KPRE * KG <= ROW_SLOTS_MIN, "the entries read before the length lie inside a row");

__device__ __forceinline__ void finish_part(const Tis& t, int pb, int nb, int nblk) {
  Status* st = t.st;
  const int n = st->n;
  const int ob = 1 - nb;
  __shared__ int s_row[K_GROUPS][KCAP];
  __shared__ int s_bt[K_GROUPS][KCAP];
  __shared__ long long s_ru[K_GROUPS][KCAP];
  __shared__ long long s_ou[K_GROUPS][KCAP];
  __shared__ double s_og[K_GROUPS][KCAP];
  const int lane = threadIdx.x & (KG - 1);
  const int grp = threadIdx.x / KG;
  const double gj_init = t.prm.gj_init, THRESH_SP = t.prm.THRESH_SP;   // read before any store (a store could alias the descriptor)
  int mylen = 0;
  const int stride = nblk * K_GROUPS;
  for (int c = blockIdx.x * K_GROUPS + grp; c < n; c += stride) {
    const bool memb = c < t.nmemb;
    const int base = memb ? MEMB_ADJ : 0;
    const int na0 = t.nlo[c];
    const int nbh = t.bcnt[c];
    const int src = t.src_row[c];
    const int bkt = t.bucket_of[c];
    const long long my_uid = t.uid[c];
    const uint8_t s = t.state[c];
    const P3 pc = ld_pos(t, pb, c);
    const int pair = t.pair[c], dermis = t.dermis[c], rdt = t.rest_div_times[c];
    const bool strong = t.agek[c] > THRESH_SP;
    const int na = memb ? 0 : na0;
    const int len = base + na + nbh;
    int* const row = t.col[nb] + (size_t)c * t.ns;
    const int* bt = t.btmp + (size_t)c * t.ns;
    const int osrc = src >= 0 ? src : c;
    const int* orow = t.col[ob] + (size_t)osrc * t.ns;
    const double* og = t.gj[ob] + (size_t)osrc * t.ns;
    const int* const lo = memb ? t.memb6 + 6 * c : row;   // the row's first part: base + na entries
    const int nl = base + na;
    int lo_e[KPRE], bt_e[KPRE], or_e[KPRE];
    double og_e[KPRE];
#pragma unroll
    for (int k = 0; k < KPRE; k++) {
      const int i = lane + k * KG;
      lo_e[k] = lo[i < nl ? i : 0];
      bt_e[k] = bt[i];
      or_e[k] = orow[i];
      og_e[k] = og[i];
    }
    const int olen = src >= 0 ? t.nlen[ob][src] : 0;
    if (lane == 0) {
      t.src_row[c] = c;
      t.old_uid[nb][c] = my_uid;
      if (bkt >= 0) t.bucket[(size_t)bkt * BUCKET_HEAD] = 0;
    }
    // the reference asserts a list shorter than N2 = 400 (:122)
    if (len >= MAX_CONN || len > t.ns) {
      if (lane == 0) { set_err(st, ERR_CAPACITY); t.nlen[nb][c] = 0; }
      continue;
    }
    mylen = max(mylen, len);
    const bool fits = len <= KCAP;
    const bool staged = olen <= KCAP;
    if (lane == 0) t.nlen[nb][c] = len;
    // the uids: entries past a row's end read cell 0's and are not kept
    long long lo_u[KPRE], bt_u[KPRE], or_u[KPRE];
#pragma unroll
    for (int k = 0; k < KPRE; k++) {
      const int i = lane + k * KG;
      lo_u[k] = t.uid[i < nl ? lo_e[k] : 0];
      bt_u[k] = t.uid[i < nbh ? bt_e[k] : 0];
      or_u[k] = t.old_uid[ob][i < olen ? or_e[k] : 0];
    }
    if (fits) {
#pragma unroll
      for (int k = 0; k < KPRE; k++) {
        const int i = lane + k * KG;
        if (i < nl) { s_row[grp][i] = lo_e[k]; s_ru[grp][i] = lo_u[k]; }
        if (i < nbh) s_bt[grp][i] = bt_e[k];
      }
      for (int i = lane + KPRE * KG; i < nl; i += KG) {
        const int o = lo[i];
        s_row[grp][i] = o;
        s_ru[grp][i] = t.uid[o];
      }
      for (int i = lane + KPRE * KG; i < nbh; i += KG) s_bt[grp][i] = bt[i];
    } else if (memb) {
      if (lane < MEMB_ADJ) row[lane] = lo[lane];
    }
    if (staged) {
#pragma unroll
      for (int k = 0; k < KPRE; k++) {
        const int i = lane + k * KG;
        if (i < olen) { s_ou[grp][i] = or_u[k]; s_og[grp][i] = og_e[k]; }
      }
      for (int f = lane + KPRE * KG; f < olen; f += KG) {
        s_ou[grp][f] = t.old_uid[ob][orow[f]];
        s_og[grp][f] = og[f];
      }
    }
    wave_sync();
    {
      const int* const b = fits ? s_bt[grp] : bt;
      int k = 0;
      for (int i = lane; i < nbh; i += KG, k++) {
        const int v = b[i];
        int rk = 0;
        for (int m = 0; m < nbh; m++) rk += b[m] < v;
        if (fits) {
          s_row[grp][nl + rk] = v;
          s_ru[grp][nl + rk] = k == 0 ? bt_u[0] : k == 1 ? bt_u[1] : t.uid[v];
        } else {
          row[nl + rk] = v;
        }
      }
    }
    wave_sync();
    const bool want_dermis = !memb && c >= t.nmemb + t.nder && (s == FIX || s == MUSUME);
    const int* const r = fits ? s_row[grp] : row;
    double bd = t.LX * t.LX;
    int be = 0x7fffffff;
    double* const g = t.gj[nb] + (size_t)c * t.ns;
    for (int e = lane; e < len; e += KG) {
      const int o = r[e];
      if (fits && (e < base || e >= nl)) row[e] = o;
      const long long u = fits ? s_ru[grp][e] : t.uid[o];
      const long long* const ou = s_ou[grp];
      const int q = gj_carry_slot(e, olen, u, [&](int k) { return staged ? ou[k] : t.old_uid[ob][orow[k]]; });
      g[e] = q < 0 ? gj_init : staged ? s_og[grp][q] : og[q];
      if (want_dermis && t.state[o] == MEMB) {
        const double d = dist_sq(t, pc, ld_pos(t, pb, o));
        if (d < bd) { bd = d; be = e; }   // entries of a lane ascend
      }
    }
    int found = dermis;
    if (want_dermis) {
#pragma unroll
      for (int o = 1; o < KG; o <<= 1) {
        const double d2 = __shfl_xor(bd, o, KG);
        const int e2 = __shfl_xor(be, o, KG);
        if (d2 < bd || (d2 == bd && e2 < be)) { bd = d2; be = e2; }
      }
      found = be == 0x7fffffff ? -1 : r[be];
      if (lane == 0) t.dermis[c] = found;
    }
    if (lane == 0) t.fa[c] = force_attr(pair, found, rdt, s, strong);   // what the force laws read (k_mech.hip)
    wave_sync();
  }
  // maxlen only grows: a wave that cannot raise it skips the atomic, which
  // would otherwise serialise every wave of the launch on one address
  for (int o = 32; o > 0; o >>= 1) mylen = max(mylen, __shfl_down(mylen, o, 64));
  if ((threadIdx.x & 63) == 0 && mylen > __hip_atomic_load(&st->maxlen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax(&st->maxlen, mylen);
}

// Blocks [0, finish_blocks) finish the rows; with ZB planes per tile the rest
// take the B stencil (ZB = 0: there is none), which needs the maps that the
// sweep's launch stamped.
template <int ZB>
__global__ void __launch_bounds__(K_BLOCK) k_finish(const Tis* __restrict__ T, int pb, int nb, int finish_blocks, int bp,
                                                    int xcd) {
  const Tis& t = T[blockIdx.y];
  if constexpr (ZB > 0) {
    if ((int)blockIdx.x >= finish_blocks) {
      ext_stim_part<ZB>(t, bp, xcd, blockIdx.x - finish_blocks, gridDim.x - finish_blocks);
      return;
    }
  }
  finish_part(t, pb, nb, finish_blocks);
}

__global__ void __launch_bounds__(256) k_zzmax(const Tis* __restrict__ T, int pb) {
  const Tis& t = T[blockIdx.y];
  Status* st = t.st;
  const int n = st->n;
  double m = 0;
  for (int c = t.nmemb + t.nder + blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    if (counts_zzmax(t.state[c])) {
      const double z = t.pos[pb][2][c];
      if (m < z) m = z;
    }
  }
  zzmax_add(st, m);
}

__global__ void k_zz_set(const Tis* __restrict__ T) {
  const Tis& t = T[blockIdx.x];
  if (threadIdx.x == 0) t.st->zzmax_bits = 0ull;
}

// CellManager::output's per-cell record (cellmanager.cpp:451-538) packed for
// an asynchronous download: one thread per cell; touch is an ALIVE cell with
// a DEAD cell in its list, as output computes it
__global__ void __launch_bounds__(256) k_out_pack(const Tis* __restrict__ T, int tissue, int pb, int cp, int cb,
                                                  int n, long long m, char* __restrict__ out) {
  const Tis& t = T[tissue];
  double* __restrict__ f = reinterpret_cast<double*>(out + OUT_HDR);
  int* __restrict__ iv = reinterpret_cast<int*>(out + OUT_HDR + 8 * OUT_NF64 * m);
  uint8_t* __restrict__ bv = reinterpret_cast<uint8_t*>(out + OUT_HDR + (8 * OUT_NF64 + 4 * OUT_NI32) * m);
  if (blockIdx.x == 0 && threadIdx.x == 0) *reinterpret_cast<int*>(out) = t.st->n;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    const uint8_t s = t.state[c];
    uint8_t touch = 0;
    if (s == ALIVE) {
      const int len = t.nlen[cb][c];
      const int* row = t.col[cb] + (size_t)c * t.ns;
      for (int e = 0; e < len; e++)
        if (t.state[row[e]] == DEAD) {
          touch = 1;
          break;
        }
    }
    const double v[OUT_NF64] = {t.radius[c], t.ageb[c], t.agek[c], t.ca2p[cp][c], t.pos[pb][0][c],
                                t.pos[pb][1][c], t.pos[pb][2][c], t.ca2p_avg[c], t.ex_fat[c], t.in_fat[c],
                                t.spr_nat_len[c]};
#pragma unroll
    for (int k = 0; k < OUT_NF64; k++) f[k * m + c] = v[k];
    iv[c] = t.rest_div_times[c];
    iv[m + c] = t.pair[c];
    iv[2 * m + c] = t.fix_origin[c];
    bv[c] = s;
    bv[m + c] = touch;
  }
}

void launch_out_pack(hipStream_t s, const Tis* dT, int tissue, int pb, int cp, int cb, int n, long long m,
                     char* out) {
  const unsigned g = (unsigned)std::max(1, std::min((n + 255) / 256, 4096));
  EPI_LAUNCH(K_OUT_PACK, k_out_pack, dim3(g), dim3(256), 0, s, dT, tissue, pb, cp, cb, n, m, out);
}

void launch_connect_insert(hipStream_t s, const Tis* dT, int ntis, int pb, int max_n, unsigned clear_blocks) {
  const unsigned gc = (max_n + 255) / 256;
  if (clear_blocks) {
    EPI_LAUNCH(K_BUCKET_INSERT, k_bucket_insert<true>, dim3(gc + clear_blocks, ntis), dim3(256), 0, s, dT, pb, 1,
               (int)gc);
  } else {
    EPI_LAUNCH(K_BUCKET_INSERT, k_bucket_insert<false>, dim3(gc, ntis), dim3(256), 0, s, dT, pb, 0, (int)gc);
  }
}

namespace {
// A whole wave takes a cell where that leaves the GPU's waves few: fewer
// buckets a lane, a shorter chain (a step of 160 swept cells 43.5 -> 41.7 us, of
// 2,000 3 % less, of 20,000 the same, 32 tissues of 140,000 1 % slower).
constexpr long long SWEEP_WAVE_CELLS = 8192;
template <int MS>
void launch_sweep(hipStream_t s, const Tis* dT, int ntis, int pb, int nb, int max_n, int max_swept, int sweep_wave) {
  const bool wave = sweep_wave || (long long)max_swept * ntis <= SWEEP_WAVE_CELLS;
  const unsigned gs = wave ? (max_swept + 3) / 4 : (max_swept + 7) / 8, gm = ((unsigned)max_n * MS + 255) / 256;
  const int id = sweep_wave ? K_SWEEP_WAVE : K_SWEEP;   // timed under the shape asked for
  const auto kfn = wave ? k_sweep<64, MS> : k_sweep<32, MS>;
  EPI_LAUNCH(id, kfn, dim3(gs + gm, ntis), dim3(256), 0, s, dT, pb, nb, (int)gs);
}
}  // namespace

void launch_connect_rest(hipStream_t s, const Tis* dT, int ntis, int pb, int nb, int max_n, int max_swept,
                         int sweep_wave) {
  launch_sweep<0>(s, dT, ntis, pb, nb, max_n, max_swept, sweep_wave);
  const unsigned gk = (max_n + K_GROUPS - 1) / K_GROUPS;
  EPI_LAUNCH(K_FINISH, k_finish<0>, dim3(gk, ntis), dim3(K_BLOCK), 0, s, dT, pb, nb, (int)gk, 0, 0);
}

void launch_connect_field(hipStream_t s, const Tis* dT, int ntis, int pb, int nb, int bp, int max_n, int max_swept,
                          long long b_tiles, const Tuning& tu) {
  static_assert(K_BLOCK == BUILD_FIELD_BS, "the caller counts tiles of this many points");
  if (tu.map_lanes == 16) launch_sweep<16>(s, dT, ntis, pb, nb, max_n, max_swept, tu.sweep_wave);
  else if (tu.map_lanes == 4) launch_sweep<4>(s, dT, ntis, pb, nb, max_n, max_swept, tu.sweep_wave);
  else launch_sweep<1>(s, dT, ntis, pb, nb, max_n, max_swept, tu.sweep_wave);
  // a multiple of 8 blocks, so that the XCD split applies
  const unsigned gk = (max_n + K_GROUPS - 1) / K_GROUPS;
  const unsigned gb = (unsigned)((std::min(std::max(b_tiles, 1LL), 1LL << 24) + 7) / 8 * 8);
  by_zb(tu.b_zb, [&](auto zbc) {
    EPI_LAUNCH(K_FINISH, k_finish<decltype(zbc)::value>, dim3(gk + gb, ntis), dim3(K_BLOCK), 0, s, dT, pb, nb, (int)gk, bp,
               tu.b_xcd);
  });
}

void launch_connect(hipStream_t s, const Tis* dT, int ntis, int pb, int nb, int max_n, int max_swept, int sweep_wave) {
  launch_connect_insert(s, dT, ntis, pb, max_n, 0);
  launch_connect_rest(s, dT, ntis, pb, nb, max_n, max_swept, sweep_wave);
}

void launch_zzmax(hipStream_t s, const Tis* dT, int ntis, int pb, int max_n) {
  EPI_LAUNCH(K_ZZ_SET, k_zz_set, dim3(ntis), dim3(64), 0, s, dT);
  dim3 gc((max_n + 255) / 256, ntis);
  EPI_LAUNCH(K_ZZMAX, k_zzmax, gc, dim3(256), 0, s, dT, pb);
}

}  // namespace epi
