// k_renew.hip -- cell_state_renew (cell_state_renew.cpp:400-429) on CDNA4.
//
// The reference walks the non-membrane cells in one loop; each cell only
// changes itself and the daughter it appends, but the replayed random draws
// are consumed in loop order and a division consumes extra draws.  So:
//   k_renew_cells  every cell that needs no draw applies its own rule; the
//                  cells that need one, and those that go, are packed in index
//                  order per block of 256 cells;
//   k_renew_tail   one workgroup per tissue places the packed lists behind
//                  each other, decides the divisions 256 ready cells a round (a
//                  ballot finds the first division; draws after it shift by
//                  its direction draws), applies the ready cells' rule
//                  (daughters are written at n_old + division rank, parent
//                  order), and then takes remove_exec's swap-with-tail and
//                  pair_disperse from the higher-index partner.
// k_renew_one does both in one launch where the tissues are small.
#include "epi_dev.h"
#include "launch.h"
#include "epi_group.h"

namespace epi {

// cell_state_renew.cpp:17-119: the rates and thresholds are runtime values
// (Tis::prm); these two are fixed by the reference's code
constexpr double stoch_corr_coef = 1;
constexpr double PI_D = 3.14159265358979323846;

// an error of the renewal; one of the forces before it comes first
__device__ __forceinline__ void renew_err(Status* st, int e) { set_err(st, st->force_err ? st->force_err : e); }

// The constants of the renewal laws, copied out of the tissue's record once,
// before a kernel's first store: the compiler cannot tell a cell store from
// the descriptor, so a record field read after a store would be loaded from
// memory again.
struct RenewK {
  double DT_Cell, THRESH_DEAD, THRESH_SP, ca2p_init, stoch_div_time_ratio, S2, accel_div, eps_kb, alpha_b, S0, eps_ks,
      accel_diff, alpha_k, eps_kk, S1, ubar, delta_lipid, delta_sig_r1, lipid_rel, lipid, ADHE_CONST, DISA;
};
__device__ __forceinline__ RenewK renew_k(const Params& pm) {
  return RenewK{pm.DT_Cell, pm.THRESH_DEAD, pm.THRESH_SP, pm.ca2p_init, pm.stoch_div_time_ratio, pm.S2, pm.accel_div,
                pm.eps_kb, pm.alpha_b, pm.S0, pm.eps_ks, pm.accel_diff, pm.alpha_k, pm.eps_kk, pm.S1, pm.ubar,
                pm.delta_lipid, pm.delta_sig_r1, pm.lipid_rel, pm.lipid, pm.ADHE_CONST, pm.DISA_conn_num_thresh};
}

__device__ __forceinline__ double weighted_eps_kb(const RenewK& k, uint8_t malig) {
  return malig ? k.accel_div * k.eps_kb : k.eps_kb;
}

// what the renewal reads of a cell, loaded in one round trip
struct RCell {
  double ageb, agek, div_age_thresh, ca2p_avg, in_fat, ex_fat;
  int dermis, pair, rest_div_times, nlen;
  uint8_t s, is_malignant;
};
__device__ __forceinline__ RCell load_rcell(const Tis& t, int cb, int c) {
  return RCell{t.ageb[c], t.agek[c], t.div_age_thresh[c], t.ca2p_avg[c], t.in_fat[c], t.ex_fat[c], t.dermis[c], t.pair[c],
               t.rest_div_times[c], t.nlen[cb][c], t.state[c], t.is_malignant[c]};
}

// is_divide_ready without the draw (:147-155), with the MUSUME/FIX guards of
// _MUSUME_state_renew (:282-298) and _FIX_state_renew (:308-318)
__device__ __forceinline__ bool needs_draw(const RenewK& k, const RCell& r) {
  if (r.s == FIX) {
    if (r.dermis < 0) return false;
  } else if (r.s == MUSUME) {
    if (r.dermis < 0 && r.pair < 0) return false;
    if (!(r.rest_div_times > 0)) return false;
  } else {
    return false;
  }
  return r.pair < 0 && (r.ageb >= r.div_age_thresh * (1.0 - k.stoch_div_time_ratio));
}

__device__ __forceinline__ bool to_remove(const RenewK& k, const RCell& r) {
  return (r.s == DEAD || r.s == AIR) && r.agek >= k.ADHE_CONST && (double)r.nlen <= k.DISA;
}

// ageing and lipid laws (:31-119)
__device__ __forceinline__ double ageb_const(const RenewK& k, double ca2p_avg, uint8_t malig) {
  return weighted_eps_kb(k, malig) * (k.S2 + k.alpha_b * min0(ca2p_avg - k.ca2p_init));
}
__device__ __forceinline__ double agek_ALIVE_const(const RenewK& k, double ca2p_avg, uint8_t malig) {
  return (malig ? k.accel_diff * k.eps_ks : k.eps_ks) * (k.S0 + k.alpha_k * min0(ca2p_avg - k.ca2p_init));
}
// k_lipid_release and k_lipid share their tanh: the arguments are the same, or
// differ in sign alone, which the subtraction, the division and tanh keep exactly
struct Lipid { double release, make; };
__device__ __forceinline__ Lipid lipid_rates(const RenewK& k, double ca2p_avg, double agek) {
  const double tc = tanh((ca2p_avg - k.ubar) / k.delta_sig_r1);
  const double ta = 1 + tanh((agek - k.THRESH_SP) / k.delta_lipid);
  return Lipid{0.25 * k.lipid_rel * (1 + tc) * ta, 0.25 * k.lipid * (1 + -tc) * ta};
}

// cell_divide (:227-270) for division rank k of parent c
__device__ void divide(const Tis& t, int pb, int cpar, int c, int k, int n_old, long long next_uid) {
  const int d = n_old + k;
  if (d >= t.cap) { renew_err(t.st, ERR_CAPACITY); return; }
  const P3 p = ld_pos(t, pb, c);
  const double divx = t.div_dir[3 * k], divy = t.div_dir[3 * k + 1], divz = t.div_dir[3 * k + 2];
  const double cav = t.ca2p[cpar][c];
  const double ipv = t.ip3[cpar][c];
  const int rdt = t.rest_div_times[c];
  const bool mus = t.state[c] == MUSUME;
  // daughter: CellManager::create(MUSUME, ...) (cellmanager.cpp:366-390)
  t.state[d] = MUSUME;
  t.fix_origin[d] = t.fix_origin[c];
  t.radius[d] = t.radius[c];
  t.div_age_thresh[d] = t.prm.agki_max;
  t.ca2p[0][d] = cav; t.ca2p[1][d] = cav;
  t.ca2p_avg[d] = cav;
  t.ip3[0][d] = ipv; t.ip3[1][d] = ipv;
  t.ex_inert[d] = t.ex_inert[c];
  t.agek[d] = 0; t.ageb[d] = 0; t.ex_fat[d] = 0; t.in_fat[d] = 0;
  const double delta_L = t.prm.delta_L;   // :231
  t.spr_nat_len[d] = delta_L;
  t.rest_div_times[d] = mus ? rdt - 1 : rdt;
  t.is_malignant[d] = t.is_malignant[c];
  t.pair[d] = c;
  t.dermis[d] = -1;
  t.diff_u[d] = 0;
  t.uid[d] = next_uid + k;
  t.cst[3 * d] = -1; t.cst[3 * d + 1] = -1; t.cst[3 * d + 2] = -1;
  t.src_row[d] = -1;
  t.touch_air[d] = 0;
  t.lat[3 * d] = 0; t.lat[3 * d + 1] = 0; t.lat[3 * d + 2] = 0;
  t.pos[pb][0][d] = p.x - divx * 0.5 * delta_L;
  t.pos[pb][1][d] = p.y - divy * 0.5 * delta_L;
  t.pos[pb][2][d] = p.z - divz * 0.5 * delta_L;
  // parent
  t.pair[c] = d;
  t.spr_nat_len[c] = delta_L;
  t.ageb[c] = 0;
  if (mus) t.rest_div_times[c] = rdt - 1;
  t.pos[pb][0][c] = p.x + divx * 0.5 * delta_L;
  t.pos[pb][1][c] = p.y + divy * 0.5 * delta_L;
  t.pos[pb][2][c] = p.z + divz * 0.5 * delta_L;
}

// the rule of a cell that needs no draw; 1 if it cornifies
__device__ __forceinline__ int renew_cell(const Tis& t, const RenewK& pm, const RCell& r, int c, long long ts) {
  const double cav = r.ca2p_avg, in_fat = r.in_fat;
  const uint8_t malig = r.is_malignant;
  const double DT_Cell = pm.DT_Cell;
  switch (r.s) {
    case ALIVE:   // _ALIVE_state_renew :347-358
      if (r.agek >= pm.THRESH_DEAD) {
        t.state[c] = DEAD;   // cornificate (cellmanager.cpp:48-53)
        t.cst[3 * c + 1] = ts;
        return 1;
      } else {
        const Lipid l = lipid_rates(pm, cav, r.agek);
        const double tmp = l.release * in_fat;
        t.in_fat[c] = in_fat + DT_Cell * (l.make * (1.0 - in_fat) - tmp);
        t.ex_fat[c] = r.ex_fat + DT_Cell * tmp;
        t.agek[c] = r.agek + DT_Cell * agek_ALIVE_const(pm, cav, malig);
      }
      break;
    case DEAD: case AIR:   // _DEAD_AIR_state_renew :330-341
      if (!to_remove(pm, r)) t.agek[c] = r.agek + DT_Cell * (pm.eps_kk * pm.S1);
      break;
    case FIX: case MUSUME: {
      if (r.s == FIX) {   // _FIX_state_renew :308-324
        if (r.dermis < 0) { renew_err(t.st, ERR_NO_DERMIS); break; }
      } else if (r.dermis < 0 && r.pair < 0) {   // _MUSUME_state_renew :282-302 (SYSTEM == WHOLE)
        t.state[c] = ALIVE;
        t.cst[3 * c] = ts;   // :287
        break;
      }
      t.ageb[c] = r.ageb + DT_Cell * ageb_const(pm, cav, malig);
      break;
    }
    default:
      break;
  }
  return 0;
}

// The cells of each block of 256 that need a draw, and those that go, in
// index order at the block's place of rd_list and rm_pack; the others' rule.
// No cell's rule touches another cell, and a cell that needs a draw waits for
// k_renew_tail, so the two parts need no order between them.
constexpr int RBLOCK = 256;

__global__ void __launch_bounds__(RBLOCK) k_renew_cells(const Tis* __restrict__ T, int cb) {
  const Tis& t = T[blockIdx.y];
  Status* st = t.st;
  __shared__ int s_rd[4], s_rm[4];
  const RenewK rk = renew_k(t.prm);
  const int start = t.nmemb + t.nder;
  const int n = st->n;
  const long long ts = st->timestep;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int ncorn = 0;
  for (int b = blockIdx.x; start + b * RBLOCK < n; b += gridDim.x) {
    const int c = start + b * RBLOCK + tid;
    const RCell r = load_rcell(t, cb, c < n ? c : n - 1);
    const bool rd = c < n && needs_draw(rk, r), rm = c < n && to_remove(rk, r);
    const unsigned long long mr = __ballot(rd), mm = __ballot(rm);
    if (lane == 0) { s_rd[wv] = __popcll(mr); s_rm[wv] = __popcll(mm); }
    __syncthreads();
    int at_r = b * RBLOCK, at_m = b * RBLOCK, nr = 0, nm = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      if (w < wv) { at_r += s_rd[w]; at_m += s_rm[w]; }
      nr += s_rd[w]; nm += s_rm[w];
    }
    const unsigned long long below = (1ull << lane) - 1;
    if (rd) t.rd_list[at_r + __popcll(mr & below)] = c;
    if (rm) t.rm_pack[at_m + __popcll(mm & below)] = c;
    if (tid == 0) { t.rd_n[b] = nr; t.rm_n[b] = nm; }
    if (c < n && !rd) ncorn += renew_cell(t, rk, r, c, ts);
    __syncthreads();   // the counts are the next block's from here
  }
  if (ncorn) atomicAdd(&st->sw, ncorn);
}

// the ordered part: one workgroup of RCHUNK lanes decides the divisions of up
// to RCHUNK ready cells at a time
constexpr int RCHUNK = 1024;
struct RenewSh {
  int ready[RCHUNK], der[RCHUNK], slot[RCHUNK];   // slot: the division's rank, or -1
  double thr[RCHUNK], rhs[RCHUNK];
  double rng[2 * RCHUNK];
  int off_r[RCHUNK], off_m[RCHUNK];
  int wcnt[16], wrm[16];
  int ndiv;
  long long cursor;
};

// the replay window for the next decisions (the caller synchronises)
__device__ __forceinline__ void renew_window(const Tis& t, RenewSh& sh, long long cur0) {
  for (int i = threadIdx.x; i < 2 * RCHUNK; i += RCHUNK) {
    const long long q = cur0 + i;
    sh.rng[i] = q < t.rng_n ? t.rng[q] : 2.0;
  }
}

// the first wave decides sh.ready[0 .. tot_r) in index order, RENEW_U * 64
// ready cells per round as long as none of them divides; draws past the window
// come from memory.  A round is a chain of LDS reads and a ballot, whatever it
// holds; a division adds its cell's positions and direction.
constexpr int RENEW_U = 4;
__device__ __forceinline__ void renew_decide(const Tis& t, RenewSh& sh, int pb, Status* st, int tot_r) {
  const int lane = threadIdx.x;
  const long long cur0 = sh.cursor;
  long long cur = cur0;
  int ndiv = sh.ndiv;
  auto draw = [&](long long dpos) {
    const long long wi = dpos - cur0;
    return wi < 2 * RCHUNK ? sh.rng[wi] : t.rng[dpos];
  };
  int i = 0;
  while (i < tot_r) {
    bool act[RENEW_U], dv[RENEW_U];
#pragma unroll
    for (int u = 0; u < RENEW_U; u++) {
      const int idx = i + 64 * u + lane;
      const long long dpos = cur + 64 * u + lane;
      act[u] = idx < tot_r;
      dv[u] = act[u] && dpos < t.rng_n && draw(dpos) * sh.thr[idx] <= sh.rhs[idx];
    }
    int f0 = -1;   // the first division's place in the round
#pragma unroll
    for (int u = RENEW_U - 1; u >= 0; u--) {
      const unsigned long long md = __ballot(dv[u]);
      if (md) f0 = 64 * u + __ffsll((long long)md) - 1;
    }
    const int k = f0 < 0 ? min(64 * RENEW_U, tot_r - i) : f0;   // cells of the round that do not divide
    // the cells up to the first division took their draws
    if (cur + min(k + (f0 >= 0), tot_r - i) > t.rng_n && lane == 0) renew_err(st, ERR_RNG_EXHAUSTED);
#pragma unroll
    for (int u = 0; u < RENEW_U; u++)
      if (64 * u + lane < k) sh.slot[i + 64 * u + lane] = -1;
    cur += k;
    i += k;
    if (f0 < 0) continue;
    int att = 0;
    if (lane == (f0 & 63)) {
      // div_direction (:192-217) with draws after the decision draw
      const P3 me = ld_pos(t, pb, sh.ready[i]), dm = ld_pos(t, pb, sh.der[i]);
      const double nvx = p_diff_x(t, me.x, dm.x);
      const double nvy = p_diff_y(t, me.y, dm.y);
      const double nvz = me.z - dm.z;
      const double norm = sqrt(nvx * nvx + nvy * nvy + nvz * nvz);
      const double nx = nvx / norm, ny = nvy / norm, nz = nvz / norm;
      double ox, oy, oz, sum;
      long long dp = cur + 1;
      do {
        if (dp + 1 >= t.rng_n) { renew_err(st, ERR_RNG_EXHAUSTED); ox = 1; oy = 0; oz = 0; att++; break; }
        const double rand_theta = PI_D * draw(dp);
        const double cr1 = cos(rand_theta);
        const double sr1 = sin(rand_theta);
        const double rand_phi = 2 * PI_D * draw(dp + 1);
        const double cr2 = cos(rand_phi);
        const double sr2 = sin(rand_phi);
        const double rvx = sr1 * cr2;
        const double rvy = sr1 * sr2;
        const double rvz = cr1;
        ox = ny * rvz - nz * rvy;
        oy = nz * rvx - nx * rvz;
        oz = nx * rvy - ny * rvx;
        dp += 2;
        att++;
      } while ((sum = ox * ox + oy * oy + oz * oz) < 1.0e-14);
      sum = sqrt(sum);
      sh.slot[i] = ndiv;
      t.div_dir[3 * ndiv + 0] = ox / sum;
      t.div_dir[3 * ndiv + 1] = oy / sum;
      t.div_dir[3 * ndiv + 2] = oz / sum;
    }
    att = __shfl(att, f0 & 63, 64);
    ndiv++;
    cur += 1 + 2 * att;
    i++;
  }
  if (lane == 0) { sh.cursor = cur; sh.ndiv = ndiv; }
}

// a ready cell, its dermis and the two sides of its division test
__device__ __forceinline__ void renew_ready(const Tis& t, RenewSh& sh, const RenewK& rk, int k, int c) {
  sh.ready[k] = c;
  sh.der[k] = t.dermis[c];
  sh.thr[k] = t.div_age_thresh[c] * rk.stoch_div_time_ratio;
  sh.rhs[k] = stoch_corr_coef * rk.DT_Cell * weighted_eps_kb(rk, t.is_malignant[c]) * rk.S2;
}

// the rule of the k-th ready cell, decided
__device__ __forceinline__ void renew_ready_rule(const Tis& t, const RenewSh& sh, const RenewK& rk, int pb, int cpar, int k,
                                                 int n_old, long long next_uid) {
  const int c = sh.ready[k];
  if (sh.slot[k] >= 0) divide(t, pb, cpar, c, sh.slot[k], n_old, next_uid);
  else t.ageb[c] = t.ageb[c] + rk.DT_Cell * ageb_const(rk, t.ca2p_avg[c], t.is_malignant[c]);
}

// exclusive offsets of the block's values a and b, and their sums
__device__ __forceinline__ void renew_offsets(RenewSh& sh, int a, int b, int* off_a, int* off_b, int* sum_a, int* sum_b) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int ta, tb;
  int oa = group_exclusive_scan<64>(a, lane, &ta), ob = group_exclusive_scan<64>(b, lane, &tb);
  if (lane == 0) { sh.wcnt[wv] = ta; sh.wrm[wv] = tb; }
  __syncthreads();
  int sa = 0, sb = 0;
#pragma unroll
  for (int w = 0; w < 16; w++) {
    if (w < wv) { oa += sh.wcnt[w]; ob += sh.wrm[w]; }
    sa += sh.wcnt[w]; sb += sh.wrm[w];
  }
  *off_a = oa; *off_b = ob; *sum_a = sa; *sum_b = sb;
}

// the last block whose offset is not past i (off ascends over m blocks)
__device__ __forceinline__ int renew_block_of(const int* off, int m, int i) {
  int lo = 0;
  for (int step = RCHUNK / 2; step > 0; step >>= 1)
    if (lo + step < m && off[lo + step] <= i) lo += step;
  return lo;
}

// CellManager::remove_exec (cellmanager.cpp:338-352): queued slot q_i takes
// the cell at the current tail N-1-i.  A queued slot at or past the current
// end means a queued cell had already been moved (the reference deletes a
// live cell there): ERR_REMOVE_ALIAS.  A removed DEAD cell's cell_stat goes
// to cst_store with k_disap = the current timestep (:343-346), in queue
// order; the timestep then advances (one renewal per step).
__device__ __forceinline__ void remove_cells(const Tis& t, int pb, int zero_zz, int N, int ndiv, int nrm) {
  Status* st = t.st;
  if (threadIdx.x < 64) {   // the first wave, 64 of the queue at a time
    const long long ts = st->timestep;
    int ns = st->nstat;
    for (int i0 = 0; i0 < nrm; i0 += 64) {
      const int i = i0 + threadIdx.x;
      const int q = t.rm_list[min(i, nrm - 1)];
      const long long c0 = t.cst[3 * q], c1 = t.cst[3 * q + 1];
      const bool keep = i < nrm && q < N - i && t.state[q] == DEAD;
      const unsigned long long mk = __ballot(keep);
      const int at = ns + __popcll(mk & ((1ull << threadIdx.x) - 1));
      if (keep && at < t.cap) {
        long long* o = t.cst_store + 3 * (size_t)at;
        o[0] = c0; o[1] = c1; o[2] = ts;
      }
      ns += __popcll(mk);
    }
    if (threadIdx.x == 0) {
      if (ns > t.cap) renew_err(st, ERR_CAPACITY);
      st->nstat = min(ns, t.cap);
      st->timestep = ts + 1;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nrm; i += blockDim.x) {
    const int q = t.rm_list[i];
    if (q >= N - i) { renew_err(st, ERR_REMOVE_ALIAS); continue; }
    if (t.pair[q] >= 0) renew_err(st, ERR_PAIR_REMOVED);
    const int s = N - 1 - i;
    if (s == q) continue;
    t.state[q] = t.state[s]; t.is_malignant[q] = t.is_malignant[s]; t.touch_air[q] = t.touch_air[s];
    t.fix_origin[q] = t.fix_origin[s]; t.rest_div_times[q] = t.rest_div_times[s];
    t.pair[q] = t.pair[s]; t.dermis[q] = t.dermis[s];
    for (int a = 0; a < 3; a++) {
      t.lat[3 * q + a] = t.lat[3 * s + a];
      t.pos[pb][a][q] = t.pos[pb][a][s];
      t.cst[3 * q + a] = t.cst[3 * s + a];
    }
    t.radius[q] = t.radius[s]; t.div_age_thresh[q] = t.div_age_thresh[s];
    t.ca2p[0][q] = t.ca2p[0][s]; t.ca2p[1][q] = t.ca2p[1][s];
    t.ip3[0][q] = t.ip3[0][s]; t.ip3[1][q] = t.ip3[1][s];
    t.ca2p_avg[q] = t.ca2p_avg[s]; t.ex_inert[q] = t.ex_inert[s]; t.agek[q] = t.agek[s];
    t.ageb[q] = t.ageb[s]; t.ex_fat[q] = t.ex_fat[s]; t.in_fat[q] = t.in_fat[s];
    t.spr_nat_len[q] = t.spr_nat_len[s]; t.diff_u[q] = t.diff_u[s];
    t.uid[q] = t.uid[s]; t.src_row[q] = t.src_row[s];
  }
  __syncthreads();
  // pair pointers follow the moved cells (Cell* identity in the reference)
  for (int i = threadIdx.x; i < nrm; i += blockDim.x) {
    const int q = t.rm_list[i];
    const int s = N - 1 - i;
    if (q >= N - i || s == q) continue;
    const int p = t.pair[q];
    if (p < 0) continue;
    int np = p;
    if (p >= N - nrm) {
      const int j = N - 1 - p;
      np = t.rm_list[j];
      if (np == p || np >= N - j) { renew_err(st, ERR_PAIR_REMOVED); continue; }
    } else {
      t.pair[p] = q;
    }
    t.pair[q] = np;
  }
  if (threadIdx.x == 0) {
    st->n = N - nrm;
    st->next_uid += ndiv;
    if (zero_zz) st->zzmax_bits = 0ull;
  }
}

// pair_disperse (:364-385), from the higher-index partner (:422-428), by one
// workgroup of RCHUNK lanes; few cells have a partner, so the pair words of
// four cells per lane are read at a time
__device__ __forceinline__ void disperse_pair(const Tis& t, int pb, int c, int p) {
  const double eps_L = t.prm.eps_L, unpair_dist_coef = t.prm.unpair_dist_coef;
  const double rad_sum = t.radius[c] + t.radius[p];
  const double unpair_th = unpair_dist_coef * rad_sum;
  const double snl = t.spr_nat_len[c];
  if (snl < 2.0 * t.radius[c]) {
    const double v = snl + t.prm.DT_Cell * eps_L;
    t.spr_nat_len[c] = v;
    t.spr_nat_len[p] = v;
  } else if (dist_sq(t, ld_pos(t, pb, c), ld_pos(t, pb, p)) > unpair_th * unpair_th) {
    t.spr_nat_len[c] = 0;
    t.spr_nat_len[p] = 0;
    t.pair[p] = -1;
    t.pair[c] = -1;
  }
}
__device__ __forceinline__ void disperse_pairs(const Tis& t, int pb, int n) {
  constexpr int U = 4;
  for (int c0 = t.nmemb + t.nder + threadIdx.x; c0 < n; c0 += U * RCHUNK) {
    int p[U];
#pragma unroll
    for (int u = 0; u < U; u++) p[u] = t.pair[min(c0 + u * RCHUNK, n - 1)];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int c = c0 + u * RCHUNK;
      if (c < n && p[u] >= 0 && c > p[u]) disperse_pair(t, pb, c, p[u]);
    }
  }
}

// What follows a tissue's decisions: the counts, removals and pairs
__device__ __forceinline__ void renew_end(const Tis& t, const RenewSh& sh, int pb, int zero_zz, int n_old, int nrm) {
  Status* st = t.st;
  const int ndiv = sh.ndiv;
  if (threadIdx.x == 0) {
    st->rng_pos = sh.cursor;
    st->ndiv = ndiv;
    st->nrm = nrm;
    st->n_old = n_old;
  }
  if (threadIdx.x == 64 && st->force_err) set_err(st, st->force_err);
  remove_cells(t, pb, zero_zz, n_old + ndiv, ndiv, nrm);
  __syncthreads();
  disperse_pairs(t, pb, n_old + ndiv - nrm);
}

// What bounds it is the chain of round trips of its one workgroup: the
// blocks' counts, the packed cells, their words and the draws, each for up to
// RCHUNK blocks or ready cells at once, then the rounds of renew_decide, the
// removals and the pairs.  With k_renew_cells, 2,000 cells past the membrane:
// 4.3 + 9.8 us (five launches that waited for each other, the walk 1024 cells
// at a time: 20.8 and four gaps); 20,000 cells: 5.1 + 26.4 (43.2).
__global__ void __launch_bounds__(RCHUNK) k_renew_tail(const Tis* __restrict__ T, int pb, int cpar, int zero_zz) {
  const Tis& t = T[blockIdx.y];
  Status* st = t.st;
  __shared__ RenewSh sh;
  const int tid = threadIdx.x;
  const int start = t.nmemb + t.nder;
  const int n_old = st->n;
  const long long next_uid = st->next_uid;
  const RenewK rk = renew_k(t.prm);
  if (tid == 0) { sh.cursor = st->rng_pos; sh.ndiv = 0; }
  const int nblk = n_old > start ? (n_old - start + RBLOCK - 1) / RBLOCK : 0;
  int nrm = 0;
  for (int b0 = 0; b0 < nblk; b0 += RCHUNK) {
    const int nb = min(nblk - b0, RCHUNK);
    const int cr = tid < nb ? t.rd_n[b0 + tid] : 0, cm = tid < nb ? t.rm_n[b0 + tid] : 0;
    int off_r, off_m, tot_r, tot_m;
    renew_offsets(sh, cr, cm, &off_r, &off_m, &tot_r, &tot_m);
    sh.off_r[tid] = off_r;
    sh.off_m[tid] = off_m;
    __syncthreads();
    for (int i = tid; i < tot_m; i += RCHUNK) {
      const int b = renew_block_of(sh.off_m, nb, i);
      t.rm_list[nrm + i] = t.rm_pack[(size_t)(b0 + b) * RBLOCK + i - sh.off_m[b]];
    }
    nrm += tot_m;
    for (int r0 = 0; r0 < tot_r; r0 += RCHUNK) {
      const int m = min(tot_r - r0, RCHUNK);
      renew_window(t, sh, sh.cursor);
      if (tid < m) {
        const int b = renew_block_of(sh.off_r, nb, r0 + tid);
        renew_ready(t, sh, rk, tid, t.rd_list[(size_t)(b0 + b) * RBLOCK + r0 + tid - sh.off_r[b]]);
      }
      __syncthreads();
      if (tid < 64) renew_decide(t, sh, pb, st, m);
      __syncthreads();
      if (tid < m) renew_ready_rule(t, sh, rk, pb, cpar, tid, n_old, next_uid);
      __syncthreads();   // the lists are the next cells' from here
    }
    __syncthreads();   // off_r, off_m and the counts are the next blocks' from here
  }
  __syncthreads();
  renew_end(t, sh, pb, zero_zz, n_old, nrm);
}

// The whole renewal of tissues with few cells, one workgroup per tissue.  A
// tissue of 420 cells: 9.6 us, against about 3.5 and 7 and the gap.  A tissue is
// sent here by the count of the last status read-back; renewals called one after
// the other without one may have outgrown a chunk.
__global__ void __launch_bounds__(RCHUNK) k_renew_one(const Tis* __restrict__ T, int pb, int cb, int cpar, int zero_zz) {
  const Tis& t = T[blockIdx.y];
  Status* st = t.st;
  __shared__ RenewSh sh;
  __shared__ int s_corn;
  const int tid = threadIdx.x;
  const int start = t.nmemb + t.nder;
  const int n_old = st->n;
  const long long next_uid = st->next_uid, ts = st->timestep, cur0 = st->rng_pos;
  const RenewK rk = renew_k(t.prm);
  if (tid == 0) { sh.cursor = cur0; sh.ndiv = 0; s_corn = 0; }
  renew_window(t, sh, cur0);
  int nrm = 0, ncorn = 0;
  for (int base = start; base < n_old; base += RCHUNK) {
    const int c = base + tid;
    const RCell r = load_rcell(t, cb, min(c, n_old - 1));
    const bool rd = c < n_old && needs_draw(rk, r), rm = c < n_old && to_remove(rk, r);
    int off_r, off_m, tot_r, tot_m;
    renew_offsets(sh, rd, rm, &off_r, &off_m, &tot_r, &tot_m);
    if (base > start && tot_r) renew_window(t, sh, sh.cursor);
    if (rd) renew_ready(t, sh, rk, off_r, c);
    if (rm) t.rm_list[nrm + off_m] = c;
    nrm += tot_m;
    __syncthreads();
    if (tot_r && tid < 64) renew_decide(t, sh, pb, st, tot_r);
    if (c < n_old && !rd) ncorn += renew_cell(t, rk, r, c, ts);
    __syncthreads();
    if (tid < tot_r) renew_ready_rule(t, sh, rk, pb, cpar, tid, n_old, next_uid);
    __syncthreads();   // the lists are the next cells' from here
  }
  if (ncorn) atomicAdd(&s_corn, ncorn);
  __syncthreads();
  if (tid == 0) st->sw += s_corn;
  renew_end(t, sh, pb, zero_zz, n_old, nrm);
}

// initialize_sc (:435-443)
__global__ void __launch_bounds__(256) k_initialize_sc(const Tis* __restrict__ T, const int* tlist, int pb) {
  const Tis& t = T[tlist ? tlist[blockIdx.y] : blockIdx.y];
  const int n = t.st->n;
  const double zzmax = __longlong_as_double((long long)t.st->zzmax_bits);
  for (int c = t.nmemb + t.nder + blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    const double THRESH_DEAD = t.prm.THRESH_DEAD;
    if (t.state[c] == ALIVE && zzmax - t.pos[pb][2][c] < 8 * t.prm.R_max) {
      t.agek[c] = t.agek[c] > THRESH_DEAD ? t.agek[c] : THRESH_DEAD;
      t.state[c] = AIR;
    }
  }
}

// cell_pos_periodic_fix (cellmanager.cpp:395-414)
__global__ void __launch_bounds__(256) k_periodic_fix(const Tis* __restrict__ T, int pb) {
  const Tis& t = T[blockIdx.y];
  const int n = t.st->n;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    const double x = t.pos[pb][0][c], y = t.pos[pb][1][c];
    if (x > t.LX) t.pos[pb][0][c] = x - t.LX;
    else if (x < 0) t.pos[pb][0][c] = x + t.LX;
    if (y > t.LY) t.pos[pb][1][c] = y - t.LY;
    else if (y < 0) t.pos[pb][1][c] = y + t.LY;
  }
}

void launch_renew(hipStream_t s, const Tis* dT, int ntis, int pb, int cb, int cpar, int max_free, int zero_zz) {
  if (max_free <= RENEW_ONE) {
    EPI_LAUNCH(K_RENEW_ONE, k_renew_one, dim3(1, ntis), dim3(RCHUNK), 0, s, dT, pb, cb, cpar, zero_zz);
    return;
  }
  EPI_LAUNCH(K_RENEW_CELLS, k_renew_cells, dim3((max_free + RBLOCK - 1) / RBLOCK, ntis), dim3(RBLOCK), 0, s, dT, cb);
  EPI_LAUNCH(K_RENEW_TAIL, k_renew_tail, dim3(1, ntis), dim3(RCHUNK), 0, s, dT, pb, cpar, zero_zz);
}

void launch_initialize_sc(hipStream_t s, const Tis* dT, const int* tlist, int ntis, int pb, int max_n) {
  dim3 g((max_n + 255) / 256, ntis);
  EPI_LAUNCH(K_INIT_SC, k_initialize_sc, g, dim3(256), 0, s, dT, tlist, pb);
}

void launch_periodic_fix(hipStream_t s, const Tis* dT, int ntis, int pb, int max_n) {
  dim3 g((max_n + 255) / 256, ntis);
  EPI_LAUNCH(K_PERIODIC_FIX, k_periodic_fix, g, dim3(256), 0, s, dT, pb);
}

}  // namespace epi
