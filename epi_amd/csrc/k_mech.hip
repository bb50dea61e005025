// k_mech.hip -- cell_interaction (cell_interaction.cpp:648-685) on CDNA4.
//
// The reference scatters every pair force into both cells with CAS atomics
// (cell_interaction.cpp:48-66, atomics.h:42-47), so its result depends on the
// order of the additions.  Here every cell gathers its own contributions and
// adds them in the order of the serial loop: bending, wall, its own handler
// over its list, lower-index handlers before and higher-index handlers after
// (cell_interaction.cpp:650-679).  In k_forces a group of FG = 16 lanes owns
// one cell: the lanes compute the cell's terms (neighbour deltas and the 12
// bend dihedrals) into LDS and the group's leader adds them in that order;
// k_forces_long, for rows longer than the LDS slots, gives one lane one
// cell.  No atomics: the FP64 result is the serial one bit for bit.
#include "epi_dev.h"
#include "launch.h"
#include "epi_group.h"
#include "mech_dev.h"

namespace epi {

struct CV {           // what a force law reads of a cell
  P3 p;
  double r, agek, snl;
  int pair, dermis, rdt;
  uint8_t s;
};

__device__ __forceinline__ CV load_cv(const Tis& t, int pb, int c) {
  CV v;
  v.p = ld_pos(t, pb, c);
  v.r = t.radius[c];
  v.agek = t.agek[c];
  v.snl = t.spr_nat_len[c];
  v.pair = t.pair[c];
  v.dermis = t.dermis[c];
  v.rdt = t.rest_div_times[c];
  v.s = t.state[c];
  return v;
}

// The law cell c's handler applies to its list entry q, or LAW_NONE.
// _DER_ :549-561, _FIX_ :581-604, _MUSUME_ :613-634, _AL_AIR_DE_ :563-579.
__device__ __forceinline__ int proc_law(const CV& c, int ci, const CV& q, int qi) {
  switch (c.s) {
    case DER:
      return (q.s == DER && ci > qi) ? LAW_DER_DER : LAW_OTHER;
    case FIX:
      if (q.s == FIX) return (c.pair != qi && ci > qi) ? LAW_FIXMU : LAW_NONE;
      if (q.s == MUSUME) return (c.pair != qi) ? LAW_FIXMU : LAW_NONE;
      if (q.s == MEMB) return (c.dermis == qi) ? LAW_FIX_MEMB : LAW_OTHER;
      return LAW_NONE;
    case MUSUME:
      if (q.s == MEMB) return (c.dermis == qi) ? LAW_MU_MEMB : LAW_OTHER;
      if (q.s == MUSUME && c.pair != qi && ci > qi) return LAW_FIXMU;
      return LAW_NONE;
    case ALIVE: case AIR: case DEAD:
      if (q.s == ALIVE || q.s == AIR || q.s == DEAD) return ci > qi ? LAW_ALAIRDE : LAW_NONE;
      if (q.s == DER) return LAW_NONE;
      return LAW_ALAIRDE;
    default:
      return LAW_NONE;
  }
}

// Coefficient of law `law` with c1 = a, c2 = b (cell_interaction.cpp:77-285).
//
// Most laws are one of three forms, and neighbouring lanes meet all of them:
//   L  4 eps Q (Q - 1) / s     ljmain, and MEMB-MEMB below cr_dist
//   A  -(K / d) x (1 - x^2 / c) adhesion, x = Q - 1 (0 past LJ_THRESH)
//   S  -(K / d) (Q - 1)         the FIX-MEMB anchor, and MEMB-MEMB up to contact
// with s = d^2.  Q and the second quotient are each a numerator over a
// denominator chosen per lane, so a wave pays for one square root and three
// FP64 divisions whatever its lanes hold, not for every law's own; the
// operands and their order are each law's.  The rare forms (DER-DER,
// stretched MEMB-MEMB, the pair spring) follow in branches of their own.
// PAIR false leaves out the pair spring, which no list entry takes.
template <bool PAIR>
__device__ __forceinline__ double coef_law(const Tis& t, int law, const CV& a, const CV& b, Status* st) {
  const double distSq = dist_sq(t, a.p, b.p);
  const double rad_sum = a.r + b.r;
  const double dist = sqrt(distSq);
  if (PAIR && law == LAW_PAIR) {
    const double force = t.prm.Kspring_division * (dist - a.snl);
    return -force / dist;
  }
  if (law == LAW_DER_DER) {
    if (dist + t.prm.delta_R < rad_sum) {
      const double dist2 = dist + t.prm.delta_R;
      const double LJ6 = POW6(rad_sum) / POW6(dist2);
      return 4.0 * t.m_eps * LJ6 * (LJ6 - 1) / (dist * dist2) + t.prm.para_ljp2;
    }
    if (distSq < rad_sum * rad_sum) return t.prm.para_ljp2;
    const double dist2 = dist + t.prm.delta_R;
    const double LJ6 = POW6(rad_sum) / POW6(dist2);
    return 4.0 * t.m_eps * LJ6 * (LJ6 - 1) / (dist * dist) + t.prm.para_ljp2;
  }
  const bool memb = law == LAW_MEMB_MEMB;
  const double rad_sum_sq = rad_sum * rad_sum;
  const double cr_dist = rad_sum * t.prm.P_MEMB;
  const double cr_dist_sq = rad_sum_sq * t.prm.P_MEMB * t.prm.P_MEMB;
  if (memb && !(distSq < cr_dist_sq) && !(distSq < rad_sum_sq)) {   // stretched MEMB-MEMB
    const double lambda_dist = (1.0 + t.prm.P_MEMB) * rad_sum;
    const double LJ6 = POW6(cr_dist) / POW6(lambda_dist - dist);
    const double tmp = -(t.prm.DER_DER_CONST / rad_sum) * ((1.0 - t.prm.P_MEMB) / t.prm.P_MEMB)
                       - 4 * t.m_eps * (LJ6 * (LJ6 - 1.0)) / ((lambda_dist - dist) * dist);
    if (fabs(tmp) > 100) set_force_err(st, ERR_STRONG_INTERACTION);
    return tmp;
  }
  // is_near: every law but LAW_OTHER takes ljmain within contact
  const bool L = law == LAW_OTHER || (memb ? distSq < cr_dist_sq : distSq < rad_sum * rad_sum);
  double K = t.m_kadh * t.prm.K_DESMOSOME_RATIO;   // LAW_FIXMU, LAW_ALAIRDE
  if (law == LAW_ALAIRDE) {
    if (a.agek > t.prm.THRESH_SP && b.agek > t.prm.THRESH_SP) K = t.m_kadh;
  } else if (law == LAW_MU_MEMB) {
    // spring_force_to_memb, set at the top of _MUSUME_interaction (:613-620)
    K = 0;
    if (!L) {
      if (a.pair >= 0 && t.state[a.pair] == FIX) K = t.m_kspring;
      else if (a.rdt > 0) K = t.prm.Kspring_d;
    }
  } else if (law == LAW_FIX_MEMB) {
    K = t.m_kspring;
  } else if (memb) {
    K = t.prm.DER_DER_CONST;
  }
  const double n1 = L ? (memb ? POW3(cr_dist_sq) : POW6(rad_sum)) : dist;
  const double d1 = L ? POW3(distSq) : (memb ? cr_dist : rad_sum);
  const double Q = n1 / d1;
  const double x = Q - 1.0;
  const double k2 = (L ? 4.0 * t.m_eps * Q * x : K) / (L ? distSq : dist);
  if (L) {
    if (memb && fabs(k2) > 100) set_force_err(st, ERR_STRONG_INTERACTION);
    return k2;
  }
  if (law == LAW_FIX_MEMB) return -k2 * x;
  if (memb) {
    const double tmp = -k2 * x;
    if (fabs(tmp) > 100) set_force_err(st, ERR_STRONG_INTERACTION);
    return tmp;
  }
  const double c2 = (t.prm.LJ_THRESH - 1.0) * (t.prm.LJ_THRESH - 1.0);
  return x + 1 > t.prm.LJ_THRESH ? 0.0 : -k2 * x * (1 - x * x / c2);
}

// cell_interaction_apply (:48-66): the displacement added to c1, subtracted from c2
template <bool PAIR>
__device__ __forceinline__ P3 delta_law(const Tis& t, int law, const CV& a, const CV& b, Status* st) {
  const double coef = coef_law<PAIR>(t, law, a, b, st);
  if (fabs(coef) > 1000) set_force_err(st, ERR_STRONG_INTERACTION);
  const double d = t.prm.DT_Cell * coef;
  return P3{d * p_diff_x(t, a.p.x, b.p.x), d * p_diff_y(t, a.p.y, b.p.y), d * (a.p.z - b.p.z)};
}
__device__ P3 delta(const Tis& t, int law, const CV& a, const CV& b, Status* st) { return delta_law<true>(t, law, a, b, st); }

// wall_interaction (:287-294): the z increment
__device__ __forceinline__ double wall_dz(const Tis& t, const CV& c) {
  const double distlj = 2.0 * c.p.z;
  const double LJ6 = POW6(c.r) / POW6(c.p.z);
  const double ljm = 4.0 * t.m_eps * LJ6 * (LJ6 - 1.0) / (distlj * distlj);
  return t.prm.DT_Cell * ljm * 2.0 * c.p.z;
}

// ---- triangular bending (:451-499) ---------------------------------------
__device__ __forceinline__ P3 v_cross(P3 a, P3 b) {
  return P3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ double v_dot(P3 a, P3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ double v_norm(P3 a) { return sqrt(a.x * a.x + a.y * a.y + a.z * a.z); }
__device__ __forceinline__ P3 v_normalize(P3& a) {   // vec3::normalize mutates
  double nm = v_norm(a);
  a.x /= nm; a.y /= nm; a.z /= nm;
  return a;
}
__device__ __forceinline__ P3 v_scale(double c, P3 v) { return P3{c * v.x, c * v.y, c * v.z}; }
__device__ __forceinline__ P3 v_div(P3 v, double c) { return P3{v.x / c, v.y / c, v.z / c}; }
__device__ __forceinline__ P3 v_sub(P3 a, P3 b) { return P3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ P3 v_add(P3 a, P3 b) { return P3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ P3 vpsub(const Tis& t, P3 a, P3 b) {
  return P3{p_diff_x(t, a.x, b.x), p_diff_y(t, a.y, b.y), a.z - b.z};
}
__device__ __forceinline__ double bend_factor(double cdot) {   // :349-360
  if (cdot >= 0) return (1.0 - cdot);
  return 1.0 / ((1.0 + cdot) * (1.0 + cdot));
}
__device__ __forceinline__ P3 tri_rho(P3 n1, P3 b1) { return v_sub(b1, v_scale(v_dot(n1, b1), n1)); }

// Term i of a membrane particle's 12 dihedral terms: tri_bend_1 (:468-474) of
// (a, b, c) for i < 6, tri_bend_2 (:476-486) for the others.  With
//   n1 = |A1 x A2|, n2 = |B1 x B2|, both unit,
//   1: A1 = r - b, A2 = a - b, B1 = a - b, B2 = c - b, f(n1.n2) (a - b) x rho(n1, n2) / |n1|
//   2: A1 = r - c, A2 = b - c, B1 = r - b, B2 = a - b,
//      f(n1.n2) ((b - c) x rho(n1, n2) / |n1| + (a - b) x rho(n2, n1) / |n2|)
// the two differ in the vectors they take and in the second summand, so the
// lanes of a particle run one code path for both.
__device__ __forceinline__ P3 p3_sel(bool c, P3 a, P3 b) { return P3{c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z}; }
__device__ __forceinline__ P3 tri_bend(const Tis& t, bool second, P3 r1v, P3 a1v, P3 b1v, P3 c1v) {
  const P3 ab = vpsub(t, a1v, b1v), rb = vpsub(t, r1v, b1v);
  const P3 rc = vpsub(t, r1v, c1v);
  // c - b of form 1, b - c of form 2 (vpsub is not antisymmetric at half a box)
  const P3 bc = vpsub(t, p3_sel(second, b1v, c1v), p3_sel(second, c1v, b1v));
  P3 norm1_pre = v_cross(p3_sel(second, rc, rb), p3_sel(second, bc, ab));
  P3 norm2_pre = v_cross(p3_sel(second, rb, ab), p3_sel(second, ab, bc));
  const P3 norm1 = v_normalize(norm1_pre), norm2 = v_normalize(norm2_pre);
  const double dot1 = v_dot(norm1, norm2);
  P3 s = v_div(v_cross(p3_sel(second, bc, ab), tri_rho(norm1, norm2)), v_norm(norm1_pre));
  if (second) s = v_add(s, v_div(v_cross(ab, tri_rho(norm2, norm1)), v_norm(norm2_pre)));
  return v_scale(bend_factor(dot1), s);
}
__device__ P3 tri_bend_1(const Tis& t, P3 r1v, P3 a1v, P3 b1v, P3 c1v) { return tri_bend(t, false, r1v, a1v, b1v, c1v); }
__device__ P3 tri_bend_2(const Tis& t, P3 r1v, P3 a1v, P3 b1v, P3 c1v) { return tri_bend(t, true, r1v, a1v, b1v, c1v); }

// ---- serial form: one lane does a whole cell --------------------------------
// Used for rows longer than the LDS slots of the cooperative kernel.
__device__ void forces_serial(const Tis& t, int pb, int cb, int X, Status* st) {
  const CV cx = load_cv(t, pb, X);
  P3 acc = cx.p;
  const int* row = t.col[cb] + (size_t)X * t.ns;
  const int len = t.nlen[cb][X];
  if (X < t.nmemb) {
    const int* md = t.memb6 + 6 * X;
    P3 dr = P3{0, 0, 0};
    for (int i = 0; i < 6; i++) {
      const int i1 = (i + 1) % 6;
      dr = v_add(dr, tri_bend_1(t, cx.p, ld_pos(t, pb, md[i]), ld_pos(t, pb, md[i1]),
                                ld_pos(t, pb, t.memb6[6 * md[i1] + i])));
    }
    for (int i = 0; i < 6; i++)
      dr = v_add(dr, tri_bend_2(t, cx.p, ld_pos(t, pb, md[i]), ld_pos(t, pb, md[(i + 1) % 6]),
                                ld_pos(t, pb, md[(i + 2) % 6])));
    acc.x += t.prm.DT_Cell * t.m_kbend * dr.x;
    acc.y += t.prm.DT_Cell * t.m_kbend * dr.y;
    acc.z += t.prm.DT_Cell * t.m_kbend * dr.z;
    if (cx.p.z < cx.r) acc.z += wall_dz(t, cx);
    int hi[6], nhi = 0;
    for (int i = 0; i < 6; i++) {
      const int q = md[i];
      if (t.state[q] != MEMB) continue;
      if (X > q) {
        const P3 d = delta(t, LAW_MEMB_MEMB, cx, load_cv(t, pb, q), st);
        acc.x += d.x; acc.y += d.y; acc.z += d.z;
      } else if (q > X) {
        int k = nhi++;
        while (k > 0 && hi[k - 1] > q) { hi[k] = hi[k - 1]; k--; }
        hi[k] = q;
      }
    }
    for (int i = 0; i < nhi; i++) {
      const P3 d = delta(t, LAW_MEMB_MEMB, load_cv(t, pb, hi[i]), cx, st);
      acc.x -= d.x; acc.y -= d.y; acc.z -= d.z;
    }
    for (int i = MEMB_ADJ; i < len; i++) {
      const int p = row[i];
      const CV cp = load_cv(t, pb, p);
      const int law = proc_law(cp, p, cx, X);
      if (law != LAW_NONE) {
        const P3 d = delta(t, law, cp, cx, st);
        acc.x -= d.x; acc.y -= d.y; acc.z -= d.z;
      }
    }
  } else {
    const int nlo = t.nlo[X];
    // lower-index handlers in ascending order (selection over the lower part)
    int last = -1;
    for (int r = 0; r < nlo; r++) {
      int best = 0x7fffffff;
      for (int i = 0; i < nlo; i++) { const int v = row[i]; if (v > last && v < best) best = v; }
      last = best;
      if (t.state[best] == MEMB) continue;
      const CV cp = load_cv(t, pb, best);
      const int law = proc_law(cp, best, cx, X);
      if (law != LAW_NONE) {
        const P3 d = delta(t, law, cp, cx, st);
        acc.x -= d.x; acc.y -= d.y; acc.z -= d.z;
      }
    }
    if (cx.s == DER && cx.p.z < cx.r) acc.z += wall_dz(t, cx);
    for (int i = 0; i < len; i++) {
      const int q = row[i];
      const CV cq = load_cv(t, pb, q);
      const int law = proc_law(cx, X, cq, q);
      if (law != LAW_NONE) {
        const P3 d = delta(t, law, cx, cq, st);
        acc.x += d.x; acc.y += d.y; acc.z += d.z;
      }
    }
    if (cx.pair >= 0 && X > cx.pair) {
      const P3 d = delta(t, LAW_PAIR, cx, load_cv(t, pb, cx.pair), st);
      acc.x += d.x; acc.y += d.y; acc.z += d.z;
    }
    int P = cx.pair > X ? cx.pair : -1;
    for (int i = nlo; i < len; i++) {
      const int p = row[i];
      if (P >= 0 && P < p) {
        const P3 d = delta(t, LAW_PAIR, load_cv(t, pb, P), cx, st);
        acc.x -= d.x; acc.y -= d.y; acc.z -= d.z;
        P = -1;
      }
      const CV cp = load_cv(t, pb, p);
      const int law = proc_law(cp, p, cx, X);
      if (law != LAW_NONE) {
        const P3 d = delta(t, law, cp, cx, st);
        acc.x -= d.x; acc.y -= d.y; acc.z -= d.z;
      }
      if (p == P) {
        const P3 d = delta(t, LAW_PAIR, cp, cx, st);
        acc.x -= d.x; acc.y -= d.y; acc.z -= d.z;
        P = -1;
      }
    }
    if (P >= 0) {
      const P3 d = delta(t, LAW_PAIR, load_cv(t, pb, P), cx, st);
      acc.x -= d.x; acc.y -= d.y; acc.z -= d.z;
    }
  }
  t.pos[1 - pb][0][X] = acc.x;
  t.pos[1 - pb][1][X] = acc.y;
  t.pos[1 - pb][2][X] = acc.z;
}

// ---- cooperative form --------------------------------------------------------
// A group of FG lanes owns one cell.  Every list entry e is handled by lane
// e % FG, which evaluates the displacement the pair contributes to the cell:
// "own" (the cell's handler processes the entry, added) or "oth" (the entry's
// handler processes the cell, subtracted).  Only a DER-DER pair has both; it
// takes a second turn of the same code, so the laws are compiled once.  The
// group's first three lanes then add them, one coordinate each, in the serial
// order of cell_interaction (:650-679): bending, wall, lower-index handlers
// ascending, the cell's own list, its pair, higher-index handlers ascending
// with a higher-index partner's spring after that partner's list.  Lane 0..11
// evaluate the 12 dihedral terms of a membrane particle.
//
// An absent "own" term is stored as -0.0 and an absent "oth" term as +0.0:
// x + (-0.0) and x - (+0.0) are x for every x, so the sums take every slot
// without flags or branches, four slots' LDS reads ahead of their adds, in
// the same order and with the same results.
//
// Each group takes one cell, so the grid must cover all cells (a launch that
// does not is reported as ERR_INVALID); a loop over cells would keep the
// math's loop-invariant constants in registers and cost occupancy.
//
// What bounds it: FP64 issue of the laws (divergent lanes run one after the
// other) and, on a small tissue, the chain of round trips and the ordered
// sum.  One copy of the laws with shared divisions, one path for both
// dihedral forms and one coordinate per summing lane, against every law and
// form on its own and a leader summing all three: 100 steps of one tissue of
// 3,900 cells 1490 -> 1073 us, of 24 tissues (with their reverse pass) 30.3 ->
// 26.9 ms.
//
// FCAP, the LDS slots per cell, is chosen per launch from the longest list
// built so far: 40 keeps a 128-lane block's LDS small enough for 4 waves per
// SIMD, 48 and 64 take longer lists at lower occupancy, and rows beyond 64 go
// to k_forces_long.
constexpr int FG = 16;
constexpr int F_BLOCK = 128;
constexpr int F_GROUPS = F_BLOCK / FG;

// a group's LDS slots, padded by 8 bytes so that the summing lanes of a
// wave's groups read different banks
template <int FCAP>
struct FRow {
  P3 v[FCAP];
  double pad;
};

// acc +- the coordinate at v[3 e] for e in [e0, e1), in order
template <bool ADD>
__device__ __forceinline__ double sum_slots(double acc, const double* v, int e0, int e1) {
  int e = e0;
#pragma unroll 1
  for (; e + 4 <= e1; e += 4) {
    double d[4];
#pragma unroll
    for (int j = 0; j < 4; j++) d[j] = v[3 * (e + j)];
#pragma unroll
    for (int j = 0; j < 4; j++) acc = ADD ? acc + d[j] : acc - d[j];
  }
  for (; e < e1; e++) acc = ADD ? acc + v[3 * e] : acc - v[3 * e];
  return acc;
}
__device__ __forceinline__ double p3_at(const P3& p, int k) { return k == 0 ? p.x : k == 1 ? p.y : p.z; }

// the tissue's status into pinned host memory, then the number the host waits
// for.  The kernel follows the build in the stream, so the status is final but
// for what runs beside it (the force kernel's own errors have their own word).
__device__ __forceinline__ void status_out(const Tis& t, const StatusOut& out) {
  static_assert(sizeof(Status) % 8 == 0 && sizeof(Status) / 8 <= 64, "status copied in 8-byte words by one wave");
  if (threadIdx.x >= 64) return;
  if (threadIdx.x < sizeof(Status) / 8)
    reinterpret_cast<unsigned long long*>(out.host + blockIdx.y)[threadIdx.x] =
        reinterpret_cast<const unsigned long long*>(static_cast<const Status*>(t.st))[threadIdx.x];
  __threadfence_system();
  if (threadIdx.x == 0)
    __hip_atomic_store(out.seq + blockIdx.y, out.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int FCAP>
__global__ void __launch_bounds__(F_BLOCK) k_forces(const Tis* __restrict__ T, int pb, int cb, StatusOut out) {
  const Tis& t = T[blockIdx.y];
  Status* st = t.st;
  if (out.host && blockIdx.x == 0) status_out(t, out);
  __shared__ FRow<FCAP> s_own[F_GROUPS];
  __shared__ FRow<FCAP> s_oth[F_GROUPS];
  __shared__ __align__(16) int s_idx[F_GROUPS][FCAP];
  __shared__ uint8_t s_perm[F_GROUPS][FCAP];
  __shared__ P3 s_bend[F_GROUPS][12];
  const int lane = threadIdx.x & (FG - 1);
  const int grp = threadIdx.x / FG;
  const int X = blockIdx.x * F_GROUPS + grp;
  if (X >= t.cap) return;
  // the cell's own words (and its lane's list words) are loaded before the
  // cell count arrives, in one round trip with it: a cell past the count
  // reads allocated, stale slots and leaves once the count is in
  const int len = t.nlen[cb][X];
  const CV cx = load_cv(t, pb, X);
  const bool memb = X < t.nmemb;
  const int nA = memb ? 0 : t.nlo[X];
  const int* row = t.col[cb] + (size_t)X * t.ns;
  const int q0 = row[lane];   // a row holds ns >= 64 > FG slots
  const int n = st->n;
  if (blockIdx.x == 0 && threadIdx.x == 0 && (long long)gridDim.x * F_GROUPS < n) set_force_err(st, ERR_INVALID);
  if (X >= n) return;
  if (len > FCAP) return;   // k_forces_long
  bool hi = false;          // this lane's membrane slot is subtracted (its handler has the higher index)
#pragma unroll 1
  for (int e = lane; e < len; e += FG) {
    const int q = e == lane ? q0 : row[e];
    const CV cq = load_cv(t, pb, q);
    int law = LAW_NONE, law2 = LAW_NONE;
    bool own = false;
    if (memb) {
      if (e >= MEMB_ADJ) {
        law = proc_law(cq, q, cx, X);
      } else if (cq.s == MEMB && X != q) {
        law = LAW_MEMB_MEMB;
        own = X > q;
        hi = !own;
      }
    } else {
      law = proc_law(cx, X, cq, q);
      if (e >= nA || cq.s != MEMB) law2 = proc_law(cq, q, cx, X);
      own = law != LAW_NONE;
      if (!own) {
        law = law2;
        law2 = LAW_NONE;
      }
    }
    s_idx[grp][e] = q;
    s_own[grp].v[e] = P3{-0.0, -0.0, -0.0};
    s_oth[grp].v[e] = P3{0, 0, 0};
#pragma unroll 1
    while (law != LAW_NONE) {
      CV a, b;
      a.p = p3_sel(own, cx.p, cq.p); b.p = p3_sel(own, cq.p, cx.p);
      a.r = cx.r; b.r = cq.r;            // the sum of the two radii alone is read
      a.agek = cx.agek; b.agek = cq.agek;   // and whether both ages pass a threshold
      a.pair = own ? cx.pair : cq.pair;
      a.rdt = own ? cx.rdt : cq.rdt;
      const P3 d = delta_law<false>(t, law, a, b, st);
      if (own) s_own[grp].v[e] = d;
      else s_oth[grp].v[e] = d;
      law = law2;
      law2 = LAW_NONE;
      own = false;
    }
  }
  if (memb && lane < 12) {
    const int* md = t.memb6 + 6 * X;
    const int i = lane < 6 ? lane : lane - 6;
    const int ma = md[i], mb = md[(i + 1) % 6];
    const int mc = lane < 6 ? t.memb6[6 * mb + i] : md[(i + 2) % 6];
    s_bend[grp][lane] = tri_bend(t, lane >= 6, cx.p, ld_pos(t, pb, ma), ld_pos(t, pb, mb), ld_pos(t, pb, mc));
  }
  wave_sync();
  int nhi = 0;
  if (memb) {
    // the membrane slots that are subtracted, ascending by cell index
    const unsigned m = (unsigned)(__ballot(hi) >> (threadIdx.x & 48)) & 0x3fu;
    nhi = __popc(m);
    if (hi) {
      const int v = s_idx[grp][lane];
      int r = 0;
      for (int k = 0; k < MEMB_ADJ; k++) r += ((m >> k) & 1u) && s_idx[grp][k] < v;
      s_perm[grp][r] = (uint8_t)lane;
    }
  } else {
    // rank of each lower-part entry by cell index
    for (int e = lane; e < nA; e += FG) {
      const int v = s_idx[grp][e];
      int r = 0, k = 0;
      for (; k + 4 <= nA; k += 4) {
        const int4 w = *reinterpret_cast<const int4*>(&s_idx[grp][k]);
        r += (w.x < v) + (w.y < v) + (w.z < v) + (w.w < v);
      }
      for (; k < nA; k++) r += s_idx[grp][k] < v;
      s_perm[grp][r] = (uint8_t)e;
    }
  }
  wave_sync();
  if (lane >= 3) return;
  const double* own = reinterpret_cast<const double*>(s_own[grp].v) + lane;
  const double* oth = reinterpret_cast<const double*>(s_oth[grp].v) + lane;
  double acc = p3_at(cx.p, lane);
  if (memb) {
    const double* bend = reinterpret_cast<const double*>(s_bend[grp]) + lane;
    double dr = 0;
#pragma unroll
    for (int i = 0; i < 12; i++) dr = dr + bend[3 * i];
    acc += t.prm.DT_Cell * t.m_kbend * dr;
    if (lane == 2 && cx.p.z < cx.r) acc += wall_dz(t, cx);
#pragma unroll
    for (int e = 0; e < MEMB_ADJ; e++) acc += own[3 * e];
    for (int i = 0; i < nhi; i++) acc -= oth[3 * s_perm[grp][i]];
    acc = sum_slots<false>(acc, oth, MEMB_ADJ, len);
  } else {
    {
      int r = 0;
#pragma unroll 1
      for (; r + 4 <= nA; r += 4) {
        int k[4];
        double d[4];
#pragma unroll
        for (int j = 0; j < 4; j++) k[j] = s_perm[grp][r + j];
#pragma unroll
        for (int j = 0; j < 4; j++) d[j] = oth[3 * k[j]];
#pragma unroll
        for (int j = 0; j < 4; j++) acc -= d[j];
      }
      for (; r < nA; r++) acc -= oth[3 * s_perm[grp][r]];
    }
    if (lane == 2 && cx.s == DER && cx.p.z < cx.r) acc += wall_dz(t, cx);
    acc = sum_slots<true>(acc, own, 0, len);
    if (cx.pair < 0) {
      acc = sum_slots<false>(acc, oth, nA, len);
    } else {
      // the pair's spring: added after the own list when this cell has the
      // higher index, else subtracted after the partner's list
      const CV cp = load_cv(t, pb, cx.pair);
      const bool up = X > cx.pair;
      const double dp = p3_at(up ? delta(t, LAW_PAIR, cx, cp, st) : delta(t, LAW_PAIR, cp, cx, st), lane);
      if (up) {
        acc = sum_slots<false>(acc + dp, oth, nA, len);
      } else {
        int P = cx.pair;
        for (int e = nA; e < len; e++) {
          const int p = s_idx[grp][e];
          if (P >= 0 && P < p) {
            acc -= dp;
            P = -1;
          }
          acc -= oth[3 * e];
          if (p == P) {
            acc -= dp;
            P = -1;
          }
        }
        if (P >= 0) acc -= dp;
      }
    }
  }
  t.pos[1 - pb][lane][X] = acc;
}

// cells whose rows exceed the LDS slots (cap) of k_forces, one lane per cell
__global__ void __launch_bounds__(256) k_forces_long(const Tis* __restrict__ T, int pb, int cb, int cap) {
  const Tis& t = T[blockIdx.y];
  const int n = t.st->n;
  for (int X = blockIdx.x * blockDim.x + threadIdx.x; X < n; X += gridDim.x * blockDim.x)
    if (t.nlen[cb][X] > cap) forces_serial(t, pb, cb, X, t.st);
}

int launch_forces_rows(hipStream_t s, const Tis* dT, int ntis, int pb, int cb, int max_other, int max_len,
                       const StatusOut& out) {
  dim3 g((max_other + F_GROUPS - 1) / F_GROUPS, ntis);
  int cap;
  if (max_len <= 40) {
    cap = 40;
    EPI_LAUNCH(K_FORCES, k_forces<40>, g, dim3(F_BLOCK), 0, s, dT, pb, cb, out);
  } else if (max_len <= 48) {
    cap = 48;
    EPI_LAUNCH(K_FORCES, k_forces<48>, g, dim3(F_BLOCK), 0, s, dT, pb, cb, out);
  } else {
    cap = FORCES_ROW_CAP;
    EPI_LAUNCH(K_FORCES, k_forces<FORCES_ROW_CAP>, g, dim3(F_BLOCK), 0, s, dT, pb, cb, out);
  }
  return cap;
}

void launch_forces_long(hipStream_t s, const Tis* dT, int ntis, int pb, int cb, int max_other, int cap) {
  dim3 gl((max_other + 255) / 256, ntis);
  EPI_LAUNCH(K_FORCES_LONG, k_forces_long, gl, dim3(256), 0, s, dT, pb, cb, cap);
}

void launch_forces(hipStream_t s, const Tis* dT, int ntis, int pb, int cb, int max_memb, int max_other,
                   int max_len) {
  (void)max_memb;
  const int cap = launch_forces_rows(s, dT, ntis, pb, cb, max_other, max_len, StatusOut{});
  if (max_len > cap) launch_forces_long(s, dT, ntis, pb, cb, max_other, cap);
}

// ==== frozen mechanics window: the reverse pass ==============================
// The window is the plain k_forces step repeated with lists, states, pairs
// and dermis frozen.  Which interactions apply depends only on that frozen
// data, so the reverse pass enumerates them from each handler cell (its own
// list, its pair, the membrane slots), evaluates the derivative of the
// active branch of each law at the step's positions, and scatters
// lam_c1 - lam_c2 through the pair's Jacobian with FP64 atomics.

namespace {
struct LawD { double coef, ds, deps, dadh, dspr; };

__device__ LawD ljmain_d(double s, double R, double eps) {
  const double L = POW6(R) / POW3(s);
  return LawD{4.0 * eps * L * (L - 1) / s, 4.0 * eps * (4.0 * L - 7.0 * L * L) / (s * s), 4.0 * L * (L - 1) / s, 0, 0};
}
__device__ LawD adhesion_d(double s, double R, double K, double lj) {
  LawD r{0, 0, 0, 0, 0};
  const double d = sqrt(s);
  const double x = d / R - 1;
  if (x + 1 > lj) return r;
  const double c2 = (lj - 1.0) * (lj - 1.0);
  const double g = x * (1 - x * x / c2);
  r.coef = -(K / d) * g;
  const double dg = (1 - 3 * x * x / c2) / R;
  r.ds = (K * g / (d * d) - (K / d) * dg) / (2 * d);
  return r;
}

// coef of `law` (c1 = a, c2 = b) and its derivatives with respect to the
// squared distance and to eps_m, K_TOTAL, Kspring
__device__ LawD coef_law_d(const Tis& t, int law, const CV& a, const CV& b) {
  const double s = dist_sq(t, a.p, b.p);
  const double R = a.r + b.r;
  const double eps = t.m_eps;
  LawD r{0, 0, 0, 0, 0};
  switch (law) {
    case LAW_OTHER:
      return ljmain_d(s, R, eps);
    case LAW_DER_DER: {
      const double d = sqrt(s), D = d + t.prm.delta_R;
      const double L = POW6(R) / POW6(D);
      const double dL = -6.0 * L / D;
      double g, dgd;
      if (D < R) {
        g = L * (L - 1) / (d * D);
        dgd = (2 * L - 1) * dL / (d * D) - L * (L - 1) * (D + d) / ((d * D) * (d * D));
      } else if (s < R * R) {
        return r;
      } else {
        g = L * (L - 1) / (d * d);
        dgd = (2 * L - 1) * dL / (d * d) - 2 * L * (L - 1) / (d * d * d);
      }
      return LawD{4.0 * eps * g + t.prm.para_ljp2, 4.0 * eps * dgd / (2 * d), 4.0 * g, 0, 0};
    }
    case LAW_ALAIRDE:
      if (s < R * R) return ljmain_d(s, R, eps);
      {
        const bool strong = a.agek > t.prm.THRESH_SP && b.agek > t.prm.THRESH_SP;
        r = adhesion_d(s, R, strong ? t.m_kadh : t.m_kadh * t.prm.K_DESMOSOME_RATIO, t.prm.LJ_THRESH);
        r.dadh = r.coef / t.m_kadh;
        return r;
      }
    case LAW_FIXMU:
      if (s < R * R) return ljmain_d(s, R, eps);
      r = adhesion_d(s, R, t.m_kadh * t.prm.K_DESMOSOME_RATIO, t.prm.LJ_THRESH);
      r.dadh = r.coef / t.m_kadh;
      return r;
    case LAW_MU_MEMB: {
      if (s < R * R) return ljmain_d(s, R, eps);
      const bool fixpair = a.pair >= 0 && t.state[a.pair] == FIX;
      const double spring = fixpair ? t.m_kspring : (a.rdt > 0 ? t.prm.Kspring_d : 0.0);
      r = adhesion_d(s, R, spring, t.prm.LJ_THRESH);
      if (fixpair) r.dspr = r.coef / t.m_kspring;
      return r;
    }
    case LAW_FIX_MEMB:
      if (s < R * R) return ljmain_d(s, R, eps);
      {
        const double d = sqrt(s);
        return LawD{-(t.m_kspring / d) * (d / R - 1.0), -t.m_kspring / (2 * d * d * d), 0, 0,
                    -(1.0 / d) * (d / R - 1.0)};
      }
    case LAW_MEMB_MEMB: {
      const double cr = R * t.prm.P_MEMB, cr2 = cr * cr;
      if (s < cr2) {
        const double L = POW3(cr2) / POW3(s);
        return LawD{4.0 * eps * L * (L - 1) / s, 4.0 * eps * (4.0 * L - 7.0 * L * L) / (s * s),
                    4.0 * L * (L - 1) / s, 0, 0};
      } else if (s < R * R) {
        const double d = sqrt(s);
        return LawD{-(t.prm.DER_DER_CONST / d) * (d / cr - 1.0), -t.prm.DER_DER_CONST / (2 * d * d * d), 0, 0, 0};
      } else {
        const double d = sqrt(s);
        const double lam = (1.0 + t.prm.P_MEMB) * R;
        const double m = lam - d;
        const double L = POW6(cr) / POW6(m);
        const double dL = 6.0 * L / m;
        const double q = L * (L - 1.0) / (m * d);
        const double dq = (2 * L - 1) * dL / (m * d) + L * (L - 1.0) * (d - m) / ((m * d) * (m * d));
        return LawD{-(t.prm.DER_DER_CONST / R) * ((1.0 - t.prm.P_MEMB) / t.prm.P_MEMB) - 4 * eps * q, -4 * eps * dq / (2 * d), -4 * q,
                    0, 0};
      }
    }
    case LAW_PAIR: {
      const double d = sqrt(s);
      return LawD{-(t.prm.Kspring_division * (d - a.snl)) / d, -t.prm.Kspring_division * a.snl / (2 * d * d * d), 0, 0, 0};
    }
    default:
      return r;
  }
}

__device__ __forceinline__ void atomic_add3(double* lam, long long cap, int c, P3 g) {
  atomicAdd(&lam[c], g.x);
  atomicAdd(&lam[cap + c], g.y);
  atomicAdd(&lam[2 * cap + c], g.z);
}
__device__ __forceinline__ P3 ld3(const double* lam, long long cap, int c) {
  return P3{lam[c], lam[cap + c], lam[2 * cap + c]};
}

struct ParAcc { double eps, adh, spr; };

// scatters the pair's term to ib and returns the one for ia (the caller's
// cell, whose lanes reduce their terms before one atomic)
__device__ __forceinline__ P3 pair_bwd(const Tis& t, int law, const CV& a, int ia, const CV& b, int ib,
                                       const double* lam, double* nl, long long cap, ParAcc& pa) {
  const LawD ld = coef_law_d(t, law, a, b);
  const P3 r{p_diff_x(t, a.p.x, b.p.x), p_diff_y(t, a.p.y, b.p.y), a.p.z - b.p.z};
  const P3 la = ld3(lam, cap, ia), lb = ld3(lam, cap, ib);
  const P3 av{la.x - lb.x, la.y - lb.y, la.z - lb.z};
  const double ar = v_dot(av, r);
  const double k2 = 2 * ld.ds * ar;
  const P3 g{t.prm.DT_Cell * (ld.coef * av.x + k2 * r.x), t.prm.DT_Cell * (ld.coef * av.y + k2 * r.y),
             t.prm.DT_Cell * (ld.coef * av.z + k2 * r.z)};
  atomic_add3(nl, cap, ib, P3{-g.x, -g.y, -g.z});
  pa.eps += t.prm.DT_Cell * ld.deps * ar;
  pa.adh += t.prm.DT_Cell * ld.dadh * ar;
  pa.spr += t.prm.DT_Cell * ld.dspr * ar;
  return g;
}

// adjoint of n = N / |N|
__device__ __forceinline__ P3 unit_bar(P3 N, P3 nb) {
  const double nn = v_norm(N);
  const P3 n = v_div(N, nn);
  return v_div(v_sub(nb, v_scale(v_dot(nb, n), n)), nn);
}
__device__ __forceinline__ double bend_factor_d(double c) {
  if (c >= 0) return -1.0;
  return -2.0 / ((1.0 + c) * (1.0 + c) * (1.0 + c));
}
// y = scale f(d) (v x (n2 - d n1)), d = n1.n2
__device__ __forceinline__ void bend_pair_bar(P3 n1, P3 n2, P3 v, double scale, P3 ob, P3& vb, P3& n1b, P3& n2b,
                                              double& db) {
  const double d = v_dot(n1, n2);
  const P3 rho = v_sub(n2, v_scale(d, n1));
  const P3 oy = v_scale(scale * bend_factor(d), ob);
  db += scale * bend_factor_d(d) * v_dot(ob, v_cross(v, rho));
  vb = v_add(vb, v_cross(rho, oy));
  const P3 rb = v_cross(oy, v);
  n2b = v_add(n2b, rb);
  db += -v_dot(rb, n1);
  n1b = v_add(n1b, v_scale(-d, rb));
}
// reverse of tri_bend_1(r, a, b, c); bar[0..3] get the adjoints of r, a, b, c
__device__ void tri_bend_1_bar(const Tis& t, P3 rv, P3 avp, P3 bv, P3 cv, P3 ob, P3* bar) {
  const P3 u = vpsub(t, rv, bv), v = vpsub(t, avp, bv), w = vpsub(t, cv, bv);
  P3 N1 = v_cross(u, v), N2 = v_cross(v, w);
  P3 t1 = N1, t2 = N2;
  const P3 n1 = v_normalize(t1), n2 = v_normalize(t2);
  const double div = v_norm(t1);
  P3 vb{0, 0, 0}, n1b{0, 0, 0}, n2b{0, 0, 0};
  double db = 0;
  bend_pair_bar(n1, n2, v, 1.0 / div, ob, vb, n1b, n2b, db);
  n1b = v_add(n1b, v_scale(db, n2));
  n2b = v_add(n2b, v_scale(db, n1));
  const P3 N1b = unit_bar(N1, n1b), N2b = unit_bar(N2, n2b);
  const P3 ub = v_cross(v, N1b);
  vb = v_add(vb, v_add(v_cross(N1b, u), v_cross(w, N2b)));
  const P3 wb = v_cross(N2b, v);
  bar[0] = v_add(bar[0], ub);
  bar[1] = v_add(bar[1], vb);
  bar[3] = v_add(bar[3], wb);
  bar[2] = v_sub(bar[2], v_add(ub, v_add(vb, wb)));
}
// reverse of tri_bend_2(r, a, b, c)
__device__ void tri_bend_2_bar(const Tis& t, P3 rv, P3 avp, P3 bv, P3 cv, P3 ob, P3* bar) {
  const P3 p = vpsub(t, rv, cv), q = vpsub(t, bv, cv);
  const P3 u = vpsub(t, rv, bv), v = vpsub(t, avp, bv);
  P3 N1 = v_cross(p, q), N2 = v_cross(u, v);
  P3 t1 = N1, t2 = N2;
  const P3 n1 = v_normalize(t1), n2 = v_normalize(t2);
  const double div1 = v_norm(t1), div2 = v_norm(t2);
  P3 qb{0, 0, 0}, vb{0, 0, 0}, n1b{0, 0, 0}, n2b{0, 0, 0};
  double db = 0;
  bend_pair_bar(n1, n2, q, 1.0 / div1, ob, qb, n1b, n2b, db);
  bend_pair_bar(n2, n1, v, 1.0 / div2, ob, vb, n2b, n1b, db);
  n1b = v_add(n1b, v_scale(db, n2));
  n2b = v_add(n2b, v_scale(db, n1));
  const P3 N1b = unit_bar(N1, n1b), N2b = unit_bar(N2, n2b);
  const P3 pb = v_cross(q, N1b);
  qb = v_add(qb, v_cross(N1b, p));
  const P3 ub = v_cross(v, N2b);
  vb = v_add(vb, v_cross(N2b, u));
  bar[0] = v_add(bar[0], v_add(pb, ub));
  bar[1] = v_add(bar[1], vb);
  bar[2] = v_add(bar[2], v_sub(qb, v_add(ub, vb)));
  bar[3] = v_sub(bar[3], v_add(pb, qb));
}
}  // namespace

// positions between the tissue's current buffer and the window's storage:
// dir 0 save to slot, 1 restore from slot, 2 save checkpoint, 3 restore
// checkpoint, 4 restore the snapshot (both buffers), 5 take the snapshot
__global__ void __launch_bounds__(256) k_mech_state(const Tis* __restrict__ T, const MechTis* __restrict__ M,
                                                     int slot, int dir, int pb) {
  const Tis& t = T[blockIdx.y];
  const MechTis& m = M[blockIdx.y];
  const int n = t.st->n;
  const long long cap = t.cap;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    for (int a = 0; a < 3; a++) {
      if (dir <= 3) {
        double* st = (dir < 2 ? m.slot : m.ck) + (long long)slot * 3 * cap + a * cap;
        if (dir == 0 || dir == 2) st[c] = t.pos[pb][a][c];
        else t.pos[pb][a][c] = st[c];
      } else if (dir == 4) {
        t.pos[pb][a][c] = m.x0[0][a * cap + c];
        t.pos[1 - pb][a][c] = m.x0[1][a * cap + c];
      } else {
        m.x0[0][a * cap + c] = t.pos[pb][a][c];
        m.x0[1][a * cap + c] = t.pos[1 - pb][a][c];
      }
    }
  }
}

// loss = mean over cells of |x - target|^2 (minimum image in x, y) and the seed
__global__ void __launch_bounds__(256) k_mech_seed(const Tis* __restrict__ T, MechTis* __restrict__ M, int pb,
                                                    int q) {
  const Tis& t = T[blockIdx.y];
  MechTis& m = M[blockIdx.y];
  const int n = t.st->n;
  const long long cap = t.cap;
  double part = 0;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    const double dx = p_diff_x(t, t.pos[pb][0][c], m.target[c]);
    const double dy = p_diff_y(t, t.pos[pb][1][c], m.target[cap + c]);
    const double dz = t.pos[pb][2][c] - m.target[2 * cap + c];
    part += dx * dx + dy * dy + dz * dz;
    m.lam[q][c] = 2 * dx / n;
    m.lam[q][cap + c] = 2 * dy / n;
    m.lam[q][2 * cap + c] = 2 * dz / n;
  }
  for (int o = 32; o > 0; o >>= 1) part += __shfl_down(part, o, 64);
  if ((threadIdx.x & 63) == 0 && part != 0) atomicAdd(&m.scal[0], part / n);
}

// restore the state of slot `slot` and start the next adjoint at the identity
__global__ void __launch_bounds__(256) k_mech_bwd_begin(const Tis* __restrict__ T, MechTis* __restrict__ M, int slot,
                                                         int pb, int q) {
  const Tis& t = T[blockIdx.y];
  MechTis& m = M[blockIdx.y];
  const int n = t.st->n;
  const long long cap = t.cap;
  const double* st = m.slot + (long long)slot * 3 * cap;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x)
    for (int a = 0; a < 3; a++) {
      t.pos[pb][a][c] = st[a * cap + c];
      m.lam[1 - q][a * cap + c] = m.lam[q][a * cap + c];
    }
}

// The reverse kernels take one lane per cell.  A cell's own terms are summed
// by its lane and added with one atomic; the terms of other cells are
// scattered with atomics and the parameter sums are reduced at the end, so
// no order is kept (a gradient need not follow the forward's).  (Lane groups
// per cell measured slower: the laws' branches and the dihedral terms' two
// code paths then run one after the other within a group.)

// every interaction a cell's handler applies (cell_interaction.cpp:529-641)
__global__ void __launch_bounds__(256) k_mech_bwd_pairs(const Tis* __restrict__ T, MechTis* __restrict__ M, int pb,
                                                         int cb, int q) {
  const Tis& t = T[blockIdx.y];
  MechTis& m = M[blockIdx.y];
  const int n = t.st->n;
  const long long cap = t.cap;
  const double* lam = m.lam[q];
  double* nl = m.lam[1 - q];
  ParAcc pa{0, 0, 0};
  for (int X = blockIdx.x * blockDim.x + threadIdx.x; X < n; X += gridDim.x * blockDim.x) {
    const CV cx = load_cv(t, pb, X);
    P3 gx{0, 0, 0};
    if (X < t.nmemb) {
      for (int i = 0; i < MEMB_ADJ; i++) {
        const int o = t.memb6[6 * X + i];
        if (t.state[o] == MEMB && X > o)
          gx = v_add(gx, pair_bwd(t, LAW_MEMB_MEMB, cx, X, load_cv(t, pb, o), o, lam, nl, cap, pa));
      }
    } else {
      const int* row = t.col[cb] + (size_t)X * t.ns;
      const int len = t.nlen[cb][X];
      for (int e = 0; e < len; e++) {
        const int o = row[e];
        const CV co = load_cv(t, pb, o);
        const int law = proc_law(cx, X, co, o);
        if (law != LAW_NONE) gx = v_add(gx, pair_bwd(t, law, cx, X, co, o, lam, nl, cap, pa));
      }
      if (cx.pair >= 0 && X > cx.pair)
        gx = v_add(gx, pair_bwd(t, LAW_PAIR, cx, X, load_cv(t, pb, cx.pair), cx.pair, lam, nl, cap, pa));
    }
    atomic_add3(nl, cap, X, gx);
  }
  for (int o = 32; o > 0; o >>= 1) {
    pa.eps += __shfl_down(pa.eps, o, 64);
    pa.adh += __shfl_down(pa.adh, o, 64);
    pa.spr += __shfl_down(pa.spr, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    if (pa.eps != 0) atomicAdd(&m.scal[1], pa.eps);
    if (pa.adh != 0) atomicAdd(&m.scal[2], pa.adh);
    if (pa.spr != 0) atomicAdd(&m.scal[3], pa.spr);
  }
}

// the wall (membrane and DER cells, :287-294) and the bending of every
// membrane particle (:488-499)
__global__ void __launch_bounds__(256) k_mech_bwd_memb(const Tis* __restrict__ T, MechTis* __restrict__ M, int pb,
                                                        int q) {
  const Tis& t = T[blockIdx.y];
  MechTis& m = M[blockIdx.y];
  const int n = t.st->n;
  const long long cap = t.cap;
  const double* lam = m.lam[q];
  double* nl = m.lam[1 - q];
  double peps = 0, pbend = 0;
  for (int X = blockIdx.x * blockDim.x + threadIdx.x; X < n; X += gridDim.x * blockDim.x) {
    const bool memb = X < t.nmemb;
    if (!memb && t.state[X] != DER) continue;
    const CV cx = load_cv(t, pb, X);
    if (cx.p.z < cx.r) {
      const double z = cx.p.z;
      const double L = POW6(cx.r) / POW6(z);
      atomicAdd(&nl[2 * cap + X], lam[2 * cap + X] * t.prm.DT_Cell * 2.0 * t.m_eps * (7.0 * L - 13.0 * L * L) / (z * z));
      peps += lam[2 * cap + X] * t.prm.DT_Cell * 2.0 * L * (L - 1.0) / z;
    }
    if (!memb) continue;
    const P3 lm = ld3(lam, cap, X);
    const P3 ob = v_scale(t.prm.DT_Cell * t.m_kbend, lm);
    const int* md = t.memb6 + 6 * X;
    P3 dr{0, 0, 0};
    for (int i = 0; i < 6; i++) {
      const int i1 = (i + 1) % 6;
      const int idx[4] = {X, md[i], md[i1], t.memb6[6 * md[i1] + i]};
      const P3 pr = ld_pos(t, pb, idx[1]), pbv = ld_pos(t, pb, idx[2]), pc = ld_pos(t, pb, idx[3]);
      dr = v_add(dr, tri_bend_1(t, cx.p, pr, pbv, pc));
      P3 bar[4] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
      tri_bend_1_bar(t, cx.p, pr, pbv, pc, ob, bar);
      for (int k = 0; k < 4; k++) atomic_add3(nl, cap, idx[k], bar[k]);
    }
    for (int i = 0; i < 6; i++) {
      const int idx[4] = {X, md[i], md[(i + 1) % 6], md[(i + 2) % 6]};
      const P3 pa = ld_pos(t, pb, idx[1]), pbv = ld_pos(t, pb, idx[2]), pc = ld_pos(t, pb, idx[3]);
      dr = v_add(dr, tri_bend_2(t, cx.p, pa, pbv, pc));
      P3 bar[4] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
      tri_bend_2_bar(t, cx.p, pa, pbv, pc, ob, bar);
      for (int k = 0; k < 4; k++) atomic_add3(nl, cap, idx[k], bar[k]);
    }
    pbend += t.prm.DT_Cell * v_dot(lm, dr);
  }
  for (int o = 32; o > 0; o >>= 1) {
    peps += __shfl_down(peps, o, 64);
    pbend += __shfl_down(pbend, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    if (peps != 0) atomicAdd(&m.scal[1], peps);
    if (pbend != 0) atomicAdd(&m.scal[4], pbend);
  }
}

void launch_mech_state(hipStream_t s, const Tis* dT, const MechTis* dM, int ntis, int slot, int dir, int pb,
                       int max_n) {
  EPI_LAUNCH(K_MECH_STATE, k_mech_state, dim3((max_n + 255) / 256, ntis), dim3(256), 0, s, dT, dM, slot, dir, pb);
}
void launch_mech_seed(hipStream_t s, const Tis* dT, MechTis* dM, int ntis, int pb, int q, int max_n) {
  EPI_LAUNCH(K_MECH_SEED, k_mech_seed, dim3((max_n + 255) / 256, ntis), dim3(256), 0, s, dT, dM, pb, q);
}
void launch_mech_backward_step(hipStream_t s, const Tis* dT, MechTis* dM, int ntis, int slot, int pb, int cb, int q,
                               int max_n) {
  const dim3 g((max_n + 255) / 256, ntis);
  EPI_LAUNCH(K_MECH_BWD_BEGIN, k_mech_bwd_begin, g, dim3(256), 0, s, dT, dM, slot, pb, q);
  EPI_LAUNCH(K_MECH_BWD_PAIRS, k_mech_bwd_pairs, g, dim3(256), 0, s, dT, dM, pb, cb, q);
  EPI_LAUNCH(K_MECH_BWD_MEMB, k_mech_bwd_memb, g, dim3(256), 0, s, dT, dM, pb, q);
}

}  // namespace epi
