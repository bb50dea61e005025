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

// What a force law reads of a cell, from two records: pk[pb] (position and
// radius, 32 bytes) and fa (pair, dermis, rest_div_times, and state with
// whether the age passes THRESH_SP, 16 bytes).  A gather touches two cache
// lines a lane, where the ten arrays the records are made from touched ten
// (the address units were busy for half of k_forces).  In a step the bucket
// insertion writes pk and k_finish fa; force_pack writes both where a force
// kernel does not follow a build; in a window k_forces writes the next pk.
// snl is read for a pair's spring alone (load_cv_snl).
struct CV {
  P3 p;
  double r, snl;
  bool strong;   // agek > THRESH_SP
  int pair, dermis, rdt;
  uint8_t s;
};

__device__ __forceinline__ CV load_cv(const Tis& t, int pb, int c) {
  const double4 p = t.pk[pb][c];
  const int4 f = t.fa[c];
  CV v;
  v.p = P3{p.x, p.y, p.z};
  v.r = p.w;
  v.pair = f.x;
  v.dermis = f.y;
  v.rdt = f.z;
  v.s = (uint8_t)(f.w & 255);
  v.strong = f.w >> 8;
  return v;
}
__device__ __forceinline__ CV load_cv_snl(const Tis& t, int pb, int c) {
  CV v = load_cv(t, pb, c);
  v.snl = t.spr_nat_len[c];
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
    if (a.strong && b.strong) K = t.m_kadh;
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
      const P3 d = delta(t, LAW_PAIR, load_cv_snl(t, pb, X), load_cv(t, pb, cx.pair), st);
      acc.x += d.x; acc.y += d.y; acc.z += d.z;
    }
    int P = cx.pair > X ? cx.pair : -1;
    for (int i = nlo; i < len; i++) {
      const int p = row[i];
      if (P >= 0 && P < p) {
        const P3 d = delta(t, LAW_PAIR, load_cv_snl(t, pb, P), cx, st);
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
        const P3 d = delta(t, LAW_PAIR, load_cv_snl(t, pb, p), cx, st);
        acc.x -= d.x; acc.y -= d.y; acc.z -= d.z;
        P = -1;
      }
    }
    if (P >= 0) {
      const P3 d = delta(t, LAW_PAIR, load_cv_snl(t, pb, P), cx, st);
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
// form on its own and a leader summing all three; then the packed records and
// the dihedrals' indices asked for early: 100 steps of one tissue of 3,900
// cells 1490 -> 1083 -> 1043 us, a launch for 24 tissues of 105,000 cells
// 82.6 -> 63.5 -> 60.1 us (without the laws 50, without the sums 57).
//
// FCAP, the LDS slots per cell, is chosen per launch from the longest list
// built so far: 40 keeps a 128-lane block's LDS small enough for 4 waves per
// SIMD, 48 and 64 take longer lists at lower occupancy, and rows beyond 64 go
// to k_forces_long.
constexpr int FG = 16;
constexpr int F_BLOCK = 128;
constexpr int F_GROUPS = F_BLOCK / FG;
static_assert(FG <= ROW_SLOTS_MIN, "a lane's first entry lies inside its cell's row");

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
__global__ void __launch_bounds__(F_BLOCK) k_forces(const Tis* __restrict__ T, int pb, int cb, StatusOut out,
                                                    MechSave save) {
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
  const int q0 = row[lane];   // a row holds ns >= ROW_SLOTS_MIN > FG slots
  const int n = st->n;
  if (blockIdx.x == 0 && threadIdx.x == 0 && (long long)gridDim.x * F_GROUPS < n) set_force_err(st, ERR_INVALID);
  if (X >= n) return;
  if (len > FCAP) return;   // k_forces_long
  // a membrane particle's dihedral of this lane: its cells' indices are asked
  // for before the laws, so that only their positions are left to wait for
  int ma = 0, mb = 0, mc = 0;
  if (memb && lane < 12) {
    const int* md = t.memb6 + 6 * X;
    const int i = lane < 6 ? lane : lane - 6;
    ma = md[i];
    mb = md[i == 5 ? 0 : i + 1];
    mc = lane < 6 ? t.memb6[6 * mb + i] : md[i >= 4 ? i - 4 : i + 2];
  }
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
      a.strong = cx.strong; b.strong = cq.strong;
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
    const double4 ap = t.pk[pb][ma], bp = t.pk[pb][mb], cp = t.pk[pb][mc];
    s_bend[grp][lane] = tri_bend(t, lane >= 6, cx.p, P3{ap.x, ap.y, ap.z}, P3{bp.x, bp.y, bp.z}, P3{cp.x, cp.y, cp.z});
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
  if (lane >= 3) {
    if (lane == 3 && save.chain) t.pk[1 - pb][X].w = cx.r;
    return;
  }
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
      const bool up = X > cx.pair;   // the handler of the pair is the higher index
      const CV ca = load_cv_snl(t, pb, up ? X : cx.pair), cp = load_cv(t, pb, up ? cx.pair : X);
      const double dp = p3_at(delta(t, LAW_PAIR, ca, cp, st), lane);
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
  if (save.chain) reinterpret_cast<double*>(static_cast<double4*>(t.pk[1 - pb]))[4LL * X + lane] = acc;
  if (save.m) save.m[blockIdx.y].slot[(3LL * save.slot + lane) * t.cap + X] = acc;
}

// cells whose rows exceed the LDS slots (cap) of k_forces, one lane per cell
__global__ void __launch_bounds__(256) k_forces_long(const Tis* __restrict__ T, int pb, int cb, int cap,
                                                     MechSave save) {
  const Tis& t = T[blockIdx.y];
  const int n = t.st->n;
  for (int X = blockIdx.x * blockDim.x + threadIdx.x; X < n; X += gridDim.x * blockDim.x)
    if (t.nlen[cb][X] > cap) {
      forces_serial(t, pb, cb, X, t.st);
      if (save.chain) t.pk[1 - pb][X] = make_double4(t.pos[1 - pb][0][X], t.pos[1 - pb][1][X], t.pos[1 - pb][2][X], t.radius[X]);
      if (save.m)
        for (int a = 0; a < 3; a++) save.m[blockIdx.y].slot[(3LL * save.slot + a) * t.cap + X] = t.pos[1 - pb][a][X];
    }
}

int launch_forces_rows(hipStream_t s, const Tis* dT, int ntis, int pb, int cb, int max_other, int max_len,
                       const StatusOut& out, const MechSave& save) {
  dim3 g((max_other + F_GROUPS - 1) / F_GROUPS, ntis);
  int cap;
  if (max_len <= 40) {
    cap = 40;
    EPI_LAUNCH(K_FORCES, k_forces<40>, g, dim3(F_BLOCK), 0, s, dT, pb, cb, out, save);
  } else if (max_len <= 48) {
    cap = 48;
    EPI_LAUNCH(K_FORCES, k_forces<48>, g, dim3(F_BLOCK), 0, s, dT, pb, cb, out, save);
  } else {
    cap = FORCES_ROW_CAP;
    EPI_LAUNCH(K_FORCES, k_forces<FORCES_ROW_CAP>, g, dim3(F_BLOCK), 0, s, dT, pb, cb, out, save);
  }
  return cap;
}

void launch_forces_long(hipStream_t s, const Tis* dT, int ntis, int pb, int cb, int max_other, int cap,
                        const MechSave& save) {
  dim3 gl((max_other + 255) / 256, ntis);
  EPI_LAUNCH(K_FORCES_LONG, k_forces_long, gl, dim3(256), 0, s, dT, pb, cb, cap, save);
}

// the records load_cv reads, from the cells' arrays
__global__ void __launch_bounds__(256) k_force_pack(const Tis* __restrict__ T, int pb) {
  const Tis& t = T[blockIdx.y];
  const double THRESH_SP = t.prm.THRESH_SP;
  const int n = t.st->n;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    const P3 p = P3{t.pos[pb][0][c], t.pos[pb][1][c], t.pos[pb][2][c]};
    const int4 f = force_attr(t.pair[c], t.dermis[c], t.rest_div_times[c], t.state[c], t.agek[c] > THRESH_SP);
    t.pk[pb][c] = make_double4(p.x, p.y, p.z, t.radius[c]);
    t.fa[c] = f;
  }
}

void launch_force_pack(hipStream_t s, const Tis* dT, int ntis, int pb, int max_n) {
  EPI_LAUNCH(K_FORCE_PACK, k_force_pack, dim3((max_n + 255) / 256, ntis), dim3(256), 0, s, dT, pb);
}

void launch_forces(hipStream_t s, const Tis* dT, int ntis, int pb, int cb, int max_other, int max_len,
                   const MechSave& save) {
  const int cap = launch_forces_rows(s, dT, ntis, pb, cb, max_other, max_len, StatusOut{}, save);
  if (max_len > cap) launch_forces_long(s, dT, ntis, pb, cb, max_other, cap, save);
}

// ==== frozen mechanics window: the reverse pass ==============================
// The window is the plain k_forces step repeated with lists, states, pairs
// and dermis frozen.  Which interactions apply depends only on that frozen
// data, so the reverse pass enumerates them from each handler cell (its own
// list, its pair, the membrane slots), evaluates the derivative of the
// active branch of each law at the step's positions, and takes
// lam_c1 - lam_c2 through the pair's Jacobian.
//
// A group of lanes owns a cell (16 a membrane particle, whose 12 dihedrals
// and six neighbours they take; 4 another cell), over the interactions that
// k_mech_plan has packed, and for the same reason as in k_forces the laws and
// the two dihedral forms each run as one code path: the quotients the common
// laws share (1 / d^2, 1 / R, d) are taken once, and the operands chosen per
// lane.  An interaction is evaluated from both of its cells, each keeping its
// own side, so that the cells past the membrane need no atomics: those leave
// the chip's L2s, which cost more than evaluating a law twice.  A membrane
// particle's terms of its six neighbours, which the dihedrals meet two to three
// times each, are summed before an atomic (39 a particle instead of 144).  Sums
// are reduced in another order than the serial reverse's, as a gradient may.
//
// One lane per cell before (two launches and a third for the copies): its
// waves, fewer than two a SIMD, each walked a whole list through every law's
// own branch.  24 tissues, 105,000 cells, a step: 134 us; lane groups over the
// handlers' entries with atomics for the other cell 76 (8 lanes a cell 79; of
// it the atomics 25); both sides evaluated 63.
constexpr int MG = 16;   // of a membrane particle
constexpr int MC = 4;    // of another cell
static_assert(MG <= MECH_ROW_MIN && MC <= MECH_ROW_MIN, "a lane's first slot lies inside its cell's plan row");

namespace {
struct LawD { double coef, ds, deps, dadh, dspr; };

// What the reverse pass needs to know of an interaction besides the two cells'
// positions and radii: the law and the one choice inside it that frozen data
// make.  They hold for a whole window, so k_mech_plan stores them, with the
// entries that have a law, once per gradient.
enum : int { CODE_LAW = 15, CODE_1 = 16, CODE_2 = 32, CODE_OWN = 64 };   // CODE_OWN: this cell is the handler
__device__ __forceinline__ int law_code(const Tis& t, int law, const CV& a, const CV& b) {
  if (law == LAW_ALAIRDE) return law | (a.strong && b.strong ? CODE_1 : 0);
  if (law == LAW_MU_MEMB) return law | (a.pair >= 0 && t.state[a.pair] == FIX ? CODE_1 : a.rdt > 0 ? CODE_2 : 0);
  return law;
}

// coef of the law of `code` at squared distance s and radius sum R (snl: the
// pair spring's natural length) and its derivatives with respect to s and to
// eps_m, K_TOTAL, Kspring.  Forms as in coef_law.
__device__ __forceinline__ LawD coef_law_d(const Tis& t, int code, double R, double snl, double s) {
  const int law = code & CODE_LAW;
  const double eps = t.m_eps;
  LawD r{0, 0, 0, 0, 0};
  if (law == LAW_PAIR) {
    const double d = sqrt(s);
    r.coef = -(t.prm.Kspring_division * (d - snl)) / d;
    r.ds = -t.prm.Kspring_division * snl / (2 * d * d * d);
    return r;
  }
  if (law == LAW_DER_DER) {
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
  const bool memb = law == LAW_MEMB_MEMB;
  const double cr = memb ? R * t.prm.P_MEMB : R;
  if (memb && !(s < cr * cr) && !(s < R * R)) {   // stretched MEMB-MEMB
    const double d = sqrt(s);
    const double lam = (1.0 + t.prm.P_MEMB) * R;
    const double m = lam - d;
    const double L = POW6(cr) / POW6(m);
    const double dL = 6.0 * L / m;
    const double q = L * (L - 1.0) / (m * d);
    const double dq = (2 * L - 1) * dL / (m * d) + L * (L - 1.0) * (d - m) / ((m * d) * (m * d));
    return LawD{-(t.prm.DER_DER_CONST / R) * ((1.0 - t.prm.P_MEMB) / t.prm.P_MEMB) - 4 * eps * q, -4 * eps * dq / (2 * d),
                -4 * q, 0, 0};
  }
  const double is = 1.0 / s;
  if (law == LAW_OTHER || s < cr * cr) {   // ljmain
    const double Q = POW6(cr) * (is * is * is);
    const double c1 = 4.0 * Q * (Q - 1.0) * is;
    return LawD{eps * c1, 4.0 * eps * (4.0 * Q - 7.0 * Q * Q) * (is * is), c1, 0, 0};
  }
  // K times the unit of the parameter that scales it: ka of K_TOTAL, ks of
  // Kspring, kc of neither
  double ka = 0, ks = 0, kc = 0;
  if (law == LAW_ALAIRDE) {
    ka = code & CODE_1 ? 1.0 : t.prm.K_DESMOSOME_RATIO;
  } else if (law == LAW_FIXMU) {
    ka = t.prm.K_DESMOSOME_RATIO;
  } else if (law == LAW_FIX_MEMB) {
    ks = 1.0;
  } else if (law == LAW_MU_MEMB) {
    if (code & CODE_1) ks = 1.0;
    else if (code & CODE_2) kc = t.prm.Kspring_d;
  } else {
    kc = t.prm.DER_DER_CONST;
  }
  const double K = ka * t.m_kadh + ks * t.m_kspring + kc;
  const double d = sqrt(s), id = d * is, iR = 1.0 / cr;
  const double x = d * iR - 1.0;
  double g = x, dg = iR;   // the anchor and the relaxed membrane
  if (!memb && law != LAW_FIX_MEMB) {   // adhesion
    if (x + 1 > t.prm.LJ_THRESH) return r;
    const double c2 = (t.prm.LJ_THRESH - 1.0) * (t.prm.LJ_THRESH - 1.0);
    const double y = x * x / c2;
    g = x * (1 - y);
    dg = (1 - 3 * y) * iR;
  }
  r.coef = -K * id * g;
  r.ds = 0.5 * K * id * (g * is - id * dg);
  r.dadh = -ka * id * g;
  r.dspr = -ks * id * g;
  return r;
}

struct ParAcc { double eps, adh, spr, bend; };
__device__ __forceinline__ P3 ld3(const double* v, long long cap, int c) { return P3{v[c], v[cap + c], v[2 * cap + c]}; }
__device__ __forceinline__ void atomic_add3(double* v, long long cap, int c, P3 g) {
  atomicAdd(&v[c], g.x);
  atomicAdd(&v[cap + c], g.y);
  atomicAdd(&v[2 * cap + c], g.z);
}
template <int G>
__device__ __forceinline__ P3 p3_group_sum(P3 v) {
#pragma unroll
  for (int o = 1; o < G; o <<= 1) {
    v.x += __shfl_xor(v.x, o, G);
    v.y += __shfl_xor(v.y, o, G);
    v.z += __shfl_xor(v.z, o, G);
  }
  return v;
}
__device__ __forceinline__ P3 p3_shfl(P3 v, int src) {
  return P3{__shfl(v.x, src, MG), __shfl(v.y, src, MG), __shfl(v.z, src, MG)};
}

// the adjoint term of an interaction for one of its two cells, at a; the
// formula is the same from either side (r and la - lb change sign together).
// The parameters' sums take it once, with the handler.
__device__ __forceinline__ P3 pair_bwd(const Tis& t, int code, P3 a, P3 b, double R, double snl, P3 la, P3 lb,
                                       ParAcc& pa) {
  const P3 r = vpsub(t, a, b);
  const LawD ld = coef_law_d(t, code, R, snl, v_dot(r, r));
  const P3 av = v_sub(la, lb);
  const double ar = v_dot(av, r), DT = t.prm.DT_Cell;
  const double k2 = 2 * ld.ds * ar;
  const double once = code & CODE_OWN ? DT * ar : 0.0;
  pa.eps += ld.deps * once;
  pa.adh += ld.dadh * once;
  pa.spr += ld.dspr * once;
  return P3{DT * (ld.coef * av.x + k2 * r.x), DT * (ld.coef * av.y + k2 * r.y), DT * (ld.coef * av.z + k2 * r.z)};
}

// the wall's term for z (:287-294)
__device__ __forceinline__ double wall_bwd(const Tis& t, double z, double radius, double lz, ParAcc& pa) {
  const double L = POW6(radius) / POW6(z), DT = t.prm.DT_Cell;
  pa.eps += lz * DT * 2.0 * L * (L - 1.0) / z;
  return lz * DT * 2.0 * t.m_eps * (7.0 * L - 13.0 * L * L) / (z * z);
}

__device__ __forceinline__ double bend_factor_d(double c) {
  if (c >= 0) return -1.0;
  return -2.0 / ((1.0 + c) * (1.0 + c) * (1.0 + c));
}
// v with its part along the unit vector n taken out, over |N|
__device__ __forceinline__ P3 unit_bar(P3 n, double inv, P3 nb) { return v_scale(inv, v_sub(nb, v_scale(v_dot(nb, n), n))); }

// reverse of tri_bend(second; r, a, b, c) for the adjoint ob = kb lm of its
// value: bar[0..3] are the adjoints of r, a, b, c; lm . value is returned.
// With y = f(d) (A2 x rho1 + [2] ab x rho2), d = n1.n2, rho1 = n2 - d n1,
// rho2 = n1 - d n2 (the normals' own norms, 1, carry no derivative).
__device__ __forceinline__ double tri_bend_bar(const Tis& t, bool second, P3 rv, P3 av, P3 bv, P3 cv, P3 lm, double kb,
                                               P3* bar) {
  const P3 ab = vpsub(t, av, bv), rb = vpsub(t, rv, bv);
  const P3 rc = vpsub(t, rv, cv);
  const P3 bc = vpsub(t, p3_sel(second, bv, cv), p3_sel(second, cv, bv));   // c - b of form 1
  const P3 A1 = p3_sel(second, rc, rb), A2 = p3_sel(second, bc, ab);
  const P3 B1 = p3_sel(second, rb, ab), B2 = p3_sel(second, ab, bc);
  const P3 N1 = v_cross(A1, A2), N2 = v_cross(B1, B2);
  const double inv1 = 1.0 / v_norm(N1), inv2 = 1.0 / v_norm(N2);
  const P3 n1 = v_scale(inv1, N1), n2 = v_scale(inv2, N2);
  const double d = v_dot(n1, n2);
  const P3 rho1 = v_sub(n2, v_scale(d, n1)), rho2 = v_sub(n1, v_scale(d, n2));
  const double f = bend_factor(d);
  const P3 oy = v_scale(f * kb, lm);
  P3 V = v_cross(A2, rho1), ab_b{0, 0, 0}, n1b{0, 0, 0}, n2b = v_cross(oy, A2);
  P3 A2b = v_cross(rho1, oy);
  double db = -v_dot(n2b, n1);
  n1b = v_scale(-d, n2b);
  if (second) {
    V = v_add(V, v_cross(ab, rho2));
    ab_b = v_cross(rho2, oy);
    const P3 q = v_cross(oy, ab);
    n1b = v_add(n1b, q);
    db -= v_dot(q, n2);
    n2b = v_sub(n2b, v_scale(d, q));
  }
  const double val = v_dot(lm, V);
  db += bend_factor_d(d) * kb * val;
  n1b = v_add(n1b, v_scale(db, n2));
  n2b = v_add(n2b, v_scale(db, n1));
  const P3 N1b = unit_bar(n1, inv1, n1b), N2b = unit_bar(n2, inv2, n2b);
  const P3 A1b = v_cross(A2, N1b);
  A2b = v_add(A2b, v_cross(N1b, A1));
  const P3 B1b = v_cross(B2, N2b), B2b = v_cross(N2b, B1);
  // form 1: A1 = rb, A2 = B1 = ab, B2 = cb; form 2: A1 = rc, A2 = bc, B1 = rb, B2 = ab
  const P3 rbb = p3_sel(second, B1b, A1b);
  const P3 abb = p3_sel(second, v_add(ab_b, B2b), v_add(A2b, B1b));
  const P3 zero{0, 0, 0};
  const P3 rcb = p3_sel(second, A1b, zero);
  const P3 bcb = p3_sel(second, A2b, v_scale(-1.0, B2b));   // of b - c
  bar[0] = v_add(rbb, rcb);
  bar[1] = abb;
  bar[2] = v_sub(bcb, v_add(rbb, abb));
  bar[3] = v_sub(v_scale(-1.0, rcb), bcb);
  return f * val;
}

// this lane's share of a cell's planned interactions
template <int G>
__device__ __forceinline__ P3 planned_bwd(const Tis& t, const MechTis& m, const double* px, const double* lam, int X, P3 xp,
                                          P3 lx, double xr, int lane, ParAcc& pa) {
  const long long cap = t.cap;
  const int* ent = m.ent + (size_t)X * m.es;
  const uint8_t* code = m.code + (size_t)X * m.es;
  const int o0 = ent[lane], k0 = code[lane];   // in one round trip with the row's length (a row has MECH_ROW_MIN slots)
  const int len = m.ent_n[X];
  P3 own{0, 0, 0};
  for (int e = lane; e < len; e += G) {
    const int o = e == lane ? o0 : ent[e], k = e == lane ? k0 : code[e];
    // a pair's spring has the natural length of its handler, the higher index
    const double snl = (k & CODE_LAW) == LAW_PAIR ? t.spr_nat_len[max(X, o)] : 0.0;
    own = v_add(own, pair_bwd(t, k, xp, ld3(px, cap, o), xr + t.radius[o], snl, lx, ld3(lam, cap, o), pa));
  }
  return own;
}

// a membrane particle: its dihedrals (:488-499), its membrane neighbours, the wall
__device__ __forceinline__ void bwd_membrane(const Tis& t, const MechTis& m, const double* px, const double* lam, double* nl,
                                             int X, int lane, ParAcc& pa) {
  const long long cap = t.cap;
  const int i = lane < 6 ? lane : lane < 12 ? lane - 6 : 0;   // lanes from 12 on take no term
  const int ma = t.memb6[6 * X + i];
  const P3 xp = ld3(px, cap, X), lm = ld3(lam, cap, X);
  const double xr = t.radius[X];
  P3 own = planned_bwd<MG>(t, m, px, lam, X, xp, lm, xr, lane, pa);
  if (lane == 12 && xp.z < xr) own.z += wall_bwd(t, xp.z, xr, lm.z, pa);
  const int mb = __shfl(ma, i == 5 ? 0 : i + 1, MG);
  const int m2 = __shfl(ma, i >= 4 ? i - 4 : i + 2, MG);
  const int mc = lane < 6 ? t.memb6[6 * mb + i] : m2;
  const P3 ap = ld3(px, cap, ma), bp = ld3(px, cap, mb), cp = ld3(px, cap, mc);
  // the membrane pair before the dihedral: its operands are done with by then
  P3 nb{0, 0, 0};
  if (lane < 6 && t.state[ma] == MEMB && X > ma) {
    const P3 g = pair_bwd(t, LAW_MEMB_MEMB | CODE_OWN, xp, ap, xr + t.radius[ma], 0.0, lm, ld3(lam, cap, ma), pa);
    own = v_add(own, g);
    nb = v_scale(-1.0, g);
  }
  P3 bar[4];
  const double val = tri_bend_bar(t, lane >= 6, xp, ap, bp, cp, lm, t.prm.DT_Cell * t.m_kbend, bar);
  if (lane < 12) {
    pa.bend += t.prm.DT_Cell * val;
    own = v_add(own, bar[0]);
  }
  if (lane < 6) atomic_add3(nl, cap, mc, bar[3]);
  // neighbour i of X (lanes 0 to 5): a of the dihedrals i, b of those before
  // it, c of form 2's two before
  const int i1 = i == 0 ? 5 : i - 1, i2 = i < 2 ? i + 4 : i - 2;
  nb = v_add(v_add(nb, v_add(bar[1], p3_shfl(bar[2], i1))), v_add(p3_shfl(bar[1], 6 + i), p3_shfl(bar[2], 6 + i1)));
  nb = v_add(nb, p3_shfl(bar[3], 6 + i2));
  if (lane < 6) atomic_add3(nl, cap, ma, nb);
  own = v_add(p3_group_sum<MG>(own), lm);
  if (lane < 3) atomicAdd(&nl[lane * cap + X], lane == 0 ? own.x : lane == 1 ? own.y : own.z);
}

// the planned interactions of another cell, and a DER cell's wall; nothing
// else reaches the cell's adjoint, so it is stored, not added
__device__ __forceinline__ void bwd_cell(const Tis& t, const MechTis& m, const double* px, const double* lam, double* nl,
                                         int X, int lane, ParAcc& pa) {
  const long long cap = t.cap;
  const P3 xp = ld3(px, cap, X), lx = ld3(lam, cap, X);
  const double xr = t.radius[X];
  const bool der = t.state[X] == DER;
  P3 own = planned_bwd<MC>(t, m, px, lam, X, xp, lx, xr, lane, pa);
  if (lane == MC - 1 && der && xp.z < xr) own.z += wall_bwd(t, xp.z, xr, lx.z, pa);
  own = v_add(p3_group_sum<MC>(own), lx);
  if (lane < 3) nl[lane * cap + X] = lane == 0 ? own.x : lane == 1 ? own.y : own.z;
}
}  // namespace

// positions between the tissue's current buffer and the window's storage:
// dir 0 save to slot, 1 restore from slot, 2 save checkpoint, 3 restore
// checkpoint (and keep it as slot 0), 4 restore the snapshot (both buffers),
// 5 take the snapshot
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
        if (dir == 3) m.slot[a * cap + c] = st[c];
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
                                                    int q, int nblk) {
  const Tis& t = T[blockIdx.y];
  MechTis& m = M[blockIdx.y];
  const int n = t.st->n;
  const long long cap = t.cap;
  double part = 0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < 4 * nblk; i += gridDim.x * blockDim.x) m.part[i] = 0;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) {
    const double dx = p_diff_x(t, t.pos[pb][0][c], m.target[c]);
    const double dy = p_diff_y(t, t.pos[pb][1][c], m.target[cap + c]);
    const double dz = t.pos[pb][2][c] - m.target[2 * cap + c];
    part += dx * dx + dy * dy + dz * dz;
    m.lam[q][c] = 2 * dx / n;
    m.lam[q][cap + c] = 2 * dy / n;
    m.lam[q][2 * cap + c] = 2 * dz / n;
    for (int a = 0; a < 3; a++) m.lam[q + 1][a * cap + c] = 0;
  }
  for (int o = 32; o > 0; o >>= 1) part += __shfl_down(part, o, 64);
  if ((threadIdx.x & 63) == 0 && part != 0) atomicAdd(&m.scal[0], part / n);
}

// Every interaction a cell takes part in, as its handler or as the other cell
// (cell_interaction.cpp:529-641; rows are symmetric but for the membrane's six
// slots, which bwd_membrane takes), and its pair's spring, packed by ballots of
// MG lanes per cell.  A row's entry has two where both cells are DER.
__global__ void __launch_bounds__(256) k_mech_plan(const Tis* __restrict__ T, MechTis* __restrict__ M, int pb, int cb) {
  const Tis& t = T[blockIdx.y];
  const MechTis& m = M[blockIdx.y];
  const int n = t.st->n;
  const int lane = threadIdx.x & (MG - 1), sh = threadIdx.x & 63 & ~(MG - 1);
  for (int X = blockIdx.x * (256 / MG) + threadIdx.x / MG; X < n; X += gridDim.x * (256 / MG)) {
    const bool memb = X < t.nmemb;
    const int* row = t.col[cb] + (size_t)X * t.ns;
    const CV cx = load_cv(t, pb, X);
    const int len = t.nlen[cb][X], all = len + (!memb && cx.pair >= 0);
    int at = 0;
    for (int e0 = memb ? MEMB_ADJ : 0; e0 < all; e0 += MG) {
      const int e = e0 + lane;
      const int o = e < len ? row[e] : e < all ? cx.pair : X;
      const CV co = load_cv(t, pb, o);
      int code[2] = {LAW_NONE, LAW_NONE};   // as the handler, as the other cell
      if (e < len) {
        const int own = memb ? (int)LAW_NONE : proc_law(cx, X, co, o);
        const int oth = o < t.nmemb ? (int)LAW_NONE : proc_law(co, o, cx, X);
        if (own != LAW_NONE) code[0] = law_code(t, own, cx, co) | CODE_OWN;
        if (oth != LAW_NONE) code[1] = law_code(t, oth, co, cx);
      } else if (e < all) {
        code[0] = LAW_PAIR | (X > o ? CODE_OWN : 0);
      }
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const unsigned mk = (unsigned)(__ballot(code[k] != LAW_NONE) >> sh) & ((1u << MG) - 1);
        if (code[k] != LAW_NONE) {
          const int slot = at + __popc(mk & ((1u << lane) - 1));
          m.ent[(size_t)X * m.es + slot] = o;
          m.code[(size_t)X * m.es + slot] = (uint8_t)code[k];
        }
        at += __popc(mk);
      }
    }
    if (lane == 0) m.ent_n[X] = at;
  }
}

// One reverse step from the state in slot `slot`: lam[q] (after the step) to
// lam[q + 1] (before it), which the step before cleared, and lam[q + 2] cleared
// for the next.  Blocks [0, mblk) take the membrane, the rest the other cells.
// A block adds its share of the parameters' adjoints to its own words of part.
__global__ void __launch_bounds__(256) k_mech_bwd(const Tis* __restrict__ T, MechTis* __restrict__ M, int slot, int q,
                                                   int mblk) {
  const Tis& t = T[blockIdx.y];
  MechTis& m = M[blockIdx.y];
  const long long cap = t.cap;
  const double* px = m.slot + (long long)slot * 3 * cap;
  const double* lam = m.lam[q];
  double* nl = m.lam[q == 2 ? 0 : q + 1];
  double* dead = m.lam[q == 0 ? 2 : q - 1];
  const bool memb = (int)blockIdx.x < mblk;
  const int nblk = memb ? mblk : gridDim.x - mblk, bid = memb ? blockIdx.x : blockIdx.x - mblk;
  ParAcc pa{0, 0, 0, 0};
  if (memb) {
    const int lane = threadIdx.x & (MG - 1), step = nblk * (256 / MG);
    for (int X = bid * (256 / MG) + threadIdx.x / MG; X < t.nmemb; X += step) {
      if (lane < 3) dead[lane * cap + X] = 0;
      bwd_membrane(t, m, px, lam, nl, X, lane, pa);
    }
  } else {
    const int lane = threadIdx.x & (MC - 1), step = nblk * (256 / MC), n = t.st->n;
    for (int X = t.nmemb + bid * (256 / MC) + threadIdx.x / MC; X < n; X += step) {
      if (lane < 3) dead[lane * cap + X] = 0;
      bwd_cell(t, m, px, lam, nl, X, lane, pa);
    }
  }
  __shared__ double s_pa[4][4];
  double v[4] = {pa.eps, pa.adh, pa.spr, pa.bend};
#pragma unroll
  for (int k = 0; k < 4; k++) {
    for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_down(v[k], o, 64);
    if ((threadIdx.x & 63) == 0) s_pa[threadIdx.x >> 6][k] = v[k];
  }
  __syncthreads();
  if (threadIdx.x < 4)
    m.part[4 * blockIdx.x + threadIdx.x] +=
        s_pa[0][threadIdx.x] + s_pa[1][threadIdx.x] + s_pa[2][threadIdx.x] + s_pa[3][threadIdx.x];
}

// the parameters' adjoints of a window from its blocks' sums, one block per tissue
__global__ void __launch_bounds__(256) k_mech_sums(MechTis* __restrict__ M, int nblk) {
  MechTis& m = M[blockIdx.y];
  double v = 0;   // the thread's values all belong to one parameter: 256 is a multiple of 4
  for (int i = threadIdx.x; i < 4 * nblk; i += 256) v += m.part[i];
  __shared__ double s_v[4][4];
  for (int o = 32; o >= 4; o >>= 1) v += __shfl_down(v, o, 64);
  if ((threadIdx.x & 63) < 4) s_v[threadIdx.x >> 6][threadIdx.x & 3] = v;
  __syncthreads();
  if (threadIdx.x < 4)
    m.scal[1 + threadIdx.x] = s_v[0][threadIdx.x] + s_v[1][threadIdx.x] + s_v[2][threadIdx.x] + s_v[3][threadIdx.x];
}

void launch_mech_state(hipStream_t s, const Tis* dT, const MechTis* dM, int ntis, int slot, int dir, int pb,
                       int max_n) {
  EPI_LAUNCH(K_MECH_STATE, k_mech_state, dim3((max_n + 255) / 256, ntis), dim3(256), 0, s, dT, dM, slot, dir, pb);
}
void launch_mech_seed(hipStream_t s, const Tis* dT, MechTis* dM, int ntis, int pb, int q, int max_n, int nblk) {
  EPI_LAUNCH(K_MECH_SEED, k_mech_seed, dim3((max_n + 255) / 256, ntis), dim3(256), 0, s, dT, dM, pb, q, nblk);
}
namespace {
int mech_blocks(int cells, int lanes) { return (int)(((long long)cells * lanes + 255) / 256); }
}  // namespace
int mech_bwd_blocks(int max_memb, int max_other) { return mech_blocks(max_memb, MG) + mech_blocks(max_other, MC); }
void launch_mech_plan(hipStream_t s, const Tis* dT, MechTis* dM, int ntis, int pb, int cb, int max_n) {
  EPI_LAUNCH(K_MECH_PLAN, k_mech_plan, dim3(mech_blocks(max_n, MG), ntis), dim3(256), 0, s, dT, dM, pb, cb);
}
void launch_mech_backward_step(hipStream_t s, const Tis* dT, MechTis* dM, int ntis, int slot, int q, int max_memb,
                               int max_other) {
  EPI_LAUNCH(K_MECH_BWD, k_mech_bwd, dim3(mech_bwd_blocks(max_memb, max_other), ntis), dim3(256), 0, s, dT, dM, slot, q,
             mech_blocks(max_memb, MG));
}
void launch_mech_sums(hipStream_t s, MechTis* dM, int ntis, int nblk) {
  EPI_LAUNCH(K_MECH_SUMS, k_mech_sums, dim3(1, ntis), dim3(256), 0, s, dM, nblk);
}

}  // namespace epi
