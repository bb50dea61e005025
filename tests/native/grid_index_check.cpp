// Host build of the grid index arithmetic of the Ca corners
// (epi_amd/csrc/ca_corner.h) and of the voxel-map stamp
// (epi_amd/csrc/field_step.h), for tests/test_grid_indices.py.  The grids are
// sparse: a reservation of address space whose pages exist once written, so that
// grids far larger than the memory of this machine can be addressed.
#include <algorithm>
#include <sys/mman.h>

#include "device_on_host.h"
#include "../../epi_amd/csrc/ca_corner.h"
#include "../../epi_amd/csrc/field_step.h"

using namespace epi;

namespace {
template <class T>
struct Sparse {
  T* p = nullptr;
  size_t bytes;
  explicit Sparse(long long n) : bytes(sizeof(T) * (size_t)n) {
    void* m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m != MAP_FAILED) p = static_cast<T*>(m);
  }
  ~Sparse() { if (p) munmap(p, bytes); }
};

struct Grid {   // the members that corner_word, corner_load and corner_new read
  int NX, NY, NZ, XP;
  long long PL;
  const uint8_t* cmap2;
  const unsigned* vox;
  const double* A0;
  double* A1;
  const double* dfo;
  const uint8_t* cm2;
};
}  // namespace

// The eight corners of the cell at lattice point (x, y, z) of an NX x NY x NZ
// grid, as a lane each: out[k] is corner k's new value, want[k] the seven-point
// update of its point (ca2p.cpp:302-338) written out, or, from plane izb on, the
// value that lies at the point; raw[k] and raw_want[k] are the index that a cell
// reads in an unfused launch and the point's own.  Values come from `seed`;
// mask > 1: masks of 0, 1 and 2.  Returns 0, or 1 if the grid cannot be
// reserved.
extern "C" int corner_check(int NX, int NY, int NZ, int izb, int x, int y, int z, int mask, unsigned seed, double* out,
                            double* want, long long* raw, long long* raw_want) {
  Grid g{};
  g.NX = NX; g.NY = NY; g.NZ = NZ;
  g.XP = (NX + 1 + 15) / 16 * 16;
  g.PL = (long long)g.XP * (NY + 1);
  const long long size = g.PL * (NZ + 1);
  Sparse<double> a0(size), a1(size);
  Sparse<uint8_t> m2(size);
  Sparse<unsigned> vox(size);
  if (!a0.p || !a1.p || !m2.p || !vox.p) return 1;
  double dfo[64];
  unsigned long long s = seed * 2654435761ull + 12345;
  auto rnd = [&] { s = s * 6364136223846793005ull + 1442695040888963407ull; return (unsigned)(s >> 33); };
  for (double& d : dfo) d = rnd() / 2147483648.0 - 0.3;
  // the point (j, k, l), written out in 64 bits
  auto at = [&](int j, int k, int l) { return (long long)l * g.PL + (long long)k * g.XP + (long long)j; };
  auto fill = [&](int j, int k, int l) {
    const long long v = at(j, k, l);
    if (a0.p[v] != 0) return;
    a0.p[v] = 0.05 + rnd() / 2147483648.0;
    a1.p[v] = 0.05 + rnd() / 2147483648.0;
    m2.p[v] = mask > 1 ? rnd() % 3 : rnd() % 2;
    vox.p[v] = (rnd() % 64) | (rnd() % 2 ? 0x80000000u : 0u);
  };
  struct Nb { int px, nx, py, ny, pz, nz; };
  auto around = [&](int j, int k, int l) {
    return Nb{(j + NX - 1) % NX, (j + 1) % NX, (k + NY - 1) % NY, (k + 1) % NY, l == 0 ? 1 : l - 1,
              l == NZ - 1 ? NZ - 1 : l + 1};
  };
  for (int k = 0; k < 8; k++) {
    const int rj = x + (k & 1), rk = y + (k >> 1 & 1), l = z + (k >> 2), j = rj % NX, kk = rk % NY;
    fill(rj, rk, l);
    fill(j, kk, l);
    if (l >= NZ) continue;
    const Nb n = around(j, kk, l);
    fill(n.px, kk, l); fill(n.nx, kk, l); fill(j, n.py, l); fill(j, n.ny, l); fill(j, kk, n.pz); fill(j, kk, n.nz);
  }
  // a plain corner's periodic copy holds the point's value, as the sub-steps leave it
  for (int k = 0; k < 8; k++) {
    const int rj = x + (k & 1), rk = y + (k >> 1 & 1), l = z + (k >> 2);
    a1.p[at(rj, rk, l)] = a1.p[at(rj % NX, rk % NY, l)];
  }
  g.cmap2 = g.cm2 = m2.p;
  g.vox = vox.p; g.A0 = a0.p; g.A1 = a1.p; g.dfo = dfo;
  const AtpK ak{0.01, 1.2, 0.0025, 0.5, 0.1};
  const double inv = 1.25;
  uint4 q[8];
  Corner c[8];
  for (int k = 0; k < 8; k++) {
    q[k] = corner_word(g, izb, x, y, z, k);
    c[k] = corner_load(g, k, q[k]);
  }
  for (int k = 0; k < 8; k++) {
    out[k] = corner_new(ak, inv, g, k, q[k], c[k], c[k ^ 1].c0, c[k ^ 2].c0, c[k ^ 4].c0);
    const int rj = x + (k & 1), rk = y + (k >> 1 & 1), l = z + (k >> 2), j = rj % NX, kk = rk % NY;
    raw[k] = corner_raw(q[k]);
    raw_want[k] = at(rj, rk, l);
    const double c0 = a0.p[at(j, kk, l)];
    if (l >= izb) {
      want[k] = a1.p[at(j, kk, l)];
      continue;
    }
    const Nb n = around(j, kk, l);
    const long long p[6] = {at(n.px, kk, l), at(n.nx, kk, l), at(j, n.py, l), at(j, n.ny, l), at(j, kk, n.pz), at(j, kk, n.nz)};
    double lap = 0;
    for (long long v : p) lap += (double)m2.p[v] * (a0.p[v] - c0);
    const unsigned w = vox.p[at(j, kk, l)];
    const double du = w & 0x7fffffffu ? dfo[(w & 0x7fffffffu) - 1] : 0.0;
    want[k] = c0 + ak.DT_Ca * (ak.Da * lap * inv * inv + ak.STIM11 * (du < 0 ? 0 : du) - c0 * ak.Kaa +
                               (w >> 31) * ak.AIR_STIM);
  }
  return 0;
}

// setup_map_lat's stamp (map.cpp:39-166) of n cells by `lanes` lanes a cell: the
// number of voxels of the cells' boxes, their periodic copies included, whose
// maps differ from the loops written out, or -1 if the grid cannot be reserved.
// Cell 0 is not looked at (an empty voxel of the sparse map reads 0).
extern "C" long long stamp_check(int NX, int NY, int NZ, double lx, double ly, double lz, int n, const double* x,
                                 const double* y, const double* z, const double* radius, const uint8_t* state, int lanes) {
  Tis t;
  std::memset(&t, 0, sizeof t);
  t.NX = NX; t.NY = NY; t.NZ = NZ;
  t.XP = (NX + 1 + 15) / 16 * 16;
  t.PL = (long long)t.XP * (NY + 1);
  t.LX = lx; t.LY = ly; t.LZ = lz;
  t.dx = lx / NX; t.dy = ly / NY; t.dz = lz / NZ;
  t.inv_dx = NX / lx; t.inv_dy = NY / ly; t.inv_dz = NZ / lz;
  t.irx = (int)(1.4 * NX / lx); t.iry = (int)(1.4 * NY / ly); t.irz = (int)(1.4 * NZ / lz);
  t.prm.FAC_MAP = 2.0;
  t.cap = n;
  Status st{};
  st.n = n;
  t.st = &st;
  Sparse<int> m1(t.PL * (NZ + 1));
  Sparse<uint8_t> m2(t.PL * (NZ + 1));
  if (!m1.p || !m2.p) return -1;
  t.cmap1 = m1.p; t.cmap2 = m2.p;
  t.pos[0][0] = const_cast<double*>(x); t.pos[0][1] = const_cast<double*>(y); t.pos[0][2] = const_cast<double*>(z);
  t.radius = const_cast<double*>(radius);
  t.state = const_cast<uint8_t*>(state);
  int* lat = new int[3 * n];
  t.lat = lat;
  blockDim.x = lanes;
  for (int l = 0; l < lanes; l++) {
    threadIdx.x = l;
    if (lanes == 16) map_stamp_part<16>(t, 0, 0, 1);
    else if (lanes == 4) map_stamp_part<4>(t, 0, 0, 1);
    else map_stamp_part<1>(t, 0, 0, 1);
  }
  long long bad = st.err != 0;
  auto wrap = [](long v, int N) { return (int)((v % N + N) % N); };
  auto diff = [](double a, double b, double L) {
    const double d = a - b;
    return d > 0.5 * L ? d - L : d <= -0.5 * L ? d + L : d;
  };
  struct Cell { int i, j, k; };
  auto lattice = [&](int c) { return Cell{wrap((long)(x[c] * t.inv_dx), NX), wrap((long)(y[c] * t.inv_dy), NY),
                                          wrap((long)(z[c] * t.inv_dz), NZ)}; };
  for (int c = 0; c < n; c++) {
    const Cell at = lattice(c);
    bad += lat[3 * c] != at.i || lat[3 * c + 1] != at.j || lat[3 * c + 2] != at.k;
    if (c == 0) continue;
    const int f = is_afm(state[c]) ? 2 : 1;
    for (int k = std::max(at.k - f * t.irz, 1); k <= std::min(at.k + f * t.irz, NZ - 1); k++)
      for (int j = at.j - f * t.iry; j <= at.j + f * t.iry; j++)
        for (int i = at.i - f * t.irx; i <= at.i + f * t.irx; i++) {
          // the owner and the mask of voxel (i, j, k) from every cell
          int own = 0, mask = 0;
          for (int o = 1; o < n; o++) {
            const bool afm = is_afm(state[o]);
            const int g = afm ? 2 : 1;
            const Cell ao = lattice(o);
            auto off = [](int a, int b, int N) { const int d = ((a - b) % N + N) % N; return d > N / 2 ? d - N : d; };
            const int ii = ao.i + off(i, ao.i, NX), jj = ao.j + off(j, ao.j, NY);
            if (std::abs(ii - ao.i) > g * t.irx || std::abs(jj - ao.j) > g * t.iry || std::abs(k - ao.k) > g * t.irz) continue;
            const double dx = diff(ii * t.dx, x[o], lx), dy = diff(jj * t.dy, y[o], ly), dz = k * t.dz - z[o];
            const double d2 = dx * dx + dy * dy + dz * dz, r = radius[o];
            if (d2 < r * r) own = o;
            if (afm && d2 < (2.0 * r) * (2.0 * r)) mask = 1;
          }
          const long long wi = wrap(i, NX), wj = wrap(j, NY);
          for (int copy = 0; copy < 4; copy++) {
            if (((copy & 1) && wi != 0) || ((copy & 2) && wj != 0)) continue;
            const long long v = (long long)k * t.PL + (wj + (copy & 2 ? NY : 0)) * (long long)t.XP + wi + (copy & 1 ? NX : 0);
            bad += m1.p[v] != own || m2.p[v] != mask;
          }
        }
  }
  delete[] lat;
  return bad;
}
