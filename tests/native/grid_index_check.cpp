// Host build of the grid index arithmetic of the Ca corners
// (epi_amd/csrc/ca_corner.h), for tests/test_grid_indices.py.  The grids are sparse: a
// reservation of address space whose pages exist once written, so that grids
// far larger than the memory of this machine can be addressed.
#include <algorithm>
#include <sys/mman.h>

#include "device_on_host.h"
#include "../../epi_amd/csrc/ca_corner.h"

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
