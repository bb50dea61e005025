// noalloc.hip -- calc_ext_stim (ext_stim.cpp:18-69) over caller-held device
// grids, allocating nothing: epi_calc_ext_stim_noalloc (include/epi_amd.h).
//
// The context path keeps its grid descriptors (Tis), per-tissue status and
// the B stencil's tile work list in memory the library allocates.  Here they
// live in one static device array, `scratch`, of a fixed size per GPU: a
// first kernel writes one descriptor per caller view, the tile list and the
// caller's codes, then the context path's own k_ext_stim runs on them.  The array's device address
// is looked up once per device (hipGetSymbolAddress) and that address, not
// the symbol, is what host code hands to kernels.
#include <mutex>

#include "epi_dev.h"
#include "launch.h"
#include "field_step.h"
#include "../../include/epi_amd.h"

namespace epi {
namespace {

constexpr size_t al256(size_t v) { return (v + 255) / 256 * 256; }
constexpr int NA_MAX = EPI_NOALLOC_MAX_GRIDS;
constexpr size_t NA_TIS = al256(sizeof(Tis) * NA_MAX);         // descriptors
constexpr size_t NA_WL = al256(sizeof(int) * (2 * NA_MAX + 1));  // tile list: offsets, iz_bound
constexpr size_t NA_BYTES = NA_TIS + NA_WL;

}  // namespace
}  // namespace epi

// Scratch of epi_calc_ext_stim_noalloc: every call on a GPU shares that GPU's
// copy, which keeps the last call's contents; each call rewrites what it
// reads (descriptors, list) before reading it.
static __device__ __align__(256) unsigned char scratch[epi::NA_BYTES];

namespace epi {
namespace {

constexpr int NA_DEVICES = 64;
std::mutex g_na_mu;
unsigned char* g_na_ptr[NA_DEVICES] = {};

// the current device's address of `scratch`, looked up on the first call per
// device with that device current
int na_scratch(unsigned char** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NA_DEVICES) return EPI_ERR_HIP;
  std::lock_guard<std::mutex> lk(g_na_mu);
  if (!g_na_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return EPI_ERR_HIP;
    g_na_ptr[dev] = static_cast<unsigned char*>(p);
  }
  *out = g_na_ptr[dev];
  return EPI_OK;
}

// One block: per view the descriptor fields that k_ext_stim reads (the same
// expressions as epi_create's for dz and inv_dz), with epi5_MT's parameters,
// its tiles in the list and its code.  The parameter records are written by
// the whole block, a word a thread.  (A thread a view writing whole records,
// k_wl_b after it and a launch to copy the codes took 14.3 us of a call's 42
// with their gaps; this 3.5.)
__global__ void __launch_bounds__(1024) k_na_setup(const epi_bfield_view* __restrict__ views, int n, Tis* __restrict__ T,
                                                   int bs, int zb, int* __restrict__ off, int* __restrict__ izb_out,
                                                   int32_t* __restrict__ err, const Params prm) {
  static_assert(sizeof(Params) % 8 == 0, "the parameters are copied in 8-byte words");
  constexpr int W = sizeof(Params) / 8;
  __shared__ unsigned long long s_prm[W];
  if (threadIdx.x < W) s_prm[threadIdx.x] = reinterpret_cast<const unsigned long long*>(&prm)[threadIdx.x];
  const double margin = prm.iz_margin;
  int carry = 0;
  for (int base = 0; base < n; base += blockDim.x) {
    const int i = base + threadIdx.x;
    int cnt = 0;
    if (i < n) {
      const epi_bfield_view v = views[i];
      Tis& t = T[i];
      t.NX = v.nx; t.NY = v.ny; t.NZ = v.nz; t.XP = v.xp;
      t.PL = v.pl;
      t.inv_dz = v.nz / v.lz;
      t.bf[0] = const_cast<double*>(v.b_in);
      t.bf[1] = v.b_out;
      t.cmap1 = const_cast<int*>(v.cmap1);
      t.cmap2 = const_cast<uint8_t*>(v.cmap2);
      t.state = const_cast<uint8_t*>(v.state);
      t.agek = const_cast<double*>(v.agek);
      int izb = (int)((v.zzmax + margin) * (v.nz / v.lz));   // b_iz_bound
      const bool out = izb > v.nz || izb < 0;
      if (out) izb = 0;
      err[i] = out ? ERR_OUT_OF_GRID : OK;
      izb_out[i] = izb;
      cnt = ((v.nx * v.ny + bs - 1) / bs) * ((izb + zb - 1) / zb);
    }
    int tot;
    const int ex = block_exclusive_scan(cnt, &tot);
    if (i < n) off[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) off[n] = carry;
  __syncthreads();
  for (int k = threadIdx.x; k < n * W; k += blockDim.x)
    reinterpret_cast<unsigned long long*>(&T[k / W].prm)[k % W] = s_prm[k % W];
}

}  // namespace
}  // namespace epi

extern "C" int64_t epi_noalloc_scratch_bytes(void) { return (int64_t)epi::NA_BYTES; }

extern "C" int epi_calc_ext_stim_noalloc(const epi_bfield_view* views, int32_t ngrids, int32_t* err, void* stream) {
  using namespace epi;
  if (!views || !err || ngrids < 1 || ngrids > NA_MAX) return EPI_ERR_INVALID;
  unsigned char* base = nullptr;
  const int rc = na_scratch(&base);
  if (rc != EPI_OK) return rc;
  Tis* T = reinterpret_cast<Tis*>(base);
  int* wl = reinterpret_cast<int*>(base + NA_TIS);
  hipStream_t s = static_cast<hipStream_t>(stream);
  static const Params prm = [] {
    epi_params d;
    epi_params_default(&d);
    Params p;
    derive_params(d, p);
    return p;
  }();
  const Tuning tu{};
  hipLaunchKernelGGL(k_na_setup, dim3(1), dim3(ngrids <= 256 ? 256 : 1024), 0, s, views, ngrids, T, 64 * tu.b_rows, tu.b_zb,
                     wl, wl + ngrids + 1, err, prm);
  // the grid sizes are in device memory: the blocks walk the list grid-stride
  // from a grid sized for 256 tiles per view
  launch_ext_stim_list(s, T, ngrids, 0, 256LL * ngrids, wl, tu);
  return hipGetLastError() == hipSuccess ? EPI_OK : EPI_ERR_HIP;
}
