// launch.h -- host-side launchers of the kernel families (one per .hip file)
// and the optional per-kernel event timer.
#pragma once
#include <type_traits>
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

namespace epi {
struct Tis;
struct Status;
struct MechTis;

enum KernelId {
  K_FORCES, K_FORCES_LONG, K_RENEW_CELLS, K_RENEW_TAIL,
  K_INIT_SC, K_PERIODIC_FIX, K_BUCKET_INSERT, K_SWEEP,
  K_FINISH, K_ZZ_SET, K_ZZMAX, K_MAP_CLEAR, K_MAP_STAMP,
  K_EXT_STIM, K_CA_BEGIN, K_CA_VOX, K_CA_CELLS, K_ATP, K_CA_END, K_SW_RESET,
  K_RD_SNAPSHOT, K_RD_RESTORE, K_RD_PUT_GJ, K_RD_STATE, K_RD_SEED, K_RD_STEP,
  K_RD_SUMS, K_RD_OWN, K_MECH_STATE, K_MECH_SEED, K_MECH_BWD, K_MECH_SUMS, K_MECH_PLAN,
  K_CA_FUSED, K_CA_CORNERS, K_SWEEP_WAVE, K_WL, K_CA_SWAP, K_OUT_PACK, K_RENEW_ONE, K_FORCE_PACK, K_COUNT
};

// ints of a context's work-list buffer: the offsets and per-tissue iz_bound
// of the B stencil's list, the rest for the Ca solve's lists
constexpr long long WL_INTS(int ntis) { return 8LL * (ntis + 1); }

// Launch shapes that the autotuner may change (values checked by the host).
struct Tuning {
  int b_zb = 4, b_rows = 4;   // k_ext_stim: z planes per tile, 64-lane rows per block (points per tile)
  int a_zb = 4, a_rows = 4;   // k_atp: the same (a fused solve's tiles are 128 points)
  int ca_group = 8;           // Ca cell kernels: lanes per cell (8, or 16; 4 takes 8)
  int xcd = 1;                // Ca cells and ATP: XCD-contiguous workgroup order (launches of many workgroups)
  int b_xcd = 0;              // k_ext_stim: its tile list in one contiguous run per XCD
  int sweep_wave = 0;         // k_sweep: 1, one wave per cell whatever the number of cells (0: only for few)
  int side_fork = 0;          // 1: the side stream forks after the whole build
  int rd_group = 8;           // k_rd_step: lanes per cell
  int ca_fuse = 2;            // Ca solves: ATP of a sub-step and cells of the next in one launch
                              // (0 never, 1 always, 2 for solves of at most 196608 cells)
  int ca_group_small = 8;     // k_ca_cells lanes per cell in the solves that ca_fuse 2 fuses
  int map_lanes = 16;         // k_map_stamp: lanes per cell (1, 4 or 16, along x of the stamp box)
  int step_graph = 0;         // epi_step: 1 replays the renewal and build from a captured graph
};

// Event timer: when the bit of a kernel id is set, its launches carry a
// start and a stop event that the dispatch itself records
// (hipExtLaunchKernelGGL), so the elapsed time is the kernel's own duration
// without the cost of separate event packets (see host.hip).
bool prof_on(int k, bool* counted);
void prof_events(hipEvent_t* a, hipEvent_t* b);
void prof_add(int k, hipEvent_t a, hipEvent_t b, bool counted);

#define EPI_LAUNCH(kid, kernel, grid, block, shmem, stream, ...)                              \
  do {                                                                                        \
    bool cnt_ = false;                                                                        \
    if (::epi::prof_on(kid, &cnt_)) {                                                         \
      hipEvent_t a_ = nullptr, b_ = nullptr;                                                  \
      ::epi::prof_events(&a_, &b_);                                                           \
      hipExtLaunchKernelGGL(kernel, grid, block, shmem, stream, a_, b_, 0, __VA_ARGS__);      \
      ::epi::prof_add(kid, a_, b_, cnt_);                                                     \
    } else {                                                                                  \
      hipLaunchKernelGGL(kernel, grid, block, shmem, stream, __VA_ARGS__);                    \
    }                                                                                         \
  } while (0)

// f with a z chunk as a compile-time constant
template <class F>
inline void by_zb(int zb, F f) {
  switch (zb) {
    case 1: f(std::integral_constant<int, 1>()); break;
    case 2: f(std::integral_constant<int, 2>()); break;
    case 8: f(std::integral_constant<int, 8>()); break;
    case 16: f(std::integral_constant<int, 16>()); break;
    default: f(std::integral_constant<int, 4>()); break;
  }
}

// where a force kernel leaves the statuses for a waiting host (pinned,
// coherent memory; host == nullptr: nowhere): a Status per tissue, then value
// into every tissue's seq
struct StatusOut {
  Status* host = nullptr;
  unsigned long long* seq = nullptr;
  unsigned long long value = 0;
};

// where a force kernel also leaves the new positions: slot `slot` of a
// mechanics window (m == nullptr: nowhere)
struct MechSave {
  MechTis* m = nullptr;
  int slot = 0;
  bool chain = false;   // and the next force kernel's records (no build between the two)
};

// Rows of up to FORCES_ROW_CAP entries go to the cooperative kernel (whose
// LDS slots per cell, 40, 48 or 64, follow max_len), longer ones to a
// one-lane-per-cell kernel, launched only when max_len exceeds the slots.
constexpr int FORCES_ROW_CAP = 64;
void launch_forces(hipStream_t s, const Tis* dT, int ntis, int pb, int cb, int max_other, int max_len,
                   const MechSave& save = {});
// the two halves of launch_forces: the cooperative kernel for rows of up to
// the returned number of slots (chosen from max_len), and the long rows
int launch_forces_rows(hipStream_t s, const Tis* dT, int ntis, int pb, int cb, int max_other, int max_len,
                       const StatusOut& out, const MechSave& save = {});
// the records the force kernels read, where no build has just written them
void launch_force_pack(hipStream_t s, const Tis* dT, int ntis, int pb, int max_n);
void launch_forces_long(hipStream_t s, const Tis* dT, int ntis, int pb, int cb, int max_other, int cap,
                        const MechSave& save = {});
// zero_zz: also clear zzmax, for a build whose insertion takes it.  max_free:
// the most cells past membrane and dermis of any tissue.  Up to RENEW_ONE the
// renewal is one launch of a workgroup per tissue (160 cells: 9.6 us against
// 11.5 with the gap for two launches; with 2,000 cells it took 20.1 against 15,
// the lipid laws' tanh on one CU)
constexpr int RENEW_ONE = 768;
void launch_renew(hipStream_t s, const Tis* dT, int ntis, int pb, int cb, int cpar, int max_free, int zero_zz);
void launch_initialize_sc(hipStream_t s, const Tis* dT, const int* tlist, int ntis, int pb, int max_n);
void launch_periodic_fix(hipStream_t s, const Tis* dT, int ntis, int pb, int max_n);
// the bucket insertion and the rest of the build, for callers that run the
// voxel maps beside the rest.  With clear_blocks (a step), the insertion also
// applies the periodic fix, takes zzmax (cleared by launch_renew) and empties
// the voxel maps with that many more blocks
void launch_connect_insert(hipStream_t s, const Tis* dT, int ntis, int pb, int max_n, unsigned clear_blocks);
void launch_connect_rest(hipStream_t s, const Tis* dT, int ntis, int pb, int nb, int max_n, int max_swept,
                         int sweep_wave);
// the rest of the build of a step with the stamping of the voxel maps as
// further blocks of the sweep and the B stencil as further blocks of k_finish:
// up to b_tiles tiles of BUILD_FIELD_BS points per tissue
constexpr int BUILD_FIELD_BS = 128;
void launch_connect_field(hipStream_t s, const Tis* dT, int ntis, int pb, int nb, int bp, int max_n, int max_swept,
                          long long b_tiles, const Tuning& tu);
void launch_connect(hipStream_t s, const Tis* dT, int ntis, int pb, int nb, int max_n, int max_swept, int sweep_wave);
void launch_zzmax(hipStream_t s, const Tis* dT, int ntis, int pb, int max_n);
// A snapshot's output record (CellManager::output's fields): a header of
// OUT_HDR bytes whose first int is the device's cell count, then m >= n
// slots per array: the doubles radius, ageb, agek, ca2p, x, y, z, ca2p_avg,
// ex_fat, in_fat, spr_nat_len, the ints rest_div_times, pair, fix_origin and
// the bytes state, touch.  m is a multiple of 32, so every array is aligned.
constexpr int OUT_NF64 = 11, OUT_NI32 = 3, OUT_NU8 = 2;
constexpr long long OUT_HDR = 256;
constexpr long long out_record_bytes(long long m) { return OUT_HDR + m * (8 * OUT_NF64 + 4 * OUT_NI32 + OUT_NU8); }

// the output record of one tissue's first n cells into out, positions from
// buffer pb, Ca2+ from cp, lists from cb
void launch_out_pack(hipStream_t s, const Tis* dT, int tissue, int pb, int cp, int cb, int n, long long m, char* out);
// setup_map_lat: the maps emptied (map_clear_blocks blocks a tissue), then stamped
unsigned map_clear_blocks(long long max_gsize);
void launch_map_clear(hipStream_t s, const Tis* dT, int ntis, long long max_gsize);
void launch_map_stamp(hipStream_t s, const Tis* dT, int ntis, int pb, int max_n, const Tuning& tu);
// the B stencil over a work list of (tissue, tile) built on the device from
// zzmax (d_wl: 2 ntis + 1 ints); tiles_est sizes the grid (any value covers
// the list: the blocks walk it grid-stride)
// k_ext_stim over a list that is in d_wl already: ntis + 1 offsets, ntis iz_bounds
void launch_ext_stim_list(hipStream_t s, const Tis* dT, int ntis, int bp, long long tiles_est, const int* d_wl,
                          const Tuning& tu);
void launch_ext_stim(hipStream_t s, const Tis* dT, int ntis, int bp, long long tiles_est, int* d_wl,
                     const Tuning& tu);
// a solve's or window's set-up: packed entries, pairs, laws' constants (and
// ca2p_avg cleared with zero_avg), voxel words, corners.  launch_ca_corners
// alone renews what depends on B (buffer bp)
void launch_ca_begin(hipStream_t s, const Tis* dT, const int* tlist, int ntis, int cb, int bp, int max_n,
                     long long max_plane, int max_izb, int zero_avg);
void launch_ca_corners(hipStream_t s, const Tis* dT, const int* tlist, int ntis, int bp, int max_n);
struct RdTis;
// A Ca solve's work, flattened over its tissues (built on the host once per
// solve, device pointers): blocks of the cell kernels map to (tissue, block
// of that tissue, blocks of that tissue) through cmap (ncb entries); the ATP
// grid is a list of tiles of `abs` plane points by a_zb planes, aoff[i]
// being the first tile of the list's i-th tissue (aoff[ntis] = atiles), with
// its iz_bound aizb[i] and tissue id atis[i].
// A list of one tissue (a single-tissue solve) also carries that tissue id
// and iz_bound by value (t0, izb0): the kernels then read no list memory.
struct CaList {
  const int* aoff;
  const int* aizb;
  const int* atis;
  const int4* cmap;
  int ntis, ncb, atiles, abs;
  int t0, izb0;
  const Tis* h0;   // host: that tissue's descriptor, passed to the kernels by value
  unsigned mg_npt; // its tiles per plane, for div_by
  bool wide;       // a plane of some tissue is past 32-bit byte offsets
};
// points per ATP tile of a solve: the fused kernel's block, or the ATP
// kernel's 64 a_rows
int ca_list_bs(const Tuning& tu, bool fused);
// lanes per cell that a CA_GROUP value asks for (8 serves 4 too: a cell's
// eight corners take eight lanes)
constexpr int ca_lanes(int ca_group) { return ca_group <= 8 ? 8 : 16; }
// n_sub sub-steps (fused when tu.ca_fuse), flipping cp and ap after each.
// sv: a reaction-diffusion window's reverse-pass storage; the cells then also
// save the state before each sub-step into segment slots slot, slot + 1, ...;
// last_cells_only skips the ATP update of the last one
void launch_ca_substeps(hipStream_t s, const Tis* dT, const CaList& cl, int& cp, int& ap, int n_sub, const Tuning& tu,
                        const RdTis* sv = nullptr, int slot = 0, bool last_cells_only = false);
// packed gj and pairs back into the cells' arrays (CA_END_PUT), with diff_u
// cleared (CA_END_SUBSTEP), and the rest of a solve's end (CA_END_SOLVE)
enum { CA_END_PUT = 0, CA_END_SUBSTEP = 1, CA_END_SOLVE = 2 };
void launch_ca_end(hipStream_t s, const Tis* dT, const int* tlist, int ntis, int cb, int max_n, int what);
// the listed tissues' two Ca, IP3 and ATP buffers trade contents (after a
// solve of part of a context with an odd sub-step count, whose buffer
// parities are shared by every tissue)
void launch_ca_swap(hipStream_t s, const Tis* dT, const int* tlist, int ntis, int max_n, long long max_gsize);
// frozen reaction-diffusion window (k_adjoint.hip)
void launch_rd_snapshot(hipStream_t s, const Tis* dT, RdTis* dR, int ntis, int cb, int cp, int ap, long long items);
void launch_rd_own(hipStream_t s, const Tis* dT, RdTis* dR, int ntis, int max_n);
void launch_rd_restore(hipStream_t s, const Tis* dT, RdTis* dR, const double* gj0, int ntis, int cb, int cp, int ap,
                       int use_kpa, long long items);
void launch_rd_put_gj(hipStream_t s, const Tis* dT, RdTis* dR, int ntis, int cb, long long items);
void launch_rd_state(hipStream_t s, const Tis* dT, RdTis* dR, int ntis, int slot, int save, int cp, int ap,
                     long long items);
void launch_rd_seed(hipStream_t s, const Tis* dT, RdTis* dR, int ntis, int cp, int q, long long items);
void launch_rd_backward_substep(hipStream_t s, const Tis* dT, RdTis* dR, int ntis, int slot, int q, int qa, int max_n,
                                long long max_box, int rg);
// frozen mechanics window (k_mech.hip)
void launch_mech_state(hipStream_t s, const Tis* dT, const MechTis* dM, int ntis, int slot, int dir, int pb,
                       int max_n);
// blocks of a reverse step, each with four words of MechTis::part
int mech_bwd_blocks(int max_memb, int max_other);
void launch_mech_seed(hipStream_t s, const Tis* dT, MechTis* dM, int ntis, int pb, int q, int max_n, int nblk);
void launch_mech_backward_step(hipStream_t s, const Tis* dT, MechTis* dM, int ntis, int slot, int q, int max_memb,
                               int max_other);
void launch_mech_plan(hipStream_t s, const Tis* dT, MechTis* dM, int ntis, int pb, int cb, int max_n);
void launch_mech_sums(hipStream_t s, MechTis* dM, int ntis, int nblk);
void launch_rd_sums(hipStream_t s, const Tis* dT, RdTis* dR, int ntis, int q, long long items);
}  // namespace epi
