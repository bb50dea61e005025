// mech_dev.h -- device record of the frozen mechanics window and its
// adjoint (k_mech.hip, host.hip).
//
// A window is cell_interaction + pos_copy (cell_interaction.cpp:648-685,
// cellmanager.cpp:19-26) run n_steps times from a snapshot of the positions,
// with lists, states, pairs and dermis frozen, without the periodic fix, and
// with eps_m, K_TOTAL, Kspring and KBEND (Tis::m_*) as runtime values.
#pragma once
#include "epi_dev.h"

namespace epi {

// the fewest slots of a plan row: lanes ask for a row's first slots before they
// know its length
constexpr int MECH_ROW_MIN = 16;

struct MechTis {
  GPtr<double> x0[2];      // snapshot of both position buffers, [0] = current
  GPtr<double> slot;       // positions of the states of one segment (slot-major, 3 * cap each)
  GPtr<double> ck;         // checkpoints (3 * cap each)
  // position adjoints (3 * cap each) in three rotating buffers: [q] after the
  // step, [q + 1] before it, [q + 2] cleared for the next, q = step mod 3
  GPtr<double> lam[3];
  // the interactions each cell takes part in, es slots a cell: the other cell
  // and the law's code (k_mech_plan).  lam, the plan and part are a gradient's
  // alone and lie in its work memory
  GPtr<int> ent;
  GPtr<uint8_t> code;
  GPtr<int> ent_n;
  int es;
  GPtr<double> part;       // four parameter sums per block of the reverse kernel
  GPtr<double> target;     // 3 * cap: x, y, z
  GPtr<double> scal;       // [0] loss, [1] dL/deps, [2] dL/dK_TOTAL, [3] dL/dKspring, [4] dL/dKBEND
};

}  // namespace epi
