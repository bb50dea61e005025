"""What a mechanics window holds on the device: positions and targets from its
opening (72 bytes a cell of capacity), the adjoints, states and plan only from its
first gradient on and sized by the longest list, and nothing after its end."""
import ctypes as C

import numpy as np
import pytest

from epi_amd import configs

pytestmark = pytest.mark.gpu

MIB = 1 << 20
CAP = 400_000   # cells of capacity: the window's arrays stand out from the allocator's granularity


def free_bytes(native):
    a, b = C.c_size_t(), C.c_size_t()
    assert native.load_library().hipMemGetInfo(C.byref(a), C.byref(b)) == 0   # found through its own HIP runtime
    return a.value


def test_memory_of_a_window():
    from epi_amd import native
    spec = configs.config_tiny(7, 160)
    spec["geometry"].max_cells = CAP
    t = native.Tissue(spec["geometry"])
    t.load(spec)
    longest = t.status().maxlen
    # a first window of its own: the runtime loads kernels and takes their scratch at first launches
    warm = native.Tissue(configs.config_tiny(7, 160)["geometry"])
    warm.load(configs.config_tiny(7, 160))
    warm.set.mech_begin()
    warm.set.mech_adjoint([{}], 4, 2, [warm.set.mech_get_positions(0)])
    warm.close()
    before = free_bytes(native)
    t.set.mech_begin()
    opened = before - free_bytes(native)
    t.set.mech_forward([{}], 4)
    assert before - free_bytes(native) == opened
    assert opened <= 72 * CAP + 8 * MIB
    x = t.set.mech_get_positions(0)
    for every in (2, 2):
        t.set.mech_adjoint([{}], 4, every, [x + 0.01])
    with_grad = before - free_bytes(native)
    # two states of a segment, two checkpoints, three adjoints; a plan slot is an index and a code
    assert with_grad <= opened + ((2 + 2 + 3) * 24 + 5 * (2 * longest + 8) + 4) * CAP + 8 * MIB
    t.set.mech_end()
    assert before - free_bytes(native) <= 8 * MIB
    t.close()
