"""When the node clusters' plan is made: by a disc's first Jacobian that takes
it.  Creating a mechanics, residuals, functionals, features and FP32-tangent
Jacobians must not pay for it (seen in the device memory they take); a first
Jacobian through the entry point that allocates nothing settles the disc on the
element pass and gather, so that later Jacobians keep its bits.

Bounds: the plan of these boxes takes more than 8 MiB (16 bytes for each of a
lane per pair, 28 and 7 pairs a node); what else the calls allocate is named
where it is measured, and the device's pool rounds up by 2 MiB an allocation."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from tests.helpers import MATS, RTOL, mat_row, oracle_mesh_from, random_state, rel

pytestmark = pytest.mark.gpu

g = pytest.importorskip("goal_amd")

g.lib.goal_asm_jacobian_noalloc.restype = C.c_int
g.lib.goal_asm_jacobian_noalloc.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int]


def used():
    """Device memory in use, bytes (the HIP runtime is a dependency of the library)."""
    g.sync()
    free, total = C.c_size_t(), C.c_size_t()
    assert g.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return total.value - free.value


def make(order, model, dims):
    disc = g.Disc.box(*dims, order=order, jitter=0.1, seed=3)
    disc.set_soln(random_state(disc.num_nodes, 4, scale_u=0.001))
    st = g.States(disc, model, order)
    return disc, st, lambda: g.Mechanics(disc, st, [g.MaterialSpec(**MATS[model])], quad_order=order)


@pytest.mark.parametrize("order,model,dims", [(2, 1, (24, 24, 24)), (1, 1, (48, 48, 48))])
def test_plan_is_not_made_for_other_calls(order, model, dims):
    disc, st, mechanics = make(order, model, dims)
    si = g.SolInfo(disc)
    si.zero_all()
    si.norm_R()
    npe, ne, nn = 4 if order == 1 else 10, disc.num_elems, disc.num_nodes
    before = used()
    mech = mechanics()
    assert used() - before < 8 * ne + (4 << 20)  # a value per element
    feat = g.learn_features(mech, 0.25)
    mech.residual(si)
    mech.qoi(g.QOI_AVG_VM, si)
    # element residuals, the features and their scratch
    assert used() - before < 8 * ne + 8 * 4 * npe * ne + (8 * 12 + 4 * 12) * ne + 8 * 10 * nn + (12 << 20)
    del feat
    before = used()
    mech.set_option("tangent", 32)
    mech.jacobian(si)
    assert used() - before < 8 * (4 * npe) ** 2 * ne + (4 << 20)  # element matrices
    before = used()
    mech.set_option("tangent", 64)
    mech.jacobian(si)
    assert used() - before > 8 << 20  # the plan


@pytest.mark.parametrize("order,model", [(1, 1), (1, 2), (2, 1)])
def test_first_jacobian_without_allocation(order, model):
    disc, st, mechanics = make(order, model, (5, 4, 3))
    mech = mechanics()
    si = g.SolInfo(disc)
    om = oracle_mesh_from(disc)
    ost = O.States(om, model, order)
    Ro, Vo = O.assemble(O.K_JACOBIAN, om, model, [mat_row(MATS[model])], disc.soln(), ost, quad_order=order)
    runs = []
    for noalloc in (True, True, False, True):
        si.zero_all()
        if noalloc:
            g.check(g.lib.goal_asm_jacobian_noalloc(mech.h, si.h, 0, 1))
        else:
            mech.jacobian(si)
        runs.append((si.R(), si.vals()))
        assert rel(runs[-1][0], Ro) < RTOL and rel(runs[-1][1], Vo) < RTOL
    for R, V in runs[1:]:
        assert np.array_equal(R, runs[0][0]) and np.array_equal(V, runs[0][1])
