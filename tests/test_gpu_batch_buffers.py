"""A captured batch keeps its buffers: assemblies of another kind on the same
mechanics (FP32 tangent, adjoint, residual, functional) after the capture leave
the memory that the replays write to alone.  Buffers of the linear elements'
point states' size, allocated after those assemblies, stand where a buffer
given up by one of them would be: the replays must not write to them.

Tolerance: none, every replay gives the first one's bits."""
import numpy as np
import pytest

from tests.helpers import MATS, random_history, random_state

pytestmark = pytest.mark.gpu

g = pytest.importorskip("goal_amd")

STATE = 32  # doubles per linear element


@pytest.mark.parametrize("order,model", [(1, 2), (1, 1), (2, 1)])
def test_replays_after_other_assemblies(order, model):
    disc = g.Disc.box(*((12, 6, 6) if order == 1 else (4, 3, 3)), order=order, jitter=0.1, seed=3)
    st = g.States(disc, model, order)
    mech = g.Mechanics(disc, st, [g.MaterialSpec(**MATS[model])], quad_order=order)
    disc.set_soln(random_state(disc.num_nodes, 4, scale_u=0.002))
    if model == 2:
        Fp, eq = random_history(disc.num_elems * st.nq, 5)
        for k, v in (("Fp_old", Fp), ("eqps_old", eq), ("Fp", Fp), ("eqps", eq)):
            st.set(k, v)
    si, other = g.SolInfo(disc), g.SolInfo(disc)
    b = g.Batch([mech], [si])
    b.capture()
    b.run()
    g.sync()
    R, V = si.R(), si.vals()
    assert np.isfinite(R).all() and np.isfinite(V).all() and V.any()
    for tangent in (32, 64):
        mech.set_option("tangent", tangent)
        for adjoint in (False, True):
            other.zero_all()
            mech.jacobian(other, adjoint=adjoint, save_states=False)
        mech.residual(other, save_states=False)
        mech.qoi(g.QOI_AVG_VM, other)
        standins = [g.DeviceArray(STATE * disc.num_elems) for _ in range(4)]
        for s in standins:
            s.fill(7.0)
        for _ in range(3):
            si.set(R=np.full(disc.num_dofs, 3.0), vals=np.full(disc.nnz, 5.0))
            b.run()
            g.sync()
            assert np.array_equal(si.R(), R) and np.array_equal(si.vals(), V), tangent
        for s in standins:
            assert (s.numpy() == 7.0).all(), tangent
