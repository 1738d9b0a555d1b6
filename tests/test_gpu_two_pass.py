"""The element pass and gather of the kinds that node clusters took over, FP64
neo-Hookean (quadratic, four points; linear, one) and one-point linear J2, on
meshes that the clusters refuse (one node without elements): in chunks with the
gathers beside them against one pass, and on enough elements that workgroups
walk several groups, against the oracle.

Tolerance: none for chunks (the same kernels over disjoint work), RTOL of the
parity tests (1e-11 normwise, FP64 on both sides) for the oracle."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import MATS, RTOL, mat_row, random_history, random_state, rel

pytestmark = pytest.mark.gpu

g = pytest.importorskip("goal_amd")


def refused(order, model, dims):
    X, conn = g.mesh_box(*dims, order=order, jitter=0.1, seed=7)
    X = np.vstack([X, [[2.0, 2.0, 2.0]]])
    sets = np.zeros(conn.shape[0], dtype=np.int32)
    disc = g.Disc.from_arrays(order, X, conn, sets)
    st = g.States(disc, model, order)
    mech = g.Mechanics(disc, st, [g.MaterialSpec(**MATS[model])], quad_order=order)
    h = 1.0 / max(dims)  # no element turns inside out
    x = random_state(X.shape[0], 4, scale_u=0.02 * h)
    disc.set_soln(x)
    om = O.Mesh(order, X, conn, sets)
    ost = O.States(om, model, order)
    if model == 2:
        Fp, eq = random_history(conn.shape[0] * st.nq, 9)
        for f, v in (("Fp_old", Fp), ("Fp", Fp), ("eqps_old", eq), ("eqps", eq)):
            getattr(ost, f)[:] = v
            st.set(f, v)
    return disc, st, mech, x, om, ost


@pytest.mark.parametrize("order,dims", [(2, (4, 4, 4)), (2, (9, 5, 7)), (1, (7, 7, 7)), (1, (16, 9, 11))])
def test_chunks_equal_one_pass(order, dims):
    disc, st, mech, x, om, ost = refused(order, 1, dims)
    si = g.SolInfo(disc)
    mech.set_option("overlap", 0)
    ref = {}
    for adjoint in (False, True):
        si.zero_all()
        mech.jacobian(si, adjoint=adjoint)
        ref[adjoint] = si.R(), si.vals()
        assert np.isfinite(ref[adjoint][0]).all() and ref[adjoint][1].any()
    for chunks, blocks in ((2, 0), (5, 0), (8, 16)):
        mech.set_option("overlap", chunks)
        mech.set_option("overlap_blocks", blocks)
        for adjoint in (False, True):
            si.set(R=np.full(disc.num_dofs, 3.0), vals=np.full(disc.nnz, 2.0))
            si.zero_all()
            mech.jacobian(si, adjoint=adjoint)
            assert np.array_equal(si.R(), ref[adjoint][0]), (chunks, adjoint)
            assert np.array_equal(si.vals(), ref[adjoint][1]), (chunks, adjoint)


@pytest.mark.parametrize("order,model,dims", [(2, 1, (16, 16, 16)), (1, 1, (28, 26, 24)), (1, 2, (28, 26, 24))])
def test_many_groups_match_oracle(order, model, dims):
    disc, st, mech, x, om, ost = refused(order, model, dims)
    si = g.SolInfo(disc)
    si.zero_all()
    mech.jacobian(si)
    Ro, Vo = O.assemble(O.K_JACOBIAN, om, model, [mat_row(MATS[model])], x, ost, quad_order=order)
    assert np.isfinite(Ro).all() and np.isfinite(Vo).all()
    assert rel(si.R(), Ro) < RTOL and rel(si.vals(), Vo) < RTOL
    for f in ("sigma",) + (("Fp", "eqps") if model == 2 else ()):
        assert rel(st.get(f), getattr(ost, f)) < RTOL
