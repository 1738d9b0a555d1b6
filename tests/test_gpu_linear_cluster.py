"""Linear tets' Jacobians over node clusters (one point, neo-Hookean and J2,
FP64) against the oracle where the plan can go wrong: one cell, several runs
with a ragged end, a renumbered mesh, a node whose elements fill most of a run,
and the meshes left to the element pass and gather (a node with more elements
than a run holds, a node without elements); several element sets, sums added
to earlier ones, and grids smaller than the runs.

Tolerance: RTOL of the parity tests (1e-11 normwise, FP64 on both sides)."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import MATS, RTOL, fan_mesh, mat_row, random_history, random_state, rel

pytestmark = pytest.mark.gpu

g = pytest.importorskip("goal_amd")


def mesh(kind):
    if kind.startswith("fan"):  # 80 or 320 tets around one node
        return fan_mesh(order=1, subdiv=1 if kind == "fan80" else 2, jitter=0.05, seed=3)
    dims = dict(cell=(1, 1, 1), ragged=(9, 2, 3), renumbered=(5, 4, 6), bare=(2, 2, 1))[kind]
    X, conn = g.mesh_box(*dims, order=1, jitter=0.1, seed=7)
    if kind == "renumbered":
        p = np.random.default_rng(5).permutation(X.shape[0]).astype(np.int32)
        Y = np.empty_like(X)
        Y[p] = X
        conn = p[conn][np.random.default_rng(6).permutation(conn.shape[0])]
        X = Y
    if kind == "bare":
        X = np.vstack([X, [[2.0, 2.0, 2.0]]])
    return X, np.ascontiguousarray(conn)


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("model", [1, 2])
@pytest.mark.parametrize("kind", ["cell", "ragged", "renumbered", "fan80", "fan320", "bare"])
def test_linear_clusters_match_oracle(kind, model, adjoint):
    X, conn = mesh(kind)
    ne = conn.shape[0]
    sets = (np.arange(ne) % 2).astype(np.int32)
    mats = [dict(MATS[model]), dict(MATS[model], E=700.0, nu=0.3, c0=0.5)]
    x = random_state(X.shape[0], 4, scale_u=0.005)
    om = O.Mesh(1, X, conn, sets)
    K = O.K_ADJOINT if adjoint else O.K_JACOBIAN
    disc = g.Disc.from_arrays(1, X, conn, sets)
    disc.set_elem_sets(2, sets)
    disc.set_soln(x)
    st, ost = g.States(disc, model, 1), O.States(om, model, 1)
    mech = g.Mechanics(disc, st, [g.MaterialSpec(**m) for m in mats], quad_order=1)
    if model == 2:
        Fp, eq = random_history(ne, 9)
        for f, v in (("Fp_old", Fp), ("Fp", Fp), ("eqps_old", eq), ("eqps", eq)):
            getattr(ost, f)[:] = v
            st.set(f, v)
    rows = [mat_row(m) for m in mats]
    Ro, Vo = O.assemble(K, om, model, rows, x, ost, quad_order=1)
    si = g.SolInfo(disc)
    si.zero_all()
    mech.jacobian(si, adjoint=adjoint)
    R, V = si.R(), si.vals()
    assert rel(R, Ro) < RTOL and rel(V, Vo) < RTOL
    for f in ("sigma",) + (("Fp", "eqps") if model == 2 else ()):
        assert rel(st.get(f), getattr(ost, f)) < RTOL
    mech.jacobian(si, adjoint=adjoint)  # added to what is there
    assert rel(si.R(), 2 * Ro) < RTOL and rel(si.vals(), 2 * Vo) < RTOL
    mech.qoi(g.QOI_AVG_DISP, si)
    dm = si.dMdu()
    mech.jacobian(si, adjoint=adjoint)
    assert dm.any() and np.array_equal(si.dMdu(), dm)  # no clear is pending
    si.zero_all()
    mech.jacobian(si, adjoint=adjoint)
    assert not si.dMdu().any()
    for blocks in (1, 8, 40):  # grids smaller than the runs, with and without the XCD slabs
        mech.set_option("blocks", blocks)
        si.zero_all()
        mech.jacobian(si, adjoint=adjoint)
        assert np.array_equal(si.R(), R) and np.array_equal(si.vals(), V)
    mech.set_option("blocks", 0)
    mech.set_option("stabilization", 0)
    si.zero_all()
    mech.jacobian(si, adjoint=adjoint, save_states=False)
    Ro, Vo = O.assemble(K, om, model, rows, x, ost, quad_order=1, stabilization=False, save=False)
    assert rel(si.R(), Ro) < RTOL and rel(si.vals(), Vo) < RTOL
