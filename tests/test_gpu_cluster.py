"""The one-kernel assembly of neo-Hookean quadratic tets (four points, FP64)
against the oracle where its plan can go wrong: a node with more elements than
one chunk holds, ragged and renumbered meshes, the smallest mesh, several
element sets, sums added to earlier ones, and the meshes that it leaves to the
element pass and gather (a node without elements).

Tolerance: RTOL of the parity tests (1e-11 normwise, FP64 on both sides)."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import NH, RTOL, fan_mesh, mat_row, random_state, rel

pytestmark = pytest.mark.gpu

g = pytest.importorskip("goal_amd")


def mesh(kind):
    if kind.startswith("fan"):  # 80 or 320 tets around one node
        return fan_mesh(order=2, subdiv=1 if kind == "fan80" else 2, jitter=0.05, seed=3)
    dims = dict(cell=(1, 1, 1), ragged=(5, 1, 3), renumbered=(4, 3, 2), bare=(2, 2, 1))[kind]
    X, conn = g.mesh_box(*dims, order=2, jitter=0.1, seed=7)
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
@pytest.mark.parametrize("kind", ["cell", "ragged", "renumbered", "fan80", "fan320", "bare"])
def test_one_kernel_assembly_matches_oracle(kind, adjoint):
    X, conn = mesh(kind)
    sets = (np.arange(conn.shape[0]) % 2).astype(np.int32)
    disc = g.Disc.from_arrays(2, X, conn, sets)
    disc.set_elem_sets(2, sets)
    st = g.States(disc, 1, 2)
    mats = [dict(NH), dict(NH, E=700.0, nu=0.3, c0=0.5)]
    mech = g.Mechanics(disc, st, [g.MaterialSpec(**m) for m in mats], quad_order=2)
    x = random_state(X.shape[0], 4)
    disc.set_soln(x)
    om = O.Mesh(2, X, conn, sets)
    ost = O.States(om, 1, 2)
    K = O.K_ADJOINT if adjoint else O.K_JACOBIAN
    Ro, Vo = O.assemble(K, om, 1, [mat_row(m) for m in mats], x, ost, quad_order=2)
    si = g.SolInfo(disc)
    si.zero_all()
    mech.jacobian(si, adjoint=adjoint)
    R, V = si.R(), si.vals()
    assert rel(R, Ro) < RTOL and rel(V, Vo) < RTOL
    assert rel(st.get("sigma"), ost.sigma) < RTOL
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
    Ro, Vo = O.assemble(K, om, 1, [mat_row(m) for m in mats], x, ost, quad_order=2, stabilization=False, save=False)
    assert rel(si.R(), Ro) < RTOL and rel(si.vals(), Vo) < RTOL
