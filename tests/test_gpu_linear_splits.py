"""Linear tets over node clusters where a group of eight vertices has to be split
into two, four and eight runs, and where a vertex' pairs take 32 and 64 lanes (49
to 96 and 97 to 160 elements), against the oracle.

The meshes are fans of n tets around a centre, many of them with their centres
together, so that groups of eight centres follow each other on the Morton curve:
they hold 8 n elements, and a run takes 160.  runs_per_group() restates how the
groups are cut, from the node order and the limits of a run.

Tolerance: RTOL of the parity tests (1e-11 normwise, FP64 on both sides)."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import MATS, RTOL, fan_mesh, mat_row, random_history, random_state, rel

g = pytest.importorskip("goal_amd")

FANS = [(20, 1), (40, 2), (80, 4), (97, 8), (160, 8)]  # tets of a fan, runs of a group of eight centres


def fans(n, copies=20):
    """`copies` fans of n tets, their centres within a thousandth of each other."""
    X, conn = fan_mesh(order=1, subdiv=0 if n == 20 else 2, jitter=0.02, seed=3)
    conn = conn[:n]
    used = np.unique(conn)
    conn, X = np.searchsorted(used, conn).astype(np.int32), X[used]  # the centre stays node 0
    rng = np.random.default_rng(5)
    Xs = [X + 1e-3 * rng.uniform(-1, 1, 3) for _ in range(copies)]
    return np.vstack(Xs), np.vstack([conn + k * X.shape[0] for k in range(copies)]).astype(np.int32)


def runs_per_group(X, conn):
    lo = X.min(axis=0)
    cell = np.clip((X - lo) * (1024.0 / (X.max(axis=0) - lo).max()), 0.0, 1023.0).astype(np.int64)
    code = sum(((cell[:, c, None] >> np.arange(10) & 1) << (3 * np.arange(10) + c)).sum(axis=1) for c in range(3))
    order = np.argsort(code, kind="stable")
    elems = [set() for _ in range(X.shape[0])]
    near = [set() for _ in range(X.shape[0])]
    for e, row in enumerate(conn.tolist()):
        for a in row:
            elems[a].add(e)
            near[a].update(row)
    out = []
    for i in range(0, len(order), 8):
        group = order[i:i + 8]
        for p in (1, 2, 4, 8):
            parts = [group[k:k + 8 // p] for k in range(0, len(group), 8 // p)]
            if all(len(set().union(*(elems[a] for a in q))) <= 160 and sum(len(near[a]) for a in q) <= 512
                   for q in parts):
                out.append((p, sum(a % (X.shape[0] // 20) == 0 for a in group)))
                break
        else:
            out.append((0, 0))
    return out


@pytest.mark.parametrize("n,runs", FANS)
def test_groups_are_cut_as_meant(n, runs):
    cut = runs_per_group(*fans(n))
    assert (runs, 8) in cut and all(p > 0 for p, _ in cut)


@pytest.mark.gpu
@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("model", [1, 2])
@pytest.mark.parametrize("n", [n for n, _ in FANS])
def test_split_groups_match_oracle(n, model, adjoint):
    X, conn = fans(n)
    ne = conn.shape[0]
    sets = np.zeros(ne, dtype=np.int32)
    disc = g.Disc.from_arrays(1, X, conn, sets)
    x = random_state(X.shape[0], 4, scale_u=0.002)
    disc.set_soln(x)
    st = g.States(disc, model, 1)
    mech = g.Mechanics(disc, st, [g.MaterialSpec(**MATS[model])], quad_order=1)
    om = O.Mesh(1, X, conn, sets)
    ost = O.States(om, model, 1)
    if model == 2:
        Fp, eq = random_history(ne, 9)
        for f, v in (("Fp_old", Fp), ("Fp", Fp), ("eqps_old", eq), ("eqps", eq)):
            getattr(ost, f)[:] = v
            st.set(f, v)
    Ro, Vo = O.assemble(O.K_ADJOINT if adjoint else O.K_JACOBIAN, om, model, [mat_row(MATS[model])], x, ost,
                        quad_order=1)
    assert np.isfinite(Ro).all() and np.isfinite(Vo).all()
    si = g.SolInfo(disc)
    for _ in range(2):
        si.set(R=np.full(disc.num_dofs, 3.0), vals=np.full(disc.nnz, 2.0))
        si.zero_all()
        mech.jacobian(si, adjoint=adjoint)
        assert rel(si.R(), Ro) < RTOL and rel(si.vals(), Vo) < RTOL
        assert rel(st.get("sigma"), ost.sigma) < RTOL
