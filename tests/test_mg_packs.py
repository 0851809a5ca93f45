"""Fine-level FP16 product of the multigrid smoother (GPU) at node rows whose
neighbour counts fill a pack of four, leave one to three over or are shorter
than a pack group, with and (nodes fixed at random, small patches) without row
shapes.

The product enters the V-cycle only, so the cycle itself is checked: it is a
symmetric positive definite preconditioner up to the FP32 rounding of its sums
(1e-5 of |<u, M v>| bounds, a few hundred products per sum and some tens of
sums), and multigrid-preconditioned CG reaches the direct solution.  A lost or
doubled block breaks the symmetry at order one over the row length, 1e-2."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from ifem_amd import FP64, PC_MG, Session
from ifem_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fix", ["faces", "nodes"])
@pytest.mark.parametrize("p,nel", [(1, (6, 5, 9)), (1, (4, 8, 8)), (2, (6, 8, 7)), (2, (12, 5, 6)),
                                   (3, (6, 6, 7))])
def test_cycle_is_symmetric_and_solves(p, nel, fix):
    P = M.cube_patch(p, list(nel), 0.1, seed=p)
    msc = np.asarray(M.face_status(P, 3, [7, 0, 0, 0, 0, 0])).copy()
    if fix == "nodes":
        msc[np.repeat(M.uniform(5, P.nnod) < 0.05, 3)] = 0
    meqn, neq = M.equation_numbers(msc)
    itg = M.Integrand(M.ELASTICITY, E=1.3, nu=0.28, body=(0.2, -0.1, 0.3))
    print(f"[gpu] mg packs p={p} nel={nel} fix={fix} neq={neq}", flush=True)
    rng = np.random.default_rng(neq)
    u, v = rng.standard_normal(neq), rng.standard_normal(neq)
    with Session() as s:
        s.bind(s.add_patch(P), 3, meqn, neq)
        s.init_assembly()
        s.assemble(itg, (p + 1,) * 3, FP64)
        rp, ci, A, b = s.system()
        s.mg_setup(2)
        mu, mv = s.mg_apply(u), s.mg_apply(v)
        st = s.solve(rtol=1e-11, maxits=500, pc=PC_MG)
        x = s.solution()
    K = sp.csr_matrix((A, ci, rp), shape=(neq, neq))
    scale = np.sqrt((u @ mu) * (v @ mv))
    assert u @ mu > 0 and v @ mv > 0
    assert abs(u @ mv - v @ mu) <= 1e-5 * scale
    assert st["converged"] and not st["fallback"]
    xd = spla.spsolve(K.tocsc(), b)
    e = x - xd
    assert np.sqrt(e @ (K @ e)) <= 1e-7 * np.sqrt(xd @ (K @ xd))


@pytest.mark.parametrize("p,nel", [(1, (37, 33, 34)), (2, (24, 21, 22))])
def test_cycle_from_row_shapes(p, nel):
    """Systems whose products read row shapes (2^20 node couplings and more)."""
    P = M.cube_patch(p, list(nel), 0.1, seed=p)
    meqn, neq = M.equation_numbers(M.face_status(P, 3, [7, 0, 0, 0, 0, 0]))
    itg = M.Integrand(M.ELASTICITY, E=1.3, nu=0.28, body=(0.2, -0.1, 0.3))
    print(f"[gpu] mg packs shapes p={p} nel={nel} neq={neq}", flush=True)
    rng = np.random.default_rng(neq)
    u, v = rng.standard_normal(neq), rng.standard_normal(neq)
    with Session() as s:
        s.bind(s.add_patch(P), 3, meqn, neq)
        s.init_assembly()
        s.assemble(itg, (p + 1,) * 3, FP64)
        rp, ci, A, b = s.system()
        s.mg_setup(2)
        mu, mv = s.mg_apply(u), s.mg_apply(v)
        st = s.solve(rtol=1e-11, maxits=500, pc=PC_MG)
        x = s.solution()
    assert len(ci) // 9 >= 1 << 20
    K = sp.csr_matrix((A, ci, rp), shape=(neq, neq))
    assert u @ mu > 0 and v @ mv > 0
    assert abs(u @ mv - v @ mu) <= 1e-5 * np.sqrt((u @ mu) * (v @ mv))
    assert st["converged"] and not st["fallback"]
    assert np.linalg.norm(b - K @ x) <= 1e-11 * np.linalg.norm(b) * 1.01
