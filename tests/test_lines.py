"""Line kernels of the volume assembly (GPU): K and b against the oracle at
the sizes where their work split can go wrong -- one element per direction,
line groups of full and partial size, row segments of a long line, rows with
full and with compacted windows.

Tolerances: the sums are a few hundred to a few thousand products long, so
1e-12 of the largest entry in FP64; FP32 values to 1e-5 of it."""
import numpy as np
import pytest

import oracle
from ifem_amd import FP32, FP64, Session
from ifem_amd import model as M
from ifem_amd import problems
from test_gpu_parity import _prescribed_case
from test_multipatch import _global_status, _oracle_system

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (1, 8, 2), (3, 11, 1), (29, 4, 3), (64, 2, 2), (9, 22, 5)]


def _problem(nc, p, nel, fix):
    P = M.cube_patch(p, list(nel), 0.1, seed=p + nc)
    if fix == "random":
        msc = np.where(M.uniform(77, P.nnod * nc) < 0.7, 1, 0).astype(np.int32)
    else:
        msc = M.face_status(P, nc, [0, 0, 0, 0, 0, 0] if fix == "none" else [7, 0, 0, 1, 0, 0])
    meqn, neq = M.equation_numbers(msc)
    if nc == 3:
        itg = M.Integrand(M.ELASTICITY, E=1.3, nu=0.28, body=(0.2, -0.1, 0.3))
    else:
        itg = M.Integrand(M.POISSON, kappa=M.lognormal_conductivity(3, 0.7, 0.3, 8),
                          source=M.smooth_source(4, 4))
    return problems.Problem("lines", P, itg, (p + 1,) * 3, meqn, neq)


@pytest.mark.parametrize("fix", ["none", "faces", "random"])
@pytest.mark.parametrize("nel", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("nc,p", [(1, 1), (1, 2), (3, 1), (3, 2)])
def test_lines_match_oracle(nc, p, nel, fix):
    if nc == 3 and nel[0] * nel[1] * nel[2] > 400:
        nel = (nel[0], nel[1] // 2, nel[2])
    pb = _problem(nc, p, nel, fix)
    print(f"[gpu] lines nc={nc} p={p} nel={nel} fix={fix} neq={pb.neq}", flush=True)
    if pb.neq == 0:
        pytest.skip("no free DOF")
    rp, ci, A, b = oracle.system(pb.patch, pb.integrand, pb.ng, pb.meqn, pb.neq, None, 0)
    with Session() as s:
        s.bind(s.add_patch(pb.patch), nc, pb.meqn, pb.neq)
        s.init_assembly()
        s.assemble(pb.integrand, pb.ng, FP64)
        grp, gci, gA, gb = s.system()
        s.assemble(pb.integrand, pb.ng, FP32)
        A32 = s.values_fp32().astype(np.float64)
    assert np.array_equal(grp, rp) and np.array_equal(gci, ci)
    assert np.max(np.abs(gA - A)) <= 1e-12 * np.max(np.abs(A))
    assert np.max(np.abs(gb - b)) <= 1e-12 * max(np.max(np.abs(b)), 1e-300)
    assert np.max(np.abs(A32 - A)) <= 1e-5 * np.max(np.abs(A))


@pytest.mark.parametrize("nel", [(1, 1, 1), (5, 5, 5), (8, 3, 2), (29, 4, 3), (64, 2, 2)],
                         ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("nc,p,ng", [(1, 1, 2), (1, 1, 3), (1, 2, 3), (3, 1, 2), (3, 1, 3), (3, 2, 3)])
def test_row_splits_give_the_same_bits(nc, p, ng, nel):
    """Variants 0 (the built-in rule: down to one row per segment on small
    patches), 1 (twice as many segments) and 2 (whole lines)."""
    pb = _problem(nc, p, nel, "none")
    print(f"[gpu] row splits nc={nc} p={p} ng={ng} nel={nel}", flush=True)
    out = []
    with Session() as s:
        s.bind(s.add_patch(pb.patch), nc, pb.meqn, pb.neq)
        s.init_assembly()
        for variant in (-1, 0, 1, 2):
            for precision in (FP64, FP32):
                if (nc, p, precision) != (3, 2, FP32):  # a kernel without row segments
                    s.set_assembly_variant(p, ng, nc, precision, variant)
                s.assemble(pb.integrand, (ng,) * 3, precision)
            _, _, A, b = s.system()
            out.append((A.copy(), b.copy(), s.values_fp32().copy()))
    for got in out[1:]:
        for x, y in zip(out[0], got):
            assert np.array_equal(x, y)


def _against(s, itg, ng, rp, ci, A, b):
    """K and b of both precisions of a bound session against the oracle's."""
    s.init_assembly()
    s.assemble(itg, (ng,) * 3, FP64)
    grp, gci, gA, gb = s.system()
    s.assemble(itg, (ng,) * 3, FP32)
    A32 = s.values_fp32().astype(np.float64)
    assert np.array_equal(grp, rp) and np.array_equal(gci, ci)
    assert np.max(np.abs(gA - A)) <= 1e-12 * np.max(np.abs(A))
    assert np.max(np.abs(gb - b)) <= 1e-12 * max(np.max(np.abs(b)), 1e-300)
    assert np.max(np.abs(A32 - A)) <= 1e-5 * np.max(np.abs(A))


@pytest.mark.parametrize("rhs", [True, False], ids=["rhs", "norhs"])
@pytest.mark.parametrize("fix", ["none", "faces", "random"])
@pytest.mark.parametrize("nel", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("nc", [1, 3])
def test_linear_elements_with_three_points(nc, nel, fix, rhs):
    pb = _problem(nc, 1, nel, fix)
    if not rhs:
        pb.integrand.source = M.Function()
        pb.integrand.body = (0.0, 0.0, 0.0)
    print(f"[gpu] lines nc={nc} p=1 ng=3 nel={nel} fix={fix} rhs={rhs}", flush=True)
    if pb.neq == 0:
        pytest.skip("no free DOF")
    want = oracle.system(pb.patch, pb.integrand, (3, 3, 3), pb.meqn, pb.neq, None, 0)
    with Session() as s:
        s.bind(s.add_patch(pb.patch), nc, pb.meqn, pb.neq)
        _against(s, pb.integrand, 3, *want)


@pytest.mark.parametrize("nel", [(1, 8, 2), (29, 4, 3), (9, 22, 5)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("nc,p,ng", [(1, 1, 2), (1, 1, 3), (1, 2, 3), (3, 1, 2), (3, 1, 3), (3, 2, 3)])
def test_prescribed_values_at_split_sizes(nc, p, ng, nel):
    if nc == 3:
        nel = (nel[0], (nel[1] + 3) // 4, nel[2])
    pb = _problem(nc, p, nel, "none")
    sam = _prescribed_case(pb, seed=p + ng)
    g = sam.prescribed_values()
    print(f"[gpu] lines prescribed nc={nc} p={p} ng={ng} nel={nel} neq={sam.neq}", flush=True)
    if sam.neq == 0:
        pytest.skip("no free DOF")
    rp, ci = oracle.pattern(pb.patch, nc, sam.meqn, sam.neq)
    A, b = oracle.assemble(pb.patch, pb.integrand, (ng,) * 3, sam.meqn, sam.neq, rp, ci, gdof=g)
    with Session() as s:
        s.bind_constraints(s.add_patch(pb.patch), nc, sam)
        _against(s, pb.integrand, ng, rp, ci, A, b)


@pytest.mark.parametrize("nels,nyz", [((1, 1), 1), ((2, 9), 4), ((17, 12), 2)])
@pytest.mark.parametrize("nc,p,ng", [(1, 1, 2), (1, 1, 3), (1, 2, 3), (3, 1, 2), (3, 1, 3), (3, 2, 3)])
def test_rows_shared_by_two_patches(nc, p, ng, nels, nyz):
    mp = M.x_split_patches(p, list(nels), nyz, 0.1, 3)
    meqn, neq = M.equation_numbers(_global_status(mp, nc, [7 if nc == 3 else 1, 0, 0, 0, 0, 0]))
    itg = _problem(nc, p, (1, 1, 1), "none").integrand
    print(f"[gpu] lines shared nc={nc} p={p} ng={ng} nels={nels} nyz={nyz} neq={neq}", flush=True)
    want = _oracle_system(mp, itg, [ng] * 3, meqn, neq)
    with Session() as s:
        s.bind_patches([s.add_patch(P) for P in mp.patches], mp.mlgn, nc, meqn, neq)
        _against(s, itg, ng, *want)
