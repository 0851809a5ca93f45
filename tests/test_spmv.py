"""Matrix-vector products (GPU) over the row layouts they tell apart: scalar
rows and node triples, columns from row shapes (free or face-fixed patches of
at least 2^20 column indices) and from the column indices (smaller patches,
fixings strewn over the patch), rows shorter and longer than a round of their
lanes, each number of lanes.

A sum of n products is within n units of roundoff of its exact value, relative
to the sum of the absolute products; rows hold at most 1029 entries and both
sides round: 2.3e-13 (FP64), 6.2e-5 (FP32 against an FP64 sum)."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp
import torch

from ifem_amd import FP32, FP64, Session, lib
from ifem_amd import model as M
from ifem_amd._native import check

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (2, 9, 1), (5, 4, 6), (41, 7, 5)]


def _status(P, nc, fix):
    if fix == "none":
        return M.face_status(P, nc, [0] * 6)
    if fix == "faces":
        return M.face_status(P, nc, [7, 0, 0, 1, 0, 0])
    if fix == "nodes":  # whole nodes: node triples without common shapes
        return np.repeat(np.where(M.uniform(5, P.nnod) < 0.7, 1, 0), nc).astype(np.int32)
    return np.where(M.uniform(77, P.nnod * nc) < 0.7, 1, 0).astype(np.int32)


@pytest.mark.parametrize("fix", ["none", "faces", "nodes", "dofs"])
@pytest.mark.parametrize("nel", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("nc,p", [(1, 1), (1, 2), (1, 3), (3, 1), (3, 2), (3, 3)])
def test_product_of_every_row_layout(nc, p, nel, fix):
    if nc == 3 and nel[0] > 9:
        nel = (17, 3, 4)
    P = M.cube_patch(p, list(nel), 0.1, seed=p + nc)
    meqn, neq = M.equation_numbers(_status(P, nc, fix))
    if nc == 3:
        itg = M.Integrand(M.ELASTICITY, E=1.3, nu=0.28, body=(0.2, -0.1, 0.3))
    else:
        itg = M.Integrand(M.POISSON, source=M.smooth_source(4, 4))
    print(f"[gpu] spmv nc={nc} p={p} nel={nel} fix={fix} neq={neq}", flush=True)
    _check_products(P, itg, nc, p, meqn, neq)


def _shapes_kept(rp, ci, nodal):
    """Whether there are at least 2^20 (node) column indices and the distinct
    lists of column offsets take at most an eighth of them: the products then
    read the lists."""
    if nodal:
        n = (len(rp) - 1) // 3
        cnt = np.diff(rp)[::3] // 3
        start = np.concatenate([[0], np.cumsum(cnt)])
        ci = np.concatenate([ci[rp[3 * k]:rp[3 * k + 1]:3] // 3 for k in range(n)])
    else:
        n, start = len(rp) - 1, rp
    lists = {(ci[start[r]:start[r + 1]] - r).tobytes() for r in range(n)}
    return start[-1] >= 1 << 20 and sum(map(len, lists)) // ci.itemsize <= start[-1] // 8


# lanes: of the rows or nodes of this size (4 or 16: short lists; 32 or 64: long
# lists of few rows; 8 or 32: others)
@pytest.mark.parametrize("nc,p,nel,lanes", [
    (1, 1, (48, 36, 31), 4), (1, 2, (25, 23, 22), 8), (1, 3, (22, 21, 20), 32),
    (1, 3, (30, 26, 24), 8), (3, 1, (37, 33, 34), 16), (3, 2, (24, 21, 22), 32),
    (3, 3, (18, 15, 16), 64), (3, 3, (150, 20, 2), 32)])
def test_products_from_row_shapes(nc, p, nel, lanes):
    P = M.cube_patch(p, list(nel), 0.1, seed=p + nc)
    fix = [7, 0, 0, 7, 0, 0] if nc == 3 else [0] * 6
    meqn, neq = M.equation_numbers(M.face_status(P, nc, fix))
    if nc == 3:
        itg = M.Integrand(M.ELASTICITY, E=1.3, nu=0.28, body=(0.2, -0.1, 0.3))
    else:
        itg = M.Integrand(M.POISSON, source=M.smooth_source(4, 4))
    print(f"[gpu] spmv shapes nc={nc} p={p} nel={nel} neq={neq}", flush=True)
    rp, ci = _check_products(P, itg, nc, p, meqn, neq)
    assert _shapes_kept(rp, ci, nc == 3)
    length = len(ci) / neq / nc
    if nc == 1:
        want = 4 if length <= 40 else 32 if length > 120 and neq <= 16384 else 8
    else:
        want = 16 if length <= 32 else 64 if length > 128 and neq <= 3 * 16384 else 32
    assert want == lanes


def _check_products(P, itg, nc, p, meqn, neq):
    x = np.random.default_rng(neq).standard_normal(neq)
    hole = neq // 2
    xi = x.copy()
    xi[hole] = np.inf
    with Session() as s:
        s.bind(s.add_patch(P), nc, meqn, neq)
        s.init_assembly()
        s.assemble(itg, (p + 1,) * 3, FP64)
        rp, ci, A, _ = s.system()
        y = s.spmv(x)
        yi = s.spmv(xi)
        s.assemble(itg, (p + 1,) * 3, FP32)
        A32 = s.values_fp32().astype(np.float64)
        x32 = torch.from_numpy(x.astype(np.float32)).cuda()
        y32 = torch.empty_like(x32)
        torch.cuda.synchronize()
        s.spmv_device(x32.data_ptr(), y32.data_ptr(), FP32)
        s.synchronize()
        y32 = y32.cpu().numpy().astype(np.float64)
        x32 = x32.cpu().numpy().astype(np.float64)
    K = sp.csr_matrix((A, ci, rp), shape=(neq, neq))
    K32 = sp.csr_matrix((A32, ci, rp), shape=(neq, neq))
    assert np.all(np.abs(y - K @ x) <= 2.3e-13 * (abs(K) @ np.abs(x)))
    assert np.all(np.abs(y32 - K32 @ x32) <= 6.2e-5 * (abs(K32) @ np.abs(x32)))
    # an infinite entry reaches exactly the rows that hold its column
    rows = np.zeros(neq, bool)
    rows[np.repeat(np.arange(neq), np.diff(rp))[ci == hole]] = True
    assert np.array_equal(np.isfinite(yi), ~rows)
    assert np.array_equal(yi[~rows], y[~rows])
    return rp, ci


def _hip(name, *args):
    """A call of the HIP runtime that the library is linked with."""
    rc = getattr(lib(), name)(*args)
    assert rc == 0, (name, rc)


def test_first_products_of_every_kind():
    """The first product of a system gives the same bits whichever way it is
    made: plain, without allocation, recorded in a graph, and in a session that
    held a system of another pattern before."""
    def bind(s, nel, p):
        P = M.cube_patch(p, list(nel), 0.1, seed=p)
        meqn, neq = M.equation_numbers(M.face_status(P, 1, [0] * 6))
        s.bind(s.add_patch(P), 1, meqn, neq)
        s.init_assembly()
        s.assemble(M.Integrand(M.POISSON, source=M.smooth_source(4, 4)), (p + 1,) * 3, FP64)
        return neq

    def noalloc(s, x):
        y = np.empty_like(x)
        check(lib().ifem_gpu_spmv_noalloc(s.h, x.ctypes.data_as(C.c_void_p), y.ctypes.data_as(C.c_void_p)))
        return y
    nel = (16, 14, 12)
    print("[gpu] spmv first products", flush=True)
    with Session() as s:
        neq = bind(s, nel, 2)
        x = np.random.default_rng(neq).standard_normal(neq)
        plain = s.spmv(x)
        assert np.array_equal(noalloc(s, x), plain)
        n2 = bind(s, (9, 20, 11), 1)  # another pattern, shapes of the first one held
        rp, ci, A, _ = s.system()
        x2 = np.random.default_rng(n2).standard_normal(n2)
        K = sp.csr_matrix((A, ci, rp), shape=(n2, n2))
        assert np.all(np.abs(s.spmv(x2) - K @ x2) <= 2.3e-13 * (abs(K) @ np.abs(x2)))
    with Session() as s:
        bind(s, nel, 2)
        assert np.array_equal(noalloc(s, x), plain)
        assert np.array_equal(s.spmv(x), plain)
    with Session() as s:
        bind(s, nel, 2)
        xd = torch.from_numpy(x).cuda()
        yd = torch.zeros_like(xd)
        torch.cuda.synchronize()
        stream, graph, run = C.c_void_p(s.stream), C.c_void_p(), C.c_void_p()
        s.synchronize()
        _hip("hipStreamBeginCapture", stream, C.c_int(0))  # global: no allocation meanwhile
        s.spmv_device(xd.data_ptr(), yd.data_ptr())
        _hip("hipStreamEndCapture", stream, C.byref(graph))
        _hip("hipGraphInstantiate", C.byref(run), graph, None, None, C.c_size_t(0))
        for scale in (1.0, 2.0, -1.0):
            xd.copy_(torch.from_numpy(scale * x))
            torch.cuda.synchronize()
            _hip("hipGraphLaunch", run, stream)
            s.synchronize()
            assert np.array_equal(yd.cpu().numpy(), scale * plain)
            assert np.array_equal(s.spmv(x), plain)
        _hip("hipGraphExecDestroy", run)
        _hip("hipGraphDestroy", graph)
