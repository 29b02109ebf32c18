"""Staged tiles whose nodes are shared by one to many tiles (tiles of single
elements to tiles that hold a mesh), one and three values per node, one and
two incremented maps: float64 within 1e-12 and float32 within 1e-5 of the
float64 oracle, added to values the Dats already hold."""
import numpy as np
import pytest

from helpers import TetProblem, TriProblem, oracle_p1, oracle_p2, relerr, repeated_edge_nodes
from oracle import seqwrap
from pyop2_amd import device as dev, elements, op2
from pyop2_amd.meshes import unit_cube_tet_p2, unit_square_tri, workload_rng

pytestmark = pytest.mark.gpu

TILES = [(1, 64), (3, 64), (16, 128), (61, 64), (200, 192), (384, 256)]


def _check(pl, n, outs, refs, tol, tile, block):
    """Two launches over Dats that hold values, twice."""
    held = [np.random.default_rng(k).standard_normal(r.shape) for k, r in enumerate(refs)]
    ex = pl.global_kernel.compile()
    seen = []
    for _ in range(2):
        for d, h in zip(outs, held):
            d.device_data.copy_(dev.to_device(h.astype(d.dtype)))
        for _ in range(2):
            ex.launch(0, n, pl, {"strategy": "staged", "tile": tile, "block": block, "partials": True})
        assert ex.strategy_used == "staged"
        seen.append([dev.to_host(d.device_data_ro).copy() for d in outs])
    for d, h, r, first, again in zip(outs, held, refs, *seen):
        assert relerr(first, h.astype(d.dtype).astype(np.float64) + 2 * r) < tol
        assert relerr(again, first) < tol


@pytest.mark.parametrize("tile,block", TILES)
def test_one_value_per_node(device, tile, block):
    m = unit_square_tri(23, rng=workload_rng(1))
    p = TriProblem(m)
    R = op2.Dat(p.verts, name="R")
    pl = op2.ParLoop(elements.p1_laplace_residual(), p.cells, R(op2.INC, p.c2v), p.X(op2.READ, p.c2v),
                     p.u(op2.READ, p.c2v))
    _check(pl, m.ncells, [R], [oracle_p1("p1_laplace_residual", m)], 1e-12, tile, block)


@pytest.mark.parametrize("dtype,tol", [(np.float64, 1e-12), (np.float32, 1e-5)])
@pytest.mark.parametrize("tile,block", TILES)
@pytest.mark.parametrize("repeated", [False, True])
def test_three_values_per_node(device, dtype, tol, tile, block, repeated):
    m = unit_cube_tet_p2(5, rng=workload_rng(3))
    m = repeated_edge_nodes(m) if repeated else m
    p = TetProblem(m, dtype=dtype)
    R = op2.Dat(p.nodes ** 3, dtype=dtype, name="R")
    pl = op2.ParLoop(elements.p2_elasticity_residual(1.3, 0.7), p.cells, R(op2.INC, p.c2n),
                     p.X(op2.READ, p.c2v), p.u(op2.READ, p.c2n))
    _check(pl, m.ncells, [R], [oracle_p2("p2_elasticity_residual", m, 1.3, 0.7)], tol, tile, block)


@pytest.mark.parametrize("tile,block", TILES)
def test_two_incremented_maps(device, tile, block):
    m = unit_cube_tet_p2(5, rng=workload_rng(4))
    rng = np.random.default_rng(7)
    X = m.coords + rng.uniform(-0.01, 0.01, m.coords.shape)
    E = rng.standard_normal((m.nnodes, 3))
    p = TetProblem(m)
    p.X.data[:] = X
    Rb, ub, Xb = op2.Dat(p.nodes ** 3, E), op2.Dat(p.nodes ** 3), op2.Dat(p.verts ** 3)
    pl = op2.ParLoop(elements.p2_elasticity_adjoint(1.3, 0.7), p.cells, ub(op2.INC, p.c2n), Xb(op2.INC, p.c2v),
                     Rb(op2.READ, p.c2n), p.X(op2.READ, p.c2v), p.u(op2.READ, p.c2n))
    rub, rXb = np.zeros((m.nnodes, 3)), np.zeros((m.nverts, 3))
    seqwrap.run(elements.kernel_source("p2_elasticity_adjoint", lam=1.3, mu=0.7), "p2_elasticity_adjoint",
                [seqwrap.DatArg(rub, "INC", m.cell_node), seqwrap.DatArg(rXb, "INC", m.cell_vertex),
                 seqwrap.DatArg(E, "READ", m.cell_node), seqwrap.DatArg(X, "READ", m.cell_vertex),
                 seqwrap.DatArg(m.u, "READ", m.cell_node)], [(0, m.ncells)])
    _check(pl, m.ncells, [ub, Xb], [rub, rXb], 1e-12, tile, block)
