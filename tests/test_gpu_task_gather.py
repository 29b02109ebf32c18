"""The task row gather of the P2 elasticity matrix against the oracle: batches
from single rows to the largest its LDS takes (so first values at every
alignment, fewer and more tasks and elements than threads, blocks of one and of
several tasks), float64 within 1e-12 and float32 within 1e-5 of the float64
oracle, added to values the Mat already holds."""
import numpy as np
import pytest

from helpers import TetProblem, oracle_p2, relerr, repeated_edge_nodes, unreferenced_nodes
from pyop2_amd import device as dev, elements, op2
from pyop2_amd.configuration import configuration
from pyop2_amd.meshes import unit_cube_tet_p2, workload_rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def meshes():
    m = unit_cube_tet_p2(7, rng=workload_rng(3))
    rng = np.random.default_rng(4)
    m.coords[:] += rng.uniform(-0.01, 0.01, m.coords.shape)
    out = {"plain": m, "repeated": repeated_edge_nodes(m), "holes": unreferenced_nodes(m)[0]}
    return {k: (v, oracle_p2("p2_elasticity_matrix", v, lam=1.3, mu=0.7)) for k, v in out.items()}


def _loop(m, dtype, core=None):
    p = TetProblem(m, dtype=dtype, core=core)
    A = op2.Mat(p.sparsity(), dtype)
    pl = op2.ParLoop(elements.p2_elasticity_matrix(1.3, 0.7), p.cells, A(op2.INC, (p.c2n, p.c2n)),
                     p.X(op2.READ, p.c2v))
    return p, A, pl


@pytest.mark.parametrize("dtype,tol", [(np.float64, 1e-12), (np.float32, 1e-5)])
@pytest.mark.parametrize("batch,block", [((1, 1), 64), ((16, 40), 128), ((64, 97), 64), ((192, 240), 256),
                                         ((384, 480), 512), ((400, 500), 256)])
def test_batches(device, meshes, dtype, tol, batch, block):
    m, ref = meshes["plain"]
    _, A, pl = _loop(m, dtype)
    held = np.random.default_rng(1).standard_normal(ref.values.size).astype(dtype)
    A.device_values.copy_(dev.to_device(held))
    ex = pl.global_kernel.compile()
    for _ in range(2):
        ex.launch(0, m.ncells, pl, {"strategy": "rowgather_tasks", "batch": list(batch), "block": block})
    assert ex.strategy_used == "rowgather_tasks"
    want = held.astype(np.float64).reshape(ref.values.shape) + 2 * ref.values
    assert relerr(dev.to_host(A.device_values).reshape(ref.values.shape), want) < tol


@pytest.mark.parametrize("dtype,tol", [(np.float64, 1e-12), (np.float32, 1e-5)])
@pytest.mark.parametrize("mesh,core", [("plain", 777), ("plain", 0), ("repeated", None), ("holes", 900)])
def test_bands_and_odd_maps(device, meshes, dtype, tol, mesh, core):
    """Core and owned bands (each skips the other's elements), map rows that
    name a node twice, rows without elements."""
    m, ref = meshes[mesh]
    configuration["strategy"] = "rowgather_tasks"
    _, A, pl = _loop(m, dtype, core)
    pl()
    A.assemble()
    assert pl.global_kernel.compile().strategy_used == "rowgather_tasks"
    rp, ci, v = A._host_csr()
    assert np.array_equal(rp, ref.rowptr) and np.array_equal(ci, ref.colidx)
    assert relerr(v, ref.values) < tol


def test_batches_that_do_not_fit_take_the_slot_table(device, meshes, monkeypatch):
    from pyop2_amd import registry
    m, ref = meshes["plain"]
    monkeypatch.setattr(registry, "_LDS", 20000)
    configuration["strategy"] = "rowgather_tasks"
    _, A, pl = _loop(m, np.float64)
    pl()
    assert pl.global_kernel.compile().strategy_used == "rowgather_slots"
    assert relerr(dev.to_host(A.device_values).reshape(ref.values.shape), ref.values) < 1e-12


def test_fused_loop_as_split_with_tasks(device, meshes):
    m, ref = meshes["plain"]
    p = TetProblem(m, dtype=np.float32)
    A, R = op2.Mat(p.sparsity(), np.float32), op2.Dat(p.nodes ** 3, dtype=np.float32)
    pl = op2.ParLoop(elements.p2_elasticity_fused(1.3, 0.7), p.cells, A(op2.INC, (p.c2n, p.c2n)),
                     R(op2.INC, p.c2n), p.X(op2.READ, p.c2v), p.u(op2.READ, p.c2n))
    ex = pl.global_kernel.compile()
    cfg = {"strategy": "split", "overlap": "after",
           "parts": [{"strategy": "rowgather_tasks"}, {"strategy": "staged_coloured"}]}
    for _ in range(2):
        ex.launch(0, m.ncells, pl, cfg)
    f = lambda a: a.astype(np.float32).astype(np.float64)  # noqa: E731
    res = oracle_p2("p2_elasticity_residual", m, lam=1.3, mu=0.7, coords=f(m.coords), u=f(m.u))
    assert relerr(dev.to_host(A.device_values).reshape(ref.values.shape), 2 * ref.values) < 1e-5
    assert relerr(R.data_ro, 2 * res) < 1e-5
