"""Launches that a loop and its maps keep ready: a call follows what has changed
since (strategy, replaced data, another loop's data on the same maps, new maps),
and keeping them does not keep the maps."""
import gc
import weakref

import numpy as np
import pytest

from helpers import oracle_p1, relerr
from pyop2_amd import elements, op2
from pyop2_amd.configuration import configuration
from pyop2_amd.meshes import unit_square_tri, workload_rng

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _objects(n=12):
    m = unit_square_tri(n, rng=workload_rng(1), permute=True)
    cells, verts = op2.Set(m.ncells), op2.Set(m.nverts)
    c2v = op2.Map(cells, verts, 3, m.cell_vertex)
    return m, cells, verts, c2v, op2.Dat(verts ** 2, m.coords), op2.Dat(verts, m.u)


def test_strategy_and_data_changes(device):
    m, cells, verts, c2v, X, u = _objects()
    want = oracle_p1("p1_laplace_residual", m)
    R = op2.Dat(verts)
    pl = op2.ParLoop(elements.p1_laplace_residual(), cells, R(op2.INC, c2v), X(op2.READ, c2v), u(op2.READ, c2v))
    ex = pl.global_kernel.compile()
    passes = 0
    for strategy in ("atomic", "staged", "coloured", "auto", "atomic"):
        configuration["strategy"] = strategy
        for _ in range(2):
            pl()
            passes += 1
        assert strategy == "auto" or ex.strategy_used == strategy
        assert relerr(R.data_ro, passes * want) < TOL
    configuration["strategy"], configuration["staged_partials"] = "staged", False
    pl()
    assert relerr(R.data_ro, (passes + 1) * want) < TOL
    # newer host data, then another Dat in its place
    u.data[:] *= 2.0
    R.zero()
    pl()
    assert relerr(R.data_ro, 2.0 * want) < TOL
    S = op2.Dat(verts)
    pl.replace_data(0, S)
    pl()
    assert relerr(S.data_ro, 2.0 * want) < TOL and relerr(R.data_ro, 2.0 * want) < TOL


def test_two_mats_and_another_pattern(device):
    m, cells, verts, c2v, X, _ = _objects()
    want = oracle_p1("p1_laplace_matrix", m)
    sp = op2.Sparsity((verts ** 1, verts ** 1), [(c2v, c2v, None)])
    far = np.full((m.ncells, 1), m.nverts - 1, dtype=np.int32)
    wide = op2.Sparsity((verts ** 1, verts ** 1), [(c2v, c2v, None), (op2.Map(cells, verts, 1, far),) * 2 + (None,),
                                                   (c2v, op2.Map(cells, verts, 1, far), None)])
    mats = [op2.Mat(sp, np.float64), op2.Mat(sp, np.float64), op2.Mat(wide, np.float64)]
    loops = [op2.ParLoop(elements.p1_laplace_matrix(), cells, A(op2.INC, (c2v, c2v)), X(op2.READ, c2v)) for A in mats]
    for strategy in ("rowgather_slots", "rowgather_rows"):
        configuration["strategy"] = strategy
        for A in mats:
            A.zero()
        for pl in loops + loops[:1]:
            pl()
        dense = np.zeros((m.nverts, m.nverts))
        for r in range(m.nverts):
            s = slice(want.rowptr[r], want.rowptr[r + 1])
            dense[r, want.colidx[s]] = np.asarray(want.values[s]).ravel()
        for A, times in zip(mats, (2, 1, 1)):
            assert relerr(A.values, times * dense) < TOL
    # a kept loop given a Mat of the wide pattern
    loops[0].replace_data(0, mats[2])
    mats[2].zero()
    loops[0]()
    assert relerr(mats[2].values, dense) < TOL


def test_new_maps_and_freed_ones(device):
    configuration["strategy"] = "staged"
    for n in (6, 9, 6, 7):
        m, cells, verts, c2v, X, u = _objects(n)
        R = op2.Dat(verts)
        for _ in range(2):
            op2.par_loop(elements.p1_laplace_residual(), cells, R(op2.INC, c2v), X(op2.READ, c2v), u(op2.READ, c2v))
        assert relerr(R.data_ro, 2 * oracle_p1("p1_laplace_residual", m)) < TOL
    gone = weakref.ref(c2v)
    gc.collect()
    gc.disable()
    try:
        del c2v, R, X, u, cells, verts
        assert gone() is None
    finally:
        gc.enable()
