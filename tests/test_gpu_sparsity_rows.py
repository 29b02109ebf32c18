"""Sparsity rows and row incidences on the device against the oracle, at the
sizes where the row kernels change: rows around the candidates a group of
lanes takes (192 and 384), around 2,048 candidates, rows without elements,
negative map entries, several pairs, rectangular patterns, and incidence
lists that do not fit the sort's stage."""
import numpy as np
import pytest

from oracle import sparsity as osp
from pyop2_amd import op2, plans
from pyop2_amd import device as dev

pytestmark = pytest.mark.gpu


def _heavy_map(rng, nrows, arity, heavy, ncells, negative=False):
    """Random cells, node 3 in the first ``heavy`` of them."""
    t = rng.integers(8, nrows, size=(ncells, arity)).astype(np.int32)
    t[:heavy, 0] = 3
    if negative:
        t[rng.random(t.shape) < 0.1] = -1
        t[:heavy, 0] = 3
    return t


def _check(rowsize, colsize, pairs, diag):
    rows = op2.Set(rowsize)
    cols = rows if colsize is None else op2.Set(colsize)
    maps, host = [], []
    for r, c in pairs:
        it = op2.Set(len(r))
        rm = op2.Map(it, rows, r.shape[1], r)
        cm = rm if c is None else op2.Map(it, cols, c.shape[1], c)
        maps.append((rm, cm, None))
        host.append((r, r if c is None else c, len(r)))
    sp = op2.Sparsity((rows ** 1, cols ** 1), maps)
    rp, ci = osp.pattern(rowsize, cols.total_size, host, set_diag=diag)
    grp, gci = (dev.to_host(t) for t in sp.block_pattern)
    assert np.array_equal(grp, rp) and np.array_equal(gci, ci)


@pytest.mark.parametrize("heavy", [0, 47, 48, 511, 512, 700])
def test_half_wave_rows(device, heavy):
    """Few candidates a row on average: half a wave a row, up to 192; 47, 48,
    511 and 512 cells of four make 189, 193, 2,045 and 2,049 with the diagonal."""
    rng = np.random.default_rng([5, heavy])
    _check(3000, None, [(_heavy_map(rng, 3000, 4, heavy, 1500), None)], True)


@pytest.mark.parametrize("heavy", [0, 38, 39, 204, 205])
def test_whole_wave_rows(device, heavy):
    """Many candidates a row: a wave a row, up to 384 (38 and 39 cells of ten
    make 381 and 391 with the diagonal, 204 and 205 make 2,041 and 2,051)."""
    rng = np.random.default_rng([6, heavy])
    _check(700, None, [(_heavy_map(rng, 700, 10, heavy, 500), None)], True)


def test_pairs_negative_entries_and_rectangular(device):
    rng = np.random.default_rng(7)
    a = _heavy_map(rng, 400, 3, 30, 300, negative=True)
    b = _heavy_map(rng, 400, 5, 90, 200, negative=True)
    _check(400, None, [(a, None), (b, None)], True)
    c = rng.integers(0, 97, size=(300, 4)).astype(np.int32)
    c[::7, 1] = -1
    _check(400, 97, [(a, c)], False)


@pytest.mark.parametrize("nrows", [1, 255, 256, 257])
@pytest.mark.parametrize("ncells", [0, 2, 900, 4000])
def test_incidences_ascend(device, nrows, ncells):
    """Sorted incidence lists around the 256 rows and 7,168 entries of a stage."""
    rng = np.random.default_rng([nrows, ncells])
    t = rng.integers(0, nrows, size=(ncells, 3)).astype(np.int32)
    m = op2.Map(op2.Set(ncells), op2.Set(nrows), 3, t)
    tr = plans.transpose(m, nrows, ncells)
    order = np.argsort(t.ravel(), kind="stable")
    assert np.array_equal(dev.to_host(tr.inc_ptr), np.searchsorted(t.ravel()[order], np.arange(nrows + 1)))
    assert np.array_equal(dev.to_host(tr.inc_ent)[:tr.total], order)


@pytest.mark.parametrize("n", [0, 1, 7, 2048, 2049, 300000, 1024 * 2048, 1024 * 2048 + 1, 2500000])
def test_exclusive_scan(device, n):
    """One tile, several, the most whose sums the blocks take themselves, more."""
    import ctypes
    v = np.random.default_rng(n).integers(0, 7, n).astype(np.int32)
    t, out = dev.to_device(v), dev.empty((n + 1,), np.int32)
    L, need, total = dev.lib(), ctypes.c_size_t(), ctypes.c_int64()
    dev.check(L.op2hip_scan_workspace(n, ctypes.byref(need)))
    work = dev.empty((need.value,), np.uint8)
    for _ in range(2):
        dev.check(L.op2hip_exclusive_scan(n, dev.ptr(t), dev.ptr(out), ctypes.byref(total), dev.ptr(work),
                                          need.value, dev.stream()))
        want = np.concatenate(([0], np.cumsum(v)))
        assert total.value == want[-1] and np.array_equal(dev.to_host(out), want)


@pytest.mark.parametrize("nrows", [1, 64, 65, 5000])
def test_entries_beyond_the_set_are_counted(device, nrows):
    """The counter lies behind the counts, whatever their number."""
    import ctypes
    v = np.random.default_rng(1).integers(0, nrows, (900, 3)).astype(np.int32)
    L, need, total = dev.lib(), ctypes.c_size_t(), ctypes.c_int64()
    dev.check(L.op2hip_transpose_workspace(nrows, ctypes.byref(need)))
    work, ptr = dev.empty((need.value,), np.uint8), dev.empty((nrows + 1,), np.int32)

    def count():
        return L.op2hip_transpose_count(nrows, dev.ptr(t), 3, 900, dev.ptr(ptr), ctypes.byref(total),
                                        dev.ptr(work), need.value, dev.stream())
    t = dev.to_device(v)
    dev.check(count())
    assert total.value == v.size
    assert np.array_equal(np.diff(dev.to_host(ptr)), np.bincount(v.ravel(), minlength=nrows))
    v[5, 1] = v[899, 2] = nrows
    t = dev.to_device(v)
    with pytest.raises(dev.DeviceError, match="2 map entries"):
        dev.check(count())
