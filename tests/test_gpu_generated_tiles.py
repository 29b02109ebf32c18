"""Generated loops in tiles and their reduced Globals: the tiled launch against
the device-atomic one and numpy over the forms it takes (types, shapes, several
outputs, one or two maps, CSR and BSR Mats, split bands), the loops that must
keep the atomic launch, and reductions around the sizes where they change."""
import numpy as np
import pytest

from pyop2_amd import codegen, op2
from pyop2_amd import device as dev
from pyop2_amd.configuration import configuration

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _tiles_at_test_sizes(monkeypatch):
    monkeypatch.setattr(codegen, "_TILED_LEAST", 32768)

# float sums of a few tens of terms of size one, in any order, on numbers of
# size ten: some hundred roundings of the type at most
TOL = {"float64": 1e-12, "float32": 1e-4, "int32": 0, "int64": 0}


def _mesh(n, nodes, arity, rng):
    """Elements whose nodes are near each other."""
    base = np.sort(rng.integers(0, max(nodes - 40, 1), size=n))
    return ((base[:, None] + rng.integers(0, 40, size=(n, arity))) % nodes).astype(np.int32)


def _kernel(arity, dim, ctype):
    return op2.Kernel(f"""
static void spread({ctype} *r, const {ctype} *x) {{
  for (int i = 0; i < {arity}; ++i) for (int j = 0; j < {dim}; ++j)
    r[i * {dim} + j] += x[i] * ({ctype})(j + 1) + x[0];
}}""", "spread")


@pytest.mark.parametrize("dtype,ctype", [("float64", "double"), ("float32", "float"), ("int32", "int"),
                                         ("int64", "long long")])
@pytest.mark.parametrize("n,arity,dim,core", [(9000, 2, 4, None), (16385, 3, 1, None), (4097, 4, 3, None),
                                              (30000, 2, 1, 11111), (2049, 10, 2, None), (1000, 1, 120, 450)])
def test_dat_increments(device, dtype, ctype, n, arity, dim, core):
    rng = np.random.default_rng([n, arity, dim])
    nodes = n // 3 if arity > 1 else 60
    table = _mesh(n, nodes, arity, rng)
    x = rng.integers(-9, 9, nodes).astype(dtype)
    it, ns = op2.Set(n if core is None else (core, n, n)), op2.Set(nodes)
    m = op2.Map(it, ns, arity, table)
    start = rng.integers(-5, 5, (nodes, dim)).astype(dtype)
    got = {}
    for strategy in ("auto", "atomic"):
        configuration["strategy"] = strategy
        R = op2.Dat(ns ** dim, start.copy(), dtype)
        pl = op2.ParLoop(_kernel(arity, dim, ctype), it, R(op2.INC, m), op2.Dat(ns, x, dtype)(op2.READ, m))
        for _ in range(2):
            pl()
        got[strategy] = np.asarray(R.data_ro).reshape(nodes, dim).astype(np.float64)
        assert pl.global_kernel.compile().strategy_used == ("staged" if strategy == "auto" else "atomic")
    want = start.astype(np.float64).reshape(nodes, dim).copy()
    xe = x.astype(np.float64)[table]
    add = xe[:, :, None] * (1.0 + np.arange(dim)) + xe[:, :1, None]
    for _ in range(2):
        np.add.at(want, table, add)
    scale = np.abs(want).max()
    for g in got.values():
        assert np.abs(g - want).max() <= TOL[dtype] * scale


def test_two_outputs_on_two_maps(device):
    """Two Dats on one map, a third on another, a direct output beside them."""
    rng = np.random.default_rng(3)
    n, na, nb = 12000, 4000, 3000
    ta, tb = _mesh(n, na, 3, rng), _mesh(n, nb, 2, rng)
    it, A, B = op2.Set(n), op2.Set(na), op2.Set(nb)
    ma, mb = op2.Map(it, A, 3, ta), op2.Map(it, B, 2, tb)
    x = rng.random(n)
    k = op2.Kernel("""
static void three(double *p, double *q, double *s, double *d, const double *x) {
  for (int i = 0; i < 3; ++i) { p[i] += x[0] + i; q[2 * i] += x[0]; q[2 * i + 1] -= x[0]; }
  for (int i = 0; i < 2; ++i) s[i] += x[0] * (i + 1);
  d[0] = 3.0 * x[0];
}""", "three")
    P, Q, S, D = op2.Dat(A), op2.Dat(A ** 2), op2.Dat(B), op2.Dat(it)
    pl = op2.ParLoop(k, it, P(op2.INC, ma), Q(op2.INC, ma), S(op2.INC, mb), D(op2.WRITE),
                     op2.Dat(it, x)(op2.READ))
    pl()
    assert pl.global_kernel.compile().strategy_used == "staged"
    p, q, s = np.zeros(na), np.zeros((na, 2)), np.zeros(nb)
    np.add.at(p, ta, x[:, None] + np.arange(3))
    np.add.at(q, ta, np.stack([x, -x], axis=1)[:, None, :])
    np.add.at(s, tb, x[:, None] * np.array([1.0, 2.0]))
    for got, want in ((P, p), (Q, q), (S, s), (D, 3.0 * x)):
        assert np.allclose(np.asarray(got.data_ro), want, rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("dim,block", [(1, True), (2, True), (2, False)])
def test_mat_increments(device, dim, block):
    """CSR and BSR Mats run in tiles, a dof-level Mat with atomics."""
    rng = np.random.default_rng(dim)
    n, nodes = 6000, 2500
    t = _mesh(n, nodes, 3, rng)
    it, ns = op2.Set(n), op2.Set(nodes)
    m = op2.Map(it, ns, 3, t)
    x = rng.random(n)
    w = 3 * dim
    k = op2.Kernel(f"""
static void outer(double *A, const double *x) {{
  for (int i = 0; i < {w}; ++i) for (int j = 0; j < {w}; ++j) A[i * {w} + j] += x[0] * (i + 1) - j;
}}""", "outer")
    sp = op2.Sparsity((ns ** dim, ns ** dim), [(m, m, None)], block_sparse=block)
    vals = {}
    for strategy in ("auto", "atomic"):
        configuration["strategy"] = strategy
        A = op2.Mat(sp, np.float64)
        pl = op2.ParLoop(k, it, A(op2.INC, (m, m)), op2.Dat(it, x)(op2.READ))
        pl()
        pl()
        A.assemble()
        staged = strategy == "auto" and (block or dim == 1)
        assert pl.global_kernel.compile().strategy_used == ("staged" if staged else "atomic")
        vals[strategy] = dev.to_host(A.device_values)
    assert np.allclose(vals["auto"], vals["atomic"], rtol=1e-12, atol=1e-11)
    local = x[:, None, None] * np.arange(1, w + 1)[:, None] - np.arange(w)
    assert abs(vals["auto"].sum() - 2 * local.sum()) <= 1e-10 * np.abs(local).sum()


@pytest.mark.parametrize("why", ["negative", "small", "spread", "subset", "rw", "capture"])
def test_loops_that_keep_the_atomic_launch(device, why):
    rng = np.random.default_rng(5)
    n, nodes = (2000, 700) if why == "small" else (30000, 9000)
    t = _mesh(n, nodes, 2, rng)
    if why == "spread":
        nodes = 2 ** 20
        t = rng.permutation(nodes)[:2 * n].reshape(n, 2).astype(np.int32)
    if why == "negative":
        t[::9, 1] = -1
    it, ns = op2.Set(n), op2.Set(nodes)
    m = op2.Map(it, ns, 2, t)
    x = rng.random(n)
    over = op2.Subset(it, np.arange(0, n, 2, dtype=np.int32)) if why == "subset" else it
    R = op2.Dat(ns)
    k = op2.Kernel("static void two(double *r, const double *x) { r[0] += x[0]; r[1] += 2.0 * x[0]; }", "two")
    args = [R(op2.RW if why == "rw" else op2.INC, m), op2.Dat(it, x)(op2.READ)]
    pl = op2.ParLoop(k, over, *args)
    passes = 1
    if why == "capture":
        torch = dev.torch()
        R.device_data_ro, [a.data._device_array() for a in pl.arguments], m.device_values
        ex = pl.global_kernel.compile()
        ex._loaded(pl, ex._flags(pl))
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            pl()
        passes = 3
        for _ in range(passes):
            g.replay()
    else:
        pl()
    assert pl.global_kernel.compile().strategy_used == ("coloured" if why == "rw" else "atomic")
    want = np.zeros(nodes)
    sel = np.arange(0, n, 2) if why == "subset" else np.arange(n)
    if why != "rw":
        ok = t[sel] >= 0
        np.add.at(want, t[sel][ok], (passes * x[sel][:, None] * np.array([1.0, 2.0]))[ok])
        assert np.allclose(np.asarray(R.data_ro), want, rtol=1e-12, atol=1e-12)


def test_tiles_in_a_captured_graph(device):
    rng = np.random.default_rng(6)
    n, nodes = 30000, 9000
    t = _mesh(n, nodes, 2, rng)
    it, ns = op2.Set(n), op2.Set(nodes)
    m = op2.Map(it, ns, 2, t)
    x = rng.random(n)
    R, X, G = op2.Dat(ns), op2.Dat(it, x), op2.Global(1, 0.0, np.float64)
    k = op2.Kernel("static void two(double *r, double *g, const double *x)"
                   " { r[0] += x[0]; r[1] += 2.0 * x[0]; g[0] += x[0]; }", "two")
    pl = op2.ParLoop(k, it, R(op2.INC, m), G(op2.INC), X(op2.READ))
    pl()
    torch = dev.torch()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        pl()
    want = np.zeros(nodes)
    np.add.at(want, t, x[:, None] * np.array([1.0, 2.0]))
    for rep in range(2, 5):
        g.replay()
        torch.cuda.synchronize()
        torch.ones(1000, device=R.device_data_ro.device).sum().item()
        assert np.allclose(dev.to_host(R._device_array()), rep * want, rtol=1e-12, atol=1e-12)
        assert abs(float(G._device_array().item()) - rep * x.sum()) <= 1e-10 * x.sum() * rep


@pytest.mark.parametrize("dtype", ["float64", "float32", "int32", "int64"])
@pytest.mark.parametrize("n", [1, 64, 4096, 4097, 256 * 2048, 256 * 2048 + 1])
def test_reduced_globals(device, dtype, n):
    """Sums, minima and maxima of one workgroup, of those that send atomics
    (16 of 256), of more, and past the grid; integers exactly."""
    ct = {"float64": "double", "float32": "float", "int32": "int", "int64": "long long"}[dtype]
    rng = np.random.default_rng(n)
    x = rng.integers(-50, 50, (n, 2)).astype(dtype)
    it = op2.Set(n)
    k = op2.Kernel(f"""
static void stats({ct} *s, {ct} *lo, {ct} *hi, const {ct} *x) {{
  s[0] += x[0]; s[1] += x[0] * x[1]; s[2] += 1;
  if (x[0] < lo[0]) lo[0] = x[0];
  if (x[1] > hi[0]) hi[0] = x[1];
}}""", "stats")
    S, lo, hi = op2.Global(3, [1, 2, 3], dtype), op2.Global(1, 40, dtype), op2.Global(1, -40, dtype)
    pl = op2.ParLoop(k, it, S(op2.INC), lo(op2.MIN), hi(op2.MAX), op2.Dat(it ** 2, x, dtype)(op2.READ))
    pl()
    pl()
    xl = x.astype(np.float64)
    want = np.array([1, 2, 3]) + 2 * np.array([xl[:, 0].sum(), (xl[:, 0] * xl[:, 1]).sum(), n])
    # every partial sum is a whole number below 2^24 in n = 4,097; above that
    # float32 sums of 2,048 workgroups are off by their roundings
    tol = 0 if dtype != "float32" or n <= 4097 else 1e-5 * np.abs(xl).max() ** 2 * n
    assert np.abs(np.asarray(S.data_ro, dtype=np.float64) - want).max() <= tol
    assert lo.data_ro[0] == min(40, x[:, 0].min()) and hi.data_ro[0] == max(-40, x[:, 1].max())
