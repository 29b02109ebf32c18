"""Workloads whose speed stands for what this framework is used for.

A case is one pass of a finite element or finite volume program through the
``op2`` interface: par_loops that scatter into Dats, par_loops that assemble
matrices, the gradient of a residual, many small meshes in one launch, kernels
that the user wrote in C, and the pattern of a new mesh.  The sizes are those of
the benchmark's configurations (256^2, 1024^2, 64^3, 32^3 and the quick set of
batched meshes), with odd and small ones beside them.

A program makes its mesh (Sets, Maps, Sparsity) once and runs many loops on
it with changing fields, so the mesh of a size is kept for all states of a
process; coordinates, fields, Dats and Mats are a state's own.
"""
import functools

import numpy as np
import torch

from pyop2_amd import elements, op2
from pyop2_amd.adjoint import P2Elasticity
from pyop2_amd.batch import BatchedLaplace
from pyop2_amd.meshes import TET_EDGES, unit_cube_tet_p2, unit_square_tri

# Screened Poisson stiffness plus mass, as a user writes it in C.
HELMHOLTZ = r"""
static void helmholtz(double A[3][3], const double X[3][2])
{
  const double a = X[1][0] - X[0][0], b = X[2][0] - X[0][0];
  const double c = X[1][1] - X[0][1], d = X[2][1] - X[0][1];
  const double det = a * d - b * c, area = 0.5 * fabs(det);
  double g[3][2];
  g[1][0] = d / det;  g[1][1] = -b / det;
  g[2][0] = -c / det; g[2][1] = a / det;
  g[0][0] = -g[1][0] - g[2][0];
  g[0][1] = -g[1][1] - g[2][1];
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j)
      A[i][j] += area * (g[i][0] * g[j][0] + g[i][1] * g[j][1] + (i == j ? 2.0 : 1.0) / 12.0);
}
"""

# Upwind advection of four tracers over the edges of a mesh: flux and update.
EDGE_FLUX = r"""
static void edge_flux(double r[2][4], const double x[2][2], const double w[2][2], const double q[2][4])
{
  const double nx = x[1][1] - x[0][1], ny = x[0][0] - x[1][0];
  const double un = 0.5 * ((w[0][0] + w[1][0]) * nx + (w[0][1] + w[1][1]) * ny);
  const double s = fabs(un);
  for (int k = 0; k < 4; ++k) {
    const double f = 0.5 * (un * (q[0][k] + q[1][k]) - s * (q[1][k] - q[0][k]));
    r[0][k] -= f;
    r[1][k] += f;
  }
}
"""
EDGE_UPDATE = r"""
static void edge_update(double *q, const double *r, double *rms)
{
  for (int k = 0; k < 4; ++k) {
    q[k] += 1e-3 * r[k];
    rms[0] += r[k] * r[k];
  }
}
"""


def listed():
    return [
        # a small loop called once a step by a program that builds the call
        # each time: the host path and one launch
        {"name": "p1 mass 32", "kind": "p1_mass", "n": 32},
        # the plain P1 residual of the 256^2 configuration, loop object kept
        {"name": "p1 residual 256", "kind": "p1_residual", "n": 256, "permute": False},
        # P1 CSR assembly, vertices numbered as an unstructured mesh numbers them
        {"name": "p1 matrix 1024 permuted", "kind": "p1_matrix", "n": 1024, "permute": True},
        # vector P2 residual of the 64^3 configuration: one operator application
        {"name": "p2 residual 64", "kind": "p2_residual", "n": 64, "dtype": "float64"},
        # residual and tangent matrix of a Newton step in one loop, added to held values
        {"name": "p2 fused 64", "kind": "p2_fused", "n": 64, "dtype": "float64", "zero": False},
        # the same in single precision at an odd size, from zero
        {"name": "p2 fused 45 f32", "kind": "p2_fused", "n": 45, "dtype": "float32", "zero": True},
        # stiffness matrix of a small cube, assembled and finalised
        {"name": "p2 matrix 11", "kind": "p2_matrix", "n": 11, "dtype": "float64"},
        # value and gradient of an objective of the residual (forward and backward)
        {"name": "p2 gradient 32", "kind": "p2_gradient", "n": 32},
        # many small meshes: assembly and residual of each in one launch
        {"name": "batched 32", "kind": "batched", "count": 32, "nmin": 16, "nmax": 128},
        # a matrix kernel of the user's own
        {"name": "user matrix 500", "kind": "user_matrix", "n": 500},
        # a time step of the user's own kernels: edge fluxes, update, residual norm
        {"name": "user step 600", "kind": "user_step", "n": 600},
        # the pattern of a new mesh
        {"name": "p2 pattern 24", "kind": "p2_pattern", "n": 24},
    ]


def draw(rng):
    def size(lo, hi):
        return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))
    kind = rng.choice(["p1_mass", "p1_residual", "p1_matrix", "p2_residual", "p2_fused", "p2_matrix",
                       "p2_gradient", "batched", "user_matrix", "user_step", "p2_pattern"])
    if kind == "p1_mass":
        return {"kind": kind, "n": size(8, 300)}
    if kind in ("p1_residual", "p1_matrix"):
        return {"kind": kind, "n": size(24, 1000), "permute": rng.random() < 0.5}
    if kind in ("p2_residual", "p2_matrix"):
        return {"kind": kind, "n": size(5, 48), "dtype": rng.choice(["float64", "float32"])}
    if kind == "p2_fused":
        return {"kind": kind, "n": size(5, 48), "dtype": rng.choice(["float64", "float32"]),
                "zero": rng.random() < 0.5}
    if kind == "p2_gradient":
        return {"kind": kind, "n": size(5, 36)}
    if kind == "batched":
        lo = size(8, 40)
        return {"kind": kind, "count": size(3, 32), "nmin": lo, "nmax": lo + size(8, 100)}
    if kind == "user_matrix":
        return {"kind": kind, "n": size(16, 700)}
    if kind == "user_step":
        return {"kind": kind, "n": size(16, 700)}
    return {"kind": kind, "n": size(4, 28)}


# ---------------------------------------------------------------------------
# Meshes: connectivity, and the op2 objects a program builds on it once

class _Tri:
    def __init__(self, n, permute):
        m = unit_square_tri(n, rng=np.random.default_rng([n, 1]), jitter=0.0, draw_u=False, permute=permute)
        self.n, self.base, self.cv = n, m.coords, m.cell_vertex
        inside = (m.coords > 0.5 / n) & (m.coords < 1.0 - 0.5 / n)
        self.inside = inside.all(axis=1)
        self.cells, self.verts = op2.Set(m.ncells), op2.Set(m.nverts)
        self.c2v = op2.Map(self.cells, self.verts, 3, m.cell_vertex)

    @functools.cached_property
    def sparsity(self):
        return op2.Sparsity((self.verts ** 1, self.verts ** 1), [(self.c2v, self.c2v, None)])

    @functools.cached_property
    def edge_vertex(self):
        n1 = self.n + 1
        v = np.arange(n1 * n1, dtype=np.int32).reshape(n1, n1)
        pairs = [(v[:, :-1], v[:, 1:]), (v[:-1, :], v[1:, :]), (v[:-1, :-1], v[1:, 1:])]
        e = np.concatenate([np.stack([a.ravel(), b.ravel()], axis=1) for a, b in pairs])
        return np.ascontiguousarray(e[np.lexsort((e[:, 1], e[:, 0]))])

    @functools.cached_property
    def e2v(self):
        return op2.Map(op2.Set(len(self.edge_vertex)), self.verts, 2, self.edge_vertex)

    def coords(self, rng):
        """Interior vertices moved by up to a fifth of a mesh width."""
        x = self.base.copy()
        x[self.inside] += rng.uniform(-0.2 / self.n, 0.2 / self.n, (int(self.inside.sum()), 2))
        return x


class _Tet:
    def __init__(self, n):
        m = unit_cube_tet_p2(n)
        self.n, self.base, self.cv, self.cn = n, m.coords, m.cell_vertex, m.cell_node
        self.inside = ((m.coords > 0.5 / n) & (m.coords < 1.0 - 0.5 / n)).all(axis=1)
        self.nnodes = m.nnodes
        self.cells, self.verts, self.nodes = op2.Set(m.ncells), op2.Set(m.nverts), op2.Set(m.nnodes)
        self.c2v = op2.Map(self.cells, self.verts, 4, m.cell_vertex)
        self.c2n = op2.Map(self.cells, self.nodes, 10, m.cell_node)

    @functools.cached_property
    def sparsity(self):
        return op2.Sparsity((self.nodes ** 3, self.nodes ** 3), [(self.c2n, self.c2n, None)])

    def coords(self, rng):
        """Interior vertices moved by up to a tenth of a mesh width."""
        x = self.base.copy()
        x[self.inside] += rng.uniform(-0.1 / self.n, 0.1 / self.n, (int(self.inside.sum()), 3))
        return x


@functools.lru_cache(maxsize=64)
def _tri(n, permute=False):
    return _Tri(n, permute)


@functools.lru_cache(maxsize=4)
def _tet(n):
    return _Tet(n)


def _batch_sizes(case):
    rng = np.random.default_rng([case["count"], case["nmin"], case["nmax"]])
    return [int(v) for v in rng.integers(case["nmin"], case["nmax"] + 1, size=case["count"])]


def _batch_meshes(case):
    return [_tri_copy(n, k) for k, n in enumerate(_batch_sizes(case))]


@functools.lru_cache(maxsize=256)
def _tri_copy(n, k):
    """Mesh ``k`` of a batch: its own Sets and Maps, also where two have one size."""
    return _Tri(n, False)


def _inputs(case, seed):
    """The host arrays of a case: made from the seed alone."""
    kind, rng = case["kind"], np.random.default_rng([int(seed), 7])
    if kind == "p2_pattern":
        # the same mesh with its nodes numbered anew
        t = _tet(case["n"])
        return t, rng.permutation(t.nnodes).astype(np.int32)[t.cn]
    if kind == "batched":
        ms = _batch_meshes(case)
        return ms, [(m.coords(rng), rng.uniform(-1.0, 1.0, len(m.base))) for m in ms]
    if kind.startswith("p2_"):
        t, dt = _tet(case["n"]), np.dtype(case.get("dtype", "float64"))
        return t, t.coords(rng).astype(dt), rng.uniform(-1.0, 1.0, (t.nnodes, 3)).astype(dt)
    m = _tri(case["n"], bool(case.get("permute", False)))
    nv = len(m.base)
    if kind == "user_step":
        return m, m.coords(rng), rng.uniform(-1.0, 1.0, (nv, 2)), rng.uniform(0.5, 1.5, (nv, 4))
    return m, m.coords(rng), rng.uniform(-1.0, 1.0, nv)


def _dat(dset, values=None, dtype=np.float64):
    d = op2.Dat(dset, values, dtype)
    d.device_data_ro  # a program's fields live on the device
    return d


# ---------------------------------------------------------------------------

def prepare(case, seed):
    kind, given = case["kind"], _inputs(case, seed)
    m = given[0]
    s = {"kind": kind, "case": case, "mesh": m}
    if kind == "p2_pattern":
        s["table"] = given[1]
    elif kind == "batched":
        pairs, s["out"] = [], []
        for t, (x, u) in zip(m, given[1]):
            X, U, R = _dat(t.verts ** 2, x), _dat(t.verts, u), _dat(t.verts)
            A = op2.Mat(t.sparsity, np.float64)
            pairs.append((op2.ParLoop(elements.p1_laplace_matrix(), t.cells, A(op2.INC, (t.c2v, t.c2v)),
                                      X(op2.READ, t.c2v)),
                          op2.ParLoop(elements.p1_laplace_residual(), t.cells, R(op2.INC, t.c2v),
                                      X(op2.READ, t.c2v), U(op2.READ, t.c2v))))
            s["out"] += [A.device_values, R.device_data_ro]
        s["batch"] = BatchedLaplace(pairs)
    elif kind == "p2_gradient":
        X, U = op2.Dat(m.verts ** 3, given[1]), op2.Dat(m.nodes ** 3, given[2])
        s["problem"] = P2Elasticity(m.cells, m.c2v, m.c2n, X, U)
        s["X"], s["u"] = X.device_data_ro, U.device_data_ro
    elif kind.startswith("p2_"):
        dt = np.dtype(case["dtype"])
        s["X"], s["u"] = _dat(m.verts ** 3, given[1], dt), _dat(m.nodes ** 3, given[2], dt)
        X, u = s["X"](op2.READ, m.c2v), s["u"](op2.READ, m.c2n)
        inc = []
        if kind != "p2_residual":
            s["A"] = op2.Mat(m.sparsity, dt)
            s["A"].device_values
            inc.append(s["A"](op2.INC, (m.c2n, m.c2n)))
        if kind != "p2_matrix":
            s["R"] = _dat(m.nodes ** 3, None, dt)
            inc.append(s["R"](op2.INC, m.c2n))
        kernel = {"p2_residual": elements.p2_elasticity_residual, "p2_matrix": elements.p2_elasticity_matrix,
                  "p2_fused": elements.p2_elasticity_fused}[kind]()
        s["loop"] = op2.ParLoop(kernel, m.cells, *inc, X, *([] if kind == "p2_matrix" else [u]))
    else:
        s["X"] = _dat(m.verts ** 2, given[1])
        if kind == "p1_mass":
            s["M"], s["kernel"] = _dat(m.verts), elements.p1_lumped_mass()
        elif kind == "p1_residual":
            s["u"], s["R"] = _dat(m.verts, given[2]), _dat(m.verts)
            s["loop"] = op2.ParLoop(elements.p1_laplace_residual(), m.cells, s["R"](op2.INC, m.c2v),
                                    s["X"](op2.READ, m.c2v), s["u"](op2.READ, m.c2v))
        elif kind in ("p1_matrix", "user_matrix"):
            s["A"] = op2.Mat(m.sparsity, np.float64)
            s["A"].device_values
            kernel = elements.p1_laplace_matrix() if kind == "p1_matrix" else op2.Kernel(HELMHOLTZ, "helmholtz")
            s["loop"] = op2.ParLoop(kernel, m.cells, s["A"](op2.INC, (m.c2v, m.c2v)), s["X"](op2.READ, m.c2v))
        else:
            s["w"], s["q"] = _dat(m.verts ** 2, given[2]), _dat(m.verts ** 4, given[3])
            s["r"], s["rms"] = _dat(m.verts ** 4), op2.Global(1, 0.0, np.float64)
            s["flux"] = op2.ParLoop(op2.Kernel(EDGE_FLUX, "edge_flux"), m.e2v.iterset, s["r"](op2.INC, m.e2v),
                                    s["X"](op2.READ, m.e2v), s["w"](op2.READ, m.e2v), s["q"](op2.READ, m.e2v))
            s["update"] = op2.ParLoop(op2.Kernel(EDGE_UPDATE, "edge_update"), m.verts, s["q"](op2.RW),
                                      s["r"](op2.READ), s["rms"](op2.INC))
    return s


def run(s):
    kind, m = s["kind"], s["mesh"]
    if kind == "p1_mass":
        s["M"].zero()
        op2.par_loop(s["kernel"], m.cells, s["M"](op2.INC, m.c2v), s["X"](op2.READ, m.c2v))
        return s["M"].device_data_ro
    if kind in ("p1_residual", "p2_residual"):
        s["R"].zero()
        s["loop"]()
        return s["R"].device_data_ro
    if kind == "p1_matrix":
        s["A"].zero()
        s["loop"]()
        return s["A"].device_values
    if kind in ("p2_matrix", "user_matrix"):
        s["A"].zero()
        s["loop"]()
        s["A"].assemble()
        return s["A"].device_values
    if kind == "p2_fused":
        if s["case"]["zero"]:
            s["A"].zero()
            s["R"].zero()
        s["loop"]()
        return s["A"].device_values, s["R"].device_data_ro
    if kind == "p2_gradient":
        u, X = s["u"].detach().requires_grad_(), s["X"].detach().requires_grad_()
        J = s["problem"].objective(u, X)
        J.backward()
        return J.detach(), u.grad, X.grad
    if kind == "batched":
        s["batch"]()
        return s["out"]
    if kind == "user_step":
        s["r"].zero()
        s["rms"].zero()
        s["flux"]()
        s["update"]()
        return s["q"].device_data_ro, s["r"].device_data_ro, s["rms"].device_data_ro
    nodes = op2.Set(m.nnodes)
    cells = op2.Set(len(s["table"]))
    c2n = op2.Map(cells, nodes, 10, s["table"])
    return list(op2.Sparsity((nodes ** 3, nodes ** 3), [(c2n, c2n, None)]).block_pattern)


# ---------------------------------------------------------------------------
# What a pass cannot do without

def _tri_nnz(n):
    return (n + 1) ** 2 + 2 * (3 * n * n + 2 * n)


def _tet_counts(n):
    """Vertices, P2 nodes and P2 block non-zeros of the cube of n^3 hexes."""
    nv = (n + 1) ** 3
    edges = 3 * n * (n + 1) ** 2 + 3 * n * n * (n + 1) + n ** 3
    faces = 12 * n ** 3 + 6 * n * n
    tets = 6 * n ** 3
    # node pairs that share a tetrahedron: those of a common edge (vertex and
    # vertex, vertex and midpoint), of a common face (vertex and the opposite
    # edge, two edges) and of a tetrahedron alone (opposite edges)
    pairs = edges * 3 + faces * 6 + tets * 3
    return nv, nv + edges, nv + edges + 2 * pairs


def work(case):
    kind = case["kind"]
    if kind == "batched":
        ns = _batch_sizes(case)
        b = sum(2 * n * n * 12 + (n + 1) ** 2 * (16 + 8 + 16 + 4) + _tri_nnz(n) * 20 for n in ns)
        return {"bytes": b, "flops": sum(2 * n * n * 100 for n in ns)}
    n = case["n"]
    if kind.startswith("p2_"):
        nv, nn, nnz = _tet_counts(n)
        nc, it = 6 * n ** 3, np.dtype(case.get("dtype", "float64")).itemsize
        maps, x, u = nc * 56, nv * 3 * it, nn * 3 * it
        if kind == "p2_pattern":
            return {"bytes": nc * 40 + (nn + 1) * 4 + nnz * 4, "flops": 0}
        if kind == "p2_residual":
            return {"bytes": maps + x + 2 * u, "flops": nc * 1100}
        if kind == "p2_gradient":
            return {"bytes": 2 * maps + 3 * x + 5 * u, "flops": nc * 4000}
        held = 0 if kind == "p2_matrix" or case["zero"] else 1
        mat = nnz * 9 * it * (1 + held) + nnz * 4 + (nn + 1) * 4 + maps + x
        if kind == "p2_matrix":
            return {"bytes": mat, "flops": nc * 4500}
        return {"bytes": mat + u * (2 + held), "flops": nc * 5600}
    nc, nv = 2 * n * n, (n + 1) ** 2
    if kind == "p1_mass":
        return {"bytes": nc * 12 + nv * 24, "flops": nc * 12}
    if kind == "p1_residual":
        return {"bytes": nc * 12 + nv * 32, "flops": nc * 50}
    if kind == "user_step":
        ne = 3 * n * n + 2 * n
        return {"bytes": ne * 8 + nv * (16 + 16 + 32 + 32 + 32), "flops": ne * 45 + nv * 16}
    return {"bytes": nc * 12 + nv * (16 + 4) + _tri_nnz(n) * 12, "flops": nc * 60}


# ---------------------------------------------------------------------------
# The same in plain torch, 64 bits

def _to(a, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a)).to("cuda" if torch.cuda.is_available() else "cpu")
    return t if dtype is None else t.to(dtype)


def _scatter(n, index, values):
    out = torch.zeros((n,) + tuple(values.shape[2:]), dtype=torch.float64, device=values.device)
    return out.index_add(0, index.reshape(-1), values.reshape((-1,) + tuple(values.shape[2:])))


def _tri_terms(x, cv):
    """Gradients of the vertex functions and areas."""
    p = x[cv]
    e = p[:, [2, 0, 1]] - p[:, [1, 2, 0]]
    det = e[:, 2, 0] * e[:, 0, 1] - e[:, 2, 1] * e[:, 0, 0]
    g = torch.stack([-e[..., 1], e[..., 0]], dim=2) / det[:, None, None]
    return g, 0.5 * det.abs()


def _csr_values(n, cv, local):
    """Values in CSR order of element matrices ``local`` (cells, k, k, ...)."""
    keys = cv[:, :, None] * n + cv[:, None, :]
    pattern = torch.unique(torch.cat([keys.reshape(-1), torch.arange(n, device=cv.device) * (n + 1)]))
    return pattern, torch.searchsorted(pattern, keys.reshape(-1)).reshape(keys.shape)


def _p2_derivatives(device):
    """d phi_i / d lambda_m at the four points of the degree 2 rule."""
    d = torch.zeros((4, 10, 4), dtype=torch.float64)
    for q in range(4):
        bary = [0.5854101966249685 if q == m else 0.1381966011250105 for m in range(4)]
        for i in range(4):
            d[q, i, i] = 4.0 * bary[i] - 1.0
        for k, (a, b) in enumerate(TET_EDGES):
            d[q, 4 + k, a], d[q, 4 + k, b] = 4.0 * bary[b], 4.0 * bary[a]
    return d.to(device)


def _p2_gradients(x, cv, d):
    """Basis gradients (cells, point, basis, 3) and quadrature weights."""
    p = x[cv]
    jac = (p[:, 1:] - p[:, :1]).transpose(1, 2)
    inv = torch.linalg.inv(jac)
    gl = torch.cat([-inv.sum(dim=1, keepdim=True), inv], dim=1)
    return torch.einsum("qim,cmk->cqik", d, gl), torch.linalg.det(jac).abs() / 24.0


def _p2_element_residual(x, u, cv, cn, d, lam=1.0, mu=0.5):
    g, w = _p2_gradients(x, cv, d)
    gu = torch.einsum("cib,cqik->cqbk", u[cn], g)
    eye = torch.eye(3, dtype=x.dtype, device=x.device)
    s = mu * (gu + gu.transpose(2, 3)) + lam * gu.diagonal(dim1=2, dim2=3).sum(-1)[..., None, None] * eye
    return torch.einsum("c,cqak,cqik->cia", w, s, g)


def _p2_exact(case, t, x, u, lam=1.0, mu=0.5):
    cv, cn, x, u = _to(t.cv, torch.int64), _to(t.cn, torch.int64), _to(x, torch.float64), _to(u, torch.float64)
    d, n, step = _p2_derivatives(x.device), t.nnodes, 32768
    R = A = None
    if case["kind"] != "p2_matrix":
        R = torch.zeros((n, 3), dtype=torch.float64, device=x.device)
        for lo in range(0, len(cv), step):
            e = _p2_element_residual(x, u, cv[lo:lo + step], cn[lo:lo + step], d, lam, mu)
            R.index_add_(0, cn[lo:lo + step].reshape(-1), e.reshape(-1, 3))
    if case["kind"] != "p2_residual":
        pattern = torch.unique((cn[:, :, None] * n + cn[:, None, :]).reshape(-1))
        A = torch.zeros((len(pattern), 3, 3), dtype=torch.float64, device=x.device)
        eye = torch.eye(3, dtype=x.dtype, device=x.device)
        for lo in range(0, len(cv), step):
            c = cn[lo:lo + step]
            g, w = _p2_gradients(x, cv[lo:lo + step], d)
            M = torch.einsum("c,cqia,cqjb->cijab", w, g, g)
            tr = M.diagonal(dim1=3, dim2=4).sum(-1)
            K = lam * M + mu * M.transpose(3, 4) + mu * tr[..., None, None] * eye
            at = torch.searchsorted(pattern, (c[:, :, None] * n + c[:, None, :]).reshape(-1))
            A.index_add_(0, at, K.reshape(-1, 3, 3))
        A = A.reshape(-1)
    return {"p2_residual": R, "p2_matrix": A, "p2_fused": (A, R)}[case["kind"]]


def exact(case, seed):
    kind, given = case["kind"], _inputs(case, seed)
    if kind == "p2_pattern":
        return None  # whole numbers only
    m = given[0]
    if kind == "batched":
        out = []
        for t, (x, u) in zip(m, given[1]):
            cv, x, u = _to(t.cv, torch.int64), _to(x), _to(u)
            g, area = _tri_terms(x, cv)
            K = area[:, None, None] * torch.einsum("cia,cja->cij", g, g)
            pattern, at = _csr_values(len(x), cv, K)
            out += [_scatter(len(pattern), at, K[..., None].reshape(len(cv), 9)),
                    _scatter(len(x), cv, torch.einsum("cij,cj->ci", K, u[cv]))]
        return out
    if kind == "p2_gradient":
        t, x, u = given[0], _to(given[1]).requires_grad_(), _to(given[2]).requires_grad_()
        cv, cn = _to(t.cv, torch.int64), _to(t.cn, torch.int64)
        e = _p2_element_residual(x, u, cv, cn, _p2_derivatives(x.device))
        J = 0.5 * _scatter(t.nnodes, cn, e).square().sum()
        J.backward()
        return J.detach(), u.grad, x.grad
    if kind.startswith("p2_"):
        return _p2_exact(case, *given)
    x, nv = _to(given[1]), len(m.base)
    if kind == "user_step":
        ev, w, q = _to(m.edge_vertex, torch.int64), _to(given[2]), _to(given[3])
        dx = x[ev[:, 1]] - x[ev[:, 0]]
        wm = 0.5 * (w[ev[:, 0]] + w[ev[:, 1]])
        un = (wm[:, 0] * dx[:, 1] - wm[:, 1] * dx[:, 0])[:, None]
        q0, q1 = q[ev[:, 0]], q[ev[:, 1]]
        f = 0.5 * (un * (q0 + q1) - un.abs() * (q1 - q0))
        r = _scatter(nv, ev, torch.stack([-f, f], dim=1))
        return q + 1e-3 * r, r, r.square().sum().reshape(1)
    cv = _to(m.cv, torch.int64)
    g, area = _tri_terms(x, cv)
    if kind == "p1_mass":
        return _scatter(nv, cv, (area / 3.0)[:, None].expand(-1, 3))
    K = area[:, None, None] * torch.einsum("cia,cja->cij", g, g)
    if kind == "p1_residual":
        return _scatter(nv, cv, torch.einsum("cij,cj->ci", K, _to(given[2])[cv]))
    if kind == "user_matrix":
        K = K + area[:, None, None] * (1.0 + torch.eye(3, dtype=x.dtype, device=x.device)) / 12.0
    pattern, at = _csr_values(nv, cv, K)
    return _scatter(len(pattern), at.reshape(len(cv), 9), K.reshape(len(cv), 9))
