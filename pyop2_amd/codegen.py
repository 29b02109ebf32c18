"""Generated gather/compute/scatter kernels for arbitrary C-string kernels.

For a local kernel with no hand-written implementation, the executor emits
one HIP kernel per GlobalKernel signature: each work-item takes one
iteration element ``n`` and follows the reference wrapper's per-element
semantics (``pyop2/codegen/builder.py``):

* indirect Dat READ/RW/MIN/MAX arguments are gathered into private buffers
  ``buf[i*dim + j] = dat[map[n][i]*dim + j]``; INC/WRITE buffers start at
  zero; direct Dats pass ``&dat[n*dim]``;
* Globals: READ passes the device array; INC uses a zeroed buffer and
  MIN/MAX a copy, reduced over the workgroup (``_REDUCE_BLOCKS``);
* Mats: a zeroed ``(ar_r*rdim) x (ar_c*cdim)`` buffer, added (INC) or
  stored (WRITE) block by block at the slot found by binary search of the
  row's sorted column indices;
* the user's C function is compiled unchanged as a device function
  (``#pragma clang force_cuda_host_device``) and called with pointer
  adaptors that convert to whatever pointer types it declares;
* unpack: INC adds (device-scope atomics, or plain adds inside a colour),
  MIN/MAX atomic min/max, WRITE/RW stores.

Indirect WRITE/RW arguments and Mat WRITE need exclusive targets, so such
loops run coloured (greedy colouring, one launch per colour); INC-only
loops run with atomics, or in tiles (``_tiles``): a workgroup adds the
increments of consecutive elements up in LDS, writes one partial sum per
distinct target, and a second pass adds a target's partial sums.  Sources
are compiled for gfx950 with hiprtc and the code objects cached in memory
and under ``<cache_dir>/hip``.
"""
import ctypes
import hashlib
import operator
import os
import re
import threading

import numpy as np

from pyop2_amd import device as dev
from pyop2_amd.configuration import configuration
from pyop2_amd.datatypes import as_cstr
from pyop2_amd.exceptions import CompilationError
from pyop2_amd.global_kernel import (DatKernelArg, GlobalKernelArg, MatKernelArg, MixedDatKernelArg,
                                     MixedMatKernelArg)
from pyop2_amd.types import region as reg
from pyop2_amd.types.access import INC, MAX, MIN, READ, RW, WRITE
from pyop2_amd.types.set import Subset

__all__ = ["GeneratedKernel", "generate_source", "compile_options"]

_PRELUDE = r"""
typedef signed char int8_t;
typedef unsigned char uint8_t;
typedef short int16_t;
typedef unsigned short uint16_t;
typedef int int32_t;
typedef unsigned int uint32_t;
typedef long long int64_t;
typedef unsigned long long uint64_t;
#define restrict __restrict__

/* Converts to any pointer type a user kernel declares for an argument. */
struct op2_ptr_ {
  void *p;
  template <typename U> __host__ __device__ operator U *() const { return static_cast<U *>(p); }
};

template <typename T> __device__ inline void op2_atomic_add(T *p, T v) { atomicAdd(p, v); }
__device__ inline void op2_atomic_add(int64_t *p, int64_t v) {
  atomicAdd(reinterpret_cast<unsigned long long *>(p), static_cast<unsigned long long>(v));
}
__device__ inline void op2_atomic_add(uint64_t *p, uint64_t v) {
  atomicAdd(reinterpret_cast<unsigned long long *>(p), static_cast<unsigned long long>(v));
}
template <typename T> __device__ inline void op2_atomic_min(T *p, T v) { atomicMin(p, v); }
template <typename T> __device__ inline void op2_atomic_max(T *p, T v) { atomicMax(p, v); }
__device__ inline void op2_atomic_min(int64_t *p, int64_t v) { atomicMin(reinterpret_cast<long long *>(p), (long long)v); }
__device__ inline void op2_atomic_max(int64_t *p, int64_t v) { atomicMax(reinterpret_cast<long long *>(p), (long long)v); }
__device__ inline void op2_atomic_min(uint64_t *p, uint64_t v) { atomicMin(reinterpret_cast<unsigned long long *>(p), (unsigned long long)v); }
__device__ inline void op2_atomic_max(uint64_t *p, uint64_t v) { atomicMax(reinterpret_cast<unsigned long long *>(p), (unsigned long long)v); }
__device__ inline void op2_atomic_min(double *p, double v) {
  unsigned long long *a = reinterpret_cast<unsigned long long *>(p);
  unsigned long long old = *a, assumed;
  while (__longlong_as_double(old) > v) {
    assumed = old;
    old = atomicCAS(a, assumed, __double_as_longlong(v));
    if (old == assumed) break;
  }
}
__device__ inline void op2_atomic_max(double *p, double v) {
  unsigned long long *a = reinterpret_cast<unsigned long long *>(p);
  unsigned long long old = *a, assumed;
  while (__longlong_as_double(old) < v) {
    assumed = old;
    old = atomicCAS(a, assumed, __double_as_longlong(v));
    if (old == assumed) break;
  }
}
__device__ inline void op2_atomic_min(float *p, float v) {
  unsigned int *a = reinterpret_cast<unsigned int *>(p);
  unsigned int old = *a, assumed;
  while (__uint_as_float(old) > v) {
    assumed = old;
    old = atomicCAS(a, assumed, __float_as_uint(v));
    if (old == assumed) break;
  }
}
__device__ inline void op2_atomic_max(float *p, float v) {
  unsigned int *a = reinterpret_cast<unsigned int *>(p);
  unsigned int old = *a, assumed;
  while (__uint_as_float(old) < v) {
    assumed = old;
    old = atomicCAS(a, assumed, __float_as_uint(v));
    if (old == assumed) break;
  }
}
template <typename T> __device__ inline T op2_min(T a, T b) { return b < a ? b : a; }
template <typename T> __device__ inline T op2_max(T a, T b) { return b > a ? b : a; }

template <typename T> __device__ inline T op2_wave_sum(T v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
template <typename T> __device__ inline T op2_wave_min(T v) {
  for (int o = 32; o > 0; o >>= 1) v = op2_min(v, (T)__shfl_xor(v, o, 64));
  return v;
}
template <typename T> __device__ inline T op2_wave_max(T v) {
  for (int o = 32; o > 0; o >>= 1) v = op2_max(v, (T)__shfl_xor(v, o, 64));
  return v;
}

/* Remainder of a periodic column's layer offset, a in [0, 2n). */
__device__ inline int32_t op2_rem(int32_t a, int32_t n) { return a < n ? a : a - n; }

__device__ inline int32_t op2_find_slot(const int32_t *__restrict__ rowptr,
                                         const int32_t *__restrict__ colidx,
                                         int32_t row, int32_t col) {
  int32_t l = rowptr[row], h = rowptr[row + 1] - 1;
  while (l <= h) {
    const int32_t m = l + ((h - l) >> 1);
    const int32_t c = colidx[m];
    if (c == col) return m;
    if (c < col) l = m + 1; else h = m - 1;
  }
  return -1;
}
"""

_STD_HEADER = re.compile(r'^\s*#\s*include\s*<(math|stdlib|stdio|string|stdint|stdbool|float|limits|complex|inttypes|stddef|assert)\.h>\s*$',
                         re.M)

# Integer types without wavefront shuffles / atomics (Global reductions refused).
_SHUFFLE_T = {"int8_t": "int32_t", "uint8_t": "uint32_t", "int16_t": "int32_t",
              "uint16_t": "uint32_t"}


def compile_options():
    return ["--offload-arch=gfx950", "-O3", "-std=c++17", "-munsafe-fp-atomics",
            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def _strip_headers(text):
    return _STD_HEADER.sub("", text)


def _kernel_maps(garg):
    """MapKernelArgs of a kernel argument in the order of its parloop
    argument's ``maps``."""
    if isinstance(garg, DatKernelArg):
        return (garg.map_,) if garg.map_ is not None else ()
    if isinstance(garg, MatKernelArg):
        return tuple(garg.maps)
    if isinstance(garg, (MixedDatKernelArg, MixedMatKernelArg)):
        return tuple(garg.maps)
    return ()


def _dat_store(acc, tgt, val):
    """Statement storing a Dat pack entry ``val`` into ``tgt`` for ``acc``
    (atomic when the launch is not coloured)."""
    if acc == INC:
        return f"if (atomic) op2_atomic_add(&{tgt}, {val}); else {tgt} += {val};"
    if acc == MIN:
        return f"if (atomic) op2_atomic_min(&{tgt}, {val}); else {tgt} = op2_min({tgt}, {val});"
    if acc == MAX:
        return f"if (atomic) op2_atomic_max(&{tgt}, {val}); else {tgt} = op2_max({tgt}, {val});"
    return f"{tgt} = {val};"


def _region_bounds(region, periodic=False):
    """C expressions of the first and one-past-last layer a column runs in
    ``region``, from its ``bottom_`` and cell end ``cend_``
    (``builder.py:771-795``; a column with no cells runs no top cell; a
    periodic column has as many interior facets as cells)."""
    region = reg.normalise(region)
    if region == reg.ON_INTERIOR_FACETS and periodic:
        return "bottom_", "cend_"
    if region == reg.ON_BOTTOM:
        return "bottom_", "bottom_ + 1"
    if region == reg.ON_TOP:
        return "(cend_ - 1 > bottom_ ? cend_ - 1 : bottom_)", "cend_"
    if region == reg.ON_INTERIOR_FACETS:
        return "bottom_", "cend_ - 1"
    return "bottom_", "cend_"


def generate_source(gk, map_index, block_flags=None, tiled=None):
    """HIP source of the wrapper kernel ``op2_wrap`` for GlobalKernel ``gk``.

    ``map_index[(arg, j)]`` is the position of an argument's j-th map in the
    unique-map list; ``block_flags[arg]`` says whether a Mat argument is
    stored as BSR (else scalar CSR over dofs).  ``tiled`` (argument -> plan
    number) makes the tiled form: the increments of those arguments go to
    LDS accumulators through the plan's local ids and leave the workgroup as
    partial sums.
    """
    block_flags = block_flags or {}
    tiled = tiled or {}
    lk = gk.local_kernel
    extruded = getattr(gk, "_extruded", False)
    region = getattr(gk, "_iteration_region", None) if extruded else None
    # interior facets: every map names the cell below, then the cell above
    nf = reg.facet_factor(region)
    periodic = extruded and bool(getattr(gk, "_extruded_periodic", False))
    # map offsets per unique map (extruded maps step by offset[i] per layer)
    # and, on a periodic set, their offset quotients
    offsets, quots = {}, {}
    for k, garg in enumerate(gk.arguments):
        for j, mk in enumerate(_kernel_maps(garg)):
            if mk.offset is not None and extruded:
                offsets[map_index[(k, j)]] = mk.offset
                if periodic and mk.offset_quotient is not None:
                    quots[map_index[(k, j)]] = mk.offset_quotient

    def _step(m, ar, i, f):
        """Layer offset of entry ``i`` of map ``m``: the cells above the
        column's bottom (``f`` adds the cell above), wrapped on a periodic
        set (``builder.py:103-121``)."""
        st = "lyr_" if f is None else f"(lyr_ + {f})"
        if not periodic:
            return st
        if m not in quots:
            return f"op2_rem({st}, nl_)"
        return f"(op2_rem({st} + quo{m}[{i}], nl_) - op2_rem(quo{m}[{i}], nl_))"

    def _mv(m, ar, i):
        """Entry ``i`` of unique map ``m`` (arity ``ar``) for element ``n``
        (and layer); with interior facets ``i`` runs over ``2 * ar`` entries,
        the cell below first (``builder.py:81-129``)."""
        if nf == 1:
            base = f"map{m}[(int64_t)n * {ar} + {i}]"
            if m in offsets:
                return f"(({base}) >= 0 ? ({base}) + off{m}[{i}] * {_step(m, ar, i, None)} : -1)"
            return base
        if m not in offsets:
            raise ValueError("ON_INTERIOR_FACETS needs extruded maps (maps with an offset)")
        i_ = f"({i}) % {ar}"
        base = f"map{m}[(int64_t)n * {ar} + {i_}]"
        return f"(({base}) >= 0 ? ({base}) + off{m}[{i_}] * {_step(m, ar, i_, f'({i}) / {ar}')} : -1)"
    headers = "\n".join(_strip_headers(h) for h in lk.headers)
    code = _strip_headers(lk.code)
    params = ["int32_t lo", "int32_t hi", "const int32_t *__restrict__ list", "int32_t atomic"]
    pre, call, post, red = [], [], [], []
    accs = []            # (argument, plan, values per target) of the tiled form
    reduced = []         # (argument, element type, components, operation) of the reduced Globals
    nmaps = len(set(map_index.values()))
    for k, (larg, garg) in enumerate(zip(lk.arguments, gk.arguments)):
        acc = larg.access
        t = as_cstr(np.dtype(larg.dtype))
        if isinstance(garg, DatKernelArg):
            dim = int(np.prod(garg.dim))
            # a DatView passes one component: stride dim, offset comp, width 1
            # (builder.py:303-410, view_index)
            comp = 0 if garg.index is None else int(np.ravel_multi_index(garg.index, garg.dim))
            stride, dim = dim, (dim if garg.index is None else 1)
            params.append(f"{t} *__restrict__ arg{k}")
            if garg.map_ is None:
                call.append(f"op2_ptr_{{(void *)(arg{k} + (int64_t)n * {stride} + {comp})}}")
                continue
            m = map_index[(k, 0)]
            ar = garg.map_.arity
            ear = nf * ar
            pre.append(f"    int32_t mi{k}[{ear}];")
            pre.append(f"    for (int i = 0; i < {ear}; ++i) mi{k}[i] = {_mv(m, ar, 'i')};")
            pre.append(f"    {t} buf{k}[{ear * dim}];")
            if acc in (INC, WRITE):
                pre.append(f"    for (int q = 0; q < {ear * dim}; ++q) buf{k}[q] = ({t})0;")
            else:
                pre.append(f"    for (int i = 0; i < {ear}; ++i) for (int j = 0; j < {dim}; ++j)"
                           f" buf{k}[i * {dim} + j] = mi{k}[i] >= 0 ? arg{k}[(int64_t)mi{k}[i] * {stride} + {comp} + j] : ({t})0;")
            call.append(f"op2_ptr_{{(void *)buf{k}}}")
            if acc == READ:
                continue
            if k in tiled:
                accs.append((k, tiled[k], dim))
                post.append(f"    for (int i = 0; i < {ar}; ++i) {{ const int l_ = loc{tiled[k]}_[(int64_t)(n - base_) * {ar} + i];"
                            f" for (int j = 0; j < {dim}; ++j) op2_atomic_add(&acc{k}_[l_ * {dim} + j],"
                            f" ({_acc_type(t)})buf{k}[i * {dim} + j]); }}")
                continue
            tgt = f"arg{k}[(int64_t)mi{k}[i] * {stride} + {comp} + j]"
            val = f"buf{k}[i * {dim} + j]"
            post.append(f"    for (int i = 0; i < {ear}; ++i) {{ if (mi{k}[i] < 0) continue;"
                        f" for (int j = 0; j < {dim}; ++j) {{ {_dat_store(acc, tgt, val)} }} }}")
        elif isinstance(garg, GlobalKernelArg):
            dim = int(np.prod(garg.dim)) if len(garg.dim) else 1
            params.append(f"{t} *__restrict__ arg{k}")
            if acc == READ:
                call.append(f"op2_ptr_{{(void *)arg{k}}}")
                continue
            # a buffer per element, as for the other outputs, added to the
            # thread's result after it
            start = f"({t})0" if acc == INC else f"arg{k}[q]"
            join = {INC: "sum{k}_[q] + buf{k}[q]", MIN: "op2_min(sum{k}_[q], buf{k}[q])",
                    MAX: "op2_max(sum{k}_[q], buf{k}[q])"}.get(acc, "").format(k=k)
            red.append((f"  {t} sum{k}_[{dim}];\n  for (int q = 0; q < {dim}; ++q) sum{k}_[q] = {start};",
                        f"    {t} buf{k}[{dim}];\n    for (int q = 0; q < {dim}; ++q) buf{k}[q] = {start};",
                        f"    for (int q = 0; q < {dim}; ++q) sum{k}_[q] = {join};"))
            call.append(f"op2_ptr_{{(void *)buf{k}}}")
            fn = {INC: "sum", MIN: "min", MAX: "max"}.get(acc)
            if fn is None:
                raise NotImplementedError(f"Global access {acc!r} in a par_loop")
            if t in _SHUFFLE_T:
                raise NotImplementedError(f"Global reductions of {t} are not supported on the device")
            reduced.append((k, t, dim, fn))
        elif isinstance(garg, MixedDatKernelArg):
            # one buffer: the packs of the components one after the other
            comps = garg.arguments
            total = sum(nf * c.map_.arity * int(np.prod(c.dim)) for c in comps)
            pre.append(f"    {t} buf{k}[{total}];")
            if acc in (INC, WRITE):
                pre.append(f"    for (int q = 0; q < {total}; ++q) buf{k}[q] = ({t})0;")
            off = 0
            for c, comp in enumerate(comps):
                dim, ar, m = int(np.prod(comp.dim)), comp.map_.arity, map_index[(k, c)]
                ear = nf * ar
                a_, mi_ = f"arg{k}_{c}", f"mi{k}_{c}"
                params.append(f"{t} *__restrict__ {a_}")
                pre.append(f"    int32_t {mi_}[{ear}];")
                pre.append(f"    for (int i = 0; i < {ear}; ++i) {mi_}[i] = {_mv(m, ar, 'i')};")
                if acc not in (INC, WRITE):
                    pre.append(f"    for (int i = 0; i < {ear}; ++i) for (int j = 0; j < {dim}; ++j)"
                               f" buf{k}[{off} + i * {dim} + j] = {mi_}[i] >= 0 ?"
                               f" {a_}[(int64_t){mi_}[i] * {dim} + j] : ({t})0;")
                if acc != READ:
                    tgt = f"{a_}[(int64_t){mi_}[i] * {dim} + j]"
                    val = f"buf{k}[{off} + i * {dim} + j]"
                    post.append(f"    for (int i = 0; i < {ear}; ++i) {{ if ({mi_}[i] < 0) continue;"
                                f" for (int j = 0; j < {dim}; ++j) {{ {_dat_store(acc, tgt, val)} }} }}")
                off += ear * dim
            call.append(f"op2_ptr_{{(void *)buf{k}}}")
        elif isinstance(garg, MixedMatKernelArg):
            # one element matrix; block (i, j) is rows of row component i
            # times columns of column component j, added into block Mat (i, j)
            nr, nc = garg.shape
            blocks = garg.arguments
            rds = [blocks[i * nc].dims[0][0][0] for i in range(nr)]
            cds = [blocks[j].dims[0][0][1] for j in range(nc)]
            rars = [nf * blocks[i * nc].maps[0].arity for i in range(nr)]
            cars = [nf * blocks[j].maps[1].arity for j in range(nc)]
            roff = [sum(rars[q] * rds[q] for q in range(i)) for i in range(nr)]
            coff = [sum(cars[q] * cds[q] for q in range(j)) for j in range(nc)]
            NR, NC = roff[-1] + rars[-1] * rds[-1], coff[-1] + cars[-1] * cds[-1]
            pre.append(f"    {t} buf{k}[{NR * NC}];")
            pre.append(f"    for (int q = 0; q < {NR * NC}; ++q) buf{k}[q] = ({t})0;")
            call.append(f"op2_ptr_{{(void *)buf{k}}}")
            flags = block_flags.get(k) or (False,) * (nr * nc)
            store = ("if (atomic) op2_atomic_add(&{tgt}, {val}); else {tgt} += {val};" if acc == INC
                     else "{tgt} = {val};")
            for i in range(nr):
                for j in range(nc):
                    b = i * nc + j
                    rd, cd, rar, car = rds[i], cds[j], rars[i], cars[j]
                    rm, cm = map_index[(k, i)], map_index[(k, nr + j)]
                    params += [f"const int32_t *__restrict__ rowptr{k}_{b}",
                               f"const int32_t *__restrict__ colidx{k}_{b}", f"{t} *__restrict__ arg{k}_{b}"]
                    val = f"buf{k}[({roff[i]} + ii * {rd} + ri) * {NC} + {coff[j]} + jj * {cd} + cj]"
                    # flags[b]: True = BSR block Mat; False = scalar CSR;
                    # ("offset", r0, c0) = block of a monolithic Mat, rows and
                    # columns shifted by its offsets in the parent's CSR
                    shift = flags[b] if isinstance(flags[b], tuple) else ("offset", 0, 0)
                    if flags[b] is True:
                        tgt = f"arg{k}_{b}[(int64_t)s_ * {rd * cd} + ri * {cd} + cj]"
                        post.append(
                            f"    for (int ii = 0; ii < {rar}; ++ii) {{ const int32_t r_ = {_mv(rm, rar // nf, 'ii')}; if (r_ < 0) continue;\n"
                            f"      for (int jj = 0; jj < {car}; ++jj) {{ const int32_t c_ = {_mv(cm, car // nf, 'jj')}; if (c_ < 0) continue;\n"
                            f"        const int32_t s_ = op2_find_slot(rowptr{k}_{b}, colidx{k}_{b}, r_, c_); if (s_ < 0) {{ atomicAdd(status, 1); continue; }}\n"
                            f"        for (int ri = 0; ri < {rd}; ++ri) for (int cj = 0; cj < {cd}; ++cj) {{ {store.format(tgt=tgt, val=val)} }} }} }}")
                    else:
                        tgt = f"arg{k}_{b}[s_]"
                        post.append(
                            f"    for (int ii = 0; ii < {rar}; ++ii) {{ const int32_t r_ = {_mv(rm, rar // nf, 'ii')}; if (r_ < 0) continue;\n"
                            f"      for (int ri = 0; ri < {rd}; ++ri) for (int jj = 0; jj < {car}; ++jj) {{ const int32_t c_ = {_mv(cm, car // nf, 'jj')}; if (c_ < 0) continue;\n"
                            f"        for (int cj = 0; cj < {cd}; ++cj) {{ const int32_t s_ = op2_find_slot(rowptr{k}_{b}, colidx{k}_{b}, {shift[1]} + r_ * {rd} + ri, {shift[2]} + c_ * {cd} + cj);"
                            f" if (s_ < 0) {{ atomicAdd(status, 1); continue; }} {store.format(tgt=tgt, val=val)} }} }} }}")
        elif isinstance(garg, MatKernelArg):
            rd, cd = garg.dims[0][0]
            params += [f"const int32_t *__restrict__ rowptr{k}", f"const int32_t *__restrict__ colidx{k}",
                       f"{t} *__restrict__ arg{k}"]
            rm, cm = map_index[(k, 0)], map_index[(k, 1)]
            rar, car = nf * garg.maps[0].arity, nf * garg.maps[1].arity
            ncol = car * cd
            pre.append(f"    {t} buf{k}[{rar * rd * ncol}];")
            pre.append(f"    for (int q = 0; q < {rar * rd * ncol}; ++q) buf{k}[q] = ({t})0;")
            call.append(f"op2_ptr_{{(void *)buf{k}}}")
            block = bool(block_flags.get(k, False))
            if acc == INC:
                store = "if (atomic) op2_atomic_add(&{tgt}, {val}); else {tgt} += {val};"
            else:
                store = "{tgt} = {val};"
            if k in tiled:
                # targets are the blocks of the pattern, one local id per (i, j)
                accs.append((k, tiled[k], rd * cd))
                post.append(
                    f"    for (int i = 0; i < {rar}; ++i) for (int j = 0; j < {car}; ++j) {{"
                    f" const int l_ = loc{tiled[k]}_[(int64_t)(n - base_) * {rar * car} + i * {car} + j];"
                    f" for (int ri = 0; ri < {rd}; ++ri) for (int cj = 0; cj < {cd}; ++cj)"
                    f" op2_atomic_add(&acc{k}_[l_ * {rd * cd} + ri * {cd} + cj],"
                    f" ({_acc_type(t)})buf{k}[(i * {rd} + ri) * {ncol} + j * {cd} + cj]); }}")
            elif block:
                tgt = f"arg{k}[(int64_t)s_ * {rd * cd} + ri * {cd} + cj]"
                val = f"buf{k}[(i * {rd} + ri) * {ncol} + j * {cd} + cj]"
                post.append(
                    f"    for (int i = 0; i < {rar}; ++i) {{ const int32_t r_ = {_mv(rm, rar // nf, 'i')}; if (r_ < 0) continue;\n"
                    f"      for (int j = 0; j < {car}; ++j) {{ const int32_t c_ = {_mv(cm, car // nf, 'j')}; if (c_ < 0) continue;\n"
                    f"        const int32_t s_ = op2_find_slot(rowptr{k}, colidx{k}, r_, c_); if (s_ < 0) {{ atomicAdd(status, 1); continue; }}\n"
                    f"        for (int ri = 0; ri < {rd}; ++ri) for (int cj = 0; cj < {cd}; ++cj) {{ {store.format(tgt=tgt, val=val)} }} }} }}")
            else:
                tgt = f"arg{k}[s_]"
                val = f"buf{k}[(i * {rd} + ri) * {ncol} + j * {cd} + cj]"
                post.append(
                    f"    for (int i = 0; i < {rar}; ++i) {{ const int32_t r_ = {_mv(rm, rar // nf, 'i')}; if (r_ < 0) continue;\n"
                    f"      for (int ri = 0; ri < {rd}; ++ri) for (int j = 0; j < {car}; ++j) {{ const int32_t c_ = {_mv(cm, car // nf, 'j')}; if (c_ < 0) continue;\n"
                    f"        for (int cj = 0; cj < {cd}; ++cj) {{ const int32_t s_ = op2_find_slot(rowptr{k}, colidx{k}, r_ * {rd} + ri, c_ * {cd} + cj);"
                    f" if (s_ < 0) {{ atomicAdd(status, 1); continue; }} {store.format(tgt=tgt, val=val)} }} }} }}")
        else:
            raise NotImplementedError("Passthrough arguments are not supported on the device")
    for m in range(nmaps):
        params.append(f"const int32_t *__restrict__ map{m}")
    params.append("int32_t *__restrict__ status")
    if extruded:
        params.append("const int32_t *__restrict__ layers")
    offdecl = [f"    const int32_t off{m}[{len(o)}] = {{{', '.join(str(int(v)) for v in o)}}};"
               for m, o in sorted(offsets.items())]
    offdecl += [f"    const int32_t quo{m}[{len(o)}] = {{{', '.join(str(int(v)) for v in o)}}};"
                for m, o in sorted(quots.items())]
    params += [f"{t} *__restrict__ red{k}_" for k, t, _, _ in reduced]
    if accs:
        plans_used = sorted({g for _, g, _ in accs})
        params += ["int32_t tile_", "int32_t base_"]
        params += [p for g in plans_used for p in (f"const int32_t *__restrict__ tptr{g}_",
                                                   f"const uint16_t *__restrict__ loc{g}_")]
        params += [f"{_acc_type(_arg_ctype(lk, k))} *__restrict__ part{k}_" for k, _, _ in accs]
        head = _tiled_head(lk, accs, plans_used)
        loop = ["  for (int64_t t_ = first_ + threadIdx.x; t_ < last_; t_ += blockDim.x) {",
                "    const int32_t n = (int32_t)t_;"]
        tail = _tiled_tail(accs)
    elif reduced:
        # a workgroup runs several elements a lane, so that few partial
        # results leave it
        head, tail = [], []
        loop = ["  for (int64_t t_ = lo + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t_ < hi;"
                " t_ += (int64_t)gridDim.x * blockDim.x) {",
                "    const int32_t n = list ? list[t_] : (int32_t)t_;"]
    else:
        head, tail = ["  const int32_t t_ = lo + (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);"], []
        loop = ["  if (t_ < hi) {", "    const int32_t n = list ? list[t_] : t_;"]
    src = [_PRELUDE,
           "#pragma clang force_cuda_host_device begin",
           headers, code,
           "#pragma clang force_cuda_host_device end",
           'extern "C" __global__ void __launch_bounds__(256)',
           "op2_wrap(" + ", ".join(params) + ")",
           "{",
           "  (void)status;",
           *[d for d, _, _ in red],
           *head,
           *loop,
           *[d for _, d, _ in red],
           *([] if not extruded else [
               *offdecl,
               "    const int32_t lay_ = %s;" % ("0" if gk._constant_layers else "n"),
               "    const int32_t bottom_ = layers[2 * lay_], cend_ = layers[2 * lay_ + 1] - 1;",
               "    const int32_t lo_ = %s, hi_ = %s;" % _region_bounds(region, periodic),
               "    const int32_t nl_ = cend_ - bottom_;",
               "    (void)nl_;",
               "    for (int32_t layer_ = lo_; layer_ < hi_; ++layer_) {",
               "    const int32_t lyr_ = layer_ - bottom_;",
               "    (void)lyr_;"]),
           *pre,
           f"    {lk.name}({', '.join(call + (['layer_'] if getattr(gk, '_pass_layer_arg', False) else []))});",
           *post,
           *(["    }"] if extruded else []),
           *[d for _, _, d in red],
           "  }",
           *tail,
           *_reduction_tail(reduced),
           "}",
           *_finish_kernel(reduced)]
    return "\n".join(s for s in src if s is not None)


def _acc_type(t):
    """Type the increments of a tile are added up in: float64 for floats
    (LDS float32 adds run at a quarter of the float64 rate on gfx950)."""
    return "double" if t in ("float", "double") else t


def _arg_ctype(lk, k):
    return as_cstr(np.dtype(lk.arguments[k].dtype))


def _tiled_head(lk, accs, plans_used):
    """The workgroup's tile, its accumulators in LDS, zeroed.  Each XCD takes
    a contiguous range of tiles (workgroups go to the 8 XCDs in turn), so
    that neighbouring tiles' shared targets meet in one L2."""
    out = ["  extern __shared__ double smem_[];",
           "  const int32_t q_ = (int32_t)gridDim.x / 8, m_ = (int32_t)gridDim.x % 8, x_ = (int32_t)blockIdx.x % 8;",
           "  const int32_t b_ = x_ * q_ + (x_ < m_ ? x_ : m_) + (int32_t)blockIdx.x / 8;",
           "  const int64_t first_ = lo + (int64_t)b_ * tile_;",
           "  const int64_t last_ = first_ + tile_ < hi ? first_ + tile_ : hi;"]
    out += [f"  const int32_t p{g}_ = tptr{g}_[b_], u{g}_ = tptr{g}_[b_ + 1] - p{g}_;" for g in plans_used]
    out.append("  double *free_ = smem_;")
    for k, g, dim in accs:
        t = _acc_type(_arg_ctype(lk, k))
        out += [f"  {t} *acc{k}_ = reinterpret_cast<{t} *>(free_);", f"  free_ += u{g}_ * {dim};",
                f"  for (int32_t i = threadIdx.x; i < u{g}_ * {dim}; i += blockDim.x) acc{k}_[i] = ({t})0;"]
    out.append("  __syncthreads();")
    return out


def _tiled_tail(accs):
    """Every accumulator to its partial slot, contiguous per tile."""
    out = ["  __syncthreads();"]
    out += [f"  for (int32_t i = threadIdx.x; i < u{g}_ * {dim}; i += blockDim.x)"
            f" part{k}_[(int64_t)p{g}_ * {dim} + i] = acc{k}_[i];" for k, g, dim in accs]
    return out


def _reduction_tail(reduced):
    """Each reduced Global over the workgroup: waves, then LDS, then one
    partial result (or, for launches of few workgroups, one atomic)."""
    out = []
    if reduced:
        out.append("  const int lane_ = threadIdx.x & 63, wave_ = threadIdx.x >> 6, waves_ = (blockDim.x + 63) >> 6;")
    for k, t, dim, fn in reduced:
        step = {"sum": "w + buf", "min": "op2_min(w, buf)", "max": "op2_max(w, buf)"}[fn].replace("buf", f"s{k}_[v]")
        atomic = {"sum": "op2_atomic_add", "min": "op2_atomic_min", "max": "op2_atomic_max"}[fn]
        out += [f"  __shared__ {t} s{k}_[4];",
                f"  for (int q = 0; q < {dim}; ++q) {{",
                f"    {t} w = op2_wave_{fn}(sum{k}_[q]);",
                f"    if (lane_ == 0) s{k}_[wave_] = w;",
                "    __syncthreads();",
                "    if (threadIdx.x == 0) {",
                f"      for (int v = 1; v < waves_; ++v) w = {step};",
                f"      if (red{k}_) red{k}_[(int64_t)q * gridDim.x + blockIdx.x] = w; else {atomic}(&arg{k}[q], w);",
                "    }",
                "    __syncthreads();",
                "  }"]
    return out


def _finish_kernel(reduced):
    """``op2_finish``: one workgroup per component adds (or takes the minimum
    or maximum of) the partial results of ``n`` workgroups."""
    if not reduced:
        return []
    params = ", ".join(f"{t} *__restrict__ arg{k}, const {t} *__restrict__ red{k}_" for k, t, _, _ in reduced)
    out = ['extern "C" __global__ void __launch_bounds__(256)', f"op2_finish(int32_t n, {params})", "{",
           "  int c = blockIdx.x;", "  const int lane_ = threadIdx.x & 63, wave_ = threadIdx.x >> 6;"]
    for k, t, dim, fn in reduced:
        start = f"({t})0" if fn == "sum" else f"arg{k}[c]"
        join = {"sum": "{a} + {b}", "min": "op2_min({a}, {b})", "max": "op2_max({a}, {b})"}[fn]
        out += [f"  __shared__ {t} s{k}_[4];",
                f"  if (c >= 0 && c < {dim}) {{",
                f"    {t} w = {start};",
                "    for (int32_t i = threadIdx.x; i < n; i += 256) w = "
                + join.format(a="w", b=f"red{k}_[(int64_t)c * n + i]") + ";",
                f"    w = op2_wave_{fn}(w);",
                f"    if (lane_ == 0) s{k}_[wave_] = w;",
                "    __syncthreads();",
                "    if (threadIdx.x == 0) {",
                "      for (int v = 1; v < 4; ++v) w = " + join.format(a="w", b=f"s{k}_[v]") + ";",
                f"      arg{k}[c] = " + (join.format(a=f"arg{k}[c]", b="w")) + ";",
                "    }",
                "  }",
                f"  c -= {dim};"]
    out.append("}")
    return out


_gen_lock = threading.Lock()
_modules = {}


def _code_object(src, opts):
    """Code object bytes for ``src`` (memory, then disk cache, then hiprtc)."""
    key = hashlib.sha256(("\0".join(opts) + "\0" + src).encode()).hexdigest()[:32]
    cdir = os.path.join(configuration["cache_dir"], "hip")
    path = os.path.join(cdir, key + ".co")
    try:
        with open(path, "rb") as f:
            return key, f.read()
    except OSError:
        pass
    L = dev.lib()
    copts = (ctypes.c_char_p * len(opts))(*[o.encode() for o in opts])
    size = ctypes.c_size_t(0)
    log = ctypes.create_string_buffer(65536)
    rc = L.op2hip_jit_code_object(src.encode(), copts, len(opts), None, ctypes.byref(size), log, len(log))
    if rc != 0:
        raise CompilationError("device compilation of the generated wrapper failed:\n"
                               + log.value.decode(errors="replace") + "\n--- source ---\n" + src)
    buf = ctypes.create_string_buffer(size.value)
    rc = L.op2hip_jit_code_object(src.encode(), copts, len(opts), buf, ctypes.byref(size), log, len(log))
    dev.check(rc, "jit_code_object")
    data = buf.raw[:size.value]
    try:
        os.makedirs(cdir, exist_ok=True)
        tmp = path + ".tmp%d" % os.getpid()
        with open(tmp, "wb") as f:
            f.write(data)
        os.replace(tmp, path)
    except OSError:
        pass
    return key, data


def _module(src):
    opts = compile_options()
    key, data = _code_object(src, opts)
    with _gen_lock:
        mod = _modules.get(key)
        if mod is None:
            dev.device()
            L = dev.lib()
            h = ctypes.c_void_p()
            buf = ctypes.create_string_buffer(data, len(data))
            dev.check(L.op2hip_jit_load(buf, ctypes.byref(h)), "jit_load")
            mod = _modules[key] = h
    return mod


# Workgroups of a launch that reduces into Globals: each adds up its elements
# and leaves one partial result per component, which op2_finish adds (one
# atomic per wave on a Global's one address takes 52 ns after the other: 295 of
# 310 us for 361,201 elements); up to _ATOMIC_BLOCKS workgroups send atomics,
# cheaper than the second launch.
_REDUCE_BLOCKS = 2048
_ATOMIC_BLOCKS = 16

# Least increments of a loop that runs in tiles: below, device atomics hide
# behind the host's issue of the call, and the second pass costs one launch more
# (a pass with a P1 matrix kernel of 0.35, 0.72 and 2.9 million increments takes
# 33, 44 and 107 us with atomics, 32, 32 and 42 us in tiles; one with an edge
# flux of 0.47, 0.96 and 3.8 million, 39, 44 and 149 against 46 us).  Most
# distinct targets per increment: with less reuse a partial sum costs as much
# as an atomic.
_TILED_LEAST = 3 << 18
_TILED_REUSE = 0.75
_TILED_CODES = {"float64": 0, "float32": 1, "int32": 2, "int64": 3}


class GeneratedKernel:
    """Executor of a generated wrapper (``(start, end, ptrs, parloop)``)."""

    BLOCK = 256

    def __init__(self, gk):
        self.gk = gk
        self.strategy_used = None
        self._src = {}
        self._mods = {}
        lk = gk.local_kernel
        # components of every reduced Global
        self._reduced = [(k, int(np.prod(garg.dim)) if len(garg.dim) else 1)
                         for k, (larg, garg) in enumerate(zip(lk.arguments, gk.arguments))
                         if isinstance(garg, GlobalKernelArg) and larg.access != READ]
        self._tile_dims = self._tileable()

    def _tileable(self):
        """Values per target of every argument whose increments a tile can
        add up (``{arg: dim}``; None if the loop has another kind of indirect
        output, or none)."""
        gk, lk = self.gk, self.gk.local_kernel
        if getattr(gk, "_extruded", False) or gk._subset:
            return None
        out = {}
        for k, (larg, garg) in enumerate(zip(lk.arguments, gk.arguments)):
            if isinstance(garg, (MixedDatKernelArg, MixedMatKernelArg)):
                return None
            if isinstance(garg, DatKernelArg):
                if garg.map_ is None or larg.access == READ:
                    continue
                if larg.access != INC or garg.index is not None or garg.map_.offset is not None:
                    return None
                dim = int(np.prod(garg.dim))
            elif isinstance(garg, MatKernelArg):
                if larg.access != INC or garg.unroll or any(m.offset is not None for m in garg.maps):
                    return None
                dim = int(np.prod(garg.dims[0][0]))
            else:
                continue
            if np.dtype(larg.dtype).name not in _TILED_CODES:
                return None
            out[k] = dim
        return out or None

    def _unique_maps(self, parloop):
        seen, index = [], {}
        for k, a in enumerate(parloop.arguments):
            for j, m in enumerate(a.maps):
                for q, s in enumerate(seen):
                    if s is m:
                        index[(k, j)] = q
                        break
                else:
                    index[(k, j)] = len(seen)
                    seen.append(m)
        return seen, index

    def _flags(self, parloop):
        out = []
        for k, (garg, a) in enumerate(zip(self.gk.arguments, parloop.arguments)):
            if isinstance(garg, MatKernelArg):
                out.append((k, a.data._block))
            elif isinstance(garg, MixedMatKernelArg):
                out.append((k, tuple(getattr(b, "_gen_flag", b._block) for b in a.data)))
        return tuple(out)

    def source(self, parloop, groups=()):
        """The wrapper's source; ``groups``, the (argument, plan) pairs of
        the tiled form."""
        flags = self._flags(parloop)
        src = self._src.get((flags, groups))
        if src is None:
            _, index = self._unique_maps(parloop)
            src = self._src[flags, groups] = generate_source(self.gk, index, dict(flags), dict(groups))
        return src

    def _loaded(self, parloop, flags, groups=()):
        mod = self._mods.get((flags, groups))
        if mod is None:
            mod = self._mods[flags, groups] = _module(self.source(parloop, groups))
        return mod

    def _tiles(self, parloop, start, end):
        """The loop's tiling (``plans.target_tiles``) and its (argument,
        plan) pairs when it runs in tiles: large enough, every target
        present, and targets shared by a tile's elements often enough; else
        None and no pairs."""
        if (self._tile_dims is None or configuration["strategy"] not in ("auto", "staged") or end <= start
                or isinstance(parloop.iterset, Subset)):
            return None, ()
        from pyop2_amd import plans
        targets, groups, width = [], [], 0
        for k, dim in self._tile_dims.items():
            a = parloop.arguments[k]
            if any(m.has_negative for m in a.maps):
                return None, ()
            if a.kind == "mat":
                if hasattr(a.data, "_gen_flag") or (dim > 1 and not a.data._block):
                    return None, ()
                target = (a.maps[0], a.maps[1], a.data)
                width += a.maps[0].arity * a.maps[1].arity * dim
            else:
                target = (a.maps[0], None, None)
                width += a.maps[0].arity * dim
            g = next((i for i, t in enumerate(targets) if all(x is y for x, y in zip(t, target))), len(targets))
            if g == len(targets):
                targets.append(target)
            groups.append((k, g))
        if (end - start) * width < _TILED_LEAST:
            return None, ()
        tiles = plans.target_tiles(targets, start, end, width, _TILED_REUSE)
        return tiles, tuple(groups) if tiles is not None else ()

    def _conflict_maps(self, parloop):
        """Maps whose targets must be exclusive within a launch."""
        out = []
        need = False
        for larg, garg, a in zip(self.gk.local_kernel.arguments, self.gk.arguments, parloop.arguments):
            if isinstance(garg, DatKernelArg) and garg.map_ is not None:
                if larg.access in (RW, WRITE):
                    need = True
                if larg.access in (RW, WRITE, INC, MIN, MAX):
                    out.append(a.maps[0])
            elif isinstance(garg, MixedDatKernelArg):
                if larg.access in (RW, WRITE):
                    need = True
                if larg.access in (RW, WRITE, INC, MIN, MAX):
                    out.extend(a.maps)
            elif isinstance(garg, MatKernelArg):
                if larg.access == WRITE:
                    need = True
                out.append(a.maps[0])
            elif isinstance(garg, MixedMatKernelArg):
                if larg.access == WRITE:
                    need = True
                out.extend(a.maps[:garg.shape[0]])
        return (out if need else []), need

    def __call__(self, start, end, ptrs, parloop):
        if parloop is None:
            raise RuntimeError("generated loops are launched by a Parloop")
        own = parloop.__dict__.setdefault("_launches", {})
        launch = own.get((start, end, self))
        if launch is None or not launch.holds(parloop):
            launch = _GeneratedLaunch(self, start, end, parloop)
            # tiles cannot be planned while a graph is captured: later calls may
            if not dev.torch().cuda.is_current_stream_capturing():
                own[(start, end, self)] = launch
        launch(parloop)
        self.strategy_used = launch.strategy

    def _colours(self, start, end, parloop):
        """The colour plan of a loop that runs coloured, else None."""
        conflict, need_colour = self._conflict_maps(parloop)
        if configuration["strategy"] == "coloured" and not need_colour:
            conflict = []
            for larg, garg, a in zip(self.gk.local_kernel.arguments, self.gk.arguments, parloop.arguments):
                if (isinstance(garg, DatKernelArg) and garg.map_ is not None and larg.access != READ) \
                        or isinstance(garg, MatKernelArg):
                    conflict.append(a.maps[0])
                elif isinstance(garg, MixedDatKernelArg) and larg.access != READ:
                    conflict.extend(a.maps)
                elif isinstance(garg, MixedMatKernelArg):
                    conflict.extend(a.maps[:garg.shape[0]])
            need_colour = bool(conflict)
        if not (need_colour and conflict):
            return None
        from pyop2_amd import plans
        iterset, region = parloop.iterset, getattr(self.gk, "_iteration_region", None)
        if isinstance(iterset, Subset):
            elems = iterset.indices[start:end]
        else:
            elems = np.arange(start, end, dtype=np.int32)
        key = (iterset._plan_key(), start, end, tuple(id(m) for m in conflict), int(region or 0))
        if not getattr(self.gk, "_extruded", False):
            return plans.colour_plan(conflict[0], elems, [(m, id(m.toset)) for m in conflict], key)
        # a column's targets over all its layers (a thread runs the
        # layers of its column one after the other)
        cols = np.ascontiguousarray(elems, dtype=np.int32)   # column ids, in launch order
        targets = [(_ColumnTargets(m, iterset, cols, region), id(m.toset)) for m in conflict]
        plan = plans.colour_plan(conflict[0], np.arange(len(cols), dtype=np.int32), targets,
                                 ("extruded",) + key)
        return _column_plan(plan, cols, conflict[0], ("extruded-cols",) + key)


class _GeneratedLaunch:
    """One band of a generated loop, ready but for the addresses of its data:
    the loaded kernel, its argument block, and the colours or tiles it runs
    by.  Held by the loop it was made for; ``holds`` says whether what it was
    made from is still the loop's."""

    def __init__(self, kernel, start, end, parloop):
        self.kernel, self.start, self.end = kernel, start, end
        gk = kernel.gk
        self.lock = threading.Lock()
        flags = kernel._flags(parloop)
        tiles, self.groups = kernel._tiles(parloop, start, end)
        self.tiles = tiles
        self.mod = kernel._loaded(parloop, flags, self.groups)
        maps, _ = kernel._unique_maps(parloop)
        iterset = parloop.iterset
        self.made_for = self._made_of(parloop)
        self.flags, self.strategies = flags, (configuration["strategy"], _TILED_LEAST)
        # data arguments: (argument block entries, argument, what)
        self.data, vals, self.status_of = [], [], None
        for k, (garg, a) in enumerate(zip(gk.arguments, parloop.arguments)):
            n = {True: 3, False: 1}[isinstance(garg, MatKernelArg)]
            if isinstance(garg, MixedMatKernelArg):
                n = 3 * sum(1 for _ in a.data)
            elif isinstance(garg, MixedDatKernelArg):
                n = sum(1 for _ in a.data)
            if isinstance(garg, (MatKernelArg, MixedMatKernelArg)) and self.status_of is None:
                self.status_of = k
            slots = [ctypes.c_void_p() for _ in range(n)]
            self.data.append((slots, k, garg))
            vals += slots
        vals += [ctypes.c_void_p(dev.ptr(m.device_values)) for m in maps]
        self.keep = [m.device_values for m in maps]
        self.status = ctypes.c_void_p(dev.ptr(_dummy_status()) if self.status_of is None else 0)
        vals.append(self.status)
        if getattr(gk, "_extruded", False):
            region = getattr(gk, "_iteration_region", None)
            for m in maps:
                if getattr(m, "offset", None) is not None:
                    m.check_extruded(iterset, region)
            vals.append(ctypes.c_void_p(dev.ptr(iterset.device_layers)))
            self.keep.append(iterset.device_layers)
        self.colours = kernel._colours(start, end, parloop)
        self.list = 0
        if isinstance(iterset, Subset):
            self.list = dev.ptr(iterset.device_indices)
            self.keep.append(iterset.device_indices)
        self.strategy = "coloured" if self.colours else "staged" if tiles is not None else "atomic"
        # the argument block: bounds, list, atomic flag, data, maps, partial
        # results of the reduced Globals, and the tiles' plan and partial sums
        self.head = [ctypes.c_int32(), ctypes.c_int32(), ctypes.c_void_p(), ctypes.c_int32()]
        self.reds = [ctypes.c_void_p() for _ in kernel._reduced]
        self.parts, extra, self.lds = [], [], 0
        if tiles is not None:
            extra = [ctypes.c_int32(tiles.tile), ctypes.c_int32(start)]
            for p in tiles.plans:
                extra += [ctypes.c_void_p(dev.ptr(p.tile_ptr)), ctypes.c_void_p(dev.ptr(p.local))]
            for k, g in self.groups:
                dt = np.dtype(gk.local_kernel.arguments[k].dtype)
                plan, dim, slot = tiles.plans[g], kernel._tile_dims[k], ctypes.c_void_p()
                acc = np.dtype(np.float64) if dt.kind == "f" else dt
                self.parts.append((slot, k, plan, dim, _TILED_CODES[dt.name], acc))
                self.lds += plan.max_targets * dim * 8
                extra.append(slot)
        block = self.head + vals + self.reds + extra
        self.argv = (ctypes.c_void_p * len(block))(*[ctypes.addressof(v) for v in block])
        self.block = block
        self.count = ctypes.c_int32()
        self.globals = [ctypes.c_void_p() for _ in kernel._reduced]
        finish = [self.count] + [v for pair in zip(self.globals, self.reds) for v in pair]
        self.finish = (ctypes.c_void_p * len(finish))(*[ctypes.addressof(v) for v in finish])
        self.name = "op2_wrap:" + gk.name

    @staticmethod
    def _made_of(parloop):
        """Maps and patterns the launch's plans follow from."""
        out = [parloop.iterset]
        for a in parloop.arguments:
            out += a.maps
            if a.kind in ("mat", "mixed_mat"):
                out.append(a.data.sparsity)
        return out

    def holds(self, parloop):
        now = self._made_of(parloop)
        return (self.strategies == (configuration["strategy"], _TILED_LEAST) and len(now) == len(self.made_for)
                and all(map(operator.is_, self.made_for, now))
                and (self.status_of is None or self.flags == self.kernel._flags(parloop)))

    def _fill(self, parloop):
        args = parloop.arguments
        for slots, k, garg in self.data:
            data = args[k].data
            if isinstance(garg, MatKernelArg):
                blocks = (data,)
            elif isinstance(garg, MixedMatKernelArg):
                blocks = tuple(data)
            elif isinstance(garg, MixedDatKernelArg):
                for s, d in zip(slots, data):
                    s.value = d._device_array().data_ptr()
                continue
            else:
                slots[0].value = data._device_array().data_ptr()
                continue
            for i, b in enumerate(blocks):
                slots[3 * i].value = b.rowptr.data_ptr()
                slots[3 * i + 1].value = b.colidx.data_ptr()
                slots[3 * i + 2].value = b.device_values.data_ptr()
        if self.status_of is not None:
            data = args[self.status_of].data
            if isinstance(self.kernel.gk.arguments[self.status_of], MixedMatKernelArg):
                data = data[0, 0]
            self.status.value = data._status.data_ptr()

    def __call__(self, parloop):
        with self.lock:   # the argument block is this launch's own
            self._fill(parloop)
            with dev.timed_launch(self.name):
                if self.colours is not None:
                    plan = self.colours
                    ep = dev.ptr(plan.elems)
                    for c in range(plan.ncolours):
                        lo, hi = int(plan.offsets[c]), int(plan.offsets[c + 1])
                        if hi > lo:
                            self._launch(parloop, lo, hi, ep, 0)
                elif self.tiles is not None:
                    self._launch_tiles(parloop)
                else:
                    self._launch(parloop, self.start, self.end, self.list, 1)

    def _launch(self, parloop, lo, hi, lst, atomic, grid=0, block=GeneratedKernel.BLOCK, lds=0):
        L, kernel, stream = dev.lib(), self.kernel, dev.raw_stream()
        if not grid:
            grid = (hi - lo + block - 1) // block
            if self.reds:
                grid = min(grid, _REDUCE_BLOCKS)
        self.head[0].value, self.head[1].value, self.head[2].value, self.head[3].value = lo, hi, lst, atomic
        finish = self.reds and grid > _ATOMIC_BLOCKS
        if self.reds:
            # partial results of the workgroups, free again behind the launches
            parts = [dev.empty((dim * grid,), kernel.gk.local_kernel.arguments[k].dtype) if finish else None
                     for k, dim in kernel._reduced]
            for slot, p in zip(self.reds, parts):
                slot.value = dev.ptr(p)
        rc = L.op2hip_jit_launch(self.mod, b"op2_wrap", grid, block, lds, self.argv, stream)
        if not rc and finish:
            self.count.value = grid
            for slot, (k, _) in zip(self.globals, kernel._reduced):
                slot.value = parloop.arguments[k].data._device_array().data_ptr()
            rc = L.op2hip_jit_launch(self.mod, b"op2_finish", sum(d for _, d in kernel._reduced),
                                     GeneratedKernel.BLOCK, 0, self.finish, stream)
        if rc:
            dev.check(rc, f"launch of generated {kernel.gk.name}")

    def _launch_tiles(self, parloop):
        """The tiles' launch, then one pass per output that adds its targets'
        partial sums (float64 for floats)."""
        L, tiles = dev.lib(), self.tiles
        bufs = [dev.empty((max(p.nslots * dim, 1),), acc) for _, _, p, dim, _, acc in self.parts]
        for buf, part in zip(bufs, self.parts):
            part[0].value = buf.data_ptr()
        self._launch(parloop, self.start, self.end, 0, 1, tiles.ntiles, tiles.block, self.lds)
        for buf, (_, k, p, dim, code, _) in zip(bufs, self.parts):
            a = parloop.arguments[k]
            out = a.data.device_values if a.kind == "mat" else a.data._device_array()
            rc = L.op2hip_tile_targets_add(code, p.nrows, dim, dev.ptr(p.row_ptr), dev.ptr(p.row_slots),
                                           buf.data_ptr(), out.data_ptr(), dev.raw_stream())
            if rc:
                dev.check(rc, f"partial sums of generated {self.kernel.gk.name}")


class _ColumnTargets:
    """Duck-typed map for colouring the columns ``cols`` of an extruded loop
    (a range of the set, or a Subset's columns): row c lists every target
    column cols[c] touches over the layers it runs."""

    def __init__(self, m, iterset, cols, region=None):
        self._table = m.column_table(iterset, cols, region)
        self.toset = m.toset


def _column_plan(plan, cols, owner, key):
    """A colour plan over positions in ``cols`` turned into column ids."""
    from pyop2_amd import plans
    got = owner._cache.get(key)
    if got is None:
        elems = cols[dev.to_host(plan.elems).astype(np.int64)].astype(np.int32)
        got = plans.ColourPlan(plan.colours, dev.to_device(elems), plan.offsets, plan.ncolours)
        owner._cache[key] = got
    return got


_STATUS = None


def _dummy_status():
    global _STATUS
    if _STATUS is None:
        _STATUS = dev.zeros((1,), np.int32)
    return _STATUS
