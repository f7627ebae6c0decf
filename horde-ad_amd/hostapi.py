"""Binding of include/hordead_host.h (libhordead_host.so): values and their operations through the CPython extension
`lib/_pyvalues.*.so` (host/pyvalues.cpp), everything else through ctypes.

`Host` is a context of the host layer on some provider of the array ABI, `V` a
tensor value whose methods carry the names of horde-ad's tensor operations
(`ssum`, `sgather`, `smatmul2`, ...; reference export list:
src/HordeAd/OpsTensor.hs:16-78), and `IxV` a lane-batched scalar with Python
operators, so that an index function is written as a lambda exactly like the
reference's `\\[i, k] -> [i + k]` and is called once, symbolically.
"""
import ctypes as C
import hashlib
import importlib.machinery
import importlib.util
import os
import sysconfig

import numpy as np

from . import capi
from .capi import _DT2NP, _NP2DT, CMP, OP1, OP2, HgpuError, _larr

P, PP, I, L = C.c_void_p, C.POINTER(C.c_void_p), C.c_int, C.c_int64
LP, IP = C.POINTER(C.c_int64), C.POINTER(C.c_int)
D = C.c_double
SIG = {
    "create_gpu": (I, [I, PP]), "create": (I, [P, I, PP]), "destroy": (I, [P]),
    "last_error": (C.c_char_p, [P]), "sync": (I, [P]), "array_ctx": (P, [P]), "tape_reset": (I, [P]), "set_fusion": (I, [P, I]),
    "upload": (I, [P, I, I, LP, P, I, PP]), "from_array": (I, [P, P, I, PP]),
    "constant": (I, [P, I, D, I, LP, PP]), "array": (I, [P, PP]), "download": (I, [P, P, P]),
    "val_rank": (I, [P]), "val_dtype": (I, [P]), "val_shape": (I, [P, LP]), "free": (I, [P]),
    "backward": (I, [P, P, P, I, PP, PP]),
    "ewise1": (I, [P, I, P, PP]), "ewise2": (I, [P, I, P, P, PP]), "compare": (I, [P, I, P, P, PP]),
    "compare_all": (I, [P, I, P, P, IP]), "select": (I, [P, P, P, P, PP]), "convert": (I, [P, P, I, I, PP]),
    "tssumN": (I, [P, P, I, PP]), "tssum0": (I, [P, P, PP]), "tsdot0": (I, [P, P, P, PP]),
    "tsdot1In": (I, [P, P, P, PP]), "tsdotNIn": (I, [P, P, P, I, PP]), "tD": (I, [P, P, P, PP]), "tprimalPart": (I, [P, P, PP]), "as_input": (I, [P, P, PP]), "tsmatvecmul": (I, [P, P, P, PP]), "tsmatmul2": (I, [P, P, P, PP]),
    "tsreplicateN": (I, [P, P, I, LP, PP]), "tsappend": (I, [P, P, P, PP]), "tsslice": (I, [P, P, L, L, PP]),
    "tsreverse": (I, [P, P, PP]), "tstranspose": (I, [P, P, I, IP, PP]), "tsreshape": (I, [P, P, I, LP, PP]),
    "tsindex": (I, [P, P, I, LP, PP]), "tsargminmax": (I, [P, P, I, PP]), "tsiota": (I, [P, L, I, PP]),
    "ix_var": (I, [P, I, LP, I, PP]), "ix_const": (I, [P, I, LP, I, D, PP]), "ix_lift": (I, [P, I, LP, P, PP]),
    "ix_op1": (I, [P, I, P, PP]), "ix_op2": (I, [P, I, P, P, PP]), "ix_compare": (I, [P, I, P, P, PP]),
    "ix_select": (I, [P, P, P, P, PP]), "ix_convert": (I, [P, P, I, I, PP]),
    "ix_index0": (I, [P, P, I, PP, PP]), "ix_argminmax": (I, [P, P, I, PP, I, PP]), "ix_free": (I, [P]),
    "ix_is_affine": (I, [P]), "counter": (L, [P, C.c_char_p]),
    "ix_from_val": (I, [P, P, PP]), "ix_to_val": (I, [P, P, PP]), "ix_dtype": (I, [P]),
    "tconvert": (I, [P, I, P, I, LP, PP]), "dense": (I, [P, P, PP]),
    "tsgather": (I, [P, P, I, LP, I, PP, PP]), "tsscatter": (I, [P, P, I, I, LP, PP, PP]),
    "capture_begin": (I, [P]), "capture_end": (I, [P, PP]), "graph_launch": (I, [P, P]), "graph_free": (I, [P, P]),
    "force": (I, [P, P]), "overwrite": (I, [P, P, P]), "assign": (I, [P, P, P]),
    "update_with_gradient": (I, [P, D, P, P, PP]),
    "update_with_gradient_adam": (I, [P, D, D, D, D, I, P, P, P, P, PP, PP, PP]),
    "adam_step_size": (I, [P, I, D, D, D, I, PP]),
    "adam_apply": (I, [P, P, D, D, D, P, P, P, P, PP, PP, PP]),
}

EXTENSION = os.path.join(capi.HERE, "lib", "_pyvalues" + sysconfig.get_config_var("EXT_SUFFIX"))


def _extension():
    loader = importlib.machinery.ExtensionFileLoader("_pyvalues", EXTENSION)
    mod = importlib.util.module_from_spec(importlib.util.spec_from_file_location("_pyvalues", EXTENSION, loader=loader))
    loader.exec_module(mod)
    _check_source(mod.SOURCE, os.path.join(capi.HERE, "host", "pyvalues.cpp"))
    return mod


def _check_source(built_from, path):
    """The extension takes signatures and addresses on trust: one that another source was built to is not used."""
    if os.path.exists(path):
        with open(path, "rb") as f:
            if hashlib.sha256(f.read()).hexdigest()[:16] != built_from:
                raise ImportError(f"{EXTENSION} is not built from {path} as it is now; run __graft_entry__.build()")


_py = _extension()
_dll = None
# entry points called through the extension: name -> (arguments, result); pyvalues.cpp says what the letters are
NATIVE = {
    "tape_reset": ("", "N"), "constant": ("idS", "V"), "ewise1": ("iv", "V"), "ewise2": ("ivv", "V"), "compare": ("ivv", "V"),
    "select": ("vvv", "V"), "convert": ("vii", "V"), "tssumN": ("vi", "V"), "tssum0": ("v", "V"), "tsdot0": ("vv", "V"),
    "tsdot1In": ("vv", "V"), "tsdotNIn": ("vvi", "V"), "tD": ("vv", "V"), "tprimalPart": ("v", "V"), "as_input": ("v", "V"),
    "tsmatvecmul": ("vv", "V"), "tsmatmul2": ("vv", "V"), "tsreplicateN": ("vS", "V"), "tsappend": ("vv", "V"), "tsslice": ("vnn", "V"),
    "tsreverse": ("v", "V"), "tstranspose": ("vQ", "V"), "tsreshape": ("vS", "V"), "tsindex": ("vS", "V"), "tsargminmax": ("vi", "V"),
    "tsiota": ("ni", "V"), "dense": ("v", "V"), "tsgather": ("vSK", "V"), "tconvert": ("ivS", "V"),
    "ix_var": ("Si", "X"), "ix_const": ("Sid", "X"), "ix_lift": ("Sv", "X"), "ix_op1": ("ix", "X"), "ix_op2": ("ixx", "X"),
    "ix_compare": ("ixx", "X"), "ix_select": ("xxx", "X"), "ix_convert": ("xii", "X"), "ix_index0": ("vK", "X"),
    "ix_argminmax": ("vKi", "X"), "ix_from_val": ("v", "X"), "ix_to_val": ("x", "V"),
    "force": ("v", "N"), "download": ("vp", "N"), "overwrite": ("vp", "N"), "assign": ("vv", "N"), "graph_launch": ("p", "N"),
}


class _Native:
    """The entry points of NATIVE as functions of a host and their arguments, once the library is loaded."""


_c = _Native()


def _lib():
    global _dll
    if _dll is None:
        if not os.path.exists(capi.HOST_LIB):
            raise FileNotFoundError(f"{capi.HOST_LIB} is not built; run __graft_entry__.build()")
        dll = C.CDLL(capi.HOST_LIB)
        for name, (res, args) in SIG.items():
            fn = getattr(dll, "hh_" + name)
            fn.restype, fn.argtypes = res, args
        address = lambda name: C.cast(getattr(dll, "hh_" + name), C.c_void_p).value  # noqa: E731
        _py.setup(V, IxV, HgpuError, *[address(f) for f in ("free", "ix_free", "val_rank", "val_dtype", "val_shape", "ix_dtype", "last_error", "backward")])
        for name, (args, out) in NATIVE.items():
            setattr(_c, name, _py.Fn(address(name), args, out))
        _dll = dll
    return _dll


def _values(x):
    if isinstance(x, V):
        yield x
    elif isinstance(x, (list, tuple)):
        for y in x:
            yield from _values(y)


class Graph:
    def __init__(self, host, h):
        self.host, self.h = host, h

    def launch(self):
        _c.graph_launch(self.host, self.h)

    def free(self):
        if self.h:
            self.host.check(self.host.dll.hh_graph_free(self.host.h, self.h))
            self.h = None
            self.keeps = None


class Host(_py.HostBase):
    """A host-layer context: on the gfx950 library by default, or on the provider
    whose ABI table `api_lib.get_api()` returns."""

    def __init__(self, api_lib=None, device=0):
        self.dll = _lib()
        h = C.c_void_p()
        if api_lib is None:
            rc = self.dll.hh_create_gpu(device, C.byref(h))
        else:
            self._api_lib = api_lib  # keep the provider loaded
            rc = self.dll.hh_create(api_lib.get_api(), device, C.byref(h))
        if rc:
            raise HgpuError(rc, "cannot create a host-layer context (no usable device?)")
        self.h = h
        self._bind(h)

    def check(self, rc):
        if rc:
            raise HgpuError(rc, self.dll.hh_last_error(self.h).decode())

    def _out(self, fn, *args):
        o = C.c_void_p()
        self.check(fn(self.h, *args, C.byref(o)))
        return V(self, o)

    def sync(self):
        self.check(self.dll.hh_sync(self.h))

    def set_fusion(self, on):
        self.check(self.dll.hh_set_fusion(self.h, int(on)))

    def counter(self, name):
        """How often the named rewrite onto a fused entry point was taken (diagnostic)."""
        return int(self.dll.hh_counter(self.h, name.encode()))

    def tape_reset(self):
        _c.tape_reset(self)

    def submit(self, *values):
        """Sends out now what gives these values, not when they are read."""
        for v in values:
            _c.force(self, v)

    def destroy(self):
        self.dll.hh_destroy(self.h)

    # -- one recorded program, launched many times
    def capture(self, program):
        """Records the device work of `program()` (run it once without capture
        first) and returns (graph, what program returned); every value made
        inside is refreshed by graph.launch()."""
        self.check(self.dll.hh_capture_begin(self.h))
        try:
            result = program()
            for v in _values(result):
                _c.force(self, v)
        except BaseException:
            g = C.c_void_p()
            self.dll.hh_capture_end(self.h, C.byref(g))
            if g:
                self.dll.hh_graph_free(self.h, g)
            raise
        g = C.c_void_p()
        self.check(self.dll.hh_capture_end(self.h, C.byref(g)))
        graph = Graph(self, g)
        # The recording reads, at every launch, the arrays that existed before it:
        # they must outlive it.  The recorded function holds them (its closure), so the graph holds the function.
        graph.keeps = program
        return graph, result

    # -- values
    def concrete(self, x, requires_grad=False):
        x = np.asarray(x)
        if not x.flags.c_contiguous:
            x = x.copy(order="C")
        return self._out(self.dll.hh_upload, _NP2DT[x.dtype], x.ndim, _larr(x.shape),
                         x.ctypes.data_as(C.c_void_p), int(requires_grad))

    def param(self, x):
        return self.concrete(x, requires_grad=True)

    def sconcrete(self, x):
        """A small constant of the program (`sconcrete (sfromListLinear ..)`: an index table,
        the [0.0, 1.0] of a mask): uploaded the first time its value is asked for and kept, so
        a program that names constants can be recorded after one eager run."""
        x = np.ascontiguousarray(x)
        key = (x.dtype.str, x.shape, x.tobytes())
        cache = self.__dict__.setdefault("_constants", {})
        if key not in cache:
            if x.nbytes > 1 << 16:
                return self.concrete(x)
            cache[key] = self.concrete(x)
        return cache[key]

    def srepl(self, shape, value, dtype=capi.F64):
        """sconcrete (sreplicate shape value)"""
        return _c.constant(self, dtype, float(value), shape)

    def siota(self, n, dtype=capi.I64):
        return _c.tsiota(self, n, dtype)

    def grad(self, out, inputs, dt=None):
        """Cotangents of `inputs` for d(out) = dt (default: ones, as `grad` uses).

        The tape keeps what the reverse pass may read until `tape_reset`, and what it keeps counts as wanted: a
        zero-extension that a convolution's kernels read through, or a gather that is multiplied and summed at once, is
        written after all while the tape has it.  Reset the tape when the gradients have been asked for, as
        `Workload.gradient` does; values made before stay usable as constants, but an input made before a reset
        has no derivative after it."""
        return _py.backward(self, out, dt, inputs)

    # -- host loops of the tensor class (the reference's `Concrete` instance runs
    #    these closures once per index on the host as well)
    def sfromVector(self, vs):
        """tsfromVector (OpsConcrete.hs:144-151): stacks values of one shape along a new outermost dim."""
        out = None
        for v in vs:
            row = v.sreshape([1] + list(v.shape))
            out = row if out is None else out.sappend(row)
        return out

    def sbuild1(self, k, f):
        """tsbuild1 (OpsConcrete.hs:1761-1774): [f 0, ..., f (k-1)] stacked; f gets a concrete index."""
        return self.sfromVector([f(i) for i in range(k)])

    def kbuild(self, shm, f, dtype=None):
        """tkbuild @shm f (Ops.hs:863-880; Concrete: one vector generate, OpsConcrete.hs:1081-1087):
        f gets the position variables as lane values and runs once; its result (a lane
        value, or a Python number with `dtype`) is written out as an array of shape shm."""
        shm = tuple(int(s) for s in shm)
        r = f(*self.ix_space(shm))
        if not isinstance(r, IxV):
            r = IxV.const(self, shm, r, capi.I64 if dtype is None else dtype)
        elif dtype is not None and r.dtype != dtype:
            raise HgpuError(1, "kbuild: the closure's result is not of the element type asked for")
        return r.to_val()

    def kbuild1(self, k, f, dtype=None):
        """tkbuild1 @k f (Ops.hs:860-862)."""
        return self.kbuild((k,), f, dtype)

    def sbuild(self, shm, f):
        """tsbuild @shm f for a closure that yields arrays (Ops.hs:913-928, OpsConcrete.hs:1776-1789):
        the reference's nest of tsbuild1 host loops, f gets concrete indices.  With scalar
        elements (shn = []) the reference takes tbuildK instead: that is `kbuild`."""
        shm = tuple(int(s) for s in shm)

        def level(prefix, rest):
            if not rest:
                return f(*prefix)
            return self.sbuild1(rest[0], lambda i: level(prefix + [i], rest[1:]))
        return level([], list(shm))

    def smapAccumL(self, f, acc0, xs):
        """tmapAccumL (OpsConcrete.hs:990-1019): threads `acc` through the outermost
        dim of xs; f(acc, x) -> (acc', y).  Returns (final acc, stacked ys)."""
        acc, ys = acc0, []
        for t in range(xs.shape[0]):
            acc, y = f(acc, xs.sindex([t]))
            ys.append(y)
        return acc, self.sfromVector(ys)

    # -- index functions
    def ix_space(self, shm):
        return [_c.ix_var(self, shm, d) for d in range(len(shm))]

    def _apply_index_fn(self, shm, f):
        shm = tuple(int(s) for s in shm)
        vars_ = self.ix_space(shm)
        res = f(*vars_)
        res = [r if isinstance(r, IxV) else IxV.const(self, shm, int(r)) for r in res]
        return shm, res


class IxV(_py.Lane):
    """A scalar inside an index function, for all positions at once (`host`, `h`, `shm`: its index space, `dtype`)."""

    @staticmethod
    def const(host, shm, value, dtype=capi.I64):
        return _c.ix_const(host, shm, dtype, float(value))

    @staticmethod
    def from_val(v):
        """The elements of an array as a lane value over the array's own index space
        (what the scalar closure of tsmap0N / tszipWith0N is applied to)."""
        return _c.ix_from_val(v.host, v)

    def to_val(self):
        """This lane value as an array of shape shm."""
        return _c.ix_to_val(self.host, self)

    def _coerce(self, o, dtype=None):
        """A Python number beside a lane value is a literal of the lane value's element type."""
        return o if isinstance(o, IxV) else _c.ix_const(self.host, self.shm, self.dtype if dtype is None else dtype, float(o))

    def _op2(self, op, o, dtype=None):
        return _c.ix_op2(self.host, OP2[op], self, o if isinstance(o, IxV) else self._coerce(o, dtype))

    def _rop2(self, op, o, dtype=None):
        return self._coerce(o, dtype)._op2(op, self)

    @property
    def is_affine(self):
        return bool(self.host.dll.hh_ix_is_affine(self.h))

    def __add__(self, o): return self._op2("add", o)
    def __radd__(self, o): return self._rop2("add", o)
    def __sub__(self, o): return self._op2("sub", o)
    def __rsub__(self, o): return self._rop2("sub", o)
    def __mul__(self, o): return self._op2("mul", o)
    def __rmul__(self, o): return self._rop2("mul", o)
    def __truediv__(self, o): return self._op2("div", o)
    def __rtruediv__(self, o): return self._rop2("div", o)
    def __pow__(self, o): return self._op2("pow", o)
    def atan2H(self, o): return self._op2("atan2", o)
    def __neg__(self): return _c.ix_op1(self.host, OP1["neg"], self)
    def quotH(self, o): return self._op2("quot", o)
    def remH(self, o): return self._op2("rem_scalar", o)      # scalar rule: remH a 0 = a (Types.hs:402-419)
    def minH(self, o): return self._op2("min", o)
    def maxH(self, o): return self._op2("max", o)
    def op1(self, name): return _c.ix_op1(self.host, OP1[name], self)

    def _cmp(self, c, o, dtype):
        return _c.ix_compare(self.host, CMP[c], self, self._coerce(o, dtype))

    def leq(self, o, dtype=None): return self._cmp("leq", o, dtype)     # <=.
    def lt(self, o, dtype=None): return self._cmp("lt", o, dtype)       # <.
    def eq(self, o, dtype=None): return self._cmp("eq", o, dtype)       # ==.
    def notB(self): return self.op1("not")
    def andB(self, o): return self._op2("and", o)                        # &&*

    def convert(self, dtype, mode=0):
        return _c.ix_convert(self.host, self, dtype, mode)


def ifH(cond, a, b, dtype=None):
    """ifH / kcond on lane-batched scalars.  Python numbers take the other branch's element
    type, or `dtype`, or Int."""
    if dtype is None:
        dtype = a.dtype if isinstance(a, IxV) else b.dtype if isinstance(b, IxV) else capi.I64
    a = a if isinstance(a, IxV) else IxV.const(cond.host, cond.shm, a, dtype)
    b = b if isinstance(b, IxV) else IxV.const(cond.host, cond.shm, b, dtype)
    return _c.ix_select(cond.host, cond, a, b)


class V(_py.Val):
    """A tensor value of the `Gpu` carrier, possibly carrying a tape node (`host`, `h`, `shape`, `dtype`)."""

    def numpy(self):
        out = np.empty(self.shape, dtype=_DT2NP[self.dtype])
        _c.download(self.host, self, out.__array_interface__["data"][0])
        return out

    def overwrite(self, x):
        """New contents for an input of a recorded program (same shape and dtype)."""
        x = np.asarray(x, dtype=_DT2NP[self.dtype])
        if not x.flags.c_contiguous:
            x = x.copy(order="C")
        assert tuple(x.shape) == tuple(self.shape)
        _c.overwrite(self.host, self, x.__array_interface__["data"][0])

    def assign(self, src):
        """This array's memory takes src's elements (how a recorded training step
        hands updated parameters to its next launch)."""
        _c.assign(self.host, self, src)

    def _lift(self, o):
        if isinstance(o, V):
            return o
        return self.host.srepl(self.shape, o, self.dtype)

    # -- Num / Fractional / Floating
    def op1(self, name): return _c.ewise1(self.host, OP1[name], self)
    def op2(self, name, o): return _c.ewise2(self.host, OP2[name], self, o if isinstance(o, V) else self._lift(o))
    def _cmp(self, c, o): return _c.compare(self.host, CMP[c], self, o if isinstance(o, V) else self._lift(o))
    def __add__(self, o): return self.op2("add", o)
    def __radd__(self, o): return self._lift(o).op2("add", self)
    def __sub__(self, o): return self.op2("sub", o)
    def __rsub__(self, o): return self._lift(o).op2("sub", self)
    def __mul__(self, o): return self.op2("mul", o)
    def __rmul__(self, o): return self._lift(o).op2("mul", self)
    def __truediv__(self, o): return self.op2("div", o)
    def __rtruediv__(self, o): return self._lift(o).op2("div", self)
    def __pow__(self, o): return self.op2("pow", o)
    def __neg__(self): return self.op1("neg")
    def atan2H(self, o): return self.op2("atan2", o)
    def quotH(self, o): return self.op2("quot", o)
    def remH(self, o): return self.op2("rem", o)

    # -- comparisons, conditionals, conversions
    def leq(self, o): return self._cmp("leq", o)
    def lt(self, o): return self._cmp("lt", o)
    def eq(self, o): return self._cmp("eq", o)

    def compare_all(self, cmp, o):
        r = C.c_int()
        self.host.check(self.host.dll.hh_compare_all(self.host.h, CMP[cmp], self.h, o.h, C.byref(r)))
        return bool(r.value)

    def select(self, a, b):
        """Elementwise ifH on a Bool tensor."""
        return _c.select(self.host, self, a, b)

    def scast(self, dtype): return _c.convert(self.host, self, dtype, 0)
    def sfromIntegral(self, dtype): return _c.convert(self.host, self, dtype, 0)
    def sfloor(self, dtype=capi.I64): return _c.convert(self.host, self, dtype, 1)

    # -- maps of scalar closures (Ops.hs:929-941): the closure runs once, on lane values
    def smap0N(self, f):
        """tsmap0N f self"""
        return f(IxV.from_val(self)).to_val()

    def szipWith0N(self, f, o):
        """tszipWith0N f self o"""
        if tuple(self.shape) != tuple(o.shape):
            raise HgpuError(1, "szipWith0N: the two arrays differ in shape")
        return f(IxV.from_val(self), IxV.from_val(o)).to_val()

    # -- reductions and contractions
    def ssum(self): return _c.tssumN(self.host, self, 1)
    def ssumN(self, k): return _c.tssumN(self.host, self, k)
    def ssum0(self): return _c.tssum0(self.host, self)
    def sdot0(self, o): return _c.tsdot0(self.host, self, o)
    def sdot1In(self, o): return _c.tsdot1In(self.host, self, o)
    def sdotNIn(self, o, n): return _c.tsdotNIn(self.host, self, o, n)
    def as_input(self): return _c.as_input(self.host, self)
    def sprimalPart(self): return _c.tprimalPart(self.host, self)
    def tD(self, dual): return _c.tD(self.host, self, dual)
    def tconvert(self, conv, shape=None):
        """ConvertTensor: "kfromS", "sfromK", "sfromR", "rfromS", "sfromX", "xfromS", "nest", "unnest";
        shape = the shape the shaped type names (sfromR / sfromX) or the outer dims (nest / unnest)."""
        kinds = ["kfromS", "sfromK", "sfromR", "rfromS", "sfromX", "xfromS", "nest", "unnest"]
        sh = list(shape) if shape is not None else []
        return _c.tconvert(self.host, kinds.index(conv), self, sh)

    def smatvecmul(self, v): return _c.tsmatvecmul(self.host, self, v)
    def smatmul2(self, o): return _c.tsmatmul2(self.host, self, o)
    def sargMax(self): return _c.tsargminmax(self.host, self, 1)
    def sargMin(self): return _c.tsargminmax(self.host, self, 0)

    # -- structure
    def sreplicate(self, k): return _c.tsreplicateN(self.host, self, (k,))
    def sreplicateN(self, shm): return _c.tsreplicateN(self.host, self, shm)
    sreplicate0N = sreplicateN
    def sappend(self, o): return _c.tsappend(self.host, self, o)
    def sslice(self, i, n): return _c.tsslice(self.host, self, i, n)
    def sreverse(self): return _c.tsreverse(self.host, self)
    def stranspose(self, perm): return _c.tstranspose(self.host, self, perm)
    def str_(self): return self.stranspose([1, 0])
    def sreshape(self, shape): return _c.tsreshape(self.host, self, shape)
    def sindex(self, ix): return _c.tsindex(self.host, self, ix)   # `!$` with concrete indices

    # -- indexing with index functions
    def dense(self):
        """The primal part as a dense row-major array (a copy when the value is a strided view)."""
        return _c.dense(self.host, self)

    def sgather(self, shm, f):
        """sgather @shm self (\\[i...] -> [ix...])"""
        shm, ix = self.host._apply_index_fn(shm, f)
        return _c.tsgather(self.host, self, shm, ix)

    def sscatter(self, rank_m, shp, f):
        """sscatter @shm self (\\[i...] -> [ix...]) with shm = the first rank_m dims; result shp ++ rest"""
        shm, ix = self.host._apply_index_fn(self.shape[:rank_m], f)
        if len(ix) != len(shp):
            raise HgpuError(1, "sscatter: the index function must return one index per dim of shp")
        return self.host._out(self.host.dll.hh_tsscatter, self.h, rank_m, len(ix), _larr(shp), (C.c_void_p * max(len(ix), 1))(*[x.h for x in ix]))

    # inside index functions
    def sindex0(self, ix):
        """self `sindex0` [ix...] with lane-batched indices"""
        first = next(x for x in ix if isinstance(x, IxV))
        ix = [x if isinstance(x, IxV) else IxV.const(self.host, first.shm, x) for x in ix]
        return _c.ix_index0(self.host, self, ix)

    def kargMax(self, ix, want_max=True):
        """kargMax (self !$ [ix...])"""
        first = next(x for x in ix if isinstance(x, IxV))
        ix = [x if isinstance(x, IxV) else IxV.const(self.host, first.shm, x) for x in ix]
        return _c.ix_argminmax(self.host, self, ix, int(want_max))

    def kargMin(self, ix):
        return self.kargMax(ix, want_max=False)

    def lift(self, shm):
        """A rank-0 tensor as a scalar of the position space shm."""
        return _c.ix_lift(self.host, shm, self)


# Ranked (`tr*`, user-facing `r*`) and mixed (`tx*` / `x*`) methods of the tensor
# class (Ops.hs:297-1255): the ABI takes shapes at run time, so a ranked or
# mixed method is its shaped twin under another name -- the same entry point,
# the same kernel.  `rtr` = `str_`, `rmaxIndex` / `rminIndex` = `sargMax` /
# `sargMin` as in the reference's naming.
_TWINS = ["map0N", "zipWith0N", "cast", "fromIntegral", "floor", "sum", "sumN", "sum0", "dot0", "dot1In", "dotNIn", "matvecmul", "matmul2",
          "replicate", "replicateN", "append", "slice", "reverse", "transpose", "reshape", "index", "gather", "scatter", "index0"]
for _n in _TWINS:
    for _p in ("r", "x"):
        setattr(V, _p + _n, getattr(V, "s" + _n))
for _p in ("r", "x"):
    setattr(V, _p + "tr", V.str_)
    setattr(V, _p + "maxIndex", V.sargMax)
    setattr(V, _p + "minIndex", V.sargMin)
    setattr(Host, _p + "concrete", Host.sconcrete)
    setattr(Host, _p + "repl", Host.srepl)
    setattr(Host, _p + "iota", Host.siota)
    setattr(Host, _p + "fromVector", Host.sfromVector)
    setattr(Host, _p + "build1", Host.sbuild1)
    setattr(Host, _p + "build", Host.sbuild)
    setattr(Host, _p + "mapAccumL", Host.smapAccumL)
