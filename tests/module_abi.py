"""The Module vtable of include/nn_modules.h for tests that drive modules from Python."""
from __future__ import annotations

import ctypes as C

import numpy as np

P, I, F = C.c_void_p, C.c_int, C.c_float


class _CondSlot(C.Structure):
    _fields_ = [("fwd", P), ("grad", P), ("dim", I)]


class Context(C.Structure):
    _fields_ = [("blas", P), ("rng", C.c_uint64 * 4), ("stream", P), ("cond", _CondSlot * 4), ("n_cond", I)]


class _Param(C.Structure):
    _fields_ = [("param", P), ("grad", P), ("size", I)]


class _ParamList(C.Structure):
    _fields_ = [("items", C.POINTER(_Param)), ("count", I), ("capacity", I)]


class _Module(C.Structure):
    pass


_Module._fields_ = [("name", C.c_char_p), ("in_dim", I), ("out_dim", I), ("state", P),
                    ("forward", C.CFUNCTYPE(None, C.POINTER(_Module), P, P, I, C.POINTER(Context))),
                    ("backward", C.CFUNCTYPE(None, C.POINTER(_Module), P, P, P, P, I, C.POINTER(Context))),
                    ("parameters", C.CFUNCTYPE(None, C.POINTER(_Module), C.POINTER(_ParamList))),
                    ("free", C.CFUNCTYPE(None, C.POINTER(_Module)))]

_CREATE = {"linear_create": [I, I], "mp_linear_create": [I, I, F], "conv2d_create": [I] * 9 + [F]}


class Module:
    """A module of library L with its own context: create(name, *args), then params() and calls on device pointers."""

    def __init__(self, L, name, *args, stream=None):
        self.d = L.dll
        self.ctx = Context()
        self.d.nn_context_init.argtypes = [C.POINTER(Context), C.c_uint64, P]
        self.d.nn_context_destroy.argtypes = [C.POINTER(Context)]
        self.d.nn_context_init(C.byref(self.ctx), 17, stream)
        create = getattr(self.d, name)
        create.restype, create.argtypes = C.POINTER(_Module), [C.POINTER(Context)] + _CREATE[name]
        self.m = create(C.byref(self.ctx), *args)

    def params(self):
        """[(value pointer, gradient pointer, floats)]"""
        pl = _ParamList()
        self.d.param_list_init.argtypes = self.d.param_list_free.argtypes = [C.POINTER(_ParamList)]
        self.d.param_list_init(C.byref(pl))
        self.m.contents.parameters(self.m, C.byref(pl))
        got = [(pl.items[i].param, pl.items[i].grad, pl.items[i].size) for i in range(pl.count)]
        self.d.param_list_free(C.byref(pl))
        return got

    def set(self, i, value):
        value = np.ascontiguousarray(value, np.float32)
        ptr, _, n = self.params()[i]
        assert n == value.size
        self.d.nnhip_memcpy_htod(C.c_void_p(ptr), value.ctypes.data_as(P), C.c_size_t(4 * n))

    def get(self, i, grad=False):
        ptr, gptr, n = self.params()[i]
        out = np.empty(n, np.float32)
        self.d.nnhip_memcpy_dtoh(out.ctypes.data_as(P), C.c_void_p(gptr if grad else ptr), C.c_size_t(4 * n))
        return out

    def forward(self, x, y, batch):
        self.m.contents.forward(self.m, x, y, batch, C.byref(self.ctx))

    def backward(self, x, y, gy, gx, batch):
        self.m.contents.backward(self.m, x, y, gy, gx, batch, C.byref(self.ctx))

    def free(self):
        self.m.contents.free(self.m)
        self.d.nn_context_destroy(C.byref(self.ctx))
