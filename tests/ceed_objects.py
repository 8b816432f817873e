"""libCEED objects made through the C API on a problem's Ceed, for tests of operators that the framework's own setup does not make."""
import ctypes as ct

import numpy as np

from pyhonee.driver import CEED_MEM_HOST, load_libs

COPY_VALUES, (NONE, INTERP, GRAD) = 0, (0, 1, 2)


class CeedObjects:
    def __init__(self, prob):
        self.lib, self.prob, self.ceed = load_libs()[0], prob, ct.c_void_p(prob.ceed)
        self.host = ct.CFUNCTYPE(ct.c_int, ct.c_void_p, ct.c_int, ct.c_void_p, ct.c_void_p)(lambda *a: 1)
    def _symbol(self, name):
        return ct.byref(ct.c_int.in_dll(self.lib, name))

    def _pointer(self, name):
        return ct.c_void_p.in_dll(self.lib, name)

    def _call(self, name, *args):
        if getattr(self.lib, name)(*args):
            msg = ct.c_char_p()
            self.lib.CeedGetErrorMessage(self.ceed, ct.byref(msg))
            raise RuntimeError(f"{name}: {msg.value.decode()}")

    def _made(self, name, *args):
        h = ct.c_void_p()
        self._call(name, *args, ct.byref(h))
        return h

    def _restriction(self, nelem, size, ncomp, length, offsets):
        off = np.ascontiguousarray(offsets, dtype=np.int32)
        return self._made("CeedElemRestrictionCreate", self.ceed, nelem, size, ncomp, 1, ct.c_longlong(length), CEED_MEM_HOST, COPY_VALUES,
                          off.ctypes.data_as(ct.c_void_p))

    def _basis(self, ncomp, P, B, D):
        k = self.prob._keep
        return self._made("CeedBasisCreateTensorH1", self.ceed, 3, ncomp, P, self.prob.tab.Q, *(a.ctypes.data_as(ct.c_void_p) for a in (B, D, k["qref"], k["qweight"])))

    def vector(self, a):
        a = np.ascontiguousarray(a, dtype=np.float64).ravel()
        v = self._made("CeedVectorCreate", self.ceed, ct.c_longlong(a.size))
        self._call("CeedVectorSetArray", v, CEED_MEM_HOST, COPY_VALUES, a.ctypes.data_as(ct.c_void_p))
        return v

    def strided(self, n):
        nelem, Q3 = self.prob.mesh.nelem, self.prob.tab.Q ** 3
        return self._made("CeedElemRestrictionCreateStrided", self.ceed, nelem, Q3, n, ct.c_longlong(nelem * Q3 * n), self._symbol("CEED_STRIDES_BACKEND"))

    def operator(self, source, context, ins, outs, fields):
        """ins, outs: (name, size, mode); fields: name -> (restriction, basis, vector)."""
        qf = self._made("CeedQFunctionCreateInterior", self.ceed, 1, self.host, source.encode())
        if context is not None:
            self._call("CeedQFunctionSetContext", qf, context)
        for name, size, mode in ins:
            self._call("CeedQFunctionAddInput", qf, name.encode(), size, mode)
        for name, size, mode in outs:
            self._call("CeedQFunctionAddOutput", qf, name.encode(), size, mode)
        op = self._made("CeedOperatorCreate", self.ceed, qf, None, None)
        for name, f in fields.items():
            self._call("CeedOperatorSetField", op, name.encode(), *f)
        return op

    def read(self, v, n):
        p, out = ct.POINTER(ct.c_double)(), np.zeros(n)
        self._call("CeedVectorGetArrayRead", v, CEED_MEM_HOST, ct.byref(p))
        out[:] = np.ctypeslib.as_array(p, (n,))
        self._call("CeedVectorRestoreArrayRead", v, ct.byref(p))
        return out
