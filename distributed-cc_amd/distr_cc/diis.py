"""Pulay DIIS on device vectors (reference distr_cc/diis.py:25-177).

The history vectors, error vectors and the extrapolation live in HBM; only
the (space+1)^2 B matrix and its solve are on the host, as in the reference
(diis.py:118-167).  Error vectors are x - x_prev (diis.py:114); the B-matrix
row of the newest error is built from dot products (diis.py:122-132); the
coefficients come from eigh with a 1e-14 cutoff or a plain solve
(diis.py:157-167).  Every reduction is a deterministic FP64 device sum.
"""
import ctypes
import weakref

import numpy as np

from distr_cc import _lib as L
from distr_cc.device import DeviceArray


class _Iterate(DeviceArray):
    """An extrapolated vector.  Freed, it leaves its memory to its DIIS for the next one (one vector at most,
    released with the DIIS): allocating and releasing a vector of 116 MB costs as much as half a step.  As
    hipFree does, it first waits for everything on the device that may still read the vector."""

    def __init__(self, diis):
        spare, diis._spare = diis._spare, None
        super().__init__((diis.size,), ptr=spare)
        self._owner = True
        self._diis = weakref.ref(diis)

    def free(self):
        diis = self._diis()
        if self.ptr and diis is not None and diis._spare is None:
            L.call("dcc_device_synchronize")
            # another iterate may have been freed during the wait (by a thread, or by the garbage collector): its
            # memory is in this one's hands then
            self.ptr, diis._spare = diis._spare or 0, self.ptr
        super().free()


class DeviceDIIS:
    def __init__(self, size, space=6, stream=None):
        if int(space) <= 0:
            raise ValueError("DIIS space must be a positive integer")
        self.size, self.space, self.stream = int(size), int(space), stream
        self.xs = [None] * self.space
        self.es = [None] * self.space
        self._head, self._H, self._xprev = 0, None, None
        self.last_delta_norm_sq = None
        self._partials = DeviceArray((int(L._lib.dcc_diis_partials()),))
        self._out = DeviceArray((self.space,))
        self._spare = None    # memory of a freed extrapolated vector

    def __del__(self):
        try:
            if self._spare:
                L.call("dcc_free", ctypes.c_void_p(self._spare))
        except Exception:
            pass

    # device primitives
    def _h(self):
        return self.stream.handle if self.stream is not None else None

    def _copy(self, src):
        dst = DeviceArray((self.size,))
        L.call("dcc_memcpy_dtod", dst.vp, src.vp, dst.nbytes, self._h())
        return dst

    @staticmethod
    def _pointers(arrays):
        return (ctypes.c_void_p * len(arrays))(*[a.ptr for a in arrays])

    def update(self, x):
        """x: DeviceArray of ``size`` doubles; returns the extrapolated vector (a new
        DeviceArray) and keeps a copy of it as the next x_prev (diis.py:105-145)."""
        if self._xprev is None:
            self._xprev = self._copy(x)
            self.last_delta_norm_sq = None
            return self._copy(x)
        h = self._head
        if self.xs[h] is None:
            self.xs[h] = DeviceArray((self.size,))
            self.es[h] = DeviceArray((self.size,))
        nd = sum(v is not None for v in self.xs)
        if self._H is None:
            self._H = np.zeros((self.space + 1, self.space + 1))
            self._H[0, 1:] = self._H[1:, 0] = 1
        L.call("dcc_diis_push_f64", x.vp, self._xprev.vp, self.xs[h].vp, self._pointers(self.es[:nd]), nd, h, self.size,
               self._partials.vp, self._out.vp, self._h())
        self._H[h + 1, 1:nd + 1] = self._H[1:nd + 1, h + 1] = self._out.download(stream=self.stream)[:nd]
        self._head = (h + 1) % self.space
        return self._combine(nd, self._xprev)

    def coefficients(self, nd):
        h = self._H[:nd + 1, :nd + 1]
        g = np.zeros(nd + 1)
        g[0] = 1
        w, v = np.linalg.eigh(h)
        if np.any(abs(w) < 1e-14):
            idx = abs(w) > 1e-14
            return np.dot(v[:, idx] * (1 / w[idx]), np.dot(v[:, idx].T, g))
        return np.linalg.solve(h, g)

    def extrapolate(self, nd):
        """The extrapolated vector of the first ``nd`` history vectors (a new DeviceArray); nothing is kept."""
        c = self.coefficients(nd)[1:]
        xnew = DeviceArray((self.size,))
        lay = L.Strided()
        lay.ndim, lay.shape[0], lay.dst_stride[0], lay.src_stride[0] = 1, self.size, 1, 1
        for i, ci in enumerate(c):
            L.call("dcc_tensor_axpby_f64", xnew.vp, self.xs[i].vp, ctypes.byref(lay), float(ci), 0.0 if i == 0 else 1.0,
                   self._h())
        return xnew

    def _combine(self, nd, xprev):
        """The extrapolated vector, which also replaces ``xprev``; keeps the norm of the change."""
        c = np.ascontiguousarray(self.coefficients(nd)[1:], dtype=np.float64)
        xnew = _Iterate(self)
        L.call("dcc_diis_combine_f64", xnew.vp, xprev.vp, self._pointers(self.xs[:nd]),
               c.ctypes.data_as(ctypes.c_void_p), nd, self.size, self._partials.vp, self._out.vp, self._h())
        self.last_delta_norm_sq = max(float(self._out.download(stream=self.stream)[0]), 0.0)
        return xnew
