"""The vectors that N_VInvTest and N_VConstrMask store are written when the calls return, on
MI355X: read at once through another stream."""
import ctypes as C

import numpy as np
import pytest

from pihm_amd import _lib

pytestmark = pytest.mark.gpu


def _dp(a):
    return a.ctypes.data_as(_lib.c_double_p)


@pytest.mark.parametrize("n", [1, 512, 513, 4097, 64 * 512 - 1, 64 * 512, 64 * 512 + 1, 200001])
def test_stored_vector_on_another_stream(n):
    L = _lib.lib()
    print(f"[tests that store] n {n}", flush=True)
    streams = [C.c_void_p(), C.c_void_p()]
    for s in streams:
        assert L.pihm_stream_create(C.byref(s)) == 0
    X, Cv, Z = (L.N_VNew_Hip(n) for _ in range(3))
    for v in (X, Cv, Z):
        L.N_VSetStream_Hip(v, streams[0])
    W = L.N_VMake_Hip(n, L.N_VGetDeviceArrayPointer_Hip(Z))     # the same memory, the other stream
    L.N_VSetStream_Hip(W, streams[1])
    got = np.zeros(n)
    for k in range(8):
        rng = np.random.default_rng([n, k])
        x = rng.choice([-1.0, 1.0], n) * rng.uniform(0.5, 2.0, n)
        c = rng.choice([-2.0, -1.0, 0.0, 1.0, 2.0], n)
        assert L.N_VCopyToDevice_Hip(X, _dp(x)) == 0 and L.N_VCopyToDevice_Hip(Cv, _dp(c)) == 0
        assert L.N_VInvTest_Hip(X, Z) == 1
        assert L.N_VCopyFromDevice_Hip(W, _dp(got)) == 0
        assert np.array_equal(got, 1.0 / x)
        bad = (x * c < 0).astype(float)
        assert L.N_VConstrMask_Hip(Cv, X, Z) == int(not bad.any())
        assert L.N_VCopyFromDevice_Hip(W, _dp(got)) == 0
        assert np.array_equal(got, bad)
    for v in (W, X, Cv, Z):
        L.N_VDestroy_Hip(v)
    for s in streams:
        L.pihm_stream_destroy(s)
