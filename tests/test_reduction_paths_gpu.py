"""Reductions on either side of the line where the second pass is a launch of its own, and
vectors kept by a context from one run to the next, on MI355X."""
import ctypes as C
import math

import numpy as np
import pytest

from pihm_amd import _lib
from pihm_amd.forcing import StormForcing, run_config
from pihm_amd.rhs import HipRHS, run_gpu

pytestmark = pytest.mark.gpu
TICKET = 64 * 512     # entries of 64 workgroups: up to here the last workgroup does the second pass


def _dp(a):
    return a.ctypes.data_as(_lib.c_double_p)


def _vec(L, a):
    v = L.N_VNew_Hip(len(a))
    assert L.N_VCopyToDevice_Hip(v, _dp(a)) == 0
    return v


@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 512, 513, 1025, TICKET - 1, TICKET, TICKET + 1, 2 * TICKET,
                               1024 * 512 - 1, 1024 * 512 + 1, 608190])
def test_reductions_at_every_length(n):
    """The sums equal the two-launch dot product of the no-allocation entry point bit for bit
    at every length (one tree for both), twice in a row; the others equal numpy's exactly or
    within n roundings."""
    L = _lib.lib()
    rng = np.random.default_rng(n)
    x, w = np.ascontiguousarray(rng.standard_normal(n)), np.ascontiguousarray(rng.uniform(0.5, 2.0, n))
    print(f"[reductions] n {n}", flush=True)
    X, W, R = _vec(L, x), _vec(L, w), L.N_VNew_Hip(1)
    one = np.zeros(1)
    for _ in range(2):
        d = L.N_VDotProd_Hip(X, W)
        assert L.pihm_nv_dotprod_noalloc(n, L.N_VGetDeviceArrayPointer_Hip(X), L.N_VGetDeviceArrayPointer_Hip(W),
                                         L.N_VGetDeviceArrayPointer_Hip(R), None) == 0
        assert L.N_VCopyFromDevice_Hip(R, _dp(one)) == 0
        assert d == one[0]
        arr = (C.c_void_p * 3)(W, X, W)
        out = np.zeros(3)
        assert L.N_VDotProdMulti_Hip(3, X, arr, _dp(out)) == 0
        assert out[0] == d and out[2] == d and out[1] == L.N_VDotProd_Hip(X, X)
        assert L.N_VMaxNorm_Hip(X) == np.max(np.abs(x))
        assert L.N_VMin_Hip(X) == np.min(x)
        assert L.N_VMinQuotient_Hip(X, W) == np.min(x / w)
        # n additions of terms whose magnitudes sum to S: at most n roundings of S
        assert abs(L.N_VL1Norm_Hip(X) - math.fsum(np.abs(x))) <= n * 2.0 ** -53 * math.fsum(np.abs(x))
        q = math.fsum((x * w) ** 2)
        assert abs(L.N_VWrmsNorm_Hip(X, W) - math.sqrt(q / n)) <= (n + 4) * 2.0 ** -53 * math.sqrt(q / n)
    for v in (X, W, R):
        L.N_VDestroy_Hip(v)


def test_runs_on_one_context_equal_runs_on_new_ones(tree_small):
    """A context keeps the integrator's vectors: a second run, a run after the state's length
    changed (closure on and off) and a run after one that failed give the bits of a run on a
    context of its own."""
    m = tree_small
    f = StormForcing(3, seed=5, nelem=m.nelem, p_wet=0.8)
    y0, cfg = m.initial_state(), run_config(300.0)
    rc, ref, _ = run_gpu(m, f, cfg, y0)
    assert rc == 0
    _, refc, _ = run_gpu(m, f, cfg, y0, closure=True)
    h = HipRHS(m, nan_check=False)
    fs = f.struct()
    bad = run_config(300.0, max_steps_per_call=1)
    zero = np.zeros(3 * m.nelem)
    for k, kind in enumerate(["plain", "plain", "closure", "plain", "fails", "plain"]):
        print(f"[reuse] run {k} {kind}", flush=True)
        assert h.L.pihm_ctx_set_closure(h.ctx, 1 if kind == "closure" else 0) == 0
        h.set_river_edge_ovlflow(zero)
        y = np.concatenate([y0, np.zeros(4)]) if kind == "closure" else y0.copy()
        st = _lib.RunStats()
        c = bad if kind == "fails" else cfg
        rc = h.L.pihm_run_gpu(h.ctx, C.byref(fs), C.byref(c), _dp(y), C.byref(st))
        if kind == "fails":
            assert rc != 0
        else:
            assert rc == 0 and np.array_equal(y, refc if kind == "closure" else ref)
    h.close()
