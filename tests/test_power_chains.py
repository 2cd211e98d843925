"""The powers outside their ordinary range: xpow's special and extreme arguments against
the host libm, and on MI355X the retention curve where the RHS leaves its paired powers
(beta / (beta - 1) of 300 or more, or beta <= 1) and on either side of that line."""
import copy

import numpy as np
import pytest

import oracle as O
from conftest import assert_rhs_close
from test_xmath import _ulps, xpow


def test_xpow_special_arguments_follow_libm():
    v = np.array([0.0, -0.0, 1.0, -1.0, 2.0, -2.0, 0.5, -0.5, 3.0, -3.0, 1e300, -1e300, 1e-300, np.inf, -np.inf, np.nan])
    x, y = (a.ravel() for a in np.meshgrid(v, v))
    with np.errstate(all="ignore"):
        ref = np.power(x, y)
    got = xpow(x, y)
    # exact cases are exact; finite, non-zero results within the ulps of the ordinary range
    plain = np.isfinite(ref) & (ref != 0.0)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[~plain & ~np.isnan(ref)], ref[~plain & ~np.isnan(ref)])
    assert np.array_equal(np.signbit(got[~np.isnan(ref)]), np.signbit(ref[~np.isnan(ref)]))
    assert np.all(_ulps(got[plain], ref[plain]) <= 2)


def test_xpow_at_the_ends_of_the_range():
    rng = np.random.default_rng(4)
    x = 10 ** rng.uniform(-300, 300, 20000)
    y = np.log(10.0) * rng.choice([-1, 1], 20000) * rng.uniform(306, 330, 20000) / np.log(x)
    with np.errstate(all="ignore"):
        ref = np.power(x, y)
    got = xpow(x, y)
    normal = np.isfinite(ref) & (ref > 2.3e-308)
    # ln x carries 1.2e-16 absolute, y ln x |y| times that, and exp about an ulp each side
    ulps = 2.0 + 1.2e-16 * np.abs(y) / 2.0 ** -53
    assert np.all(_ulps(got[normal], ref[normal]) <= ulps[normal])
    # subnormal results: the same relative error and the rounding to a step, on each side
    small = ref <= 2.3e-308
    assert np.all(np.abs(got[small] - ref[small]) <= 2 * 4.95e-324 + ulps[small] * 2.0 ** -52 * ref[small])
    assert np.array_equal(got[~np.isfinite(ref)], ref[~np.isfinite(ref)])


@pytest.mark.gpu
@pytest.mark.parametrize("beta", [1.003, 1.0034, 1.01, 1.3, 2.0, 5.0])
@pytest.mark.parametrize("path", [0, 1])
def test_rhs_over_the_range_of_beta(c0, beta, path):
    from pihm_amd.rhs import HipRHS
    m = copy.copy(c0)
    m.a = dict(c0.a)
    m.a["beta"] = np.full(m.nelem, beta)
    m._keep = []
    rng = np.random.default_rng(3)
    y = m.initial_state()
    ne = m.nelem
    y[:ne] = rng.uniform(0.0, 2e-2, ne)
    # saturations between dry and full, some exactly full
    gw = m.a["depth"] * rng.uniform(0.1, 0.9, ne)
    y[ne:2 * ne] = (m.a["depth"] - gw) * np.where(rng.random(ne) < 0.1, 1.0, rng.uniform(0.05, 1.0, ne))
    y[2 * ne:3 * ne] = gw
    inp = dict(pcpdrp=rng.uniform(0, 3e-6, ne), ws0_surf=rng.uniform(0, 1e-3, ne))
    print(f"[beta] {beta} path {path}", flush=True)
    h, o = HipRHS(m, rhs_path=path), O.OracleRHS(m)
    h.set_step_inputs(**inp)
    o.set_step_inputs(**inp)
    rc_h, dh = h.ode(y)
    rc_o, do, mag = o.ode(y, with_mag=True)
    h.close()
    assert rc_h == rc_o
    # an exponent of e1 = beta / (beta - 1) multiplies the half-ulp of ln s: e1 |ln s| eps on the
    # power, and (1/s)^e1 - 1 near s = 1 again by its own size; 1e-12 holds for e1 up to a few tens
    e1 = beta / (beta - 1.0)
    fin = np.isfinite(do) & np.isfinite(mag)     # at 1.003 (1/s)^e1 overflows on both sides
    assert np.array_equal(dh[~fin], do[~fin], equal_nan=True)
    assert_rhs_close(dh[fin], do[fin], mag[fin], 1e-12 * max(1.0, e1 / 10.0), f"beta {beta}")
