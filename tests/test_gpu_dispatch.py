"""Runs that the dispatch sends to kernels or layouts of their own: they return
the bits of the general form."""
import numpy as np
import pytest

from rapt_amd import _native as N
from rapt_amd import batch
from rapt_amd import constants as K
from rapt_amd import fields as F
from rapt_amd import params, workloads as W

pytestmark = pytest.mark.gpu


def _same(got, ref):
    np.testing.assert_array_equal(got.status, ref.status)
    for a, b in zip(got.rows, ref.rows):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("adaptive", [False, True])
def test_static_field_kernels_equal_the_general_ones(adaptive):
    """Protons in the equatorial plane of the dipole: the equatorial constraint
    changes nothing there, and with it a run takes the general kernel.  (A
    momentum converted from a guiding centre has a rounding's pz, 1e-36 kg m/s,
    that the constraint drops: compared up to a tracer's first conversion.)"""
    rng = np.random.default_rng(7)
    n = 67
    r, phi, a = rng.uniform(3, 7, n) * K.Re, *rng.uniform(0, 2 * np.pi, (2, n))
    pos = np.stack([r * np.cos(phi), r * np.sin(phi), 0 * r], axis=1)
    v = 10.0 ** rng.uniform(6.5, 8.3, n)
    vel = np.stack([v * np.cos(a), v * np.sin(a), 0 * v], axis=1)
    f = F.EarthDipole()
    runs = []
    for eq in (False, True):
        prm = dict(params, **{"enforce equatorial": eq, "GCtimestep": 0.2})
        if adaptive:
            runs.append(batch.advance_adaptive(f, pos, vel, 0.0, K.m_pr, K.e, 2.0, params=prm))
        else:
            g = 1 / np.sqrt(1 - (v / K.c) ** 2)
            last = np.c_[0 * r, pos, K.m_pr * g[:, None] * vel]
            runs.append(batch.advance_particles(f, last, K.m_pr, K.e, 2.0, params=prm))
    assert np.all(runs[0].status == 1) and min(len(x) for x in runs[0].rows) > 3
    np.testing.assert_array_equal(runs[1].status, runs[0].status)
    for got, ref in zip(runs[1].rows, runs[0].rows):
        to_p = np.flatnonzero(np.diff(ref[:, 0]) < 0) if adaptive else []
        k = to_p[0] + 2 if len(to_p) else len(ref)
        assert len(to_p) or len(got) == len(ref)
        np.testing.assert_array_equal(got[:k], ref[:k])


@pytest.mark.parametrize("n", [1, 1025, 2049])
def test_adaptive_particles_spread_over_waves(n):
    """One, two and four particles a wave (one wave a SIMD is 1,024), the last
    wave not full, against 64 a wave."""
    w = W.current_sheet_protons(n=n)
    f = F.CurrentSheet()
    prm = dict(params, GCtimestep=0.5)
    arg = (f, w["pos"], w["vel"], 0.0, K.m_pr, K.e, 3.0)
    _same(batch.advance_adaptive(*arg, params=prm),
          batch.advance_adaptive(*arg, params=prm, lanes=n + 63 & ~63))


@pytest.mark.parametrize("n", [1, 9, 8193, 16385, 32769, 98305])
def test_default_guiding_centre_layout_and_order(n):
    """Octets up to 16,384, quads up to 32,768, quads and pairs up to 98,304 and
    pairs above, taken in the order of r / v where the output steps are equal;
    against one lane a particle, and that in input order (one step differs by a
    part in 1e12 from the rest)."""
    w = W.doubledipole_electrons_gc(n=n)
    f = F.DoubleDipole()
    v = w["v"]
    g = 1 / np.sqrt(1 - (v / K.c) ** 2)
    last = np.c_[np.zeros(n), w["pos"], K.m_el * g * v * np.cos(np.radians(w["pa"]))]
    B = N.context().field_eval(f.descriptor(), "magB", last[:, :4])[:, 0]
    mu = (K.m_el * g * v * np.sin(np.radians(w["pa"]))) ** 2 / (2 * K.m_el * B)
    prm = dict(params, solvertolerances=(1e-8, 1e-8))
    dt = np.full(n, 0.05)
    got = batch.advance_gcs(f, last, K.m_el, -K.e, mu, v, dt, 0.2, params=prm)
    one = batch.advance_gcs(f, last, K.m_el, -K.e, mu, v, dt, 0.2, params=prm,
                            lanes_per_particle=1)
    dt[0] *= 1 + 1e-12
    ref = batch.advance_gcs(f, last, K.m_el, -K.e, mu, v, dt, 0.2, params=prm,
                            lanes_per_particle=1)
    assert np.all(got.status == 1)
    _same(got, one)
    np.testing.assert_array_equal(got.status[1:], ref.status[1:])
    for a, b in zip(got.rows[1:], ref.rows[1:]):
        np.testing.assert_array_equal(a, b)
