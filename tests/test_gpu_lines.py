"""The field-line kernels' lane pairs (rapt_halfbounce, rapt_eye,
rapt_bounce_labels, rapt_bounce_center_advance), where they can go wrong:

- lines of few points and of many (three, four and five points, odd and even
  counts, more points than the first scratch size holds) against the host
  restatement of flutils.halfbouncepath (rapt/flutils.py:254-316), which
  traces and interpolates the same points and integrates with QUADPACK at
  epsrel 1e-4, the bar here;
- batches around the sizes of a wave, a group of lines and an ordered chunk:
  every line's result is its own, whatever the batch it is in, bit for bit."""
import numpy as np
import pytest

import rapt_amd as rapt
from rapt_amd import _native as N
from rapt_amd import constants as K
from rapt_amd import fields as F
from rapt_amd import flutils

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res,alpha", [(2, 20), (2, 60), (5, 35), (5, 75), (50, 89.9), (50, 89.3),
                                       (50, 88.6), (50, 88.0), (50, 40), (400, 20)])
@pytest.mark.parametrize("model", ["dipole", "double"])
def test_point_counts_vs_host(monkeypatch, model, res, alpha):
    f = F.EarthDipole() if model == "dipole" else F.DoubleDipole()
    monkeypatch.setitem(rapt.params, "fieldlineresolution", res)
    tpos = np.array([0.0, 3.1 * K.Re, 2.4 * K.Re, 0.0])
    Bm = f.magB(tpos) / np.sin(np.radians(alpha)) ** 2
    ref = flutils.halfbouncepath(tpos, f, Bm)
    sb, st = N.context().halfbounce(f.descriptor(), tpos, Bm, res)
    assert st[0] == 1
    np.testing.assert_allclose(sb[0], ref, rtol=1e-4)


def _starts(n):
    rng = np.random.default_rng(n)
    L, ph = rng.uniform(3, 7, n) * K.Re, rng.uniform(0, 6.28, n)
    f = F.DoubleDipole()
    tpos = np.c_[np.zeros(n), L * np.cos(ph), L * np.sin(ph), np.zeros(n)]
    ctx = N.context()
    B = ctx.field_eval(f.descriptor(), "magB", tpos)[:, 0]
    return ctx, f.descriptor(), tpos, B / np.sin(np.radians(rng.uniform(15, 89.9, n))) ** 2, rng


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 4095, 4096, 4099, 70001])
@pytest.mark.parametrize("what", ["halfbounce", "eye"])
def test_lines_do_not_depend_on_their_batch(what, n):
    ctx, d, tpos, Bm, rng = _starts(n)
    fn = getattr(ctx, what)
    out, st = fn(d, tpos, Bm, 50)
    assert np.all(st == 1)
    back, _ = fn(d, tpos[::-1], Bm[::-1], 50)
    np.testing.assert_array_equal(back[::-1], out)
    for i in rng.integers(0, n, 5):
        np.testing.assert_array_equal(fn(d, tpos[i], Bm[i], 50)[0], out[i:i + 1])


@pytest.mark.parametrize("n", [1, 5, 6, 7, 61, 4096, 12300])
def test_labels_do_not_depend_on_their_batch(n):
    rng = np.random.default_rng(n)
    q = np.c_[rng.uniform(2, 8, n), rng.uniform(10, 89.9, n), rng.uniform(4, 7, n)]
    d = F.DipolePlusUniform(Bu=(0.0, 0.0, -10e-9)).descriptor()

    def labels(x):
        return N.context().bounce_labels(d, x, K.m_pr, K.e, 0.03 * K.Re, 50)
    out, st = labels(q)
    back, sb = labels(q[::-1])
    np.testing.assert_array_equal(back[::-1], out)
    np.testing.assert_array_equal(sb[::-1], st)
    for i in rng.integers(0, n, 5):
        np.testing.assert_array_equal(labels(q[i])[0], out[i:i + 1])


def test_long_lines_take_the_larger_scratch():
    """More points a half line than the first attempt's scratch holds: labels
    and bounce centres agree with the default resolution's to the quadrature's
    5e-5, and centres come out the same alone and in a batch."""
    d = F.EarthDipole().descriptor()
    ctx = N.context()
    q = np.array([[4.0, 15.0, 6.0], [6.5, 70.0, 5.0], [5.0, 12.0, 6.5]])
    fine, st = ctx.bounce_labels(d, q, K.m_pr, K.e, 0.03 * K.Re, 300)
    base, _ = ctx.bounce_labels(d, q, K.m_pr, K.e, 0.03 * K.Re, 50)
    assert np.all(st == 1)
    np.testing.assert_allclose(fine[:, [0, 2]], base[:, [0, 2]], rtol=5e-5)
    tpos = np.c_[np.zeros(3), q[:, 0] * K.Re, np.zeros((3, 2))]
    Bm = K.B0 / q[:, 0] ** 3 / np.sin(np.radians(q[:, 1])) ** 2
    coef, dt = 2e6 + np.zeros(3), np.array([1.0, 0.5, 2.0])
    rows, end, st, _ = ctx.bounce_center_advance(d, tpos, Bm, coef, dt, 0.0, 2, 1e-6, 1e-6,
                                                 0.03 * K.Re, 300)
    assert np.all(st == 1)
    for i in range(3):
        r1, e1, _, _ = ctx.bounce_center_advance(d, tpos[i], Bm[i], coef[i], dt[i], 0.0, 2, 1e-6,
                                                 1e-6, 0.03 * K.Re, 300)
        np.testing.assert_array_equal(r1[0], rows[i])
        np.testing.assert_array_equal(e1[0], end[i])
