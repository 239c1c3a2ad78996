"""Surrogate labels on more than 72 waves (gridded and user-written fields, and
the second attempt at lines of many points): every query's labels are its own,
whatever the batch it is in, bit for bit."""
import numpy as np
import pytest

from rapt_amd import _native as N
from rapt_amd import constants as K
from rapt_amd import fields as F

pytestmark = pytest.mark.gpu


class _Written(F._Field):
    def __init__(self):
        F._Field.__init__(self)
        self.gradientstepsize = K.Re / 1000

    def B(self, tpos):
        t, x, y, z = tpos
        r2 = x * x + y * y + z * z
        return -K.B0 * K.Re ** 3 * np.array([3 * x * z, 3 * y * z, 2 * z * z - x * x - y * y]) \
            / pow(r2, 5.0 / 2.0)


class _Sampled(F.Grid):
    def parsefile(self, filename):
        a = (np.linspace(-8, 8, 65) + 0.02) * K.Re
        z = (np.linspace(-4, 4, 65) + 0.02) * K.Re
        X, Y, Z = np.meshgrid(a, a, z, indexing="ij")
        r2 = X * X + Y * Y + Z * Z
        s = -3 * K.B0 * K.Re ** 3 / np.maximum(r2, K.Re ** 2) ** 2.5
        return dict(time=0.0, x=a, y=a, z=z, Bx=s * X * Z, By=s * Y * Z,
                    Bz=s * (Z * Z - r2 / 3), Ex=0 * X, Ey=0 * X, Ez=0 * X)


@pytest.mark.parametrize("field,compiled,n,res", [(_Written, True, 2500, 50),
                                                  (_Written, True, 500, 400),
                                                  (_Written, False, 500, 50),
                                                  (lambda: _Sampled(["0"]), True, 2500, 50),
                                                  (F.EarthDipole, True, 500, 400)])
def test_labels_do_not_depend_on_their_wave(field, compiled, n, res):
    rng = np.random.default_rng(n)
    q = np.c_[rng.uniform(3, 5, n), rng.uniform(35, 89, n), rng.uniform(4, 7, n)]
    ctx = N.context()
    d = field().descriptor()
    ctx.set_expr_mode(compiled)
    try:
        def labels(x):
            return ctx.bounce_labels(d, x, K.m_pr, K.e, 0.05 * K.Re, res)
        out, st = labels(q)
        back, sb = labels(q[::-1])
        np.testing.assert_array_equal(back[::-1], out)
        np.testing.assert_array_equal(sb[::-1], st)
        assert np.mean(st == 1) > 0.99
        for i in rng.integers(0, n, 3):
            np.testing.assert_array_equal(labels(q[i])[0], out[i:i + 1])
    finally:
        ctx.set_expr_mode(True)
