"""The host side of librapt_hip.so (what it launches, allocates, keeps and
copies) on a HIP runtime without a device (fake_hip.c), whose kernels do
nothing.  Each case runs in a process of its own, with that runtime loaded in
front of the library."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import rapt_amd as rapt  # noqa: E402
from rapt_amd import _native as N  # noqa: E402
from rapt_amd import fields as F  # noqa: E402

GIB = 1 << 30


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.check_call(["cc", "-shared", "-fPIC", "-O1", "-I/opt/rocm/include", "-o", so,
                           os.path.join(HERE, "fake_hip.c")])
    return so


def _run(fake, case, *args):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), fake, case] +
                       [str(a) for a in args], capture_output=True, text=True, cwd=ROOT)
    assert r.returncode == 0, r.stderr[-2000:]


class _Grid(F.Grid):
    def parsefile(self, filename):
        a = np.linspace(-8, 8, 9) * rapt.Re
        X = np.meshgrid(a, a, a, indexing="ij")[0]
        z = 0 * X
        return dict(time=0.0, x=a, y=a, z=a, Bx=z, By=z, Bz=z + 1e-7, Ex=z, Ey=z, Ez=z)


class _User(F._Field):
    def B(self, tpos):
        t, x, y, z = tpos
        return np.array([0 * x, 0 * y, 1e-7 * (1 + x * x)])


def _field(name):
    return {"dipole": F.EarthDipole, "double": F.DoubleDipole, "uniform": F.DipolePlusUniform,
            "grid": lambda: _Grid(["0"]), "user": _User}[name]()


def _ctx(field):
    ctx = N.context()
    ctx.set_expr_mode(False)
    ctx.set_field(field.descriptor())
    return ctx


class _Var:
    """A variable of the fake runtime."""

    def __init__(self, lib):
        self._lib = lib

    def __getattr__(self, name):
        t = {"fake_budget": C.c_size_t, "fake_used": C.c_size_t, "fake_largest_copy": C.c_size_t,
             "fake_overflow_bytes": C.c_size_t, "fake_last_grid": C.c_uint,
             "fake_last_kernel": C.c_char_p}.get(name, C.c_int)
        return t.in_dll(self._lib, name)


# ---- field-line launches ------------------------------------------------------------


def case_labels(rt, name, n, attempt):
    f = _field(name)
    q = np.tile([4.0, 45.0, 5.0], (n, 1))
    if attempt == 2:
        rt.fake_overflow_bytes.value = 4 * n  # every status of the first attempt
    _ctx(f).bounce_labels(f.descriptor(), q, rapt.m_pr, rapt.e, 1e3, 50)
    assert b"k_bounce_labels" in rt.fake_last_kernel.value
    assert rt.fake_last_grid.value == min((n + 5) // 6, 2048 if attempt == 1 else 512)


@pytest.mark.parametrize("name,n,attempt", [("grid", 16384, 1), ("user", 16384, 1),
                                            ("user", 65536, 1), ("grid", 300, 1),
                                            ("dipole", 16384, 2), ("uniform", 4000, 2),
                                            ("user", 65536, 2)])
def test_labels_fill_the_gpu(fake, name, n, attempt):
    """Labels in fields whose evaluation is most of a line, and lines too long
    for the first scratch size, run with every wave that the scratch has."""
    _run(fake, "case_labels", name, n, attempt)


if __name__ == "__main__":
    _lib = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
    globals()[sys.argv[2]](_Var(_lib), *[int(a) if a.lstrip("-").isdigit() else a
                                         for a in sys.argv[3:]])
