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


def _arg(text):
    try:
        return int(text)
    except ValueError:
        pass
    try:
        return float(text)
    except ValueError:
        return text


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
             "fake_overflow_bytes": C.c_size_t, "fake_last_grid": C.c_uint, "fake_last_block": C.c_uint,
             "fake_epoch_lanes": C.c_uint,
             "fake_last_kernel": C.c_char_p, "fake_epoch_kernel": C.c_char_p}.get(name, C.c_int)
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


# ---- guiding-centre layouts ----------------------------------------------------------


def case_layout(rt, name, n, costs, kernel, lanes):
    f = {"sheet": F.CurrentSheet, "bz": F.UniformBz}[name]() if name in ("sheet", "bz") \
        else _field(name)
    ctx = _ctx(f)
    S = np.zeros((N.NSLOT, n))
    S[N.S_Y0] = 5 * rapt.Re
    c = {"equal": np.ones(n), "spread": ((np.arange(n) + 1.0) / n) ** 2}[costs]
    S[N.S_V] = 1e8 * c
    S[N.S_DT] = 1.0
    b = N.Batch(ctx, n)
    b.upload(S, np.zeros(n, np.int32))
    b.set_rows(5, np.full(n, 1, np.int64))
    desc = N.make_desc(N.MODE_GC, rapt.params, 10.0)
    for how in ("uploaded", "set_cost"):
        if how == "set_cost":
            b.set_cost(c)
        b.run(desc)
        assert kernel in rt.fake_last_kernel.value.decode(), rt.fake_last_kernel.value
        assert rt.fake_last_grid.value * rt.fake_last_block.value == lanes


def case_short(rt, rows, n, v_r, kernel):
    """Runs and epochs of `rows` output steps of v_r times r / v."""
    ctx = _ctx(_field("double"))
    S = np.zeros((N.NSLOT, n))
    S[N.S_Y0] = 5 * rapt.Re
    S[N.S_V] = np.linspace(1e8, 0.2e8, n)
    S[N.S_DT] = v_r * S[N.S_Y0] / S[N.S_V]
    if n > 1:
        S[N.S_DT] *= np.linspace(0.999, 1.0, n)  # (output steps that differ)
    b = N.Batch(ctx, n)
    b.upload(S, np.zeros(n, np.int32))
    b.set_rows(5, np.full(n, 1, np.int64))
    b.run(N.make_desc(N.MODE_GC, rapt.params, rows * v_r * S[N.S_Y0, 0] / 1e8))
    assert kernel in rt.fake_last_kernel.value.decode(), rt.fake_last_kernel.value
    if n <= 8192:
        for _ in b.epochs(N.make_desc(N.MODE_GC, rapt.params, 1e6), rows, 1):
            pass
        assert kernel in rt.fake_epoch_kernel.value.decode()


_Q, _O, _MIX = "k_trace_gcnILi%dELi4E", "k_trace_gcnILi%dELi8E", "k_trace_gcmixILi%dE"
ONE = 65536  # lanes of one wave a SIMD


@pytest.mark.parametrize("name,model,n,costs,kernel,lanes", [
    # particles that cost the same: none wait for others to end
    ("double", 2, 8192, "equal", _O, ONE), ("double", 2, 8193, "equal", _Q, 4 * 8193 + 60),
    ("double", 2, 16384, "equal", _Q, ONE), ("dipole", 1, 32768, "equal", _Q, 2 * ONE),
    ("uniform", 8, 40000, "equal", _Q, 160000), ("double", 2, 65536, "equal", _MIX, 2 * ONE + 64),
    # of different cost: one wave a SIMD, refilled
    ("double", 2, 16384, "spread", _O, ONE), ("double", 2, 32768, "spread", _Q, ONE),
    ("double", 2, 65536, "spread", _MIX, ONE), ("grid", 9, 16384, "equal", _O, ONE),
    # fields that the order says nothing of, or with short steps
    ("sheet", 7, 32768, "equal", _Q, ONE), ("sheet", 7, 40000, "spread", _Q, 160000),
    ("sheet", 7, 131072, "spread", _Q, 8 * ONE),
    ("bz", 3, 8192, "equal", _Q, 32768), ("bz", 3, 1, "equal", _Q, 64)])
def test_default_guiding_centre_layout(fake, name, model, n, costs, kernel, lanes):
    _run(fake, "case_layout", name, n, costs, kernel % model, lanes)


@pytest.mark.parametrize("rows,n,v_r,kernel", [
    (1, 16, 0.4, _O), (1, 4096, 0.4, _Q), (8, 4096, 0.4, _O), (1, 8192, 0.4, _Q),
    (32, 8192, 0.4, _O), (4, 12000, 0.4, _Q), (16, 12000, 0.4, _O)])
def test_short_guiding_centre_runs(fake, rows, n, v_r, kernel):
    """Octets where the steps make up for the launch of twice the waves."""
    _run(fake, "case_short", rows, n, v_r, kernel % 2)


def case_brief(rt, n, kernel, lanes):
    """Particles alike, a run of few steps: one wave a SIMD, in rounds."""
    ctx = _ctx(_field("double"))
    S = np.zeros((N.NSLOT, n))
    S[N.S_Y0] = 5 * rapt.Re
    S[N.S_V] = 1e8
    S[N.S_DT] = 0.1
    b = N.Batch(ctx, n)
    b.upload(S, np.zeros(n, np.int32))
    b.set_rows(5, np.full(n, 1, np.int64))
    b.run(N.make_desc(N.MODE_GC, rapt.params, 0.3))
    assert kernel in rt.fake_last_kernel.value.decode()
    assert rt.fake_last_grid.value * rt.fake_last_block.value == lanes


@pytest.mark.parametrize("n,kernel,lanes", [(16385, _Q, ONE), (32768, _Q, ONE),
                                            (65536, _MIX, ONE)])
def test_brief_runs_of_particles_alike(fake, n, kernel, lanes):
    _run(fake, "case_brief", n, kernel % 2, lanes)


def test_epochs_of_particles_that_cost_the_same(fake):
    """Output steps of a bounce period's fraction: an epoch's particles cost the
    same, so all are resident; equal output steps: as they differ in r / v."""
    _run(fake, "case_epochs")


def case_epochs(rt):
    n = 16384
    ctx = _ctx(_field("double"))
    S = np.zeros((N.NSLOT, n))
    S[N.S_Y0] = 5 * rapt.Re
    S[N.S_V] = 1e8 * ((np.arange(n) + 1.0) / n) ** 2
    for dt, kernel in ((0.4 * S[N.S_Y0] / S[N.S_V], _Q % 2), (np.ones(n), _O % 2)):
        S[N.S_DT] = dt
        b = N.Batch(ctx, n)
        b.upload(S, np.zeros(n, np.int32))
        b.set_rows(5, np.full(n, 1, np.int64))
        for _ in b.epochs(N.make_desc(N.MODE_GC, rapt.params, 1e9), 32, 1):
            pass
        assert kernel in rt.fake_epoch_kernel.value.decode()


# ---- full orbits and adaptive runs ---------------------------------------------------


def case_orbits(rt, name, mode, n, rows, kernel, waves):
    ctx = _ctx(_field(name))
    S = np.zeros((N.NSLOT, n))
    S[N.S_Y0] = 5 * rapt.Re
    b = N.Batch(ctx, n)
    b.upload(S, np.zeros(n, np.int32))
    b.set_rows(N.ROW_WIDTH[mode], np.full(n, rows + 11, np.int64))
    desc = N.make_desc(mode, dict(rapt.params, GCtimestep=0.1), 1.0)
    b.run(desc)
    assert kernel in rt.fake_last_kernel.value.decode(), rt.fake_last_kernel.value
    assert rt.fake_last_grid.value * rt.fake_last_block.value == 64 * waves
    if mode == N.MODE_ADAPTIVE:
        for _ in b.epochs(desc, rows, 1):
            pass
        assert kernel in rt.fake_epoch_kernel.value.decode()
        assert rt.fake_epoch_lanes.value == 64 * waves


_P, _A = N.MODE_PARTICLE, N.MODE_ADAPTIVE
_DIP, _GRID = "ILi1ELi2ELi0ELb1E", "ILi9ELi2ELi0ELb0E"


@pytest.mark.parametrize("name,mode,n,rows,kernel,waves", [
    # the static kernel where it is the faster one
    ("dipole", _P, 1024, 9, "ILi1ELi0ELi0ELb1E", 16),
    ("grid", _P, 1024, 9, "ILi9ELi0ELi0ELb0E", 16), ("user", _P, 64, 9, "ILi10ELi0ELi0ELb0E", 1),
    # a wave each, one wave a CU, 64 a wave, one wave a SIMD
    ("dipole", _A, 1, 1, _DIP, 1), ("dipole", _A, 256, 1, _DIP, 256),
    ("dipole", _A, 1024, 3, _DIP, 1024), ("dipole", _A, 1024, 2, _DIP, 256),
    ("dipole", _A, 1025, 99, _DIP, 129), ("dipole", _A, 4096, 99, _DIP, 256),
    ("dipole", _A, 4097, 99, _DIP, 65), ("dipole", _A, 16383, 99, _DIP, 256),
    ("dipole", _A, 16384, 8, _DIP, 1024), ("dipole", _A, 16384, 7, _DIP, 256),
    ("grid", _A, 1, 99, _GRID, 1), ("grid", _A, 1024, 99, _GRID, 256),
    ("grid", _A, 4096, 99, _GRID, 256), ("grid", _A, 16384, 99, _GRID, 256)])
def test_orbit_kernels_and_spread(fake, name, mode, n, rows, kernel, waves):
    _run(fake, "case_orbits", name, mode, n, rows, kernel, waves)


# ---- kept scratch --------------------------------------------------------------------


def _keep_scratch(rt, ctx):
    """A call that leaves the context with scratch; what is free beside it."""
    f = _field("dipole")
    n = 65536
    tpos = np.tile([0.0, 5 * rapt.Re, 0.0, 0.0], (n, 1))
    ctx.halfbounce(f.descriptor(), tpos, np.full(n, 1e-5), 50)
    assert rt.fake_used.value > 2 * GIB


def case_memory(rt, call):
    """Every allocation that the call makes beside the kept scratch: with that
    much free and less, where the scratch has to give."""
    dip = _field("dipole")
    ctx = _ctx(dip)
    tp = np.array([[0.0, 5 * rapt.Re, 0.0, 0.0]])
    net = None
    if call in ("train", "forward", "targets"):
        from rapt_amd import surrogate as SG
        net = SG.Surrogate(dip, members=2)
    b = N.Batch(ctx, 1000) if call in ("epochs", "set_rows") else None
    if call == "epochs":
        b.upload(np.ones((N.NSLOT, 1000)), np.zeros(1000, np.int32))
        b.set_rows(7, np.ones(1000, np.int64))

    def run():
        if call == "train":
            z = np.zeros((4096, 3), np.float32)
            net.train_steps(z, z, np.zeros(4096, np.int64), 4096, 1e-3, 1e-3)
        elif call == "forward":
            net.forward(np.zeros((4096, 3), np.float32))
        elif call == "targets":
            net.targets(np.ones((4096, 3)), np.ones((4096, 3)))
        elif call == "surrogate":
            from rapt_amd import surrogate as SG
            SG.Surrogate(dip, members=2).close()
        elif call == "equatorial":
            ctx.bounce_center_equatorial(dip.descriptor(), np.tile(tp, (999, 1)), 1.0, 1.0, 0.0,
                                         3, 1e-6, 1e-6)
        elif call == "epochs":
            for _ in b.epochs(N.make_desc(N.MODE_PARTICLE, rapt.params, 1.0), 4, 1):
                pass
        elif call == "rhs":
            ctx.rhs_eval(dip.descriptor(), N.MODE_GC, np.ones((999, 5)), np.ones((999, 4)))
        elif call == "program":
            ctx.set_field(_field("user").descriptor())
        elif call == "grid":
            ctx.set_field(_Grid(["0"]).descriptor())
            assert b"k_grid_cells" in rt.fake_last_kernel.value  # (the faster layout)
        elif call == "batch":
            N.Batch(ctx, 1000).close()
        else:
            b.set_rows(7, np.full(1000, 10, np.int64))

    for room in (0, 64, 4096, 100000, 1 << 20, 3 << 20):
        ctx.set_field(dip.descriptor())
        rt.fake_budget.value = 1 << 40
        _keep_scratch(rt, ctx)
        rt.fake_budget.value = rt.fake_used.value + room
        run()


@pytest.mark.parametrize("call", ["train", "forward", "targets", "surrogate", "equatorial",
                                  "epochs", "rhs", "program", "grid", "batch", "set_rows"])
def test_kept_scratch_is_given_back_to_calls(fake, call):
    _run(fake, "case_memory", call)


def case_release(rt):
    ctx = _ctx(_field("dipole"))
    before = rt.fake_used.value
    _keep_scratch(rt, ctx)
    ctx.release_scratch()
    assert rt.fake_used.value == before
    ctx.release_scratch()
    _keep_scratch(rt, ctx)


def test_kept_scratch_is_given_back_on_request(fake):
    _run(fake, "case_release")


# ---- calls that fail half way ----------------------------------------------------------


def case_failed_copy(rt, call):
    """The k-th copy fails, for every k that the call reaches: it raises, and
    leaves nothing on the stream that could still use its arrays."""
    from rapt_amd import surrogate as SG
    dip = _field("dipole")
    ctx, d = _ctx(dip), dip.descriptor()
    n = 700000 if call in ("field_eval", "particle_gc") else 50  # (staged copies: 4 MB)
    tp = np.tile([0.0, 5 * rapt.Re, 0.0, 0.0], (n, 1))
    net = SG.Surrogate(dip, members=2) if call in ("train", "infer", "values") else None
    q = np.ones((1 << 18 if call == "values" else 50, 3), np.float32)
    fn = {"halfbounce": lambda: ctx.halfbounce(d, tp, 1e-5, 50),
          "labels": lambda: ctx.bounce_labels(d, np.ones((n, 3)), 1.0, 1.0, 1e3, 50),
          "centres": lambda: ctx.bounce_center_advance(d, tp, 1e-5, 1.0, 1.0, 0.0, 2, 1e-6, 1e-6,
                                                       1e3, 50),
          "field_eval": lambda: ctx.field_eval(d, "B", tp),
          "particle_gc": lambda: ctx.particle_gc(d, np.ones((n, 7)), 1.0, 1.0),
          "infer": lambda: net.infer(q, raw=True), "values": lambda: net.infer(q, raw=True),
          "train": lambda: net.train_steps(q[:50], q[:50], np.zeros(64, np.int64), 64, 1e-3, 1e-3,
                                           want_grad=True)}[call]
    for k in range(100):
        rt.fake_fail_copy.value = k
        try:
            fn()
        except RuntimeError:
            assert rt.fake_pending.value == 0, k
            rt._lib.hipGetLastError()
        else:
            break
    assert 1 < k < 99


@pytest.mark.parametrize("call", ["halfbounce", "labels", "centres", "field_eval", "particle_gc",
                                  "infer", "values", "train"])
def test_failed_calls_leave_nothing_queued(fake, call):
    _run(fake, "case_failed_copy", call)


# ---- large results ---------------------------------------------------------------------


def case_destination(rt, known):
    n = 700000
    dip = _field("dipole")
    ctx = _ctx(dip)
    rt.fake_pinned_lookup.value = known
    out = ctx.field_eval(dip.descriptor(), "magB", np.ones((n, 4)))
    assert out.nbytes > 4 << 20
    assert rt.fake_largest_copy.value == (out.nbytes if known else 1 << 20)
    assert rt._lib.hipGetLastError() == 0  # (the runtime's "not mine" is no error of the call)


@pytest.mark.parametrize("known", [0, 1])
def test_large_results_to_the_runtimes_own_memory_are_one_copy(fake, known):
    _run(fake, "case_destination", known)


if __name__ == "__main__":
    _lib = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
    globals()[sys.argv[2]](_Var(_lib), *[_arg(a) for a in sys.argv[3:]])
