"""Results large enough for the staged copies (rapt_copy.hip), a megabyte a
slot of a ring of eight: one slot short of the threshold, at it, a last slot
that is not full, the ring more than once round; and from two threads at once."""
import ctypes as C
import threading

import numpy as np
import pytest

from rapt_amd import _native as N
from rapt_amd import constants as K
from rapt_amd import fields as F

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _points(n):
    rng = np.random.default_rng(n)
    return np.c_[np.zeros(n), rng.uniform(2, 8, (n, 3)) * K.Re]


@pytest.mark.parametrize("nbytes", [4 * MB - 8, 4 * MB, 4 * MB + 8, 8 * MB, 21 * MB + 1000])
def test_large_results_equal_small_ones(nbytes):
    f = F.EarthDipole().descriptor()
    ctx = N.context()
    tp = _points(nbytes // 8)
    got = ctx.field_eval(f, "magB", tp)
    step = 100000
    ref = np.concatenate([ctx.field_eval(f, "magB", tp[i:i + step])
                          for i in range(0, len(tp), step)])
    np.testing.assert_array_equal(got, ref)


def test_large_results_on_two_threads():
    f = F.EarthDipole().descriptor()
    ctx = N.context()
    tp = [_points(700001), _points(900003)]
    ref = [ctx.field_eval(f, "B", t) for t in tp]
    got = [None, None]

    def work(i):
        for _ in range(3):
            got[i] = ctx.field_eval(f, "B", tp[i])

    th = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for g, r in zip(got, ref):
        np.testing.assert_array_equal(g, r)


def test_inference_values_on_either_side_of_the_device_widening():
    """From 262,144 queries on the device widens the values and applies the
    drift's sign: the bits of the float path."""
    from rapt_amd import surrogate as S
    rng = np.random.default_rng(4)
    n = 1 << 18
    q = np.c_[rng.uniform(2, 8, n), rng.uniform(10, 89, n), rng.uniform(4, 7, n)]
    for charge in (K.e, -K.e):
        s = S.Surrogate(F.EarthDipole(), charge=charge, members=2, seed=1)
        v, flag, raw, _ = s.infer(q, raw=True)
        a, b = s.infer(q[:-1], raw=True), s.infer(q[-1:], raw=True)
        np.testing.assert_array_equal(v, np.r_[a[0], b[0]])
        np.testing.assert_array_equal(flag, np.r_[a[1], b[1]])
        np.testing.assert_array_equal(raw, np.concatenate([a[2], b[2]], axis=1))


def test_large_results_to_pinned_memory():
    """A destination that the runtime has pinned takes the copy directly."""
    f = F.EarthDipole().descriptor()
    ctx = N.context()
    tp = np.ascontiguousarray(_points(900003))
    ref = ctx.field_eval(f, "B", tp)
    hip = C.CDLL("libamdhip64.so")
    p = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(p), C.c_size_t(ref.nbytes), 0) == 0
    try:
        ptr = C.cast(p, C.POINTER(C.c_double))
        ctx.check(N.lib().rapt_field_eval(ctx.h, N.EVAL["B"], len(tp), N._dp(tp), ptr),
                  "rapt_field_eval")
        np.testing.assert_array_equal(np.ctypeslib.as_array(ptr, ref.shape), ref)
    finally:
        hip.hipHostFree(p)
