"""Scratch that the full-orbit kernels spill to, at most what they spilled
before their divisions were shortened: beyond it they are slower."""
import pytest

from test_kernel_resources import sizes  # noqa: F401  (fixture)


@pytest.mark.parametrize("model,precision,limit", [(1, 0, 20), (5, 0, 140), (7, 0, 60), (9, 0, 0),
                                                   (1, 1, 12), (5, 1, 140), (7, 1, 52)])
def test_general_full_orbit_kernels(sizes, model, precision, limit):  # noqa: F811
    name = "_ZN4rapt7k_traceILi%dELi0ELi%dELb0EEEvNS_5KArgsE" % (model, precision)
    assert sizes[name] <= limit
