"""Calls that stay refused, without a GPU: sizes that name no work are errors,
not silent successes."""
import ctypes as C

import numpy as np
import pytest

from prismplan_amd import _ppl


@pytest.mark.parametrize("extent", [(-0.1, 0.1, 0.1), (0.1, -0.05, 0.1), (0.1, 0.1, -0.1), (-0.1, -0.1, 0.1),
                                    (float("nan"), 0.1, 0.1)])
def test_esdf_of_an_empty_grid_is_refused(extent):
    """A negative (or undefined) extent gives a grid without nodes along it."""
    view = _ppl.SceneView()
    prm = np.array([*extent, 0.05], np.float32)
    pose = np.array([0, 0, 0, 1, 0, 0, 0, 0], np.float32)
    out = np.zeros(64, np.float32)
    f = lambda a: a.ctypes.data_as(C.POINTER(C.c_float))
    st = _ppl.lib().ppl_esdf_from_obbs(C.byref(view), f(prm), f(pose), C.c_void_p(out.ctypes.data), None)
    assert st != _ppl.PPL_OK
    assert not out.any()
