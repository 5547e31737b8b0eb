"""A solver with sequential dot products holds no second array of directions:
only the fused vector update of tree-ordered dots uses one (levels 3 and 6-8).
Its device memory is a solver's without the fused update, one array of
doubles over the skewed layout less than with it."""
import ctypes

import pytest

import oracle_lib as ol
from gpu_util import make_product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [3, 7])
def test_no_second_direction_array(level, monkeypatch):
    import ifl_fluids as F

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        # of the runtime that the library is linked to
        assert F.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    sc = ol.REF_SCENES[level]
    w, h = 2000, 1900
    make_product(level, 16, 16, sc["params"], []).close()  # the library's own one-time memory

    def held(order, fused):
        monkeypatch.setenv("IFL_NO_FUSED_UPDATE", "0" if fused else "1")
        before = free_bytes()
        s = make_product(level, w, h, sc["params"], [], dot_order=order)
        n = before - free_bytes()
        s.close()
        return n

    array = 8 * 64 * ((h + 63) // 64) * ((w + 63 + 15) // 16 * 16)
    tree, plain, seq = held(F.DOT_TREE, True), held(F.DOT_TREE, False), held(F.DOT_SEQUENTIAL, True)
    print(f"level {level} {w}x{h}: tree {tree}, not fused {plain}, sequential {seq}, one array {array}", flush=True)
    assert tree - plain >= array // 2
    assert abs(seq - plain) < array // 2
