"""Parameters of a batch handle that were read can be set again without a change (host calls only)."""
import ctypes

import pytest


@pytest.mark.parametrize("grid", [0, 1, 2048])
def test_params_round_trip(grid):
    from neighbor_amd import _capi
    L = _capi.lib()
    h = ctypes.c_void_p()
    assert L.nb_batch_create(ctypes.byref(h)) == _capi.NB_OK
    try:
        assert L.nb_batch_set_params(h, 512, 32, _capi.NB_BATCH_WAVE, grid) == _capi.NB_OK
        for _ in range(2):
            b, k, g, v = ctypes.c_uint32(), ctypes.c_uint32(), ctypes.c_uint32(), ctypes.c_int()
            assert L.nb_batch_get_params(h, ctypes.byref(b), ctypes.byref(k), ctypes.byref(v), ctypes.byref(g)) == _capi.NB_OK
            assert (b.value, k.value, v.value, g.value) == (512, 32, _capi.NB_BATCH_WAVE, grid)
            assert L.nb_batch_set_params(h, b.value, k.value, v.value, g.value) == _capi.NB_OK
    finally:
        assert L.nb_batch_destroy(h) == _capi.NB_OK
