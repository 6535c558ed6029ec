"""Which kernel a size takes, at the sizes where both sides were measured
(the rules and the figures stand beside them in the sources)."""

import ctypes

import pytest

import hyperdeal_amd as H


def _lib():
    return ctypes.CDLL(H.library_path())


@pytest.mark.parametrize("k,nx,strips", [
    (3, [16, 2], 1), (3, [2, 2], 1), (3, [32, 32], 1), (3, [4, 256], 1),
    (3, [64, 2], 1), (3, [64, 16], 1), (3, [65, 2], 0), (3, [100, 2], 0),
    (3, [128, 4], 0), (3, [128, 5], 1), (3, [100, 10], 1), (3, [5, 1], 0),
    (2, [24, 24], 1), (2, [32, 32], 1), (2, [56, 10], 1), (2, [4, 200], 1),
    (2, [22, 23], 0), (2, [16, 16], 0), (2, [57, 9], 0), (2, [200, 4], 0),
    (1, [2, 2], 0), (1, [32, 32], 0), (1, [4, 250], 0),
])
def test_strips_only_where_they_are_faster(k, nx, strips):
    assert _lib().hd_probe_vp_strips(k, *nx) == strips


@pytest.mark.parametrize("dims,k,x,v,prec,stage,curved", [
    ((1, 1), 1, 220, 220, H.FP64, 0, 1), ((1, 1), 1, 270, 270, H.FP64, 0, 0),
    ((1, 1), 1, 220, 220, H.FP32, 1, 1), ((1, 1), 1, 300, 300, H.FP32, 1, 0),
    ((1, 1), 2, 1500, 1500, H.FP64, 0, 1), ((1, 1), 2, 600, 600, H.FP64, 1, 1),
    ((1, 1), 2, 1100, 1100, H.FP64, 1, 0),
    ((1, 1), 2, 1100, 1100, H.FP32, 0, 0), ((1, 1), 3, 1100, 1100, H.FP32, 0, 1),
    ((1, 1), 2, 270, 270, H.FP32, 1, 1), ((1, 1), 2, 330, 330, H.FP32, 1, 0),
    ((1, 1), 3, 1100, 1100, H.FP64, 1, 1), ((1, 1), 4, 1100, 1100, H.FP64, 1, 0),
    ((1, 1), 4, 500, 500, H.FP32, 1, 1), ((1, 1), 4, 800, 800, H.FP32, 1, 0),
    ((2, 1), 1, 1600, 40, H.FP32, 1, 1), ((2, 1), 1, 2500, 50, H.FP32, 1, 0),
    ((1, 2), 1, 100, 10000, H.FP32, 1, 1), ((1, 2), 1, 140, 19600, H.FP32, 1, 0),
    ((2, 1), 1, 19600, 140, H.FP64, 1, 1),
    ((2, 2), 1, 1024, 1024, H.FP32, 1, 1), ((2, 2), 3, 576, 576, H.FP64, 0, 1),
    # the tables of a space stay within 64 MB
    ((2, 1), 4, 5461, 2, H.FP64, 0, 1), ((2, 1), 4, 5462, 2, H.FP64, 0, 0),
    ((1, 2), 4, 2, 5462, H.FP64, 0, 0), ((1, 1), 2, 70000, 2, H.FP64, 0, 0),
    ((3, 1), 2, 12, 4, H.FP64, 0, 0), ((1, 1), 5, 4, 4, H.FP64, 0, 0),
])
def test_factorised_form_only_where_it_is_faster(dims, k, x, v, prec, stage,
                                                 curved):
    f = _lib().hd_probe_curved
    assert f(*dims, k, ctypes.c_longlong(x), ctypes.c_longlong(v), prec,
             stage) == curved
