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
    (3, [128, 5], 0), (3, [5, 1], 0),
    (2, [24, 24], 1), (2, [32, 32], 1), (2, [56, 10], 1), (2, [4, 200], 1),
    (2, [22, 23], 0), (2, [16, 16], 0), (2, [57, 9], 0), (2, [200, 4], 0),
    (1, [2, 2], 0), (1, [32, 32], 0), (1, [4, 250], 0),
])
def test_strips_only_where_they_are_faster(k, nx, strips):
    assert _lib().hd_probe_vp_strips(k, *nx) == strips
