"""Matrices between the caller's arrays and the device: every element, and
nothing else, where the pieces and the slots of the copies change."""
import numpy as np
import pytest

from mopac_gpu_amd import lib as L

pytestmark = pytest.mark.gpu


# one value; columns without gaps; ragged ones in one and in several pieces;
# 13 and 27 MB (slots at their largest); one and two columns of 64 KB to 4 MB,
# a slot's smallest and largest size between them; columns longer than that
@pytest.mark.parametrize("m,n,pad", [(1, 1, 0), (1, 40, 3), (7, 301, 2), (300, 77, 0), (123, 701, 5),
                                     (1237, 1301, 5), (1901, 1777, 1), (8193, 2, 3),
                                     (9000, 2, 3), (12000, 2, 3), (20000, 1, 3), (24000, 1, 3), (40000, 2, 1),
                                     (524288, 2, 3), (600001, 2, 3)])
def test_pitched_copies_touch_only_their_rows(gpu_ctx, m, n, pad):
    rng = np.random.default_rng(m + n)
    lib, ld = L.load(), m + pad
    lib.mhip_destroy_resources()  # slots only grow: these are this matrix's own
    a = np.asfortranarray(rng.integers(-8, 9, (ld, 1)).astype(float))
    b = np.asfortranarray(rng.integers(-8, 9, (1, n)).astype(float))
    c = np.asfortranarray(rng.integers(-8, 9, (ld, n)).astype(float))
    want = c.copy(order="F")
    want[:m] = 2.0 * a[:m] @ b + 3.0 * c[:m]  # whole numbers: exact
    lib.mhip_call_gemm(b"N", b"N", m, n, 1, 2.0, L.ptr(a), ld, L.ptr(b), 1, 3.0, L.ptr(c), ld)
    assert np.array_equal(c, want)
