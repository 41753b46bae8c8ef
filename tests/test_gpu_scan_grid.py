"""A scan over more rows than one dimension of a grid has threads for (2^30 of
them at 64 rows a block of 256), against the definition: a row of one element
is its own running sum."""
import numpy as np
import pytest
import torch

from pdl_amd import core as C

pytestmark = pytest.mark.gpu


class Seen:
    """an ndarray's memory as torch takes it in"""
    def __init__(self, x, typestr):
        self.x = x
        self.__cuda_array_interface__ = {"shape": tuple(x.dims[::-1]), "typestr": typestr, "data": (x._buf.ptr, False),
                                         "version": 2}


@pytest.mark.parametrize("rows", [(1 << 30) + 65])
def test_scan_of_very_many_rows(rows):
    C.init(0)
    host = np.random.default_rng(3).integers(0, 256, (rows, 1), dtype=np.uint8)
    x = C.ndarray.from_numpy(host, C.L.B)
    y = x.cumusumover()
    assert y.dims == [1, rows] and y.dtype == C.L.L
    C.synchronize()
    a, b = torch.as_tensor(Seen(x, "|u1"), device="cuda"), torch.as_tensor(Seen(y, "<i4"), device="cuda")
    for lo in range(0, rows, 1 << 28):   # piecewise: no large copy
        assert torch.equal(a[lo:lo + (1 << 28)].to(torch.int32), b[lo:lo + (1 << 28)]), lo
