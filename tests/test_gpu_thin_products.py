"""Float products of any size with a side below 64 or fewer than 32 k run on
the FP32 matrix cores like the small ones, in sums of a few k.  A long inner
dimension: partial sums of 32 k leave about sqrt(k / 64) rounding errors of
2^-25.5 each in an output, 3e-7 of its size at 12000 k at most; one chain of
all k leaves 1.7e-6; 2^-21 lies between.  Few k: a row's outputs have the same
bits whether few or many rows are multiplied."""
import pytest
import torch

from pdl_amd import core as C

pytestmark = pytest.mark.gpu


class Seen:
    def __init__(self, x):
        self.x = x
        self.__cuda_array_interface__ = {"shape": tuple(x.dims[::-1]), "typestr": "<f4", "data": (x._buf.ptr, False),
                                         "version": 2}


def tensor(x):
    return torch.as_tensor(Seen(x), device="cuda")


def normal(rows, cols, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = C.ndarray.new_dense(C.L.F, [cols, rows])
    tensor(x).normal_(generator=g)
    torch.cuda.synchronize()
    return x


@pytest.fixture(autouse=True)
def device():
    C.init(0)
    yield
    torch.cuda.empty_cache()


@pytest.mark.parametrize("h,t,w", [(32, 12000, 12000), (12000, 12000, 33), (8, 24000, 24000), (63, 9000, 8000)])
def test_long_inner_dimension(h, t, w):
    a, b = normal(h, t, 1), normal(t, w, 2)
    c = C.matmult(a, b)
    C.synchronize()
    truth = tensor(a).double() @ tensor(b).double()
    assert float((tensor(c).double() - truth).norm() / truth.norm()) <= 2.0 ** -21


@pytest.mark.parametrize("t", [9, 16, 31])
def test_few_k(t):
    h, w = 28000, 27000
    a, b = normal(h, t, 3), normal(t, w, 4)
    c = C.matmult(a, b)
    for lo in (0, h - 1000):
        part = C.matmult(a.slice(None, (lo, lo + 999, 1)), b)
        C.synchronize()
        assert torch.equal(tensor(c)[lo:lo + 1000], tensor(part)), lo
