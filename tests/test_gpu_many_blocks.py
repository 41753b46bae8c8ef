"""Work of 2^24 blocks and more, where one dimension of a grid would wrap:
batches of small products on the matrix cores (8x8x8), the SIMT kernel (4x4x4
and whole-number types) and the split-FP16 kernel (33x33x33, operands and
outputs shared so that they fit), and an elementwise op over 2^24 rows of a
broadcast.  Small whole numbers: every result is exact."""
import pytest
import torch

from pdl_amd import core as C

pytestmark = pytest.mark.gpu

TORCH = {C.L.B: torch.uint8, C.L.L: torch.int32, C.L.F: torch.float32, C.L.D: torch.float64}
TYPESTR = {C.L.B: "|u1", C.L.L: "<i4", C.L.F: "<f4", C.L.D: "<f8"}
STEP = 1 << 20


class Seen:
    def __init__(self, x):
        self.x = x
        self.__cuda_array_interface__ = {"shape": tuple(x.dims[::-1]), "typestr": TYPESTR[x.dtype],
                                         "data": (x._buf.ptr, False), "version": 2}


def tensor(x):
    return torch.as_tensor(Seen(x), device="cuda")


@pytest.fixture(autouse=True)
def device():
    C.init(0)
    yield
    torch.cuda.empty_cache()


def filled(t, dims, lo, hi, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = C.ndarray.new_dense(t, dims)
    for part in tensor(x).split(STEP):
        part.copy_(torch.randint(lo, hi, part.shape, generator=g, device="cuda", dtype=torch.int32))
    torch.cuda.synchronize()
    return x


@pytest.mark.parametrize("t,n", [(C.L.F, 8), (C.L.D, 8), (C.L.F, 4), (C.L.L, 4)],
                         ids=["float 8", "double 8", "float 4", "long 4"])
def test_batches_of_small_products(t, n):
    count = (1 << 24) + 3
    a, b = filled(t, [n, n, count], -9, 10, 1), filled(t, [n, n, 1], -9, 10, 2)
    c = C.matmult(a, b)
    assert c.dims == [n, n, count]
    C.synchronize()
    tb = tensor(b)[0].double()
    for pa, pc in zip(tensor(a).split(STEP), tensor(c).split(STEP)):
        want = (pa.double().reshape(-1, n) @ tb).reshape(pa.shape)
        assert torch.equal(pc.double(), want)


def test_batch_of_split16_products():
    count, n = (1 << 24) + 3, 33
    a, b = filled(C.L.F, [n, n], -9, 10, 3), filled(C.L.F, [n, n], -9, 10, 4)
    c = C.ndarray.new_dense(C.L.F, [n, n, count])
    tensor(c).fill_(float("nan"))
    torch.cuda.synchronize()
    C._run("matmult", [a.dummy(2, count), b.dummy(2, count), c])
    C.synchronize()
    want = (tensor(a).double() @ tensor(b).double()).float()
    for part in tensor(c).split(STEP):
        assert bool((part == want).all())


def test_one_product_of_many_tiles():
    h, w = (1 << 18) + 5, (1 << 18) + 3     # 64 GiB of bytes
    a, b = filled(C.L.B, [1, h], 0, 256, 7), filled(C.L.B, [w, 1], 0, 256, 8)
    c = C.matmult(a, b)
    assert c.dims == [w, h]
    C.synchronize()
    tb = tensor(b)
    for pa, pc in zip(tensor(a).split(1 << 12), tensor(c).split(1 << 12)):
        assert torch.equal(pc, pa * tb)


def test_rows_of_a_broadcast():
    rows = (1 << 24) + 5
    a, b = filled(C.L.B, [128, rows], 0, 256, 5), filled(C.L.B, [128], 0, 256, 6)
    c = a + b
    assert c.dims == [128, rows]
    C.synchronize()
    tb = tensor(b)
    for pa, pc in zip(tensor(a).split(STEP), tensor(c).split(STEP)):
        assert torch.equal(pc, pa + tb)
