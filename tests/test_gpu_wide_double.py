"""Double products of 17 to 48 k and 8e7 outputs or more (blocks of 128x128)
and their neighbours on the tiles: ragged sides, operands and output along
either index, whole numbers exactly, infinities and NaN as in the plain loop."""
import numpy as np
import pytest
import torch

from pdl_amd import core as C
from test_gpu_dgemm import LAYOUTS, whole

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def device():
    C.init(0)
    C.set_matmult_precision("split16")
    yield
    torch.cuda.empty_cache()


def tensor(x):
    class Seen:
        __cuda_array_interface__ = {"shape": tuple(x.dims[::-1]), "typestr": "<f8", "data": (x._buf.ptr, False),
                                    "version": 2}
    return torch.as_tensor(Seen(), device="cuda")


@pytest.mark.parametrize("h,t,w", [(9001, 17, 9003), (9001, 16, 9003), (400, 31, 200010), (128, 48, 625001),
                                   (127, 48, 640001), (9000, 49, 8900), (8900, 33, 8900)])
@pytest.mark.parametrize("la,lb", [("dense", "dense"), ("transposed", "dense"), ("dense", "transposed")])
def test_whole_numbers_exact(h, t, w, la, lb):
    rng = np.random.default_rng(h + t)
    a, b = whole(rng, h, t), whole(rng, t, w)
    c = C.matmult(LAYOUTS[la](a), LAYOUTS[lb](b))
    C.synchronize()
    d, tb = tensor(c), torch.from_numpy(b).cuda()
    for lo in range(0, h, 2048):
        assert torch.equal(d[lo:lo + 2048], torch.from_numpy(a[lo:lo + 2048]).cuda() @ tb), lo


def test_output_through_a_view_and_nonfinite_entries():
    h, t, w = 9001, 20, 9003
    rng = np.random.default_rng(2)
    a, b = whole(rng, h, t), whole(rng, t, w)
    out = C.ndarray.new_dense(C.L.D, [h, w])
    C.matmult(LAYOUTS["dense"](a), LAYOUTS["dense"](b), out.xchg(0, 1))
    C.synchronize()
    assert torch.equal(tensor(out).T, torch.from_numpy(a).cuda() @ torch.from_numpy(b).cuda())
    del out
    a[3, 19], a[8000, 0], b[7, 5], b[2, 9002] = np.inf, np.nan, -np.inf, np.nan
    c = C.matmult(LAYOUTS["dense"](a), LAYOUTS["dense"](b))
    C.synchronize()
    rows = [0, 3, 8000, 9000]
    with np.errstate(invalid="ignore"):
        want = (a[rows][:, :, None] * b[None]).sum(axis=1)
    np.testing.assert_array_equal(tensor(c)[rows].cpu().numpy(), want)
