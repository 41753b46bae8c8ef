"""Ragged integer scans whose long items are cut into pieces: lengths around
the pieces' and segments' ends, several long items, strided views, wrapping
sums and products, against numpy's wrapping cumulative ops, run twice and
replayed in a graph."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SEG = 4096
LENGTHS = [[3 * SEG], [SEG, SEG + 1], [40 * SEG + 7] + [5] * 50, [0, 9 * SEG - 1, 0, 9 * SEG, 9 * SEG + 1, 1, 300],
           [300 * SEG + 11, 100 * SEG, 17, 0, SEG - 1] + [2000] * 700, [1100 * SEG + 1]]


@pytest.mark.parametrize("lengths", LENGTHS, ids=lambda x: "n%d_max%d" % (len(x), max(x)))
@pytest.mark.parametrize("t,dtype,op,step", [("B", np.uint8, "cumusumover", 1), ("L", np.int32, "cumusumover", 2),
                                             ("LL", np.int64, "cumusumover", 1), ("LL", np.int64, "cumuprodover", 1)])
def test_ragged_scan_pieces(lengths, t, dtype, op, step):
    from pdl_amd import core as C
    C.init(0)
    rng = np.random.default_rng(len(lengths))
    info = np.iinfo(dtype)
    hosts, views = [], []
    for n in lengths:
        x = rng.integers(info.min, info.max, max(n, 1) * step, dtype=dtype, endpoint=True)
        if op == "cumuprodover":
            x |= 1   # (an even factor now and then would leave zeros)
        hosts.append(x[:n * step:step])
        views.append(C.ndarray.from_numpy(x, getattr(C.L, t))._view([n], [step], 0))
    f = np.cumsum if op == "cumusumover" else np.cumprod
    r = C.Ragged([[v] for v in views], [], op)
    for _ in range(2):
        r.run()
    graph = C.Graph(lambda: r.run())
    for _ in range(2):
        graph.launch()
        for x, o in zip(hosts, r.outputs):
            got = o.numpy()
            want = f(x.astype(got.dtype), dtype=got.dtype)   # in the op's own output type, which wraps
            assert np.array_equal(got, want), (len(x), np.argmax(got != want))


@pytest.mark.parametrize("lengths", [[1, 511, 512, 513, 1025, 0, 4097], [1 << 21] * 8 + [4096, 4097, 1], [60000] * 70],
                         ids=["512", "4096", "1024"])
def test_ragged_sum_segments(lengths):
    """sums over segments of 512 to 4096 elements, as the list's size has them"""
    from pdl_amd import core as C
    C.init(0)
    rng = np.random.default_rng(3)
    hosts = [rng.standard_normal(n).astype(np.float32) for n in lengths]
    r = C.Ragged([[C.ndarray.from_numpy(x, C.L.F)] for x in hosts], [], "sumover")
    r.run()
    for x, o in zip(hosts, r.outputs):
        x = x.astype(np.float64)
        assert abs(float(o.numpy()) - x.sum()) <= (len(x) + 1) * 2.0 ** -24 * np.abs(x).sum()
