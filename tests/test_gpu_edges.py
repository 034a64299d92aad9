"""Edge tiles of the doubles kernels: only the occupied row and column
fragments of a tile and only the columns of valid tuples are computed.

Bar: per-tuple energies within 1e-12 (FP64) and 1e-5 (FP32 products) of the
largest, the tolerances of the parity tests, against the oracle, where No^2
and the valid columns end on, just before and just after a fragment (16 or 32
wide), half a tile and a whole tile, for every tile variant, over the whole
space and over ranges that cut an A-pair's columns at either end; the bits are
those of the automatic tile and window.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REL = {"fp64": 1e-12, "split_fp32": 1e-5, "bf16x3": 1e-5}
TILES = {"fp64": range(8), "split_fp32": range(10), "bf16x3": range(10)}


# No^2 = 16, 25, 64, 81, 121, 144, 324: one fragment and around whole ones;
# the window edge sets how many columns a pair holds (edge * No)
@pytest.mark.parametrize("no,nv,window", [(4, 11, 1), (5, 13, 7), (8, 12, 4),
                                          (9, 10, 3), (11, 9, 8), (12, 14, 5),
                                          (18, 10, 9)])
@pytest.mark.parametrize("precision", ["fp64", "split_fp32", "bf16x3"])
def test_edge_tiles(hip_ctx, oracle, no, nv, window, precision):
    seed = 900 + no
    t = oracle.synthetic(no, nv, seed)
    _, _, ref, _ = oracle.run(no, nv, t, per_tuple=True)
    n = oracle.n_tuples(nv)
    s = hip_ctx.upload(no, nv, t)
    try:
        base = hip_ctx.tuple_energies(s, 0, n, precision)
        assert np.max(np.abs(base - ref)) <= REL[precision] * np.max(np.abs(ref))
        hip_ctx.set_option("window", window)
        for tile in TILES[precision]:
            print("edge tiles", no, nv, window, precision, tile, flush=True)
            hip_ctx.set_option("tile", tile)
            for first, count in ((0, n), (1, 1), (n // 3, n // 2), (n - 5, 5)):
                e = hip_ctx.tuple_energies(s, first, count, precision)
                assert np.array_equal(e, base[first:first + count]), (tile, first)
    finally:
        hip_ctx.set_option("tile", -1)
        hip_ctx.set_option("window", 0)
        hip_ctx.release(s)


# The epilogue that does a whole tuple at once (No <= 18, with (cT) or FP32
# buffers <= 20): one pair of elements, odd and even No around the limits of a
# wave (8) and of four (14), and the last No and the first beyond.  W is the same
# bits as in the cube epilogue and the up to 1771 terms of a tuple are added in
# another order: within 1771 roundings of 1.1e-16 of the sum of their
# magnitudes, bounded here by 1e-12 of the largest tuple.
@pytest.mark.parametrize("no", [1, 2, 3, 7, 8, 9, 14, 15, 16, 18, 19, 20, 21])
@pytest.mark.parametrize("precision", ["fp64", "bf16x3"])
def test_small_epilogue(hip_ctx, no, precision):
    nv = 13
    n = nv * (nv + 1) * (nv + 2) // 6 - nv
    for with_j in (False, True):
        print("small epilogue", no, precision, with_j, flush=True)
        s = hip_ctx.upload_synthetic(no, nv, 700 + no, with_j=with_j)
        out = []
        try:
            for epi in (0, 1):
                hip_ctx.set_option("epilogue", epi)
                out.append(hip_ctx.tuple_energies(s, 0, n, precision, with_ct=True))
        finally:
            hip_ctx.set_option("epilogue", 0)
            hip_ctx.release(s)
        for x, y in zip(*out):
            assert np.max(np.abs(x - y)) <= 1e-12 * np.max(np.abs(y))


# The complex one (No <= 20, with (cT) <= 16), likewise; up to 1771 terms.
@pytest.mark.parametrize("no", [1, 2, 3, 7, 8, 9, 15, 16, 17, 20, 21])
def test_small_epilogue_complex(hip_ctx, no):
    nv = 11
    n = nv * (nv + 1) * (nv + 2) // 6 - nv
    for with_j in (False, True):
        print("small complex epilogue", no, with_j, flush=True)
        s = hip_ctx.upload_synthetic_complex(no, nv, 800 + no, with_j=with_j)
        out = []
        try:
            for epi in (0, 1):
                hip_ctx.set_option("epilogue", epi)
                out.append(hip_ctx.tuple_energies(s, 0, n, with_ct=True))
        finally:
            hip_ctx.set_option("epilogue", 0)
            hip_ctx.release(s)
        for x, y in zip(*out):
            assert np.max(np.abs(x - y)) <= 1e-12 * np.max(np.abs(y))
