"""Systems whose row-swapped operand copies were given back: an upload that no
device holds, in another context, takes them back before it fails.

Bar: the same bits, real and complex, with and without (cT), whole runs,
ranges and the batched form, before and after.
"""
import numpy as np
import pytest

from atrip_amd import hip

pytestmark = pytest.mark.gpu


def _pad(n, m):
    return (n + m - 1) // m * m


# No^2 on and off a 16-row tile, Nv on and off an 8-deep one
@pytest.mark.parametrize("no,nv", [(5, 19), (8, 24), (13, 21)])
@pytest.mark.parametrize("with_j", [False, True])
def test_same_bits_without_swapped_copies(no, nv, with_j):
    n = nv * (nv + 1) * (nv + 2) // 6 - nv
    h3 = 8 * nv * _pad(no * no, 16) * _pad(no, 16)
    t3 = 8 * nv * _pad(no * no, 16) * _pad(nv, 16)
    swaps = t3 + h3 * (2 if with_j else 1)
    # a complex system's swapped planes: real, imaginary and negated imaginary
    with hip.Context(0) as ctx, hip.Context(0) as other:
        real = ctx.upload_synthetic(no, nv, 40 + no, with_j=with_j)
        comp = ctx.upload_synthetic_complex(no, nv, 60 + no, with_j=with_j)

        def results():
            out = [np.array(ctx.run(s, first=f, count=c)) for s in (real, comp)
                   for f, c in ((0, None), (n // 3, n // 2))]
            for s in (real, comp):
                out += list(ctx.tuple_energies(s, 0, n, with_ct=True))
            return out + [ctx.batch_run([real])]

        print("swapped copies", no, nv, with_j, flush=True)
        before = results()
        size = [ctx.sys_info(s)["bytes"] for s in (real, comp)]
        with pytest.raises(hip.HipError, match="out of memory"):
            other.upload_synthetic(200, 3000, 1)
        assert [ctx.sys_info(s)["bytes"] for s in (real, comp)] == [
            size[0] - swaps, size[1] - 3 * swaps]
        print("without them", flush=True)
        for x, y in zip(before, results()):
            assert np.array_equal(x, y) and np.any(x != 0.0)
