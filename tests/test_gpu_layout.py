"""The FP64 operand tiles and their row-swapped copies, through the C-ABI.

Bar: a system without the row-swapped copies (a server whose budget does not
hold them admits it without) gives the same bits as one with them: the
kernels read the same values from the straight arrays.
"""
import pytest

from atrip_amd import serve

pytestmark = pytest.mark.gpu


def _pad(n, m):
    return (n + m - 1) // m * m


def _swap_bytes(no, nv):
    """Bytes of the row-swapped copies of T3 and H3 (rows padded to 16)."""
    return 8 * nv * _pad(no * no, 16) * (_pad(nv, 16) + _pad(no, 16))


# both served paths (No below and from 16), No^2 on and off a 16-row tile,
# Nv on and off an 8-deep tile
@pytest.mark.parametrize("no,nv,seed", [(5, 23, 1), (8, 40, 2), (16, 24, 3),
                                        (19, 17, 4)])
def test_without_swapped_copies(hip_ctx, no, nv, seed):
    s = hip_ctx.upload_synthetic(no, nv, seed)
    full = hip_ctx.sys_info(s)["bytes"]
    hip_ctx.release(s)
    least = full - _swap_bytes(no, nv)
    energy = {}
    for budget in (full, least):
        print("layout", no, nv, budget, flush=True)
        with serve.Server(hip_ctx, hbm_budget_gb=(budget + 0.5) / 1e9) as srv:
            rid = srv.submit_synthetic(no, nv, seed)
            energy[budget] = srv.drain([rid])[rid]["energy"]
            assert srv.stats()["peak_bytes"] == budget
    assert energy[full] == energy[least] != 0.0
    with serve.Server(hip_ctx, hbm_budget_gb=(least - 0.5) / 1e9) as srv:
        rid = srv.submit_synthetic(no, nv, seed)
        srv.step()
        assert srv.result(rid, raise_failed=False)["state"] == serve.FAILED
