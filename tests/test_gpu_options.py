"""The "batch" option (windows per launch): 0 is its default and automatic
value, so a program that reads it and writes it back changes nothing.

Bar: the number of launches of a run (timing events of the energy kernel) is
the automatic one after writing back what get_option returned and after 4 has
been set and taken back; 4 windows per launch take as many launches as windows
/ 4.
"""
import pytest

from atrip_amd import hip

pytestmark = pytest.mark.gpu


def test_batch_zero_is_automatic():
    with hip.Context(0) as ctx:
        s = ctx.upload_synthetic(6, 33, 1)
        ctx.set_option("window", 8)
        ctx.set_option("timing", 1)

        def launches():
            ctx.reset_stats()
            ctx.run(s)
            return ctx.kernel_stats("energy").launches

        assert launches() == 1  # 34 windows of edge 8: 215 MB of class buffers
        ctx.set_option("batch", ctx.get_option("batch"))
        assert launches() == 1
        ctx.set_option("batch", 4)
        assert ctx.get_option("batch") == 4
        assert launches() == 9
        ctx.set_option("batch", 0)
        assert launches() == 1
        for bad in (-1, 4097):
            with pytest.raises(hip.HipError, match="batch must be"):
                ctx.set_option("batch", bad)
