"""What a call does when the device has little memory left, on the CPU: the
library runs on a stand-in for the HIP runtime (fake_hip.c) whose allocations
have a limit and whose kernels do nothing.

Bar: a call succeeds wherever the least that it needs fits.
"""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", out,
                    os.path.join(HERE, "fake_hip.c")], check=True)
    return out


def _run(fake, body):
    """Runs `body` in a process of its own, the stand-in loaded first."""
    code = ("import ctypes, sys\n"
            f"sys.path.insert(0, {os.path.dirname(HERE)!r})\n"
            f"fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)\n"
            "fake.fake_set_limit.argtypes = [ctypes.c_size_t]\n"
            "fake.fake_used.restype = ctypes.c_size_t\n"
            "from atrip_amd import hip\n"
            "GiB = 1 << 30\n") + body
    r = subprocess.run([sys.executable, "-c", code], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_smaller_launch_gives_back_what_the_larger_had(fake):
    # No=20, W cubes: 510 MB of class buffers and 170 MB of cubes for three
    # windows of 512 tuples, so 12 windows take 2.04 + 0.68 GB and the least
    # launch, four, 0.68 + 0.23.  With 2.14 GB only the larger one's class
    # buffers fit, and beside them the smaller one's cubes do not.
    _run(fake, """
ctx = hip.Context(0)
ctx.set_option("epilogue", 1)
ctx.set_option("window", 8)
s = ctx.upload_synthetic(20, 48, 1)
fake.fake_set_limit(fake.fake_used() + 2140 * 10**6)
ctx.run(s)
assert fake.fake_used() < 2140 * 10**6
""")


# `full`: bytes of a No=12, Nv=48 system, `swaps` of them (3.5 MB) its
# row-swapped copies; a run of it grows launch buffers of more than 1 GiB
SIZES = """
probe = hip.Context(0)
before = fake.fake_used()
p = probe.upload_synthetic(12, 48, 1)
full = fake.fake_used() - before
probe.run(p)
grown = fake.fake_used() - before - full
assert grown > GiB
probe.close()
assert fake.fake_used() == before
swaps = 8 * 48 * 144 * (48 + 16)
"""


def test_upload_takes_back_what_its_context_grew(fake):
    _run(fake, SIZES + """
ctx = hip.Context(0)
a = ctx.upload_synthetic(12, 48, 1)
ctx.run(a)
fake.fake_set_limit(fake.fake_used() + full // 2)
b = ctx.upload_synthetic(12, 48, 2)
ctx.run(b)
""")


def test_upload_takes_back_what_another_context_holds(fake):
    # room for the second system only without its own copies and without the
    # first's copies or launch buffers
    _run(fake, SIZES + """
for run in (False, True):
    one, two = hip.Context(0), hip.Context(0)
    a = one.upload_synthetic(12, 48, 1)
    assert one.sys_info(a)["bytes"] > full - swaps
    if run:
        one.run(a)
    fake.fake_set_limit(fake.fake_used() + full - swaps - 10**6)
    b = two.upload_synthetic(12, 48, 2)
    assert one.sys_info(a)["bytes"] <= full - swaps
    fake.fake_set_limit(1 << 40)
    one.run(a)
    two.run(b)
    two.close()
    one.close()
""")


def test_waits_for_a_run_of_another_context(fake):
    # the other context's run has 0.2 s to go when the upload finds no memory
    _run(fake, SIZES + """
import threading, time
one, two = hip.Context(0), hip.Context(0)
a = one.upload_synthetic(12, 48, 1)
one.run(a)
fake.fake_set_limit(fake.fake_used() + full - swaps - 10**6)
fake.fake_set_launch_us(100000)
ended = []
t = threading.Thread(target=lambda: (one.run(a), ended.append(time.time())))
t.start()
time.sleep(0.1)
b = two.upload_synthetic(12, 48, 2)
t.join()
assert one.sys_info(a)["bytes"] <= full - swaps
one.run(a)
two.run(b)
""")


def test_fewer_windows_where_four_do_not_fit(fake):
    # No=9, edge 16: 12288 class buffers of 4096 values for one window of 4096
    # tuples, 403 MB (four in GEMM order, 9^2 rows of 16: 510 MB)
    _run(fake, """
ctx = hip.Context(0)
ctx.set_option("window", 16)
s = ctx.upload_synthetic(9, 48, 1)
for batch in (0, 4):
    ctx.set_option("batch", batch)
    fake.fake_set_limit(fake.fake_used() + 512 * 10**6)
    ctx.run(s)
    fake.fake_set_limit(fake.fake_used() + 10**9)
    ctx.run(s, first=10, count=20000)
    fake.fake_set_limit(1 << 40)
""")
