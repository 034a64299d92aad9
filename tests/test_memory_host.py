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
