"""Host side of the serving loop's results, run against a HIP runtime in host
memory (fake_hip.cpp): a thread that cannot be started costs speed only, and the
library's streams and events stay on the server's device whatever device a
caller has current."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEAD = """
import ctypes, sys, threading
sys.path.insert(0, %r)
import numpy as np
import le2d_amd
fake = ctypes.CDLL(%r)
NX, NY = 300, 100  # 1.2 MB: several pieces and helpers


def result(s, i):
    a = np.ones((NY, NX, 5))
    rc = s.lib.le2d_server_result(s.h, i, a.ctypes.data)
    assert rc == 0, s.lib.le2d_last_error()
    assert not a.any()  # the device state is zero: nothing runs on it


def requests(s, n):
    ids = [s.submit(NX, NY, 2, np.float64, keep=True) for _ in range(n)]
    s.drain(60)
    return ids
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-o", so,
                    os.path.join(ROOT, "tests", "fake_hip.cpp")], check=True)
    return so


def _run(fake, body):
    out = subprocess.run([sys.executable, "-c", HEAD % (ROOT, fake) + body],
                         env=dict(os.environ, LD_PRELOAD=fake), capture_output=True, text=True,
                         timeout=120)
    assert out.returncode == 0 and "done" in out.stdout, out.stderr[-2000:]


@pytest.mark.parametrize("k", [1, 2, 3])
def test_no_memory_for_a_helper(fake, k):
    _run(fake, """
with le2d_amd.Server(1 << 28, 4) as s:
    for i in requests(s, 2):
        fake.fake_fail_new(%d)
        result(s, i)
        fake.fake_fail_new(0)
print("done")
""" % k)


def test_callers_with_another_device(fake):
    _run(fake, """
with le2d_amd.Server(1 << 28, 4) as s:
    ids = requests(s, 3)

    def caller():
        fake.hipSetDevice(1)
        result(s, ids[0])
        d = ctypes.c_int()
        fake.hipGetDevice(ctypes.byref(d))
        assert d.value == 1
        left.append(True)

    left = []
    t = threading.Thread(target=caller)
    t.start()
    t.join()
    assert left
    result(s, ids[1])
    assert fake.fake_foreign() == 0 and fake.fake_cross() == 0, (fake.fake_foreign(), fake.fake_cross())
print("done")
""")


def test_server_on_the_creating_thread_s_device(fake):
    _run(fake, """
fake.hipSetDevice(1)
with le2d_amd.Server(1 << 28, 4) as s:
    for i in requests(s, 2):
        result(s, i)
assert fake.fake_cross() == 0, fake.fake_cross()
print("done")
""")
