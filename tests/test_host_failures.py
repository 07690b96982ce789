"""What the host code does when a device operation fails, and what it holds, on the CPU: the
library on a stand-in HIP runtime (tests/c_abi/hip_stub.c) whose kernels do nothing, whose
launches fail where a test says so and which counts the bytes of device memory."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = tmp_path_factory.mktemp("stub") / "libhip_stub.so"
    subprocess.run(["gcc", "-O1", "-std=c11", "-fPIC", "-shared", "-I/opt/rocm/include", "-o",
                    str(out), os.path.join(HERE, "c_abi", "hip_stub.c")], check=True, timeout=120)
    return str(out)


def _run(stub, code):
    head = f"import sys; sys.path.insert(0, {ROOT!r})\n" + """
import os
import numpy as np
from proxima_amd import FlatIndex, Metric, PqIndex

import ctypes
stub = ctypes.CDLL(os.environ["LD_PRELOAD"].split(":")[0])
def fail(name):
    os.environ["PX_STUB_FAIL_LAUNCH"] = name
def live():
    return ctypes.c_size_t.in_dll(stub, "px_stub_live").value
def launches(name, call):
    n = ctypes.c_long.in_dll(stub, "px_stub_launches")
    n.value, os.environ["PX_STUB_COUNT_LAUNCH"] = 0, name
    call()
    os.environ["PX_STUB_COUNT_LAUNCH"] = ""
    return n.value
"""
    preload = ":".join([stub, *filter(None, [os.environ.get("LD_PRELOAD")])])
    r = subprocess.run([sys.executable, "-c", head + code],
                       env=dict(os.environ, LD_PRELOAD=preload), capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-4000:])


# An add's rows are in place before the screening copy is brought up to date: a failure there
# leaves the index without a copy, not the caller with an error for rows that searches return.
@pytest.mark.parametrize("kernel", ["abs_max_kernel", "screen_rows_kernel", "screen_spread_kernel"])
def test_flat_add_survives_a_failed_screening_copy(stub, kernel):
    _run(stub, f"""
x = np.arange(5000 * 8, dtype=np.float32).reshape(5000, 8)
idx = FlatIndex(8, Metric.L2)
fail({kernel!r})
idx.add(x)
assert len(idx) == 5000 and np.array_equal(idx.vectors(), x)
idx.add(x[:7])
assert len(idx) == 5007
fail("")
idx.add(x[:1])
assert len(idx) == 5008
""")


@pytest.mark.parametrize("kernel", ["abs_max_kernel", "screen_rows_kernel"])
def test_flat_add_survives_a_failure_beside_it(stub, kernel):
    # an index with a copy: the rows added go to it in the same pass
    _run(stub, f"""
x = np.arange(5000 * 8, dtype=np.float32).reshape(5000, 8)
idx = FlatIndex(8, Metric.L2)
idx.add(x)
idx.add(x[:1])  # (room for 10,000 rows)
one = live()
idx.add(x[:1])
assert live() == one
fail({kernel!r})
idx.add(x[:7])
assert len(idx) == 5009 and live() < one - 10_000 * 256 + (1 << 16)
fail("")
idx.add(x[:1000])
assert len(idx) == 6009 and live() >= one - (1 << 16)
assert np.array_equal(idx.vectors(), np.concatenate([x, x[:1], x[:1], x[:7], x[:1000]]))
""")


@pytest.mark.parametrize("kernel", ["screen_codes_kernel", "screen_spread_kernel"])
def test_pq_add_survives_a_failed_screening_copy(stub, kernel):
    _run(stub, f"""
pq = PqIndex(8, Metric.L2, m=2, train_iters=0, train_sample=300)
pq.train(np.arange(300 * 8, dtype=np.float32).reshape(300, 8))
codes = np.arange(10000, dtype=np.uint8).reshape(5000, 2)
fail({kernel!r})
pq.add_codes(codes)
assert len(pq) == 5000 and np.array_equal(pq.codes(), codes)
fail("")
pq.add_codes(codes[:1])
assert len(pq) == 5001
""")


def test_a_failed_upload_still_fails_the_add(stub):
    _run(stub, """
x = np.ones((5000, 8), dtype=np.float32)
idx = FlatIndex(8, Metric.L2)
fail("row_norms_kernel")
try:
    idx.add(x)
except RuntimeError:
    assert len(idx) == 0
else:
    raise AssertionError("no error")
fail("")
idx.add(x)
assert len(idx) == 5000
""")


# The screening copy of an index of codes takes at most 8 GiB, room for more rows counted, and
# nothing once the rows are past that: 256 bytes a row, 33.5M rows. (The copy is never touched
# here: the stand-in's kernels do nothing.)
def test_pq_screening_copy_is_bounded_and_given_back(stub):
    _run(stub, """
pq = PqIndex(4, Metric.L2, m=4, train_iters=0, train_sample=256)
pq.train(np.arange(256 * 4, dtype=np.float32).reshape(256, 4))
codes = np.zeros((17_000_000, 4), dtype=np.uint8)
pq.add_codes(codes)
one = live()
assert one > 17_000_000 * 256
pq.add_codes(codes[:10])  # room for 34M codes
assert 17_000_000 * 256 < live() < (8 << 30) + 34_000_000 * 8 + (1 << 20), live()
pq.add_codes(codes[:16_600_000])
assert live() < 68_000_010 * 4 + (1 << 20), live()
""")


def test_flat_screening_copy_is_bounded_and_given_back(stub):
    # 8 dims: 32 bytes a row and 256 of copy
    _run(stub, """
idx = FlatIndex(8, Metric.L2)
x = np.zeros((17_000_000, 8), dtype=np.float32)
x[0, 0] = 1
idx.add(x)
idx.add(x[:16_900_000])  # room for 34M rows: their copy would be 8.7 GB
assert live() < 34_000_000 * 37 + (1 << 20), live()
""")


def test_pq_copy_that_cannot_be_had_is_not_tried_at_every_search(stub):
    # device memory for the codes and not for the copy: one try an eighth more rows
    _run(stub, """
pq = PqIndex(8, Metric.L2, m=8, train_iters=0, train_sample=256)
pq.train(np.arange(256 * 8, dtype=np.float32).reshape(256, 8))
codes = np.zeros((40_000, 8), dtype=np.uint8)
os.environ["PX_DEVICE_BUDGET"] = str(9_000_000)
pq.add_codes(codes)
assert live() < 1_000_000
del os.environ["PX_DEVICE_BUDGET"]
q = np.zeros((1, 8), dtype=np.float32)
assert launches("screen_codes", lambda: [pq.search_batch(q, k=1) for _ in range(5)]) == 0
assert launches("screen_codes", lambda: pq.add_codes(codes[:10])) == 0
assert launches("screen_codes", lambda: pq.add_codes(codes[:5000])) == 1
assert live() > 45_000 * 256
""")


def test_an_add_of_a_few_rows_waits_no_more_than_without_a_copy(stub):
    # the waits of the host are what such an add costs
    _run(stub, """
def waits(call):
    n = ctypes.c_long.in_dll(stub, "px_stub_waits")
    n.value = 0
    call()
    return n.value
x = np.arange(5000 * 8, dtype=np.float32).reshape(5000, 8)
n = []
for screening in (False, True):
    idx = FlatIndex(8, Metric.L2)
    idx._screening(screening)
    idx.add(x)
    idx.add(x[:1])
    n.append(waits(lambda: idx.add(x[:1])))
assert n[0] == n[1] == 1, n
""")
