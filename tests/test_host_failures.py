"""What the host code does when a device operation fails, on the CPU: the library on a stand-in
HIP runtime (tests/c_abi/hip_stub.c) whose kernels do nothing and whose launches fail where a
test says so."""
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

def fail(name):
    os.environ["PX_STUB_FAIL_LAUNCH"] = name
"""
    r = subprocess.run([sys.executable, "-c", head + code], env=dict(os.environ, LD_PRELOAD=stub),
                       capture_output=True, text=True, timeout=120)
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
