"""Out-of-device-memory paths on the GPU, simulated with PX_DEVICE_BUDGET.

PX_DEVICE_BUDGET (bytes, read at every device allocation of the library) caps the library's
own device memory; an allocation past it fails with hipErrorOutOfMemory as on a full device
(the reference returns NULL from gpu_knn_create on a failed cudaMalloc, gpu.rs:31-33, and its
Python surface raises). Each failure must leave the index as it was -- rows counted, results
unchanged -- and the same index must work again once memory is there.
"""
import contextlib
import gc
import os

import numpy as np
import pytest

import oracle
from proxima_amd import FlatIndex, Metric, PqIndex, datagen

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def device_budget(nbytes):
    os.environ["PX_DEVICE_BUDGET"] = str(nbytes)
    try:
        yield
    finally:
        del os.environ["PX_DEVICE_BUDGET"]


def test_flat_add_and_search_out_of_memory(gpu):
    data = datagen.sift_like(30_000, 48, 301)
    more = datagen.sift_like(40_000, 48, 302)
    q = datagen.sift_like(40, 48, 303)
    big_q = datagen.sift_like(3000, 48, 304)
    idx = FlatIndex(48, Metric.L2)
    idx.add(data)
    ids0, d0 = idx.search_batch(q, k=10)
    print("case flat add past the budget", flush=True)
    with device_budget(1):  # nothing more can be allocated
        with pytest.raises(RuntimeError, match="out of memory"):
            idx.add(more)  # the corpus mirror must grow
        assert len(idx) == 30_000
        ids, d = idx.search_batch(q, k=10)  # its workspace is already there
        assert np.array_equal(ids, ids0) and np.array_equal(d, d0)
        print("case flat search past the budget", flush=True)
        with pytest.raises(RuntimeError, match="out of memory"):
            idx.search_batch(big_q, k=10)  # a larger batch needs a larger workspace
        with pytest.raises(RuntimeError, match="out of memory"):
            idx.search_batch(q, k=500)  # the collect path's buffers
    print("case flat after the budget", flush=True)
    idx.add(more)
    both = np.concatenate([data, more])
    assert len(idx) == 70_000
    for qq, k in ((q, 10), (big_q, 10), (q, 500)):
        ids, d = idx.search_batch(qq, k=k)
        o_ids, o_d, _ = oracle.flat_search(both, qq, k, oracle.L2)
        assert np.array_equal(ids, o_ids) and np.array_equal(d, o_d), k


def test_pq_train_and_add_out_of_memory(gpu):
    data = datagen.gaussian(6000, 32, 311)
    q = datagen.gaussian(20, 32, 312)
    pq = PqIndex(32, Metric.L2, m=8, nbits=6, train_iters=5, train_sample=4000)
    print("case pq train past the budget", flush=True)
    with device_budget(1):
        with pytest.raises(RuntimeError, match="out of memory"):
            pq.train(data)
    pq.train(data)
    pq.add(data[:2000])
    ids0, d0 = pq.search_batch(q, k=10)
    print("case pq add past the budget", flush=True)
    with device_budget(1):
        with pytest.raises(RuntimeError, match="out of memory"):
            pq.add(data[2000:])  # 6,000 codes pass the first code buffer's 4,096 rows
        assert len(pq) == 2000
        ids, d = pq.search_batch(q, k=10)
        assert np.array_equal(ids, ids0) and np.array_equal(d, d0)
    pq.add(data[2000:])
    assert len(pq) == 6000
    ids, d = pq.search_batch(q, k=10)
    o_ids, o_d, _ = oracle.pq_search(pq.codebooks(), pq.codes(), q, 10, oracle.L2)
    assert np.array_equal(ids, o_ids) and np.array_equal(d, o_d)


def test_flat_add_that_fits_without_the_screening_copy(gpu):
    # 40,000 rows of 128 dims: 20.5 MB and a screening copy of 10.2; the next row grows the index
    # to 80,000 rows' room, 41 MB beside the old rows. 67 MB hold both and a search's scratch, not
    # the copy too: the copy gives way, and is made again (20.5 MB) once the old rows are gone.
    gc.collect()
    data = datagen.gaussian(40_001, 128, 321)
    q = datagen.gaussian(30, 128, 322)
    idx = FlatIndex(128, Metric.L2)
    idx.add(data[:40_000])
    idx.search_batch(q, k=10)
    assert idx._last_timing()["screened"]
    print("case flat add that fits without the copy", flush=True)
    with device_budget(67_000_000):
        idx.add(data[40_000:])
        ids, d = idx.search_batch(q, k=10)
    assert idx._last_timing()["screened"]
    o_ids, o_d, _ = oracle.flat_search(data, q, 10, oracle.L2)
    assert np.array_equal(ids, o_ids) and np.array_equal(d, o_d)


def test_pq_add_that_fits_without_the_screening_copy(gpu):
    # 100,000 codes of 64 bytes: 6.4 MB and a copy of 26; room for twice as many is 12.8 MB more,
    # which 40 MB hold without the copy (and not the 51 MB copy after)
    gc.collect()
    rng = np.random.default_rng(323)
    pq = PqIndex(64, Metric.L2, m=64, train_iters=1, train_sample=1000)
    pq.train(datagen.gaussian(1000, 64, 324))
    codes = rng.integers(0, 256, size=(100_001, 64)).astype(np.uint8)
    pq.add_codes(codes[:100_000])
    q = datagen.gaussian(20, 64, 325)
    pq.search_batch(q, k=10)
    assert pq._last_timing()["screened"]
    print("case pq add that fits without the copy", flush=True)
    with device_budget(40_000_000):
        pq.add_codes(codes[100_000:])
        ids, d = pq.search_batch(q, k=10)
        assert not pq._last_timing()["screened"]
    o_ids, o_d, _ = oracle.pq_search(pq.codebooks(), codes, q, 10, oracle.L2)
    assert np.array_equal(ids, o_ids) and np.array_equal(d, o_d)
    pq.search_batch(q, k=10)


@pytest.mark.parametrize("budget,copy_kept", [(78_700_000, True), (77_400_000, False)])
def test_flat_search_that_fits_without_screening(gpu, budget, copy_kept):
    # 100,000 rows of 128 dims and their copy: 77.2 MB. A screened search of 17 queries wants 2.3
    # MB of candidates, the fp32 lists 0.6: 78.7 MB hold those, 77.4 only without the copy.
    gc.collect()
    data = datagen.gaussian(100_000, 128, 331)
    q = datagen.gaussian(17, 128, 332)
    idx = FlatIndex(128, Metric.L2)
    idx.add(data)
    o_ids, o_d, _ = oracle.flat_search(data, q, 10, oracle.L2)
    print(f"case flat search without screening, budget {budget}", flush=True)
    with device_budget(budget):
        ids, d = idx.search_batch(q, k=10)
        assert not idx._last_timing()["screened"]
        assert np.array_equal(ids, o_ids) and np.array_equal(d, o_d)
    ids, d = idx.search_batch(q, k=10)
    assert idx._last_timing()["screened"] == copy_kept
    assert np.array_equal(ids, o_ids) and np.array_equal(d, o_d)
    idx.add(data[:15_000])  # (room for it: the copy is brought up to date, or made again)
    idx.search_batch(q, k=10)
    assert idx._last_timing()["screened"]


def test_pq_search_that_fits_without_screening(gpu):
    # 100,000 codes of 16 bytes of 32 dims: 1.6 MB and a copy of 26; 500 queries, k = 10
    gc.collect()
    data = datagen.gaussian(100_000, 32, 341)
    q = datagen.gaussian(500, 32, 342)
    pq = PqIndex(32, Metric.L2, m=16, train_iters=1, train_sample=1000)
    pq.train(data)
    pq.add(data)
    print("case pq search without screening", flush=True)
    with device_budget(29_500_000):
        ids, d = pq.search_batch(q, k=10)
        assert not pq._last_timing()["screened"]
    o_ids, o_d, _ = oracle.pq_search(pq.codebooks(), pq.codes(), q, 10, oracle.L2)
    assert np.array_equal(ids, o_ids) and np.array_equal(d, o_d)
