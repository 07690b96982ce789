"""GPU parity of screened FlatIndex searches (px_screen.hip).

Indexes of at least 4,096 rows keep a copy of them rounded to fp16 (rows of 128 dims that are
exact in fp16 have one as they are). A search multiplies that copy, rules out every row proven to lie outside the
best k by a bound on the rounding, and recomputes the keys of the rest in the reference's
arithmetic (flat.rs:106-148 with distance.rs:3-39), so its results equal the oracle's: ids and
distances bit for bit, with no exemption for near ties. Queries that cannot be screened
(bounds too wide for the data, scales too far apart) take the fp32 scans and must give what
those give.
"""
import numpy as np
import pytest

import oracle
from proxima_amd import FlatIndex, Metric, PqIndex, datagen

pytestmark = pytest.mark.gpu


def _index(data, metric):
    idx = FlatIndex(data.shape[1], Metric.L2 if metric == oracle.L2 else Metric.InnerProduct)
    idx.add(data)
    return idx


def _search(idx, q, k, mask=None):
    ids, d = (idx.search_batch(q, k=k) if mask is None
              else idx.search_batch_filtered(q, mask, k=k))
    return ids, d, idx._last_timing()


def _same(a, b):
    assert np.array_equal(a[0], b[0])
    assert np.array_equal(a[1].view(np.uint32), b[1].view(np.uint32))


def _exact(data, q, k, metric, mask=None, idx=None):
    print(f"case screen n={data.shape[0]} dim={data.shape[1]} nq={q.shape[0]} k={k} "
          f"metric={metric} mask={mask is not None}", flush=True)
    idx = idx or _index(data, metric)
    ids, d, info = _search(idx, q, k, mask)
    assert info["screened"] and info["path"] == "screened" and not info["scan_f16"], info
    o_ids, o_d, _ = oracle.flat_search(data, q, k, metric, mask=mask)
    _same((ids, d), (o_ids, o_d))
    return idx, info


# row groups of 128, tiles of 32, waves of 64 queries, workgroups of 512, chunks of 128 dims:
# whole ones, one more and one less; the fewest rows; the largest k (a 64th of the rows)
@pytest.mark.parametrize("n,dim,nq,k,metric,kind", [
    (4_096, 128, 17, 1, oracle.L2, "gauss"),
    (4_097, 8, 64, 64, oracle.IP, "gauss"),
    (9_999, 36, 1, 3, oracle.L2, "unit"),
    (70_000, 77, 16, 100, oracle.IP, "gauss"),
    (5_001, 1100, 3, 10, oracle.L2, "gauss"),
    (50_017, 100, 65, 100, oracle.L2, "gauss"),
    (49_279, 129, 513, 37, oracle.L2, "unit"),
    (52_000, 384, 300, 812, oracle.IP, "unit"),
    (50_000, 1000, 40, 10, oracle.L2, "gauss"),
    (120_000, 120, 1025, 16, oracle.IP, "unit"),
    (300_000, 64, 260, 24, oracle.L2, "sift"),
])
def test_sizes(gpu, n, dim, nq, k, metric, kind):
    gen = {"gauss": datagen.gaussian, "unit": datagen.unit_gaussian, "sift": datagen.sift_like}[kind]
    _, info = _exact(gen(n, dim, 901), gen(nq, dim, 902), k, metric)
    assert info["collect_rounds"] == 1


@pytest.mark.parametrize("n,k,nq", [(262_144, 4_096, 20), (192_000, 3_000, 20), (140_000, 2_000, 3),
                                    (64_000, 1_000, 300), (5_000, 78, 40)])
def test_most_neighbours(gpu, n, k, nq):
    # k a 64th of the rows or little less: the sample's threshold still lets no more through than
    # the select holds, and every query finishes in the first round
    _, info = _exact(datagen.gaussian(n, 32, 905), datagen.gaussian(nq, 32, 906), k, oracle.L2)
    assert info["collect_rounds"] == 1, info


@pytest.mark.parametrize("dim", [96, 200])
@pytest.mark.parametrize("metric", [oracle.L2, oracle.IP])
def test_filtered(gpu, dim, metric):
    data = datagen.gaussian(120_003, dim, 911)
    q = datagen.gaussian(70, dim, 912)
    for density in (0.5, 0.98):
        _exact(data, q, 20, metric, mask=datagen.mask(120_003, density, 913))
    # fewer kept rows than screening takes: the fp32 scans
    idx = _index(data, metric)
    mask = datagen.mask(120_003, 0.03, 914)
    ids, d, info = _search(idx, q, 20, mask)
    assert not info["screened"]


def test_near_rows_in_one_run(gpu):
    # every near row lies in one run of the corpus: the regions of one split overflow and the
    # queries go round again
    rng = np.random.default_rng(921)
    data = (rng.standard_normal((60_000, 40)) * 3 + 20).astype(np.float32)
    data[30_000:32_500] -= 20
    q = rng.standard_normal((100, 40)).astype(np.float32)
    _, info = _exact(data, q, 500, oracle.L2)
    assert info["collect_rounds"] >= 2, info


def test_near_rows_are_the_sampled_ones(gpu):
    # the sample (every 14th row) is near, the rest far: its thresholds admit too few rows
    rng = np.random.default_rng(931)
    n = 60_000
    data = (rng.standard_normal((n, 24)) * 30).astype(np.float32)
    data[::n // 4096] = rng.standard_normal((len(data[::n // 4096]), 24)) * 2
    q = (rng.standard_normal((80, 24)) * 2).astype(np.float32)
    _exact(data, q, 900, oracle.L2)


def test_ties(gpu):
    # few distinct distances: thousands of equal keys at the cut go to the lower row
    rng = np.random.default_rng(941)
    data = rng.integers(0, 2, size=(60_000, 14)).astype(np.float32)
    q = rng.integers(0, 2, size=(40, 14)).astype(np.float32)
    for metric in (oracle.L2, oracle.IP):
        idx = _index(data, metric)
        ids, d, info = _search(idx, q, 20)
        assert info["screened"]
        _same((ids, d), oracle.flat_search(data, q, 20, metric)[:2])


@pytest.mark.parametrize("name", ["offset", "query scale", "zero queries", "outlier row"])
def test_what_screening_leaves_open(gpu, name):
    # the bound spans every row (a large common offset), is infinite (scales 2^45 apart), or is
    # widened by one row of huge norm, added later: whatever screening finishes or leaves, the
    # results are the fp32 scans'
    rng = np.random.default_rng(951)
    data = rng.standard_normal((60_000, 64)).astype(np.float32)
    q = rng.standard_normal((90, 64)).astype(np.float32)
    if name == "offset":
        # (multiples of 2^-8 near 128: sums of a few of them are exact, so that the fp32 scan's
        # own candidates are right)
        data = (np.round(data * 2) / 2 + 128).astype(np.float32)
        q = (np.round(q * 2) / 2 + 128).astype(np.float32)
    elif name == "query scale":
        q *= np.float32(2.0 ** 45)
    elif name == "zero queries":
        q[::3] = 0
    metric = oracle.IP if name == "query scale" else oracle.L2
    idx = _index(data, metric)
    if name == "outlier row":
        assert _search(idx, q, 10)[2]["screened"]
        idx.add(np.full((1, 64), 3e4, dtype=np.float32))
    print(f"case screen left open: {name}", flush=True)
    ids, d, info = _search(idx, q, 10)
    # (rows so far from the origin that fp16 cannot tell them apart are not screened)
    assert info["screened"] == (name != "offset")
    if name == "query scale":
        assert info["collect_rounds"] == 1  # (90 queries: the fp32 lists finish them)
    # an index on which such a search is no accident is not screened again; one whose rows can be
    # told apart by queries of their own kind is
    ids2, d2, info = _search(idx, q, 10)
    assert info["screened"] == (name in ("query scale", "zero queries"))
    _same((ids, d), (ids2, d2))
    idx._scan_f16(False)
    ids32, d32, info32 = _search(idx, q, 10)
    assert not info32["screened"]
    _same((ids, d), (ids32, d32))


def test_rows_added_later(gpu):
    # the copy grows with the rows, is made again when a row passes its scale, and starts when
    # an index gets its 4,096th row or its first row that is not exact in fp16
    a, b = datagen.gaussian(4_000, 72, 961), datagen.gaussian(30_000, 72, 962)
    big = (datagen.gaussian(40_000, 72, 963) * 128).astype(np.float32)
    q = datagen.gaussian(50, 72, 964)
    idx = _index(a, oracle.IP)
    assert not _search(idx, q, 5)[2]["screened"]
    idx.add(b)
    both = np.concatenate([a, b])
    _exact(both, q, 5, oracle.IP, idx=idx)
    idx.add(big)
    _exact(np.concatenate([both, big]), q, 5, oracle.IP, idx=idx)
    s, g = datagen.sift_like(50_000, 128, 965), datagen.gaussian(10_000, 128, 966)
    q = datagen.sift_like(60, 128, 967)
    idx = _index(s, oracle.L2)
    info = _search(idx, q, 100)[2]
    assert not info["screened"]
    idx.add(g)
    _exact(np.concatenate([s, g]), q, 10, oracle.L2, idx=idx)


def test_magnitudes(gpu):
    # rows and queries of any common scale within [2^-40, 2^40]; none past it
    data, q = datagen.gaussian(50_000, 48, 971), datagen.gaussian(40, 48, 972)
    for e in (-30, 30):
        _exact(np.ldexp(data, e), np.ldexp(q, e), 10, oracle.IP)
    idx = _index(np.ldexp(data, 50), oracle.IP)
    assert not _search(idx, q, 10)[2]["screened"]
    # ... added later too, where the copy's scale could still carry them
    idx = _index(np.ldexp(data, 37), oracle.IP)
    assert _search(idx, q, 10)[2]["screened"]
    idx.add(np.ldexp(data[:100], 42))
    assert not _search(idx, q, 10)[2]["screened"]
    # rows added later may all be smaller than that
    idx = _index(data, oracle.IP)
    tiny = np.ldexp(datagen.gaussian(100, 48, 973), -60)
    idx.add(tiny)
    _exact(np.concatenate([data, tiny]), q, 10, oracle.IP, idx=idx)


def test_queries_whose_residuals_square_to_nothing(gpu):
    # Inner products of tiny queries: every rounding residual is about 2^-75, whose square is
    # no fp32 number, while the largest element, 2^-60, is exact. For each query two rows whose
    # fp16 keys differ by 0.3 (in units of 2^-89; the other terms of the bound are 0.05) in
    # favour of one and whose keys differ by 0.5 in favour of the other, 60 residuals of 0.9 / 64
    # all pulling one way: a bound without the residuals drops the nearest row.
    rng = np.random.default_rng(975)
    n, dim, nq = 20_000, 64, 5
    data = rng.choice([-1, 0, 1], size=(n, dim)).astype(np.float32) * np.float32(2.0 ** -5)
    data[:, 63] = 0
    up, down, gap, big = slice(0, 30), slice(30, 60), 60, 63
    q = np.zeros((nq, dim))
    q[:, up], q[:, down], q[:, gap], q[:, big] = 40 + 0.9 / 64, 40 - 0.9 / 64, 0.3125, 512
    for i in range(nq):
        sign = rng.choice([-1, 1], size=dim)
        q[i] *= sign
        data[100 + i] = data[7000 + i] = 0
        data[100 + i, up] = sign[up]
        data[7000 + i, down] = sign[down]
        data[7000 + i, gap] = sign[gap]
    q = np.ldexp(q, -69).astype(np.float32)
    _exact(np.ldexp(data, -20), q, 1, oracle.IP)


def test_give_up(gpu):
    # a stage wait that gives up (one poll) fails the search; the next one is right
    data, q = datagen.gaussian(200_000, 128, 981), datagen.gaussian(100, 128, 982)
    idx = _index(data, oracle.L2)
    idx._spin_limit(1)
    with pytest.raises(RuntimeError, match="stage sync"):
        idx.search_batch(q, k=10)
    idx._spin_limit(0)
    _exact(data, q, 10, oracle.L2, idx=idx)


@pytest.mark.parametrize("nq", [3, 300])
def test_too_many_rows_within_the_bound(gpu, nq):
    # two thirds of the rows spread widely, a third in one tight group about a far point, all of
    # it within the bound of the neighbours of queries beside it: the ladder gives such queries
    # up and the scans without screening answer them; others of the batch are screened (values
    # near the group as in the offset case above)
    rng = np.random.default_rng(985)
    data = np.round(rng.standard_normal((30_000, 64)) * 100).astype(np.float32)

    def tight(n):
        return 128 + np.round(rng.standard_normal((n, 64)) * 2) / 2

    data[::3] = tight(10_000)  # (a period that a whole step of a row sample would meet)
    q = tight(nq).astype(np.float32)
    q[::4] = np.round(rng.standard_normal((len(q[::4]), 64)) * 100)
    _, info = _exact(data, q, 10, oracle.L2)
    assert info["collect_rounds"] == (2 if nq == 3 else 1)  # (3: the vector-ALU scan collects)


@pytest.mark.parametrize("kind", ["two groups", "fifty groups", "copies"])
def test_rows_too_close_together_for_screening(gpu, kind):
    # rows in groups that the bound cannot tell apart, larger than a select is worth: after one
    # search that screening left open such an index is not screened, until it has other rows too
    rng = np.random.default_rng(986)
    centres = {"two groups": 2, "fifty groups": 50, "copies": 16}[kind]
    c = rng.standard_normal((centres, 64)) * 64

    def near(n):
        off = rng.standard_normal((n, 64)) / 256 if kind != "copies" else 0
        return (c[rng.integers(centres, size=n)] + off).astype(np.float32)

    data, q = near(60_000), near(20)
    idx = _index(data, oracle.L2)
    first, second = _search(idx, q, 10), _search(idx, q, 10)
    assert first[2]["screened"] and not second[2]["screened"]
    _same(first[:2], second[:2])
    other = (datagen.gaussian(200_000, 64, 987) * 64).astype(np.float32)
    idx.add(other)
    assert _search(idx, other[:20], 10)[2]["screened"]


def test_rows_exact_in_fp16_too_close_together(gpu):
    # the same of the fp16 copy of exact rows, whose vector and list routes are screened: copies
    # of 16 rows
    rng = np.random.default_rng(989)
    data = rng.integers(0, 256, size=(16, 128)).astype(np.float32)[rng.integers(16, size=70_000)]
    q = rng.integers(0, 256, size=(20, 128)).astype(np.float32)
    idx = _index(data, oracle.L2)
    o = oracle.flat_search(data, q, 10, oracle.L2)[:2]
    for screened in (True, False, False):
        ids, d, info = _search(idx, q, 10)
        assert info["screened"] == screened
        _same((ids, d), o)
    more = rng.integers(0, 256, size=(200_000, 128)).astype(np.float32)
    idx.add(more)
    for _ in range(2):
        ids, d, info = _search(idx, more[:20], 10)
        assert info["screened"]
        _same((ids, d), oracle.flat_search(np.concatenate([data, more]), more[:20], 10,
                                           oracle.L2)[:2])


def test_codes_of_few_distinct_rows_are_not_screened(gpu):
    rng = np.random.default_rng(988)
    data = rng.standard_normal((100_000, 8)).astype(np.float32)
    pq = PqIndex(8, Metric.L2, m=1, nbits=8, train_iters=2, train_sample=4000)
    pq.train(data)
    pq.add(data)
    q = rng.standard_normal((20, 8)).astype(np.float32)
    ids, d, info = _search(pq, q, 10)
    assert not info["screened"]
    _same((ids, d), oracle.pq_search(pq.codebooks(), pq.codes(), q, 10, oracle.L2)[:2])


# ADC searches: the rows that the codes stand for, screened the same way; a key recomputed as
# the ADC sum (pq.rs:299-347)
@pytest.mark.parametrize("m,nbits,dim,nq,k,metric,density", [
    (16, 8, 128, 300, 10, oracle.L2, None),
    (16, 8, 128, 65, 100, oracle.IP, 0.9),
    (9, 8, 36, 40, 128, oracle.L2, None),     # a group of 8 subspaces and one more
    (4, 6, 8, 70, 129, oracle.IP, None),      # past the lists' k; few distinct rows, ties
    (3, 4, 24, 50, 30, oracle.L2, None),      # 4,096 distinct rows: ties at every cut
    (20, 8, 240, 513, 5, oracle.L2, 0.95),
])
def test_adc(gpu, m, nbits, dim, nq, k, metric, density):
    n = 56_003
    data = datagen.gaussian(n, dim, 991)
    q = datagen.gaussian(nq, dim, 992)
    mask = datagen.mask(n, density, 993) if density else None
    pq = PqIndex(dim, Metric.L2 if metric == oracle.L2 else Metric.InnerProduct, m=m, nbits=nbits,
                 train_iters=3, train_sample=4000)
    pq.train(data)
    pq.add(data[:50_000])
    pq.add(data[50_000:])
    print(f"case screen adc m={m} nbits={nbits} dim={dim} nq={nq} k={k} metric={metric}", flush=True)
    ids, d, info = _search(pq, q, k, mask)
    assert info["screened"]
    o_ids, o_d, _ = oracle.pq_search(pq.codebooks(), pq.codes(), q, k, metric, mask=mask)
    _same((ids, d), (o_ids, o_d))


def test_adc_rows_added_and_trained_again(gpu):
    # the copy of the coded rows follows the codes and the codebooks
    data, q = datagen.gaussian(60_000, 32, 994), datagen.gaussian(30, 32, 995)
    pq = PqIndex(32, Metric.L2, m=8, train_iters=2, train_sample=3000)
    pq.train(data)
    pq.add(data)
    for step in range(3):
        ids, d, info = _search(pq, q, 10)
        assert info["screened"]
        o_ids, o_d, _ = oracle.pq_search(pq.codebooks(), pq.codes(), q, 10, oracle.L2)
        _same((ids, d), (o_ids, o_d))
        if step == 0:
            pq.add(data[:7_000])
        elif step == 1:
            pq.train((data * 3)[::-1].copy())
            pq.add(data[:55_000])


# rows of 128 dims exact in fp16 (their fp16 copy has no residual): the vector route whatever
# the queries hold, the list route (from 65,536 rows on) exact queries or not, host arrays and
# device queries alike
@pytest.mark.parametrize("nq,k", [(1, 10), (16, 50), (17, 10), (200, 100)])
@pytest.mark.parametrize("exact", [True, False])
def test_rows_exact_in_fp16(gpu, nq, k, exact):
    import ctypes
    from proxima_amd import _lib
    lib = _lib.load()
    data = datagen.sift_like(70_001, 128, 996)
    q = datagen.sift_like(nq, 128, 997)
    if not exact:
        q = (q + 0.3).astype(np.float32)
    for metric in (oracle.L2, oracle.IP):
        idx = _index(data, metric)
        o = oracle.flat_search(data, q, k, metric)[:2]
        ids, d, info = _search(idx, q, k)
        assert info["screened"] and not info["scan_f16"], info
        _same((ids, d), o)
        bufs = [(ctypes.c_void_p(), n) for n in (q.nbytes, nq * k * 8, nq * k * 4)]
        try:
            for p, n in bufs:
                assert lib.px_dev_alloc(ctypes.byref(p), n) == 0
            (dq, _), (di, _), (dd, _) = bufs
            assert lib.px_dev_upload(dq, q.ctypes.data, q.nbytes) == 0
            assert lib.px_flat_search_device(idx._h, dq, nq, k, None, di, dd) == 0
            info = idx._last_timing()
            assert info["screened"] and not info["scan_f16"], info
            assert lib.px_dev_download(ids.ctypes.data, di, ids.nbytes) == 0
            assert lib.px_dev_download(d.ctypes.data, dd, d.nbytes) == 0
            _same((ids, d), o)
        finally:
            for p, _ in bufs:
                lib.px_dev_free(p)


def test_what_ran_is_reported(gpu):
    # a screened search reports the screening scan, its own rounds and no other scan; with
    # screening off the same search reports the scan that takes its place, and so does the
    # no-allocation entry point, which is never screened
    import ctypes
    from proxima_amd import _lib
    lib = _lib.load()
    data, q = datagen.gaussian(30_000, 64, 1001), datagen.gaussian(40, 64, 1002)
    idx = _index(data, oracle.L2)

    def said():
        t = idx._last_timing()
        return [t[x] for x in ("screened", "path", "scan_f16", "collect_rounds")]

    _search(idx, q, 10)
    assert said() == [True, "screened", False, 1]
    bufs = [(ctypes.c_void_p(), n) for n in (q.nbytes, 40 * 10 * 8, 40 * 10 * 4)]
    try:
        for p, n in bufs:
            assert lib.px_dev_alloc(ctypes.byref(p), n) == 0
        (dq, _), (di, _), (dd, _) = bufs
        assert lib.px_dev_upload(dq, q.ctypes.data, q.nbytes) == 0
        assert lib.px_flat_search_device_noalloc(idx._h, dq, 40, 10, None, di, dd) == 0
    finally:
        for p, _ in bufs:
            lib.px_dev_free(p)
    assert said() == [False, "lists", False, 0]
    idx._screening(False)
    _search(idx, q, 10)
    assert said() == [False, "lists", False, 0]
    idx.add(data[:10])
    _search(idx, q, 10)
    assert said() == [False, "lists", False, 0]
    idx._screening(True)
    _same(_search(idx, q, 10)[:2], oracle.flat_search(np.concatenate([data, data[:10]]), q, 10,
                                                      oracle.L2)[:2])
    assert said() == [True, "screened", False, 1]
    idx._scan_f16(False)
    _search(idx, q, 10)
    assert said() == [False, "lists", False, 0]

    pq = PqIndex(64, Metric.L2, m=16, train_iters=1, train_sample=1000)
    pq.train(data)
    pq.add(data)
    a = pq.search_batch(q, k=10)
    assert pq._last_timing()["screened"]
    pq._screening(False)
    _same(pq.search_batch(q, k=10), a)
    assert not pq._last_timing()["screened"]
    pq._screening(True)
    _same(pq.search_batch(q, k=10), a)
    assert pq._last_timing()["screened"]


def test_results_past_the_mapped_buffer(gpu):
    # results of more than 16 MB are copied back, smaller ones written to host memory directly;
    # queries of up to 65,536 values are read from there: one handle through all of them
    data = datagen.gaussian(30_000, 40, 998)
    idx = _index(data, oracle.L2)
    for nq, k in ((3, 7), (1639, 50), (2987, 468), (2988, 468), (2, 400), (40, 300)):
        q = datagen.gaussian(nq, 40, 1000 + nq)
        _exact(data, q, k, oracle.L2, idx=idx)
