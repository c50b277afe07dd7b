"""The scan + pick kernel pair (long last-axis rows) and the sampling-style entry
point, on the GPU, through the C ABI.

* The pair against the chunk + merge kernels it stands in for (vkop_hip_tune
  "rows.path"): bit-identical results -- both implement "top-k by (probability, then
  lower index) of the row's softmax" and sum the row's terms in orders of their own,
  so a value may differ by an ulp where the sums round apart; indices, and values
  where the sums agree, are compared exactly, values otherwise to one ulp -- and
  against the oracle: the monotone-ranking invariants on every row, exact indices
  wherever the oracle's probabilities around the cut are well apart.
* vkop_hip_softmax_topk_sampling against the oracle's sampling variant and against
  the plain entry point on a tensor scaled on the host.
* The NaN replacement option of the softmax on axes other than the last.
"""
import numpy as np
import pytest

import oracle
from helpers import check_fused_invariants, check_topk_invariants, half_ulp_diff, ulp_diff, well_separated_cut
from vkop_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ops():
    from vkop_amd import capi, ops as _ops
    capi.lib()              # raises if the HIP library is not built: no fallback
    capi.init(0)
    yield _ops
    capi.tune("rows.path", 0)


def dev(a):
    a = np.ascontiguousarray(a)
    if a.dtype == np.uint16:
        a = a.view(np.float16)
    return torch.from_numpy(a).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def _rows(kind, rows, n, rng):
    if kind == "llm":
        return synth.llm_logits(rows, n, seed=int(rng.integers(1, 1 << 30)))
    if kind == "grid":        # 513 levels, hundreds of elements on each
        return synth.grid_values(rows, n, seed=int(rng.integers(1, 1 << 30)))
    x = (rng.standard_normal((rows, n)) * 1.5).astype(np.float32)
    if kind == "bf16":        # what a bf16 head hands over: equal logits straddle the cut
        return np.ascontiguousarray((x.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32))
    if kind == "levels":      # 64 levels: massive ties
        return (np.round(x * 8) / 8).astype(np.float32)
    if kind == "sorted":
        x = np.sort(x, axis=1)
        x[1::2] = x[1::2, ::-1]
        return np.ascontiguousarray(x)
    if kind == "masked":      # a few allowed tokens per row, the rest -inf
        m = rng.random((rows, n)) < (40.0 / n)
        x[~m] = -np.inf
        x[0, :] = -np.inf
        x[0, min(5, n - 1)] = 1.0
        return x
    if kind == "constant":
        x[:] = np.float32(-2.5)
        x[1, n // 2:] = np.float32(3.0)
        return x
    if kind == "spikes":      # elements far above their wave's first vectors, and a dominant one
        x[:, n // 3] += 40.0
        x[2, 17::4099] += 25.0
        return x
    if kind == "tenth":       # one value everywhere, not a round one (its key has low bits set)
        x[:] = np.float32(0.1)
        x[rows - 1, :] = np.float32(-7.3)
        return x
    if kind == "two_values":
        return np.where(rng.random((rows, n)) < 0.5, np.float32(1.7), np.float32(1.7000002)).astype(np.float32)
    if kind == "sorted_desc":
        return np.ascontiguousarray(np.sort(x, axis=1)[:, ::-1])
    if kind == "flat_with_peaks":   # one value, and a few larger ones scattered over the row
        x[:] = np.float32(-0.3)
        for r in range(rows):
            at = rng.choice(n, size=min(n, 3 + 2 * r), replace=False)
            x[r, at] = np.float32(2.0) + rng.random(at.size).astype(np.float32)
        return x
    if kind == "runs":        # sorted inside runs of 4096: clustered, not sorted as a whole
        x = x.copy()
        for s0 in range(0, n, 4096):
            x[:, s0:s0 + 4096] = np.sort(x[:, s0:s0 + 4096], axis=1)
        return x
    if kind == "half_half":   # two values, either one in half of the places: the threshold's value is everywhere
        return np.where(rng.random((rows, n)) < 0.5, np.float32(1.0), np.float32(-1.0)).astype(np.float32)
    if kind == "three_allowed":   # three finite elements a row: the rest of the result is -inf, in index order
        x[:] = -np.inf
        x[:, [n // 7, n // 2, n - 3]] = np.float32(0.5)
        return x
    if kind == "nan_and_inf":  # rows of NaN probabilities (NaN ranks first in the plain top-k)
        x[0, n // 2] = np.nan
        x[1, n // 3] = np.inf
        x[2, 5] = np.nan
        x[2, n - 1] = np.nan
        return x
    if kind == "huge":        # differences of thousands: all but a few probabilities are 0 and tie
        return (x * np.float32(1e4)).astype(np.float32)
    if kind == "masked90":    # nine in ten -inf: block maxima of both signs (coarse histogram bins)
        x[rng.random((rows, n)) < 0.9] = -np.inf
        return x
    if kind == "coarse_levels":   # a dozen levels, thousands of elements on the one at the cut
        return (np.round(x) / 2).astype(np.float32)
    if kind == "signed_zeros":    # -0 == +0: one rank group, in index order
        x = np.where(rng.random((rows, n)) < 0.5, np.float32(0.0), np.float32(-0.0)).astype(np.float32)
        x[:, ::1000] = np.float32(1.0)
        return x
    raise ValueError(kind)


KINDS = ["llm", "bf16", "levels", "sorted", "masked", "constant", "spikes"]
TIE_KINDS = ["tenth", "two_values", "sorted_desc", "flat_with_peaks", "runs"]
WALK_KINDS = ["half_half", "three_allowed", "nan_and_inf", "huge", "masked90", "coarse_levels", "signed_zeros", "sorted", "runs",
              "flat_with_peaks"]


# a row of halves has half as many blocks as one of floats: too few for the pick kernel, or few enough for the large-k pair
OTHER_TYPE_ONLY = {(50257, 300, "float16"), (40000, 255, "float16"), (50257, 200, "float32")}


def _compare_paths(ops, n, k, dtype, rows, kinds, path):
    """The library's choice of kernels (which has to be `path`) against the kernels
    rows.path = 1 selects, and both against the oracle."""
    from vkop_amd import capi
    rng = np.random.default_rng(n * 31 + k)
    dt = capi.F32 if dtype == np.float32 else capi.F16
    capi.tune("rows.path", 0)
    if (n, k, np.dtype(dtype).name) in OTHER_TYPE_ONLY:
        pytest.skip("not a shape these kernels take in this element type")
    assert capi.measure_path(dt, (rows, n), -1, k) == path, (rows, n, k)
    for kind in kinds:
        x = np.ascontiguousarray(_rows(kind, rows, n, rng).astype(dtype))
        xd = dev(x)
        capi.tune("rows.path", 0)
        v, ix = ops.softmax_topk(xd, k)
        t, tj = ops.topk(xd, k)
        v, ix, t, tj = host(v), host(ix), host(t), host(tj)
        capi.tune("rows.path", 1)
        v1, ix1 = ops.softmax_topk(xd, k)
        t1, tj1 = ops.topk(xd, k)
        v1, ix1, t1, tj1 = host(v1), host(ix1), host(t1), host(tj1)
        capi.tune("rows.path", 0)
        bits = np.uint16 if dtype == np.float16 else np.uint32
        what = (kind, n, k, np.dtype(dtype).name)
        # plain top-k: no arithmetic, everything exact, both pairs and the oracle
        et, ej = oracle.topk(x, k)
        assert np.array_equal(tj, ej) and np.array_equal(t.view(bits), et.view(bits)), what
        assert np.array_equal(tj1, ej) and np.array_equal(t1.view(bits), et.view(bits)), what
        # fused: values within an ulp of the other pair's, to the bar against the oracle
        ov, oix, op = oracle.softmax_topk(x, k, return_probs=True)
        if dtype == np.float16:
            assert half_ulp_diff(v, v1).max() <= 1 and half_ulp_diff(v, ov).max() <= 1, what
        else:
            # (the bar is the distance to the oracle; the radix select behind rows.path = 1 at
            # large k sums accurate terms only, the scan sums fast ones: on rows of few distinct
            # values the two row sums may lie an ulp from the oracle's on either side)
            assert ulp_diff(v, ov).max() <= 2 and ulp_diff(v1, ov).max() <= 2 and ulp_diff(v, v1).max() <= 2, what
        differ = 0
        xf = x.astype(np.float32)
        for r in range(rows):
            vr = v[r].astype(np.float32)
            if not np.array_equal(ix[r], ix1[r]):
                differ += 1      # only where the two row sums round a tie open or closed
                assert not np.array_equal(v[r].view(bits), v1[r].view(bits)) or \
                    sorted(ix[r].tolist()) != sorted(ix1[r].tolist()), what
            if np.isfinite(vr).all():
                check_fused_invariants(xf[r], vr, ix[r])
            else:
                assert np.array_equal(ix[r], np.arange(k)), what       # all-NaN row: lowest indices
            if well_separated_cut(op[r].astype(np.float32), xf[r], k, 4 if dtype == np.float32 else 1 << 14):
                assert np.array_equal(ix[r], oix[r]), (what, r)
        assert differ <= 2, (what, differ)


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("n,k", [(128256, 50), (128256, 1), (128256, 255), (40000, 7), (16385, 20), (13057, 50),
                                 (262144, 64), (100003, 33), (500000, 100), (300000, 511), (50257, 300)])
def test_scan_pick_pair_equals_chunk_merge_and_oracle(ops, n, k, dtype):
    """(From k = 256 on the pair is the library's choice on more than 16 rows only, there also
    with fewer than two blocks per wanted place; of rows that one workgroup holds on more than 256.)"""
    _compare_paths(ops, n, k, dtype, 20 if k >= 256 else 260 if n <= 16384 else 6, KINDS, 2)


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("n,k", [(262144, 1024), (262144, 600), (524288, 2048), (200003, 700), (131072, 512),
                                 (300000, 1500), (200000, 300), (50257, 200), (100000, 400)])
def test_scan_with_spread_out_pick_for_large_k_equals_radix_select_and_oracle(ops, n, k, dtype):
    """k beyond one workgroup's candidate list (and, on a few rows, from k = 256 on, or from
    k = 160 where the row has too few blocks for the pick kernel): scan, then the gather and rank kernels
    that spread a row's candidates over many workgroups, against the multi-pass radix
    select (rows.path = 1) and the oracle -- the regular rows, and the ones the pair hands
    to its exact fallback (constant and masked rows, levels with thousands of equals)."""
    _compare_paths(ops, n, k, dtype, 4, KINDS + ["grid"], 3)


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("n,k", [(1000, 5), (1000, 16), (33, 5), (5, 5), (1024, 1), (2048, 7), (777, 10), (256, 3), (64, 16),
                                 (1001, 5), (130, 2), (1000, 32), (2048, 24), (1500, 20), (40, 32)])
def test_one_wave_kernel_for_short_rows_equals_chunk_kernel_and_oracle(ops, n, k, dtype):
    """Short rows, small k (a classifier head): the one-wave-per-row kernel against the
    chunk kernel (rows.path = 1) and the oracle, on regular rows and on the ones it hands
    to its exact fallback (ties en masse, masked rows, constant rows), and on rows whose
    probabilities underflow to 0 for all but a few elements (a tie at 0 that runs to the row's end)."""
    _compare_paths(ops, n, k, dtype, 6, KINDS + ["huge", "masked90"], 4)


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("n,k,path", [(128256, 50, 2), (40000, 255, 2), (262144, 200, 2), (1048576, 100, 2), (262144, 1024, 3), (300000, 600, 3), (131072, 800, 3), (1000, 5, 4),
                                      (2048, 16, 4), (2048, 32, 4)])
def test_rows_of_equal_and_clustered_values_on_every_route(ops, n, k, path, dtype):
    """Rows that defeat a threshold taken from block or lane maxima -- one value everywhere
    (with a key that is not a round number), two values a float apart, rows sorted
    downwards, a flat row with a few peaks, rows sorted in runs -- settled by each route's
    own means (a second threshold, the first elements equal to the tie value, block
    minima), against the other kernels and the oracle."""
    _compare_paths(ops, n, k, dtype, 4, TIE_KINDS, path)


@pytest.mark.parametrize("n,k", [(262144, 1024), (262144, 2000), (524288, 2048), (300000, 600), (300001, 700), (65536, 512),
                                 (100000, 1200)])
def test_large_k_rows_whose_cut_falls_into_a_crowd(ops, n, k):
    """The large-k kernels on rows where the threshold's own rank group is too large for the
    candidate lists (one value in half of the places, -inf nearly everywhere, probabilities
    that underflow to 0, -0 and +0, a dozen levels) -- its first members come from a walk over
    the row in index order, also on rows that do not start on 16 bytes -- on rows of NaN
    probabilities, on block maxima of both signs and on sorted rows at a k close to the
    lists' capacity, and on rows with hardly more blocks than wanted places (1.3 a place:
    most of the row is a candidate); against the radix select and the oracle."""
    _compare_paths(ops, n, k, np.float32, 4, WALK_KINDS, 3)


@pytest.mark.parametrize("rows,n,k", [(16, 131072, 1), (32, 50000, 3), (4, 262144, 1024), (8, 100000, 600), (64, 8192, 3),
                                      (256, 1000, 5), (7, 128255, 50)])
def test_rows_of_one_repeated_value_and_a_few_peaks(ops, rows, n, k):
    """One value everywhere but in three places: the row's sum is that value's term times its
    count, and the term is, by definition, the correctly rounded float exponential of the
    ROUNDED difference to the maximum -- off the exact exponential of the exact difference by up
    to 3e-7, the same for every copy.  A streaming pass that sums against a reference of its
    own has to say so exactly (the scan kernel records a wave of equal elements as a count and
    the value), or the probabilities drift by several ulp; every route, the plain softmax too."""
    rng = np.random.default_rng(rows + n + k)
    for rep in range(2):
        x = np.zeros((rows, n), np.float32) + (rng.standard_normal((rows, 1)) * 2).astype(np.float32)
        for r in range(rows):
            x[r, rng.choice(n, 3, replace=False)] = x[r, 0] + (rng.random(3) * 8 + 1).astype(np.float32)
        v, ix = ops.softmax_topk(dev(x), k)
        v, ix = host(v), host(ix)
        ov, oix = oracle.softmax_topk(x, k)
        assert ulp_diff(v, ov).max() <= 2, (rows, n, k, int(ulp_diff(v, ov).max()))
        assert np.array_equal(ix, oix), (rows, n, k)
        y = host(ops.softmax(dev(x)))
        assert ulp_diff(y, oracle.softmax(x)).max() <= 2, (rows, n, k)


@pytest.mark.parametrize("seed", [21, 22, 23])
def test_random_shapes_k_and_row_kinds_on_whatever_route_they_take(ops, seed):
    """A dozen draws a seed of (rows, n, k, element type, three kinds of rows) through the
    comparison of the library's own choice of kernels with the kernels rows.path = 1 selects and
    with the oracle: the shapes between the ones the other tests name (this is how the rows of
    one repeated value and three peaks, and a row that overflowed a wave's stage twice, were found).
    A flat row with dozens of peaks per thousand copies ([n = 20001, k = 16] under seed 23) measured
    3 ulp on every streaming route until their waves counted the copies of a value that fills them
    apart (a record word of its own: the scan kernel's, then the chunk kernel's): the kind
    "flat_with_peaks" is drawn like any other."""
    from vkop_amd import capi
    rng = np.random.default_rng(seed)
    kinds_all = list(dict.fromkeys(KINDS + TIE_KINDS + WALK_KINDS))
    ns = [33, 64, 100, 255, 256, 257, 777, 1000, 1024, 2047, 2048, 4096, 5000, 8191, 8192, 8400, 12000, 16384, 20001, 32768, 40000,
          50257, 65536, 100000, 128256, 200003]
    ks = [1, 2, 5, 8, 16, 31, 32, 33, 50, 64, 65, 100, 128, 159, 160, 200, 255, 256, 257, 300, 408, 409, 500, 511, 512, 600, 1024, 2000, 2048]
    for _ in range(12):
        n = int(rng.choice(ns))
        k = int(min(n, rng.choice(ks)))
        rows = int(rng.choice([3, 4, 5, 8, 16, 17, 24, 40])) if n <= 65536 else int(rng.choice([3, 4, 8, 16, 17, 20]))
        dtype = np.float32 if rng.random() < 0.6 else np.float16
        kinds = [str(t) for t in rng.choice(kinds_all, size=3, replace=False)]
        capi.tune("rows.path", 0)
        path = capi.measure_path(capi.F32 if dtype == np.float32 else capi.F16, (rows, n), -1, k)
        _compare_paths(ops, n, k, dtype, rows, kinds, path)


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("n,k", [(1040, 128), (2048, 129), (4095, 255), (4096, 256), (4097, 200), (8192, 300), (8193, 300), (12288, 408), (12289, 256),
                                 (16384, 409), (16385, 500), (32768, 511), (9000, 511), (2200, 511)])
def test_wide_workgroups_with_the_vectors_a_row_needs(ops, n, k, dtype):
    """A row in a workgroup of 512 or 1024 threads, at and just past what each number of vectors a thread holds, and as
    many places as its list takes: plain top-k exactly, in either direction; the fused call to the bars."""
    rng = np.random.default_rng(n + k)
    bits = np.uint16 if dtype == np.float16 else np.uint32
    for kind in ("llm", "levels", "sorted", "runs", "masked", "nan_and_inf", "signed_zeros", "tenth", "half_half"):
        x = np.ascontiguousarray(_rows(kind, 17, n, rng).astype(dtype))
        xd = dev(x)
        for largest in (True, False):
            t, tj = ops.topk(xd, k, largest=largest)
            et, ej = oracle.topk(x, k, largest=largest)
            assert np.array_equal(host(tj), ej) and np.array_equal(host(t).view(bits), et.view(bits)), (kind, largest)
        v, ix = (host(t) for t in ops.softmax_topk(xd, k))
        ov, oix = oracle.softmax_topk(x, k)
        assert (half_ulp_diff if dtype == np.float16 else ulp_diff)(v, ov).max() <= (1 if dtype == np.float16 else 2), kind
        xf, op = x.astype(np.float32), oracle.softmax(x).astype(np.float32)
        for r in range(17):
            if np.isfinite(v[r]).all():
                check_fused_invariants(xf[r], v[r].astype(np.float32), ix[r])
            else:
                assert np.array_equal(ix[r], np.arange(k)), (kind, r)  # all-NaN row: lowest indices
            if well_separated_cut(op[r], xf[r], k, 4 if dtype == np.float32 else 1 << 14):
                assert np.array_equal(ix[r], oix[r]), (kind, r)


@pytest.mark.parametrize("rows,n,k", [(17, 20001, 16), (8, 20001, 16), (24, 50000, 40), (5, 131072, 64), (16, 16385, 5)])
def test_flat_rows_with_dozens_of_peaks_on_the_chunk_and_merge_kernels(ops, rows, n, k):
    """The chunk + merge kernels over several chunks (rows.path = 1: no shape takes them by itself any
    more) on rows that are one value and dozens of peaks: most waves hold a larger element beside the
    copies, all of them sum against references of their own, and the copies' common term error came to
    3 ulp of the probabilities (n = 20001, k = 16) until the chunk kernel's waves counted the copies
    apart, in a record word of their own, for the merge to add them as the sum is defined."""
    from vkop_amd import capi
    rng = np.random.default_rng(rows * 1000 + k)
    x = np.full((rows, n), np.float32(-0.3))
    for r in range(rows):
        at = rng.choice(n, size=20 + 13 * r, replace=False)
        x[r, at] = np.float32(2.0) + rng.random(at.size).astype(np.float32)
    ov, oix = oracle.softmax_topk(x, k)
    try:
        capi.tune("rows.path", 1)
        assert capi.measure_path(capi.F32, (rows, n), -1, k) == 1 and capi.rows_plan(capi.F32, (rows, n), -1, k)[2] > 1
        v, ix = ops.softmax_topk(dev(x), k)
        v, ix = host(v), host(ix)
    finally:
        capi.tune("rows.path", 0)
    assert np.array_equal(ix, oix), (rows, n, k)
    assert ulp_diff(v, ov).max() <= 2, (rows, n, k, int(ulp_diff(v, ov).max()))
    v0, ix0 = ops.softmax_topk(dev(x), k)
    assert np.array_equal(host(ix0), oix) and ulp_diff(host(v0), ov).max() <= 2, (rows, n, k)


@pytest.mark.parametrize("n", [16388, 40002, 128255])
def test_scan_pick_pair_on_rows_that_do_not_start_on_16_bytes(ops, n):
    """n not a multiple of the vector width (rows after the first are unaligned), and a
    tensor that starts two elements into an allocation: the element-wise load variants."""
    rng = np.random.default_rng(n)
    for dtype in (np.float32, np.float16):
        x = np.ascontiguousarray((rng.standard_normal((5, n)) * 2).astype(dtype))
        x[3, ::5] = x[3, 1]
        big = torch.empty(5 * n + 8, dtype=torch.float32 if dtype == np.float32 else torch.float16, device="cuda")
        xd = big[2:2 + 5 * n].view(5, n)
        xd.copy_(dev(x))
        for k in (5, 60):
            v, ix = ops.softmax_topk(xd, k)
            t, tj = ops.topk(xd, k)
            v, ix, t, tj = host(v), host(ix), host(t), host(tj)
            et, ej = oracle.topk(x, k)
            bits = np.uint16 if dtype == np.float16 else np.uint32
            assert np.array_equal(tj, ej) and np.array_equal(t.view(bits), et.view(bits)), (n, k)
            ov, oix, op = oracle.softmax_topk(x, k, return_probs=True)
            if dtype == np.float16:
                assert half_ulp_diff(v, ov).max() <= 1
            else:
                assert ulp_diff(v, ov).max() <= 2
            for r in range(5):
                check_fused_invariants(x[r].astype(np.float32), v[r].astype(np.float32), ix[r])
                if well_separated_cut(op[r].astype(np.float32), x[r].astype(np.float32), k, 4 if dtype == np.float32 else 1 << 14):
                    assert np.array_equal(ix[r], oix[r]), (n, k, r)


def test_plain_topk_nan_ranks_first_through_the_scan_pick_pair(ops):
    rng = np.random.default_rng(3)
    x = rng.standard_normal((4, 70000)).astype(np.float32)
    x[0, [5, 69999, 30000]] = np.nan
    x[1, ::3] = np.nan                       # more NaN than k
    x[2, 1000] = np.inf
    x[2, 2000] = -np.inf
    x[3, :] = np.nan
    for k in (1, 4, 100):
        t, tj = ops.topk(dev(x), k)
        et, ej = oracle.topk(x, k)
        assert np.array_equal(host(tj), ej) and np.array_equal(host(t).view(np.uint32), et.view(np.uint32)), k


# ------------------------------------------------------------ sampling variant --

@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("shape,k", [((16, 128256), 50), ((3, 40000), 7), ((256, 1000), 5), ((2, 33), 33), ((5, 2, 4097), 9),
                                     ((64, 8192), 40), ((16, 8400), 300), ((40, 4096), 64), ((300, 257), 8), ((7, 20000), 100),
                                     ((4, 262144), 1024)])
def test_sampling_variant_against_the_oracle(ops, shape, k, dtype):
    rng = np.random.default_rng(shape[-1] + k)
    x = synth.llm_logits(int(np.prod(shape[:-1])), shape[-1], seed=shape[-1], temperature=1.0).reshape(shape)
    x = np.ascontiguousarray(x.astype(dtype))
    bits = np.uint16 if dtype == np.float16 else np.uint32
    for scale, top_p in ((1.25, 0.9), (1.0, 0.5), (0.5, 0.999), (3.0, 0.2)):
        v, ix, c = ops.softmax_topk_sampling(dev(x), k, scale, top_p)
        v, ix, c = host(v), host(ix), host(c)
        ov, oix, oc = oracle.softmax_topk_sampling(x, k, scale, top_p)
        what = (shape, k, scale, top_p)
        if dtype == np.float16:
            assert half_ulp_diff(v, ov).max() <= 1, what
        else:
            assert ulp_diff(v, ov).max() <= 2, what
        # the count is a function of the stored values: exact against the pinned CPU rule on them,
        # and equal to the separate entry point's
        vf = v.astype(np.float32).reshape(-1, k)
        assert np.array_equal(c.reshape(-1), oracle.topp_count(vf, top_p)), what
        same_values = np.array_equal(v.view(bits), ov.view(bits))
        if same_values:
            assert np.array_equal(c, oc), what
        # bit for bit the plain entry point on a tensor scaled on the host (one float32 product per element)
        xs = (x.astype(np.float32) * np.float32(scale)).astype(np.float32)
        # (bit for bit where both run the scan + pick kernels; other shapes take the line kernels here and the
        # one-workgroup streaming kernels there, which add up the row in different orders: both within the 2-ulp bar of the oracle)
        if dtype == np.float32:
            from vkop_amd import capi
            pv, pix = ops.softmax_topk(dev(xs), k)
            pv, pix = host(pv), host(pix)
            if capi.measure_path(capi.F32, shape, -1, k) == 2:
                assert np.array_equal(pix, ix) and np.array_equal(pv.view(np.uint32), v.view(np.uint32)), what
            else:
                assert ulp_diff(pv, v).max() <= 2, what
        xf = (x.astype(np.float32) * np.float32(scale)).reshape(-1, shape[-1])
        op = oracle.softmax(xf)
        for r in range(xf.shape[0]):
            check_fused_invariants(xf[r], vf[r], ix.reshape(-1, k)[r])
            if dtype == np.float32 and well_separated_cut(op[r], xf[r], k):
                assert np.array_equal(ix.reshape(-1, k)[r], oix.reshape(-1, k)[r]), (what, r)


@pytest.mark.parametrize("k", [1, 5, 20, 31, 32, 40, 63, 64, 100, 150, 200, 255])
@pytest.mark.parametrize("n", [50257, 131072])
def test_sampling_half_rows_whose_probabilities_tie(ops, n, k):
    """Long half rows under a temperature: the probabilities near the k-th place are subnormal halves, and elements
    of different logits share one.  They are in order of index, whether the candidates at hand settle the group at
    the k-th place or the row has to be read again: rows spread out, of a coarse grid, and ones whose tail all
    rounds to the smallest half or to nothing."""
    rng = np.random.default_rng(n + k)
    x = rng.standard_normal((12, n)).astype(np.float32)
    x[np.arange(12), rng.integers(0, n, 12)] += np.linspace(3, 16, 12, dtype=np.float32)
    x[4:7] = np.round(x[4:7] * 16) / 16
    x[7, rng.integers(0, n, 4 * k)] += np.float32(2.0)
    x = np.ascontiguousarray((x * np.float32(1.25)).astype(np.float16))
    for scale, top_p in ((1.25, 0.9), (1.0, 0.5), (0.75, 0.95)):
        v, ix, c = (host(t) for t in ops.softmax_topk_sampling(dev(x), k, scale, top_p))
        ov, oix, oc = oracle.softmax_topk_sampling(x, k, scale, top_p)
        # Sums agree to 2^-22, so a probability that close to the boundary between two normal halves, 2^-11 apart, may
        # fall on either side of it: one in 2^-10 of the values, a unit each, and where it joins or leaves the group at the
        # k-th place the row's indices move with it.
        assert half_ulp_diff(v, ov).max() <= 1 and (v.view(np.uint16) != ov.view(np.uint16)).sum() <= max(2, v.size >> 9)
        assert ((ix == oix).all(axis=-1) | (v.view(np.uint16) != ov.view(np.uint16)).any(axis=-1)).sum() >= 11, (n, k, scale)
        assert np.array_equal(c, oracle.topp_count(v.astype(np.float32), top_p))
        # equal probabilities in order of index, in every row
        equal = v[:, 1:] == v[:, :-1]
        assert np.all(ix[:, 1:][equal] > ix[:, :-1][equal])


@pytest.mark.parametrize("k", [4, 40, 120])
def test_half_rows_whose_cut_is_a_few_of_the_smallest_half(ops, k):
    """Rows whose k-th probability is 1 to 60 of the smallest half, so that its group spans a logit or a sixtieth of one, far below
    the first k: the list goes on as far as the group can, or the row is looked at again."""
    rng = np.random.default_rng(k)
    rows, n = 48, 50257
    x = rng.standard_normal((rows, n)).astype(np.float32) * np.float32(1.25)
    cut = np.sort(x, axis=-1)[:, -k]
    units = np.exp(np.linspace(np.log(0.8), np.log(60.0), rows))
    x[np.arange(rows), rng.integers(0, n, rows)] = cut + np.log(2.0 ** 24 / units).astype(np.float32)
    x = x.astype(np.float16)
    v, ix = (host(t) for t in ops.softmax_topk(dev(x), k))
    ov, oix = oracle.softmax_topk(x, k)
    # (sums agree to 2^-22: a probability that close to a boundary between two halves may fall on either side of it)
    same = (v.view(np.uint16) == ov.view(np.uint16)).all(axis=-1)
    assert half_ulp_diff(v, ov).max() <= 1 and same.sum() >= rows - 2 and np.array_equal(ix[same], oix[same])
    equal = v[:, 1:] == v[:, :-1]
    assert np.all(ix[:, 1:][equal] > ix[:, :-1][equal])


@pytest.mark.parametrize("k", [3, 20, 40, 90])
def test_half_rows_with_a_tie_at_the_cut_where_the_list_may_end(ops, k):
    """k + 5 elements above the rest, t + 1 neighbouring ones of them around the k-th place a last place of their logits apart, whose
    probabilities are equal halves: the list of candidates may end with that group, and whether it holds all of it is
    decided by the largest probability that is not listed -- of the group's own value in every other row, where an
    element a few last places below goes on with it."""
    rng = np.random.default_rng(k)
    n, rows, scale = 32000, 64, 1.25
    x = (rng.standard_normal((rows, n)) * 0.5).astype(np.float16)
    for r in range(rows):
        where = rng.permutation(n)[:k + 5]
        x[r, where] = np.linspace(5.0, 4.0, k + 5).astype(np.float16)
        x[r, where[0]] = 8.0 + rng.random() * 6.0   # the row's maximum: the others' probabilities are small halves
        t = int(rng.integers(1, 5))
        first = k - 1 - int(rng.integers(0, min(t, k - 1)))
        group = where[first:first + t + 1]
        top = x[r, group[0]]
        x[r, group] = top - np.spacing(top) * rng.integers(0, 2, len(group)).astype(np.float16)
        if r % 2:
            x[r, where[-1]] = top - np.spacing(top) * np.float16(3)
    v, ix, _ = (host(a) for a in ops.softmax_topk_sampling(dev(x), k, scale, 0.9))
    ov, oix, _ = oracle.softmax_topk_sampling(x, k, scale, 0.9)
    # sums agree to 2^-22: a probability that close to a boundary between two halves may fall on either side of it
    assert half_ulp_diff(v, ov).max() <= 1
    same = (v.view(np.uint16) == ov.view(np.uint16)).all(axis=-1)
    assert same.sum() >= rows - 2 and np.array_equal(ix[same], oix[same])
    equal = v[:, 1:] == v[:, :-1]
    assert np.all(ix[:, 1:][equal] > ix[:, :-1][equal])


@pytest.mark.parametrize("k", [3, 40, 90])
def test_float_rows_with_equal_logits_at_the_cut(ops, k):
    """k + 4 equal logits around the k-th place, where the list of candidates may end; in two rows of three a logit one float below
    with a lower index, whose difference to the row's maximum rounds to the same float (a maximum 8 above and more) or does not
    (the others).  Maxima 2 to 100 above the group (the last: subnormal probabilities), groups at 5, -3, 0, 300 and 1e-3."""
    rng = np.random.default_rng(k)
    n, rows = 40000, 60
    x = np.empty((rows, n), np.float32)
    for r in range(rows):
        v = np.float32((5.0, -3.0, 0.0, 300.0, 1e-3)[r % 5])
        x[r] = v - 1 - np.abs(rng.standard_normal(n)).astype(np.float32)
        where = np.sort(rng.permutation(n)[:k + 6])
        x[r, where[1:k + 5]] = v
        x[r, where[-1]] = v + np.float32((2.0, 8.5, 17.0, 40.0, 89.0, 100.0)[r // 5 % 6])
        if r % 3:
            x[r, where[0]] = np.nextafter(v, np.float32(-np.inf))
        if r % 3 == 2:
            x[r, where[2]] = np.nextafter(np.nextafter(v, np.float32(-np.inf)), np.float32(-np.inf))
    v, ix = (host(t) for t in ops.softmax_topk(dev(x), k))
    ev, eix = oracle.softmax_topk(x, k)
    assert np.array_equal(ix, eix) and ulp_diff(v, ev).max() <= 2


@pytest.mark.parametrize("spread", [2.0 ** -i for i in (3, 4, 5, 6, 9, 12, 13, 14, 15, 18, 21)])
@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
def test_rows_of_small_range_whose_list_goes_on_below_its_threshold(ops, spread, dtype):
    """Rows so narrow that the stretch below the threshold (0.01 of halves, 2^-13 of a float threshold) holds dozens, hundreds or
    all of their elements, with and without a peak."""
    rng = np.random.default_rng(int(1 / spread))
    x = (rng.standard_normal((9, 50257)) * spread).astype(np.float32)
    x[3:6] += np.float32(0.75)
    x[0::3, 77] = 6.0
    x = x.astype(dtype)
    for k in (5, 40, 100):
        v, ix = (host(t) for t in ops.softmax_topk(dev(x), k))
        ev, eix = oracle.softmax_topk(x, k)
        if dtype == np.float32:
            assert ulp_diff(v, ev).max() <= 2, k
        else:
            assert half_ulp_diff(v, ev).max() <= 1, k
        bits = np.uint32 if dtype == np.float32 else np.uint16
        for r in range(9):
            check_fused_invariants(x[r].astype(np.float32), v[r].astype(np.float32), ix[r])
            # the sums agree to 2^-22: where no probability fell on the other side of a boundary, neither did an index
            if np.array_equal(v[r].view(bits), ev[r].view(bits)) and (dtype == np.float16 or spread > 1e-3):
                assert np.array_equal(ix[r], eix[r]), (k, r)


def test_a_tie_at_the_cut_costs_no_second_look(ops):
    """[64,128256] k = 50 with 70 logits of 5 behind the maximum of every row: where that is 13 the next float below 5 has the same
    difference to it, rounded, where it is 13.3 it has not, and the one takes the time of the other (a row that starts over takes
    6 us of 14 longer).  The least of nine means of 40 calls each, the two in turn."""
    rng = np.random.default_rng(9)
    rows, n, k = 64, 128256, 50
    x = np.minimum(rng.standard_normal((rows, n)).astype(np.float32), np.float32(3.0))
    where = np.stack([rng.permutation(n)[:71] for _ in range(rows)])
    np.put_along_axis(x, where, np.float32(5.0), -1)
    inputs = {}
    for top in (13.0, 13.3):
        x[np.arange(rows), where[:, 0]] = top
        inputs[top] = dev(x)
        assert np.array_equal(host(ops.softmax_topk(inputs[top], k)[1]), oracle.softmax_topk(x, k)[1])
    best = dict.fromkeys(inputs, 1e9)
    for _ in range(9):
        for top, t in inputs.items():
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            ops.softmax_topk(t, k)
            a.record()
            for _ in range(40):
                ops.softmax_topk(t, k)
            b.record()
            torch.cuda.synchronize()
            best[top] = min(best[top], a.elapsed_time(b) / 40)
    assert best[13.0] < 1.2 * best[13.3], best


def test_a_row_of_small_range_costs_no_longer_list(ops):
    """[32,50257] k = 40 of rows spread by 2e-5 against rows spread by 0.3 (listed to 2^-16 below the threshold, where most of such a
    row lies, they took 2.1 times as long; 1.1 times to 2^-13 of it).  These rows have no more than 128 elements at their
    thresholds, past which the ranking takes longer.  The least of nine means of 40 calls each, the two in turn."""
    x = np.random.default_rng(6).standard_normal((32, 50257)).astype(np.float32)
    inputs = {spread: dev(x * np.float32(spread)) for spread in (0.3, 2e-5)}
    best = dict.fromkeys(inputs, 1e9)
    for _ in range(9):
        for spread, t in inputs.items():
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            ops.softmax_topk(t, 40)
            a.record()
            for _ in range(40):
                ops.softmax_topk(t, 40)
            b.record()
            torch.cuda.synchronize()
            best[spread] = min(best[spread], a.elapsed_time(b) / 40)
    assert best[2e-5] < 1.5 * best[0.3], best


@pytest.mark.parametrize("n", [50000, 8192, 1000, 8400])
def test_sampling_variant_ties_special_rows_and_errors(ops, n):
    """(n = 50000: the scan + pick kernels; the shorter rows: one workgroup, or one wave, per row)"""
    from vkop_amd import capi
    rng = np.random.default_rng(9)
    x = (np.round(rng.standard_normal((6, n)) * 4) / 4).astype(np.float32)   # ties across the cut
    x[1, 10:] = -np.inf                     # fewer elements above -inf than k
    x[2, 77] = np.nan                       # an all-NaN result
    x[3] = 1.5                              # a constant row
    k = 40
    v, ix, c = ops.softmax_topk_sampling(dev(x), k, 0.75, 0.8)
    v, ix, c = host(v), host(ix), host(c)
    with np.errstate(invalid="ignore"):
        ov, oix, oc = oracle.softmax_topk_sampling(x, k, 0.75, 0.8)
    assert np.array_equal(np.isnan(v), np.isnan(ov))
    assert ulp_diff(v, ov).max() <= 2
    assert np.array_equal(ix[2], np.arange(k)) and c[2] == k
    assert np.array_equal(ix[3], np.arange(k)) and np.array_equal(ix[1][:10], oix[1][:10])
    ok = ~np.isnan(v).any(axis=1)
    assert np.array_equal(c[ok], oracle.topp_count(v[ok], 0.8))
    xs = (x * np.float32(0.75)).astype(np.float32)
    for r in np.nonzero(ok)[0]:
        check_fused_invariants(xs[r], v[r], ix[r])
    xd = dev(x)
    out = torch.empty((6, k), dtype=torch.float32, device="cuda")
    oi = torch.empty((6, k), dtype=torch.int32, device="cuda")
    ws = torch.zeros(1 << 22, dtype=torch.uint8, device="cuda")
    ptr = (ws.data_ptr() + 255) // 256 * 256
    for bad in (0.0, -1.0, float("inf"), float("nan")):
        with pytest.raises(capi.VkopHipError) as e:
            capi.softmax_topk_sampling(xd.data_ptr(), out.data_ptr(), oi.data_ptr(), 0, capi.F32, x.shape, -1, k, bad, 0.5, ptr,
                                       1 << 21, 0)
        assert e.value.code == capi.ERR_INVALID
    with pytest.raises(capi.VkopHipError) as e:   # the count along an axis that is not the last
        capi.softmax_topk_sampling(xd.data_ptr(), out.data_ptr(), oi.data_ptr(), oi.data_ptr(), capi.F32, x.shape, 0, 3, 1.0, 0.5,
                                   ptr, 1 << 21, 0)
    assert e.value.code == capi.ERR_UNSUPPORTED


# ------------------------------------------ softmax: NaN option on the other axes --

@pytest.mark.parametrize("shape,axis", [((130, 70), 0), ((5, 130, 70), 1), ((2, 3, 40, 9), 2), ((80, 8400), 0), ((3, 4, 5, 6), 0),
                                        ((4, 3000, 3), 1)])
def test_nan_replacement_on_axes_other_than_the_last(ops, shape, axis):
    """shaders/softmax2.comp:177-181 implements the option for axis 0 of a matrix; here every axis."""
    rng = np.random.default_rng(sum(shape) + axis)
    for dtype in (np.float32, np.float16):
        x = rng.standard_normal(shape).astype(np.float32)
        idx = tuple(rng.integers(0, s, size=6) for s in shape)
        x[idx] = np.nan                                     # lines holding a NaN: all of the line's outputs are NaN
        line = [0] * len(shape)
        line[axis] = slice(None)
        x[tuple(line)] = -np.inf                            # a line of -inf: NaN too
        x = np.ascontiguousarray(x.astype(dtype))
        with np.errstate(invalid="ignore"):
            exp = oracle.softmax(x, axis)
            expn = oracle.softmax(x, axis, nan_where=1, nan_value=0.25)
        assert np.isnan(exp.astype(np.float32)).any()
        got = host(ops.softmax(dev(x), axis))
        gotn = host(ops.softmax(dev(x), axis, nan_where=True, nan_value=0.25))
        assert np.array_equal(np.isnan(got.astype(np.float32)), np.isnan(exp.astype(np.float32)))
        assert not np.isnan(gotn.astype(np.float32)).any()
        assert np.array_equal(gotn.astype(np.float32) == 0.25, (expn.astype(np.float32) == 0.25))
        if dtype == np.float16:
            assert half_ulp_diff(gotn, expn).max() <= 1
        else:
            assert ulp_diff(gotn, expn).max() <= 2


# ------------------------------------------------------------ the benchmark's timeline leg --

def test_bench_timeline_leg_sees_every_lane(ops):
    """bench.py --timeline (a child process on libvkop_hip_timeline.so, whose scan and pick kernels log their own
    device timestamps): the summary names as many lanes as calls were in flight, and its per-call time from the
    log agrees with the HIP-event figure of the same pass."""
    import json
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    if not os.path.exists(os.path.join(root, "vkop_amd", "libvkop_hip_timeline.so")):
        pytest.skip("libvkop_hip_timeline.so is not built (make -C vkop_amd/csrc timeline)")
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--timeline", "--hw-queues", "8", "--inflight", "3",
                        "--steps", "120", "--warmup", "12"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-500:]
    out = json.loads([line for line in r.stdout.splitlines() if line.startswith("{")][-1])
    assert out.get("lanes_seen") == 3, out
    assert 0.7 < out["us_per_call_from_the_log"] / out["us_per_step_by_hip_events_same_run"] < 1.3, out
    assert 1.0 < out["mean_kernels_running"] <= 3.2, out


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("rows,n,k", [(5, 3, 2), (5, 7, 3), (5, 9, 4), (4, 1001, 5), (4, 1003, 40), (3, 1462, 225), (3, 4097, 64), (3, 8195, 64),
                                      (3, 8201, 100), (20, 20003, 50), (2, 50257, 200), (3, 131075, 50), (2, 100001, 600),
                                      (2, 131077, 1100), (2, 29467, 886)])
def test_rows_that_start_off_sixteen_bytes(ops, rows, n, k, dtype):
    """Every selection route (one wave, one workgroup, scan + pick, scan + gather + rank, the radix select) on rows
    of odd length in a tensor that itself starts one element off 16 bytes, the row's largest and smallest elements
    in its last and first vectors -- loaded 16 bytes at a time, the last vector moved back into the row."""
    rng = np.random.default_rng(rows * n + k)
    x = rng.standard_normal((rows, n)).astype(dtype)
    m = min(n // 3, 11)
    for r in range(rows):
        ends = np.concatenate([np.arange(m), n - 1 - np.arange(m)])
        x[r, ends] += np.where(rng.random(ends.size) < 0.5, -5, 5).astype(dtype)
    buf = torch.empty(rows * n + 1, dtype=torch.float16 if dtype == np.float16 else torch.float32, device="cuda")
    view = buf[1:].view(rows, n)
    view.copy_(dev(x))
    bits = np.uint16 if dtype == np.float16 else np.uint32
    for largest in (True, False):
        v, ix = ops.topk(view, k, largest=largest)
        ev, eix = oracle.topk(x, k, -1, largest)
        assert np.array_equal(host(ix), eix) and np.array_equal(host(v).view(bits), ev.view(bits)), largest
    for scale, top_p in ((1.0, None), (1.25, 0.9)):
        # the aligned copy of the same rows takes the same kernels' other form: the same bits from either
        got, want = ((ops.softmax_topk(t, k) if top_p is None else ops.softmax_topk_sampling(t, k, scale, top_p))
                     for t in (view, dev(x)))
        for g, w in zip(got, want):
            assert np.array_equal(host(g), host(w)), (scale, top_p)


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("n,k", [(4096, 64), (8400, 300), (8401, 300), (32000, 40), (50257, 200), (100000, 600), (131076, 1025)])
def test_smallest_first_on_reversed_elements(ops, n, k, dtype):
    """k smallest on long rows: the kernels of the other direction on reversed elements.  NaN (largest: last, behind
    +inf) and +inf -- the reversed -inf that never becomes a candidate -- alone and side by side, where they fill the
    last places and where they do not; zeros of both signs; rows of one value, of levels, in order."""
    rng = np.random.default_rng(n + k)
    x = rng.standard_normal((12, n)).astype(dtype)
    x[1, rng.random(n) < 0.3] = np.nan
    x[2, rng.random(n) < 0.9] = np.inf
    few = rng.choice(n, k // 2, replace=False)
    x[3, :], x[3, few] = np.inf, -1.5
    x[4, :], x[4, few] = np.nan, rng.standard_normal(few.size)
    x[5, 0::2], x[5, 1::2], x[5, few] = np.nan, np.inf, 2.0          # both kinds behind the candidates, mixed
    x[6, :], x[6, few[: k // 4]] = np.nan, np.inf                    # fewer +inf than places, then NaN
    x[7, :] = np.where(rng.random(n) < 0.5, dtype(0.0), dtype(-0.0))
    x[8, :] = 0.75
    x[9, :] = np.round(x[9].astype(np.float32) * 4) / 4
    x[10, :] = np.sort(x[10])[::-1]
    x[11, rng.choice(n, 5, replace=False)] = -np.inf
    for rows in (x, np.tile(x, (2, 1))):                               # up to 16 rows, and more: other routes
        v, ix = ops.topk(dev(rows), k, largest=False)
        ev, eix = oracle.topk(rows, k, -1, False)
        for r in range(rows.shape[0]):
            assert np.array_equal(host(ix[r]), eix[r]), r
        bits = np.uint16 if dtype == np.float16 else np.uint32
        assert np.array_equal(host(v).view(bits), ev.view(bits))


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("rows,n,k", [(1023, 400, 44), (1024, 400, 57), (4096, 801, 75), (256, 1000, 150), (257, 1000, 150), (300, 1500, 219),
                                      (300, 1505, 219), (257, 1576, 393), (300, 1577, 394), (300, 1681, 394), (256, 2400, 271), (257, 2400, 271), (5, 1500, 393), (9, 999, 249), (9, 1031, 249), (9, 1383, 345), (1025, 8196, 23)])
def test_rows_of_one_workgroup_or_of_an_exact_select(ops, rows, n, k, dtype):
    """Rows on either side of the line between the one-workgroup kernel and the exact select, both directions, spread out and
    with values equal en masse; and the fused call, whose line lies elsewhere."""
    rng = np.random.default_rng(rows + n + k)
    bits = np.uint16 if dtype == np.float16 else np.uint32
    for step in (0, 0.25):
        x = rng.standard_normal((rows, n)).astype(np.float32)
        if step:
            x = np.round(x / np.float32(step)) * np.float32(step)
        x = x.astype(dtype)
        x[1, n // 2] = np.nan
        for largest in (True, False):
            v, ix = ops.topk(dev(x), k, largest=largest)
            ev, eix = oracle.topk(x, k, largest=largest)
            assert np.array_equal(host(ix), eix) and np.array_equal(host(v).view(bits), ev.view(bits)), (step, largest)
        x[1, n // 2] = 0.5
        v, ix = ops.softmax_topk(dev(x), k)
        v, ix = host(v), host(ix)
        ev, eix, ep = oracle.softmax_topk(x, k, return_probs=True)
        assert (half_ulp_diff(v, ev).max() <= 1) if dtype == np.float16 else (ulp_diff(v, ev).max() <= 2), step
        for r in range(0, rows, 37):
            check_fused_invariants(x[r].astype(np.float32), v[r].astype(np.float32), ix[r])
            if well_separated_cut(ep[r].astype(np.float32), x[r].astype(np.float32), k, 4 if dtype == np.float32 else 1 << 14):
                assert np.array_equal(ix[r], eix[r]), (step, r)


@pytest.mark.parametrize("n,k", [(1000, 5), (4096, 64), (8400, 300), (8401, 300), (32000, 40), (50257, 200), (100000, 600), (131076, 1025)])
def test_signalling_nan_ranks_as_nan(ops, n, k):
    """A NaN is a NaN whether it is quiet or signalling: last among the smallest, first among the largest, of either sign,
    alone, among +inf, and where NaN fills the last places; values are copies of the input's bits."""
    rng = np.random.default_rng(n + k)
    x = rng.standard_normal((20, n)).astype(np.float32)
    bits = x.view(np.uint32)
    kinds = np.array([0x7F800001, 0xFF800001, 0x7FBFFFFF, 0xFFBFFFFF, 0x7FC00000], np.uint32)
    bits[0, n // 2] = kinds[0]
    bits[1, 0], bits[1, n - 1] = kinds[0], kinds[1]
    at = rng.random(n) < 0.3
    bits[2, at] = rng.choice(kinds, at.sum())
    few = rng.choice(n, k // 2, replace=False)
    bits[3, :], x[3, few] = kinds[1], -1.5
    bits[4, :] = rng.choice(kinds, n)
    x[5, :], bits[5, 0::2], x[5, few] = np.inf, kinds[0], 2.0
    for largest in (False, True):
        for rows in (x[:12], x):
            v, ix = ops.topk(dev(rows), k, largest=largest)
            ev, eix = oracle.topk(rows, k, -1, largest)
            for r in range(rows.shape[0]):
                assert np.array_equal(host(ix[r]), eix[r]), (largest, r)
            assert np.array_equal(host(v).view(np.uint32), ev.view(np.uint32)), largest


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("rows,n,k", [(9, 4096, 64), (9, 4001, 64), (20, 8192, 100), (16, 8400, 300), (9, 1100, 100)])
def test_rows_of_few_values_whose_keys_end_in_ones(ops, rows, n, k, dtype):
    """One workgroup a row, rows of one value, two or a dozen: the bound from the lane maxima holds the leading 16 bits of a
    key, the low bits of which are ones for -0.75 and anything for 0.1, and is raised to the value itself where fewer than k+1
    lanes exceed it.  k - 1, k, k + 1 elements above the value, -inf beside it, and -inf alone; both directions and fused."""
    rng = np.random.default_rng(n + k)
    x = np.empty((rows, n), np.float32)
    for r in range(rows):
        v = (-0.75, 0.1, -0.1, 0.75, -3.3e-5, 1e4, -1e4)[r % 7]
        x[r] = v
        if r % 9 == 7:
            x[r, rng.permutation(n)[:n // 2]] = -np.inf
        if r % 9 == 8:
            x[r] = (np.round(rng.standard_normal(n) * 2) / 2 * 0.1)
        if r % 3 == 1:
            at = rng.choice(n, k + r % 5 - 1, replace=False)
            x[r, at] = v + np.abs(v) * (1 + rng.random(at.size))
        if r % 3 == 2:
            at = rng.choice(n, k + r % 4 - 1, replace=False)
            x[r, at] = v - np.abs(v) * (1 + rng.random(at.size))
    x[rows - 1] = -np.inf
    x[rows - 1, :k // 2] = 0.1
    x = x.astype(dtype)
    bits = np.uint16 if dtype == np.float16 else np.uint32
    for largest in (True, False):
        v, ix = ops.topk(dev(x), k, largest=largest)
        ev, eix = oracle.topk(x, k, -1, largest)
        assert np.array_equal(host(ix), eix) and np.array_equal(host(v).view(bits), ev.view(bits)), largest
    v, ix = (host(t) for t in ops.softmax_topk(dev(x), k))
    ev, eix = oracle.softmax_topk(x, k)
    assert np.array_equal(ix, eix)
    assert (half_ulp_diff(v, ev) if dtype == np.float16 else ulp_diff(v, ev)).max() <= (1 if dtype == np.float16 else 2)


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("n,k", [(33000, 5), (128256, 50), (131073, 40), (300001, 60), (1000003, 200)])
def test_rows_whose_cut_is_a_value_of_many_blocks(ops, dtype, n, k):
    """One value in every sixth block or so, with none, some and k elements above it, in the row's first and last element and in
    neighbours: more blocks reach it than are read again, and its first members come from the blocks in index order."""
    rng = np.random.default_rng(n + k)
    x = np.minimum(rng.standard_normal((5, n)).astype(np.float32), np.float32(3.0))
    for r in range(5):
        x[r, rng.choice(n, max(n // 400, 8 * (k + 1)), replace=False)] = 5.0
        if r:
            x[r, rng.choice(n, (k // 2, k - 1, k, 1)[r - 1], replace=False)] = 5.0 + rng.random((k // 2, k - 1, k, 1)[r - 1]).astype(np.float32)
    x[:, -1] = 5.0
    x[1, :3] = 5.0
    x[3, 7] = -0.0
    x = np.ascontiguousarray(x.astype(dtype))
    for largest in (True, False):
        y = x if largest else -x
        v, ix = (host(t) for t in ops.topk(dev(y), k, largest=largest))
        ov, oix = oracle.topk(y, k, largest=largest)
        assert np.array_equal(ix, oix) and np.array_equal(v.view(np.uint8), ov.view(np.uint8)), largest
    v, ix = (host(t) for t in ops.softmax_topk(dev(x), k))
    ov, oix = oracle.softmax_topk(x, k)
    if dtype == np.float32:   # (the values are within 2 ulp; which logit is the larger one, and so the order, does not depend on them)
        assert ulp_diff(v, ov).max() <= 2 and np.array_equal(ix, oix)
    else:                     # (sums agree to 2^-22: a probability on a boundary between two halves moves the row's order with it)
        same = (v == ov).all(axis=-1)
        assert half_ulp_diff(v, ov).max() <= 1 and same.sum() >= 3 and np.array_equal(ix[same], oix[same])


@pytest.mark.parametrize("n,k", [(50257, 40), (128256, 50), (262144, 600)])
def test_nan_of_any_payload_among_the_block_maxima_and_minima(ops, n, k):
    """Quiet and signalling NaN, alone, side by side and a block of nothing else: first in a plain top-k, last in the other direction."""
    rng = np.random.default_rng(n)
    x = rng.standard_normal((4, n)).astype(np.float32)
    b = x.view(np.uint32)
    b[0, rng.choice(n, 3, replace=False)] = 0x7F800001
    b[1, 64 * 9:64 * 11] = 0xFF800123
    b[2, rng.choice(n, k + 5, replace=False)] = 0x7FC00001
    b[3, [0, n - 1]] = (0x7F800001, 0xFFFFFFFF)
    xd = torch.from_numpy(x.view(np.int32)).cuda().view(torch.float32)
    for largest in (True, False):
        _, ix = (host(t) for t in ops.topk(xd, k, largest=largest))
        assert np.array_equal(ix, oracle.topk(x, k, largest=largest)[1]), largest


@pytest.mark.parametrize("n,k", [(700, 20), (2999, 100), (8192, 40), (8191, 300), (16384, 10), (30000, 120)])
def test_tie_at_the_cut_of_a_row_in_one_workgroup(ops, n, k):
    """Half probabilities of 2 to 6000 of the smallest half at the k-th place: the tied group ends within the list of
    candidates (its lower end is then read off the list) or goes on below it (it is looked for, and the row read again)."""
    rng = np.random.default_rng(n + k)
    rows = 40
    x = rng.standard_normal((rows, n)).astype(np.float32) * np.float32(1.25)
    cut = np.sort(x, axis=-1)[:, -k]
    units = np.exp(np.linspace(np.log(2.0), np.log(6000.0), rows))
    x[np.arange(rows), rng.integers(0, n, rows)] = cut + np.log(2.0 ** 24 / units).astype(np.float32)
    x = x.astype(np.float16)
    v, ix = (host(t) for t in ops.softmax_topk(dev(x), k))
    ov, oix = oracle.softmax_topk(x, k)
    # Sums agree to 2^-22, so a probability that close to a boundary between two halves, 2^-11 apart, may fall on either
    # side of it: at most one in 2^10 of the values, a unit each.
    same = (v.view(np.uint16) == ov.view(np.uint16)).all(axis=-1)
    assert half_ulp_diff(v, ov).max() <= 1 and same.sum() >= rows - max(4, 2 * v.size >> 10) and np.array_equal(ix[same], oix[same])
    equal = v[:, 1:] == v[:, :-1]
    assert np.all(ix[:, 1:][equal] > ix[:, :-1][equal])


@pytest.mark.parametrize("n", [8193, 12288, 16384, 16385, 32767])
@pytest.mark.parametrize("k", [1, 33, 64])
def test_a_small_k_of_rows_that_one_workgroup_holds(ops, n, k):
    """Past the rows that 256 threads hold: one workgroup a row, or the scan, against the chunk kernels and the select
    (rows.path = 1), bit for bit in plain top-k, whatever the order, the NaN and the equal values of the row."""
    from vkop_amd import capi
    rng = np.random.default_rng(n + k)
    for dtype in (np.float32, np.float16):
        for kind in ("llm", "levels", "sorted", "runs", "masked90", "nan_and_inf", "constant"):
            x = dev(np.ascontiguousarray(_rows(kind, 5, n, rng).astype(dtype)))
            for largest in (True, False):
                got = []
                for path in (0, 1):
                    capi.tune("rows.path", path)
                    got.append([host(t) for t in ops.topk(x, k, largest=largest)])
                capi.tune("rows.path", 0)
                (v, ix), (w, jx) = got
                assert np.array_equal(ix, jx) and v.tobytes() == w.tobytes(), (kind, largest)
        _compare_paths(ops, n, k, dtype, 5, ["llm", "levels", "masked90", "nan_and_inf", "coarse_levels"],
                       capi.measure_path(capi.F32 if dtype == np.float32 else capi.F16, (5, n), -1, k))


@pytest.mark.parametrize("rows,n,k,off,kernels", [(3, 12001, 20, 0, 2), (64, 8401, 5, 0, 2), (1, 16383, 40, 1, 2), (3, 12000, 20, 0, 1), (3, 12000, 20, 1, 1),
                                                  (65, 12001, 20, 0, 1), (257, 12001, 20, 0, 2), (257, 16384, 64, 2, 2), (16, 8193, 64, 0, 1)])
def test_sampling_of_float_rows_that_one_workgroup_or_the_scan_takes(ops, rows, n, k, off, kernels):
    """The scaled form on rows of 8193 to 16384 floats: up to 64 whose length takes them off 16 bytes, and more than 256, the scan and
    the pick kernel, others one workgroup a row (16 of 8193 and k = 64 have too few blocks for the scan); a tensor's start does not
    count.  With the first kernel alone (a library that can leave one out) the results are written by one-workgroup rows only."""
    import ctypes
    from vkop_amd import capi
    rng = np.random.default_rng(n + k)
    x = np.concatenate([_rows(kind, rows, n, rng) for kind in ("llm", "bf16")])[::2] if rows > 1 else _rows("llm", 1, n, rng)
    big = torch.empty(rows * n + 4, device="cuda")
    xd = big[off:off + rows * n].view(rows, n)
    xd.copy_(dev(x))
    v, ix, c = (host(t) for t in ops.softmax_topk_sampling(xd, k, 1.25, 0.9))
    ov, oix, _ = oracle.softmax_topk_sampling(x, k, 1.25, 0.9)
    assert ulp_diff(v, ov).max() <= 2 and np.array_equal(c, oracle.topp_count(v, 0.9))
    xs = x * np.float32(1.25)
    op = oracle.softmax(xs)
    for r in range(rows):
        check_fused_invariants(xs[r], v[r], ix[r])
        if well_separated_cut(op[r], xs[r], k):
            assert np.array_equal(ix[r], oix[r]), r
    part = ctypes.CDLL(capi.BENCH_LIB_PATH)
    part.vkop_hip_softmax_topk_sampling.argtypes = capi.lib()._signatures["vkop_hip_softmax_topk_sampling"][1]
    values, indices, counts = torch.full((rows, k), -7.0, device="cuda"), *(torch.full((m,), -7, dtype=torch.int32, device="cuda") for m in (rows * k, rows))
    ws, size = ops.Workspace().get(capi.softmax_topk_workspace_bytes(capi.F32, (rows, n), -1, k))
    try:
        assert part.vkop_hip_measure_stages(1) == 0
        assert part.vkop_hip_softmax_topk_sampling(xd.data_ptr(), values.data_ptr(), indices.data_ptr(), counts.data_ptr(), capi.F32,
                                                   (ctypes.c_int * 2)(rows, n), 2, -1, k, 1.25, 0.9, ws, size,
                                                   torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
    finally:
        part.vkop_hip_measure_stages(3)
    assert bool((values == -7.0).all()) == (kernels == 2) and (kernels == 2 or np.array_equal(host(values), v))


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("rows,n,k", [(257, 10001, 40), (300, 8400, 64), (257, 9361, 64), (257, 16640, 64), (260, 24000, 40), (1024, 8193, 5)])
def test_plain_topk_on_more_rows_than_cus(ops, rows, n, k, dtype):
    """One workgroup a row where the row has few blocks a place, the scan otherwise: the oracle's values and indices either way."""
    rng = np.random.default_rng(rows + n)
    bits = np.uint16 if dtype == np.float16 else np.uint32
    for kind in ("bf16", "levels", "runs") if rows < 1000 else ("bf16",):
        x = np.ascontiguousarray(_rows(kind, rows, n, rng).astype(dtype))
        for largest in (True, False):
            t, tj = ops.topk(dev(x), k, largest=largest)
            et, ej = oracle.topk(x, k, largest=largest)
            assert np.array_equal(host(tj), ej) and np.array_equal(host(t).view(bits), et.view(bits)), (kind, largest)
