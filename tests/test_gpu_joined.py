"""The one-launch softmax of long rows (kernels_joined.hpp): its workgroups wait for each other's chunk statistics."""
import ctypes

import numpy as np
import pytest

import oracle
from helpers import half_ulp_diff, ulp_diff

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# rows, elements: a chunk of 512 threads is 16384 / 8192 / 4096 elements, of 256 threads 10240.  Whole chunks, one element more
# and less, a last chunk of a vector or less, and each of the shapes the plan chooses between
SHAPES = [(64, 65536), (64, 65537), (40, 65535), (32, 131073), (32, 33001), (100, 9001), (150, 8200), (300, 20483), (130, 50257),
          (33, 229377)]


@pytest.fixture(scope="module")
def ops():
    from vkop_amd import capi, ops as _ops
    capi.init(0)
    return _ops


def rows_of(rows, n, dtype, seed):
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((rows, n)) * 2).astype(dtype)
    x[0] = dtype(0.5)                    # one value
    x[1, : n // 2] = dtype(-np.inf)      # masked
    x[2] = dtype(-np.inf)                # nothing left: NaN
    x[3, n - 1] = dtype(np.nan)
    x[4, 0] = dtype(np.inf)
    x[5, n - 1] = dtype(30.0)            # the maximum in the last, moved vector
    return x


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("rows,n", SHAPES)
@pytest.mark.parametrize("start", [0, 1])
def test_rows_against_the_oracle_and_the_pair_of_kernels(ops, rows, n, dtype, start):
    x = rows_of(rows, n, dtype, rows + n)
    buf = torch.empty(start + rows * n, dtype=torch.float32 if dtype == np.float32 else torch.float16, device="cuda")
    t = buf[start:].view(rows, n)
    t.copy_(torch.from_numpy(x))
    got = ops.softmax(t)
    again = ops.softmax(t)
    replaced = ops.softmax(t, nan_where=True, nan_value=7.0)
    inplace = t.clone()
    ops.softmax(inplace, out=inplace)    # (the one launch too; the pair where the last vector reaches back into the chunk before)
    best = ops.softmax_reduce_max(t, -1)
    torch.cuda.synchronize()
    bits = torch.int32 if dtype == np.float32 else torch.int16
    nan = torch.isnan(got)
    assert torch.equal(got.view(bits), again.view(bits))
    assert torch.equal(torch.isnan(inplace), nan) and torch.equal(inplace[~nan].view(bits), got[~nan].view(bits))
    assert torch.equal(replaced[~nan], got[~nan]) and bool((replaced[nan] == 7.0).all())
    top = got.max(-1).values
    assert torch.equal(torch.isnan(top), torch.isnan(best)) and torch.equal(top[~torch.isnan(top)], best[~torch.isnan(best)])
    some = [0, 1, 2, 3, 4, 5, 6, rows - 1]
    want, g = oracle.softmax(x[some]), got.cpu().numpy()[some]
    if dtype == np.float32:
        assert ulp_diff(g, want).max() <= 2
    else:
        assert half_ulp_diff(g, want).max() <= 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("rows,n", [(64, 65537), (300, 20483), (32, 33001), (100, 9001)])
def test_a_workgroup_that_does_not_wait_reads_the_other_chunks_itself(ops, rows, n, dtype):
    """Looks limited to one (a bound of the kernel's own wait): same bits, records and counters left at zero."""
    from vkop_amd import capi
    lib = ctypes.CDLL(capi.BENCH_LIB_PATH)
    f = lib.vkop_hip_softmax
    f.argtypes = capi.lib()._signatures["vkop_hip_softmax"][1]
    gen = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn((rows, n), generator=gen, device="cuda").to(dtype)
    x[1, : n // 2] = float("-inf")
    want = ops.softmax(x)
    shape = (ctypes.c_int * 2)(rows, n)
    dt = capi.F32 if dtype == torch.float32 else capi.F16
    need = capi.lib().vkop_hip_softmax_workspace_bytes(dt, shape, 2, -1)
    ws = torch.zeros(need + 256, dtype=torch.uint8, device="cuda")
    at = ws.data_ptr() + (-ws.data_ptr()) % 256
    stream = torch.cuda.current_stream().cuda_stream
    try:
        for polls in (0, 0, 1, 100, 0):
            assert lib.vkop_hip_measure_polls(polls) == 0
            out = torch.full_like(x, 5.0)
            torch.cuda.synchronize()
            assert f(x.data_ptr(), out.data_ptr(), dt, shape, 2, -1, 0, 0.0, at, need, stream) == 0
            torch.cuda.synchronize()
            assert torch.equal(out, want), polls
            assert int(ws.count_nonzero()) == 0, polls
    finally:
        lib.vkop_hip_measure_polls(100)


@pytest.mark.parametrize("rows,n", [(64, 128256), (32, 33001), (64, 200000)])
def test_nothing_is_written_behind_the_workspace(ops, rows, n):
    """With what the query asks for, and with what the pair of kernels' statistics take, 24 bytes a chunk."""
    from vkop_amd import capi
    x = torch.randn((rows, n), generator=torch.Generator(device="cuda").manual_seed(n), device="cuda")
    want = ops.softmax(x)
    need = capi.softmax_workspace_bytes(capi.F32, (rows, n), -1)
    pair = 65536 + -(-(need - 65536) * 3 // 4 // 256) * 256
    for size in (need, pair):
        ws = torch.zeros(need + 65536, dtype=torch.uint8, device="cuda")
        ws[size:] = 0xA5
        out = torch.zeros_like(x)
        capi.softmax(x.data_ptr(), out.data_ptr(), capi.F32, (rows, n), -1, 0, 0.0, ws.data_ptr(), size,
                     torch.cuda.current_stream().cuda_stream)
        assert torch.equal(out, want)
        assert bool((ws[size:] == 0xA5).all())


def test_more_rows_than_counters(ops):
    """16384 counters: two launches.  540 M halves."""
    rows, n = 16384 + 40, 32776
    x = torch.empty((rows, n), dtype=torch.float16, device="cuda").normal_(generator=torch.Generator(device="cuda").manual_seed(3))
    got = ops.softmax(x)
    for r in (0, 16383, 16384, rows - 1):
        assert half_ulp_diff(got[r:r + 1].cpu().numpy(), oracle.softmax(x[r:r + 1].cpu().numpy())).max() <= 1, r
    ops.softmax(x, out=x)
    assert torch.equal(x, got)


def test_workspace_with_other_contents_and_replays(ops):
    """What the records' place held before does not matter, in an eager call; a recording replays, with eager work and
    synchronizations in between."""
    from vkop_amd import capi
    rows, n = 64, 40000
    gen = torch.Generator(device="cuda").manual_seed(11)
    xs = [torch.randn((rows, n), generator=gen, device="cuda") for _ in range(3)]
    want = [ops.softmax(x) for x in xs]
    need = capi.softmax_workspace_bytes(capi.F32, (rows, n), -1)
    ws = torch.zeros(need + 256, dtype=torch.uint8, device="cuda")
    at = ws.data_ptr() + (-ws.data_ptr()) % 256
    counters = 65536 - (ws.data_ptr() - at)
    ws[counters:].random_(0, 256, generator=gen)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    src, out = torch.empty_like(xs[0]), torch.empty_like(xs[0])
    call = lambda: capi.softmax(src.data_ptr(), out.data_ptr(), capi.F32, (rows, n), -1, 0, 0.0, at, need, side.cuda_stream)  # noqa: E731
    with torch.cuda.stream(side):
        for i in range(3):
            src.copy_(xs[i])
            call()
            side.synchronize()
            assert torch.equal(out, want[i])
    stream = side.cuda_stream
    capi.graph_begin(stream)
    call()
    graph = capi.graph_end(stream)
    try:
        with torch.cuda.stream(side):
            for i in (0, 1, 2, 2, 1):
                src.copy_(xs[i])
                out.zero_()
                side.synchronize()
                capi.graph_launch(graph, stream)
                side.synchronize()
                assert torch.equal(out, want[i])
                src.copy_(xs[(i + 1) % 3])
                call()
                side.synchronize()
                assert torch.equal(out, want[(i + 1) % 3])
    finally:
        capi.graph_destroy(graph)


@pytest.mark.parametrize("rows,n", [(64, 65537), (300, 20483), (32, 33001), (150, 8200)])
def test_a_workspace_whose_counters_do_not_start_at_zero_ends_every_wait(ops, rows, n):
    """A workspace nobody cleared: at each of these counts some workgroup takes itself for the row's last one and clears the
    records while others still look for them.  They run out of looks and read the chunks themselves: same bits."""
    from vkop_amd import capi
    x = torch.randn((rows, n), generator=torch.Generator(device="cuda").manual_seed(n), device="cuda")
    want = ops.softmax(x)
    need = capi.softmax_workspace_bytes(capi.F32, (rows, n), -1)
    ws = torch.zeros(need + 256, dtype=torch.uint8, device="cuda")
    at = -ws.data_ptr() % 256
    stream = torch.cuda.current_stream().cuda_stream
    for count in (0, 1, 2, 3, 4, 7, 11, 1 << 30):
        ws[at:at + 65536].view(torch.int32).fill_(count)
        for _ in range(2):
            out = torch.zeros_like(x)
            capi.softmax(x.data_ptr(), out.data_ptr(), capi.F32, (rows, n), -1, 0, 0.0, ws.data_ptr() + at, need, stream)
            torch.cuda.synchronize()
            assert torch.equal(out, want), count


def test_two_streams_on_one_workspace_end(ops):
    """Against the rules: their records and counters replace each other's.  Nothing is said about the values of the first ten
    calls, but every one ends, and the workspace serves again once it is cleared."""
    from vkop_amd import capi
    rows, n = 64, 65537
    x = torch.randn((rows, n), generator=torch.Generator(device="cuda").manual_seed(5), device="cuda")
    want = ops.softmax(x)
    need = capi.softmax_workspace_bytes(capi.F32, (rows, n), -1)
    ws = torch.zeros(need + 256, dtype=torch.uint8, device="cuda")
    at = ws.data_ptr() + (-ws.data_ptr()) % 256
    outs, streams = [torch.zeros_like(x) for _ in range(2)], [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(5):
        for out, stream in zip(outs, streams):
            capi.softmax(x.data_ptr(), out.data_ptr(), capi.F32, (rows, n), -1, 0, 0.0, at, need, stream.cuda_stream)
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream().cuda_stream
    capi.workspace_init(at, need // 4 * 4, stream)
    out = torch.zeros_like(x)
    capi.softmax(x.data_ptr(), out.data_ptr(), capi.F32, (rows, n), -1, 0, 0.0, at, need, stream)
    torch.cuda.synchronize()
    assert torch.equal(out, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("rows,n", [(64, 65536), (64, 65540), (300, 20483), (32, 33001), (100, 9001), (150, 8200), (64, 200000), (64, 128256),
                                    (64, 65537), (64, 65544), (64, 65543), (300, 20484), (300, 20487), (300, 20488)])
def test_in_place_while_other_chunks_are_written(ops, rows, n, dtype):
    """In place, with looks limited to none, one and a few: workgroups read chunks whose own workgroups start and write over them
    meanwhile.  Same bits as out of place; last vectors that reach back into the chunk before and ones that just do not."""
    from vkop_amd import capi
    lib = ctypes.CDLL(capi.BENCH_LIB_PATH)
    f = lib.vkop_hip_softmax
    f.argtypes = capi.lib()._signatures["vkop_hip_softmax"][1]
    gen = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn((rows, n), generator=gen, device="cuda").sub_(4.0).to(dtype)   # (a probability is above every logit of some chunks)
    x[1, : n // 2] = float("-inf")
    want = ops.softmax(x)
    shape = (ctypes.c_int * 2)(rows, n)
    dt = capi.F32 if dtype == torch.float32 else capi.F16
    need = capi.lib().vkop_hip_softmax_workspace_bytes(dt, shape, 2, -1)
    ws = torch.zeros(need + 256, dtype=torch.uint8, device="cuda")
    at = ws.data_ptr() + (-ws.data_ptr()) % 256
    stream = torch.cuda.current_stream().cuda_stream
    try:
        for polls in (0, 0, 0, 0, 1, 1, 3, 100):
            assert lib.vkop_hip_measure_polls(polls) == 0
            y = x.clone()
            torch.cuda.synchronize()
            assert f(y.data_ptr(), y.data_ptr(), dt, shape, 2, -1, 0, 0.0, at, need, stream) == 0
            torch.cuda.synchronize()
            assert torch.equal(y, want), polls
    finally:
        lib.vkop_hip_measure_polls(100)
