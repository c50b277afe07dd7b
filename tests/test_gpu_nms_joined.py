"""NMS in one launch (kernels_nms.hpp: place_records): every workgroup waits for the numbers of the pairs before its own."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

PER_CLASS = 60
TICKETS = 65536
# batch, classes, boxes: one pair, the most of wide and of narrow workgroups in one launch and one more, and candidates by the thousand
SHAPES = [(1, 1, 500), (1, 80, 1001), (4, 128, 300), (19, 27, 300), (16, 80, 700), (12, 128, 200), (29, 53, 200), (2, 7, 3000)]


@pytest.fixture(scope="module")
def lib():
    from vkop_amd import capi
    capi.init(0)
    handle = ctypes.CDLL(capi.BENCH_LIB_PATH)
    handle.vkop_hip_nms.argtypes = capi.lib()._signatures["vkop_hip_nms"][1]
    yield handle
    handle.vkop_hip_measure_polls(100)


def make(B, C, N, dtype, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    centre = torch.rand((B, N, 2), generator=gen, device="cuda")
    half = 0.1 * torch.rand((B, N, 2), generator=gen, device="cuda")
    scores = torch.rand((B, C, N), generator=gen, device="cuda")
    scores[:, C // 2] = 0.0      # a class without a candidate
    return torch.cat([centre - half, centre + half], -1).to(dtype).contiguous(), scores.to(dtype).contiguous()


def two_launch_bytes(B, C, N):
    up = lambda v: (v + 255) // 256 * 256  # noqa: E731
    return TICKETS + up(2 * B * C * 4) + up(B * C * min(N, 2048, PER_CLASS) * 4)


class Call:
    def __init__(self, lib, boxes, scores, ws, nbytes, capacity):
        from vkop_amd import capi
        B, C, N = scores.shape
        self.out = torch.full((max(capacity, 1), 3), 77, dtype=torch.int32, device="cuda")
        self.count = torch.full((2,), 77, dtype=torch.int32, device="cuda")
        self.args = (boxes.data_ptr(), scores.data_ptr(), self.out.data_ptr(), capacity, self.count.data_ptr(),
                     capi.F32 if scores.dtype == torch.float32 else capi.F16, B, C, N, 0, PER_CLASS, 0.45, 0.4, ws, nbytes)
        self.f = lib.vkop_hip_nms

    def __call__(self, stream=None):
        assert self.f(*self.args, (stream or torch.cuda.current_stream()).cuda_stream) == 0
        return self


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("B,C,N", SHAPES)
def test_one_launch_and_two_whatever_the_wait(lib, B, C, N, dtype):
    """Looks limited to none, some and the usual number (a bound of the kernel's own wait): the records of the two launches, which a
    workspace of their size gives, also with less room than there are records, and the arrival counters left at zero.  What the
    workspace held otherwise is random."""
    from vkop_amd import capi
    boxes, scores = make(B, C, N, dtype, B + C + N)
    need = capi.lib().vkop_hip_nms_workspace_bytes(B, C, N, PER_CLASS)
    ws = torch.randint(0, 256, (need + 256,), dtype=torch.uint8, device="cuda")
    at = ws.data_ptr() + (-ws.data_ptr()) % 256
    tickets = ws[at - ws.data_ptr():][:TICKETS]
    tickets.zero_()
    capacity = B * C * min(N, PER_CLASS)
    two = Call(lib, boxes, scores, at, two_launch_bytes(B, C, N), capacity)()
    torch.cuda.synchronize()
    total = int(two.count[0])
    if B * C <= 200:
        want = oracle.nms(boxes.float().cpu().numpy(), scores.float().cpu().numpy(), 0.45, 0.4, PER_CLASS, max_candidates=2048)
        assert np.array_equal(two.out[:total].cpu().numpy(), want)
    for polls in (0, 1, 100, 0, 100):
        assert lib.vkop_hip_measure_polls(polls) == 0
        for room in (capacity, total, max(total - 1, 0), total // 2):
            one = Call(lib, boxes, scores, at, need, room)
            torch.cuda.synchronize()
            one()
            torch.cuda.synchronize()
            held = min(total, room)
            assert torch.equal(one.count, two.count) and torch.equal(one.out[:held], two.out[:held]), (polls, room)
            if room > total:
                assert one.out[total].tolist() == [-1, -1, -1]
                assert bool((one.out[total + 1:] == 77).all())
            assert int(tickets.count_nonzero()) == 0


def test_a_recording_replayed(lib):
    """Other inputs in every replay, eager calls on the same workspace between."""
    from vkop_amd import capi
    lib.vkop_hip_measure_polls(100)
    B, C, N = 8, 40, 900
    boxes, scores = make(B, C, N, torch.float32, 1)
    need = capi.lib().vkop_hip_nms_workspace_bytes(B, C, N, PER_CLASS)
    ws = torch.zeros(need + 256, dtype=torch.uint8, device="cuda")
    at = ws.data_ptr() + (-ws.data_ptr()) % 256
    capacity = B * C * PER_CLASS
    one = Call(lib, boxes, scores, at, need, capacity)
    other = torch.zeros(need + 256, dtype=torch.uint8, device="cuda")
    two = Call(lib, boxes, scores, other.data_ptr() + (-other.data_ptr()) % 256, two_launch_bytes(B, C, N), capacity)
    one()
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        one(stream)
        one(stream)
    for seed in range(2, 8):
        b, s = make(B, C, N, torch.float32, seed)
        boxes.copy_(b)
        scores.copy_(s)
        graph.replay()
        torch.cuda.synchronize()
        got, count = one.out.clone(), one.count.clone()
        two()
        one()
        torch.cuda.synchronize()
        total = int(two.count[0])
        for rec, n in ((got, count), (one.out, one.count)):
            assert torch.equal(n, two.count) and torch.equal(rec[:total], two.out[:total]), seed


@pytest.mark.parametrize("B,C", [(2, 80), (8, 20)])
def test_a_recording_whose_workspace_serves_another_operator(B, C):
    """Every replay has its arguments from the recording, and the same top-k before it in the same workspace, whose lists, keys and
    counters lie where a call's own words do; the end of that workspace is put back, too, to what it was before the replay.  (Fewer
    candidates than places: the pairs' numbers differ from replay to replay.)"""
    from vkop_amd import capi
    capi.init(0)
    N, per_class, n, k = 700, 300, 33600, 300
    boxes, scores = make(B, C, N, torch.float32, 1)
    rows = torch.randn((1, n), generator=torch.Generator(device="cuda").manual_seed(2), device="cuda")
    values, indices = torch.empty((1, k), device="cuda"), torch.empty((1, k), dtype=torch.int32, device="cuda")
    room = B * C * per_class
    out, count = torch.zeros((room, 3), dtype=torch.int32, device="cuda"), torch.zeros(2, dtype=torch.int32, device="cuda")
    nms_bytes = capi.nms_workspace_bytes(B, C, N, per_class)
    need = max(nms_bytes, capi.topk_workspace_bytes(capi.F32, (1, n), -1, k))
    memory = torch.zeros(need + 256, dtype=torch.uint8, device="cuda")
    at = memory.data_ptr() + (-memory.data_ptr()) % 256
    end = memory[at - memory.data_ptr():][nms_bytes - 256:nms_bytes]

    def calls(stream):
        capi.topk(rows.data_ptr(), values.data_ptr(), indices.data_ptr(), capi.F32, (1, n), -1, k, 1, 1, at, need, stream)
        capi.nms(boxes.data_ptr(), scores.data_ptr(), out.data_ptr(), room, count.data_ptr(), capi.F32, B, C, N, 0, per_class, 0.45, 0.8,
                 at, need, stream)

    stream = torch.cuda.Stream()
    calls(stream.cuda_stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        calls(stream.cuda_stream)
    for seed in range(3, 9):
        b, s = make(B, C, N, torch.float32, seed)
        boxes.copy_(b)
        scores.copy_(s)
        before = end.clone()
        graph.replay()
        torch.cuda.synchronize()
        want = oracle.nms(b.cpu().numpy(), s.cpu().numpy(), 0.45, 0.8, per_class, max_candidates=2048)
        assert count.tolist() == [len(want), 0], seed
        assert np.array_equal(out[:len(want)].cpu().numpy(), want), seed
        if seed % 2:
            end.copy_(before)
