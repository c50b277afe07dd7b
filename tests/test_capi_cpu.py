"""CPU-only checks of the C-ABI library: it loads, it exports every function the
header declares, and argument errors are reported without touching a GPU."""
import ctypes
import os
import subprocess

import pytest

from vkop_amd import capi


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(capi.LIB_PATH):
        capi.build()
    return capi.lib()


def test_exports_every_declared_symbol(lib):
    declared = capi.declared_symbols()
    assert len(declared) >= 25
    for name in declared:
        assert hasattr(lib, name), name
    # and the binding knows a signature for each of them, and beyond them only for the
    # measurement hooks of the internal header
    internal = capi.internal_symbols()
    assert internal and not set(internal) & set(declared)
    shipped = [name for name in internal if name not in capi.BENCH_ONLY]
    assert sorted(lib._signatures) == sorted(declared + shipped)
    for name in shipped:
        assert hasattr(lib, name), name

    def exported(path):
        out = subprocess.check_output(["nm", "-D", "--defined-only", path]).decode()
        return {line.split()[-1] for line in out.splitlines() if " T " in line}
    assert set(declared) <= exported(capi.LIB_PATH)
    # the hook that changes what a call launches is not in the shipped library, only in the benchmark's build of it
    assert not set(capi.BENCH_ONLY) & exported(capi.LIB_PATH)
    assert set(capi.BENCH_ONLY) <= set(internal)
    assert set(declared) | set(internal) <= exported(capi.BENCH_LIB_PATH)


def test_no_oracle_or_torch_linked_into_product():
    out = subprocess.check_output(["ldd", capi.LIB_PATH]).decode()
    assert "oracle" not in out and "torch" not in out
    assert "amdhip64" in out


def test_argument_errors_need_no_gpu(lib):
    shape = (ctypes.c_int * 2)(4, 1000)
    dummy = ctypes.c_void_p(256)
    f = lib.vkop_hip_softmax
    assert f(dummy, dummy, 7, shape, 2, 1, 0, 0.0, None, 0, None) == capi.ERR_INVALID
    assert "dtype" in capi.last_error()
    assert f(dummy, dummy, capi.F32, shape, 5, 1, 0, 0.0, None, 0, None) == capi.ERR_INVALID
    assert f(dummy, dummy, capi.F32, shape, 2, 2, 0, 0.0, None, 0, None) == capi.ERR_INVALID
    assert f(dummy, dummy, capi.F32, shape, 2, -3, 0, 0.0, None, 0, None) == capi.ERR_INVALID
    assert f(None, dummy, capi.F32, shape, 2, 1, 0, 0.0, None, 0, None) == capi.ERR_INVALID
    assert f(dummy, dummy, capi.F32, None, 2, 1, 0, 0.0, None, 0, None) == capi.ERR_INVALID
    t = lib.vkop_hip_topk
    assert t(dummy, dummy, dummy, capi.F32, shape, 2, -1, 0, 1, 1, None, 0, None) == capi.ERR_INVALID
    assert t(dummy, dummy, dummy, capi.F32, shape, 2, -1, 1001, 1, 1, None, 0, None) == capi.ERR_INVALID
    assert "exceeds" in capi.last_error()
    big = (ctypes.c_int * 2)(1, 100000)
    assert t(dummy, dummy, dummy, capi.F32, big, 2, -1, capi.MAX_K + 1, 1, 1, None, 0, None) == capi.ERR_UNSUPPORTED
    s = lib.vkop_hip_softmax_topk
    need = lib.vkop_hip_softmax_topk_workspace_bytes(capi.F32, shape, 2, -1, 5)
    assert need > 0
    assert s(dummy, None, dummy, dummy, capi.F32, shape, 2, -1, 5, 1, None, 0, None) == capi.ERR_WORKSPACE
    assert s(dummy, None, dummy, dummy, capi.F32, shape, 2, -1, 5, 1, dummy, need - 1, None) == capi.ERR_WORKSPACE
    assert lib.vkop_hip_reduce_max(dummy, dummy, capi.F32, (ctypes.c_int * 2)(3, 0), 2, 1, None) == capi.ERR_INVALID
    # empty tensors are a no-op, not an error
    empty = (ctypes.c_int * 2)(0, 1000)
    assert f(None, None, capi.F32, empty, 2, 1, 0, 0.0, None, 0, None) == capi.OK


def test_workspace_queries_are_pure(lib):
    shape = (ctypes.c_int * 2)(64, 128256)
    a = lib.vkop_hip_softmax_topk_workspace_bytes(capi.F32, shape, 2, -1, 50)
    b = lib.vkop_hip_softmax_topk_workspace_bytes(capi.F32, shape, 2, -1, 50)
    assert a == b and a % 256 == 0
    assert lib.vkop_hip_softmax_topk_workspace_bytes(9, shape, 2, -1, 50) == 0


def test_timeline_summary_reads_a_log_of_two_lanes():
    """bench.py --timeline: the summary of a log made up here -- two lanes, each scan 8 us and pick 6 us with 2 us
    between them, the lanes half a call apart -- gives back those durations, gaps and the overlap."""
    import importlib.util
    import numpy as np
    spec = importlib.util.spec_from_file_location("bench_for_test", os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    recs = []
    period = 18000  # ns per call of a lane: 8 + 2 + 6 + 2
    for lane, ws in enumerate((0x1000, 0x2000)):
        for call in range(40):
            s0 = 5_000_000 + lane * period // 2 + call * period
            for wg in (0, 16, 500):        # scan workgroups: enter together, the last leaves after 8 us
                recs.append(((wg << 40) | ws, (s0 + wg) // 10, (s0 + 7000 + 2 * wg) // 10))
            p0 = s0 + 8000 + 2000
            for wg in range(4):            # pick workgroups
                recs.append(((1 << 63) | (wg << 40) | ws, (p0 + wg) // 10, (p0 + 5000 + 250 * wg + (250 if wg == 3 else 0)) // 10))
    # (a warm-up stretch long before, which the summary leaves out)
    recs.append((0x1000, 100, 200))
    out = bench.timeline_summary(np.array(recs, dtype=np.uint64), 0.009, 2, 8)
    assert out["lanes_seen"] == 2
    assert abs(out["scan_kernel_us_first_entry_to_last_exit"]["mean"] - 8.0) < 0.05
    assert abs(out["pick_kernel_us_first_entry_to_last_exit"]["mean"] - 6.0) < 0.05
    assert abs(out["gap_us_scan_exit_to_pick_entry_same_lane"] - 2.0) < 0.05
    assert abs(out["gap_us_pick_exit_to_next_scan_entry_same_lane"] - 2.0) < 0.05
    assert abs(out["us_per_call_from_the_log"] - 9.0) < 0.05            # two lanes, 18 us a call each
    assert abs(out["mean_kernels_running"] - 2 * 14.0 / 18.0) < 0.05     # each lane busy 14 of 18 us


def test_route_planner_without_a_gpu(lib):
    """Which kernels a last-axis top-k / fused call takes is decided on the host (vkop_hip_measure_path: 4 one wave
    per row, 2 scan + pick, 3 scan + gather + rank, 1 chunk (+ merge), 0 radix select or general kernels;
    vkop_hip_rows_plan: threads, loads, chunks of the chunk kernel).  The five workloads' routes, the shape that a
    limit of 8192 blocks had left to the radix select, and the rule that no shape takes chunk + merge over SEVERAL
    chunks unless vkop_hip_tune asks for it."""
    F32, F16 = capi.F32, capi.F16
    assert capi.measure_path(F32, (1, 1000), -1, 5) == 4            # C1
    assert capi.measure_path(F32, (256, 1000), -1, 5) == 4          # C2
    assert capi.measure_path(F16, (256, 1000), -1, 5) == 4
    assert capi.measure_path(F32, (64, 128256), -1, 50) == 2        # C3
    assert capi.measure_path(F16, (64, 128256), -1, 50) == 2
    assert capi.measure_path(F32, (8, 262144), -1, 1024) == 3       # C4
    assert capi.measure_path(F32, (16, 8400), -1, 300) == 1         # C5's select: one workgroup a row
    assert capi.rows_plan(F32, (16, 8400), -1, 300)[2] == 1
    assert capi.measure_path(F32, (4, 1048576), -1, 100) == 2       # 16384 blocks a row
    assert capi.measure_path(F32, (1, 128256), -1, 50) == 2         # a single sequence's logits
    several = []
    for dt in (F32, F16):
        for rows in (1, 8, 16, 17, 64, 1024):
            for n in list(range(256, 40000, 997)) + [8192, 8193, 8320, 8321, 16384, 32768, 32769, 65536, 131072, 300000, 1 << 20]:
                for k in (1, 5, 32, 33, 64, 65, 100, 255, 256, 408, 511):
                    if k > n:
                        continue
                    if capi.measure_path(dt, (rows, n), -1, k) == 1 and capi.rows_plan(dt, (rows, n), -1, k)[2] > 1:
                        several.append((dt, rows, n, k))
    assert not several, several[:10]
    try:
        capi.tune("rows.path", 1)
        assert capi.measure_path(F32, (64, 128256), -1, 50) == 1 and capi.rows_plan(F32, (64, 128256), -1, 50)[2] > 1
    finally:
        capi.tune("rows.path", 0)
    # the workspace a call is told to bring covers the headline shape with room in the static scratch's 4 MiB
    need = capi.softmax_topk_workspace_bytes(F32, (64, 128256), -1, 50)
    assert 64 * 1024 < need <= 4 << 20


def test_rows_of_one_workgroup_up_to_a_row_a_cu(lib):
    """Rows that 512 threads hold go to one workgroup each while there are no more of them than CUs, and to the scan beyond."""
    for dt in (capi.F32, capi.F16):
        for n in (8193, 8400, 10001, 12000, 16383, 16384):
            for k in (1, 5, 20, 32):
                for rows in (1, 17, 255, 256, 257, 300, 1023, 1024, 5000):
                    assert capi.measure_path(dt, (rows, n), -1, k) == (1 if rows <= 256 else 2), (dt, rows, n, k)
    assert capi.measure_path(capi.F32, (256, 16385), -1, 20) == 2


def test_rows_plan_tells_the_loads_that_run(lib):
    """Rows that a wide workgroup holds are launched with as few vectors a thread as hold the row, unless the shape is forced."""
    F32, F16 = capi.F32, capi.F16
    for dt, n, k, want in ((F32, 8400, 300, (1024, 3, 1)), (F32, 8192, 300, (1024, 2, 1)), (F32, 16000, 300, (1024, 4, 1)),
                           (F32, 16385, 300, (1024, 8, 1)), (F32, 4000, 130, (512, 2, 1)), (F32, 8190, 130, (512, 4, 1)),
                           (F16, 8400, 300, (1024, 2, 1)), (F16, 8192, 300, (1024, 1, 1)), (F16, 20000, 300, (1024, 4, 1))):
        assert capi.rows_plan(dt, (16, n), -1, k) == want, (dt, n, k)
    try:
        for shape in ((1024, 8, 1), (512, 8, 1), (1024, 4, 8)):
            for name, value in zip(("rows.threads", "rows.loads", "rows.chunks"), shape):
                capi.tune(name, value)
            assert capi.rows_plan(F32, (16, 8400), -1, 100) == shape
    finally:
        for name in ("rows.threads", "rows.loads", "rows.chunks"):
            capi.tune(name, 0)


def test_native_front_end_refuses_what_the_operators_refuse():
    """vkop_amd.ops reaches the C ABI through its native front end, which is built with the library; a tensor that is not on
    a GPU, and what is no tensor, are TypeErrors before anything else happens."""
    torch = pytest.importorskip("torch")
    from vkop_amd import ops
    x = torch.zeros(2, 5)
    for call in (lambda t: ops.softmax(t), lambda t: ops.topk(t, 2), lambda t: ops.softmax_topk(t, 2),
                 lambda t: ops.softmax_topk_sampling(t, 2, 1.0, 0.9), lambda t: ops.softmax_reduce_max(t, 1), lambda t: ops.reduce_max(t, 1)):
        for bad in (x, x.numpy(), None):
            with pytest.raises(TypeError, match="GPU"):
                call(bad)


@pytest.mark.parametrize("transform", ["vmap", "jvp", "vjp"])
def test_a_tensor_without_storage_is_an_exception(transform):
    """Inside torch.vmap, jvp and vjp an operator sees a wrapper without storage.  Its pointer is asked for, and the error
    raised, while the interpreter's lock is held and before the stream is (a GPU is not needed to get there)."""
    torch = pytest.importorskip("torch")
    from torch._subclasses import FakeTensorMode
    from vkop_amd import ops
    with FakeTensorMode():
        t = torch.empty(2, 5, device="cuda")
    out = torch.empty(2, 5)
    run = {"vmap": lambda f: torch.vmap(f)(t), "jvp": lambda f: torch.func.jvp(f, (t,), (t,)), "vjp": lambda f: torch.func.vjp(f, t)}[transform]
    for op in (lambda x: ops.softmax(x), lambda x: ops.softmax(x, out=out), lambda x: ops.topk(x, 2), lambda x: ops.softmax_topk(x, 2),
               lambda x: ops.softmax_topk(x, 2, return_probs=True), lambda x: ops.softmax_topk_sampling(x, 2, 1.0, 0.9),
               lambda x: ops.softmax_reduce_max(x, 0), lambda x: ops.reduce_max(x, 0)):
        with pytest.raises(RuntimeError, match="storage"):
            run(op)


def test_native_front_end_takes_whole_numbers_only():
    """k and axis are whole numbers (Python's, numpy's, one-element integer tensors): anything else is a TypeError, as ctypes
    has it, and not rounded or parsed."""
    torch = pytest.importorskip("torch")
    import numpy as np
    from torch._subclasses import FakeTensorMode
    from vkop_amd import ops
    with FakeTensorMode():
        t = torch.empty(2, 5, device="cuda")
    for bad in (2.5, "1", np.float64(1), None, torch.tensor(1.5)):
        for call in (lambda: ops.softmax(t, bad), lambda: ops.topk(t, bad), lambda: ops.topk(t, 2, axis=bad), lambda: ops.softmax_topk(t, bad),
                     lambda: ops.softmax_topk_sampling(t, bad), lambda: ops.softmax_reduce_max(t, bad), lambda: ops.reduce_max(t, bad)):
            with pytest.raises(TypeError):
                call()
    for k in (2, np.int64(2), torch.tensor(2)):  # taken, the axis outside the tensor refused
        with pytest.raises(IndexError):
            ops.topk(t, k, axis=np.int32(7))


@pytest.mark.parametrize("dtype,rows,n,chunk", [(capi.F32, 64, 128256, 16384), (capi.F32, 150, 8200, 16384), (capi.F16, 64, 65537, 16384),
                                                (capi.F32, 32, 33001, 8192), (capi.F32, 64, 200000, 10240), (capi.F16, 500, 33001, 10240)])
def test_softmax_of_long_rows_asks_for_a_record_a_chunk(lib, dtype, rows, n, chunk):
    """32 bytes behind the 64 KiB of counters for every chunk that the one-launch softmax splits a row into."""
    assert capi.softmax_workspace_bytes(dtype, (rows, n), -1) >= 65536 + rows * -(-n // chunk) * 32


def test_no_record_tag_is_that_of_a_cleared_word(lib):
    """The one-launch softmax takes a word with the launch's tag for arrived: none of a launch's four may be 0, which a cleared
    word has, nor alike, and a launch's are not those of the one before.  All launches until the tags come again, and across
    the counter's wrap."""
    import ctypes
    import numpy as np
    f = ctypes.CDLL(capi.BENCH_LIB_PATH).vkop_hip_measure_tags
    f.argtypes = [ctypes.c_uint, ctypes.c_uint, ctypes.c_void_p]
    at_once = 1 << 20
    tags = np.zeros((at_once, 4), np.uint32)
    for first in [i * at_once for i in range(18)] + [(1 << 32) - at_once // 2]:
        assert f(first, at_once, tags.ctypes.data) == 0
        assert tags.min() > 0 and tags.max() < 1 << 24, first
        for w in range(4):
            assert not np.any(tags[:, w] == tags[:, (w + 1) % 4]) and not np.any(tags[:, w] == tags[:, (w + 2) % 4]), first
            assert not np.any(tags[1:, w] == tags[:-1, w]), first


def test_native_front_end_takes_any_object_with_get_as_workspace():
    """A workspace is what its get(nbytes) returns: an object with nothing else, and a class derived from ops.Workspace with a
    get() of its own.  (The rest of the call needs a GPU; get() is called before.)"""
    torch = pytest.importorskip("torch")
    from torch._subclasses import FakeTensorMode
    from vkop_amd import capi, ops
    with FakeTensorMode():
        t = torch.empty(2, 100000, device="cuda")
    out = torch.empty(2, 100000)
    need = capi.softmax_workspace_bytes(capi.F32, (2, 100000), -1)
    assert need > 0

    class Asked(Exception):
        pass

    class Plain:
        def get(self, nbytes):
            raise Asked(nbytes)

    class Derived(ops.Workspace):
        def get(self, nbytes):
            raise Asked(nbytes)

    for ws in (Plain(), Derived()):
        with pytest.raises(Asked, match=str(need)):
            ops.softmax(t, out=out, workspace=ws)

    class Wrong:
        def __init__(self, answer):
            self.answer = answer

        def get(self, nbytes):
            return self.answer

    for answer in ((1, 2, 3), ("x", 1), (1.5, 1), 7):
        with pytest.raises((TypeError, ValueError)):
            ops.softmax(t, out=out, workspace=Wrong(answer))


@pytest.mark.parametrize("shape,axis", [((0, 5000, 7), 1), ((3, 5000, 0), 1), ((3, 300, 0), 1), ((0, 200000), 1), ((0, 100), 1),
                                        ((3, 0), 1), ((3, 0, 5), 1), ((0, 1000, 5), 1), ((0,), 0), ((2, 0, 3, 4), 2)])
def test_tensors_without_elements(lib, shape, axis):
    """No scratch is asked for and nothing launched (a plan that divided by its number of tiles ended the process)."""
    for dt in (capi.F32, capi.F16):
        assert capi.softmax_workspace_bytes(dt, shape, axis) == 0
        assert capi.softmax_reduce_max_workspace_bytes(dt, shape, axis) == 0
        capi.softmax(0, 0, dt, shape, axis)
        if shape[axis] != 0:
            capi.softmax_reduce_max(0, 0, dt, shape, axis)
            capi.topk(0, 0, 0, dt, shape, axis, min(5, shape[axis]))
            capi.softmax_topk(0, 0, 0, 0, dt, shape, axis, min(5, shape[axis]))


def test_native_front_end_knows_what_it_was_built_for(monkeypatch):
    torch = pytest.importorskip("torch")
    from vkop_amd import ops
    monkeypatch.setattr(ops, "_native", None)
    monkeypatch.setattr(torch, "__version__", "1.0.0")
    with pytest.raises(ImportError, match="built for torch"):
        ops.softmax(torch.zeros(2, 5))


def test_polynomial_of_the_exponential():
    """exp_accurate's polynomial interpolates e^r at the nine Chebyshev points of [-0.34662, 0.34662], the coefficients rounded
    to double: made again from that sentence in 60 digits, bit for bit, and its relative error on the interval is below 2^-39."""
    import re
    from decimal import Decimal as D, getcontext
    getcontext().prec = 60
    text = open(os.path.join(os.path.dirname(os.path.dirname(__file__)), "vkop_amd", "csrc", "device_utils.hpp")).read()
    body = text[text.index("float exp_accurate(float d)"):]
    body = body[:body.index("__double2hiint")]
    have = [float.fromhex(h) for h in re.findall(r"0x1\.[0-9a-f]+p-?\d+", body)]
    have.append(float(re.findall(r"p = fma\(p, r, (1\.0)\);", body)[0]))
    have.reverse()
    assert len(have) == 9

    def cos(x):
        s, t, i = D(0), D(1), 0
        while abs(t) > D(10) ** -58:
            s, i = s + t, i + 2
            t = -t * x * x / (i * (i - 1))
        return s
    pi = D("3.14159265358979323846264338327950288419716939937510582097494459")
    r_max = D("0.34662")
    pts = [r_max * cos(pi * (2 * i + 1) / 18) for i in range(9)]
    table = [p.exp() for p in pts]  # Newton's divided differences, then the powers' coefficients
    for step in range(1, 9):
        for i in range(8, step - 1, -1):
            table[i] = (table[i] - table[i - 1]) / (pts[i] - pts[i - step])
    coeff = [table[8]] + [D(0)] * 8
    for i in range(7, -1, -1):
        coeff = [table[i] - pts[i] * coeff[0]] + [coeff[j - 1] - pts[i] * coeff[j] for j in range(1, 9)]
    assert [float(c) for c in coeff] == have
    worst = D(0)
    for i in range(2001):
        r = r_max * (D(i) / 1000 - 1)
        p = D(0)
        for c in reversed(have):
            p = p * r + D(c)
        worst = max(worst, abs(p / r.exp() - 1))
    assert worst < D(2) ** -39
