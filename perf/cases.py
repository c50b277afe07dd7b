"""Performance cases of the softmax -> top-k post-processing library.

Each case is one call -- or, for the detection chain, the two calls -- that a
program with logits or scores on the GPU makes through vkop_amd.ops: the fused
softmax -> top-k of a classifier or a language model, its sampling form, plain
top-k in both directions, plain softmax along the last and along another axis,
and the detection tail (class maximum, best anchors, non-maximum suppression;
the last through the C ABI, whose record buffer stays on the GPU).
Shapes are those of the operator benchmark, its sweeps and the tests;
draw() spreads over the same ranges.
"""
import math

import torch

from vkop_amd import capi, ops

DTYPES = {"f32": torch.float32, "f16": torch.float16}
ITEM = {"f32": 4, "f16": 2}
NMS_PER_CLASS = 100


def listed():
    return [
        # one image through a classifier head: the smallest call there is, all latency
        dict(name="classifier_1x1000_f32_k5", op="softmax_topk", rows=1, n=1000, k=5, dtype="f32"),
        # a batch of the same in half precision (the USE_FP16 build of the operators)
        dict(name="classifier_256x1000_f16_k5", op="softmax_topk", rows=256, n=1000, k=5, dtype="f16"),
        # one decoding step of a language model over a batch: the headline workload
        dict(name="vocab_64x128256_f32_k50", op="softmax_topk", rows=64, n=128256, k=50, dtype="f32"),
        # a decoding step that samples (temperature, top-p) over a vocabulary of odd size: rows start off 16 bytes
        dict(name="sampling_32x50257_f16_k40", op="sampling", rows=32, n=50257, k=40, scale=1.25, top_p=0.9, dtype="f16"),
        # candidates out of long score lists full of equal values
        dict(name="topk_ties_8x262144_f32_k1024", op="topk", rows=8, n=262144, k=1024, largest=True, data="grid",
             dtype="f32"),
        # the other direction: the nearest out of tens of thousands of distances
        dict(name="topk_smallest_64x32000_f32_k40", op="topk", rows=64, n=32000, k=40, largest=False, data="normal",
             dtype="f32"),
        # the whole probability tensor of a decoding step (scoring, distillation)
        dict(name="softmax_64x128256_f32", op="softmax", rows=64, n=128256, dtype="f32"),
        # attention weights of a vision transformer: short rows of odd length, hundreds of thousands of them
        dict(name="softmax_302592x197_f16", op="softmax", rows=128 * 12 * 197, n=197, dtype="f16"),
        # attention weights of a long sequence: the largest tensor
        dict(name="softmax_524288x1024_f16", op="softmax", rows=16 * 32 * 1024, n=1024, dtype="f16"),
        # per-pixel class probabilities of a segmentation head (softmax along the channels of NCHW)
        dict(name="softmax_axis1_8x21x262144_f32", op="softmax_axis1", batch=8, n=21, inner=512 * 512, dtype="f32"),
        # a detector's classification tail: best class probability per anchor, then the best anchors
        dict(name="detect_16x80x8400_f32_k300", op="detect", batch=16, classes=80, anchors=8400, k=300, dtype="f32"),
        # non-maximum suppression behind it: records and their number stay on the GPU, as in the C++ operator
        dict(name="nms_16x80x8400_f32", op="nms", batch=16, classes=80, anchors=8400, dtype="f32"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["softmax_topk", "softmax_topk", "sampling", "topk", "topk", "softmax", "softmax", "softmax_axis1",
                     "detect", "nms"])
    dtype = rng.choice(["f32", "f16"])
    if op == "softmax_topk":    # classifier heads to vocabularies, one row to a serving batch
        n = _log_int(rng, 100, 262144)
        return dict(op=op, rows=_log_int(rng, 1, 256), n=n, k=_log_int(rng, 1, min(500, n // 4)), dtype=dtype)
    if op == "sampling":        # vocabularies
        return dict(op=op, rows=_log_int(rng, 1, 256), n=_log_int(rng, 8192, 262144), k=_log_int(rng, 5, 100),
                    scale=rng.choice([1.0, 1.25, 1.4286]), top_p=rng.choice([0.8, 0.9, 0.95]), dtype=dtype)
    if op == "topk":
        n = _log_int(rng, 500, 262144)
        return dict(op=op, rows=_log_int(rng, 1, 256), n=n, k=_log_int(rng, 1, min(1024, n // 8)),
                    largest=rng.random() < 0.6, data=rng.choice(["normal", "normal", "grid"]), dtype=dtype)
    if op == "softmax":         # up to half of the largest listed tensor
        n = _log_int(rng, 32, 262144)
        return dict(op=op, rows=_log_int(rng, max(1, 65536 // n), (1 << 28) // n // (2 if dtype == "f32" else 1)), n=n,
                    dtype=dtype)
    if op == "softmax_axis1":   # channels of an image, classes of a detector, sequences
        n = _log_int(rng, 4, 1024)
        batch = _log_int(rng, 1, 32)
        return dict(op=op, batch=batch, n=n, inner=_log_int(rng, 64, min(512 * 512, (1 << 26) // (n * batch))), dtype=dtype)
    batch, classes = _log_int(rng, 1, 32), _log_int(rng, 20, 91)
    anchors = _log_int(rng, 1000, 8400 * 2)
    if op == "detect":
        return dict(op=op, batch=batch, classes=classes, anchors=anchors, k=rng.randint(100, 300), dtype=dtype)
    return dict(op=op, batch=min(batch, 16), classes=classes, anchors=min(anchors, 8400), dtype=dtype)


def _randn(gen, shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _logits(gen, rows, n):
    """Short rows: a classifier head's logits, N(0, 3^2).  Long rows: a vocabulary's, N(0, 1) with one to three
    values 6 to 10 above the rest in every row, over a temperature of 0.8."""
    x = _randn(gen, (rows, n))
    if n < 4096:
        return x.mul_(3.0)
    where = torch.randint(0, n, (rows, 3), generator=gen, device="cuda")
    lift = 6.0 + 4.0 * torch.rand((rows, 3), generator=gen, device="cuda")
    lift[:, 1:] *= (torch.rand((rows, 2), generator=gen, device="cuda") < 0.5).float()
    return x.scatter_add_(1, where, lift).mul_(1.25)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    op, dtype = case["op"], DTYPES[case["dtype"]]
    s = dict(op=op)
    if op in ("softmax_topk", "sampling"):
        s.update(x=_logits(gen, case["rows"], case["n"]).to(dtype), k=case["k"])
        if op == "sampling":
            s.update(scale=case["scale"], top_p=case["top_p"])
    elif op == "topk":
        shape = (case["rows"], case["n"])
        if case["data"] == "grid":  # 513 distinct values: quantised scores
            x = torch.randint(-256, 257, shape, generator=gen, device="cuda").float() / 64.0
        else:
            x = _randn(gen, shape)
        s.update(x=x.to(dtype), k=case["k"], largest=case["largest"])
    elif op == "softmax":
        x = torch.empty((case["rows"], case["n"]), dtype=dtype, device="cuda")
        x.normal_(0.0, 1.25, generator=gen)
        s.update(x=x)
    elif op == "softmax_axis1":
        s.update(x=_randn(gen, (case["batch"], case["n"], case["inner"])).mul_(2.0).to(dtype))
    else:
        # class scores of a detection head: N(-4, 2^2)
        x = _randn(gen, (case["batch"], case["classes"], case["anchors"])).mul_(2.0).sub_(4.0)
        if op == "detect":
            s.update(x=x.to(dtype), k=case["k"])
        else:
            centre = torch.rand((case["batch"], case["anchors"], 2), generator=gen, device="cuda")
            half = 0.1 * torch.rand((case["batch"], case["anchors"], 2), generator=gen, device="cuda")
            s.update(boxes=torch.cat([centre - half, centre + half], dim=-1).to(dtype).contiguous(),
                     scores=torch.softmax(x, dim=1).to(dtype).contiguous())
            shape = (case["batch"], case["classes"], case["anchors"])
            s.update(shape=shape, dtype=capi.F32 if dtype == torch.float32 else capi.F16, workspace=ops.Workspace(),
                     records=torch.zeros((shape[0] * shape[1] * NMS_PER_CLASS, 3), dtype=torch.int32, device="cuda"),
                     count=torch.zeros(2, dtype=torch.int32, device="cuda"))
            s["ws"] = s["workspace"].get(capi.nms_workspace_bytes(*shape, NMS_PER_CLASS))
    return s


def run(s):
    op = s["op"]
    if op == "softmax_topk":
        return ops.softmax_topk(s["x"], s["k"])
    if op == "sampling":
        return ops.softmax_topk_sampling(s["x"], s["k"], s["scale"], s["top_p"])
    if op == "topk":
        return ops.topk(s["x"], s["k"], largest=s["largest"])
    if op == "softmax":
        return ops.softmax(s["x"])
    if op == "softmax_axis1":
        return ops.softmax(s["x"], axis=1)
    if op == "detect":
        best = ops.softmax_reduce_max(s["x"], 1)
        return best, ops.topk(best, s["k"])
    capi.nms(s["boxes"].data_ptr(), s["scores"].data_ptr(), s["records"].data_ptr(), s["records"].shape[0],
             s["count"].data_ptr(), s["dtype"], *s["shape"], 0, NMS_PER_CLASS, 0.45, 0.25, *s["ws"],
             torch.cuda.current_stream().cuda_stream)
    return s["records"], s["count"]


def work(case):
    """Every input read once, every output written once; per element of a softmax a difference, an exponential and an
    addition, per element of a selection one comparison."""
    op, item = case["op"], ITEM[case["dtype"]]
    if op in ("softmax_topk", "sampling", "topk"):
        e, out = case["rows"] * case["n"], case["rows"] * case["k"]
        counts = 4 * case["rows"] if op == "sampling" else 0
        return {"bytes": e * item + out * (item + 4) + counts, "flops": e * (1 if op == "topk" else 4)}
    if op == "softmax":
        e = case["rows"] * case["n"]
        return {"bytes": 2 * e * item, "flops": 5 * e}
    if op == "softmax_axis1":
        e = case["batch"] * case["n"] * case["inner"]
        return {"bytes": 2 * e * item, "flops": 5 * e}
    e = case["batch"] * case["classes"] * case["anchors"]
    if op == "detect":
        return {"bytes": e * item + case["batch"] * (case["anchors"] * item + case["k"] * (item + 4)), "flops": 4 * e}
    return {"bytes": e * item + case["batch"] * case["anchors"] * 4 * item, "flops": e}


def tolerance(case):
    """Against the same path in 64 bits (48 cases of these ranges): single precision rel 9e-8, max 3.6e-7; half
    precision rel 2.3e-5, max 1e-3 (a unit of a half), and on rows of 130000, whose probabilities are subnormal halves,
    4e-3 (1.6e-2 is a unit at 1 / 262144).  No index differed; where two probabilities round to the same value in one
    implementation and not in the other, a pair of indices changes places."""
    if case["op"] in ("topk", "nms"):
        return "exact"  # copies of input elements, and indices
    if case["dtype"] == "f32":
        return {"rel": 4e-7, "max": 1.5e-6, "differ": 2e-4}
    return {"rel": 1e-4, "max": 2e-2, "differ": 2e-4}
