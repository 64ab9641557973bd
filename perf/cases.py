"""Performance cases of the framework: what a program that uses the tuned kernels has them do.

Every case goes through the entry points such a program calls: ``tuned.load`` / ``instances`` name a template instance,
``backend.Module`` loads it, and ``hostops.gemm``, ``hostops.conv2d_nhwc``, ``hostops.run_operator`` or
``hostops.OperatorPlan.run`` is called once per pass.  Shapes that have a tuned record of their own use it; any other
shape uses the record or the shipped general-purpose instance of its size class (``_gemm_instance``,
``_conv_instance``), as a program without a search of its own does.  All inputs are made on the GPU from the seed.

Case fields: ``family`` gemm | bmm | conv | op, ``dtype`` f16 | u8s8, and the sizes of the family.  An ``op`` case names
an operator of the registry, its shape arguments as text, and whether the call is replayed from an ``OperatorPlan``.
"""
import math

import torch

from heron_amd import backend, hostops, instances, tuned
from heron_amd.ops.rocm import getOpFromName

F16, U8, GEMM, CONV, D = instances.F16, instances.U8, instances.GEMM, instances.CONV, instances.D


def _gemm(name, dtype, m, n, k):
    return dict(name=name, family="gemm", dtype=dtype, m=m, n=n, k=k)


def _bmm(name, dtype, b, m, n, k, softmax=False):
    return dict(name=name, family="bmm", dtype=dtype, b=b, m=m, n=n, k=k, softmax=softmax)


def _conv(name, dtype, n, h, w, ci, co, kh, kw, stride, pad, dil):
    return dict(name=name, family="conv", dtype=dtype, n=n, h=h, w=w, ci=ci, co=co, kh=kh, kw=kw, stride=stride, pad=pad, dil=dil)


def _op(name, dtype, op, args, plan):
    return dict(name=name, family="op", dtype=dtype, op=op, args=",".join(str(a) for a in args), plan=plan)


def listed():
    return [
        # the quick-start product: nothing but the latency of one call
        _gemm("gemm-u8s8-64", "u8s8", 64, 64, 64),
        # a classifier / projection layer at batch 32: few output tiles and a long K, so K is split over workgroups
        _gemm("gemm-f16-32x4096x4096", "f16", 32, 4096, 4096),
        # an ordinary quantized product whose sizes fit no tile
        _gemm("gemm-u8s8-ragged", "u8s8", 1111, 1500, 2064),
        # the dense products the benchmark is quoted on
        _gemm("gemm-f16-4096", "f16", 4096, 4096, 4096),
        _gemm("gemm-f16-8192", "f16", 8192, 8192, 8192),
        _gemm("gemm-u8s8-8192", "u8s8", 8192, 8192, 8192),
        # attention of a BERT-base layer at batch 16, 12 heads: scores, then scores times values
        _bmm("bmm-f16-scores", "f16", 192, 512, 512, 64),
        _bmm("bmm-f16-values", "f16", 192, 512, 64, 512, softmax=True),
        # ResNet-50 stage 2 at batch 32, in both element types
        _conv("conv-f16-56x56x64", "f16", 32, 56, 56, 64, 64, 3, 3, 1, 1, 1),
        _conv("conv-u8s8-56x56x64", "u8s8", 32, 56, 56, 64, 64, 3, 3, 1, 1, 1),
        # channels-first 1-D convolution: layout change, product, layout change back, called eagerly
        _op("c1d-ncw-f16", "f16", "c1d", [16, 892, 512, 512, 3, 1, 4, 1], False),
        # channels-first transposed convolution with stride 2, recorded once and replayed
        _op("t2d-f16-plan", "f16", "t2d", [16, 56, 56, 64, 128, 1, 1, 2, 0, 1, 0], True),
    ]


def _log(rng, lo, hi, step):
    """A multiple of ``step`` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def draw(rng):
    family = rng.choice(["gemm", "gemm", "bmm", "conv", "op"])
    dtype = rng.choice(["f16", "u8s8"])
    kq = 8 if dtype == "f16" else 16                       # rows of K are whole 16-byte chunks
    while True:
        if family == "gemm":
            c = _gemm("", dtype, _log(rng, 17, 8192, 1), _log(rng, 64, 8192, 8), _log(rng, 64, 8192, kq))
        elif family == "bmm":
            if rng.random() < 0.5:
                c = _bmm("", dtype, _log(rng, 4, 192, 1), _log(rng, 64, 768, 1), _log(rng, 64, 768, 8), rng.choice([64, 128]))
            else:
                c = _bmm("", dtype, _log(rng, 4, 192, 1), _log(rng, 64, 768, 1), rng.choice([64, 128]), _log(rng, 64, 768, kq),
                         softmax=dtype == "f16")
        elif family == "conv":
            hw = _log(rng, 7, 80, 1)
            k, stride, dil = rng.choice([1, 3, 3, 3, 5]), rng.choice([1, 1, 1, 2]), rng.choice([1, 1, 1, 2])
            c = _conv("", dtype, _log(rng, 1, 32, 1), hw, max(7, hw + rng.choice([0, 0, -1, 3])), _log(rng, 32, 512, 16),
                      _log(rng, 32, 512, 16), k, k, stride, (k // 2) * dil, dil)
            if c["h"] + 2 * c["pad"] < (k - 1) * dil + 1 or c["w"] + 2 * c["pad"] < (k - 1) * dil + 1:
                continue
        else:
            op = rng.choice(["c1d", "c2d_nchw", "t2d", "c3d", "gemv", "var"])
            n, hw, ci, co = _log(rng, 1, 16, 1), _log(rng, 7, 56, 1), _log(rng, 16, 256, 8), _log(rng, 32, 256, 16)
            k = rng.choice([1, 3])
            if op == "c1d":
                args = [n, _log(rng, 100, 900, 1), 2 * ci, 2 * co, k, rng.choice([1, 2]), k // 2, 1]
            elif op == "c2d_nchw":
                args = [n, hw, hw, ci, co, k, k, rng.choice([1, 2]), k // 2, 1]
            elif op == "t2d":
                args = [n, hw, hw, ci, co, k, k, rng.choice([1, 2]), k // 2, 1, 0]
            elif op == "c3d":
                args = [max(1, n // 2), rng.choice([2, 4, 8]), hw, hw, ci, co, k, k, k, rng.choice([1, 2]), k // 2, 1]
            elif op == "gemv":
                args = [_log(rng, 64, 8192, 1), _log(rng, 64, 8192, 1)]
            else:
                dtype, args = "f16", [n, ci, hw, hw]
            c = _op("", dtype, op, args, rng.random() < 0.5)
        w = work(c)
        if w["flops"] <= 1.1e12 and w["bytes"] <= 1.2e9:
            del c["name"]
            return c


# ------------------------------------------------------------------------------------------------ instances
def _tuned(name):
    t = tuned.load(name)
    return t.desc, t.group_m, 0


def _gemm_instance(dtype, m, n, k, batch=1):
    """(descriptor, raster group, K slices).  A shape that fills the chip with 256-row tiles takes the tuned record of the
    square products; fewer tiles take the shipped 128-row, split-K (long K only) and 64-row instances, in this order."""
    f16 = dtype == "f16"

    def tiles(t):
        return batch * -(-m // t) * -(-n // t)

    if tiles(256) >= 128:
        return _tuned(("gemm_f16_8192" if m * n > 4096 * 4096 else "gemm_f16_4096") if f16 else "gemm_u8s8_8192")
    if tiles(128) >= 96:
        return (D(F16, GEMM, 128, 128, 128, 2, 2, 32, 2, 1, nt=1) if f16 else
                D(U8, GEMM, 128, 128, 128, 2, 2, 16, 2, 1, epi=1, colsum=1, nt=1)), 8, 0
    kt = -(-k * (2 if f16 else 1) // 128)
    slices = min(256 // tiles(64) if tiles(64) else 1, kt // 4)
    if batch == 1 and slices > 1:
        return instances.splitk_descs()[0 if f16 else 6], 8, slices
    return instances.BEST["small_f16" if f16 else "small"], 8, 0


def _bmm_instance(dtype, b, m, n, k):
    """Short K with wide results: the tuned scores record; narrow results: the tuned values record (fp16)."""
    if dtype == "f16" and n > 128 and k <= 128:
        return _tuned("bmm_f16_qk")
    if dtype == "f16" and n <= 128:
        return _tuned("bmm_f16_pv")
    return _gemm_instance(dtype, m, n, k, b)


def _conv_instance(dtype, n, h, w, ci, co, kh, kw, sh, sw, ph, pw, dh, dw):
    """The tuned ResNet record where its input window fits into LDS, else the shipped im2col instances, with K split where
    the output tiles alone leave most of the chip idle."""
    f16 = dtype == "f16"
    es = 2 if f16 else 1
    t = tuned.load("conv2d_f16_resnet" if f16 else "conv2d_u8s8_resnet")
    d = t.desc
    rows = d.bm + 2 * (ph * w + pw)
    same = (sh, sw, dh, dw) == (1, 1, 1, 1) and 2 * ph == kh - 1 and 2 * pw == kw - 1
    window = -(-rows * ci * es // 1024) * 1024
    if same and co <= 128 and ci * es % d.bkb == 0 and window + d.stages * d.bn * d.bkb <= 160 * 1024:
        return d, t.group_m, 0
    ho, wo = (h - ((kh - 1) * dh + 1) + 2 * ph) // sh + 1, (w - ((kw - 1) * dw + 1) + 2 * pw) // sw + 1
    kt = -(-kh * kw * ci * es // 128)
    tiles = -(-n * ho * wo // 64) * -(-co // 64)
    if tiles <= 128 and kt >= 8:
        return instances.splitk_descs()[4 if f16 else 5], 8, min(256 // tiles, kt // 4)
    if f16:
        if co >= 128:
            return D(F16, CONV, *instances.PARITY_SHAPES[2]), 8, 0
        return D(F16, CONV, 128, 64, 128, 2, 1, 32, 2, 1, epi=1), 8, 0
    return D(U8, CONV, 128, 64, 128, 2, 2, 16, 3, 1, epi=1, colsum=1), 8, 0


_modules = {}


def _module(desc):
    """A program loads each kernel once."""
    key = desc.as_tuple()
    if key not in _modules:
        _modules[key] = backend.Module(desc)
    return _modules[key]


# ------------------------------------------------------------------------------------------------ inputs
class _Ctx:
    """What an operator definition is declared on: it keeps the ``info`` dictionary ``run_operator`` takes."""

    def set_info(self, info):
        self.info = info

    def set_axis_map(self, m):
        self.axis_map = m


def _declare(case):
    dt = "float16" if case["dtype"] == "f16" else "int8"
    ctx = _Ctx()
    getOpFromName(case["op"])(ctx, *[int(a) for a in case["args"].split(",")], dt, dt)
    return ctx.info


def _activation(gen, dtype, shape, scale=1.0, relu=False):
    """uint8 over its whole range, or fp16 N(0, scale) (half of it zero after a ReLU)."""
    if dtype == "u8s8":
        return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=gen)
    x = torch.randn(shape, dtype=torch.float32, device="cuda", generator=gen)
    return (x.clamp_(min=0) if relu else x.mul_(scale)).half()


def _weights(gen, dtype, shape, scale):
    if dtype == "u8s8":
        return torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=gen)
    return torch.randn(shape, dtype=torch.float32, device="cuda", generator=gen).mul_(scale).half()


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    dt, family = case["dtype"], case["family"]
    if family == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        desc, group, split = _gemm_instance(dt, m, n, k)
        A, W = _activation(gen, dt, (m, k), 0.1), _weights(gen, dt, (n, k), 0.1)
    elif family == "bmm":
        b, m, n, k = case["b"], case["m"], case["n"], case["k"]
        desc, group, split = _bmm_instance(dt, b, m, n, k)
        A, W = _activation(gen, dt, (b, m, k)), _weights(gen, dt, (b, n, k), 1.0)
        if case["softmax"]:
            A = torch.softmax(A.float(), -1).half()
    elif family == "conv":
        s, p, d = case["stride"], case["pad"], case["dil"]
        desc, group, split = _conv_instance(dt, case["n"], case["h"], case["w"], case["ci"], case["co"], case["kh"], case["kw"],
                                            s, s, p, p, d, d)
        A = _activation(gen, dt, (case["n"], case["h"], case["w"], case["ci"]), relu=True)
        W = _weights(gen, dt, (case["co"], case["kh"], case["kw"], case["ci"]), 0.05)
    else:
        return _prepare_op(case, gen)
    mod = _module(desc)
    # the weights are fixed, so their column sums (uint8 path) are made with them; a batched right-hand side is not a weight
    bsum = hostops.column_sums(W) if desc.colsum and family != "bmm" else None
    return dict(case=case, mod=mod, A=A, W=W, group=group, split=split, bsum=bsum)


def _prepare_op(case, gen):
    dt, info = case["dtype"], _declare(case)
    ref = info["reference_args"]
    first = ref.get("input") or ref.get("A") or ref.get("In")
    second = ref.get("filter") or ref.get("B") or ref.get("Mean")
    inputs = [_activation(gen, dt, first, relu="filter" in ref)]
    if case["op"] == "var":
        inputs.append(inputs[0].float().mean(dim=(0, 2, 3), keepdim=True).expand(first).half().contiguous())
    else:
        inputs.append(_weights(gen, dt, second, 0.05 if "filter" in ref else 0.1))
    if info["operator"] == "conv2d_nhwc":
        c = info["conv"]
        desc, group, split = _conv_instance(dt, c["N"], c["H"], c["W"], c["CI"], c["CO"], c["KH"], c["KW"], c["stride"], c["stride_w"],
                                            c["pad"], c["pad_w"], c["dil"], c["dil_w"])
    else:
        g = info["gemm_view"]
        desc, group, split = _gemm_instance(dt, g["M"], g["N"], g["K"], g["batch"])
    mod = _module(desc)
    if case["plan"]:
        return dict(case=case, plan=hostops.OperatorPlan(mod, info, inputs, group_m=group, split_k=split))
    constant = hostops.prepare_constant(info, inputs)
    bsum = hostops.column_sums(constant) if desc.colsum else None
    return dict(case=case, mod=mod, info=info, inputs=inputs, group=group, split=split, constant=constant, bsum=bsum)


def run(state):
    if "plan" in state:
        return state["plan"].run()
    if "info" in state:
        return hostops.run_operator(state["mod"], state["info"], state["inputs"], group_m=state["group"], split_k=state["split"],
                                    constant=state["constant"], bsum=state["bsum"])
    case = state["case"]
    if case["family"] == "conv":
        return hostops.conv2d_nhwc(state["mod"], state["A"], state["W"], case["stride"], case["pad"], case["dil"],
                                   group_m=state["group"], split_k=state["split"], bsum=state["bsum"])
    return hostops.gemm(state["mod"], state["A"], state["W"], group_m=state["group"], split_k=state["split"], bsum=state["bsum"])


# ------------------------------------------------------------------------------------------------ work and tolerance
def work(case):
    """Bytes: every input read once, the result written once.  Operations: the products the definition asks for."""
    f16 = case["dtype"] == "f16"
    es, oes = (2, 2) if f16 else (1, 4)
    if case["family"] in ("gemm", "bmm"):
        b, m, n, k = case.get("b", 1), case["m"], case["n"], case["k"]
        return dict(bytes=b * ((m * k + n * k) * es + m * n * oes), flops=2 * b * m * n * k)
    if case["family"] == "conv":
        c, d = case, case["dil"]
        ho = (c["h"] - ((c["kh"] - 1) * d + 1) + 2 * c["pad"]) // c["stride"] + 1
        wo = (c["w"] - ((c["kw"] - 1) * d + 1) + 2 * c["pad"]) // c["stride"] + 1
        out, taps = c["n"] * ho * wo * c["co"], c["kh"] * c["kw"] * c["ci"]
        return dict(bytes=(c["n"] * c["h"] * c["w"] * c["ci"] + c["co"] * taps) * es + out * oes, flops=2 * out * taps)
    info = _declare(case)
    ref = info["reference_args"]
    if case["op"] == "gemv":
        m, k = ref["A"]
        return dict(bytes=(m * k + k) * es + m * 8 * oes, flops=2 * m * k)
    if case["op"] == "var":
        e = math.prod(ref["In"])
        return dict(bytes=2 * e * es + ref["In"][1] * 8 * oes, flops=4 * e)
    c = info["conv"]
    out = c["N"] * c["HO"] * c["WO"] * c["CO"]
    ci_taps = math.prod(ref["filter"]) // c["CO"]
    byts = (math.prod(ref["input"]) + math.prod(ref["filter"])) * es + out * oes
    if case["op"] == "t2d":                                 # every input element meets every tap once; inserted zeros do not count
        return dict(bytes=byts, flops=2 * math.prod(ref["input"]) * c["CO"] * c["KH"] * c["KW"])
    return dict(bytes=byts, flops=2 * out * ci_taps)


def tolerance(case):
    """Integer results are exact.  fp16 results carry one rounding of an fp32 sum: against the same product in float64 the
    relative error is 2.1e-4 and the largest difference 4.9e-4 of the value; four times that."""
    if case["dtype"] == "u8s8":
        return "exact"
    return dict(rel=8e-4, max=2e-3)
