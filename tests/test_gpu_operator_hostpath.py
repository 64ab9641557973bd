"""The native functions behind hostops.run_operator against the Python and ctypes path they stand in for: the same bits for every
operator whose passes or launch they carry, None for operands they do not take, the library's errors."""
import pytest
import torch

from heron_amd import backend as B
from heron_amd import hostops, instances
from heron_amd.ops.rocm import getOpFromName

pytestmark = pytest.mark.gpu

CASES = [("c1d", [2, 31, 40, 24, 3, 2, 1, 1]), ("c2d_nchw", [3, 9, 11, 24, 40, 3, 3, 1, 1, 1]), ("c2d_nchw", [1, 8, 8, 3, 16, 3, 3, 2, 1, 1]),
         ("c3d", [2, 5, 6, 7, 24, 40, 3, 3, 3, 1, 1, 1]), ("t2d", [2, 5, 7, 24, 40, 3, 3, 2, 1, 1, 1]), ("t2d", [2, 5, 7, 16, 24, 3, 3, 3, 1, 1, 0]),
         ("var", [3, 16, 9, 7]), ("mean", [3, 16, 9, 7]), ("dep", [2, 9, 11, 8, 16, 3, 3, 1, 1, 1])]


def _declared(op, args, dt):
    ctx = type("Ctx", (), dict(set_info=lambda self, i: setattr(self, "info", i), set_axis_map=lambda self, m: None))()
    getOpFromName(op)(ctx, *args, dt, dt)
    return ctx.info


def _python_only(monkeypatch):
    names = dict.fromkeys(("gemm", "conv2d", "channels_last", "gather", "conv_chw"), staticmethod(lambda *a: None))
    monkeypatch.setattr(B, "_ext", type("Declines", (), dict(names, stream=staticmethod(B.ext().stream))))


@pytest.mark.parametrize("kind", ["f16", "u8s8"])
@pytest.mark.parametrize("op,args", CASES, ids=["%s-%d" % (o, i) for i, (o, _) in enumerate(CASES)])
def test_same_bits(kind, op, args, hrn, monkeypatch):
    f16 = kind == "f16"
    if op in ("var", "mean", "dep") and not f16:
        pytest.skip("an fp16 operator")
    info = _declared(op, args, "float16" if f16 else "int8")
    ref = info["reference_args"]
    gen = torch.Generator(device="cuda").manual_seed(len(op))
    shapes = [s for s in (ref.get("input") or ref.get("In") or ref.get("A"), ref.get("filter") or ref.get("Mean") or ref.get("B")) if s]
    if f16:
        inputs = [torch.randn(s, device="cuda", generator=gen).half() for s in shapes]
    else:
        inputs = [torch.randint(0, 256, shapes[0], device="cuda", generator=gen, dtype=torch.uint8),
                  torch.randint(-128, 128, shapes[1], device="cuda", generator=gen, dtype=torch.int8)]
    conv = info["operator"] == "conv2d_nhwc"
    mod = B.Module(instances.D(instances.F16, instances.CONV, 128, 64, 128, 2, 1, 32, 2, 1, epi=1) if f16 and conv else
                   instances.D(instances.U8, instances.CONV, 128, 64, 128, 2, 2, 16, 3, 1, epi=1, colsum=1) if conv else instances.BEST["small_f16"])
    print("operator host path", op, args, kind, flush=True)
    got = hostops.run_operator(mod, info, inputs)
    _python_only(monkeypatch)
    want = hostops.run_operator(mod, info, inputs)
    assert got.shape == want.shape and got.dtype == want.dtype and torch.equal(got, want)
    mod.close()


def test_what_is_left_to_python(hrn):
    E = B.ext()
    x = torch.zeros(2, 8, 9, device="cuda").half()
    assert E.channels_last(x.transpose(1, 2), 8) is None and E.channels_last(x.cpu(), 8) is None and E.channels_last(x.double(), 8) is None
    assert E.channels_last(x[:0], 8) is None and E.channels_last(x, None) is None and E.channels_last(x, 8).shape == (2, 9, 8)
    assert E.channels_last(x, 4) not in (0, None) and type(E.channels_last(x, 4)) is int          # fewer channels than there are: refused
    out = torch.zeros(8, device="cuda").half()
    ok = (x, out, (8,), [(8, 9, {0: 1})], None, None, 0, None)
    assert E.gather(*ok) == 0
    for i, bad in [(0, x.cpu()), (1, None), (2, 8), (2, (1,) * 7), (3, [(8, 9)]), (3, [(8, 9, {1: 1})]), (3, []), (4, (1, 1)), (6, None), (7, 3)]:
        assert E.gather(*[bad if j == i else a for j, a in enumerate(ok)]) is None, (i, bad)
    assert E.gather(x, out, (8,), [(0, 9, {0: 1})], None, None, 0, None) == B.HRN_E_BADPARAM
