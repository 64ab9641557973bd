"""What the native host path of hostops hands back or refuses, beside the plain calls the parity tests make."""
import pytest
import torch

from heron_amd import backend as B
from heron_amd import hostops, instances
from heron_amd.ops.rocm import getOpFromName

pytestmark = pytest.mark.gpu

D, F16, U8, GEMM, CONV = instances.D, instances.F16, instances.U8, instances.GEMM, instances.CONV
CONV_F16 = D(F16, CONV, *instances.PARITY_SHAPES[2])


def half(*shape):
    return torch.ones(shape, device="cuda", dtype=torch.float16)


def declared(op, args, dtype="float16"):
    ctx = type("Ctx", (), dict(set_info=lambda self, i: setattr(self, "info", i), set_axis_map=lambda self, m: None))()
    getOpFromName(op)(ctx, *args, dtype, dtype)
    return ctx.info


# the dilated filter is larger than the padded input by less than the stride, by the stride and by more than it; in one direction
@pytest.mark.parametrize("h,w,k,stride,pad,dil", [(4, 4, 5, 2, 0, 1), (4, 9, 5, 2, 0, 1), (9, 4, 5, 2, 0, 1), (3, 3, 5, 2, 0, 1), (1, 1, 5, 2, 0, 1),
                                                  (4, 4, 3, 3, 0, 2), (2, 2, 5, 4, 1, 1)])
def test_filter_larger_than_the_input_is_refused(h, w, k, stride, pad, dil, hrn):
    mod = B.Module(CONV_F16)
    X, W = half(2, h, w, 64), half(8, k, k, 64)
    print("empty", h, w, k, stride, pad, dil, flush=True)
    for out in (None, half(2, 1, 1, 8)):
        with pytest.raises((B.HeronRocmError, RuntimeError)):
            hostops.conv2d_nhwc(mod, X, W, stride, pad, dil, out=out)
        if out is not None:
            assert torch.equal(out, half(2, 1, 1, 8))
    # the same layer channels first, declared for a larger image
    info = declared("c2d_nchw", [2, 16, 16, 64, 8, k, k, stride, pad, dil])
    with pytest.raises((B.HeronRocmError, RuntimeError)):
        hostops.run_operator(mod, info, [half(2, 64, h, w), half(8, 64, k, k)])
    mod.close()


@pytest.mark.parametrize("entry", ["gemm", "conv2d"])
def test_other_threads_run_during_a_call(entry, hrn):
    """With no forced switch of the interpreter lock another thread gets on only where a call gives the lock up."""
    import sys
    import threading
    import time
    if entry == "gemm":
        mod, args = B.Module(instances.BEST["small_f16"]), (half(512, 512), half(512, 512))
        call = hostops.gemm
    else:
        mod, args = B.Module(CONV_F16), (half(4, 28, 28, 64), half(64, 3, 3, 64), 1, 1, 1)
        call = hostops.conv2d_nhwc
    turns, stop = [0], []

    def other():
        while not stop:
            turns[0] += 1
            time.sleep(0)

    out = call(mod, *args)
    thread, interval = threading.Thread(target=other), sys.getswitchinterval()
    try:
        sys.setswitchinterval(1000.0)
        thread.start()
        before, end = turns[0], time.monotonic() + 5.0
        while turns[0] == before and time.monotonic() < end:
            call(mod, *args, out=out)
        ran = turns[0] - before
    finally:
        sys.setswitchinterval(interval)
        stop.append(True)
        thread.join()
    torch.cuda.synchronize()
    assert ran > 0
    mod.close()


def test_out_of_memory_keeps_its_type(hrn):
    """A result that no card holds: torch's allocator refuses it and its exception arrives as such."""
    mod = B.Module(instances.BEST["small_f16"])
    A = half(1 << 20, 16)                       # 2 TiB of results
    with pytest.raises(torch.OutOfMemoryError):
        hostops.gemm(mod, A, A)
    mod.close()
    mod = B.Module(CONV_F16)
    X, W = half(1 << 18, 2, 2, 16), half(1 << 20, 1, 1, 16)
    with pytest.raises(torch.OutOfMemoryError):
        hostops.conv2d_nhwc(mod, X, W)
    mod.close()


@pytest.mark.parametrize("entry", ["gemm", "bmm", "conv2d"])
def test_results_of_the_caller(entry, hrn):
    """``out`` is any contiguous tensor of the result's type with room for it; everything else is refused before a launch."""
    if entry == "conv2d":
        mod, args, shape, call = B.Module(CONV_F16), (half(2, 5, 7, 64), half(8, 3, 3, 64), 1, 1, 1), (2, 5, 7, 8), hostops.conv2d_nhwc
    else:
        b = (3,) if entry == "bmm" else ()
        mod, args, shape, call = B.Module(instances.BEST["small_f16"]), (half(*b, 33, 64), half(*b, 40, 64)), b + (33, 40), hostops.gemm
    want = call(mod, *args)
    assert want.shape == shape
    n = want.numel()
    for out in (torch.zeros_like(want), torch.zeros(n, device="cuda").half(), torch.zeros(n + 5, device="cuda").half()):
        got = call(mod, *args, out=out)
        assert got is out and torch.equal(out.flatten()[:n], want.flatten()) and not out.flatten()[n:].any()
    wide = torch.zeros(shape[:-1] + (2 * shape[-1],), device="cuda").half()
    for out in (torch.zeros(shape, dtype=torch.float16), torch.zeros(n - 1, device="cuda").half(), wide[..., :shape[-1]],
                torch.zeros(shape, device="cuda"), torch.zeros(shape, device="cuda", dtype=torch.bfloat16)):
        with pytest.raises(ValueError):
            call(mod, *args, out=out)
        assert not out.any()
    mod.close()


CHANNELS_FIRST = {"c1d": [2, 9, 64, 8, 3, 1, 1, 1], "c2d_nchw": [2, 5, 6, 64, 8, 3, 3, 1, 1, 1], "c3d": [2, 3, 5, 6, 16, 8, 3, 3, 3, 1, 1, 1],
                  "t2d": [2, 5, 6, 64, 8, 3, 3, 2, 1, 1, 0]}


@pytest.mark.parametrize("op", sorted(CHANNELS_FIRST))
def test_slices_of_k_need_an_instance_built_for_them(op, hrn):
    mod, info = B.Module(CONV_F16), declared(op, CHANNELS_FIRST[op])
    X, F = half(*info["reference_args"]["input"]), half(*info["reference_args"]["filter"])
    want = hostops.run_operator(mod, info, [X, F])
    assert torch.equal(hostops.run_operator(mod, info, [X, F], split_k=1), want)
    for split_k in (2, 8):
        with pytest.raises(B.HeronRocmError):
            hostops.run_operator(mod, info, [X, F], split_k=split_k)
    mod.close()


@pytest.mark.parametrize("op", sorted(CHANNELS_FIRST))
def test_no_images_are_refused_by_the_library(op, hrn):
    mod, info = B.Module(CONV_F16), declared(op, CHANNELS_FIRST[op])
    empty = half(0, *info["reference_args"]["input"][1:])
    with pytest.raises(B.HeronRocmError):
        hostops.run_operator(mod, info, [empty, half(*info["reference_args"]["filter"])])
    mod.close()


@pytest.mark.parametrize("images", [1, 3, 4])
def test_volumes_of_another_number_than_declared_are_refused(images, hrn):
    """conv3d takes the number of volumes from its declaration; the result has room for those."""
    mod, info = B.Module(CONV_F16), declared("c3d", CHANNELS_FIRST["c3d"])
    shape = info["reference_args"]["input"]
    assert shape[0] == 2
    with pytest.raises(RuntimeError):
        hostops.run_operator(mod, info, [half(images, *shape[1:]), half(*info["reference_args"]["filter"])])
    mod.close()


@pytest.mark.parametrize("shape", [(2, 64, 7, 6), (2, 64, 5, 9), (3, 64, 8, 8), (1, 64, 2, 3)])
def test_transposed_conv_of_another_image_than_declared(shape, hrn):
    """The expanded image has the declared extents: pixels beyond them are dropped, missing ones are zeros."""
    mod, info = B.Module(CONV_F16), declared("t2d", CHANNELS_FIRST["t2d"])
    gen = torch.Generator(device="cuda").manual_seed(shape[2])
    X = torch.randn(shape, device="cuda", generator=gen).half()
    F = torch.randn(info["reference_args"]["filter"], device="cuda", generator=gen).half()
    c = info["conv"]
    act, const, fin = hostops.ADAPTERS[info["adapter"]]
    want = fin(info, hostops.conv2d_nhwc(mod, act(info, X, F), const(info, X, F), 1, 0, (c["dil"], c["dil_w"])))
    assert torch.equal(hostops.run_operator(mod, info, [X, F]), want)
    mod.close()


def test_a_recorded_split_k_plan_owns_its_workspace(hrn):
    mod, info = B.Module(instances.splitk_descs()[4]), declared("c2d_nchw", [2, 7, 7, 64, 64, 3, 3, 1, 1, 1])
    gen = torch.Generator(device="cuda").manual_seed(5)
    X = torch.randn(info["reference_args"]["input"], device="cuda", generator=gen).half()
    F = torch.randn(info["reference_args"]["filter"], device="cuda", generator=gen).half()
    plan = hostops.OperatorPlan(mod, info, [X, F], split_k=3)
    want = plan.run().clone()
    bound = [a.workspace for _, args in plan.steps for a in args if isinstance(a, B.Problem)]
    assert bound and all(any(b.data_ptr() <= w < b.data_ptr() + b.numel() * b.element_size() for b in plan.buffers) for w in bound)
    # a larger launch of the same module in between, and fresh tensors on whatever memory it freed
    p = B.conv2d_problem(64, 28, 28, 64, 64, 3, 3, 1, 1, 1, split_k=3)
    big = half(64, 28, 28, 64), half(64, 3, 3, 64), half(64, 28, 28, 64)
    mod.launch(p, *(t.data_ptr() for t in big), hostops._stream())
    other = [torch.full((1 << 18,), 7.0, device="cuda") for _ in range(8)]
    plan.out.zero_()
    assert torch.equal(plan.run(), want)
    assert all(bool((t == 7.0).all()) for t in other)
    mod.close()


@pytest.mark.parametrize("captured", [False, True])
def test_channels_first_kernels_of_an_instance_not_prepared_for_them(captured, hrn, tmp_path, monkeypatch):
    """hrn_build finds no such code objects in the cache: the first launch compiles and loads them, also inside a capture."""
    monkeypatch.setenv("HRN_CACHE_DIR", str(tmp_path))
    mod, full = B.Module(CONV_F16), {}
    monkeypatch.undo()
    ready = B.Module(CONV_F16)
    monkeypatch.setenv("HRN_CACHE_DIR", str(tmp_path))
    for op in ("c2d_nchw", "t2d"):
        info = declared(op, CHANNELS_FIRST[op])
        gen = torch.Generator(device="cuda").manual_seed(11)
        X = torch.randn(info["reference_args"]["input"], device="cuda", generator=gen).half()
        F = torch.randn(info["reference_args"]["filter"], device="cuda", generator=gen).half()
        weights = hostops.prepare_constant(info, [X, F])
        want = hostops.run_operator(ready, info, [X, F], constant=weights)
        torch.cuda.synchronize()
        if captured:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                got = hostops.run_operator(mod, info, [X, F], constant=weights)
            for _ in range(3):
                got.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(got, want)
        else:
            assert torch.equal(hostops.run_operator(mod, info, [X, F], constant=weights), want)
        full[op] = len(list(tmp_path.glob("*.hsaco")))
    assert full == {"c2d_nchw": 2, "t2d": 3}
    mod.close()
    ready.close()
