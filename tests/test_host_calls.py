"""The native calls (csrc/host_calls.cpp): the same result as the Python path, and everything out of the ordinary left to it."""
import copy
import threading

import pytest
import torch

from tilelang_ascend_amd import _abi, ops
from tilelang_ascend_amd.ops.dequant_gemm import _w4a8_kernel
from tilelang_ascend_amd.quantize import gpu


def test_plan_checks_its_description_and_leaves_host_tensors_alone():
    Plan = _abi.host().Plan
    params = (((4, 8), _abi.I8, 0), ((4, 4), 5, 0), ((4, 4), _abi.I32, 1))
    assert Plan("w4a8", params, (4, 4, 8, 0), 0.0)(torch.zeros(4, 8, dtype=torch.int8), torch.zeros(4, 4, dtype=torch.uint8)) is NotImplemented
    assert Plan("w4a8", params, (4, 4, 8, 0), 0.0)() is NotImplemented
    for kind, p, ints in (("none such", params, (4, 4, 8, 0)), ("w4a8", params, (4, 4)), ("w4a8", params[:2], (4, 4, 8, 0)),
                          ("w4a8", (((4, -8), _abi.I8, 0),) + params[1:], (4, 4, 8, 0)), ("w4a8", (((4, 8), 77, 0),) + params[1:], (4, 4, 8, 0))):
        with pytest.raises(ValueError):
            Plan(kind, p, ints, 0.0)


def test_kernel_objects_are_copied_after_their_plan_is_made():
    kernel = ops.w4a16_gemm(3, 64, 256, group_size=128, zeros="tensor")
    kernel._fast = kernel._native_plan()  # what the first call on a GPU does
    holder = torch.nn.Module()
    holder.kernel = kernel
    for twin in (copy.deepcopy(kernel), copy.copy(kernel), copy.deepcopy(holder).kernel):
        assert twin is not kernel and twin.params == kernel.params and twin.result_idx == kernel.result_idx
        assert twin._plan is None and twin._fast == twin._first_call
        assert twin._native_plan() is not kernel._plan
    assert kernel._fast is kernel._plan


def _calls():
    g = torch.Generator().manual_seed(3)
    i8 = lambda *s: torch.randint(-100, 100, s, dtype=torch.int8, generator=g).cuda()  # noqa: E731
    u8 = lambda *s: torch.randint(0, 256, s, dtype=torch.uint8, generator=g).cuda()  # noqa: E731
    f = lambda t, *s: (torch.rand(s, generator=g) + 0.5).to(t).cuda()  # noqa: E731
    h, b, s32 = torch.float16, torch.bfloat16, torch.float32
    return {
        "w4a16": (ops.w4a16_gemm(3, 64, 256, group_size=128, zeros="tensor"), [f(h, 3, 256), u8(64, 128), f(h, 64, 2), f(h, 64, 2)]),
        "w4a16 no scales": (ops.w4a16_gemm(70, 64, 256, in_dtype="bfloat16", out_dtype="float32", with_scales=False, zeros=8), [f(b, 70, 256), u8(64, 128)]),
        "w4a16 workspace": (ops.w4a16_gemm(70, 256, 4096, group_size=128), [f(h, 70, 4096), u8(256, 2048), f(h, 256, 32)]),
        "w8a8": (ops.simple_quant_batch_matmul(2, 8, 32, 64, "1", 1, 1, 1), [i8(2, 8, 64), i8(2, 64, 32), f(s32, 1)]),
        "w8a8 slices": (ops.int8_gemm_kernel_corrected(64, 2048), [i8(5, 2048), i8(64, 2048), f(s32, 5), f(s32, 64)]),
        "act_quant": (ops.act_quant_kernel_int8_optimized(96, round_scale=True), [f(b, 7, 96)]),
        "w4a8_ws": (ops.w4a8_gemm_cv(4, 32, 256), [i8(4, 256), u8(32, 128), i8(32, 256)]),
        "w4a8": (_w4a8_kernel(9, 16, 128, "unsigned"), [i8(9, 128), u8(16, 64)]),
        "i8": (ops.int8_gemm(4, 32, 64, 1, 1, 1), [i8(4, 64), i8(64, 32)]),
        "f16": (ops.fp16_gemm(4, 32, 2048, 1, 1, 1), [f(h, 4, 2048), f(h, 2048, 32)]),
        "f16_batched": (ops.batch_matmul(2, 4, 32, 64, 1, 1, 1, "bfloat16"), [f(b, 2, 4, 64), f(b, 2, 64, 32)]),
        "gemv": (ops.simple_gemv(32, 64, 1, 1), [f(h, 64), f(h, 32, 64)]),
    }


@pytest.mark.gpu
def test_native_call_is_the_python_path():
    other = torch.cuda.Stream()
    for what, (kernel, args) in _calls().items():
        assert isinstance(kernel(*args), (torch.Tensor, list))
        assert type(kernel._fast).__name__ == "Plan", what
        got = kernel._fast(*args, torch.zeros(1))  # (a surplus positional)
        want = kernel.forward(list(args))
        torch.cuda.synchronize()
        elsewhere = kernel(*args, stream=other.cuda_stream)
        other.synchronize()
        for x, y, z in zip(*([v] if isinstance(v, torch.Tensor) else v for v in (got, want, elsewhere))):
            assert x.dtype == y.dtype and torch.equal(x, y) and torch.equal(x, z), what
        assert kernel._fast(*args[:-1], args[-1].cpu()) is NotImplemented
        assert kernel._fast(*args[:-1], args[-1].double()) is NotImplemented
        assert kernel._fast(*args[:-1], torch.stack([args[-1], args[-1]], -1)[..., 0]) is NotImplemented or args[-1].numel() == 1
        with pytest.raises(ValueError, match="dtype mismatch"):
            kernel(*args[:-1], args[-1].double())
    # an entry point that refuses the call: its own message
    bad = ops.int8_gemm(4, 30, 64, 1, 1, 1)
    with pytest.raises(RuntimeError, match="N"):
        bad(torch.zeros(4, 64, dtype=torch.int8).cuda(), torch.zeros(64, 30, dtype=torch.int8).cuda())


@pytest.mark.gpu
def test_native_helpers_and_threads():
    W = torch.randn(16, 256, generator=torch.Generator().manual_seed(1)).half().cuda()
    results, kernel, args = [], *_calls()["w4a16 workspace"]

    def work():
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                q, s = gpu.quantize_sym4(W, 64)
                p = gpu.pack_int4((q + 8).clamp_(max=15), None, torch.uint8)
                out = (q, s, p, ops.dequantize_w4(p, s, 8, 64), ops.unpack_int4(p), kernel(*args))
            torch.cuda.current_stream().synchronize()
            results.append(out)

    threads = [threading.Thread(target=work) for _ in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert len(results) == 4
    want = results[0]
    for r in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(r, want))
    q, s, p, w, u, _ = want
    assert torch.equal(u, (q + 8).clamp(max=15)) and torch.equal(w, ((u.half() - 8) * s.repeat_interleave(64, 1)))
