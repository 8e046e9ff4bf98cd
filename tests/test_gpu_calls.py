"""The operator's calls as one native step (csrc/bind.cpp) against fused.py's own lines: every form of a call gives the same bits, shapes and
types, or the same refusal, whichever of the two takes it."""
import numpy as np
import pytest

from llvq_amd import _ffi, synth

pytestmark = pytest.mark.gpu
D_IN = 400


@pytest.fixture()
def projs(gpu_rt):
    import torch  # noqa: F401

    assert gpu_rt._calls is not None, "csrc/bind.cpp was not built"
    got = [gpu_rt.upload(synth.make_matrix(f"model.layers.0.c{d}.weight", d, D_IN, seed=d)) for d in (48, 17, 64)]
    yield got
    for p in got:
        gpu_rt.free(p)


def _both(rt, call):
    """What `call` returns or raises: natively first, by fused.py alone, and whether the native step took it."""
    import torch

    calls, took, got = rt._calls, [], []

    class Spy:
        def __getattr__(self, name):
            def f(*a):
                r = getattr(calls, name)(*a)
                took.append(r is not None)
                return r
            return f

    for c in (Spy(), None):
        rt._calls = c
        try:
            y = call()
            got.append([t.clone() for t in (y if isinstance(y, (list, tuple)) else [y])])
            torch.cuda.synchronize()
        except Exception as e:  # noqa: BLE001
            got.append((type(e), str(e)))
        finally:
            rt._calls = calls
    return got[0], got[1], bool(took and took[0])


def _same(a, b):
    import torch

    if isinstance(a, tuple) or isinstance(b, tuple):
        return a == b
    return len(a) == len(b) and all(type(p) is type(q) and p.dtype == q.dtype and p.shape == q.shape and p.device == q.device and
                                    p.requires_grad == q.requires_grad and p.stride() == q.stride() and torch.equal(p, q) for p, q in zip(a, b))


def _forms():
    import torch

    x = torch.from_numpy(synth.make_activation(4 * D_IN, seed=5)[0].view(np.int16).copy()).view(torch.float16).cuda()
    row = x[:D_IN].clone()
    grad = row.clone().requires_grad_()
    return [  # (activation, whether it is one for the native step)
        (row, True), (row.view(1, D_IN), True), (row.view(1, 1, D_IN), True), (x[3:3 + D_IN], True), (grad, True),
        (x[::4], False), (row.float(), False), (row.double(), False), (row.to(torch.bfloat16), False), (row.cpu(), False), (row[:-1], False),
        (x[: 2 * D_IN].view(2, D_IN), None), (torch.nn.Parameter(row.clone()), True), (torch.conj(row), True), (torch.tensor(1.0, device="cuda").half(), False)]


def test_one_projection_and_groups(gpu_rt, projs):
    import torch

    for x, native in _forms():
        for dtype in (None, torch.float16, torch.float32, torch.bfloat16, "f16"):
            a, b, took = _both(gpu_rt, lambda: gpu_rt.forward(projs[0], x, out_dtype=dtype))
            assert _same(a, b), (x.shape, x.dtype, dtype, a, b)
            assert native is None or took == (native and dtype in (None, torch.float16, torch.float32)), (x.shape, x.dtype, dtype)
            if x.numel() != 2 * D_IN:  # (rows past the first are nobody's there)
                for group in (projs, tuple(projs), projs[:1], []):
                    a, b, _ = _both(gpu_rt, lambda: gpu_rt.forward_group(group, x, out_dtype=dtype))
                    assert _same(a, b), (x.shape, x.dtype, dtype, len(group), a, b)


def test_batches(gpu_rt, projs):
    import torch

    for rows in (1, 2, 5, 70):
        x = torch.randn(rows, D_IN, device="cuda", dtype=torch.float16, generator=torch.Generator("cuda").manual_seed(rows))
        for v, native in ((x, True), (x.t().contiguous().t(), rows == 1), (x.float(), False), (x[:, :-1].contiguous(), False), (x[0], False), (x[:0], False)):
            for dtype in (None, torch.float16, torch.float32, torch.bfloat16):
                a, b, took = _both(gpu_rt, lambda: gpu_rt.forward_batched(projs[0], v, out_dtype=dtype))
                assert _same(a, b), (v.shape, v.dtype, dtype, a, b)
                assert took == (native and dtype is not torch.bfloat16)
        for dtype in (torch.float16, torch.float32, torch.bfloat16):
            ys = [torch.zeros(rows, p.d_out, device="cuda", dtype=dtype) for p in projs]
            wrong = ys[:2] + [torch.zeros(rows, projs[2].d_out, device="cuda", dtype=torch.float64)]
            for outs in (ys, tuple(ys), ys[:2], wrong, [ys[1], ys[0], ys[2]], ys[:2] + [ys[2].t().contiguous().t()]):
                a, b, took = _both(gpu_rt, lambda: gpu_rt.forward_batched_group_into(projs, x, outs))
                assert _same(a, b), (rows, dtype, a, b)
                assert took or outs is not ys or dtype is torch.bfloat16


def test_what_wants_to_see_a_call_sees_it(gpu_rt, projs):
    import torch
    from torch.overrides import TorchFunctionMode

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x = _forms()[0][0]
    with Mode():
        a, b, took = _both(gpu_rt, lambda: gpu_rt.forward(projs[0], x))
        assert _same(a, b) and not took
    with torch.inference_mode():
        a, b, took = _both(gpu_rt, lambda: gpu_rt.forward(projs[0], x))
        assert _same(a, b) and a[0].is_inference() and b[0].is_inference()
    a, b, took = _both(gpu_rt, lambda: torch.func.vmap(lambda v: gpu_rt.forward(projs[0], v))(x.view(1, D_IN)))
    assert not took and isinstance(a, tuple) and isinstance(b, tuple) and a[0] is b[0]


def test_a_freed_projection_is_refused(gpu_rt):
    p = gpu_rt.upload(synth.make_matrix("model.layers.0.gone.weight", 16, D_IN, seed=1))
    x = _forms()[0][0]
    gpu_rt.free(p)
    a, b, took = _both(gpu_rt, lambda: gpu_rt.forward(p, x))
    assert _same(a, b) and a[0] is _ffi.LlvqError and not took
