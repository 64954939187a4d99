"""``fx_hybrid_restore`` (the hybrid Linear's dense fallback) against the torch
arithmetic it replaces on the GPU: bitwise in every output type and both code
formats at row counts off a workgroup's 64 and a wave's 8, the same refusals, and the
calls that keep the torch arithmetic."""
import pytest
import torch
from torch.autograd import forward_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from marlin_style_fluxbin_amd import deployment as d
from oracle import two_base as tb

pytestmark = pytest.mark.gpu


def _layout(o, g, kernel, device):
    p = {k: torch.from_numpy(v) for k, v in tb.make_hybrid_payload(o, g, seed=o + g).items()}
    return {k: v.to(device) for k, v in d.convert_artifact(p, kernel=kernel).items()}


@pytest.mark.parametrize("kernel", ["v1", "v5_p1024"])
@pytest.mark.parametrize("o,g", [(1, 1), (16, 2), (17, 3), (129, 2), (300, 32), (1024, 96)])
def test_restore_is_bitwise_the_torch_weight(gpu, o, g, kernel):
    layout = _layout(o, g, kernel, gpu)
    layout["rows"][0, 0] = -0.0  # signed zeros sum as the torch adds do
    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        assert d._restore_kernel_takes(layout, dtype)
        got = d.decode_layout(layout, dtype)
        want = d._decode_layout_torch(layout, dtype)
        bits = torch.int32 if dtype == torch.float32 else torch.int16
        assert torch.equal(got.view(bits), want.view(bits))


@pytest.mark.parametrize("field,where,value,message", [
    ("rows", (1, 200, 0), float("inf"), "finite"), ("columns", (0, 127, 1), float("nan"), "finite"),
    ("sparse_rows", (2, 0, 1), float("nan"), "finite"), ("sparse_columns", (1, 7, 0), float("-inf"), "finite"),
    ("indices", (2, 7), 128, "outside the group"), ("indices", (0, 0), -1, "outside the group"),
    ("indices", (1, 3), 0, "sorted and unique")])
def test_restore_refuses_what_torch_refuses(gpu, field, where, value, message):
    p = {k: torch.from_numpy(v) for k, v in tb.make_hybrid_payload(201, 3, seed=5).items()}
    module = d.PackedHybridLinear(p, fallback="dense", kernel="v5_p1024").to(gpu)
    x = torch.randn(3, 384, device=gpu).to(torch.bfloat16)
    with torch.inference_mode():
        want = torch.nn.functional.linear(x, d._decode_layout_torch(module.layout(), torch.bfloat16))
        assert torch.equal(module(x), want)
    getattr(module, field)[where] = value
    with torch.inference_mode(), pytest.raises(ValueError, match=message):
        module(x)
    with pytest.raises(ValueError, match=message):
        d.decode_layout(module.layout())


def test_restore_under_a_default_device(gpu):
    """The verdict lives in pinned host memory whatever device new tensors go to."""
    layout = _layout(17, 3, "v5_p1024", gpu)
    want = d._decode_layout_torch(layout, torch.bfloat16)
    with torch.device(gpu):
        assert torch.equal(d.decode_layout(layout), want)


class _Seen(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_traced_calls_keep_the_torch_arithmetic(gpu):
    """A tracer records torch ops: the weight has to be formed by them."""
    p = {k: torch.from_numpy(v) for k, v in tb.make_hybrid_payload(48, 2, seed=5).items()}
    module = d.PackedHybridLinear(p, fallback="dense", kernel="v5_p1024").to(gpu)
    x = torch.randn(3, 256, device=gpu).to(torch.bfloat16)
    with _Seen():
        assert not d._restore_kernel_takes(module.layout(), torch.bfloat16)
    with torch.no_grad():
        want = module(x)
        traced = torch.jit.trace(module, x, check_trace=False)
        assert "aten::empty(" not in str(traced.inlined_graph.findNode("aten::linear").inputsAt(1).node())
        assert torch.equal(traced(x), want)


def _module(gpu, o=48, g=2):
    p = {k: torch.from_numpy(v) for k, v in tb.make_hybrid_payload(o, g, seed=5).items()}
    return d.PackedHybridLinear(p, fallback="dense", kernel="v5_p1024").to(gpu)


@pytest.mark.parametrize("field", ["rows", "columns", "sparse_rows", "sparse_columns"])
def test_restored_weight_keeps_derivatives(gpu, field):
    """Scales with a gradient or a tangent: the weight is a function of them."""
    layout = _layout(33, 2, "v5_p1024", gpu)
    head = torch.randn(33, 256, generator=torch.Generator().manual_seed(1)).to(gpu)

    def gradient(decode):
        leaf = layout[field].clone().requires_grad_()
        return torch.autograd.grad((decode(dict(layout, **{field: leaf}), torch.float32) * head).sum(), leaf)[0]

    want = gradient(d._decode_layout_torch)
    assert bool(want.any()) and torch.equal(gradient(d.decode_layout), want)
    leaf = layout[field].clone().requires_grad_()
    with torch.no_grad():  # no graph is asked for: the kernel may form the values
        assert torch.equal(d.decode_layout(dict(layout, **{field: leaf})), d.decode_layout(layout))
    tangent = torch.randn(layout[field].shape, generator=torch.Generator().manual_seed(2)).to(gpu)
    with torch.no_grad(), forward_ad.dual_level():
        dual = dict(layout, **{field: forward_ad.make_dual(layout[field], tangent)})
        got = forward_ad.unpack_dual(d.decode_layout(dual, torch.float32)).tangent
        want = forward_ad.unpack_dual(d._decode_layout_torch(dual, torch.float32)).tangent
    assert got is not None and torch.equal(got, want)


def test_transforms_over_the_module(gpu):
    module = _module(gpu)
    x, t = (torch.randn(3, 256, generator=torch.Generator().manual_seed(i)).to(torch.bfloat16).to(gpu) for i in (0, 1))
    w = d._decode_layout_torch(module.layout(), torch.bfloat16)
    with torch.no_grad():
        y, dy = torch.func.jvp(module, (x,), (t,))
        assert torch.equal(y, torch.nn.functional.linear(x, w)) and torch.equal(dy, torch.nn.functional.linear(t, w))
        assert torch.equal(torch.func.vmap(module)(x.view(1, 3, 256))[0], y)


def test_restore_leaves_lazy_negation_to_torch(gpu):
    """A contiguous view whose memory holds the other sign."""
    layout = _layout(17, 3, "v5_p1024", gpu)
    want = d.decode_layout(layout)
    for field in ("rows", "columns", "sparse_rows", "sparse_columns"):
        lazy = torch._neg_view(-layout[field])
        assert lazy.is_neg() and lazy.is_contiguous()
        assert torch.equal(d.decode_layout(dict(layout, **{field: lazy})), want)


class _Doubled(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        out = func(*args, **(kwargs or {}))
        return out.mul_(2) if func is torch.Tensor.scatter_add_ else out


def test_function_modes_see_the_torch_arithmetic(gpu):
    """A function mode may change any op of the dequantize; torch's default device is
    one that changes none."""
    layout = _layout(17, 3, "v5_p1024", gpu)
    with _Doubled():
        assert not d._restore_kernel_takes(layout, torch.bfloat16)
        doubled = d.decode_layout(layout, torch.float32)
    assert torch.equal(doubled, 2 * d._decode_layout_torch(layout, torch.float32))
    with torch.device(gpu):
        assert d._restore_kernel_takes(layout, torch.bfloat16)
