"""``fx_hybrid_restore`` (the hybrid Linear's dense fallback) against the torch
arithmetic it replaces on the GPU: bitwise in every output type and both code
formats at row counts off the workgroup's 128 and 16, and the same refusals."""
import pytest
import torch
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
