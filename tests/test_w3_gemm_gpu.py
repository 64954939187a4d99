"""``fx_w3_gemm`` (the W3 dense fallback's product) against the float64 product of the
restored weight (``fx_w3_restore``, bitwise the oracle's), at the edges of its tiles
and plans.

Bar: the weights are the restored weight's bits, so what differs is the fp32
accumulation: half an output ulp of the exact value, plus 2^-18 of the terms' sum of
magnitudes (a chain of at most 16 matrix instructions a batch and batches of 512
columns, each adding one fp32 rounding of at most 2^-24 of that sum, with the pairwise
and split sums and the 32 terms inside an instruction).
"""
import pytest
import torch

from marlin_style_fluxbin_amd import PackedW3Linear
from marlin_style_fluxbin_amd import w3_lut_deployment as wl
from marlin_style_fluxbin_amd.gptq_deployment import restore_planar_w3
from tests.payloads import config_codes, layout_from_codes

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "f16": torch.float16}


def _module(gpu, o, k, *, seed=0, zeros=True, scale="bf16", permute=False, bias=None, **kwargs):
    codes, scales, zero, perm = config_codes(o, k, seed=seed, zeros=zeros, scale_dtype=DT[scale], permute=permute)
    layout = {n: v.to(gpu) for n, v in layout_from_codes(codes, scales, zero, perm).items()}
    return PackedW3Linear(layout, bias=bias, fallback="dense", row_tile=256, **kwargs)


def _check(module, x, dtype):
    """The module's output within the bar of the exact product of its dense weight."""
    assert module._gemm_takes(x)
    with torch.inference_mode():
        _within(module, x, module(x), dtype)


def _within(module, x, y, dtype):
    w = restore_planar_w3(module.layout(), dtype=x.dtype).double()
    flat = x.reshape(-1, module.in_features).double()
    exact = flat @ w.t()
    terms = flat.abs() @ w.abs().t()
    if module.bias is not None:
        exact = exact + module.bias.double()
    bits, lo = (7, -126) if dtype == "bf16" else (10, -14)
    ulp = torch.exp2(torch.floor(torch.log2(exact.abs().clamp(min=2.0 ** lo))) - bits)
    got = y.reshape(exact.shape).double()
    assert y.shape == (*x.shape[:-1], module.out_features) and y.dtype == x.dtype
    assert bool(torch.isfinite(got).all())
    assert bool(((got - exact).abs() <= 0.5 * ulp + 2.0 ** -18 * terms).all())


# rows at the edges of every activation tile; widths at the edges of the 16-row tiles and
# the plans' 2-, 3- and 4-tile blocks; K off the 512-column batch and long enough to split
@pytest.mark.parametrize("dtype,scale", [("bf16", "bf16"), ("bf16", "f16"), ("f16", "f16"), ("f16", "bf16")])
@pytest.mark.parametrize("o,k", [(1, 128), (17, 384), (63, 640), (1000, 1408), (100, 8192)])
@pytest.mark.parametrize("m", [2, 16, 17, 33, 48, 49, 65, 113, 225, 300])
def test_gemm_tiles(gpu, m, o, k, dtype, scale):
    module = _module(gpu, o, k, seed=m, scale=scale, permute=m % 2 == 1, zeros=m % 3 != 0)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(DT[dtype]).to(gpu)
    _check(module, x, dtype)


@pytest.mark.parametrize("m,o,k", [(12, 9216, 512), (20, 9217, 256), (40, 12288, 640), (60, 9230, 512),
                                   (112, 12288, 256), (128, 12300, 512), (400, 4096, 1024), (512, 1500, 512),
                                   (510, 12288, 640), (300, 12210, 1408), (400, 9000, 128), (500, 4100, 8192),
                                   (37, 512, 12288), (64, 1024, 12288), (100, 300, 16384), (200, 700, 8192)])
def test_gemm_wide_and_split_plans(gpu, m, o, k):
    module = _module(gpu, o, k, seed=3, permute=True)
    x = torch.randn(2, m // 2, k, generator=torch.Generator().manual_seed(m)).to(torch.bfloat16).to(gpu)
    _check(module, x, "bf16")


@pytest.mark.parametrize("m", [3, 50])
@pytest.mark.parametrize("k", [512, 12288])
def test_gemm_bias_views_and_extremes(gpu, m, k):
    """A bias (added before the rounding), a strided input, activations of 1e-30 and
    1e30, and infinities and NaN only in the rows that hold them."""
    bias = torch.randn(96, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(gpu)
    module = _module(gpu, 96, k, bias=bias, permute=True)
    g = torch.Generator().manual_seed(m)
    wide = torch.randn(m, 2 * k, generator=g).to(torch.bfloat16).to(gpu)
    _check(module, wide[:, :k], "bf16")
    for magnitude in (1e-30, 1e30):
        _check(_module(gpu, 96, k), (torch.randn(m, k, generator=g) * magnitude).to(torch.bfloat16).to(gpu), "bf16")
    x = wide[:, :k].contiguous()
    x[0, 5], x[1, 7] = float("inf"), float("nan")
    with torch.inference_mode():
        y = module(x)
    assert bool(torch.isnan(y[1]).all()) and not bool(torch.isfinite(y[0]).any())
    assert bool(torch.isfinite(y[2:]).all())


def test_gemm_route_leaves_other_calls_alone(gpu):
    """Calls that the kernel does not take (other types, a mismatched bias, transforms
    and modes that must see the op, more rows) keep the restored weight and F.linear."""
    module = _module(gpu, 64, 256)
    x = torch.randn(20, 256, device=gpu).to(torch.bfloat16)
    with torch.inference_mode():
        want = torch.nn.functional.linear(x, module._dense_weight(torch.bfloat16))
    assert not module._gemm_takes(x.float()) and not module._gemm_takes(x.cpu()) and not module._gemm_takes(x[:0])
    assert not module._gemm_takes(torch.empty(wl.GEMM_MAX_ROWS + 1, 256, device=gpu, dtype=torch.bfloat16))
    with torch.no_grad():
        mapped = torch.func.vmap(module)(x.view(4, 5, 256))
        assert torch.equal(mapped.reshape(20, 64), want)
        with torch.autocast("cuda", dtype=torch.float16):
            assert module(x).dtype == torch.float16
        odd = torch.zeros(20 * 256 + 1, device=gpu, dtype=torch.bfloat16)[1:].view(20, 256)
        assert torch.equal(module(odd), torch.zeros(20, 64, device=gpu, dtype=torch.bfloat16))
        assert module(x[:0]).shape == (0, 64)
    mixed = _module(gpu, 64, 256, bias=torch.zeros(64, device=gpu))
    assert not mixed._gemm_takes(x)
    with torch.inference_mode(), pytest.raises(RuntimeError):
        mixed(x)


def test_gemm_takes_only_whole_biases(gpu):
    """A bias that F.linear would broadcast keeps F.linear; one held as a Parameter is read."""
    x = torch.randn(20, 256, device=gpu).to(torch.bfloat16)
    one = _module(gpu, 64, 256, bias=torch.ones(1, device=gpu, dtype=torch.bfloat16))
    assert not one._gemm_takes(x)
    whole = _module(gpu, 64, 256, bias=torch.zeros(64, device=gpu, dtype=torch.bfloat16))
    whole.bias = torch.nn.Parameter(torch.ones(64, device=gpu, dtype=torch.bfloat16), requires_grad=False)
    _check(whole, x, "bf16")
    with torch.inference_mode():
        want = torch.nn.functional.linear(x, one._dense_weight(torch.bfloat16), one.bias)
        assert torch.equal(one(x), want)
        assert torch.equal(_module(gpu, 64, 256, bias=whole.bias, max_packed_rows=1)(x[:1]), whole(x[:1]))


def test_gemm_leaves_lazy_negation_to_torch(gpu):
    """A conjugate's imaginary part is a view whose memory holds the other sign."""
    module = _module(gpu, 64, 256, scale="f16")
    x = torch.zeros(20, 256, dtype=torch.complex32, device=gpu)
    x.copy_(torch.randn(20, 256, dtype=torch.complex64, device=gpu))
    lazy = x.conj().imag
    assert lazy.is_neg() and not module._gemm_takes(lazy)
    with torch.inference_mode():
        want = torch.nn.functional.linear(lazy, module._dense_weight(torch.float16))
        assert torch.equal(module(lazy), want)


def test_gemm_leaves_sparse_inputs_to_torch(gpu):
    """A sparse input has no memory to read by address: torch multiplies (or refuses) it."""
    module = _module(gpu, 64, 256, scale="f16")
    dense = torch.zeros(20, 256, device=gpu, dtype=torch.float16)
    dense[3, 5], dense[7, 200] = 1.5, -2.0
    for sparse in (dense.to_sparse(), dense.to_sparse_csr()):
        assert not module._gemm_takes(sparse)

        def outcome(call):
            with torch.inference_mode():
                try:
                    return call()
                except (RuntimeError, NotImplementedError) as error:
                    return str(error)

        want = outcome(lambda: torch.nn.functional.linear(sparse, module._dense_weight(torch.float16)))
        got = outcome(lambda: module(sparse))
        assert got == want if isinstance(want, str) else torch.equal(got, want)


def test_gemm_leaves_lazily_negated_biases_to_torch(gpu):
    module = _module(gpu, 64, 256, bias=torch.zeros(64, device=gpu, dtype=torch.bfloat16))
    module.bias = torch._neg_view(torch.ones(64, device=gpu, dtype=torch.bfloat16))
    x = torch.randn(20, 256, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(gpu)
    assert module.bias.is_neg() and not module._gemm_takes(x)
    with torch.inference_mode():
        want = torch.nn.functional.linear(x, module._dense_weight(torch.bfloat16), module.bias)
        assert torch.equal(module(x), want)


# more rows than the module's route takes, as a caller of the C entry may pass: plans of
# both kernels, whole and ragged sizes, one and two K splits, and the last row allowed
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("m,o,k", [(513, 17, 256), (513, 200, 8192), (700, 12300, 384), (1500, 330, 1408), (1500, 3000, 640),
                                   (4097, 65, 128), (8192, 200, 640), (8192, 1001, 384)])
def test_gemm_entry_beyond_the_modules_rows(gpu, m, o, k, dtype):
    module = _module(gpu, o, k, seed=m, permute=m % 2 == 1)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(DT[dtype]).to(gpu)
    _within(module, x, module._gemm(x, m), dtype)
