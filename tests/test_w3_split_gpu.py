"""The split contract's matrix-core kernel (``fx_w3_inline_main`` / ``fx_w3_m1_out``, one
row) against float64 partial sums of the definition: every split form it takes, ragged
sizes, both arithmetics, zero-points beyond 3 and 4 (where decoded_bf16 rounds only the
weights with |q - z| = 3, as the table kernel does) and beyond 7, scales that no finite
product has, and unaligned operands.

Bar: every product is exact, so a partial is off by its fp32 additions alone: at most 32
matrix instructions a batch (two chains of 16) and one addition a batch, each at most
2^-24 of the terms' sum of magnitudes plus the 32 terms inside an instruction: 2^-18 of
that sum for the batches here; the output adds half its own ulp."""
import pytest
import torch

from marlin_style_fluxbin_amd import _lib
from marlin_style_fluxbin_amd.gptq_deployment import decode_planar_w3_codes
from tests.payloads import config_codes, layout_from_codes

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "f16": torch.float16}


def _expected(layout, x, gps, decoded):
    """float64 partials [splits, O] and their terms' magnitudes."""
    g, _, o, _ = layout["planes"].shape
    q = decode_planar_w3_codes(layout, original_order=False).double().view(g, 128, o)
    d = q - (layout["zeros"].double()[:, None] if "zeros" in layout else 4.0)
    w = layout["scales"].double()[:, None] * d
    if decoded:
        w = torch.where(d.abs() == 3, w.to(torch.bfloat16).double(), w)
    terms = w * x.double()[0, layout["perm"].long()].view(g, 128, 1)
    splits = -(-g // gps)
    pad = torch.zeros(splits * gps - g, 128, o, dtype=torch.float64, device=terms.device)
    terms = torch.cat([terms, pad]).view(splits, gps * 128, o)
    return terms.sum(1), terms.abs().sum(1)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("decoded", [False, True])
@pytest.mark.parametrize("o,g,gps", [(1, 1, 1), (17, 2, 1), (33, 5, 1), (100, 7, 2), (16, 32, 4), (250, 33, 8),
                                     (31, 13, 13), (64, 96, 2), (40, 128, 1), (48, 128, 64), (15, 6, 7)])
def test_split_partials_and_output(gpu, o, g, gps, decoded, dtype):
    k = 128 * g
    codes, scales, _, perm = config_codes(o, k, seed=o + g, scale_dtype=DT["bf16" if decoded else dtype], permute=True)
    zeros = torch.randint(0 if o % 2 else 3, 8 if o % 2 else 5, (g, o), generator=torch.Generator().manual_seed(g),
                          dtype=torch.uint8)
    layout = {n: v.to(gpu) for n, v in layout_from_codes(codes, scales, zeros, perm).items()}
    if o % 3 == 0:
        del layout["zeros"]
    buffer = torch.randn(1, k + 8, generator=torch.Generator().manual_seed(1)).to(DT[dtype]).to(gpu)
    x = buffer[:, o % 2:k + o % 2]  # odd row counts: x off 16-byte alignment
    effective = min(gps, g)
    want, terms = _expected(layout, x, effective, decoded)
    lib, stream = _lib.library(), _lib.stream_handle(gpu)
    head = (x.data_ptr(), _lib.dtype_code(x.dtype), layout["planes"].data_ptr(), layout["scales"].data_ptr(),
            _lib.dtype_code(layout["scales"].dtype), _lib.ptr(layout.get("zeros")), layout["perm"].data_ptr())
    partial = torch.full(want.shape, float("nan"), device=gpu)
    _lib.check(lib.fx_w3_inline_main(*head, partial.data_ptr(), 1, o, k, effective, 256, int(decoded), stream), "main")
    assert bool(((partial.double() - want).abs() <= 2.0 ** -18 * terms).all())
    workspace = torch.full(want.shape, float("nan"), device=gpu)
    out = torch.empty(1, o, dtype=x.dtype, device=gpu)
    _lib.check(lib.fx_w3_m1_out(*head, workspace.data_ptr(), out.data_ptr(), 1, o, k, effective, 256, int(decoded),
                                stream), "m1_out")
    if want.shape[0] > 1:
        assert torch.equal(workspace, partial)
    else:
        assert bool(torch.isnan(workspace).all())  # one split leaves the workspace alone
    exact, total = want.sum(0), terms.sum(0)
    bits, low = (7, -126) if dtype == "bf16" else (10, -14)
    ulp = torch.exp2(torch.floor(torch.log2(exact.abs().clamp(min=2.0 ** low))) - bits)
    assert bool(((out[0].double() - exact).abs() <= 0.5 * ulp + 2.0 ** -18 * total).all())


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_split_infinities(gpu, dtype):
    """An infinite activation gives the product's infinities and NaN (a zero weight times
    infinity) and leaves no other trace."""
    codes, scales, zeros, perm = config_codes(64, 1024, seed=2, scale_dtype=torch.bfloat16, permute=True)
    layout = {n: v.to(gpu) for n, v in layout_from_codes(codes, scales, zeros, perm).items()}
    x = torch.randn(1, 1024, generator=torch.Generator().manual_seed(4)).to(DT[dtype]).to(gpu)
    x[0, 100] = float("inf")
    want, _ = _expected(layout, x, 8, False)
    partial = torch.empty(1, 64, device=gpu)
    _lib.check(_lib.library().fx_w3_inline_main(
        x.data_ptr(), _lib.dtype_code(x.dtype), layout["planes"].data_ptr(), layout["scales"].data_ptr(), _lib.FX_BF16,
        layout["zeros"].data_ptr(), layout["perm"].data_ptr(), partial.data_ptr(), 1, 64, 1024, 8, 256, 0,
        _lib.stream_handle(gpu)), "main")
    assert torch.equal(torch.isnan(partial), torch.isnan(want))
    finite_sign = ~torch.isnan(want)
    assert torch.equal(partial[finite_sign], want[finite_sign].float())


def _partials(layout, x, gps, decoded, row_tile=256):
    g, _, o, _ = layout["planes"].shape
    partial = torch.full((-(-g // gps), o), float("nan"), device=x.device)
    _lib.check(_lib.library().fx_w3_inline_main(
        x.data_ptr(), _lib.dtype_code(x.dtype), layout["planes"].data_ptr(), layout["scales"].data_ptr(),
        _lib.dtype_code(layout["scales"].dtype), layout["zeros"].data_ptr(), layout["perm"].data_ptr(),
        partial.data_ptr(), 1, o, 128 * g, gps, row_tile, int(decoded), _lib.stream_handle(x.device)), "main")
    return partial


def _payload(gpu, o, g, scale, seed):
    codes, scales, _, perm = config_codes(o, 128 * g, seed=seed, scale_dtype=DT[scale], permute=True)
    zeros = torch.randint(0, 8, (g, o), generator=torch.Generator().manual_seed(seed), dtype=torch.uint8)
    return {n: v.to(gpu) for n, v in layout_from_codes(codes, scales, zeros, perm).items()}


@pytest.mark.parametrize("dtype,scale", [("bf16", "f16"), ("f16", "f16"), ("f16", "bf16")])
@pytest.mark.parametrize("g,gps", [(5, 1), (6, 2), (8, 4), (11, 11), (33, 16)])
def test_split_zero_points_of_eight_bits(gpu, g, gps, dtype, scale):
    """Zero-points over the whole byte (the checked layouts hold 0..7): s (q - z) x has up
    to 30 bits, and a product is off by its fp32 roundings alone: a single activation,
    so that no sum hides them, within 2^-21 of the product (at most three additions of
    its digits' products, an ulp each); and whole rows as above."""
    layout = _payload(gpu, 37, g, scale, g)
    wide = torch.randint(0, 256, (g, 37), generator=torch.Generator().manual_seed(1), dtype=torch.uint8).to(gpu)
    some = torch.rand(g, 37, generator=torch.Generator().manual_seed(2)).to(gpu) < 0.3
    layout["zeros"] = torch.where(some, wide, layout["zeros"])
    decodeds = (False, True) if scale == "bf16" else (False,)
    row = torch.randn(1, 128 * g, generator=torch.Generator().manual_seed(3)).to(DT[dtype]).to(gpu)
    for decoded in decodeds:
        want, terms = _expected(layout, row, gps, decoded)
        assert bool(((_partials(layout, row, gps, decoded).double() - want).abs() <= 2.0 ** -18 * terms).all())
        for column in range(0, 128 * g, 61):
            x = torch.zeros_like(row)
            x[0, column] = row[0, column]
            want, _ = _expected(layout, x, gps, decoded)
            assert bool(((_partials(layout, x, gps, decoded).double() - want).abs() <= 2.0 ** -21 * want.abs()).all())


@pytest.mark.parametrize("decoded", [False, True])
@pytest.mark.parametrize("g,gps", [(6, 1), (7, 2), (8, 4)])
def test_split_scales_without_a_product(gpu, g, gps, decoded):
    """A scale that is not finite stays in its own row and split (the other splits of its
    four groups may be summed in another order); one so large that its products with a code
    overflow still gives the sum that does not."""
    layout = _payload(gpu, 40, g, "bf16", 3)
    x = (torch.randn(1, 128 * g, generator=torch.Generator().manual_seed(3)) * 2.0 ** -20).to(torch.bfloat16).to(gpu)
    clean = _partials(layout, x, gps, decoded)
    layout["scales"][1, 3], layout["scales"][1, 20], layout["scales"][5, 39] = float("inf"), float("nan"), 3e38
    got = _partials(layout, x, gps, decoded)
    own, near = torch.zeros_like(got, dtype=torch.bool), torch.zeros_like(got, dtype=torch.bool)
    for group, row in ((1, 3), (1, 20), (5, 39)):
        own[group // gps, row] = True
        near[[i // gps for i in range(group // 4 * 4, min(g, group // 4 * 4 + 4))], row] = True
    assert torch.equal(got[~near], clean[~near])
    want, terms = _expected(layout, x, gps, decoded)
    near &= ~own
    assert bool(((got[near].double() - want[near]).abs() <= 2.0 ** -18 * terms[near]).all())
    assert not bool(torch.isfinite(got[1 // gps, 3])) and bool(torch.isnan(got[1 // gps, 20]))
    want, terms = _expected(layout, x, gps, False)
    if not decoded:  # (three times 3e38 has no bf16 value to round to)
        assert bool(torch.isinf(got[1 // gps, 3]))
        big = (5 // gps, 39)
        assert bool((got[big].double() - want[big]).abs() <= 2.0 ** -18 * terms[big])
