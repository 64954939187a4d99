"""The row-packed RMSNorm (rows of at most 128 values) and the vectorised RoPE at the
edges of their workgroups, against the torch arithmetic they stand for: RMSNorm within
two output ulps, RoPE and copies bit for bit.

The RMSNorm bar: the sum of squares in another fp32 order moves 1 / rms by a few 2^-24,
which can flip the inner rounding round(x / rms) by one of its ulps; times the weight that
is less than two ulps of the output (an ulp of n is at most w n 2^-7 there, and an ulp of
y = w n at least half of it), so the rounded outputs are at most two apart, and where no
rounding flips they are equal."""
import pytest
import torch

from marlin_style_fluxbin_amd import _lib
from marlin_style_fluxbin_amd.fused_modules import (
    _rope_torch, add_rms_norm, fused_apply_rotary_pos_emb, head_norm_rope, rms_norm, rms_norm_reference)

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "f16": torch.float16}


def _two_ulps(got, want, dtype):
    bits, low = (7, -126) if dtype == "bf16" else (10, -14)
    ulp = torch.exp2(torch.floor(torch.log2(want.float().abs().clamp(min=2.0 ** low))) - bits)
    assert bool(((got.float() - want.float()).abs() <= 2 * ulp).all())
    assert float((got == want).float().mean()) >= 0.99


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("rows,hidden", [(1, 8), (15, 24), (16, 64), (17, 120), (255, 128), (16384, 128), (16385, 128),
                                         (20011, 72), (9, 136)])
def test_narrow_rms_norm(gpu, dtype, rows, hidden):
    g = torch.Generator().manual_seed(rows + hidden)
    x = torch.randn(rows, hidden, generator=g).to(DT[dtype]).to(gpu)
    r = torch.randn(rows, hidden, generator=g).to(DT[dtype]).to(gpu)
    w = (1 + 0.1 * torch.randn(hidden, generator=g)).to(DT[dtype]).to(gpu)
    _two_ulps(rms_norm(x, w, 1e-6), rms_norm_reference(x, w, 1e-6), dtype)
    out, s = torch.empty_like(x), x + r
    add_rms_norm(x, r, w, 1e-6, out=out, residual_out=r)  # in place on the residual
    assert torch.equal(r, s)
    _two_ulps(out, rms_norm_reference(s, w, 1e-6), dtype)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("batch,hq,hk,seq,dim", [(1, 32, 8, 8, 128), (2, 5, 1, 33, 64), (1, 7, 2, 129, 48),
                                                 (3, 4, 4, 31, 256), (1, 1, 1, 2000, 16), (1, 3, 2, 9, 40)])
def test_vector_rope_is_bit_exact(gpu, dtype, batch, hq, hk, seq, dim):
    g = torch.Generator().manual_seed(seq + dim)

    def normal(*shape):
        return torch.randn(shape, generator=g).to(DT[dtype]).to(gpu)

    cos, sin = normal(batch, seq, dim), normal(batch, seq, dim)
    q, k = normal(batch, seq, hq, dim), normal(batch, seq, hk, dim)
    for views, axis in (((q.transpose(1, 2), k.transpose(1, 2)), 1), ((q, k), 2)):
        got = fused_apply_rotary_pos_emb(*views, cos, sin, unsqueeze_dim=axis)
        # the algebra on the CPU (torch's GPU addcmul rounds rare fp16 sums differently)
        for a, b in zip(got, _rope_torch(*(v.cpu() for v in (*views, cos, sin)), axis)):
            assert torch.equal(a.cpu(), b)
    odd = normal(batch * seq * hq * dim + 1)[1:].view(batch, seq, hq, dim)  # off 16-byte alignment: the row kernel
    for a, b in zip(fused_apply_rotary_pos_emb(odd, k, cos, sin, unsqueeze_dim=2),
                    _rope_torch(*(v.cpu() for v in (odd, k, cos, sin)), 2)):
        assert torch.equal(a.cpu(), b)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("mode", [_lib.ROPE_STOCK, _lib.ROPE_FUSED])
def test_vector_rope_and_copy_into_a_cache(gpu, mode, dtype):
    """Rotation and a plain strided copy in one launch, each into its own slots, and the
    same bits as the row kernel (which a single position takes)."""
    heads, seq, dim, length = 6, 20, 128, 64
    g = torch.Generator().manual_seed(7)
    x = torch.randn(2, seq, heads, dim, generator=g).to(DT[dtype]).to(gpu)
    cos, sin = (torch.randn(seq, dim, generator=g).to(DT[dtype]).to(gpu) for _ in range(2))
    cache = torch.full((2, heads, length, dim), 7.0, dtype=DT[dtype], device=gpu)
    rows = torch.full_like(cache, 7.0)

    def tensors(dst, first, n):
        return [dict(x=x[i], out=dst[i, :, first:], heads=heads, rope=i == 0,
                     in_strides=(0, dim, heads * dim), out_strides=(0, length * dim, dim)) for i in range(n)]

    head_norm_rope(tensors(cache, 3, 2), cos=cos, sin=sin, eps=1e-6, seq=seq, rope_mode=mode, cos_strides=(0, dim))
    for s in range(seq):
        one = [dict(t, x=x[i, s:]) for i, t in enumerate(tensors(rows, 3 + s, 2))]
        head_norm_rope(one, cos=cos[s:], sin=sin[s:], eps=1e-6, seq=1, rope_mode=mode, cos_strides=(0, dim))
    assert torch.equal(cache, rows)
    assert bool((cache[:, :, :3] == 7).all()) and bool((cache[:, :, 3 + seq:] == 7).all())
    assert torch.equal(cache[1, :, 3:3 + seq], x[1].transpose(0, 1))
