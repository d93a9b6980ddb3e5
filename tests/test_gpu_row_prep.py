"""Row preparation at the edges of its row split and of its two address forms.

K in fp32 takes the 64-bit address form from 2^17 rows on; halves of such a call
take the other one and must give the same bits.

Head dim 256 takes two rows per wave, so odd row counts end in half a wave; row
indexes are split with multipliers, so head counts and lengths that are and are
not powers of two are covered; a batch stride of 2^32 elements (one batch, so
nothing lies there) takes the 64-bit address form and must give the same bits.
Against the operations in torch: fp32 row statistics, K and V rounded to bf16,
each RoPE product and the sum rounded to bf16.  The row sum's order may move the
inverse RMS by an fp32 ulp and so a rounding of the normalised value by one bf16
ulp, 2^-7 relative: the bound of V and of K's dims without RoPE.  Such a step of
x or of its partner reaches a rotary element through two products and their sum,
each of which may round to the other side as well (2 x 2^-8 each): 2^-7 + 2^-7
relative of each product and 2^-7 of the sum, 3 x 2^-7 of |x cos| + |rot(x) sin|.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 1e-6


def _reference(z, w, cos, sin, rotary):
    zf = z.float()
    n = zf * torch.rsqrt(zf.pow(2).mean(-1, keepdim=True) + EPS)
    kn = (n * w).to(torch.bfloat16)
    k, mag = kn.clone(), kn.float().abs()
    if rotary:
        x = kn[..., :rotary]
        half = rotary // 2
        rot = torch.cat((-x[..., half:], x[..., :half]), -1)
        c, s = cos[:, None], sin[:, None]
        k[..., :rotary] = x * c + rot * s
        mag[..., :rotary] = 3 * ((x * c).float().abs() + (rot * s).float().abs())
    return k, n.to(torch.bfloat16), mag


def _wide(t):
    """The same memory with a batch stride of 2^32 elements (one batch only)."""
    return t.as_strided(t.shape, (1 << 32,) + t.stride()[1:])


@pytest.mark.parametrize("d,b,h,s,rotary", [
    (256, 1, 1, 1, 256), (256, 1, 1, 7, 16), (256, 2, 3, 333, 256), (256, 3, 16, 65, 0),
    (256, 1, 32, 1025, 256), (256, 5, 5, 127, 240), (512, 1, 1, 1, 128), (512, 2, 3, 333, 512),
    (512, 3, 4, 129, 0), (512, 1, 17, 64, 496),
])
def test_row_preparation_edges(d, b, h, s, rotary):
    from gemma4_fa4_amd.kv_prep import prepare_rows_into

    g = torch.Generator().manual_seed(d + 7 * s + h)
    z = (torch.randn(b, s, h, d, generator=g) * 3).to(torch.bfloat16).transpose(1, 2)
    w = (torch.rand(d, generator=g) + 0.5).to(torch.bfloat16)
    ang = torch.rand(b, s, max(rotary, 16), generator=g) * 6
    cos, sin = torch.cos(ang).to(torch.bfloat16), torch.sin(ang).to(torch.bfloat16)
    want_k, want_v, mag = _reference(z, w.float(), cos, sin, rotary)
    zd = z.to(DEV)
    tables = {"cos": cos.to(DEV), "sin": sin.to(DEV)} if rotary else {}
    k, v = torch.empty_like(zd), torch.empty_like(zd)
    prepare_rows_into(zd, weight=w.to(DEV), rotary_dim=rotary, eps=EPS, k=k, v=v, **tables)
    for got, want, m in ((k, want_k, mag), (v, want_v, want_v.float().abs())):
        err = (got.float().cpu() - want.float()).abs()
        assert bool((err <= m * 2.0 ** -7 + 1e-6).all())
    if b == 1:
        k2, v2 = torch.empty_like(zd), torch.empty_like(zd)
        prepare_rows_into(_wide(zd), weight=w.to(DEV), rotary_dim=rotary, eps=EPS, k=_wide(k2),
                          v=_wide(v2), **tables)
        assert torch.equal(k, k2) and torch.equal(v, v2)


@pytest.mark.parametrize("heads,s", [(4, 32768), (4, 32767), (3, 43691)])
def test_large_fp32_preparation_matches_its_halves(heads, s):
    import gemma4_fa4_amd as g4

    g = torch.Generator(device=DEV).manual_seed(s)
    z = torch.randn(1, heads, s, 512, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.rand(512, generator=g, device=DEV) + 0.5
    ang = torch.rand(s, 128, generator=g, device=DEV) * 6
    cos, sin = torch.cos(ang), torch.sin(ang)
    with torch.no_grad():
        whole = g4.prepare_global_kv_from_projection_source(z, k_norm_weight=w, cos=cos, sin=sin)
        at = s // 2
        for part in (slice(0, at), slice(at, s)):
            got = g4.prepare_global_kv_from_projection_source(
                z[:, :, part], k_norm_weight=w, cos=cos[part], sin=sin[part])
            for x, y in zip(whole, got):
                assert torch.equal(x[:, :, part], y)
