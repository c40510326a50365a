"""Attention of a few row tiles: the rule that cuts the key axis into slices."""
import pytest
import torch

from tread_amd import _hip

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("hd,G,hkv", [(128, 7, 4), (64, 7, 2)])
@pytest.mark.parametrize("n,keys", [(37, 191), (37, 223), (37, 224), (37, 1500), (160, 600), (300, 700), (160, 9000)])
def test_query_attention_slices_match_fp64(hd, G, hkv, n, keys):
    """Key slices at the edges of the split rule: one slice and two, whole and cut row tiles, up to one
    work group per CU."""
    g = torch.Generator().manual_seed(keys + n)
    q = torch.randn(n, G * hkv, hd, generator=g).to(torch.bfloat16)
    K = (2 * torch.randn(1, hkv, keys, hd, generator=g)).to(torch.bfloat16)
    V = torch.randn(1, hkv, keys, hd, generator=g).to(torch.bfloat16)
    kend = torch.randperm(keys, generator=g)[:n] if n <= keys else torch.arange(n).clamp(max=keys - 1)
    kend = kend.sort().values if n <= keys else kend
    out = _hip.subset_attn(q.to(DEV), K.to(DEV), V.to(DEV), kend.to(DEV), G * hkv, hkv, hd, hd ** -0.5).cpu().double()
    see = torch.arange(keys)[None] <= kend[:, None]
    for h in range(hkv):
        s = torch.einsum("ngd,kd->ngk", q[:, h * G:(h + 1) * G].double(), K[0, h].double()) * hd ** -0.5
        p = s.masked_fill(~see[:, None], float("-inf")).softmax(-1)
        ref = (p @ V[0, h].double()).reshape(n, -1)
        got = out.view(n, hkv, -1)[:, h]
        # bf16 rounding of the scaled q (scores off by 2^-9 of their size, up to about 10 here), of P and
        # of the result
        assert (got - ref).norm() <= 1.2e-2 * ref.norm()
