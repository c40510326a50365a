"""Decoder layers of 3 to 128 rows (tread_mid_layers_bf16) and their weight-streaming projection."""
import pytest
import torch

from tread_amd import _hip, blend, forward
from tread_amd.model import ModelConfig, synthetic_model

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("m", [1, 9, 16, 17, 33, 48, 64, 65, 96, 97, 113, 128])
@pytest.mark.parametrize("n,k", [(64, 128), (192, 384), (896, 4864), (1152, 896), (4672, 3584)])
def test_mid_linear_matches_fp64(m, n, k):
    g = torch.Generator().manual_seed(m * 7 + n)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g) / k ** 0.5).to(torch.bfloat16)
    b = torch.randn(n, generator=g).to(torch.bfloat16)
    for bias in (None, b):
        y = _hip.mid_linear(x.to(DEV), w.to(DEV), None if bias is None else bias.to(DEV)).cpu().double()
        xd, wd = x.double(), w.double()
        ref = xd @ wd.t() + (0 if bias is None else bias.double())
        # one bf16 rounding (2^-9 of the value; 2^-8 leaves a tie's whole step) after fp32 sums of k
        # products, whose error is at most k 2^-24 of the sum of their magnitudes
        mag = xd.abs() @ wd.abs().t() + (0 if bias is None else bias.double().abs())
        assert ((y - ref).abs() <= 2.0 ** -8 * ref.abs() + k * 2.0 ** -24 * mag).all()


def _layer_inputs(cfg, m, t_cap, seed):
    g = torch.Generator().manual_seed(seed)
    bf = lambda *s, scale=1.0: (scale * torch.randn(*s, generator=g)).to(torch.bfloat16).to(DEV)
    model = synthetic_model(cfg, DEV, torch.bfloat16, seed=seed, std=0.05, bias_std=0.05 if cfg.attention_bias else 0.0)
    shape = (cfg.num_hidden_layers, 1, cfg.num_key_value_heads, t_cap, cfg.head_dim)
    return blend.prepared(model), bf(m, cfg.hidden_size), bf(m, cfg.hidden_size, scale=0.1), bf(*shape), bf(*shape)


@pytest.mark.parametrize("m,hd,form", [(3, 128, "tail"), (9, 64, "tail"), (16, 128, "docs"), (17, 64, "pads"), (33, 128, "tail"),
                                       (64, 64, "docs"), (65, 128, "pads"), (128, 64, "tail")])
def test_mid_layers_match_the_separate_launches(m, hd, form, monkeypatch):
    """Two layers in one call against the path for many rows (library GEMMs and separate launches):
    the same roundings, sums in another order."""
    cfg = ModelConfig(512, 384, 2, 6, 2, hd, 640)  # 128-wide units, tiles shared by work groups
    P, h, d, K, V = _layer_inputs(cfg, m, 300, seed=m + hd)
    rows = torch.arange(150, 150 + m, device=DEV)
    kseg, n_shared, kend, pos = None, 0, rows, rows
    if form == "docs":  # two packed segments after a shared prefix
        kseg = torch.where(torch.arange(m, device=DEV) < m // 2, 150, 150 + m // 2)
        n_shared, pos = 50, rows - kseg + 50
    R = forward.make_rows(P, rows, pos=pos, kseg=kseg, n_shared=n_shared)
    if form == "pads":  # padded rows: no visible key, one of them past the cache
        R.rows, R.kend = rows.clone(), kend.clone()
        R.kend[m - 3:] = -1
        R.rows[m - 1] = 300
    K2, V2 = K.clone(), V.clone()
    with torch.inference_mode():
        a = forward.run_layers(P, h, d, R, K.unbind(0), V.unbind(0), range(2))
        monkeypatch.setattr(forward, "_mid_rows", lambda *a: False)
        b = forward.run_layers(P, h, d, R, K2.unbind(0), V2.unbind(0), range(2))
    for x, y in ((a[0], b[0]), (a[1], b[1]), (K, K2), (V, V2)):
        # bf16 rounding of every intermediate, in another order: 2^-8 each, a dozen of them a layer
        assert (x.float() - y.float()).norm() <= 0.02 * y.float().norm()
    spliced = rows if form != "pads" else rows[:m - 1]
    keep = torch.ones(300, dtype=torch.bool, device=DEV)
    keep[spliced] = False
    assert torch.equal(K[..., keep, :], K2[..., keep, :]) and torch.equal(V[..., keep, :], V2[..., keep, :])


def test_mid_layers_leave_strided_weights_to_the_library():
    """A down projection stored transposed: the call is taken as before."""
    cfg = ModelConfig(512, 384, 1, 6, 2, 64, 640)
    P, h, d, K, V = _layer_inputs(cfg, 20, 100, seed=2)
    rows = torch.arange(40, 60, device=DEV)
    R = forward.make_rows(P, rows)
    with torch.inference_mode():
        a = forward.run_layers(P, h, d, R, K.unbind(0), V.unbind(0), range(1))
        P.layers[0].wd = P.layers[0].wd.t().contiguous().t()
        assert not forward._mid_rows(P, 20, [0])
        b = forward.run_layers(P, h, d, R, K.unbind(0), V.unbind(0), range(1))
    for x, y in zip(a, b):  # bf16 rounding of every intermediate, in another order
        assert (x.float() - y.float()).norm() <= 0.02 * y.float().norm()
