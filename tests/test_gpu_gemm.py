"""Projections of many rows (tread_linear_bf16, tread_linear_swiglu_bf16) and the rule that takes them."""
import pytest
import torch

from tread_amd import _hip, forward

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(m, n, k, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    bf = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)
    return bf(m, k), (bf(n, k).float() / k ** 0.5).to(torch.bfloat16), bf(n)


# edges of the tiles in both directions, one K tile and many, one partial round (cut along K or not), whole
# rounds alone and with a partial one
SHAPES = [(1, 8, 64), (255, 264, 128), (256, 256, 64), (257, 520, 192), (300, 3584, 18944), (513, 1152, 896),
          (4096, 4096, 64), (4200, 4096, 1024)]


def _check(y, ref, mag, k):
    # one bf16 rounding (2^-8 leaves a tie's whole step) after fp32 sums of k products in any order
    assert ((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + k * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_linear_matches_fp64(m, n, k):
    x, w, b = _inputs(m, n, k, m + k)
    ref = x.double() @ w.double().t().contiguous()
    mag = x.double().abs() @ w.double().abs().t().contiguous()
    _check(_hip.linear(x, w), ref, mag, k)
    _check(_hip.linear(x, w, b), ref + b.double(), mag + b.double().abs(), k)


@pytest.mark.parametrize("m,n,k", [(1, 16, 64), (257, 272, 192), (700, 1280, 18944), (4200, 4096, 896)])
def test_linear_swiglu_equals_linear_then_gating(m, n, k):
    """The gating of the fused kernel on the plain kernel's g and u: both add a tile's products in the same
    order, so the bits agree."""
    x, w, _ = _inputs(m, n, k, m)
    y = _hip.linear_swiglu(x, w)
    # a weight order that puts the same features into the same tiles does not exist for the plain kernel, but
    # an element's sum depends on the K slices alone, which the shape fixes
    assert torch.equal(y, _hip.silu_mul(_hip.linear(x, w)))


def test_workspace_is_optional():
    x, w, _ = _inputs(300, 512, 4096, 1)
    y = torch.empty(300, 512, dtype=torch.bfloat16, device=DEV)
    assert _hip.lib().tread_linear_workspace_bytes(300, 512, 4096) > 0
    _hip._check("tread_linear_bf16", _hip.lib().tread_linear_bf16(
        x.data_ptr(), w.data_ptr(), None, 300, 512, 4096, y.data_ptr(), None, 0, _hip._stream()))
    ref = x.double() @ w.double().t().contiguous()
    _check(y, ref, x.double().abs() @ w.double().abs().t().contiguous(), 4096)


@pytest.mark.parametrize("m,k,n,fused", [(3328, 896, 9728, False), (3329, 896, 9728, True), (3329, 1088, 9728, False)])
def test_mlp_route_matches_the_general_one(m, k, n, fused, monkeypatch):
    """Both sides of the fused gate|up rule give the general path's MLP up to the order of its sums."""
    from types import SimpleNamespace
    assert forward._swiglu_pays(m, n, k) == fused
    x, wgu, _ = _inputs(m, n, k, 3)
    _, wd, _ = _inputs(1, k, n // 2, 4)
    lw = SimpleNamespace(wgu=wgu, wd=wd)
    y = forward._mlp(x, lw, 0).float()
    monkeypatch.setattr(forward, "_swiglu_pays", lambda *a: False)
    r = forward._mlp(x, lw, 0).float()
    assert (y - r).norm() <= 5e-3 * r.norm()  # bf16 rounding of the gated rows (2^-9) in another order


def test_down_route_matches_the_general_one():
    m, k, n = 4700, 16384, 3584
    assert forward._linear_pays(m, n, k) and not forward._linear_pays(m, n, 8192)
    x, w, _ = _inputs(m, n, k, 5)
    y, r = _hip.linear(x, w).float(), torch.nn.functional.linear(x, w).float()
    assert (y - r).norm() <= 3e-3 * r.norm()  # two bf16 roundings of sums in another order
