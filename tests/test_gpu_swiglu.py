"""SwiGLU in one launch: the values are those of the two torch ops, over all
bf16 gates (infinities and NaN among them) and at the ends of the vector runs.

silu differs from torch's in how the exponential and the quotient round in
fp32 (a few 2^-23), which moves its bf16 rounding by one step at most, and one
step (2^-8 relative, 2^-7 at the low end of a binade) carries over to the
product: 2^-6 of the value bounds both roundings."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _check(g, u):
    import _dip_hip as K
    got, ref = K.swiglu(g, u).float(), (F.silu(g) * u).float()
    same = (got == ref) | (got.isnan() & ref.isnan())
    assert bool((same | ((got - ref).abs() <= 2.0 ** -6 * ref.abs() + 1e-38)).all())
    return float(same.float().mean())


def test_every_gate():
    print("swiglu, every bf16 gate", flush=True)
    g = torch.arange(-32768, 32768, device="cuda").to(torch.int16).view(torch.bfloat16)
    for v in (1.0, -3.0, 0.0, float("inf"), float("nan")):
        assert _check(g, torch.full_like(g, v)) > 0.99


@pytest.mark.parametrize("shape", [(1,), (7,), (8,), (9,), (2, 2047), (2, 2048), (3, 1366), (1, 33, 12288)])
def test_sizes(shape):
    print(f"swiglu {shape}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(1)
    g, u = (torch.randn(*shape, device="cuda", generator=gen).to(torch.bfloat16) for _ in "gu")
    assert _check(g, u) > 0.99 or g.numel() < 100


def test_differentiated_inputs_keep_the_torch_ops():
    from qlinear import swiglu
    g, u = (torch.randn(4, 64, device="cuda").to(torch.bfloat16) for _ in "gu")
    g.requires_grad_()
    y = swiglu(g, u)
    assert y.requires_grad and torch.equal(y, F.silu(g) * u)
    assert torch.equal(swiglu(g.detach().float(), u.float()), F.silu(g.detach().float()) * u.float())
