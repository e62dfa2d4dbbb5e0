"""GPU: dequantisation to the transpose, bit for bit the transposed
dequantisation: rows and columns that end within a tile, scales over the whole
bf16 range; and the long transposed product over the inputs it accepts."""
import numpy as np
import pytest
import torch

from gpu_util import dev, dev_bf16, random_int4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(8, 128), (120, 384), (128, 256), (136, 640), (1032, 5120)])
def test_dequant_t_is_the_transpose(rows, cols):
    import _dip_hip as K
    print(f"dequant_t {rows} x {cols}", flush=True)
    rng = np.random.default_rng(rows + cols)
    qw, sc = random_int4(rng, rows, cols)
    sc = rng.integers(0, 1 << 16, size=sc.shape).astype(np.uint16)  # infinities and NaN too
    q, s = dev(qw), dev_bf16(sc)
    want, got = K.dequant_rows(q, s, mode=1).t().contiguous(), K.dequant_t(q, s)
    assert torch.equal(got.isnan(), want.isnan())
    keep = ~want.isnan()
    assert torch.equal(got.view(torch.int16)[keep], want.view(torch.int16)[keep])


@pytest.mark.parametrize("rows", [1024, 1028])
def test_long_transposed_product(rows):
    """769 tokens through `rows` x 256, with and without a multiple of 8 rows:
    values and gradients as x @ dequantize gives them (2^-7: two bf16
    roundings), for bf16 and fp32, contiguous and strided x."""
    from qlinear import dequantize, int4_linear_t
    rng = np.random.default_rng(rows)
    qw, sc = (lambda t: (dev(t[0]), dev_bf16(t[1])))(random_int4(rng, rows, 256))
    w = dequantize(qw, sc)
    gen = torch.Generator(device="cuda").manual_seed(1)
    wide = torch.randn(769, 2 * rows, device="cuda", generator=gen)
    for x in (wide[:, :rows].to(torch.bfloat16), wide.to(torch.bfloat16)[None, :, ::2],
              wide[:, :rows]):
        x = x.detach().requires_grad_()
        ref, got = x @ w.to(x.dtype), int4_linear_t(x, qw, sc)
        assert got.shape == ref.shape and got.dtype == ref.dtype
        up = torch.randn(ref.shape, device="cuda", generator=gen).to(ref.dtype)
        pairs = [(got, ref)] + list(zip(torch.autograd.grad(got, x, up),
                                        torch.autograd.grad(ref, x, up)))
        for a, b in pairs:
            assert float((a - b).detach().abs().max()) <= 2.0 ** -7 * float(b.detach().abs().max())
