"""GPU: the prompt GEMM at the edges of its tiles and dispatch rules, against
an fp64 product of the exact q*s weights: output counts that leave a last tile
of 1 to 15 rows (and matrices of fewer than 16), token counts around 16, 32, 64
and their multiples, one group and odd group counts, row counts around each
kernel's limits, scales that are only 2-byte aligned, and K too long for the
staged scales.  One-hot tokens give each weight back: equal, bit for bit, to
bf16(q*s)."""
import numpy as np
import pytest
import torch

import dip_oracle as O
from gpu_util import dev, dev_bf16, host_bf16, random_bf16, random_int4

pytestmark = pytest.mark.gpu

CASES = [(1, 5, 128), (2, 16, 384), (3, 17, 128), (16, 31, 640), (17, 1000, 256), (31, 40, 1152),
         (33, 8, 512), (48, 1003, 384), (65, 2570, 640),   # split kernel
         (64, 20480, 256), (100, 10249, 384), (129, 9000, 512),  # tiled, two K parts
         (64, 40961, 128), (333, 7000, 640), (130, 25600, 128),  # tiled, one K part
         (700, 24001, 256),                                # tiled, four row tiles a wave
         (7, 48, 1 << 17), (40, 33, 40960),                # scales from memory
         (9, 4271, 256), (16, 8279, 256), (9, 12501, 256),  # split, 8 waves: two to four tiles
         (20, 4271, 256), (32, 8279, 256), (20, 12501, 256),
         (9, 36971, 256), (16, 16507, 256), (9, 24739, 256),  # split, 4 waves
         (768, 331, 256), (201, 2307, 256), (100, 5125, 256), (20, 16507, 256), (32, 24739, 256)]


@pytest.mark.parametrize("m,n,k", CASES)
@pytest.mark.parametrize("odd", [0, 1])
def test_gemm_tile_edges(m, n, k, odd):
    import _dip_hip as K
    print(f"int4_gemm m={m} n={n} k={k} odd={odd}", flush=True)
    rng = np.random.default_rng(m + n + k)
    qw, sc = random_int4(rng, n, k)
    x = np.stack([random_bf16(rng, k) for _ in range(m)])
    hot = rng.integers(0, k, size=m)
    x[::3] = 0
    x[np.arange(0, m, 3), hot[::3]] = 0x3F80  # bf16 1.0
    s = torch.zeros(sc.size + odd, dtype=torch.bfloat16, device="cuda")
    s[odd:] = dev_bf16(sc).view(-1)
    w, xd = dev(qw), dev_bf16(x)
    guard = torch.full((m * n + 64,), 7.0, dtype=torch.bfloat16, device="cuda")
    K._check(K.lib.dip_int4_gemm(w.data_ptr(), s.data_ptr() + 2 * odd, xd.data_ptr(),
                                 guard.data_ptr(), m, n, k, K._stream(w.device)), "dip_int4_gemm")
    assert bool((guard[m * n:] == 7.0).all())
    out = guard[:m * n].view(m, n)
    wf = torch.from_numpy(O.dequant_f32(qw, sc)).cuda().double()
    xf = xd.double()
    ref, terms = xf @ wf.t().contiguous(), xf.abs() @ wf.abs().t().contiguous()
    bound = 2.0 ** -8 * ref.abs() + 2.0 ** -17 * terms  # one bf16 rounding, fp32 sums
    assert bool(((out.double() - ref).abs() <= bound).all())
    got, want = O.bf16_to_f32(host_bf16(out[::3])), O.bf16_to_f32(O.dequantize(qw, sc)).T[hot[::3]]
    assert np.array_equal(got, want)


def test_linear_route_for_longer_prompts():
    """65 to 512 bf16 rows take the int4 GEMM; anything the kernel could not
    stand in for (another dtype, gradients, functorch, forward mode, a wrong
    width) still goes through torch's linear, as it did."""
    import torch.nn.functional as F
    import qlinear as Q
    rng = np.random.default_rng(5)
    qw, sc = (lambda a: (dev(a[0]), dev_bf16(a[1])))(random_int4(rng, 384, 256))
    w = Q.dequantize(qw, sc)
    g = torch.Generator(device="cuda").manual_seed(1)
    for rows in (65, 200, 512, 513):
        x = torch.randn(rows, 512, device="cuda", generator=g).to(torch.bfloat16)
        for v in (x[:, :256], x[:, ::2], x.t()[:256].t(), x[:, :256].reshape(1, rows, 256)):
            ref = F.linear(v, w)
            got = Q.int4_linear(v, qw, sc)
            assert got.shape == ref.shape and got.dtype == ref.dtype
            assert float((got - ref).abs().max() / ref.abs().max()) < 1e-2
    x = torch.randn(100, 256, device="cuda", generator=g)
    assert torch.equal(Q.int4_linear(x, qw, sc), F.linear(x, w.float()))
    assert torch.equal(Q.int4_linear(x.half(), qw, sc), F.linear(x.half(), w.half()))
    xb = x.to(torch.bfloat16)
    xg = xb.clone().requires_grad_()
    Q.int4_linear(xg, qw, sc).sum().backward()
    assert xg.grad is not None
    out = torch.func.vmap(lambda v: Q.int4_linear(v, qw, sc))(torch.stack([xb, 2 * xb]))
    assert torch.equal(out[0], F.linear(xb, w))
    import torch.autograd.forward_ad as fwd
    with fwd.dual_level():
        tan = fwd.unpack_dual(Q.int4_linear(fwd.make_dual(xb, xb), qw, sc)).tangent
        assert torch.equal(tan, F.linear(xb, w))
    with pytest.raises(RuntimeError):
        Q.int4_linear(torch.zeros(100, 512, device="cuda", dtype=torch.bfloat16), qw, sc)
