"""GPU: the transposed prompt GEMM at the edges of its tiles: rows that leave a
last slice of 8, 16 or 24, one 128-column group and odd counts of them, token
counts around 16, 32 and 64, several K splits and none, an output that is only
2-byte aligned.  One-hot tokens pin every weight to the reference's bf16(q*s)
bit for bit, with scales from subnormal to the largest bf16, where the fused
product gives way to the plain one."""
import numpy as np
import pytest
import torch

import dip_oracle as O
from gpu_util import dev, dev_bf16, host_bf16, random_bf16

pytestmark = pytest.mark.gpu

CASES = [(1, 8, 128), (15, 24, 384), (16, 40, 256), (17, 1000, 128), (32, 520, 640), (33, 264, 384),
         (63, 3080, 256), (65, 800, 1152), (129, 2056, 2560), (200, 9728, 256), (700, 136, 5120),
         (513, 1024, 5120)]


@pytest.mark.parametrize("m,k,n", CASES)
@pytest.mark.parametrize("odd", [0, 1])
def test_gemm_t_tile_edges(m, k, n, odd):
    import _dip_hip as K
    print(f"int4_gemm_t m={m} k={k} n={n} odd={odd}", flush=True)
    rng = np.random.default_rng(m + n + k)
    qw = O.pack_int4(rng.integers(-8, 8, size=(k, n)).astype(np.int8))
    sc = rng.uniform(0.001, 0.02, (k, n // 128)) * rng.choice([-1.0, 1.0], (k, n // 128))
    sc = O.f32_to_bf16(sc.astype(np.float32))
    x = np.stack([random_bf16(rng, k) for _ in range(m)])
    w, s, xd = dev(qw), dev_bf16(sc), dev_bf16(x)
    nbytes = K.lib.dip_int4_gemm_t_workspace_size(m, n, k)
    ws = torch.full((max(nbytes, 16) + 16,), 0x5A, dtype=torch.uint8, device="cuda")
    guard = torch.full((odd + m * n + 64,), 7.0, dtype=torch.bfloat16, device="cuda")
    K._check(K.lib.dip_int4_gemm_t(w.data_ptr(), s.data_ptr(), xd.data_ptr(),
                                   guard.data_ptr() + 2 * odd, m, n, k, ws.data_ptr(), nbytes,
                                   K._stream(w.device)), "dip_int4_gemm_t")
    assert bool((guard[odd + m * n:] == 7.0).all()) and bool((guard[:odd] == 7.0).all())
    assert bool((ws[max(nbytes, 16):] == 0x5A).all())
    wf = torch.from_numpy(O.bf16_to_f32(O.dequantize(qw, sc))).cuda().double()
    ref, terms = xd.double() @ wf, xd.double().abs() @ wf.abs()
    err = (guard[odd:odd + m * n].view(m, n).double() - ref).abs()
    assert bool((err <= 2.0 ** -8 * ref.abs() + 2.0 ** -17 * terms).all())


@pytest.mark.parametrize("m,k,n", [(7, 520, 256), (20, 1032, 128), (64, 800, 384), (130, 264, 128)])
def test_gemm_t_weights_over_the_scale_range(m, k, n):
    import _dip_hip as K
    print(f"int4_gemm_t scale range m={m} k={k} n={n}", flush=True)
    rng = np.random.default_rng(k)
    qw = O.pack_int4(rng.integers(-8, 8, size=(k, n)).astype(np.int8))
    # exponents low enough (with subnormals), around the switch, and up to the
    # largest finite ones, by runs of rows so that both products run
    expo = np.repeat(rng.choice([0, 1, 100, 127, 244, 245, 250], (k + 63) // 64), 64)[:k]
    sc = (expo[:, None].astype(np.uint16) << 7) | rng.integers(0, 128, (k, n // 128)).astype(np.uint16)
    sc |= rng.integers(0, 2, sc.shape).astype(np.uint16) << 15
    rows = rng.integers(0, k, size=m)
    rows[:2] = 0, k - 1
    x = np.zeros((m, k), dtype=np.uint16)
    x[np.arange(m), rows] = 0x3F80
    out = host_bf16(K.int4_gemm_t(dev(qw), dev_bf16(sc), dev_bf16(x)))
    want = O.dequantize(qw, sc)[rows]
    got_f, want_f = O.bf16_to_f32(out), O.bf16_to_f32(want)
    assert np.array_equal(got_f, want_f)  # zeros by value: +0 and -0 both sum to +0


def test_gemm_t_non_finite_scales():
    """An infinite or NaN scale spoils the outputs of its own column group
    only, whatever the row's place in a slice."""
    import _dip_hip as K
    rng = np.random.default_rng(3)
    k, n = 776, 384
    qw = O.pack_int4(np.full((k, n), 3, dtype=np.int8))
    for row, bits in ((0, 0x7F80), (77, 0x7FC0), (k - 1, 0xFF80)):
        sc = np.full((k, n // 128), 0x3C00, dtype=np.uint16)
        sc[row, 1] = bits
        x = np.stack([random_bf16(rng, k) for _ in range(40)])
        x[:, row] = 0x3F80
        out = O.bf16_to_f32(host_bf16(K.int4_gemm_t(dev(qw), dev_bf16(sc), dev_bf16(x))))
        want = {0x7F80: np.inf, 0xFF80: -np.inf, 0x7FC0: np.nan}[bits]
        assert np.array_equal(out[:, 128:256], np.full((40, 128), want, np.float32), equal_nan=True)
        assert np.isfinite(out[:, :128]).all() and np.isfinite(out[:, 256:]).all()


def test_transposed_route_for_longer_prompts():
    """65 to 512 bf16 rows (768 of a large matrix) take the kernel; what it could not stand in for goes
    through torch's matmul, as it did."""
    import torch.autograd.forward_ad as fwd
    import qlinear as Q
    rng = np.random.default_rng(6)
    qw = dev(O.pack_int4(rng.integers(-8, 8, size=(512, 256)).astype(np.int8)))
    sc = dev_bf16(O.f32_to_bf16(rng.uniform(0.001, 0.01, (512, 2)).astype(np.float32)))
    w = Q.dequantize(qw, sc)
    g = torch.Generator(device="cuda").manual_seed(1)
    for rows in (65, 300, 512, 513, 768, 769):
        x = torch.randn(rows, 1024, device="cuda", generator=g).to(torch.bfloat16)
        for v in (x[:, :512], x[:, ::2], x[:, :512].reshape(1, rows, 512)):
            got, ref = Q.int4_linear_t(v, qw, sc), v @ w
            assert got.shape == ref.shape and got.dtype == ref.dtype
            assert float((got - ref).abs().max() / ref.abs().max()) < 1e-2
    x = torch.randn(100, 512, device="cuda", generator=g)
    assert torch.equal(Q.int4_linear_t(x, qw, sc), x @ w.float())
    xb = x.to(torch.bfloat16)
    xg = xb.clone().requires_grad_()
    Q.int4_linear_t(xg, qw, sc).sum().backward()
    assert xg.grad is not None
    with fwd.dual_level():
        tan = fwd.unpack_dual(Q.int4_linear_t(fwd.make_dual(xb, xb), qw, sc)).tangent
        assert torch.equal(tan, xb @ w)
    with pytest.raises(RuntimeError):
        Q.int4_linear_t(xb[:, :256].contiguous(), qw, sc)
