"""GPU: gate, up and the SwiGLU in one launch, at the edges of the tiles (row
counts that leave a last tile of 1 to 15 rows, matrices of fewer than 16, odd
scale runs, 2-byte aligned scales, K too long for the staged scales) and on
both sides of each dispatch line, against fp64.

Bound: a projection p is off by d(p) = 2^-8 |p| + 2^-17 sum |w x| (one bf16
rounding, fp32 sums); |silu'| < 1.1, so silu is off by ds = 1.1 d(g) + 2^-8 |s|
and the product by |u| ds + (|s| + ds) d(u), and its own rounding 2^-8."""
import numpy as np
import pytest
import torch

import dip_oracle as O
from gpu_util import dev, dev_bf16, random_bf16, random_int4

pytestmark = pytest.mark.gpu

CASES = [(2, 5, 128), (2, 16, 384), (3, 17, 128), (16, 31, 640), (17, 1000, 256), (31, 40, 1152),
         (16, 7000, 384), (32, 6161, 256),                  # split kernel, a pair of tiles, 4 waves
         (16, 12322, 384), (9, 12321, 256), (32, 14343, 256),  # two pairs of tiles
         (33, 8, 512), (48, 1003, 384), (65, 1285, 640),    # split kernel, several token blocks
         (64, 10241, 256), (100, 5135, 384),                # tiled, two K parts
         (64, 20481, 128), (333, 3500, 640),                # tiled, one K part
         (700, 12001, 256),                                 # tiled, four row tiles a wave
         (7, 48, 1 << 17), (40, 33, 40960)]                 # scales from memory


@pytest.mark.parametrize("m,n,k", CASES)
@pytest.mark.parametrize("odd", [0, 1])
def test_gate_up_tile_edges(m, n, k, odd):
    import _dip_hip as K
    print(f"int4_gemm_swiglu m={m} n={n} k={k} odd={odd}", flush=True)
    rng = np.random.default_rng(m + n + k)
    mats = [random_int4(rng, n, k) for _ in range(2)]
    x = dev_bf16(np.stack([random_bf16(rng, k) for _ in range(m)]))
    x = (x * k ** -0.5).to(torch.bfloat16)  # gates around one
    ws, ss, ref = [], [], []
    for i, (qw, sc) in enumerate(mats):
        s = torch.zeros(sc.size + 1, dtype=torch.bfloat16, device="cuda")
        o = odd * i  # one of the two matrices' scales
        s[o:o + sc.size] = dev_bf16(sc).view(-1)
        ws.append(dev(qw))
        ss.append(s[o:])
        wf = torch.from_numpy(O.dequant_f32(qw, sc)).cuda().double()
        p, terms = x.double() @ wf.t().contiguous(), x.double().abs() @ wf.abs().t().contiguous()
        ref.append((p, 2.0 ** -8 * p.abs() + 2.0 ** -17 * terms))
    guard = torch.full((m * n + 64,), 7.0, dtype=torch.bfloat16, device="cuda")
    K._check(K.lib.dip_int4_gemm_swiglu(ws[0].data_ptr(), ss[0].data_ptr(), ws[1].data_ptr(),
                                        ss[1].data_ptr(), x.data_ptr(), guard.data_ptr(), m, n, k,
                                        K._stream(x.device)), "dip_int4_gemm_swiglu")
    assert bool((guard[m * n:] == 7.0).all())
    (g, dg), (u, du) = ref
    s = g * torch.sigmoid(g)
    ds = 1.1 * dg + 2.0 ** -8 * s.abs()
    bound = u.abs() * ds + (s.abs() + ds) * du + 2.0 ** -8 * (s * u).abs()
    assert bool(((guard[:m * n].view(m, n).double() - s * u).abs() <= bound).all())


@pytest.mark.parametrize("rows", [1, 2, 64, 65, 512, 513, 768, 769])
def test_dense_route_equals_the_separate_products(rows):
    """StreamingDIPMlp._dense over its dispatch lines against silu(gate) * up of
    the separate routes; inputs the kernel may not stand in for keep them."""
    import torch.nn.functional as F
    from dip_stream_predispatch import SharedBuffers, StreamingDIPMlp
    from qlinear import int4_linear, int4_linear_t
    H, I = 512, 1024
    rng = np.random.default_rng(rows)
    q = [(dev(a), dev_bf16(b)) for a, b in (random_int4(rng, *s) for s in ((I, H), (I, H), (I, H)))]
    shared = SharedBuffers(600, H // 2, H // 128, H, H // 128, "cuda:0")
    m = StreamingDIPMlp(*q[0], *q[1], *q[2], shared, 0.6, "cuda:0", down_transposed=True)
    gen = torch.Generator(device="cuda").manual_seed(rows)
    wide = torch.randn(rows, 2 * H, device="cuda", generator=gen).to(torch.bfloat16)
    for x in (wide[None, :, :H], wide[None, :, ::2], wide[:, :H], wide[:, :H].float()):
        print(f"dense {tuple(x.shape)} {x.dtype}", flush=True)
        h = F.silu(int4_linear(x, *q[0])) * int4_linear(x, *q[1])
        ref, got = int4_linear_t(h, *q[2]), m._dense(x)
        assert got.shape == ref.shape and got.dtype == ref.dtype
        assert float((got - ref).abs().max() / ref.abs().max()) < 1e-2
    if rows > 64:
        x = wide[None, :, :H].contiguous().requires_grad_()
        assert m._dense(x).requires_grad
