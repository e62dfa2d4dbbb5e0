"""GPU: tokens with infinite, NaN and very large values through the prompt
GEMMs, on every kernel of the dispatch, with one row past the last full tile.

The kernels sum (24 + q) * x and start from -24 * sum(x): a token for which that
leaves the range of fp32 is computed from plain q * s instead, so its outputs are
the ones of the definition (fp64 here): infinite where a non-zero weight meets
the infinity, NaN where a zero one does, finite where only the offset overflows.
Every other token keeps its bits.

Bound of a finite output: one bf16 rounding and fp32 sums, 2^-8 |ref| + 2^-17
sum |w x|; the SwiGLU's is the one of its own test."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import dip_oracle as O
from gpu_util import dev, dev_bf16, random_int4

pytestmark = pytest.mark.gpu

# (tokens, rows, K): the split kernel (staged scales, and scales from memory),
# the tiled one with two K parts, with one, and with four row tiles a wave
PLAIN = [(5, 33, 256), (40, 70, 384), (65, 2570, 640), (7, 48, 1 << 17), (100, 10249, 384),
         (64, 40961, 128), (700, 24001, 256)]
GATE_UP = [(5, 33, 256), (40, 70, 384), (7, 48, 1 << 17), (100, 5135, 384), (64, 20481, 128),
           (700, 12001, 256)]


def _tokens(m, k, seed):
    """bf16 [m, k] in (0.5, 1) and, for a few tokens, what is wrong with them."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = (torch.rand(m, k, device="cuda", generator=g) * 0.5 + 0.5).to(torch.bfloat16)
    bad = x.clone()
    at = torch.randint(0, k, (6,), generator=torch.Generator().manual_seed(seed)).tolist()
    rows = sorted({0, m // 3, m // 2, m - 1})
    bad[rows[0], at[0]] = float("inf")
    bad[rows[1], at[1]] = 3e37          # 24 times it overflows, 8 s times it does not
    if len(rows) > 2:
        bad[rows[2], at[2]] = float("nan")
    if len(rows) > 3:
        bad[rows[3], at[3]] = -float("inf")
        bad[rows[3], at[4]] = 1.0
    return x, bad, rows


def _ref(x, qw, sc):
    w = torch.from_numpy(O.dequant_f32(qw, sc)).cuda().double()
    xd = x.double()
    return xd @ w.t().contiguous(), xd.abs() @ w.abs().t().contiguous()


def _same_kind(got, ref):
    """NaN where the reference is, the same infinities."""
    assert torch.equal(got.isnan(), ref.isnan())
    inf = ref.isinf()
    assert torch.equal(got.isinf(), inf) and torch.equal(got[inf], ref[inf])


@pytest.mark.parametrize("m,n,k", PLAIN)
def test_gemm_tokens_out_of_range(m, n, k):
    import _dip_hip as K
    print(f"int4_gemm non-finite m={m} n={n} k={k}", flush=True)
    rng = np.random.default_rng(m + n + k)
    qw, sc = random_int4(rng, n, k)
    w, s = dev(qw), dev_bf16(sc)
    x, bad, rows = _tokens(m, k, seed=m + k)
    good, out = K.int4_gemm(w, s, x), K.int4_gemm(w, s, bad)
    keep = torch.ones(m, dtype=torch.bool, device="cuda")
    keep[rows] = False
    assert torch.equal(out[keep], good[keep])
    ref, terms = _ref(bad[rows], qw, sc)
    got = out[rows]
    _same_kind(got.double(), ref)
    ok = ref.isfinite()
    bound = 2.0 ** -8 * ref.abs() + 2.0 ** -17 * terms
    assert bool(ok[rows.index(m // 3)].all())
    assert bool(((got.double() - ref).abs() <= bound)[ok].all())


@pytest.mark.parametrize("m,n,k", GATE_UP)
def test_gate_up_tokens_out_of_range(m, n, k):
    import _dip_hip as K
    print(f"int4_gemm_swiglu non-finite m={m} n={n} k={k}", flush=True)
    rng = np.random.default_rng(m + n + k)
    (gq, gs), (uq, us) = random_int4(rng, n, k), random_int4(rng, n, k)
    w = dev(gq), dev_bf16(gs), dev(uq), dev_bf16(us)
    x, bad, rows = _tokens(m, k, seed=m + k)
    good, out = K.int4_gemm_swiglu(*w, x), K.int4_gemm_swiglu(*w, bad)
    keep = torch.ones(m, dtype=torch.bool, device="cuda")
    keep[rows] = False
    assert torch.equal(out[keep], good[keep])
    g, u = (_ref(bad[rows], q, s)[0].to(torch.bfloat16) for q, s in ((gq, gs), (uq, us)))
    _same_kind(out[rows].double(), (F.silu(g) * u).double())


@pytest.mark.parametrize("rows", [65, 300, 768])
def test_dense_route_with_an_infinite_activation(rows):
    """The routes of longer prompts keep what the dequantised product gives."""
    import qlinear as Q
    rng = np.random.default_rng(rows)
    qw, sc = (lambda a: (dev(a[0]), dev_bf16(a[1])))(random_int4(rng, 384, 256))
    _, x, bad = _tokens(rows, 256, seed=rows)
    ref = F.linear(x, Q.dequantize(qw, sc))
    _same_kind(Q.int4_linear(x, qw, sc), ref)
    w = Q.dequantize(qw, sc)[:256].contiguous()
    t = x.double() @ w.double()
    _same_kind(Q.int4_linear_t(x, qw[:256].contiguous(), sc[:256].contiguous()),
               t.to(torch.bfloat16))
