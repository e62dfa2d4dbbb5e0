"""GPU: attention over long caches (rows cut into splits and waves from the
position) against an fp64 softmax: every group size, one to sixteen kv heads
(few and many splits), positions at the edges of a wave's 32 rows, of a
workgroup's 128 and of the even cut, and a cache whose unused rows are NaN."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,max_len", [(1, 1, 9001), (4, 2, 5000), (32, 8, 1300), (40, 8, 4097),
                                            (64, 8, 2500), (64, 4, 3333), (32, 16, 1100)])
def test_long_cache_attention(nh, nkv, max_len):
    import _dip_hip as K
    hd, scale = 128, 1 / math.sqrt(128)
    g = torch.Generator(device="cuda").manual_seed(nh * nkv)
    q = torch.randn(nh, hd, device="cuda", generator=g).to(torch.bfloat16)
    kc = torch.randn(nkv, max_len, hd, device="cuda", generator=g).to(torch.bfloat16)
    vc = torch.randn(nkv, max_len, hd, device="cuda", generator=g).to(torch.bfloat16)
    for pos in (0, 30, 31, 32, 127, 128, 129, max_len // 2, max_len - 130, max_len - 1,
                max_len + 5):
        print(f"attention nh={nh} nkv={nkv} max_len={max_len} pos={pos}", flush=True)
        n = min(pos + 1, max_len)
        k1, v1 = kc.clone(), vc.clone()
        k1[:, n:], v1[:, n:] = math.nan, math.nan
        out = torch.empty(nh * hd, dtype=torch.bfloat16, device="cuda")
        K.decode_attention(q.view(-1), k1, v1, torch.tensor([pos], device="cuda"), out, scale)
        qd = q.double().view(nkv, nh // nkv, hd)
        ref = torch.stack([torch.softmax(qd[h] @ kc[h, :n].double().t().contiguous() * scale, -1)
                           @ vc[h, :n].double() for h in range(nkv)]).view(nh, hd)
        err = (out.view(nh, hd).double() - ref).abs()
        # the bf16 rounding of the result, and fp32 sums of at most max|v| per weight
        assert bool((err <= 2.0 ** -8 * ref.abs() + 1e-5 * vc.abs().max().double()).all())
