"""A prompt through the fused kernels: their prompt forms against the one-token
kernels bit for bit, and a whole prefill against the HF forward it replaces.

The two prefills differ by bf16 rounding only (sum order in RMSNorm, one q|k|v
product for three, the head of one row for all): the bound is the one of the
dense (keep 1.0) decode against the modules, 2e-2 of the largest logit."""
import pytest
import torch

from model_util import max_rel, tiny_config, tiny_model, write_checkpoint

pytestmark = pytest.mark.gpu


def _bf16(*shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, device="cuda", generator=g).to(torch.bfloat16)


@pytest.mark.parametrize("rows,n", [(1, 8), (3, 2048), (70, 2560), (5, 8192)])
def test_add_rmsnorm_rows_equals_single_rows(rows, n):
    import _dip_hip as K
    print(f"add_rmsnorm_rows {rows} x {n}", flush=True)
    h, add, w = _bf16(rows, n, seed=1), _bf16(rows, n, seed=2), _bf16(n, seed=3)
    for a in (add, None):
        got, out = h.clone(), torch.empty_like(h)
        K.add_rmsnorm_rows(got, a, w, out, 1e-6)
        for r in range(rows):
            one, x = h[r].clone(), torch.empty(n, dtype=h.dtype, device="cuda")
            K.add_rmsnorm(one, None if a is None else a[r], w, x, 1e-6)
            assert torch.equal(one, got[r]) and torch.equal(x, out[r])


@pytest.mark.parametrize("tokens,nh,nkv", [(1, 1, 1), (2, 4, 1), (40, 5, 1), (37, 32, 8)])
def test_qk_norm_rope_cache_rows_equals_single_tokens(tokens, nh, nkv):
    import _dip_hip as K
    print(f"qk_norm_rope_cache_rows {tokens} tokens, {nh}/{nkv} heads", flush=True)
    hd, max_len = 128, 41
    qkv = _bf16(tokens, (nh + 2 * nkv) * hd, seed=4)
    qw, kw = _bf16(hd, seed=5), _bf16(hd, seed=6)
    cos, sin = _bf16(max_len, hd, seed=7), _bf16(max_len, hd, seed=8)
    kc, vc = (torch.full((nkv, max_len, hd), 3.0, dtype=qkv.dtype, device="cuda") for _ in "kv")
    kr, vr = kc.clone(), vc.clone()
    q = torch.empty(tokens, nh * hd, dtype=qkv.dtype, device="cuda")
    K.qk_norm_rope_cache_rows(qkv, qw, kw, cos, sin, q, kc, vc, nh, nkv, 1e-6)
    for t in range(tokens):
        qt = torch.empty(nh * hd, dtype=qkv.dtype, device="cuda")
        K.qk_norm_rope_cache(qkv[t], qw, kw, cos, sin,
                             torch.tensor([t], device="cuda"), qt, kr, vr, nh, nkv, 1e-6)
        assert torch.equal(qt, q[t])
    assert torch.equal(kc, kr) and torch.equal(vc, vr)


@pytest.mark.parametrize("kv_heads,tokens", [(1, 2), (4, 65), (2, 65), (2, 300), (2, 530)])
def test_fused_prefill_matches_hf_forward(tmp_path, kv_heads, tokens):
    from dip_model import DIPDecoder
    from dip_stream_predispatch import load_streaming_dip
    print(f"prefill {tokens} tokens, {kv_heads} kv heads", flush=True)
    cfg = tiny_config(hidden=512, inter=1024, heads=4, kv_heads=kv_heads, head_dim=128, vocab=512,
                      max_pos=1024)
    write_checkpoint(tiny_model(cfg, seed=tokens), tmp_path)
    model, _, _ = load_streaming_dip(tmp_path, keep_ratio=0.6)
    ids = torch.randint(0, 512, (1, tokens), generator=torch.Generator().manual_seed(9))
    dec = DIPDecoder(model, 600)
    assert dec.fused and dec._prefill_fusible()
    got, kc, vc = dec.prefill(ids), dec.k_cache.clone(), dec.v_cache.clone()
    assert int(dec.pos) == tokens and int(dec.tok) == int(got.argmax())
    # whoever observes a module has the HF forward run it
    calls = []
    handle = model.model.norm.register_forward_hook(lambda *a: calls.append(1))
    assert not dec._prefill_fusible()
    ref = dec.prefill(ids)
    handle.remove()
    assert calls and dec._prefill_fusible()
    errs = [max_rel(a.float().cpu(), b.float().cpu())
            for a, b in ((got, ref), (kc, dec.k_cache), (vc, dec.v_cache))]
    print(f"  max_rel {errs}", flush=True)
    assert got.shape == ref.shape and max(errs) < 2e-2
