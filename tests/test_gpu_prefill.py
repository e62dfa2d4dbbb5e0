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


def _decoder(tmp_path, kv_heads=2, seed=3, **kw):
    from dip_model import DIPDecoder
    from dip_stream_predispatch import load_streaming_dip
    cfg = tiny_config(hidden=512, inter=1024, heads=4, kv_heads=kv_heads, head_dim=128, vocab=512,
                      max_pos=1024)
    write_checkpoint(tiny_model(cfg, seed=seed), tmp_path)
    model, _, _ = load_streaming_dip(tmp_path, keep_ratio=0.6)
    return DIPDecoder(model, 600, **kw)


def _ids(tokens):
    return torch.randint(0, 512, (1, tokens), generator=torch.Generator().manual_seed(9))


def _fused_against_hf(dec, ids):
    """max_rel of the logits and caches of the two prefills."""
    assert dec.fused and dec._prefill_fusible()
    got, kc, vc = dec.prefill(ids), dec.k_cache.clone(), dec.v_cache.clone()
    assert int(dec.pos) == ids.shape[1] and int(dec.tok) == int(got.argmax())
    handle = dec.model.model.norm.register_forward_hook(lambda *a: None)
    ref = dec.prefill(ids)
    handle.remove()
    return max(max_rel(a.float(), b.float())
               for a, b in ((got, ref), (kc, dec.k_cache), (vc, dec.v_cache)))


@pytest.mark.parametrize("tokens", [1, 2])
def test_fused_prefill_of_one_token(tmp_path, tokens):
    """One token takes the modules' decode step on both routes.  There the top-k
    picks channels, and a swapped one moves the logits by more than rounding: the
    bound is the sparse decode's against the modules, 8e-2."""
    print(f"prefill {tokens} token(s)", flush=True)
    assert _fused_against_hf(_decoder(tmp_path), _ids(tokens)) < (8e-2 if tokens == 1 else 2e-2)


@pytest.mark.parametrize("tokens", [1, 40, 300])
@pytest.mark.parametrize("resident", [False, True])
def test_fused_prefill_of_a_cache_aware_model(tmp_path, tokens, resident):
    from dip_ca import load_dip_ca
    from dip_model import DIPDecoder
    print(f"cache-aware prefill {tokens} tokens, resident channels {resident}", flush=True)
    cfg = tiny_config(hidden=512, inter=1024, heads=4, kv_heads=2, head_dim=128, vocab=512,
                      max_pos=1024)
    write_checkpoint(tiny_model(cfg, seed=4), tmp_path)
    model, _, cas = load_dip_ca(tmp_path, keep_ratio=0.6, cache_frac=0.3)
    if resident:
        for c in cas:
            c.set_cache(torch.randperm(c.inter, generator=torch.Generator().manual_seed(1)))
    dec = DIPDecoder(model, 600, use_graph=False)
    sparse = tokens == 1 and resident
    assert _fused_against_hf(dec, _ids(tokens)) < (8e-2 if sparse else 2e-2)


@pytest.mark.parametrize("what", ["hooks", "wrapped forward"])
@pytest.mark.parametrize("whose", ["embedding", "layers"])
def test_kept_inputs_and_outputs_stay_as_they_were(tmp_path, what, whose):
    """Whoever keeps what the embedding, the MLPs and the o projections take and
    give finds it unchanged after the prompt; the layers' keep the fused route."""
    print(f"prefill with kept tensors: {what} of the {whose}", flush=True)
    dec = _decoder(tmp_path)
    inner = dec.model.model
    mods = ([inner.embed_tokens] if whose == "embedding" else
            [m for L in inner.layers for m in (L.mlp, L.self_attn.o_proj)])
    kept = []

    def keep(*tensors):
        kept.extend((t, t.clone()) for t in tensors)

    handles = []
    for m in mods:
        if what == "hooks":
            handles.append(m.register_forward_hook(lambda mod, a, out: keep(a[0], out)))
        else:
            def forward(x, f=m.forward):
                out = f(x)
                keep(x, out)
                return out
            m.forward = forward
    assert dec._prefill_fusible() == (whose == "layers")
    dec.prefill(_ids(65))
    assert len(kept) == 2 * len(mods)
    assert all(torch.equal(t, was) for t, was in kept)
    for h in handles:
        h.remove()


def _replacements():
    import torch.nn as nn
    from transformers.models.qwen3 import modeling_qwen3 as Q

    class Wrapped(nn.Module):  # an adapter, a probe: anything around a module
        def __init__(self, inner, calls):
            super().__init__()
            self.inner, self.calls = inner, calls

        def __getattr__(self, name):
            try:
                return super().__getattr__(name)
            except AttributeError:
                return getattr(super().__getattr__("inner"), name)

        def forward(self, *a, **kw):
            self.calls.append(1)
            return self.inner(*a, **kw)

    def swap(parent, name):
        def do(dec, calls, monkeypatch):
            p = parent(dec)
            setattr(p, name, Wrapped(getattr(p, name), calls))
        return do

    def layer(dec, calls, monkeypatch):
        dec.model.model.layers[1] = Wrapped(dec.model.model.layers[1], calls)

    def class_forward(cls):
        def do(dec, calls, monkeypatch):
            orig = cls.forward

            def forward(self, *a, **kw):
                calls.append(1)
                return orig(self, *a, **kw)
            monkeypatch.setattr(cls, "forward", forward)
        return do

    def subclass(dec, calls, monkeypatch):
        norm = dec.model.model.layers[0].input_layernorm

        class Other(type(norm)):
            def forward(self, x):
                calls.append(1)
                return super().forward(x)
        norm.__class__ = Other

    def weights(dec, calls, monkeypatch):
        p = dec.model.model.layers[1].self_attn.k_proj
        p.qweight = torch.roll(p.qweight, 1, 0)
        calls.append(1)

    L0 = lambda dec: dec.model.model.layers[0]
    A0 = lambda dec: dec.model.model.layers[0].self_attn
    return {"input norm": swap(L0, "input_layernorm"),
            "post-attention norm": swap(L0, "post_attention_layernorm"),
            "q norm": swap(A0, "q_norm"), "k projection": swap(A0, "k_proj"),
            "attention": swap(L0, "self_attn"), "layer": layer,
            "final norm": swap(lambda d: d.model.model, "norm"),
            "embedding": swap(lambda d: d.model.model, "embed_tokens"),
            "norm class": class_forward(Q.Qwen3RMSNorm),
            "attention class": class_forward(Q.Qwen3Attention),
            "layer class": class_forward(Q.Qwen3DecoderLayer),
            "norm subclass": subclass, "projection weights": weights}


@pytest.mark.parametrize("what", ["input norm", "post-attention norm", "q norm", "k projection",
                                  "attention", "layer", "final norm", "embedding", "norm class",
                                  "attention class", "layer class", "norm subclass",
                                  "projection weights"])
def test_replaced_modules_run(tmp_path, what, monkeypatch):
    """A module, class method or weight replaced after the decoder was made
    serves its prompts: the logits are the model's own, now."""
    print(f"prefill with a replaced {what}", flush=True)
    dec = _decoder(tmp_path)
    ids = _ids(65)
    calls = []
    _replacements()[what](dec, calls, monkeypatch)
    assert not calls or what == "projection weights"
    got = dec.prefill(ids)
    assert calls
    with torch.no_grad():
        ref = dec.model(ids.cuda()).logits[0, -1]
    assert max_rel(got.float(), ref.float()) < 2e-2


def test_prefill_under_modes_runs_the_model(tmp_path):
    """Autocast to another type and dispatch modes act on the model's own ops."""
    from torch.utils._python_dispatch import TorchDispatchMode
    print("prefill under modes", flush=True)
    dec = _decoder(tmp_path)
    seen = []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func.name())
            return func(*args, **(kwargs or {}))

    with Dispatch():
        dec.prefill(_ids(65))
    assert any("rsqrt" in s for s in seen)  # the norms
    with torch.autocast("cuda", dtype=torch.float16):
        assert not dec._prefill_fusible()
    assert dec._prefill_fusible()


def test_two_decoders_of_one_model(tmp_path):
    """A second decoder of the model leaves the first one's prompts as they were."""
    from dip_model import DIPDecoder
    print("prefill of two decoders", flush=True)
    first = _decoder(tmp_path)
    before = first.prefill(_ids(65))
    second = DIPDecoder(first.model, 300)
    for dec in (first, second):
        assert dec._prefill_fusible()
        assert torch.equal(dec.prefill(_ids(65)), before)


def test_stand_in_for_the_model(tmp_path):
    """An object with the model's parts, but no module of its class, decodes with
    the fused steps and runs its own forward for prompts."""
    from types import SimpleNamespace
    from dip_model import DIPDecoder
    print("prefill of a stand-in", flush=True)
    dec = _decoder(tmp_path)
    want, step = dec.prefill(_ids(65)), dec.step()
    m, calls = dec.model, []

    class StandIn:
        config, lm_head = m.config, m.lm_head
        model = SimpleNamespace(layers=list(m.model.layers), embed_tokens=m.model.embed_tokens,
                                norm=m.model.norm, rotary_emb=m.model.rotary_emb)

        def __call__(self, **kw):
            calls.append(1)
            return m(**kw)

    other = DIPDecoder(StandIn(), 600)
    assert other.fused and not other._prefill_fusible()
    assert max_rel(other.prefill(_ids(65)).float(), want.float()) < 2e-2 and calls
    assert max_rel(other.step().float(), step.float()) < 8e-2  # the sparse bound
