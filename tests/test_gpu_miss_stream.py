"""The miss stream read by the device (dip_stream_rows) and the hit/miss
assembly that feeds it: bytes and whole numbers, so every comparison is exact.

The stream is compared with index_select over row sizes that allow 16, 8, 4, 2
and 1-byte vectors, counts of none, one, some and all rows; the assembly with
its definition at sizes around a wave, a step of the workgroup and the number
of steps it keeps in registers; the module's two miss paths with each other."""
import numpy as np
import pytest
import torch

import dip_oracle as O
from gpu_util import dev, dev_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("widths", [(2560, 80, 2560, 80), (64, 2), (24,), (20, 12), (33, 1, 7)])
@pytest.mark.parametrize("n", [0, 1, 130, 700])
def test_stream_rows_matches_index_select(widths, n):
    import _dip_hip as K
    print(f"stream_rows {widths} n={n}", flush=True)
    g = torch.Generator().manual_seed(n)
    rows, most = 900, 700
    srcs = [torch.randint(-128, 128, (rows, w), dtype=torch.int8, generator=g).pin_memory()
            for w in widths]
    ids = torch.randperm(rows, generator=g)[:most].to(torch.int32)
    d = torch.device("cuda:0")
    dsts = [torch.full((most + 1, w), 7, dtype=torch.int8, device=d) for w in widths]
    assert K.stream_rows(srcs, ids.to(d), torch.tensor([n], dtype=torch.int32, device=d), dsts)
    for s, t in zip(srcs, dsts):
        assert torch.equal(t[:n].cpu(), s[ids[:n].long()])
        assert bool((t[n:].cpu() == 7).all())
    short = [t[: most - 1] for t in dsts]
    with pytest.raises(RuntimeError, match="too small"):
        K.stream_rows(srcs, ids.to(d), torch.tensor([n], dtype=torch.int32, device=d), short)


@pytest.mark.parametrize("k", [1, 63, 64, 65, 1023, 1024, 1025, 8192, 8193, 16385, 25600])
@pytest.mark.parametrize("share", [0.0, 0.3, 1.0])
def test_assembly_order(k, share):
    import _dip_hip as K
    print(f"assembly k={k} share={share}", flush=True)
    rng = np.random.default_rng(k)
    inter = 30000
    id2slot = np.full(inter, -1, np.int64)
    hot = np.sort(rng.choice(inter, int(share * inter), replace=False))
    id2slot[hot] = np.arange(hot.size)
    idx = rng.choice(inter, k, replace=False).astype(np.int32)
    comb, src, row, miss, counts = (t.cpu().numpy()
                                    for t in K.ca_assemble(dev(id2slot), dev(idx)))
    hit = id2slot[idx] >= 0
    n = int(hit.sum())
    assert counts.tolist() == [n, k - n]
    assert np.array_equal(comb, np.concatenate([idx[hit], idx[~hit]]))
    assert np.array_equal(src, np.repeat([0, 1], [n, k - n]))
    assert np.array_equal(row, np.concatenate([id2slot[idx[hit]], np.arange(k - n)]))
    assert np.array_equal(miss[: k - n], idx[~hit])


def test_module_with_pinned_and_pageable_matrices():
    """Matrices in pageable memory take the host gather; both give the same
    bits and counts."""
    from dip_ca import CABuffers, CADIPMlp
    H, I, keep = 1024, 3072, 0.6
    L = O.make_layer(H, I, seed=8)
    k = O.keep_count(I, keep)
    d = torch.device("cuda:0")
    m = CADIPMlp(dev(L["gate_qw"]), dev_bf16(L["gate_sc"]), dev(L["up_qw"]),
                 dev_bf16(L["up_sc"]), dev(L["down_t_qw"]), dev_bf16(L["down_t_sc"]),
                 CABuffers(k, H // 2, H // 128, H, H // 128, d), keep, 0.3, d,
                 down_transposed=True)
    m.set_cache(torch.arange(I).flip(0))
    x = dev_bf16(O.make_x(H, seed=2)).reshape(1, 1, -1)
    print("pinned", flush=True)
    y = m(x)
    counts = m.buf.last_n_hit, m.buf.last_n_miss
    assert sum(counts) == k and min(counts) > 0
    m.up_qw, m.up_sc = m.up_qw.clone(), m.up_sc.clone()
    assert not m.up_qw.is_pinned()
    print("pageable", flush=True)
    assert torch.equal(m(x), y)
    assert (m.buf.last_n_hit, m.buf.last_n_miss) == counts


def test_host_gather_chunks_and_its_staging():
    """The host gather's chunk size moves when rows are copied, never a bit; its
    pinned staging exists only once a matrix has needed it."""
    from dip_ca import CABuffers, CADIPMlp
    H, I, keep = 1024, 3072, 0.6
    L = O.make_layer(H, I, seed=9)
    k = O.keep_count(I, keep)
    d = torch.device("cuda:0")
    buf = CABuffers(k, H // 2, H // 128, H, H // 128, d)
    m = CADIPMlp(dev(L["gate_qw"]), dev_bf16(L["gate_sc"]), dev(L["up_qw"]),
                 dev_bf16(L["up_sc"]), dev(L["down_t_qw"]), dev_bf16(L["down_t_sc"]), buf, keep,
                 0.3, d, down_transposed=True)
    m.set_cache(torch.arange(I))
    x = dev_bf16(O.make_x(H, seed=4)).reshape(1, 1, -1)
    print("read by the device", flush=True)
    y = m(x)
    assert buf._pins is None
    m.up_qw = m.up_qw.clone()  # pageable
    for chunk in (k, 333, 64, 2048):
        print(f"host gather, chunks of {chunk}", flush=True)
        buf.stream_chunk = chunk
        assert torch.equal(m(x), y)
    assert buf.pin_up_qw.is_pinned() and buf.pin_dn_sc.shape == (k, H // 128)
