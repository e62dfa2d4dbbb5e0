"""GPU: the int4 quantizer and the down transpose against the CPU oracle, bit
for bit, where the fast quotient has to give way to the division: quotients
at and one step beside half-integers, tiny, infinite and NaN values; and on
buffers that are only as aligned as the C entries ask."""
import numpy as np
import pytest
import torch

import dip_oracle as O
from gpu_util import dev, dev_bf16, host_bf16

pytestmark = pytest.mark.gpu


def _edge_rows(rng, rows, cols):
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    g = w.reshape(-1, 128)
    half = (np.arange(-7, 7) + 0.5).astype(np.float32)
    for i in range(0, len(g), 3):  # max 7 t: the scale is t, quotients n + 1/2 up to rounding
        t = np.float32(rng.uniform(0.001, 0.1))
        ties = half * t
        g[i] = rng.uniform(-6.9, 6.9, 128).astype(np.float32) * t
        g[i, :14], g[i, 14:28], g[i, 28:42] = ties, np.nextafter(ties, 9), np.nextafter(ties, -9)
        g[i, 42] = 7 * t
    g[1] = 0.0
    g[4] *= 1e-9      # below the scale's floor
    g[7, 5] = np.inf  # an infinite scale
    g[10, 3] = np.nan
    g[13] = 3e38
    return w


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("rows,cols", [(5, 384), (7, 1408), (300, 1024)])
@pytest.mark.parametrize("shift", [0, 8])
def test_quantize_edges_bit_exact(rows, cols, bf16, shift):
    import _dip_hip as K
    print(f"quantize rows={rows} cols={cols} bf16={bf16} shift={shift}", flush=True)
    w = _edge_rows(np.random.default_rng(rows), rows, cols)
    if bf16:
        w = O.bf16_to_f32(O.f32_to_bf16(w))
    # NaN: fmax skips it, and it quantizes to -8, in the oracle's terms a very
    # large negative value under the group's scale
    nan = np.isnan(w)
    with np.errstate(all="ignore"):
        m = np.nanmax(np.abs(w.reshape(-1, 128)), axis=1)
        s = np.maximum(m / np.float32(7), np.float32(1e-8)).astype(np.float32)
        q = (w.reshape(-1, 128) / s[:, None]).reshape(w.shape)
        q = np.where(nan | np.isnan(q), -8, np.clip(np.rint(q), -8, 7)).astype(np.int8)
    finite = np.where(nan | np.isinf(w), 0, w).astype(np.float32)
    want_q, want_s = O.pack_int4(q), O.f32_to_bf16(s).reshape(rows, -1)
    clean = ~(nan | np.isinf(w)).reshape(-1, 128).any(axis=1)  # groups the oracle takes as they are
    oq, osc = O.quantize_int4_groupwise(finite)
    assert np.array_equal(oq.reshape(-1, 64)[clean], want_q.reshape(-1, 64)[clean])
    assert np.array_equal(osc.reshape(-1)[clean], want_s.reshape(-1)[clean])
    src = torch.from_numpy(w).cuda().to(torch.bfloat16 if bf16 else torch.float32)
    n = shift // src.element_size()
    buf = torch.empty(src.numel() + n, dtype=src.dtype, device="cuda")
    buf[n:] = src.view(-1)
    odd = 1 if shift else 0
    qw = torch.zeros(rows * cols // 2 + odd, dtype=torch.int8, device="cuda")
    sc = torch.zeros(rows, cols // 128, dtype=torch.bfloat16, device="cuda")
    K._check(K.lib.dip_quantize_int4(buf.data_ptr() + shift, int(bf16), qw.data_ptr() + odd,
                                     sc.data_ptr(), rows, cols, K._stream(sc.device)), "quantize")
    assert np.array_equal(qw[odd:].cpu().numpy().reshape(rows, -1), want_q)
    assert np.array_equal(host_bf16(sc), want_s)


@pytest.mark.parametrize("out_f,inter", [(128, 128), (256, 384), (384, 1024), (128, 640)])
@pytest.mark.parametrize("odd", [0, 1])
def test_transpose_down_bit_exact(out_f, inter, odd):
    """Tiles cut by the last columns; scales that make groups tiny, equal
    (many quotients on half-integers) and large."""
    import _dip_hip as K
    print(f"transpose out={out_f} inter={inter} odd={odd}", flush=True)
    rng = np.random.default_rng(out_f + inter)
    q = rng.integers(-8, 8, size=(out_f, inter)).astype(np.int8)
    sc = rng.choice(np.float32([0.004, 0.02, 0.01, 1e-10, 3.5]), size=(out_f, inter // 128))
    sc[: out_f // 2] = 0.01
    qw, sb = O.pack_int4(q), O.f32_to_bf16(sc)
    want_q, want_s = O.transpose_down_to_int4(qw, sb)
    src = torch.zeros(qw.size + odd, dtype=torch.int8, device="cuda")
    src[odd:] = dev(qw).view(-1)
    tq = torch.zeros(qw.size + odd, dtype=torch.int8, device="cuda")
    ts = torch.zeros(inter, out_f // 128, dtype=torch.bfloat16, device="cuda")
    s = dev_bf16(sb)
    K._check(K.lib.dip_transpose_down_int4(src.data_ptr() + odd, s.data_ptr(), tq.data_ptr() + odd,
                                           ts.data_ptr(), out_f, inter, K._stream(s.device)),
             "transpose")
    assert np.array_equal(tq[odd:].cpu().numpy().reshape(inter, -1), want_q)
    assert np.array_equal(host_bf16(ts), want_s)
