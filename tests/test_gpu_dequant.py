"""GPU: row dequantisation against the oracle, bit for bit: runs shorter than
a block's span and with a remainder, scales over the whole bf16 range (q * s
subnormal, overflowing, of either sign), ids out of range, and buffers that
are only byte / element aligned."""
import numpy as np
import pytest
import torch

import dip_oracle as O
from gpu_util import dev, dev_bf16, host_bf16

pytestmark = pytest.mark.gpu


def _case(rows, cols, seed):
    rng = np.random.default_rng(seed)
    qw = O.pack_int4(rng.integers(-8, 8, size=(rows, cols)).astype(np.int8))
    expo = rng.integers(0, 255, size=(rows, cols // 128)).astype(np.uint16)  # 0: subnormal scales
    sc = (expo << 7) | rng.integers(0, 128, size=expo.shape).astype(np.uint16)
    return qw, sc | (rng.integers(0, 2, size=expo.shape).astype(np.uint16) << 15)


def _same(got, want):
    """Equal bits, any NaN matching any NaN."""
    g, w = np.asarray(got), np.asarray(want)
    return np.array_equal(np.isnan(g), np.isnan(w)) and np.array_equal(
        g[~np.isnan(g)].view(np.uint32), w[~np.isnan(w)].view(np.uint32))


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("rows,cols", [(1, 128), (3, 384), (65, 128), (129, 8192)])
def test_dequant_every_scale_range(mode, rows, cols):
    import _dip_hip as K
    print(f"dequant rows={rows} cols={cols} mode={mode}", flush=True)
    qw, sc = _case(rows, cols, rows + cols)
    with np.errstate(over="ignore"):
        want = O.dequant_f32(qw, sc) if mode == 0 else O.bf16_to_f32(O.dequantize(qw, sc))
    idx = np.random.default_rng(1).permutation(rows).astype(np.int32)
    idx[0] = rows  # out of range: a row of NaN
    gathered = want[np.minimum(idx, rows - 1)].copy()
    gathered[0] = np.nan

    def host(t):
        return t.cpu().numpy() if mode == 0 else O.bf16_to_f32(host_bf16(t))

    assert _same(host(K.dequant_rows(dev(qw), dev_bf16(sc), mode=mode)), want)
    assert _same(host(K.dequant_rows(dev(qw), dev_bf16(sc), dev(idx), mode=mode)), gathered)
    # the C entry on buffers that are not aligned for vector accesses
    buf = torch.zeros(qw.size + 1, dtype=torch.int8, device="cuda")
    buf[1:] = dev(qw).view(-1)
    item = 4 if mode == 0 else 2
    out = torch.zeros(rows * cols + 1, dtype=torch.float32 if mode == 0 else torch.bfloat16,
                      device="cuda")
    s = dev_bf16(sc)
    K._check(K.lib.dip_dequant_rows(buf.data_ptr() + 1, s.data_ptr(), None, out.data_ptr() + item,
                                    rows, rows, cols, mode, K._stream(s.device)), "dequant")
    assert _same(host(out[1:].reshape(rows, cols)), want)
