"""The projections' routes: what the int4 kernels may not stand in for takes the
dequantised product, as it did before they served longer prompts."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import dip_oracle as O


def _weight(rows, cols, seed=0, device="cpu"):
    rng = np.random.default_rng(seed)
    q = O.pack_int4(rng.integers(-8, 8, size=(rows, cols)).astype(np.int8))
    s = rng.uniform(0.001, 0.01, (rows, cols // 128)).astype(np.float32)
    return torch.from_numpy(q).to(device), torch.from_numpy(s).to(torch.bfloat16).to(device)


def _x(rows, cols, device="cpu"):
    g = torch.Generator().manual_seed(rows)
    return torch.randn(rows, cols, generator=g).to(torch.bfloat16).to(device)


@pytest.mark.parametrize("rows", [65, 200, 512, 513, 768])
def test_host_tensors_take_the_dequantised_product(rows):
    import qlinear as Q
    qw, sc = _weight(384, 256)
    w, x = Q.dequantize(qw, sc), _x(rows, 256)
    assert torch.equal(Q.int4_linear(x, qw, sc), F.linear(x, w))
    xt = _x(rows, 384)
    assert torch.equal(Q.int4_linear_t(xt, qw, sc), xt @ w)
    assert Q.int4_gate_up(x, qw, sc, qw, sc) is None


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [65, 512, 600])
def test_shapes_without_a_kernel_keep_their_product(rows):
    """An input dimension of the transposed layout that is no multiple of 8."""
    import qlinear as Q
    print(f"shapes without a kernel, {rows} rows", flush=True)
    qw, sc = _weight(260, 256, device="cuda")
    x = _x(rows, 260, "cuda")
    assert torch.equal(Q.int4_linear_t(x, qw, sc), x @ Q.dequantize(qw, sc))
