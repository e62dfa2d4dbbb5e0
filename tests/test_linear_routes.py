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


def _mlp(H=256, I=512):
    from dip_stream_predispatch import SharedBuffers, StreamingDIPMlp
    shared = SharedBuffers(300, H // 2, H // 128, H, H // 128, "cuda:0")
    w = [t for i in range(3) for t in _weight(I, H, i)]
    return StreamingDIPMlp(*w, shared, 0.6, "cuda:0", down_transposed=True)


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


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [65, 300, 600])
def test_autocast_decides_the_type(rows):
    """Under autocast the product is torch's, in autocast's type."""
    import qlinear as Q
    print(f"autocast, {rows} rows", flush=True)
    qw, sc = _weight(384, 256, device="cuda")
    w, x, xt = Q.dequantize(qw, sc), _x(rows, 256, "cuda"), _x(rows, 384, "cuda")
    m = _mlp()
    for dtype in (torch.float16, torch.bfloat16):
        with torch.no_grad(), torch.autocast("cuda", dtype=dtype):
            got, ref = Q.int4_linear(x, qw, sc), F.linear(x, w)
            assert got.dtype == ref.dtype == dtype
            assert float((got - ref).abs().max() / ref.abs().max()) < 1e-2
            got, ref = Q.int4_linear_t(xt, qw, sc), xt @ w
            assert got.dtype == ref.dtype == dtype
            assert float((got - ref).abs().max() / ref.abs().max()) < 1e-2
            assert m(x.view(1, rows, 256)).dtype == dtype


@pytest.mark.gpu
def test_modes_see_the_product():
    """A dispatch or function mode sees torch's product; a default device is no
    such mode."""
    import _dip_hip as K
    import qlinear as Q
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    print("modes", flush=True)
    seen = []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func.name())
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))

    qw, sc = _weight(384, 256, device="cuda")
    x, xt, m = _x(100, 256, "cuda"), _x(100, 384, "cuda"), _mlp()
    for mode, product in ((Dispatch, "mm"), (Function, "linear")):
        for f in (lambda: Q.int4_linear(x, qw, sc), lambda: m(x.view(1, 100, 256))):
            seen.clear()
            with torch.no_grad(), mode():
                f()
            assert any(product in s for s in seen), (mode, seen)
    seen.clear()
    with torch.no_grad(), Dispatch():
        Q.int4_linear_t(xt, qw, sc)
    assert any("mm" in s for s in seen)
    with torch.no_grad(), torch.device("cuda"):
        assert torch.equal(Q.int4_linear(x, qw, sc), K.int4_gemm(qw, sc, x))


# (rows, out, in, serves) on 256 CUs: both sides of each line
@pytest.mark.parametrize("rows,out_f,in_f,serves", [
    (384, 5120, 8192, True), (448, 5120, 8192, False), (512, 5120, 8192, False),
    (256, 10240, 5120, True), (257, 6144, 4096, True), (257, 6528, 4096, False),
    (257, 6656, 4096, True), (448, 4096, 4096, True), (448, 4608, 4096, False),
    (448, 6144, 4096, True), (449, 8704, 4096, False), (449, 8704, 2048, True), (449, 9600, 4096, True), (320, 9728, 2560, True),
    (448, 7040, 4096, True), (512, 7424, 8192, False), (448, 8704, 8192, True), (448, 8704, 6144, True), (384, 8704, 6144, False),
    (512, 8704, 8192, False), (512, 25600, 5120, True), (513, 25600, 5120, False),
    (65, 1024, 5120, True)])
def test_linear_rule(rows, out_f, in_f, serves):
    import qlinear as Q
    assert Q._gemm_serves(rows, out_f, in_f, 256) == serves


@pytest.mark.parametrize("rows,in_f,out_f,serves", [
    (512, 25600, 5120, True), (768, 25600, 5120, True), (769, 25600, 5120, False),
    (768, 17408, 5120, True), (832, 17408, 5120, False), (384, 6144, 5120, True),
    (448, 6144, 5120, False), (512, 12288, 4096, True), (513, 12288, 4096, False),
    (320, 12288, 4096, True), (768, 17408, 2560, True), (513, 16384, 2560, False), (192, 3072, 1024, False),
    (512, 9728, 2560, True)])
def test_transposed_rule(rows, in_f, out_f, serves):
    import _dip_hip as K
    import qlinear as Q
    splits = K.int4_gemm_t_splits(rows, out_f, in_f)  # 256 CUs, here and on the device
    assert Q._gemm_t_serves(rows, in_f, out_f, splits, 256) == serves


def _calls(monkeypatch, *names):
    import _dip_hip as K
    seen = []
    for n in names:
        def wrapped(*a, n=n, f=getattr(K, n), **kw):
            seen.append(n)
            return f(*a, **kw)
        monkeypatch.setattr(K, n, wrapped)
    return seen


def _close(got, x, w):
    """One bf16 rounding and fp32 sums, against fp64 (the weights are the
    route's: exact q * s, or rounded to bf16 once, 2^-9 of each term)."""
    ref, terms = x.double() @ w.double(), x.double().abs() @ w.double().abs()
    return bool(((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -9 * terms).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rows,entry", [(513, "int4_gemm_t"), (768, "int4_gemm_t"),
                                        (769, "dequant_t")])
def test_transposed_route_of_a_long_matrix(rows, entry, monkeypatch):
    import qlinear as Q
    print(f"transposed route, 16640 x 2560, {rows} rows", flush=True)
    qw, sc = _weight(16640, 2560, device="cuda")
    x = _x(rows, 16640, "cuda")
    w = Q.dequantize(qw, sc)
    seen = _calls(monkeypatch, "int4_gemm_t", "dequant_t")
    got = Q.int4_linear_t(x, qw, sc)
    assert seen == [entry] and _close(got, x, w)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,in_f,entry", [(384, 6144, "int4_gemm"), (448, 6144, "dequant_rows"),
                                             (448, 4096, "int4_gemm"), (513, 4096, "dequant_rows")])
def test_linear_route_by_workgroups(rows, in_f, entry, monkeypatch):
    import qlinear as Q
    print(f"linear route, 5120 x {in_f}, {rows} rows", flush=True)
    qw, sc = _weight(5120, in_f, device="cuda")
    x = _x(rows, in_f, "cuda")
    w = Q.dequantize(qw, sc).t()
    seen = _calls(monkeypatch, "int4_gemm", "dequant_rows")
    got = Q.int4_linear(x, qw, sc)
    assert seen == [entry] and _close(got, x, w)
