"""The dense route of the large products (the weight dequantized once into the workspace, then a
plain 16-bit GEMM): forward and input gradient at the sizes where its tiles end raggedly (rows
and tokens past a 256- or 128-wide tile, reductions of an odd number of 64-deep steps, whole
256x256 tiles, 128x128 tiles, both in one launch, a split reduction), against fp32 products of
the dequantized weight and, with one-hot rows, against the weight bit for bit."""

import pytest
import torch

from tests.gpu_util import OP_DX, PATH_DENSE, assert_rel, banner, linear_path, random_weight

pytestmark = pytest.mark.gpu

# ([rows of the stacked segments], K, M, splits of the reduction)
FWD = [([520, 776], 3072, 1300, 1), ([520, 776], 3072, 3001, 3), ([2312], 2048, 4100, 1),
       ([1288], 6144, 2049, 1), ([1288], 6144, 4100, 2), ([3080], 1920, 3001, 1),
       ([8960, 8960], 1536, 2048, 1)]
DX = [([3008, 64], 1536, 1300, 1), ([3008, 64], 1536, 3001, 3), ([2112], 1152, 4100, 1),
      ([4032], 1408, 2049, 1), ([10048], 1152, 3001, 4), ([1536, 256, 256], 1536, 1025, 1)]


def _need(weights, m, dtype, dx):
    from solution import _lib, kernels

    f = _lib.load().nf4_linear_dx_workspace if dx else _lib.load().nf4_linear_fwd_workspace
    return f(m, kernels._descs(weights), len(weights), _lib.DTYPE_CODE[dtype])


def _setup(rows, k, m, splits, dtype, dev, dx):
    from solution import kernels

    weights = [random_weight(n, k, seed=300 + i, dev=dev) for i, n in enumerate(rows)]
    # the route is taken: the workspace holds the 16-bit weight in strips of 128 rows, and the
    # fp32 partials of a split reduction
    p, r = (k, sum(rows)) if dx else (sum(rows), k)
    partials = 4 * splits * m * p if splits > 1 else 0
    assert _need(weights, m, dtype, dx) == -(-p // 128) * 256 * r + partials
    w = kernels.dequant(weights, dtype)
    junk = torch.full((64 << 20,), float("nan"), dtype=torch.float32, device=dev)
    del junk  # the workspace and outputs come from this memory
    return weights, w


def _lora(m, r, n_in, n_out, dtype, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    t = torch.randn(m, r, generator=g, device=dev).to(dtype)
    b = (torch.randn(n_out, r, generator=g, device=dev) * 0.05).to(dtype)
    return t, b


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,k,m,splits", FWD)
def test_dense_forward(cuda, dtype, rows, k, m, splits):
    from solution import kernels

    banner("dense fwd", dtype, rows, k, m, splits)
    weights, w = _setup(rows, k, m, splits, dtype, cuda, False)
    n = sum(rows)
    g = torch.Generator(device=cuda).manual_seed(1)
    # rows 24 elements apart from the next: what lies between is NaN
    buf = torch.full((m, k + 24), float("nan"), dtype=dtype, device=cuda)
    x = buf[:, :k]
    x.copy_(torch.randn(m, k, generator=g, device=cuda))
    bias = torch.randn(n, generator=g, device=cuda).to(dtype)
    r = 12
    t, b = _lora(m, r, k, rows[-1], dtype, cuda, 2)
    lora = [kernels.make_lora(len(rows) - 1, r, 0.5, t=t, b=b)]
    y = kernels.linear_fwd(x, weights, bias, lora)
    ref = x.float() @ w.float().T + bias.float()
    ref[:, n - rows[-1]:] += 0.5 * t.float() @ b.float().T
    assert_rel(y, ref, what="y")
    # one-hot rows pick weight columns: bit for bit
    idx = (torch.arange(m, device=cuda) * 61 + 7) % k
    hot = torch.zeros(m, k, dtype=dtype, device=cuda)
    hot[torch.arange(m, device=cuda), idx] = 1
    assert torch.equal(kernels.linear_fwd(hot, weights), w.T[idx])
    # an output that the 16-byte stores do not fit goes the other way, into the same tolerance
    out = torch.empty(m, n + 1, dtype=dtype, device=cuda)[:, 1:]
    assert_rel(kernels.linear_fwd(x, weights, bias, lora, out=out), ref, what="unaligned y")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,k,m,splits", DX)
def test_dense_input_gradient(cuda, dtype, rows, k, m, splits):
    from solution import kernels

    banner("dense dx", dtype, rows, k, m, splits)
    weights, w = _setup(rows, k, m, splits, dtype, cuda, True)
    n = sum(rows)
    g = torch.Generator(device=cuda).manual_seed(3)
    buf = torch.full((m, n + 8), float("nan"), dtype=dtype, device=cuda)
    dy = buf[:, :n]
    dy.copy_(torch.randn(m, n, generator=g, device=cuda))
    r = 20
    da, at = _lora(m, r, n, k, dtype, cuda, 4)
    a = at.T.contiguous()
    lora = [kernels.make_lora(0, r, 2.0, a=a, da=da)]  # (da holds the scale)
    ref = dy.float() @ w.float() + da.float() @ a.float()
    dx = kernels.linear_dx(dy, weights, lora)
    assert_rel(dx, ref, what="dx")
    idx = (torch.arange(m, device=cuda) * 61 + 7) % n
    hot = torch.zeros(m, n, dtype=dtype, device=cuda)
    hot[torch.arange(m, device=cuda), idx] = 1
    assert torch.equal(kernels.linear_dx(hot, weights), w[idx])
    base = dx.clone()
    assert_rel(kernels.linear_dx(dy, weights, lora, out=base, accumulate=True),
               ref + dx.float(), what="accumulated dx")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,k,m,splits", FWD[:3])
def test_dense_forward_keeps_non_finite_lora_to_its_segment(cuda, dtype, rows, k, m, splits):
    """Slabs that start or end inside a tile, one token's t infinite and one's NaN: what lies
    outside the slab's columns, and every other token, is as with a finite t, bit for bit."""
    from solution import kernels

    banner("dense fwd non-finite", dtype, rows, k, m, splits)
    rows = rows if len(rows) > 1 else [72, rows[0] - 72]
    weights, _ = _setup(rows, k, m, splits, dtype, cuda, False)
    g = torch.Generator(device=cuda).manual_seed(6)
    x = torch.randn(m, k, generator=g, device=cuda).to(dtype)
    r, starts = 12, [0, rows[0]]
    for seg in (0, 1):
        t, b = _lora(m, r, k, rows[seg], dtype, cuda, 7 + seg)
        b = b.abs() + 0.01  # (an infinity stays one)
        bad = t.clone()
        bad[5, 3], bad[m - 1] = float("inf"), float("nan")
        y, y_bad = (kernels.linear_fwd(x, weights, None, [kernels.make_lora(seg, r, 0.5, t=v, b=b)])
                    for v in (t, bad))
        inside = torch.zeros(sum(rows), dtype=torch.bool, device=cuda)
        inside[starts[seg]:starts[seg] + rows[seg]] = True
        assert torch.equal(y_bad[:, ~inside], y[:, ~inside])
        assert bool((y_bad[5, inside] == float("inf")).all())
        assert bool(y_bad[m - 1, inside].isnan().all())
        rest = torch.ones(m, dtype=torch.bool, device=cuda)
        rest[5] = rest[m - 1] = False
        assert torch.equal(y_bad[rest], y[rest])


def _mixed(rows, k, dev):
    """Segments of different formats: nested absmax with blocks of 64, fp32 absmax with blocks of
    128, nested with blocks of 256."""
    kinds = [(64, True), (128, False), (256, True)]
    return [random_weight(n, k, seed=340 + i, dev=dev, blocksize=kinds[i % 3][0], nested=kinds[i % 3][1])
            for i, n in enumerate(rows)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,k,m", [([520, 200, 576], 3072, 1300), ([520, 200, 576], 3072, 3001),
                                      ([776, 520], 2048, 4100)])
def test_dense_forward_mixed_weights_and_slabs(cuda, dtype, rows, k, m):
    """Segments of three weight formats and an adapter on the first and on the last one, their
    edges inside tiles."""
    from solution import kernels

    banner("dense fwd mixed", dtype, rows, k, m)
    weights = _mixed(rows, k, cuda)
    assert linear_path(weights, m)[0] == PATH_DENSE
    w = kernels.dequant(weights, dtype)
    n = sum(rows)
    g = torch.Generator(device=cuda).manual_seed(11)
    x = torch.randn(m, k, generator=g, device=cuda).to(dtype)
    bias = torch.randn(n, generator=g, device=cuda).to(dtype)
    ref, loras = x.float() @ w.float().T + bias.float(), []
    for seg, r, lo in ((0, 16, 0), (len(rows) - 1, 40, n - rows[-1])):
        t, b = _lora(m, r, k, rows[seg], dtype, cuda, 12 + seg)
        loras.append(kernels.make_lora(seg, r, 0.5, t=t, b=b))
        ref[:, lo:lo + rows[seg]] += 0.5 * t.float() @ b.float().T
    assert_rel(kernels.linear_fwd(x, weights, bias, loras), ref, what="y")
    idx = (torch.arange(m, device=cuda) * 61 + 7) % k
    hot = torch.zeros(m, k, dtype=dtype, device=cuda)
    hot[torch.arange(m, device=cuda), idx] = 1
    assert torch.equal(kernels.linear_fwd(hot, weights), w.T[idx])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,k,m", [([1536, 256, 320], 1536, 1025), ([3008, 64, 128], 1536, 3001)])
def test_dense_input_gradient_mixed_weights_and_slabs(cuda, dtype, rows, k, m):
    from solution import kernels

    banner("dense dx mixed", dtype, rows, k, m)
    weights = _mixed(rows, k, cuda)
    assert linear_path(weights, m, OP_DX)[0] == PATH_DENSE
    w = kernels.dequant(weights, dtype)
    n = sum(rows)
    g = torch.Generator(device=cuda).manual_seed(13)
    dy = torch.randn(m, n, generator=g, device=cuda).to(dtype)
    ref, loras = dy.float() @ w.float(), []
    for seg, r in ((0, 16), (2, 40)):
        da, at = _lora(m, r, n, k, dtype, cuda, 14 + seg)
        a = at.T.contiguous()
        loras.append(kernels.make_lora(seg, r, 2.0, a=a, da=da))
        ref += da.float() @ a.float()
    assert_rel(kernels.linear_dx(dy, weights, loras), ref, what="dx")
    idx = (torch.arange(m, device=cuda) * 61 + 7) % n
    hot = torch.zeros(m, n, dtype=dtype, device=cuda)
    hot[torch.arange(m, device=cuda), idx] = 1
    assert torch.equal(kernels.linear_dx(hot, weights), w[idx])
