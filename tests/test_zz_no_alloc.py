"""nf4_linear_dx_noalloc - the input-gradient GEMM that allocates nothing (split-K partials in a
static device array) - against nf4_linear_dx through the C ABI, on two calls in a row, the
second with a smaller input: bit for bit where nf4_linear_dx's own plan fits the array (the
same tiling and split order), and within the path's tolerance (max rel 1e-2, mean rel 1e-3)
where the array forces a smaller split."""

import pytest
import torch

from tests.gpu_util import (OP_DX, OP_DX_NOALLOC, PATH_DENSE, assert_rel, banner, linear_path,
                            random_weight)

pytestmark = pytest.mark.gpu

CAP = 64 << 20  # NF4_STATIC_SCRATCH_BYTES


def _noalloc(dy, weights, out, accumulate=False, loras=()):
    from solution import _lib, kernels

    arr = kernels._descs(weights)
    larr, nl = kernels._lora_array(list(loras))
    st = _lib.load().nf4_linear_dx_noalloc(dy.data_ptr(), dy.shape[0], dy.stride(0), arr,
                                           len(weights), larr, nl, out.data_ptr(), out.stride(0),
                                           int(accumulate), _lib.DTYPE_CODE[dy.dtype],
                                           _lib.stream_of(dy))
    _lib.check(st, "nf4_linear_dx_noalloc")
    return out


def _need(m, weights):
    from solution import _lib, kernels

    return _lib.load().nf4_linear_dx_workspace(m, kernels._descs(weights), len(weights), 0)


def test_noalloc_dx_matches_linear_dx(cuda):
    from solution import kernels

    gate = random_weight(8960, 1536, seed=104, dev=cuda)
    up = random_weight(8960, 1536, seed=105, dev=cuda)
    q = random_weight(1536, 1536, seed=100, dev=cuda)
    g = torch.Generator().manual_seed(9)
    # 1: the benchmark's gate|up input gradient (256x256 tiles split 5: 60 MiB of partials)
    banner("noalloc dx gate|up M=2048")
    dy = (torch.randn(2048, 17920, generator=g) * 1e-3).half().to(cuda)
    need = _need(2048, [gate, up])
    assert 0 < need <= CAP
    ref = kernels.linear_dx(dy, [gate, up])
    out = torch.full_like(ref, float("nan"))
    _noalloc(dy, [gate, up], out)
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
    # 2: a smaller call right after, accumulating, with a LoRA slab; the array still holds the
    # first call's partials
    banner("noalloc dx q + LoRA M=300 accumulate")
    r, s = 16, 2.0
    dy2 = (torch.randn(300, 1536, generator=g) * 1e-3).half().to(cuda)
    a = (torch.randn(r, 1536, generator=g) * 0.02).half().to(cuda)
    da = (torch.randn(300, r, generator=g) * 1e-3).half().to(cuda)
    lora = [kernels.make_lora(0, r, s, a=a, da=da)]
    base = (torch.randn(300, 1536, generator=g) * 1e-2).half().to(cuda)
    ref2 = kernels.linear_dx(dy2, [q], lora, out=base.clone(), accumulate=True)
    out2 = _noalloc(dy2, [q], base.clone(), accumulate=True, loras=lora)
    torch.cuda.synchronize()
    assert torch.equal(out2, ref2)
    # 3: a plan whose partials would not fit: a smaller split, within tolerance
    banner("noalloc dx gate|up M=8192 (plan restricted to the array)")
    dy3 = (torch.randn(8192, 17920, generator=g) * 1e-3).half().to(cuda)
    assert _need(8192, [gate, up]) > CAP
    ref3 = kernels.linear_dx(dy3, [gate, up])
    out3 = _noalloc(dy3, [gate, up], torch.empty_like(ref3))
    torch.cuda.synchronize()
    assert_rel(out3, ref3.float().cpu(), what="restricted plan")


QKV_15B = [(1536, 1536), (256, 1536), (256, 1536)]
QKV_7B = [(3584, 3584), (512, 3584), (512, 3584)]


def _problem(shapes, m, seed, dtype, dev):
    weights = [random_weight(n, k, seed=seed + i, dev=dev) for i, (n, k) in enumerate(shapes)]
    g = torch.Generator(device=dev).manual_seed(seed)
    dy = (torch.randn(m, sum(n for n, _ in shapes), generator=g, device=dev) * 1e-3).to(dtype)
    return weights, dy


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shapes,m", [(QKV_7B, 2500), ([(3584, 3584)], 3000)])
def test_noalloc_on_the_dense_route_matches_linear_dx(cuda, dtype, shapes, m):
    """The weight dequantized into the array (where the fused plan is split, and it fits): bit for
    bit nf4_linear_dx's."""
    from solution import kernels

    banner("noalloc dense", dtype, shapes, m)
    weights, dy = _problem(shapes, m, 900, dtype, cuda)
    path = linear_path(weights, m, OP_DX_NOALLOC)
    assert path[0] == PATH_DENSE and path == linear_path(weights, m, OP_DX)
    ref = kernels.linear_dx(dy, weights)
    out = _noalloc(dy, weights, torch.full_like(ref, float("nan")))
    assert torch.equal(out, ref)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shapes,m", [(QKV_15B, 1025), (QKV_7B, 4096), ([(1536, 8960)], 4096)])
def test_noalloc_without_scratch_is_the_fused_product(cuda, dtype, shapes, m):
    """Sizes at which nf4_linear_dx dequantizes into its workspace but the fused plan needs none:
    bit for bit nf4_linear_dx's result without a workspace."""
    from solution import _lib, kernels

    banner("noalloc unsplit", dtype, shapes, m)
    weights, dy = _problem(shapes, m, 910, dtype, cuda)
    assert linear_path(weights, m, OP_DX)[0] == PATH_DENSE
    ref = torch.empty(m, shapes[0][1], dtype=dtype, device=cuda)
    _lib.check(_lib.load().nf4_linear_dx(
        dy.data_ptr(), m, dy.stride(0), kernels._descs(weights), len(weights), None, 0,
        ref.data_ptr(), ref.stride(0), 0, _lib.DTYPE_CODE[dtype], None, 0, _lib.stream_of(dy)),
        "nf4_linear_dx")
    out = _noalloc(dy, weights, torch.full_like(ref, float("nan")))
    assert torch.equal(out, ref)


def test_noalloc_calls_without_scratch_overlap(cuda):
    """Two streams, two problems of a size that needs no scratch, several calls each in flight."""
    m = 1025
    problems = [_problem(QKV_15B, m, 920 + 10 * i, torch.float16, cuda) for i in range(2)]
    assert linear_path(problems[0][0], m, OP_DX_NOALLOC)[1] == 0
    banner("noalloc overlapping", QKV_15B, m)
    outs = [[torch.full((m, 1536), float("nan"), dtype=torch.float16, device=cuda)
             for _ in range(8)] for _ in problems]
    refs = [_noalloc(dy, w, torch.empty_like(outs[0][0])) for w, dy in problems]
    streams = [torch.cuda.Stream() for _ in problems]
    torch.cuda.synchronize()
    for i in range(8):
        for (w, dy), out, st in zip(problems, outs, streams):
            with torch.cuda.stream(st):
                _noalloc(dy, w, out[i])
    torch.cuda.synchronize()
    for out, ref in zip(outs, refs):
        for o in out:
            assert torch.equal(o, ref)
