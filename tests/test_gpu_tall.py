"""The 32-row kernel of the skinny forward path (17-64 tokens, weights tall enough to fill the chip
with its 160-row workgroups): ragged rows (a segment's last workgroup, its last row tile), both
token groups partly full, an odd number of super-steps (the second k-part one short), bias and
LoRA, against fp32 products of the dequantized weight and, with one-hot rows, against the weight
bit for bit.  Each size is asserted to take that kernel (its workgroups need one round of the 256
CUs, the 16-row kernel's two)."""

import pytest
import torch

from tests.gpu_util import PATH_SKINNY32, assert_rel, banner, linear_path, random_weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,k,m", [([18950, 18933], 256, 64), ([40000], 384, 33),
                                      ([18944, 18944], 640, 17), ([37770], 256, 32),
                                      ([18944, 18944], 384, 47)])
def test_tall_forward(cuda, dtype, rows, k, m):
    from solution import kernels

    banner("tall fwd", dtype, rows, k, m)
    weights = [random_weight(n, k, seed=500 + i, dev=cuda) for i, n in enumerate(rows)]
    assert linear_path(weights, m) == (PATH_SKINNY32, 0)
    w = kernels.dequant(weights, dtype)
    n = sum(rows)
    g = torch.Generator(device=cuda).manual_seed(5)
    buf = torch.full((m, k + 8), float("nan"), dtype=dtype, device=cuda)
    x = buf[:, :k]
    x.copy_(torch.randn(m, k, generator=g, device=cuda))
    bias = torch.randn(n, generator=g, device=cuda).to(dtype)
    for r in (16, 20):
        t = torch.randn(m, r, generator=g, device=cuda).to(dtype)
        b = (torch.randn(rows[-1], r, generator=g, device=cuda) * 0.05).to(dtype)
        ref = x.float() @ w.float().T + bias.float()
        ref[:, n - rows[-1]:] += 0.5 * t.float() @ b.float().T
        y = kernels.linear_fwd(x, weights, bias, [kernels.make_lora(len(rows) - 1, r, 0.5, t=t, b=b)])
        assert_rel(y, ref, what=f"y rank {r}")
    for c0 in range(0, k, m):
        idx = (torch.arange(m, device=cuda) + c0) % k
        hot = torch.zeros(m, k, dtype=dtype, device=cuda)
        hot[torch.arange(m, device=cuda), idx] = 1
        assert torch.equal(kernels.linear_fwd(hot, weights), w.T[idx]), c0


def test_tall_forward_with_down_projection_where_the_kernels_cross(cuda):
    """A size at which the 32-row kernel and a split 16-row one are nearly as fast: the adapter's
    own launch for t = x A^T does not move the call to the plan whose partials the workspace
    query, which does not see adapters, left out."""
    from solution import kernels
    from solution.quant_state import NF4_CODE, QuantState

    rows, k, m, r, dtype = 33792, 8192, 17, 32, torch.bfloat16
    banner("tall fwd with a", rows, k, m, r)
    g = torch.Generator(device=cuda).manual_seed(8)
    packed = torch.randint(0, 256, (rows * k // 2,), generator=g, device=cuda, dtype=torch.uint8)
    absmax = torch.rand(rows * k // 64, generator=g, device=cuda) * 0.04 + 0.01
    qs = QuantState(absmax=absmax, shape=torch.Size((rows, k)), dtype=dtype, blocksize=64,
                    code=torch.tensor(NF4_CODE, device=cuda), quant_type="nf4")
    x = torch.randn(m, k, generator=g, device=cuda).to(dtype)
    a = (torch.randn(r, k, generator=g, device=cuda) / k ** 0.5).to(dtype)
    b = (torch.randn(rows, r, generator=g, device=cuda) * 0.05).to(dtype)
    t = torch.empty(m, r, dtype=dtype, device=cuda)
    assert linear_path([(packed, qs)], m) == linear_path([(packed, qs)], m, xa_rank=r) == (PATH_SKINNY32, 0)
    y = kernels.linear_fwd(x, [(packed, qs)], None, [kernels.make_lora(0, r, 0.5, t=t, b=b, a=a)])
    w = kernels.dequant([(packed, qs)], dtype)
    assert_rel(t, (x.float() @ a.float().T), what="t")
    assert_rel(y, x.float() @ w.float().T + 0.5 * t.float() @ b.float().T, what="y")


@pytest.fixture(scope="module")
def gate_up_7b(cuda):
    return [random_weight(18944, 3584, seed=520 + i, dev=cuda, nested=i == 0) for i in range(2)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,r", [(64, 16), (64, 40), (31, 16), (17, 20)])
def test_tall_forward_deep(cuda, gate_up_7b, dtype, m, r):
    """The 7B gate|up pair: 14 super-steps per k-part, a 160-row workgroup ending in each segment,
    fp32 absmax in one of them, and adapters on both whose down-projection the call computes."""
    from solution import kernels

    rows, k = 18944, 3584
    banner("tall fwd deep", dtype, m, r)
    weights = gate_up_7b
    assert linear_path(weights, m, xa_rank=r) == (PATH_SKINNY32, 0)
    w = kernels.dequant(weights, dtype)
    g = torch.Generator(device=cuda).manual_seed(9)
    x = torch.randn(m, k, generator=g, device=cuda).to(dtype)
    ref, loras, ts = x.float() @ w.float().T, [], []
    for i in range(2):
        a = (torch.randn(r, k, generator=g, device=cuda) / k ** 0.5).to(dtype)
        b = (torch.randn(rows, r, generator=g, device=cuda) * 0.05).to(dtype)
        t = torch.empty(m, r, dtype=dtype, device=cuda)
        loras.append(kernels.make_lora(i, r, 0.5, t=t, b=b, a=a))
        ts.append((t, x.float() @ a.float().T))
        ref[:, i * rows:(i + 1) * rows] += 0.5 * ts[-1][1].to(dtype).float() @ b.float().T
    y = kernels.linear_fwd(x, weights, None, loras)
    for t, t_ref in ts:
        assert_rel(t, t_ref, what="t")
    assert_rel(y, ref, what="y")
