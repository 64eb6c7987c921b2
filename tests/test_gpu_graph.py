"""HIP graph capture of the projection stack: every replay must reproduce the eager launches
bit for bit (deterministic kernels, no memset nodes), with eager work between replays."""

import pytest
import torch

from tests.gpu_util import banner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 40, 300])
def test_stack_graph_replays_match_eager(cuda, m):
    from solution import kernels
    from solution.stack import ProjectionStack, Qwen2Shape

    banner("graph replay", m)
    shape = Qwen2Shape(hidden=256, inter=640, kv=64)
    st = ProjectionStack.synthetic(shape, 2, 300, torch.float16, cuda, seed_base=21)
    st.set_tokens([0, m])
    outs = lambda: [t[:m].clone() for t in (st.y_qkv, st.y_o, st.y_gu, st.y_d, st.dx_d,  # noqa
                                             st.dx_gu, st.dx_o, st.dx_qkv)] + \
        [st.per_layer[0][k].clone() for k in ("gb_q", "gb_v", "ga_q", "ga_v")]
    st.step()
    torch.cuda.synchronize()
    ref = outs()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        st.step()
    other = st.per_layer[1]
    for rep in range(3):
        for t in (st.y_qkv, st.y_d, st.dx_qkv):
            t.zero_()
        # eager work between replays, on the same buffers' neighbours
        kernels.linear_fwd(st.x2[:m], [st.layers[1]["o"]])
        g.replay()
        torch.cuda.synchronize()
        got = outs()
        for i, (a, b) in enumerate(zip(got, ref)):
            assert torch.equal(a, b), f"replay {rep}, output {i}"
    assert other is st.per_layer[1]


def test_dense_calls_replay_in_a_graph(cuda):
    """The dense route captured (its workspaces from the graph's pool, unsplit and with a split
    reduction): every replay gives the eager result, with eager calls of the same route between."""
    from solution import kernels
    from tests.gpu_util import OP_DX, PATH_DENSE, linear_path, random_weight

    banner("graph replay dense")
    g = torch.Generator(device=cuda).manual_seed(31)
    calls = []
    for rows, k, m, dx in (([520, 776], 3072, 1300, False), ([520, 776], 3072, 3001, False),
                           ([1536, 256, 256], 1536, 1025, True), ([3008, 64], 1536, 3001, True)):
        w = [random_weight(n, k, seed=350 + i, dev=cuda) for i, n in enumerate(rows)]
        assert linear_path(w, m, OP_DX if dx else 0)[0] == PATH_DENSE
        x = torch.randn(m, sum(rows) if dx else k, generator=g, device=cuda).half()
        calls.append((kernels.linear_dx if dx else kernels.linear_fwd, x, w))
    ref = [f(x, w) for f, x, w in calls]
    out = [torch.empty_like(r) for r in ref]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for (f, x, w), o in zip(calls, out):
            f(x, w, out=o)
    for rep in range(3):
        for o in out:
            o.fill_(float("nan"))
        eager = [f(x, w) for f, x, w in calls]
        graph.replay()
        torch.cuda.synchronize()
        for i, (a, b, c) in enumerate(zip(out, ref, eager)):
            assert torch.equal(a, b) and torch.equal(c, b), f"replay {rep}, call {i}"
