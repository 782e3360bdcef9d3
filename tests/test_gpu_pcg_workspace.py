"""The solver workspace of a context: whichever FP64 solve comes first, host-checked or enqueued, sizes it for
the other, so that a capture allocates nothing and a captured solve keeps the memory it was captured with."""
import pytest
import torch

from tests.cases import femhot_context, make_case

pytestmark = pytest.mark.gpu


def _system(kind, etype, n):
    case = make_case(kind, etype, n=n, seed=9)
    ctx = femhot_context(case)
    f = torch.as_tensor(case["field"], dtype=torch.float64, device="cuda")
    u = torch.as_tensor(case["u"], dtype=torch.float64, device="cuda")
    vals, R = ctx.tangent_csr(f, u)
    rp, ci = ctx.pattern()
    return ctx, rp, ci, vals, (-R).contiguous()


# the vectors are most of the workspace from about 5,000 dofs, the partial sums below about 3,000
@pytest.mark.parametrize("kind,etype,n", [("mechanical", "quad", 8), ("mechanical", "quad", 30),
                                          ("mechanical", "quad", 70), ("mechanical", "hexahedron", 13),
                                          ("thermal", "quad", 90), ("thermal", "tetra", 9)])
@pytest.mark.parametrize("first", ["pcg", "pcg_async"])
@pytest.mark.parametrize("other_pattern", [False, True])
def test_either_solve_sizes_the_workspace(kind, etype, n, first, other_pattern):
    ctx, rp, ci, vals, b = _system(kind, etype, n)
    iters = 20
    out = (torch.empty(1, dtype=torch.int32, device="cuda"), torch.empty(1, dtype=torch.float64, device="cuda"),
           torch.empty(1, dtype=torch.int32, device="cuda"))
    xg = torch.empty_like(b)

    def solve():
        xg.zero_()
        ctx.pcg_async(rp, ci, vals, b, xg, tol=1e-300, iterations=iters, context_pattern=True, out=out)

    def pcg():
        return ctx.pcg(rp, ci, vals, b, tol=1e-300, maxiter=iters, raise_on_fail=False,
                       context_pattern=not other_pattern)[0]

    pcg() if first == "pcg" else solve()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        solve()
    torch.cuda.synchronize()
    pcg()  # the other way round: the graph's memory stays
    solve()
    torch.cuda.synchronize()
    want = xg.clone()
    for rep in range(3):
        xg.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(xg, want) and int(out[0].item()) == iters, rep
        _ = float((b * 2).sum())  # eager work between replays
    ctx.close()
