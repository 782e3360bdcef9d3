"""femhot_pcg on systems that one launch holds (the context's pattern, at most 32 neighbours per node): the
cuts into workgroups where the solve can go wrong -- one workgroup, its last pass empty or full, one node
more than it holds, many workgroups, each lane count and number of dofs per node -- against a direct solve,
bit for bit against the launched form of the same solve, and with a start vector, a zero right-hand side, a
spent budget and a non-finite right-hand side."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from tests.cases import femhot_context, make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _system(kind, etype, n, seed=5):
    case = make_case(kind, etype, n=n, seed=seed)
    ctx = femhot_context(case)
    f = torch.as_tensor(case["field"], dtype=torch.float64, device="cuda")
    u = torch.as_tensor(case["u"], dtype=torch.float64, device="cuda")
    vals, R = ctx.tangent_csr(f, u)
    rp, ci = ctx.pattern()
    return ctx, rp, ci, vals, (-R).contiguous()


# quads: 4 lanes per node, 128 nodes a pass (n = 10: 121 nodes, one pass; 21: 484 of 512, four; 22: 529, the
# first with an exchange); hexahedra: 8 lanes, 64 nodes a pass (n = 3: 64, one full pass; 4: 125 of 128)
@pytest.mark.parametrize("kind,etype,n", [
    ("thermal", "quad", 10), ("thermal", "quad", 21), ("thermal", "quad", 22), ("thermal", "quad", 70),
    ("mechanical", "quad", 10), ("mechanical", "quad", 22), ("mechanical", "quad", 45), ("thermal", "hexahedron", 5),
    ("thermal", "hexahedron", 13), ("mechanical", "hexahedron", 3), ("mechanical", "hexahedron", 4),
    ("mechanical", "hexahedron", 11), ("thermal", "tetra", 9), ("mechanical", "tetra", 4), ("mechanical", "tetra", 10)])
def test_one_launch_solve(kind, etype, n):
    ctx, rp, ci, vals, b = _system(kind, etype, n)
    A = sp.csr_array((vals.cpu().numpy(), ci.cpu().numpy(), rp.cpu().numpy()), shape=(b.numel(), b.numel()))
    want = spla.spsolve(A.tocsc(), b.cpu().numpy())
    rng = np.random.default_rng(n)
    x0 = torch.as_tensor(want * (1.0 + 0.1 * rng.standard_normal(want.size)) * (b.cpu().numpy() != 0), device="cuda")
    for mode in ("f64", "mixed"):
        for start in (None, x0):
            x, it, rel, ok = ctx.pcg(rp, ci, vals, b, x0=start, tol=1e-12, maxiter=5000, mode=mode, context_pattern=True)
            assert ok and rel <= 1e-12
            # ||A x - b|| <= tol ||b|| up to the rounding of the residual itself
            r = np.linalg.norm(A @ x.cpu().numpy() - b.cpu().numpy()) / np.linalg.norm(b.cpu().numpy())
            assert r <= 1e-11, (mode, r)
            # the error is at most the residual's share times the condition number, here below 1e5
            assert np.linalg.norm(x.cpu().numpy() - want) <= 1e-6 * np.linalg.norm(want)
    # the launched form, stopped after the same number of iterations: the same bits
    for cap in (1, 7, 20):
        xs, it, _, _ = ctx.pcg(rp, ci, vals, b, tol=1e-300, maxiter=cap, raise_on_fail=False, context_pattern=True)
        xa = torch.zeros_like(b)
        ia, _, sa = ctx.pcg_async(rp, ci, vals, b, xa, tol=1e-300, iterations=cap, context_pattern=True)
        assert it == cap == int(ia.item()) and int(sa.item()) == 3 and torch.equal(xs, xa)
    ctx.close()


def test_one_launch_solve_edges():
    for kind, etype, n in (("thermal", "quad", 8), ("mechanical", "hexahedron", 8)):
        ctx, rp, ci, vals, b = _system(kind, etype, n)
        x0 = torch.full_like(b, 0.25)
        zero = torch.zeros_like(b)
        x, it, rel, ok = ctx.pcg(rp, ci, vals, zero, x0=x0, context_pattern=True)
        assert ok and it == 0 and rel == 0.0 and torch.equal(x, x0)  # b = 0: nothing to do, x as it was
        x, it, rel, ok = ctx.pcg(rp, ci, vals, b, tol=1e-14, maxiter=3, raise_on_fail=False, context_pattern=True)
        assert not ok and it == 3 and rel > 1e-14
        bad = b.clone()
        bad[1] = float("nan")
        with pytest.raises(Exception, match="non-finite"):
            ctx.pcg(rp, ci, vals, bad, context_pattern=True)
        bad.view(torch.int64)[1] = -1  # the NaN that marks an empty slot
        with pytest.raises(Exception, match="non-finite"):
            ctx.pcg(rp, ci, vals, bad, context_pattern=True)
        ctx.close()
