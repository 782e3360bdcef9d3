"""The enqueued solve where its workgroups make four or eight passes (a kernel per pass and one for p.q with one
dof per node), bit for bit against the solve in one launch; the test after the last iteration; solves that end
before their first."""
import pytest

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


# quads: 128 nodes a pass on at most 128 workgroups (n = 200: 40,401 nodes, four passes; 270: 73,441, eight), the
# last workgroup partly empty; hexahedra: 64 a pass (n = 30: 29,791, four; 44: 91,125, eight); elastic: 256 workgroups
# (quads 270: four, hexahedra 27: 21,952 nodes, two)
@pytest.mark.parametrize("kind,etype,n", [("thermal", "quad", 200), ("thermal", "quad", 270),
                                          ("thermal", "hexahedron", 30), ("thermal", "hexahedron", 44),
                                          ("thermal", "tetra", 34), ("mechanical", "quad", 270),
                                          ("mechanical", "hexahedron", 27)])
def test_many_passes_give_the_same_bits(kind, etype, n):
    ctx, rp, ci, vals, b = _system(kind, etype, n)
    for cap in (1, 2, 9):
        xs, it, _, _ = ctx.pcg(rp, ci, vals, b, tol=1e-300, maxiter=cap, raise_on_fail=False, context_pattern=True)
        xa = torch.zeros_like(b)
        ia, _, sa = ctx.pcg_async(rp, ci, vals, b, xa, tol=1e-300, iterations=cap, context_pattern=True)
        assert it == cap == int(ia.item()) and int(sa.item()) == 3 and torch.equal(xs, xa)
    ctx.close()


@pytest.mark.parametrize("kind,etype,n", [("thermal", "quad", 30), ("mechanical", "hexahedron", 6),
                                          ("thermal", "quad", 200)])
def test_ends(kind, etype, n):
    ctx, rp, ci, vals, b = _system(kind, etype, n)
    tol = 1e-6 if n < 200 else 0.5
    x = torch.zeros_like(b)
    it, rel, st = ctx.pcg_async(rp, ci, vals, b, x, tol=tol, iterations=2000, context_pattern=True)
    k = int(it.item())
    assert int(st.item()) == 1 and 0 < k < 2000 and float(rel.item()) <= tol
    # converged by the last iteration, before it, not at all (which takes at least one iteration)
    for iterations, status in ((k, 1), (k + 1, 1), (k - 1, 3))[: 2 if k == 1 else 3]:
        y = torch.zeros_like(b)
        it, rel, st = ctx.pcg_async(rp, ci, vals, b, y, tol=tol, iterations=iterations, context_pattern=True)
        assert int(st.item()) == status and int(it.item()) == min(k, iterations)
        assert torch.equal(y, x) if status == 1 else float(rel.item()) > tol
    y = x.clone()
    it, rel, st = ctx.pcg_async(rp, ci, vals, b, y, tol=tol, iterations=5, context_pattern=True)
    assert int(st.item()) == 1 and int(it.item()) == 0 and torch.equal(y, x)  # converged as it begins
    y.fill_(0.5)
    it, rel, st = ctx.pcg_async(rp, ci, vals, torch.zeros_like(b), y, tol=tol, iterations=5, context_pattern=True)
    assert int(st.item()) == 1 and int(it.item()) == 0 and bool((y == 0.5).all())
    bad = b.clone()
    bad[-1] = float("nan")
    y.fill_(0.5)
    it, rel, st = ctx.pcg_async(rp, ci, vals, bad, y, tol=tol, iterations=5, context_pattern=True)
    assert int(st.item()) == 2 and int(it.item()) == 0 and bool((y == 0.5).all())
    ctx.close()
