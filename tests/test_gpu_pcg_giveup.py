"""One-launch solves whose waits between workgroups run out (a limit of a few looks, set from the host: every
workgroup leaves normally): the call falls back to launched kernels from its own initial guess, and a Newton
solve reaches the same solution.  Two one-launch solves at once."""
import threading

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


def _direct(rp, ci, vals, b):
    A = sp.csr_array((vals.cpu().numpy(), ci.cpu().numpy(), rp.cpu().numpy()), shape=(b.numel(), b.numel()))
    return spla.spsolve(A.tocsc(), b.cpu().numpy())


def _limit(ctx, looks):
    from folax_amd import _lib as L
    L.check(ctx._lib.femhot_pcg_wait_limit(ctx._h, looks))


# systems of several workgroups, one, two and three dofs per node
@pytest.mark.parametrize("kind,etype,n", [("thermal", "quad", 40), ("mechanical", "quad", 45),
                                          ("mechanical", "hexahedron", 11), ("thermal", "tetra", 9)])
def test_gives_up_and_falls_back(kind, etype, n):
    ctx, rp, ci, vals, b = _system(kind, etype, n)
    want = _direct(rp, ci, vals, b)
    rng = np.random.default_rng(n)
    x0 = torch.as_tensor(want * (1.0 + 0.1 * rng.standard_normal(want.size)), device="cuda")
    x0 = torch.where(b == 0, torch.zeros_like(x0), x0)
    for mode in ("f64", "mixed"):
        for start in (None, x0):
            _limit(ctx, 0)
            x, it, rel, ok = ctx.pcg(rp, ci, vals, b, x0=start, tol=1e-12, maxiter=5000, mode=mode,
                                     context_pattern=True)
            assert ok and rel <= 1e-12
            assert np.linalg.norm(x.cpu().numpy() - want) <= 1e-6 * np.linalg.norm(want)  # condition below 1e5
    for cap in (1, 7, 20):  # one dof per node: the launched kernels are those of any pattern, so are the bits
        args = dict(tol=1e-300, maxiter=cap, raise_on_fail=False)
        _limit(ctx, 0)
        fall, it, _, _ = ctx.pcg(rp, ci, vals, b, x0=x0, context_pattern=True, **args)
        assert it == cap
        if kind == "thermal":
            assert torch.equal(fall, ctx.pcg(rp, ci, vals, b, x0=x0, **args)[0])
        _limit(ctx, 1 << 21)
        one = ctx.pcg(rp, ci, vals, b, x0=x0, context_pattern=True, **args)[0]
        for looks in (1, 2, 5, 20, 60):  # somewhere between the first exchange and the last, or not at all
            _limit(ctx, looks)
            got = ctx.pcg(rp, ci, vals, b, x0=x0, context_pattern=True, **args)[0]
            assert torch.equal(got, fall) or torch.equal(got, one), looks
    ctx.close()


def test_newton_falls_back():
    case = make_case("neohooke", "hexahedron", n=8, seed=6)
    f = torch.as_tensor(case["field"], dtype=torch.float64, device="cuda")
    got = []
    for looks in (1 << 21, 0):
        ctx = femhot_context(case)
        _limit(ctx, looks)
        u, hist, steps = ctx.newton(f, torch.zeros(ctx.n_dofs, dtype=torch.float64, device="cuda"), load_steps=2,
                                    abs_tol=1e-10, rel_tol=1e-10, lin_tol=1e-12)
        got.append((u, list(steps)))
        ctx.close()
    assert got[0][1] == got[1][1]
    assert float((got[0][0] - got[1][0]).norm()) <= 1e-8 * float(got[0][0].norm())


def test_two_solves_at_once():
    systems = [_system("mechanical", "hexahedron", 11), _system("thermal", "quad", 100)]
    wants = [_direct(*s[1:]) for s in systems]
    got = [None, None]

    def solve(k):
        ctx, rp, ci, vals, b = systems[k]
        _limit(ctx, 1 << 16)
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            got[k] = [ctx.pcg(rp, ci, vals, b, tol=1e-12, maxiter=5000, context_pattern=True)[0] for _ in range(5)]
            stream.synchronize()

    torch.cuda.synchronize()
    threads = [threading.Thread(target=solve, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for xs, want in zip(got, wants):
        assert xs is not None
        for x in xs:
            assert np.linalg.norm(x.cpu().numpy() - want) <= 1e-6 * np.linalg.norm(want)
    for s in systems:
        s[0].close()
