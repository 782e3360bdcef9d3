"""The Gauss-point side of responses against plain torch on the same shape functions, and the shape gradient's
two assemblies (corner buffer and atomics) against each other and the oracle, on every element type, rule and
precision; values that the caller differentiates."""
import numpy as np
import pytest

from oracle import fe
from tests.cases import femhot_context, make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
ELEMENTS = [(e, g) for e in ("quad", "hexahedron", "tetra") for g in (1, 2, 3)]


def _t(x, dtype):
    return torch.as_tensor(np.asarray(x), dtype=dtype, device="cuda")


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("etype,rule", ELEMENTS)
@pytest.mark.parametrize("kind", ["thermal", "mechanical"])
def test_values_and_gather(kind, etype, rule, dtype):
    case = make_case(kind, etype, n=3, seed=3, num_gp=rule)
    ctx = femhot_context(case)
    d, u = _t(case["field"], dtype), _t(case["u"], dtype)
    N, _, _ = ctx.gauss_point_data(rule, dtype=dtype)
    conn = torch.as_tensor(case["conn"], dtype=torch.int64, device="cuda")
    gd, gu = ctx.gauss_point_values(d, u, rule)
    P = ctx.dofs_per_node
    tol = 32 * torch.finfo(dtype).eps  # sums of at most 8 products of values of order 1
    assert float((gd - d[conn] @ N.T).abs().max()) <= tol * float(d.abs().max())
    want = torch.stack([u.view(-1, P)[conn][:, :, c] @ N.T for c in range(P)])
    assert float((gu - want).abs().max()) <= tol * float(u.abs().max())
    gen = torch.Generator(device="cuda").manual_seed(5)
    q = torch.randn(gu.shape, generator=gen, device="cuda", dtype=torch.float64).to(dtype)
    out = ctx.gauss_point_gather(q, rule)
    ref = torch.zeros(ctx.n_nodes, P, dtype=torch.float64, device="cuda")
    for c in range(P):
        ref[:, c].index_add_(0, conn.reshape(-1), (q[c].double() @ N.double()).reshape(-1))
    # at most 24 corners of 27 points: sums of about 650 terms
    assert float((out.double() - ref).abs().max()) <= 650 * torch.finfo(dtype).eps * float(q.abs().max())
    again = ctx.gauss_point_gather(q, rule, out=out.clone())
    assert float((again - 2 * out).abs().max()) <= 8 * torch.finfo(dtype).eps * float(out.abs().max())
    ctx.close()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("kind", ["thermal", "mechanical", "neohooke"])
@pytest.mark.parametrize("etype,rule", [("quad", 2), ("hexahedron", 2), ("tetra", 1), ("hexahedron", 3), ("tetra", 3)])
def test_shape_gradient(kind, etype, rule, dtype):
    body = 0.4 if kind == "thermal" else ([0.3, -0.2] if etype == "quad" else [0.3, -0.2, 0.1])
    for elemental in (False, True):
        case = make_case(kind, etype, n=3, seed=4, num_gp=rule, beta=0.5, c=2.0, elemental=elemental, body=body)
        ctx = femhot_context(case)
        from folax_amd import _lib as L
        flags = L.ELEMENT_FIELD if elemental else 0
        d, u, w = (_t(case[k], dtype) for k in ("field", "u", "w"))
        g = ctx.residual_shape_vjp(d, u, w, flags=flags)
        G = L.gauss_points_per_element(ctx.et, rule)
        phi = _t(np.random.default_rng(2).standard_normal((ctx.n_elems, G)), dtype)
        _, _, dn = ctx.gauss_point_data(rule, dtype=dtype)
        extra = ctx.residual_shape_vjp(d, u, w, flags=flags, wphi=phi) - g
        ge = torch.einsum("eg,egaj->eaj", phi.double(), dn.double())
        conn = torch.as_tensor(case["conn"], dtype=torch.int64, device="cuda")
        want = torch.zeros(ctx.n_nodes, 3, dtype=torch.float64, device="cuda")
        want[:, : ge.shape[-1]].index_add_(0, conn.reshape(-1), ge.reshape(-1, ge.shape[-1]))
        scale = max(float(want.abs().max()), float(g.abs().max()))
        assert float((extra.double() - want).abs().max()) <= 2000 * torch.finfo(dtype).eps * scale
        atomic = torch.empty_like(g)
        L.check(ctx._lib.femhot_residual_shape_vjp(ctx._h, L.F64 if dtype == torch.float64 else L.F32, d.data_ptr(),
                                                   u.data_ptr(), w.data_ptr(), atomic.data_ptr(), flags, 0))
        torch.cuda.synchronize()
        assert float((atomic - g).abs().max()) <= 200 * torch.finfo(dtype).eps * float(g.abs().max())
        if kind != "neohooke":  # the oracle differentiates by complex step: exact to rounding
            ref = fe.global_residual_shape_vjp(case["ph"], case["coords"], case["conn"], case["field"], case["u"], case["w"])
            err = np.linalg.norm(g.double().cpu().numpy() - ref) / np.linalg.norm(ref)
            assert err <= (1e-12 if dtype == torch.float64 else 1e-5)
        ctx.close()


def test_response_value_is_differentiable():
    from folax_amd import loss_functions as lf
    from folax_amd.controls import FourierControl
    from folax_amd.mesh import create_2D_square_mesh
    from folax_amd.responses import FiniteElementResponse
    m = create_2D_square_mesh(1.0, 6)
    loss = lf.MechanicalLoss2DQuad("l", {"dirichlet_bc_dict": {"Ux": {"left": 0.0}, "Uy": {"left": 0.0}},
                                         "material_dict": {"young_modulus": 1.0, "poisson_ratio": 0.3}}, m)
    fc = FourierControl("E", {"x_freqs": np.array([1]), "y_freqs": np.array([1]), "z_freqs": np.array([0]), "beta": 2}, m)
    r = FiniteElementResponse("r", "(E**2)*(U[0]**2+U[1])", loss, fc)
    r.Initialize()
    gen = torch.Generator(device="cuda").manual_seed(1)
    d = torch.rand(36, generator=gen, device="cuda", dtype=torch.float64).requires_grad_(True)
    u = torch.rand(72, generator=gen, device="cuda", dtype=torch.float64).requires_grad_(True)
    assert torch.autograd.gradcheck(r.ComputeValue, (d, u))
    assert torch.autograd.gradgradcheck(r.ComputeValue, (d, u))
