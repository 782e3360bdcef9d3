"""Response values under torch's transforms (functorch, forward mode, batched gradients) and traces, against the
same formula written with torch's operators; inputs longer than the mesh needs."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
CASES = [("mechanical", "quad"), ("thermal", "quad"), ("mechanical", "tetra"), ("thermal", "hexahedron")]


def _close(a, b):
    # two orders of sums of at most a few hundred products
    assert a.shape == b.shape
    assert float((a - b).detach().abs().max()) <= 1e-13 * max(float(b.detach().abs().max()), 1e-300)


def _response(kind, etype):
    """A response, the same value by torch's operators, and the numbers of nodes and dofs."""
    from folax_amd import loss_functions as lf
    from folax_amd.controls import FourierControl
    from folax_amd.mesh import Mesh
    from folax_amd.responses import FiniteElementResponse
    from tests.cases import make_case
    case = make_case(kind, etype, n=3, seed=12)
    m = Mesh("m", "m.")
    m.nodes_coordinates, m.node_ids = case["coords"], np.arange(len(case["coords"]))
    m.elements_nodes, m.node_sets, m.is_initialized = {etype: case["conn"]}, case["sets"], True
    where = {"quad": "2DQuad", "hexahedron": "3DHexa", "tetra": "3DTetra"}[etype]
    if kind == "thermal":
        loss = getattr(lf, "ThermalLoss" + where)("l", {"dirichlet_bc_dict": {"T": {"left": 1.0}}}, m)
        formula, phi = "(E**2)*T[0]**3", lambda e, t: e ** 2 * t[0] ** 3
    else:
        bc = {d: {"left": 0.0} for d in (["Ux", "Uy"] if etype == "quad" else ["Ux", "Uy", "Uz"])}
        loss = getattr(lf, "MechanicalLoss" + where)(
            "l", {"dirichlet_bc_dict": bc, "material_dict": {"young_modulus": 1.0, "poisson_ratio": 0.3}}, m)
        formula, phi = "(E**2)*(U[0]**2+U[1])", lambda e, u: e ** 2 * (u[0] ** 2 + u[1])
    control = FourierControl("E", {"x_freqs": np.array([1]), "y_freqs": np.array([1]), "z_freqs": np.array([0]), "beta": 2}, m)
    r = FiniteElementResponse("r", formula, loss, control)
    r.Initialize()
    # the geometry is formed by the first evaluation, outside a transform
    r.ComputeValue(np.ones(len(case["coords"])), np.ones(loss.total_number_of_dofs))
    N, wdet, _ = loss.ctx.gauss_point_data(loss.num_gp)
    conn = torch.as_tensor(case["conn"], dtype=torch.int64, device="cuda")
    p = loss.number_dofs_per_node

    def value(d, u):
        return (wdet * phi(d[conn] @ N.T, torch.einsum("ga,eac->ceg", N, u.view(-1, p)[conn]))).sum()

    return r, value, len(case["coords"]), p * len(case["coords"])


def _inputs(n, dofs, batch=4):
    gen = torch.Generator(device="cuda").manual_seed(1)
    return [torch.rand(*s, generator=gen, device="cuda", dtype=torch.float64)
            for s in ((n,), (dofs,), (batch, n), (batch, dofs))]


@pytest.mark.parametrize("kind,etype", CASES)
def test_functorch_transforms(kind, etype):
    r, ref, n, dofs = _response(kind, etype)
    d, u, ds, us = _inputs(n, dofs)
    func = torch.func
    for make, args in ((lambda f: func.grad(f, argnums=(0, 1)), (d, u)), (lambda f: func.hessian(f, argnums=1), (d, u)),
                       (lambda f: func.jacrev(func.grad(f, argnums=0), argnums=1), (d, u)),
                       (lambda f: torch.vmap(f), (ds, us)), (lambda f: torch.vmap(f, in_dims=(None, 0)), (d, us)),
                       (lambda f: torch.vmap(f, in_dims=(1, None)), (ds.T.contiguous(), u)),
                       (lambda f: torch.vmap(func.grad(f, argnums=(0, 1))), (ds, us)),
                       (lambda f: lambda a, b: func.jvp(f, (a, b), (ds[0], us[0])), (d, u))):
        got, want = make(r.ComputeValue)(*args), make(ref)(*args)
        for a, b in zip(got, want) if isinstance(got, tuple) else ((got, want),):
            _close(a, b)


@pytest.mark.parametrize("kind,etype", CASES)
def test_forward_mode_and_batched_gradients(kind, etype):
    import torch.autograd.forward_ad as fw
    r, ref, n, dofs = _response(kind, etype)
    d, u, ds, us = _inputs(n, dofs)
    got = []
    for f in (r.ComputeValue, ref):
        with fw.dual_level():
            both = fw.unpack_dual(f(fw.make_dual(d, ds[0]), fw.make_dual(u, us[0]))).tangent
            one = fw.unpack_dual(f(d, fw.make_dual(u, us[0]))).tangent
        a, b = d.clone().requires_grad_(True), u.clone().requires_grad_(True)
        factors = torch.tensor([1.0, -2.0, 0.5], dtype=torch.float64, device="cuda")
        rows = torch.autograd.grad(f(a, b), (a, b), grad_outputs=factors, is_grads_batched=True)
        functional = torch.autograd.functional
        got.append([both, one, *rows, functional.hessian(lambda x: f(d, x), u, vectorize=True),
                    functional.jacobian(lambda x: f(x, u), d, strategy="forward-mode", vectorize=True)])
    for a, b in zip(*got):
        _close(a, b)


def test_traces():
    from torch.fx.experimental.proxy_tensor import make_fx
    r, ref, n, dofs = _response("mechanical", "quad")
    d, u, ds, us = _inputs(n, dofs)
    for trace in (lambda f: torch.jit.trace(f, (d, u), check_trace=False), lambda f: make_fx(lambda a, b: f(a, b))(d, u)):
        _close(trace(r.ComputeValue)(ds[0], us[0]), ref(ds[0], us[0]))  # a graph of its inputs, not of their values


def test_input_lengths():
    r, ref, n, dofs = _response("mechanical", "quad")
    d, u, _, _ = _inputs(n, dofs)
    a, b = torch.cat([d, d]).requires_grad_(True), torch.cat([u, u]).requires_grad_(True)
    v = r.ComputeValue(a, b)
    _close(v, ref(d, u))
    for g, x in zip(torch.autograd.grad(v, (a, b)), torch.func.grad(ref, argnums=(0, 1))(d, u)):
        _close(g, torch.cat([x, torch.zeros_like(x)]))
    for args in ((d[:-1], u), (d, u[:-2])):
        with pytest.raises(IndexError):
            r.ComputeValue(*args)


def test_shape_derivatives_with_batched_gradients():
    r, _, n, dofs = _response("mechanical", "quad")
    d, u, _, us = _inputs(n, dofs)
    a, b = d.clone().requires_grad_(True), u.clone().requires_grad_(True)
    out = r.ComputeAdjointNodalShapeDerivatives(a, b, us[0])
    gen = torch.Generator(device="cuda").manual_seed(2)
    factors = torch.rand(2, out.numel(), generator=gen, device="cuda", dtype=torch.float64)
    rows = torch.autograd.grad(out, (a, b), grad_outputs=factors, is_grads_batched=True, retain_graph=True)
    for k in range(2):
        for row, want in zip(rows, torch.autograd.grad(out, (a, b), grad_outputs=factors[k], retain_graph=True)):
            _close(row[k], want)
