"""Gradients of a batch loss taken with create_graph: they can be differentiated again, as those of the loss
composed of its parts, and their second derivatives (zero: a kernel's result is a constant) are the same."""
import pytest

from tests.cases import make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
NAMES = {"quad": "2DQuad", "hexahedron": "3DHexa", "tetra": "3DTetra"}


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("which", [0, 1, 2])  # the mean, the minimum, the maximum
@pytest.mark.parametrize("kind,etype", [("thermal", "quad"), ("mechanical", "tetra"), ("neohooke", "hexahedron")])
def test_differentiated_again(kind, etype, which, dtype):
    from folax_amd import loss_functions as lf
    from folax_amd.loss_functions import _BatchEnergy, _FullDofs
    from folax_amd.mesh import Mesh
    case = make_case(kind, etype, n=3, seed=6)
    m = Mesh("m", "m.")
    m.nodes_coordinates, m.node_ids = case["coords"], range(len(case["coords"]))
    m.elements_nodes, m.node_sets, m.is_initialized = {etype: case["conn"]}, case["sets"], True
    dofs = ["T"] if kind == "thermal" else (["Ux", "Uy"] if etype == "quad" else ["Ux", "Uy", "Uz"])
    cls = {"thermal": "ThermalLoss", "mechanical": "MechanicalLoss", "neohooke": "NeoHookeMechanicalLoss"}[kind]
    loss = getattr(lf, cls + NAMES[etype])("l", {"dirichlet_bc_dict": {d: {"left": 0.0, "right": 0.01} for d in dofs},
                                                "material_dict": {"young_modulus": 1.3, "poisson_ratio": 0.3}}, m)
    loss.Initialize()
    f0, u0 = (torch.as_tensor(case[k], dtype=dtype, device="cuda") * torch.tensor([[1.0], [0.9], [1.1]], dtype=dtype,
                                                                                  device="cuda") for k in ("field", "u"))
    first, second = [], []
    for one_call in (True, False):
        f, u = f0.clone().requires_grad_(True), u0.clone().requires_grad_(True)
        if one_call:
            mean, (low, high, _) = loss.ComputeBatchLoss(f, u)
        else:
            e = _BatchEnergy.apply(loss, f, _FullDofs.apply(loss, f, u)) ** 1.0
            mean, low, high = e.mean(), e.min(), e.max()
        g = torch.autograd.grad((mean, low, high)[which], (f, u), create_graph=True)
        assert all(x.requires_grad for x in g)
        first.append([x.detach() for x in g])
        second.append(torch.autograd.grad(sum((x * x).sum() for x in g), (f, u)))
    tol = 8 * torch.finfo(dtype).eps  # the same kernels, factors in another order: 8 roundings
    for a, b in zip(*first):
        assert float((a - b).abs().max()) <= tol * float(b.abs().max())
    for pair in second:
        assert all(float(x.abs().max()) == 0.0 for x in pair)
