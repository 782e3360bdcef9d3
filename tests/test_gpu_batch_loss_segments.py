"""Gradients of a batch loss's minimum and maximum where a sample's energy is the sum of many segments' energies,
against the composition of the loss's parts: the sample that attains the extreme takes the whole gradient."""
import numpy as np
import pytest

from tests.cases import make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
NAMES = {"quad": "2DQuad", "hexahedron": "3DHexa", "tetra": "3DTetra"}


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("etype,segments", [("quad", 3), ("tetra", 17), ("hexahedron", 64)])
def test_extremes_of_many_segments(etype, segments, dtype):
    from folax_amd import loss_functions as lf
    from folax_amd.loss_functions import _BatchEnergy, _FullDofs
    from folax_amd.mesh import Mesh
    case = make_case("mechanical", etype, n=5, seed=32)
    m = Mesh("m", "m.")
    m.nodes_coordinates, m.node_ids = case["coords"], np.arange(len(case["coords"]))
    m.elements_nodes, m.node_sets, m.is_initialized = {etype: case["conn"]}, case["sets"], True
    rng = np.random.default_rng(11)
    cuts = np.sort(rng.choice(np.arange(1, len(case["conn"])), segments - 1, replace=False)) if segments < 64 else \
        np.arange(1, segments)
    offsets = np.concatenate([[0], cuts, [len(case["conn"])]]).astype(np.int64)
    dofs = ["Ux", "Uy"] if etype == "quad" else ["Ux", "Uy", "Uz"]
    loss = getattr(lf, "MechanicalLoss" + NAMES[etype])(
        "l", {"dirichlet_bc_dict": {d: {"left": 0.0, "right": 0.01 * (k + 1)} for k, d in enumerate(dofs)},
              "material_dict": {"young_modulus": 1.3, "poisson_ratio": 0.3}, "segment_offsets": offsets}, m)
    loss.Initialize()
    batch = 9
    for seed in range(4):
        rng = np.random.default_rng(seed)
        f0, u0 = (torch.as_tensor(np.stack([case[k] * rng.uniform(0.8, 1.2) for _ in range(batch)]), dtype=dtype, device="cuda")
                  for k in ("field", "u"))
        for weights in ((0.0, 1.0, 0.0), (0.0, 0.0, -2.0), (0.5, 1.5, -1.0)):
            got = []
            for one_call in (True, False):
                u = u0.clone().requires_grad_(True)
                if one_call:
                    mean, (low, high, _) = loss.ComputeBatchLoss(f0, u)
                else:
                    e = _BatchEnergy.apply(loss, f0, _FullDofs.apply(loss, f0, u))
                    mean, low, high = e.mean(), e.min(), e.max()
                total = sum(w * s for w, s in zip(weights, (mean, low, high)) if w)
                got.append(torch.autograd.grad(total, u)[0])
            # the same kernels on the same values, factors in another order: 8 roundings
            tol = 8 * torch.finfo(dtype).eps * float(got[1].abs().max())
            assert float((got[0] - got[1]).abs().max()) <= tol, (seed, weights)


def test_a_nan_sample_takes_the_extremes():
    from folax_amd import loss_functions as lf
    from folax_amd.mesh import create_2D_square_mesh
    m = create_2D_square_mesh(1.0, 6)
    loss = lf.MechanicalLoss2DQuad("l", {"dirichlet_bc_dict": {"Ux": {"left": 0.0}, "Uy": {"left": 0.0}},
                                         "material_dict": {"young_modulus": 1.0, "poisson_ratio": 0.3}}, m)
    loss.Initialize()
    u = torch.zeros(3, 72, dtype=torch.float64, device="cuda")
    u[1] = float("nan")
    u.requires_grad_(True)
    _, (low, high, _) = loss.ComputeBatchLoss(torch.ones(3, 36, dtype=torch.float64, device="cuda"), u)
    assert low.isnan() and high.isnan()
    (g,) = torch.autograd.grad(low + high, u)
    assert g[1].isnan().any() and not g[0].any() and not g[2].any()  # (a NaN counts as any)
