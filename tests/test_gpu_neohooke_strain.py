"""Neo-Hookean elements over volume changes on both sides of where the series of log J and J^(-2/D) end
(|J - 1| = 0.5, |2/D log J| = 0.5), against the oracle."""
import numpy as np
import pytest

from oracle import fe
from tests.cases import PHYS_CODE, make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("etype", ["quad", "tetra", "hexahedron"])
@pytest.mark.parametrize("volume", [0.35, 0.499, 0.501, 0.8, 1.0, 1.499, 1.501, 3.0])
def test_volume_change(etype, volume, dtype):
    from folax_amd import _lib as L
    from folax_amd.context import FemhotContext
    case = make_case("neohooke", etype, n=3, seed=23)
    ph, xyz = case["ph"], case["coords"]
    d = 2 if etype == "quad" else 3
    rng = np.random.default_rng(5)
    u = (volume ** (1.0 / d) - 1.0) * xyz[:, :d] + 1e-3 * rng.uniform(-1, 1, (len(xyz), d))
    u = u.ravel()
    ctx = FemhotContext(etype, PHYS_CODE["neohooke"], xyz, case["conn"], num_gp=ph.num_gp, young_modulus=ph.E,
                        poisson_ratio=ph.nu)
    f = torch.as_tensor(case["field"], dtype=dtype, device="cuda")
    ut = torch.as_tensor(u, dtype=dtype, device="cuda")
    none = np.zeros(0, np.int64)
    Kr, Rr = fe.assemble(ph, xyz, case["conn"], case["field"], u, none)
    # rounding of an element's inputs alone moves its vector by eps |K_e| |u_e| (an element's, not the
    # assembled matrix's: the terms of neighbouring elements cancel, their roundings do not)
    eps = 2.3e-16 if dtype == torch.float64 else 1.2e-7
    dofs = fe.element_dofs(case["conn"], d)
    _, re, Ke = ph.element(xyz[case["conn"]], np.asarray(case["field"])[case["conn"]], u[dofs], want_K=True)
    bar = np.zeros(u.size)
    np.add.at(bar, dofs, 64 * eps * (np.einsum("eij,ej->ei", np.abs(Ke), np.abs(u[dofs])) + np.abs(re)))
    for flags in (0, L.SCATTER_CHUNK):
        R, en = ctx.residual(f, ut, flags=flags)
        assert np.all(np.abs(R.double().cpu().numpy().ravel() - Rr) <= bar + 1e-300)
    K, _ = ctx.tangent_csr(f, ut, flags=L.SCATTER_ROWS)
    tol = 1e-11 if dtype == torch.float64 else 1e-4
    assert np.linalg.norm(K.double().cpu().numpy() - Kr.data) <= tol * np.linalg.norm(Kr.data)
    ctx.close()
