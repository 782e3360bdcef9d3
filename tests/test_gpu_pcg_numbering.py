"""Solves on meshes whose nodes are numbered at random, so that a workgroup's columns spread over the whole mesh: within
the range of ids that the tile kernels take (LDS holding as many nodes as their rows can name), just beyond it, and
beyond their LDS, against the solve on any pattern; the enqueued form too."""
import numpy as np
import pytest

from tests.cases import PHYS_CODE, make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# 6,561 nodes; 65,025 (of at most 65,536 ids); 66,049; two and three dofs per node (30,976 and 4,913 nodes)
@pytest.mark.parametrize("kind,etype,n", [("thermal", "quad", 80), ("thermal", "quad", 254), ("thermal", "quad", 256),
                                          ("mechanical", "quad", 175), ("mechanical", "hexahedron", 16)])
def test_random_numbering(kind, etype, n):
    from folax_amd.context import FemhotContext
    case = make_case(kind, etype, n=n, seed=4)
    rng = np.random.default_rng(n)
    nodes = len(case["coords"])
    new = rng.permutation(nodes)  # old id -> new id
    coords, field = np.empty_like(case["coords"]), np.empty_like(case["field"])
    coords[new], field[new] = case["coords"], case["field"]
    p = case["ph"].ndpn
    ids = np.asarray(case["didx"])
    ctx = FemhotContext(case["etype"], PHYS_CODE[kind], coords, new[case["conn"]].astype(np.int32),
                        young_modulus=case["ph"].E, poisson_ratio=case["ph"].nu, dirichlet_idx=new[ids // p] * p + ids % p,
                        dirichlet_val=case["dval"])
    f = torch.as_tensor(field, dtype=torch.float64, device="cuda")
    u = torch.as_tensor(rng.uniform(0.0, 1.0, p * nodes), dtype=torch.float64, device="cuda")
    vals, R = ctx.tangent_csr(f, u)
    rp, ci = ctx.pattern()
    b = -R
    for cap in (1, 8):
        args = dict(tol=1e-300, maxiter=cap, raise_on_fail=False)
        x, it, _, _ = ctx.pcg(rp, ci, vals, b, context_pattern=True, **args)
        y, _, _, _ = ctx.pcg(rp, ci, vals, b, **args)
        # eight iterations of sums in another order, the FP64 vectors some 1e2 apart in size
        assert it == cap and float((x - y).norm()) <= 1e-11 * float(y.norm())
        z = torch.zeros_like(b)
        ctx.pcg_async(rp, ci, vals, b, z, tol=1e-300, iterations=cap, context_pattern=True)
        assert float((z - y).norm()) <= 1e-11 * float(y.norm())
    ctx.close()
