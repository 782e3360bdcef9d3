"""The row-owner tangent and the residual it forms beside, where they can go wrong: nodes with more incident
elements than a batch and more neighbours than a window of columns (hexahedra in sectors around an axis),
partial batches on the boundary, a collapsed element, body forces, per-element fields, accumulation and every
physics, against the oracle and against the separate residual call."""
import numpy as np
import pytest

from oracle import fe
from tests.cases import PHYS_CODE, make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def sectors(n=12, layers=2, collapsed=False):
    """n quadrilaterals around an axis, each (axis, ring_i, outer_i, ring_i+1), in `layers` layers of hexahedra: a
    node of the axis belongs to 2 n of them and has 3 (2 n + 1) neighbours."""
    ang = 2 * np.pi * np.arange(n) / n
    ring = np.stack([np.cos(ang), np.sin(ang)], 1)
    outer = 1.6 * np.stack([np.cos(ang + np.pi / n), np.sin(ang + np.pi / n)], 1)
    plane = np.concatenate([[[0.0, 0.0]], ring, outer])
    m = len(plane)
    xyz = np.concatenate([np.column_stack([plane, np.full(m, 0.7 * k)]) for k in range(layers + 1)])
    rng = np.random.default_rng(0)
    xyz += 0.03 * rng.uniform(-1, 1, xyz.shape)
    quad = [(0, 1 + i, 1 + n + i, 1 + (i + 1) % n) for i in range(n)]
    conn = np.array([[q + k * m for q in f] + [q + (k + 1) * m for q in f] for k in range(layers) for f in quad], np.int32)
    if collapsed:
        conn[3, 6] = conn[3, 5]
    return xyz, conn


def _case(kind, body, elemental, collapsed=False):
    xyz, conn = sectors(collapsed=collapsed)
    rng = np.random.default_rng(9)
    ph = fe.Physics(kind, "hexahedron", beta=0.5, c=2.0, E=1.7, nu=0.3, body=body)
    field = rng.uniform(0.5, 2.0, len(conn) if elemental else len(xyz))
    u = rng.uniform(0.0, 1.0, len(xyz)) if kind == "thermal" else rng.uniform(-0.03, 0.03, 3 * len(xyz))
    didx = np.arange(0, ph.ndpn * len(xyz), 7)
    return dict(kind=kind, etype="hexahedron", ph=ph, coords=xyz, conn=conn, field=field, u=u, didx=didx,
                dval=np.zeros(didx.size), elemental=elemental, beta=0.5, c=2.0, body=body)


def _context(case):
    from folax_amd.context import FemhotContext
    bf = np.zeros(3)
    if case["body"] is not None:
        b = np.atleast_1d(case["body"])
        bf[: b.size] = b
    return FemhotContext(case["etype"], PHYS_CODE[case["kind"]], case["coords"], case["conn"], num_gp=case["ph"].num_gp,
                         young_modulus=case["ph"].E, poisson_ratio=case["ph"].nu, beta=case["beta"], c=case["c"],
                         body_force=bf, dirichlet_idx=case["didx"], dirichlet_val=case["dval"])


def _check(case, dtype):
    from folax_amd import _lib as L
    ctx = _context(case)
    f = torch.as_tensor(case["field"], dtype=dtype, device="cuda")
    u = torch.as_tensor(case["u"], dtype=dtype, device="cuda")
    flags = L.SCATTER_ROWS | (L.ELEMENT_FIELD if case["elemental"] else 0)
    K, R = ctx.tangent_csr(f, u, flags=flags)
    Kr, Rr = fe.assemble(case["ph"], case["coords"], case["conn"], case["field"], case["u"], case["didx"])
    tol = 1e-12 if dtype == torch.float64 else 1e-5
    assert np.linalg.norm(K.double().cpu().numpy() - Kr.data) <= tol * np.linalg.norm(Kr.data)
    assert np.linalg.norm(R.double().cpu().numpy() - Rr) <= tol * np.linalg.norm(Rr)
    R2, _ = ctx.residual(f, u, want_energy=False, flags=(flags & L.ELEMENT_FIELD) | L.MASK_DIRICHLET)
    assert float((R2.reshape(-1) - R).norm()) <= tol * float(R.norm())
    again, Ra = ctx.tangent_csr(f, u, flags=flags | L.ACCUMULATE, out_vals=K.clone())
    assert torch.equal(again, 2 * K) and Ra.shape == R.shape
    same, Rs = ctx.tangent_csr(f, u, flags=flags)
    assert torch.equal(same, K) and torch.equal(Rs, R)  # a fixed order
    ctx.close()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("kind", ["thermal", "mechanical", "neohooke"])
@pytest.mark.parametrize("with_body,elemental,collapsed", [(False, False, False), (True, True, False), (False, True, True)])
def test_wide_nodes(kind, with_body, elemental, collapsed, dtype):
    if collapsed and kind != "thermal" and dtype == torch.float32:
        pytest.skip("a collapsed corner's inverse Jacobian exceeds the FP32 bar")
    body = None if not with_body else (0.4 if kind == "thermal" else [0.2, -0.3, 0.1])
    _check(_case(kind, body, elemental, collapsed), dtype)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("kind,etype", [("thermal", "quad"), ("mechanical", "quad"), ("thermal", "tetra"),
                                        ("mechanical", "tetra"), ("mechanical", "hexahedron")])
@pytest.mark.parametrize("rule", [1, 2, 3])
def test_residual_beside_the_tangent(kind, etype, rule, dtype):
    for body in (None, 0.4 if kind == "thermal" else ([0.2, -0.3] if etype == "quad" else [0.2, -0.3, 0.1])):
        case = make_case(kind, etype, n=3, seed=17, beta=0.5, c=2.0, body=body, num_gp=rule)
        _check(case, dtype)
