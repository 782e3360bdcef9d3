"""Arguments that the Gauss-point kernels cannot index by are refused on the host, before any launch."""
import pytest

from tests.cases import femhot_context, make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("etype,rule,points", [("quad", 2, 4), ("hexahedron", 1, 1), ("tetra", 2, 4)])
def test_refused_before_a_launch(etype, rule, points):
    case = make_case("thermal", etype, n=3, seed=8, num_gp=rule)
    ctx = femhot_context(case)
    d, u, w = (torch.as_tensor(case[k], dtype=torch.float64, device="cuda") for k in ("field", "u", "w"))
    ne, nn = ctx.n_elems, ctx.n_nodes
    for other in (1, 2, 3):
        if other != rule:  # another rule than the context's
            with pytest.raises(ValueError, match="Gauss rule"):
                ctx.gauss_point_values(d, u, other)
            with pytest.raises(ValueError, match="Gauss rule"):
                ctx.gauss_point_gather(torch.zeros(1, ne, 1, dtype=torch.float64, device="cuda"), other)
    with pytest.raises(IndexError):
        ctx.gauss_point_values(d[:-1].contiguous(), u, rule)
    with pytest.raises(ValueError, match="contiguous"):
        ctx.gauss_point_values(torch.zeros(nn, 2, dtype=torch.float64, device="cuda")[:, 0], u, rule)
    with pytest.raises(ValueError, match="shape"):
        ctx.gauss_point_gather(torch.zeros(1, ne, points + 1, dtype=torch.float64, device="cuda"), rule)
    with pytest.raises(ValueError, match="device"):
        ctx.gauss_point_gather(torch.zeros(1, ne, points, dtype=torch.float64), rule)
    for size in (points - 1, 2 * points):  # whole multiples of the element count, too short or too long
        if size:
            with pytest.raises(ValueError, match="wphi"):
                ctx.residual_shape_vjp(d, u, w, wphi=torch.zeros(ne, size, dtype=torch.float64, device="cuda"))
    gd, gu = ctx.gauss_point_values(d, u, rule)
    assert gd.shape == (ne, points) and gu.shape == (1, ne, points)
    assert ctx.residual_shape_vjp(d, u, w, wphi=torch.zeros(ne, points, dtype=torch.float64, device="cuda")).isfinite().all()
    ctx.close()
