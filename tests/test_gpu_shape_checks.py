"""Arguments that the shape sensitivity refuses on the host: a field, state or adjoint of another size, type or device, or
strided."""
import pytest

from tests.cases import femhot_context, make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,etype", [("mechanical", "tetra"), ("thermal", "quad")])
def test_refused(kind, etype):
    case = make_case(kind, etype, n=3, seed=2)
    ctx = femhot_context(case)
    good = {k: torch.as_tensor(case[k], dtype=torch.float64, device="cuda") for k in ("field", "u", "w")}
    want = ctx.residual_shape_vjp(**good)
    assert want.shape == (ctx.n_nodes, 3)
    for name, t in good.items():
        for bad, error in ((t[:-1], ValueError), (torch.cat([t, t[:1]]), ValueError), (t.cpu(), ValueError),
                           (t.repeat_interleave(2)[::2], ValueError), (t.float(), TypeError)):
            if name == "u" and bad.dtype != t.dtype:
                continue  # u gives the call its type
            with pytest.raises(error):
                ctx.residual_shape_vjp(**{**good, name: bad})
    assert torch.equal(ctx.residual_shape_vjp(**{k: t.reshape(1, -1) for k, t in good.items()}), want)
    ctx.close()
