"""The scaled residual VJP under a recorded LDS-DMA configuration, the backward pass of a residual-norm loss whose
autotuner chose that kernel: the recorded kernel runs, and scales the cotangent."""
import numpy as np
import pytest

from tests.cases import femhot_context, make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

SIZES = {"quad": 20, "hexahedron": 7, "tetra": 5}


@pytest.mark.parametrize("picard", [False, True])
@pytest.mark.parametrize("elemental", [False, True])
@pytest.mark.parametrize("kind,etype", [("thermal", "quad"), ("mechanical", "hexahedron"), ("neohooke", "tetra"),
                                        ("thermal", "tetra")])
def test_recorded_kernel_scales(kind, etype, elemental, picard):
    from folax_amd import _lib as L
    extra = dict(beta=0.5, c=2.0) if kind == "thermal" else dict(u_scale=0.1 / SIZES[etype])
    case = make_case(kind, etype, n=SIZES[etype], seed=62, elemental=elemental, **extra)
    ctx = femhot_context(case)
    batch = 3
    rng = np.random.default_rng(4)
    f, u, w = (torch.as_tensor(np.stack([case[k] * rng.uniform(0.8, 1.2) for _ in range(batch)]), dtype=torch.float32,
                               device="cuda") for k in ("field", "u", "w"))
    base = L.SCATTER_CHUNK | L.MASK_DIRICHLET | (L.ELEMENT_FIELD if elemental else 0) | (L.PICARD if picard else 0)
    ctx.set_chunk_config(L.OP_VJP, torch.float32, batch, 128, 256 | L.CHUNK_DMA, -2, flags=base)
    plain = ctx.residual_vjp(f, u, w, flags=base)
    for scale, exact in ((2.0, True), (-0.25, True), (0.3, False)):
        s = torch.tensor(scale, dtype=torch.float32, device="cuda")
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
            got = ctx.residual_vjp(f, u, w, flags=base, scale=s)
            torch.cuda.synchronize()
        names = [e.key for e in prof.key_averages()]
        assert not names or any("k_chunk_pipe" in n for n in names), names  # (empty under another profiler)
        for a, b in zip(got, plain):
            if exact:  # linear in w, and powers of two commute with every rounding
                assert torch.equal(a, scale * b)
            else:  # the scaled cotangent and sums of at most 24 corners of 8 points round once more each
                assert float((a - scale * b).abs().max()) <= 400 * 2.0 ** -23 * abs(scale) * float(b.abs().max())
    ctx.close()
