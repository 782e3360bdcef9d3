"""Finite-element responses and their adjoint sensitivities over libfemhot (PyTorch-ROCm host side).

FiniteElementResponse follows fol/responses/fe_response.py:17-719 with the same method names and
meaning.  A response is f = sum_e sum_g w detJ phi(N.d, N.u) for a user formula phi written in
terms of the control's name and the first letter of the first dof ("(E**2)*U[0]" reads E = N.d
and U[c] = N.u_c at each Gauss point, fe_response.py:61-66, 92-113).

What runs where:
* the Gauss-point geometry (w detJ, N, dN/dx) comes from the library (femhot_gauss_point_data);
* the nodal field and state are brought to the Gauss points, and Gauss-point terms back to the nodes,
  by the library's gather kernels (under torch's transforms and traces, by torch's own operators);
* phi is evaluated on the device with torch on all Gauss points at once, and its derivatives with
  respect to the Gauss-point field and state come from torch autograd of that evaluation (the
  formula is arbitrary Python, as the reference's jax.grad of its eval'd lambda);
* the adjoint terms lambda^T dR/dk and lambda^T dR/dX run in the hand-written residual VJP and
  shape-VJP kernels, the transposed tangent in the CSR assembly kernel, and the adjoint solve in
  the device PCG.
"""
from __future__ import annotations

import torch
from torch.autograd import forward_ad

from . import _lib as L
from .loss_functions import FiniteElementLoss, _as_device_tensor, _has_memory


class _ArrayNamespace:
    """The `jnp` a response formula may call (fe_response.py:64 evaluates it with jnp in scope):
    numpy-named functions resolved to torch's elementwise ones."""

    _alias = {"power": torch.pow, "arctan": torch.atan, "arcsin": torch.asin, "arccos": torch.acos,
              "absolute": torch.abs}

    def __getattr__(self, name):
        if name in self._alias:
            return self._alias[name]
        return getattr(torch, name)


def _kernels_read(*tensors):
    """Whether the gather kernels can take these tensors: plain ones with memory of their own, outside torch's
    transforms (functorch, forward mode, batched gradients) and traces, which need operators they know."""
    if (forward_ad._current_level >= 0 or torch._C._len_torch_dispatch_stack() or torch._C._is_tracing()
            or torch.compiler.is_compiling()):
        return False
    for t in tensors:
        if not (type(t) in (torch.Tensor, torch.nn.Parameter) and _has_memory(t)) \
                or torch._C._functorch.is_functorch_wrapped_tensor(t):
            return False
    return True


def _point_values(r, d, u):
    """N.d (n_elems, G) and N.u (dofs per node, n_elems, G) of response r's mesh: by the kernel, or by torch's own
    operators where that cannot be (the linear map is the same)."""
    if _kernels_read(d, u):
        if not (torch.is_grad_enabled() and (d.requires_grad or u.requires_grad)):  # nothing to record
            return r.fe_loss.ctx.gauss_point_values(d.contiguous(), u.contiguous(), r.fe_loss.num_gp)
        return _PointValues.apply(r, d, u)
    N, conn = r._geometry(u.dtype, u.device)[0], r._connectivity(u.device)
    return d[conn] @ N.T, u.view(-1, r.fe_loss.number_dofs_per_node)[conn].permute(2, 0, 1) @ N.T


def _point_gather(r, q):
    """The transpose of _point_values per component: q (ncomp, n_elems, G) -> (n_nodes, ncomp)."""
    if _kernels_read(q):
        return _PointGather.apply(r, q)
    N, conn = r._geometry(q.dtype, q.device)[0], r._connectivity(q.device)
    corners = (q @ N).permute(1, 2, 0).reshape(-1, q.shape[0])
    zero = torch.zeros(r.fe_loss.ctx.n_nodes, q.shape[0], dtype=q.dtype, device=q.device)
    return zero.index_add(0, conn.reshape(-1), corners)


class _PointValues(torch.autograd.Function):
    """N.d and N.u at the Gauss points; its transpose is the gather of _PointGather, so both differentiate
    to any order."""

    @staticmethod
    def forward(ctx, r, d, u):
        ctx.r, ctx.shapes = r, (d.shape, u.shape)
        return r.fe_loss.ctx.gauss_point_values(d.contiguous(), u.contiguous(), r.fe_loss.num_gp)

    @staticmethod
    def backward(ctx, gd, gu):
        return (None, _point_gather(ctx.r, gd.unsqueeze(0)).reshape(ctx.shapes[0]) if ctx.needs_input_grad[1] else None,
                _point_gather(ctx.r, gu).reshape(ctx.shapes[1]) if ctx.needs_input_grad[2] else None)


class _PointGather(torch.autograd.Function):
    """sum of N_a q at the nodes, (n_nodes, ncomp); the transpose of _PointValues per component."""

    @staticmethod
    def forward(ctx, r, q):
        ctx.r, ctx.ncomp = r, q.shape[0]
        return r.fe_loss.ctx.gauss_point_gather(q, r.fe_loss.num_gp)

    @staticmethod
    def backward(ctx, g):
        zero = torch.zeros(ctx.r.fe_loss.ctx.n_dofs, dtype=g.dtype, device=g.device)
        return None, torch.stack([_point_values(ctx.r, g[:, c].contiguous(), zero)[0] for c in range(ctx.ncomp)])


class FiniteElementResponse:
    """fe_response.py:17-45: a named response formula over an FE loss and a control."""

    def __init__(self, name: str, response_formula: str, fe_loss: FiniteElementLoss, control):
        self.name = name
        self.response_formula = response_formula
        self.fe_loss = fe_loss
        self.control = control
        self.initialized = False

    def GetName(self):
        return self.name

    def Initialize(self, reinitialize=False):
        """fe_response.py:47-69: the formula becomes lambda <control name>, <first dof letter>: formula."""
        if self.initialized and not reinitialize:
            return
        self.fe_loss.Initialize()
        self.control.Initialize()
        variables = [self.control.GetName(), self.fe_loss.dofs[0][0]]
        self.response_function = eval(f"lambda {', '.join(variables)}: {self.response_formula}",
                                      {"jnp": _ArrayNamespace()})
        self._gp = {}
        self._conn = None
        self._has_both = False
        self.fe_loss.ctx.build_incidence()
        self.initialized = True

    # ---- Gauss-point integrand ----
    def _geometry(self, dtype, device):
        key = (dtype, device)
        if key not in self._gp:
            self._gp[key] = self.fe_loss.ctx.gauss_point_data(self.fe_loss.num_gp, dtype=dtype, device=device)
        return self._gp[key]

    def _connectivity(self, device):
        if self._conn is None or self._conn.device != device:
            with torch._C._DisableFuncTorch():  # kept beyond the transform that first needs it
                self._conn = torch.as_tensor(self.fe_loss.fe_mesh.GetElementsNodes(self.fe_loss.element_type),
                                             dtype=torch.int64, device=device)
        return self._conn

    def _inputs(self, control, dofs):
        u = _as_device_tensor(dofs)
        d = _as_device_tensor(control, dtype=u.dtype, device=u.device)
        return d.reshape(-1), u.reshape(-1)

    def _integrand(self, d, u):
        """w detJ (Ne, G) and, at the Gauss points, N.d (Ne, G) and N.u (ndpn, Ne, G): U[c] is component c."""
        _, wdet, _ = self._geometry(u.dtype, u.device)
        n, p = self.fe_loss.ctx.n_nodes, self.fe_loss.number_dofs_per_node
        if d.numel() < n or u.numel() < n * p:
            raise IndexError(f"a response reads {n} nodal control values and {n * p} dofs")
        if d.numel() > n or u.numel() > n * p:  # the nodes' values come first
            d, u = d[:n], u.view(-1, p)[:n].reshape(-1)
        gp_d, gp_u = _point_values(self, d, u)
        return wdet, gp_d, gp_u

    # ---- reference API ----
    def ComputeValue(self, nodal_control_values, nodal_dof_values):
        """fe_response.py:196-212: sum over elements and Gauss points."""
        d, u = self._inputs(nodal_control_values, nodal_dof_values)
        wdet, gp_d, gp_u = self._integrand(d, u)
        return (wdet * self.response_function(gp_d, gp_u)).sum()  # differentiable in both arguments

    def _point_grad(self, d, u, which):
        """Derivative of the response integrand, times w detJ, with respect to the Gauss-point field (which 0:
        (Ne, G)) or state (1: (ndpn, Ne, G)).  A formula that leaves out either is refused, which the
        first derivative taken finds out; later ones take the one that is asked for."""
        wdet, *points = self._integrand(d.detach(), u.detach())
        with torch.enable_grad():
            for k, p in enumerate(points):
                p.requires_grad_(k == which or not self._has_both)
            f = self.response_function(*points) * wdet
            grads = torch.autograd.grad(f, [p for p in points if p.requires_grad], torch.ones_like(f))
        self._has_both = True
        return grads[which if len(grads) == 2 else 0]

    def ComputeAdjointJacobianMatrixAndRHSVector(self, nodal_control_values, nodal_dof_values):
        """fe_response.py:244-283: rhs = -(df/du) with Dirichlet entries zeroed, and the BC-applied
        transposed tangent of the loss."""
        d, u = self._inputs(nodal_control_values, nodal_dof_values)
        q_u = self._point_grad(d, u, 1)
        idx, _ = self.fe_loss._dir_idx(u.device)
        rhs = -self.fe_loss.ctx.gauss_point_gather(q_u, self.fe_loss.num_gp).reshape(-1)
        rhs[idx] = 0.0
        K, _ = self.fe_loss.ComputeJacobianMatrixAndResidualVector(d, u, transpose_jacobian=True)
        return K, rhs

    def ComputeAdjointNodalControlDerivatives(self, nodal_control_values, nodal_dof_values, nodal_adj_dof_values):
        """fe_response.py:486-526: df/dk + lambda^T dR/dk (the residual VJP kernel)."""
        d, u = self._inputs(nodal_control_values, nodal_dof_values)
        lam = _as_device_tensor(nodal_adj_dof_values, dtype=u.dtype, device=u.device).reshape(-1)
        q_d = self._point_grad(d, u, 0)
        if self.fe_loss._has_own("ComputeResidualVJP"):
            _, gk = self.fe_loss.ComputeResidualVJP(d, u, lam)
            return self.fe_loss.ctx.gauss_point_gather(q_d.unsqueeze(0), self.fe_loss.num_gp).reshape(-1) + gk
        _, gk = self.fe_loss.ctx.residual_vjp(d.reshape(1, -1), u.reshape(1, -1), lam.reshape(1, -1), want_gu=False,
                                              flags=self.fe_loss._flags())
        if gk.numel() != self.fe_loss.ctx.n_nodes:  # an element field: the two have no common length
            return self.fe_loss.ctx.gauss_point_gather(q_d.unsqueeze(0), self.fe_loss.num_gp).reshape(-1) + gk[0]
        return self.fe_loss.ctx.gauss_point_gather(q_d.unsqueeze(0), self.fe_loss.num_gp, out=gk).reshape(-1)

    def ComputeAdjointNodalShapeDerivatives(self, nodal_control_values, nodal_dof_values, nodal_adj_dof_values):
        """fe_response.py:365-406: df/dX + lambda^T dR/dX, flattened (3 n_nodes,).  Only detJ of the
        integrand moves with the nodes: d(w detJ)/dX_a,i = w detJ dN_a/dx_i at each Gauss point; the
        residual term runs in the shape-VJP kernel."""
        d, u = self._inputs(nodal_control_values, nodal_dof_values)
        lam = _as_device_tensor(nodal_adj_dof_values, dtype=u.dtype, device=u.device).reshape(-1)
        wdet, gp_d, gp_u = self._integrand(d, u)
        wphi = (wdet * self.response_function(gp_d, gp_u)).contiguous()
        if wphi.shape != wdet.shape:
            raise RuntimeError(f"the response formula must give one value per Gauss point, got {tuple(wphi.shape)}")
        # the caller differentiates the integrand's part, or the loss has its own residual term
        if wphi.requires_grad or self.fe_loss._has_own("ComputeResidualShapeVJP"):
            _, _, dndx = self._geometry(u.dtype, u.device)
            ge = torch.einsum("eg,egaj->eaj", wphi, dndx)                # (Ne, n, dim)
            if ge.shape[-1] < 3:
                ge = torch.nn.functional.pad(ge, (0, 3 - ge.shape[-1]))
            conn = self._connectivity(u.device)
            dfdX = torch.zeros(self.fe_loss.fe_mesh.GetNumberOfNodes(), 3, dtype=u.dtype, device=u.device)
            dfdX.index_add_(0, conn.reshape(-1), ge.reshape(-1, 3))
            return dfdX.reshape(-1) + self.fe_loss.ComputeResidualShapeVJP(d, u, lam)
        flags = L.ELEMENT_FIELD if self.fe_loss.control_location == "element" else 0
        return self.fe_loss.ctx.residual_shape_vjp(d, u, lam, flags=flags, wphi=wphi).reshape(-1)

    def Finalize(self):
        pass
