"""Differentiable force evaluation: a ``torch.autograd.Function`` over the C ABI.

The forward pass is one ``rbmdx_force`` evaluation; the backward pass is
``rbmdx_force_vjp`` with the incoming gradient of the forces as the cotangent:
hand-written adjoint kernels give dL/d(positions) and, per atom type,
dL/dQ (the type's charge), dL/deps and dL/dsigma.  The structure factor is
recomputed in the backward pass, not stored per atom and k.

Per-type charges are applied as per-atom charges Q[type]; an update may not
turn a neutral type charged or back (the charged/neutral partition of the pair
work is fixed when the system is set).  dL/dQ of a neutral type is therefore 0
unless ``neutral_charge_grad=True``, which computes it as the derivative at
Q = 0 (the Coulomb pairs of charged and neutral atoms and the neutral atoms'
structure sums enter the backward pass).  The pair set (RBL sampling epoch
``step``) and the k-sample are those of the forward evaluation; the backward
pass must run before the next forward evaluation of the same context.
"""
import numpy as np
import torch

from . import ForceContext, _current_stream


class _ForceFn(torch.autograd.Function):
    @staticmethod
    def forward(fctx, pos, Q, eps, sigma, model, step, m_samples, num_k):
        model._apply(Q, eps, sigma, pos.device)
        # one transposing copy each way; the rows are the SoA arrays (a copy in any
        # memory order: the caller may change pos before the backward pass)
        x = pos.transpose(0, 1).clone(memory_format=torch.contiguous_format)
        f = torch.empty_like(x)
        model.ctx.force(step, *x.unbind()[:3], *f.unbind()[:3], m_samples=m_samples,
                        num_k=num_k)
        fctx.save_for_backward(x)
        fctx.model = model
        fctx.step = step
        fctx.pdev = (Q.device, eps.device, sigma.device)
        fctx.pdtype = (Q.dtype, eps.dtype, sigma.dtype)
        return f[:3].transpose(0, 1).contiguous()

    @staticmethod
    def backward(fctx, gF):
        x, = fctx.saved_tensors
        model = fctx.model
        g = gF.to(x.dtype).transpose(0, 1).contiguous()
        d = torch.empty_like(g)
        nt = model.ntypes
        dparam = torch.empty(3 * nt, dtype=torch.float64, device=x.device)
        model.ctx.force_vjp(fctx.step, *x.unbind()[:3], *g.unbind(), *d.unbind(), dparam,
                            neutral_q=model.neutral_charge_grad)
        dpos = d.transpose(0, 1).contiguous()
        grads = [dparam[k * nt:(k + 1) * nt].to(device=dev, dtype=dt)
                 for k, (dev, dt) in enumerate(zip(fctx.pdev, fctx.pdtype))]
        return (dpos, *grads, None, None, None, None)


class DifferentiableForce:
    """Force field of one system as a differentiable function of positions
    and per-type (Q, eps, sigma).

    >>> model = DifferentiableForce(cfg, system)
    >>> F = model(pos, Q, eps, sigma, step=0, m_samples=m)
    >>> ((F - F_target) ** 2).sum().backward()
    """

    def __init__(self, cfg, system, device=0, neutral_charge_grad=False):
        self.neutral_charge_grad = bool(neutral_charge_grad)
        self.ctx = ForceContext(cfg, device=device)
        self.types = np.asarray(system.types, dtype=np.int32)
        self.ntypes = len(system.eps)
        self.ctx.set_system(system.box_lo, system.box_len, system.types, system.ids,
                            system.charges, system.eps, system.sigma)
        self._state = None

    def _apply(self, Q, eps, sigma, device):
        par = [t.detach() for t in (Q, eps, sigma)]
        if all(t.is_cuda and t.device == Q.device for t in par):
            # one copy to the host (each waits for the device)
            flat = torch.cat([t.reshape(-1).to(torch.float64) for t in par]).cpu().numpy()
            n = [t.numel() for t in par]
            q, e, s = (a.reshape(t.shape) for a, t in
                       zip(np.split(flat, [n[0], n[0] + n[1]]), par))
        else:
            q, e, s = (np.asarray(t.cpu(), dtype=np.float64) for t in par)
        same_q = self._state is not None and np.array_equal(q, self._state[0])
        same_lj = (self._state is not None and np.array_equal(e, self._state[1])
                   and np.array_equal(s, self._state[2]))
        if not (same_q and same_lj):
            if q.shape == e.shape == s.shape == (self.ntypes,):
                self.ctx.set_type_params(q, e, s, _current_stream(device))
            else:
                if not same_q:
                    self.ctx.set_charges(q[self.types])
                if not same_lj:
                    self.ctx.set_lj(e, s)
        self._state = (q, e, s)

    def __call__(self, pos, Q, eps, sigma, step=0, m_samples=None, num_k=None):
        return _ForceFn.apply(pos, Q, eps, sigma, self, int(step), m_samples, num_k)
