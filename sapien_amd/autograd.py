"""torch.autograd.Function wrappers over the hand-written adjoint kernels.

* ``link_poses(model, q)``            -> (B, L, 7) poses; backward = FK pose VJP kernel
* ``inverse_dynamics(model, q, qd, qdd)`` -> (B, nv) torques; backward = RNEA VJP kernel
* ``pose_torque_loss(model, q, qd, qdd, tau_target, ee_link, p_target)``
      -> (B,) loss_b = |tau - tau*|^2 + |p_ee - t|^2; the forward kernel returns
      the loss and its gradients in one pass, backward only scales them.
* ``rollout(model, q0, qd0, tau, dt, checkpoint_every=16)`` -> final (q_T, qd_T)
      of semi-implicit Euler with ABA over tau (B, T, nv); the forward keeps the
      state every K steps, backward recomputes each K-step segment from its
      checkpoint and runs the step adjoint kernel backwards through it.

Backward passes recompute the forward inside the adjoint kernel from the saved
inputs (no intermediates are stored between forward and backward). Kernels run
in FP32; gradients are returned in the dtype of the inputs. The Jacobian output
of the batched API has no adjoint (its derivative is second order).
"""
from __future__ import annotations

import torch


def _as(x, dtype):
    return x if x.dtype is dtype else x.to(dtype=dtype)


class _LinkPoses(torch.autograd.Function):
    @staticmethod
    def forward(ctx, model, q):
        ctx.model = model
        ctx.save_for_backward(q)
        return _as(model.compute_forward_kinematics_batched(q), q.dtype)

    @staticmethod
    def backward(ctx, gposes):
        (q,) = ctx.saved_tensors
        dq, _, _ = ctx.model.kinematics_vjp_batched(q, grad_poses=gposes)
        return None, _as(dq, q.dtype)


class _InverseDynamics(torch.autograd.Function):
    @staticmethod
    def forward(ctx, model, q, qd, qdd):
        ctx.model = model
        ctx.save_for_backward(q, qd, qdd)
        return _as(model.compute_inverse_dynamics_batched(q, qd, qdd), q.dtype)

    @staticmethod
    def backward(ctx, gtau):
        q, qd, qdd = ctx.saved_tensors
        dq, dqd, dqdd = ctx.model.kinematics_vjp_batched(q, qd, qdd, grad_tau=gtau)
        return None, _as(dq, q.dtype), _as(dqd, qd.dtype), _as(dqdd, qdd.dtype)


class _PoseTorqueLoss(torch.autograd.Function):
    @staticmethod
    def forward(ctx, model, q, qd, qdd, tau_target, ee_link, p_target):
        loss, grads = model._pose_torque_loss_packed(q, qd, qdd, tau_target, ee_link, p_target)
        ctx.save_for_backward(grads)  # (dq, dqd, dqdd), or dq alone, in one tensor: one product scales them
        ctx.dtypes = (q.dtype, None if qd is None else qd.dtype, None if qdd is None else qdd.dtype)
        return _as(loss, q.dtype)

    @staticmethod
    def backward(ctx, gloss):
        (grads,) = ctx.saved_tensors
        s = _as(gloss.detach(), torch.float32)[:, None]
        need = ctx.needs_input_grad[1:4]
        if all(need) and len(grads) == 3:
            # one product for all three; .data: tensors over it that are not views to autograd (a view
            # made here would refuse changes in place). 208 us a training pass of 8192 9-joint arms, 228
            # with three products.
            parts = [g.data for g in (grads * s).unbind(0)]
        else:  # a product, and its memory, for each gradient asked for
            parts = [grads[k] * s if need[k] and k < len(grads) else None for k in range(3)]
        out = tuple(None if g is None else _as(g, d) for g, d in zip(parts, ctx.dtypes))
        return (None,) + out + (None, None, None)


class _Rollout(torch.autograd.Function):
    @staticmethod
    def forward(ctx, model, q0, qd0, tau, dt, K):
        qT, qdT, ckpt = model.rollout_batched(q0.detach(), qd0.detach(), tau.detach(), dt, K)
        ctx.model, ctx.dt, ctx.K = model, dt, K
        ctx.dtypes = (q0.dtype, qd0.dtype, tau.dtype)
        ctx.save_for_backward(tau.detach().to(torch.float32).contiguous(), ckpt)
        return qT.to(q0.dtype), qdT.to(qd0.dtype)

    @staticmethod
    def backward(ctx, gq, gqd):
        tau, ckpt = ctx.saved_tensors
        gq = torch.zeros_like(tau[:, 0]) if gq is None else gq.detach().to(torch.float32).contiguous()
        gqd = torch.zeros_like(tau[:, 0]) if gqd is None else gqd.detach().to(torch.float32).contiguous()
        dq0, dqd0, dtau = ctx.model.rollout_backward_batched(tau, ckpt, ctx.dt, gq, gqd, ctx.K)
        return None, dq0.to(ctx.dtypes[0]), dqd0.to(ctx.dtypes[1]), dtau.to(ctx.dtypes[2]), None, None


def link_poses(model, q):
    return _LinkPoses.apply(model, q)


def inverse_dynamics(model, q, qd, qdd):
    return _InverseDynamics.apply(model, q, qd, qdd)


def pose_torque_loss(model, q, qd=None, qdd=None, tau_target=None, ee_link=0, p_target=None):
    return _PoseTorqueLoss.apply(model, q, qd, qdd, tau_target, ee_link, p_target)


def rollout(model, q0, qd0, tau, dt, checkpoint_every=16):
    return _Rollout.apply(model, q0, qd0, tau, dt, checkpoint_every)
