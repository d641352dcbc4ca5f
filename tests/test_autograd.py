"""The gradients that sapien_amd.autograd hands to torch, on the CPU with a
stand-in for the model's kernels."""
import pytest

torch = pytest.importorskip("torch")

from sapien_amd import autograd as A  # noqa: E402

B, N = 5, 4


class _Model:
    """loss = sum of 1 q + 2 qd + 3 qdd per environment."""

    def _pose_torque_loss_packed(self, q, qd, qdd, tau_target, ee_link, p_target):
        parts = [x.detach() for x in (q, qd, qdd) if x is not None]
        loss = sum((k + 1.0) * x for k, x in enumerate(parts)).sum(1)
        return loss, torch.stack([torch.full((B, N), k + 1.0) for k in range(3 if tau_target is not None else 1)])


@pytest.mark.parametrize("wanted", [(0,), (1,), (0, 2), (0, 1, 2)])
@pytest.mark.parametrize("create_graph", [False, True])
def test_pose_torque_gradients_are_tensors_of_their_own(wanted, create_graph):
    """No views (they refuse changes in place, and detach_), and no more memory
    held than the gradients asked for need."""
    q, qd, qdd = (torch.randn(B, N).requires_grad_(k in wanted) for k in range(3))
    ins = [x for x in (q, qd, qdd) if x.requires_grad]
    scale = torch.rand(B)
    loss = A.pose_torque_loss(_Model(), q, qd, qdd, torch.zeros(B, N))
    grads = torch.autograd.grad(loss, ins, grad_outputs=scale, create_graph=create_graph)
    for k, g in zip(wanted, grads):
        assert torch.equal(g, (k + 1.0) * scale[:, None].expand(B, N)) and g.is_contiguous()
        assert not g._is_view() and not g.requires_grad
    assert sum({g.untyped_storage().data_ptr(): g.untyped_storage().nbytes() for g in grads}.values()) == \
        sum(g.numel() * 4 for g in grads)
    before = [g.clone() for g in grads[1:]]
    grads[0].mul_(torch.full((N,), 2.0, requires_grad=True))
    grads[0].detach_()
    assert torch.equal(grads[0], 2.0 * (wanted[0] + 1.0) * scale[:, None].expand(B, N))
    assert all(torch.equal(a, b) for a, b in zip(before, grads[1:]))


def test_pose_loss_alone_has_no_torque_gradients():
    q = torch.randn(B, N, requires_grad=True)
    A.pose_torque_loss(_Model(), q, p_target=torch.zeros(B, 3)).sum().backward()
    assert torch.equal(q.grad, torch.ones(B, N)) and not q.grad._is_view()
