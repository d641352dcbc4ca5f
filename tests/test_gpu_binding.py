"""GPU: how the batched methods take their tensors. A plain contiguous float32
tensor on the model's GPU is read in place; anything else goes through torch's
conversions or DLPack, to the same results, and what is refused stays refused."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from sapien_amd import synthetic as S  # noqa: E402
from test_gpu_parity import _pair, _t  # noqa: E402


class _Sub(torch.Tensor):
    pass


def _padded(x):
    return torch.cat([x, x], 1)[:, : x.shape[1]]


FORMS = {
    "parameter": torch.nn.Parameter,
    "requires grad": lambda x: x.clone().requires_grad_(True),
    "non-leaf": lambda x: x.clone().requires_grad_(True) * 1.0,
    "subclass": lambda x: x.as_subclass(_Sub),
    "strided rows": _padded,
    "transposed": lambda x: x.t().contiguous().t(),
    "float64": lambda x: x.double(),
    "cpu": lambda x: x.cpu(),
    "numpy": lambda x: x.cpu().numpy(),
    "list": lambda x: x.tolist(),
}


@pytest.fixture(scope="module")
def arm():
    rob = S.arm9()
    m, _ = _pair(rob)
    return m, [_t(x) for x in S.samples(rob, 5, 3600)]


@pytest.mark.parametrize("form", FORMS)
def test_input_forms(arm, form):
    m, (q, qd, qdd, tau) = arm
    f = FORMS[form]
    for got, want in ((m.compute_fk_jacobian_rnea_batched(f(q), f(qd), f(qdd)),
                       m.compute_fk_jacobian_rnea_batched(q, qd, qdd)),
                      (m.rollout_batched(f(q), f(qd), f(tau)[:, None] if not isinstance(f(tau), list) else
                                         [[r] for r in f(tau)], 1e-3), m.rollout_batched(q, qd, tau[:, None], 1e-3)),
                      (m.pose_torque_loss_batched(f(q), f(qd), f(qdd), f(tau)),
                       m.pose_torque_loss_batched(q, qd, qdd, tau))):
        for a, b in zip(got, want):
            assert not a.requires_grad and torch.equal(a, b)
    if form == "transposed":  # passive forces read padded rows in place: the last dimension has to be contiguous
        with pytest.raises(ValueError):
            m.compute_passive_force_batched(f(q), f(qd))
    else:
        assert torch.equal(m.compute_passive_force_batched(f(q), f(qd)), m.compute_passive_force_batched(q, qd))
    if form != "list":  # one row without its batch dimension
        assert torch.equal(m.compute_forward_kinematics_batched(f(q)[0]), m.compute_forward_kinematics_batched(q[:1]))


def test_refusals(arm):
    m, (q, qd, qdd, tau) = arm
    poses = torch.empty(5, m.nlinks, 7, device="cuda")
    body = torch.zeros(5, m.nlinks, 13, device="cuda")
    leaf = q.clone().requires_grad_(True)
    for bad in (leaf, q.double(), q.cpu(), q[:, :4], q.t().contiguous().t(), q[None]):
        with pytest.raises(Exception):
            m.compute_fk_jacobian_rnea_into(bad, poses=poses)
        with pytest.raises(Exception):
            m.compute_link_state_into(bad, body=body)
        with pytest.raises(Exception):
            m.rollout_step_(bad, qd.clone(), tau, 1e-3)
        with pytest.raises(Exception):
            m.rollout_step_(q.clone(), bad, tau, 1e-3)
    for bad in (q[:, :4], q[None], torch.empty(0, 4, device="cuda"), None):
        with pytest.raises((RuntimeError, ValueError)):
            m.compute_forward_kinematics_batched(bad)
    with pytest.raises(RuntimeError):
        m.compute_inverse_dynamics_batched(q, qd[:3], qdd)
    with pytest.raises(RuntimeError):
        m.kinematics_vjp_batched(q, grad_poses=poses[:, :1])
    assert m.compute_forward_kinematics_batched(q[:0]).shape == (0, m.nlinks, 7)


def test_streams(arm):
    """torch's current stream, and a raw stream handed in, for a tensor made on it."""
    m, (q, qd, qdd, _) = arm
    want = m.compute_inverse_dynamics_batched(q, qd, qdd)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = m.compute_inverse_dynamics_batched(q * 1.0, qd, qdd)
    raw = m.compute_inverse_dynamics_batched(q, qd, qdd, stream=side.cuda_stream)
    side.synchronize()
    assert torch.equal(got, want) and torch.equal(raw, want)
    assert np.isfinite(want.cpu().numpy()).all()


def test_expanded_rows(arm):
    """One row standing for all of them (stride 0): copied out where inputs are
    converted, refused where buffers are used in place."""
    m, (q, qd, _, _) = arm
    B, n = q.shape
    eq, eqd = q[:1].expand(B, n), qd[0].expand(B, n)
    rows = [x.contiguous() for x in (eq, eqd)]
    for f in (lambda x: x, lambda x: x.clone()[:1].expand(B, n).requires_grad_(True), torch.Tensor.double,
              lambda x: x.as_subclass(_Sub)):
        assert torch.equal(m.compute_passive_force_batched(f(eq), f(eqd)), m.compute_passive_force_batched(*rows))
        assert torch.equal(m.compute_forward_kinematics_batched(f(eq)), m.compute_forward_kinematics_batched(rows[0]))
    poses, tau = torch.empty(B, m.nlinks, 7, device="cuda"), torch.empty(B, n, device="cuda")
    body = torch.zeros(B, m.nlinks, 13, device="cuda")
    for bad in (eq, eq.as_subclass(_Sub)):
        for call in (lambda: m.compute_fk_jacobian_rnea_into(bad, poses=poses),
                     lambda: m.compute_fk_jacobian_rnea_into(q, qvel=bad, qacc=q, qf=tau),
                     lambda: m.compute_fk_jacobian_rnea_into(q, qvel=q, qacc=q, qf=bad),
                     lambda: m.compute_fk_jacobian_rnea_into(q, poses=poses[:1].expand_as(poses)),
                     lambda: m.compute_fk_jacobian_rnea_into(q, poses=poses[:, :1].expand_as(poses)),
                     lambda: m.compute_link_state_into(bad, body=body),
                     lambda: m.compute_link_state_into(q, qvel=bad, body=body),
                     lambda: m.compute_link_state_into(q, body=body[:1].expand_as(body)),
                     lambda: m.compute_passive_force_batched(q, qd, out=bad)):
            with pytest.raises(ValueError, match="expanded"):
                call()
    one = q[:1].as_strided((1, n), (0, 1))  # the stride of a single row says nothing
    m.compute_fk_jacobian_rnea_into(one, qvel=one, qacc=one, qf=tau[:1])
    assert torch.equal(tau[:1], m.compute_inverse_dynamics_batched(q[:1], q[:1], q[:1]))


def test_rollout_step_on_one_row(arm):
    """One environment's configuration without its batch dimension, updated in place."""
    m, (q, qd, _, tau) = arm
    want = q[:1].clone(), qd[:1].clone()
    m.rollout_step_(*want, tau[:1], 1e-3)
    row, v = q[0].clone(), qd[:1].clone()
    m.rollout_step_(row, v, tau[:1], 1e-3)
    assert torch.equal(row, want[0][0]) and torch.equal(v, want[1])
    with pytest.raises(Exception):
        m.rollout_step_(q[0].clone(), qd.clone(), tau, 1e-3)  # one environment against five
