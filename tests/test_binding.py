"""How the batched methods take their tensors, as far as it shows without a GPU:
a DLPack capsule that claims this model's (absent) GPU gets as far as torch's
stream of that GPU, unless the binding refuses it first."""
import ctypes
import os
import subprocess
import sys
import textwrap

import pytest

torch = pytest.importorskip("torch")

import sapien_amd as sa  # noqa: E402
from sapien_amd import synthetic as S  # noqa: E402

needs_no_gpu = pytest.mark.skipif(torch.cuda.is_available(), reason="the capsules hold host addresses")
TAKEN = "no ROCm-capable device"


class _Managed(ctypes.Structure):
    """DLManagedTensor (dlpack_abi.h) of a float32 tensor."""
    _fields_ = [("data", ctypes.c_void_p), ("device_type", ctypes.c_int32), ("device_id", ctypes.c_int32),
                ("ndim", ctypes.c_int32), ("code", ctypes.c_uint8), ("bits", ctypes.c_uint8),
                ("lanes", ctypes.c_uint16), ("shape", ctypes.POINTER(ctypes.c_int64)),
                ("strides", ctypes.POINTER(ctypes.c_int64)), ("byte_offset", ctypes.c_uint64),
                ("manager_ctx", ctypes.c_void_p), ("deleter", ctypes.c_void_p)]


class _OnDevice(torch.Tensor):
    """A host tensor whose DLPack capsule is one of the (absent) GPU of a model made without one."""

    def __dlpack__(self, **kw):
        n = self.dim()
        managed = _Managed(self.data_ptr(), 10, -1, n, 2, 32, 1, (ctypes.c_int64 * n)(*self.shape),
                                (ctypes.c_int64 * n)(*self.stride()), 0, None, None)
        self.__dict__.setdefault("managed", []).append(managed)  # they outlive their capsules
        new = ctypes.pythonapi.PyCapsule_New
        new.restype, new.argtypes = ctypes.py_object, [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p]
        return new(ctypes.addressof(managed), b"dltensor", None)


def _on_device(x):
    return x.as_subclass(_OnDevice)


@pytest.fixture(scope="module")
def arm():
    rob = S.arm9()
    m = sa.PinocchioModel(rob.urdf, [0.0, 0.0, -9.81])
    m.set_joint_order(rob.joint_names)
    m.set_link_order(rob.link_names)
    return m, rob.nv


class _Foreign:
    """No torch tensor: a shape and a DLPack capsule."""

    def __init__(self, x):
        self.tensor, self.shape = _on_device(x), tuple(x.shape)

    def __dlpack__(self, **kw):
        return self.tensor.__dlpack__()


@needs_no_gpu
def test_dlpack_objects_that_torch_does_not_know(arm):
    """The in-place methods take their buffers through DLPack alone."""
    (m, nv), B, L = arm, 3, arm[0].nlinks
    q, poses, body = (_Foreign(torch.zeros(s)) for s in ((B, nv), (B, L, 7), (B, L, 13)))
    with pytest.raises(RuntimeError, match=TAKEN):
        m.compute_fk_jacobian_rnea_into(q, qvel=q, qacc=q, poses=poses, qf=q)
    with pytest.raises(RuntimeError, match=TAKEN):
        m.compute_link_state_into(q, qvel=q, body=body)
    with pytest.raises(ValueError, match=">= nlinks"):
        m.compute_fk_jacobian_rnea_into(q, poses=_Foreign(torch.zeros(B, L - 1, 7)))


@needs_no_gpu
def test_expanded_tensors_are_refused_in_place(arm):
    """A row, environment or link stride of 0 over several entries: the C ABI
    would read it as contiguous rows, past the end of the tensor."""
    (m, nv), B, L = arm, 3, arm[0].nlinks
    q, poses, body = (_on_device(torch.zeros(s)) for s in ((B, nv), (B, L, 7), (B, L, 13)))
    expanded = {(d, n): _on_device(torch.zeros([1 if k == n else e for k, e in enumerate(d)]).expand(d))
                for d in ((B, nv), (B, L, 7), (B, L, 13)) for n in range(len(d) - 1)}
    into, state = m.compute_fk_jacobian_rnea_into, m.compute_link_state_into
    with pytest.raises(RuntimeError, match=TAKEN):
        into(q, qvel=q, qacc=q, poses=poses, qf=q)
    with pytest.raises(RuntimeError, match=TAKEN):
        state(q, qvel=q, body=body)
    eq = expanded[(B, nv), 0]
    calls = [lambda: into(eq, poses=poses), lambda: into(q, qvel=eq, qacc=q, qf=q), lambda: into(q, qvel=q, qacc=eq, qf=q),
             lambda: into(q, qvel=q, qacc=q, qf=eq), lambda: state(eq, body=body), lambda: state(q, qvel=eq, body=body)]
    calls += [lambda n=n: into(q, poses=expanded[(B, L, 7), n]) for n in (0, 1)]
    calls += [lambda n=n: state(q, body=expanded[(B, L, 13), n]) for n in (0, 1)]
    for call in calls:
        with pytest.raises(ValueError, match="expanded"):
            call()
    # one environment: its stride says nothing, and 0 is as good as any
    one = _on_device(torch.zeros(1, nv).as_strided((1, nv), (0, 1)))
    with pytest.raises(RuntimeError, match=TAKEN):
        into(one, qvel=one, qacc=one, qf=one)


def test_first_calls_from_two_threads():
    """The first batched calls of a process, from two threads at once, on numpy
    arrays and with torch not imported yet: both come back (here with torch's
    error for want of a GPU)."""
    script = textwrap.dedent("""
        import sys, threading
        import numpy as np
        import sapien_amd as sa
        from sapien_amd import synthetic as S
        assert "torch" not in sys.modules
        rob, gate, out = S.chain7(), threading.Barrier(2), [None, None]
        models = []
        for _ in out:
            m = sa.PinocchioModel(rob.urdf, [0.0, 0.0, -9.81])
            m.set_joint_order(rob.joint_names)
            m.set_link_order(rob.link_names)
            models.append(m)

        def call(i):
            gate.wait()
            try:
                out[i] = "poses", models[i].compute_forward_kinematics_batched(np.zeros((2, rob.nv))).shape
            except RuntimeError as e:
                out[i] = "error", str(e)

        threads = [threading.Thread(target=call, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert out[0] and out[0] == out[1], out
        """)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=root, HIP_VISIBLE_DEVICES="")
    subprocess.run([sys.executable, "-c", script], env=env, check=True, timeout=120)
