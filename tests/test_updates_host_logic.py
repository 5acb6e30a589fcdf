"""Batched parameter updates with the library calls replaced by a recorder (no
device): parameters that read or write each other's buffers are not put into one
launch."""
import struct
from types import SimpleNamespace

import pytest

from vulkpy_amd._lib import ADAM_STEP_FORMAT
from vulkpy_amd.nn import optimizers, parameters
from vulkpy_amd.nn.optimizers import AdamState
from vulkpy_amd.nn.parameters import Parameter, Updates

GPU = SimpleNamespace(_handle=1)


def array(ptr):
    return SimpleNamespace(_gpu=GPU, _ptr=ptr, size=4, _set_job=lambda keep=(): None)


def parameter(value, grad, m, v):
    p = Parameter.__new__(Parameter)
    p.value, p.grad, p.R = array(value), array(grad), None
    p.opt_state = st = AdamState.__new__(AdamState)
    st.opt = SimpleNamespace(lr=0.1, eps=1e-8, beta1=0.9, beta2=0.99)
    st.m, st.v, st.beta1t, st.beta2t = array(m), array(v), 1.0, 1.0
    return p


@pytest.mark.parametrize("second,together", [
    ((5, 6, 7, 8), True),
    ((5, 2, 7, 8), True),    # the same gradient, read by both
    ((1, 6, 7, 8), False),   # the same value
    ((5, 6, 3, 8), False),   # the same first moments
    ((5, 1, 7, 8), False),   # its gradient is the first one's value
    ((2, 6, 7, 8), False),   # its value is the first one's gradient
])
def test_parameters_that_share_buffers(monkeypatch, second, together):
    launches = []

    def record(name, handle, *args):
        if name == "vkh_adam_multi":
            launches.append([s[0] for s in struct.iter_unpack("@" + ADAM_STEP_FORMAT, args[0])])
        else:
            launches.append([args[0]])

    monkeypatch.setattr(parameters, "call", record)
    monkeypatch.setattr(optimizers, "call", record)
    batch = Updates()
    batch.add(parameter(1, 2, 3, 4))
    batch.add(parameter(*second))
    batch.flush()
    assert launches == ([[1, second[0]]] if together else [[1], [second[0]]])
