"""
Neural Network Parameter (:mod:`vulkpy_amd.nn.parameters`)
==========================================================

``Parameter`` with the interface of vulkpy/nn/parameters.py:14-116: a value,
an accumulated gradient (absent for frozen parameters), an optimizer state and
an optional regularizer.

On this backend every method is stream ordered and none waits on the host:

* ``zero_grad`` enqueues a fill kernel (the reference writes the mapped
  memory from the host, parameters.py:86);
* ``update`` runs the optimizer state's fused update kernel when the state
  class provides one (same FP32 operations as ``grad2diff`` + ``+=``);
* ``regular_grad`` adds the regularizer's gradient onto ``grad`` in one
  kernel for the penalties of :mod:`vulkpy_amd.nn.regularizers`.
"""
from __future__ import annotations
import struct
from typing import Callable, Iterable, List, Optional

from vulkpy_amd._lib import ADAM_MULTI_MAX, ADAM_STEP_FORMAT, FILL_MULTI_MAX, SPAN_FORMAT, call
from vulkpy_amd.vkarray import GPU, Array, zeros
from .core import Optimizer, OptimizerState, Regularizer
from .optimizers import Adam, AdamState
from .regularizers import _fused_penalty


__all__ = [
    "Parameter"
]


def _has_fused_update(state) -> bool:
    """True when the state's class provides ``_update`` and does not override
    the ``grad2diff`` that the fused kernel reproduces."""
    for klass in type(state).__mro__:
        if "_update" in vars(klass):
            return type(state).grad2diff is klass.grad2diff
    return False


class Parameter:
    """
    Parameter of a layer: value, gradient, optimizer state and regularizer

    Parameters
    ----------
    gpu : vulkpy_amd.GPU
        Device holding the value, gradient and optimizer state.
    shape : iterable of int
        Shape of the value.
    trainable : bool, optional
        Keep a gradient and an optimizer state (default ``True``).
    opt : vulkpy_amd.nn.Optimizer, optional
        Optimizer; ``Adam(gpu)`` when ``None``.
    initializer : callable, optional
        ``initializer(gpu, shape)`` returning the initial value; zeros when
        ``None``.
    regularizer : vulkpy_amd.nn.Regularizer, optional
        Penalty whose gradient ``regular_grad`` adds.
    """
    def __init__(self,
                 gpu: GPU,
                 shape: Iterable[int],
                 trainable: bool = True,
                 opt: Optional[Optimizer] = None,
                 initializer: Optional[Callable[[GPU, Iterable[int]], Array]]=None,
                 regularizer: Optional[Regularizer] = None):
        make_value = zeros if initializer is None else initializer
        self.value: Array = make_value(gpu, shape)
        self.R: Optional[Regularizer] = regularizer
        self.grad: Optional[Array] = None
        self.opt_state: Optional[OptimizerState] = None
        if not trainable:
            return
        self.grad = zeros(gpu, shape=shape)
        optimizer = Adam(gpu) if opt is None else opt
        self.opt_state = optimizer.init_state(shape)

    def is_trainable(self) -> bool:
        """Whether the parameter keeps a gradient"""
        return self.grad is not None

    def add_grad(self, grad: Array):
        """Accumulate ``grad`` (ignored for a frozen parameter)"""
        if not self.is_trainable():
            return
        self.grad += grad

    def zero_grad(self):
        """Reset the gradient to 0 (a fill kernel after earlier work on it)"""
        if not self.is_trainable():
            return
        self.grad._fill(0.0)

    def update(self):
        """Apply the optimizer step to ``value`` (trainable parameters only)"""
        if not self.is_trainable():
            return
        state = self.opt_state
        if _has_fused_update(state):
            state._update(self.value, self.grad)
            return
        step = state.grad2diff(self.grad)
        self.value += step

    def regular_loss(self) -> Array:
        """Regularization loss of the value; a (1,) zero without a regularizer"""
        if self.R is None:
            return zeros(self.value._gpu, shape=(1,))
        return self.R.loss(self.value)

    def regular_grad(self):
        """Add the regularizer's gradient to ``grad``"""
        if self.R is None or not self.is_trainable():
            return
        if _fused_penalty(self.R):
            self.R._add_grad(self.value, self.grad)
            return
        self.add_grad(self.R.grad(self.value))


def _plain(obj, method: str, own) -> bool:
    """Whether ``obj.method`` is the function ``own``, neither overridden in a
    subclass nor replaced on a class or on the object."""
    return getattr(type(obj), method, None) is own and method not in getattr(obj, "__dict__", ())


# what the batches below stand for, as defined here (a program may replace them)
_ZERO_GRAD, _UPDATE, _ADAM_UPDATE = Parameter.zero_grad, Parameter.update, AdamState._update


class ZeroGrads:
    """``Parameter.zero_grad`` of many parameters, up to ``FILL_MULTI_MAX`` a
    launch; ``flush`` issues what has been added."""

    def __init__(self):
        self._grads: List[Array] = []

    def add(self, p: Parameter):
        if type(p) is not Parameter or not _plain(p, "zero_grad", _ZERO_GRAD):
            self.flush()
            p.zero_grad()
        elif p.grad is not None:
            q = self._grads
            if q and (len(q) == FILL_MULTI_MAX or q[0]._gpu is not p.grad._gpu):
                self.flush()
            self._grads.append(p.grad)

    def flush(self):
        grads, self._grads = self._grads, []
        if len(grads) == 1:
            grads[0]._fill(0.0)
        elif grads:
            spans = [x for a in grads for x in (a._ptr, a.buffer.n)]
            call("vkh_fill_multi", grads[0]._gpu._handle, struct.pack(SPAN_FORMAT * len(grads), *spans),
                 len(grads), 0.0)
            for a in grads:
                a._set_job()


class Updates:
    """``Parameter.update`` of many parameters: those with the framework's own
    Adam state up to ``ADAM_MULTI_MAX`` a launch, with the bits of the single
    updates; any other parameter, or one that writes what one already added
    reads or writes (a shared value or state), or reads what that one writes,
    comes after those added before it."""

    def __init__(self):
        self._params: List[Parameter] = []
        self._written = set()
        self._read = set()

    def add(self, p: Parameter):
        if type(p) is not Parameter or not _plain(p, "update", _UPDATE):
            self.flush()
            p.update()
            return
        if p.grad is None:
            return
        state = p.opt_state
        if (type(state) is not AdamState or not _plain(state, "_update", _ADAM_UPDATE)
                or not (abs(state.opt.lr) < 1e38 and abs(state.opt.eps) < 1e38)
                or p.value._gpu is not p.grad._gpu or p.value.size == 0):
            self.flush()
            p.update()
            return
        mine = (p.value._ptr, state.m._ptr, state.v._ptr)
        if (len(self._params) == ADAM_MULTI_MAX or not self._written.isdisjoint(mine)
                or p.grad._ptr in self._written or not self._read.isdisjoint(mine)
                or (self._params and self._params[0].value._gpu is not p.value._gpu)):
            self.flush()
        self._params.append(p)
        self._written.update(mine)
        self._read.add(p.grad._ptr)

    def flush(self):
        params, self._params = self._params, []
        self._written.clear()
        self._read.clear()
        if len(params) == 1:
            params[0].update()
            return
        if not params:
            return
        table = []
        for p in params:
            st = p.opt_state
            st._advance_powers()
            o = st.opt
            table += (p.value._ptr, p.grad._ptr, st.m._ptr, st.v._ptr, p.value.size, o.lr, o.eps, o.beta1,
                      o.beta2, st.beta1t, st.beta2t)
        call("vkh_adam_multi", params[0].value._gpu._handle,
             struct.pack(ADAM_STEP_FORMAT * len(params), *table), len(params))
        for p in params:
            st = p.opt_state
            p.value._set_job([p.grad])
            st.m._set_job()
            st.v._set_job()
