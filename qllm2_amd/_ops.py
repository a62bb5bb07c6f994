"""Registration of the qpam:: operators with the torch dispatcher.

`op("qpam::name")` defines an operator from a Python function's annotations,
with `register_fake` and `register_autograd` as torch.library.custom_op has
them, so tracing, fake tensors, dispatch modes and functorch see one operator
as before: an argument left at its default reaches setup_context filled in, and
an output that is an input is an error.  Keyword-only arguments
are refused.  The difference is the autograd path: custom_op flattens every
argument and result through pytrees on each differentiable call (172 us for a
14-argument operator returning a list of tensors, against 33 us here; forward
and backward 315 against 110 us, one host core), which was most of a small
training step.  Here the Autograd kernel applies one torch.autograd.Function
that redispatches below autograd and keeps the saved tensors.  It needs a few
names of torch._C; where one is missing, op() is torch.library.custom_op.
"""

import sys
import threading

import torch

_LIB = torch.library.Library("qpam", "FRAGMENT")
_CALL = threading.local()  # the dispatch keys of the call that is entering its autograd function


def _kernel(name, fn):
    """fn as the operator's kernel.  It is kept out of torch.compile's tracing where it
    is called from a compiled program, and is as it is while nothing has loaded the
    compiler (which the wrapper would import on its first call).  No output may be one
    of the inputs: autograd and functionalization take an operator's outputs for tensors
    of their own.  (custom_op looks for shared storage, views included, which costs a
    small call 3 us of its 75; that no operator here returns a view of an input is tested.)"""
    traced_off = torch._disable_dynamo(fn)

    def kernel(*args):
        out = fn(*args) if "torch._dynamo" not in sys.modules else traced_off(*args)
        if not {*map(id, args)}.isdisjoint(map(id, out if isinstance(out, list) else (out,))):
            raise RuntimeError(f"{name}: an output is one of the inputs")
        return out

    return kernel


class Op:
    """One qpam:: operator, callable as the function it was made from."""

    def __init__(self, name, fn):
        ns, self._name = name.split("::")
        if ns != "qpam":
            raise ValueError(f"operator {name}: the namespace must be qpam")
        schema = torch.library.infer_schema(fn, mutates_args=())
        _LIB.define(self._name + schema, tags=(torch.Tag.pt2_compliant_tag,))
        self._op = getattr(torch.ops.qpam, self._name).default
        arguments = self._op._schema.arguments
        if any(a.kwarg_only for a in arguments):
            raise ValueError(f"operator {name}: keyword-only arguments are not supported")
        self._defaults = [a.default_value for a in arguments]  # read past the arguments a call passes
        _LIB.impl(self._name, _kernel(name, fn), "CompositeExplicitAutograd")
        self._list = schema.rstrip().endswith("[]")
        self.__doc__, self.__name__ = fn.__doc__, fn.__name__
        self._autograd(None, None)

    def __call__(self, *args, **kwargs):
        return self._op(*args, **kwargs)

    def register_fake(self, fn):
        torch.library.register_fake(f"qpam::{self._name}", fn, lib=_LIB)
        return fn

    def register_autograd(self, backward, *, setup_context):
        """backward(ctx, grads) -> one gradient (or None) per argument (a tuple; a lone
        gradient for one argument), grads a list for an operator that returns a
        list; setup_context(ctx, inputs, output), inputs every argument."""
        self._autograd(backward, setup_context)

    def _autograd(self, backward, setup_context):
        op, is_list, name, first = self._op, self._list, self._name, not hasattr(self, "_fn")
        defaults = self._defaults

        class Fn(torch.autograd.Function):
            @staticmethod
            def forward(ctx, *args):
                keyset = _CALL.keyset
                with torch._C._AutoDispatchBelowAutograd():
                    out = op.redispatch(keyset & torch._C._after_autograd_keyset, *args)
                if setup_context is not None:
                    setup_context(ctx, args, out)
                return tuple(out) if is_list else out

            @staticmethod
            def backward(ctx, *grads):
                if backward is None:
                    raise RuntimeError(f"qpam::{name} has no backward")
                return backward(ctx, list(grads) if is_list else grads[0])

        Fn.__name__ = Fn.__qualname__ = f"qpam_{name}"
        self._fn = Fn
        if first:
            def autograd_kernel(keyset, *args):
                if torch.is_grad_enabled() and torch._C._any_requires_grad(*args):
                    # the dispatcher drops trailing arguments equal to their defaults
                    if len(args) < len(defaults):
                        args = (*args, *defaults[len(args):])
                    _CALL.keyset = keyset  # beside the arguments, not one of them; read first thing in forward
                    out = self._fn.apply(*args)
                    return list(out) if is_list else out
                with torch._C._AutoDispatchBelowAutograd():
                    return op.redispatch(keyset & torch._C._after_autograd_keyset, *args)

            _LIB.impl(name, autograd_kernel, "Autograd", with_keyset=True)


_NAMES = ("_AutoDispatchBelowAutograd", "_after_autograd_keyset", "_any_requires_grad")


def op(name):
    """Decorator: the qpam:: operator made from an annotated function."""
    if all(hasattr(torch._C, n) for n in _NAMES) and hasattr(torch, "_disable_dynamo"):
        return lambda fn: Op(name, fn)
    return lambda fn: torch.library.custom_op(name, fn, mutates_args=())
