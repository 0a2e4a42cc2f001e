"""Registration of the ``molix`` ops with the dispatcher.

``op("molix::name")`` turns a function on GPU tensors into ``torch.ops.molix.name`` (schema from its
annotations, or given), with ``.register_fake`` and ``.register_autograd`` as
``torch.library.custom_op`` has them.  What differs is the path of one call: the GPU kernel and the
autograd kernel are registered directly, so a call passes through one Python function per dispatch key.
``custom_op`` also checks every result for aliasing with the arguments, at 16 us a call without and
42 us with a gradient (9 and 18 us here; forward and backward of a small op 114 against 60 us), which
is what bounds systems of a few thousand atoms.  The ops here return fresh tensors; one that writes
into an argument, or takes or returns a list of tensors (which an autograd function does not look
into), stays a ``custom_op``.
"""

from __future__ import annotations

import inspect
import re

import torch

_lib = torch.library.Library("molix", "FRAGMENT")
# Each op's own Library, kept across a reload of this module: defining an op again (importlib.reload,
# a notebook's autoreload) replaces it, as with ``custom_op``
_libs: dict[str, torch.library.Library] = globals().get("_libs", {})


def _needs_grad(args) -> bool:
    for a in args:
        if isinstance(a, torch.Tensor) and a.requires_grad:
            return True
    return False


class Op:
    """One op: callable, with its fake implementation and autograd formula registered later."""

    def __init__(self, qualname: str, fn, schema: str | None):
        ns, name = qualname.split("::")
        if ns != "molix":
            raise ValueError(f"{qualname}: the namespace is molix")
        schema = schema or torch.library.infer_schema(fn, mutates_args=())
        if re.search(r"Tensor\??\[", schema):
            raise TypeError(f"{qualname}{schema}: lists of tensors need torch.library.custom_op")
        if name in _libs:
            _libs.pop(name)._destroy()
        self._lib = _libs[name] = torch.library.Library("molix", "FRAGMENT")
        self._lib.define(name + schema, tags=(torch.Tag.pt2_compliant_tag,))
        self.qualname, self.__doc__, self.__name__ = qualname, fn.__doc__, fn.__name__
        self._op = getattr(torch.ops.molix, name).default
        # a call through the dispatcher leaves out trailing arguments that have their default value
        self._defaults = tuple(p.default for p in inspect.signature(fn).parameters.values())
        self._setup = self._backward = None
        self._function = self._make_function()
        self._lib.impl(name, fn, "CUDA")
        self._lib.impl(name, self._autograd, "Autograd")

    def __call__(self, *args, **kwargs):
        return self._op(*args, **kwargs)

    def register_fake(self, fn):
        torch.library.register_fake(self.qualname, fn, lib=self._lib)
        return fn

    def register_autograd(self, backward, *, setup_context=None) -> None:
        """``setup_context(ctx, inputs, output)`` and ``backward(ctx, *grads)`` as for
        ``torch.library.custom_op``: one gradient per argument of the schema."""
        self._backward, self._setup = backward, setup_context

    def _autograd(self, *args):
        args += self._defaults[len(args):]
        if torch.is_grad_enabled() and _needs_grad(args):
            return self._function.apply(*args)
        with torch._C._AutoDispatchBelowAutograd():
            return self._op(*args)

    def _make_function(self):
        op = self

        class Function(torch.autograd.Function):
            @staticmethod
            def forward(*args):
                with torch._C._AutoDispatchBelowAutograd():
                    return op._op(*args)

            @staticmethod
            def setup_context(ctx, inputs, output):
                if op._setup is not None:
                    op._setup(ctx, inputs, output)

            @staticmethod
            def backward(ctx, *grads):
                if op._backward is None:
                    raise RuntimeError(f"Trying to backward through {op.qualname} but no autograd formula was "
                                       "registered")
                return op._backward(ctx, *grads)

        Function.__name__ = Function.__qualname__ = op.qualname.replace("::", "_")
        return Function


def op(qualname: str, *, schema: str | None = None):
    """Decorator: registers the function as the op ``qualname`` on the GPU."""
    return lambda fn: Op(qualname, fn, schema)
