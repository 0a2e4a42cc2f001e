"""molnex_amd._ops: what the registration of an op gives its callers (on the CPU, with a stand-in kernel),
as torch.library.custom_op gives it."""

import os
import subprocess
import sys

import pytest
import torch

from molnex_amd import _ops


def _scaled(x: torch.Tensor, y: torch.Tensor, k: int = 2, z: torch.Tensor | None = None) -> tuple[torch.Tensor, torch.Tensor]:
    return x * y * k, torch.arange(x.shape[0])


def _plain(g: torch.Tensor, y: torch.Tensor, k: int) -> torch.Tensor:
    return g * y * k


scaled = _ops.op("molix::_test_scaled")(_scaled)
plain = _ops.op("molix::_test_plain")(_plain)
_ops._lib.impl("_test_scaled", _scaled, "CPU")
_ops._lib.impl("_test_plain", _plain, "CPU")
scaled.register_fake(lambda x, y, k=2, z=None: (torch.empty_like(x), x.new_empty(x.shape[0], dtype=torch.int64)))
plain.register_fake(lambda g, y, k: torch.empty_like(g))


def _setup(ctx, inputs, output):
    assert len(inputs) == 4  # defaults filled in
    ctx.save_for_backward(inputs[1])
    ctx.k = inputs[2]


scaled.register_autograd(lambda ctx, g, _: (plain(g, ctx.saved_tensors[0], ctx.k), None, None, None), setup_context=_setup)
X, Y = torch.tensor([1.0, 2.0, 3.0]), torch.tensor([4.0, 5.0, 6.0])


def test_calls_defaults_and_gradients():
    x = X.clone().requires_grad_(True)
    for out, k in ((torch.ops.molix._test_scaled(x, Y), 2), (torch.ops.molix._test_scaled(x, y=Y, k=5), 5), (scaled(x, Y, 3), 3)):
        assert torch.equal(out[0], X * Y * k) and not out[1].requires_grad
        assert torch.equal(torch.autograd.grad(out[0].sum(), x)[0], Y * k)
    with torch.no_grad():
        assert not scaled(x, Y)[0].requires_grad
    with torch.inference_mode():
        assert scaled(x, Y)[0].is_inference()
    assert not scaled(X, Y)[0].requires_grad


def test_backward_without_a_formula_raises():
    x = X.clone().requires_grad_(True)
    with pytest.raises(RuntimeError, match="_test_plain"):
        torch.autograd.grad(plain(x, Y, 2).sum(), x)
    y = Y.clone().requires_grad_(True)
    (g,) = torch.autograd.grad(scaled(X.clone().requires_grad_(True), y)[0].sum(), y, create_graph=True, allow_unused=True)
    assert g is None  # the formula gives y none
    x = X.clone().requires_grad_(True)
    (g,) = torch.autograd.grad(scaled(x, y)[0].sum(), x, create_graph=True)
    with pytest.raises(RuntimeError, match="_test_plain"):  # the second order was not given
        torch.autograd.grad(g.sum(), y)


def test_hooks_vmap_tracing_and_opcheck():
    x = X.clone().requires_grad_(True)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t, lambda t: t):
        out = scaled(x, Y)[0]
    assert len(packed) == 1 and torch.equal(torch.autograd.grad(out.sum(), x)[0], 2 * Y)
    assert torch.equal(torch.func.vmap(lambda a: scaled(a, Y)[0])(torch.stack([X, 2 * X])), torch.stack([X, 2 * X]) * Y * 2)
    f = torch.compile(lambda a: scaled(a, Y)[0].sin(), backend="aot_eager", fullgraph=True)
    assert torch.allclose(torch.autograd.grad(f(x).sum(), x)[0], torch.cos(2 * X * Y) * 2 * Y)
    torch.library.opcheck(torch.ops.molix._test_scaled.default, (x, Y, 3))


def test_lists_of_tensors_are_left_to_custom_op():
    """An autograd function does not look into lists: such an op's gradients would be lost in silence."""

    def takes(y: torch.Tensor, s: list[torch.Tensor]) -> torch.Tensor:
        return y * s[0]

    def gives(y: torch.Tensor) -> list[torch.Tensor]:
        return [y + 1]

    for fn in (takes, gives):
        with pytest.raises(TypeError, match="custom_op"):
            _ops.op(f"molix::_test_{fn.__name__}")(fn)
    with pytest.raises(TypeError, match="custom_op"):
        _ops.op("molix::_test_optional", schema="(Tensor y, Tensor?[] s) -> Tensor")(takes)
    import molnex_amd.kernels as K

    assert not any("Tensor[" in str(op._schema) or "Tensor?[" in str(op._schema)
                   for op in (v._op for v in vars(K).values() if isinstance(v, _ops.Op)))


def test_an_op_defined_again_replaces_the_first():
    """A module of ops can be reloaded (a notebook's autoreload)."""
    def first(x: torch.Tensor) -> torch.Tensor:
        return x + 1

    def second(x: torch.Tensor, k: int) -> torch.Tensor:
        return x + k

    for fn, args, want in ((first, (), 1), (second, (5,), 5)):
        op = _ops.op("molix::_test_again")(fn)
        op._lib.impl("_test_again", fn, "CPU")
        op.register_fake(lambda x, *a: torch.empty_like(x))
        op.register_autograd(lambda ctx, g, n=len(args): (g, None)[:1 + n])
        x = X.clone().requires_grad_(True)
        out = torch.ops.molix._test_again(x, *args)
        assert torch.equal(out, X + want) and torch.equal(torch.autograd.grad(out.sum(), x)[0], torch.ones(3))
        f = torch.compile(lambda a, rest=args: torch.ops.molix._test_again(a, *rest).sin(), backend="aot_eager", fullgraph=True)
        assert torch.allclose(f(x), torch.sin(X + want))


def test_the_kernels_module_can_be_reloaded():
    code = ("import importlib, torch, molnex_amd._ops as O, molnex_amd.kernels as K\n"
            "old = K.tall_tn\n"
            "for m in (K, O, K):\n"
            "    importlib.reload(m)\n"
            "assert K.tall_tn is not old and torch.ops.molix.tall_tn.default is K.tall_tn._op\n")
    subprocess.run([sys.executable, "-c", code], check=True, timeout=240, cwd=os.path.dirname(os.path.dirname(_ops.__file__)))
