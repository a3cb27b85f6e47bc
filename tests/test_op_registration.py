"""archbench_amd._op.gpu_op against torch.library.custom_op on a CPU function of the same body: gradients (also of some
inputs only), no gradient, saved-tensor hooks, dispatch modes, fake tensors, make_fx, vmap, forward mode, functorch's grad,
a missing autograd formula and a compiled call behave alike."""

from typing import Optional

import pytest
import torch
import torch.autograd.forward_ad as fw
from torch import Tensor
from torch._subclasses import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import TorchDispatchMode

from archbench_amd._op import gpu_op


def _make(kind):
    deco = (lambda n: gpu_op(f"archbench_test::{kind}_{n}")) if kind == "gpu_op" else (
        lambda n: torch.library.custom_op(f"archbench_test::{kind}_{n}", mutates_args=()))

    @deco("f")
    def f(x: Tensor, y: Tensor | None, c: float, n: int) -> tuple[Tensor, Tensor]:
        return (x * c if y is None else x * y * c), torch.full((n,), 7, dtype=torch.uint8)

    @deco("b")
    def b(x: Tensor, y: Tensor | None, g: Tensor, c: float) -> tuple[Tensor, Tensor]:
        return (g * c if y is None else g * y * c), g * x * c

    f.register_fake(lambda x, y, c, n: (torch.empty_like(x), x.new_empty(n, dtype=torch.uint8)))
    b.register_fake(lambda x, y, g, c: (torch.empty_like(x), torch.empty_like(x)))

    def setup(ctx, inputs, output):
        x, y, c, _ = inputs
        ctx.save_for_backward(x, y, output[1])
        ctx.c = c
        ctx.set_materialize_grads(False)

    def backward(ctx, g, gs):
        assert gs is None
        x, y, _ = ctx.saved_tensors
        dx, dy = b(x, y, g, ctx.c)
        return dx, (None if y is None else dy), None, None

    f.register_autograd(backward, setup_context=setup)
    return f, b


def _make_default(kind):
    deco = gpu_op if kind == "gpu_op" else lambda n: torch.library.custom_op(n, mutates_args=())

    @deco(f"archbench_test::{kind}_d")
    def d(x: Tensor, y: Tensor | None = None, c: float = 3.0, n: int = 2) -> Tensor:
        return x * c * n if y is None else x * y * c * n

    d.register_fake(lambda x, y=None, c=3.0, n=2: torch.empty_like(x))

    def setup(ctx, inputs, output):
        x, y, ctx.c, ctx.n = inputs
        ctx.save_for_backward(x, y)

    def backward(ctx, g):
        x, y = ctx.saved_tensors
        f = ctx.c * ctx.n
        return (g * f if y is None else g * y * f), (None if y is None else g * x * f), None, None

    d.register_autograd(backward, setup_context=setup)
    return d


DEFAULTS = {k: _make_default(k) for k in ("gpu_op", "custom_op")}
OPS = {k: _make(k) for k in ("gpu_op", "custom_op")}


class _Names(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func).replace("custom_op", "gpu_op"))
        return func(*args, **(kwargs or {}))


def _leaves(rx=True, ry=True):
    g = torch.Generator().manual_seed(1)
    return torch.randn(5, generator=g).requires_grad_(rx), torch.randn(5, generator=g).requires_grad_(ry)


def _grads(f, b, rx=True, ry=True):
    x, y = _leaves(rx, ry)
    o, s = f(x, y, 2.0, 3)
    o.sum().backward()
    return [o, s, x.grad, y.grad, o.requires_grad, s.requires_grad]


def _hooks(f, b):
    n = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (n.append("pack"), t)[1], lambda t: (n.append("unpack"), t)[1]):
        o, _ = f(*_leaves(), 2.0, 3)
    o.sum().backward()
    return sorted(n)


def _modes(f, b):
    with _Names() as m:
        f(*_leaves(), c=2.0, n=3)[0].sum().backward()
    return m.names


def _fake(f, b):
    with FakeTensorMode() as m:
        o, s = f(m.from_tensor(torch.zeros(5)), None, 2.0, 3)
    return [o.shape, s.shape, s.dtype]


def _dual(f, b, rx):
    with fw.dual_level():
        x = fw.make_dual(torch.ones(5).requires_grad_(rx), torch.ones(5))
        return [fw.unpack_dual(f(x, None, 2.0, 3)[0]).tangent]


def _double(f, b):
    x, y = _leaves()
    g, = torch.autograd.grad(f(x, y, 2.0, 3)[0].square().sum(), x, create_graph=True)
    g.sum().backward()


def _no_grad(f, b):
    with torch.no_grad():
        o, _ = f(*_leaves(), 2.0, 3)
    return [o, o.requires_grad]


CHECKS = {
    "grad": _grads, "grad of x": lambda f, b: _grads(f, b, True, False), "grad of y": lambda f, b: _grads(f, b, False, True),
    "no grad": _no_grad, "hooks": _hooks, "modes": _modes, "fake": _fake, "double": _double,
    "dual": lambda f, b: _dual(f, b, False), "dual grad": lambda f, b: _dual(f, b, True),
    "inference": lambda f, b: list(torch.inference_mode()(f)(torch.ones(5), None, 2.0, 3)),
    "make_fx": lambda f, b: [str(n.target).replace("custom_op", "gpu_op")
                             for n in make_fx(lambda x: f(x, None, 2.0, 3)[0])(torch.ones(5)).graph.nodes],
    "vmap": lambda f, b: [torch.vmap(lambda x: f(x, None, 2.0, 3)[0])(torch.ones(2, 5))],
    "func.grad": lambda f, b: [torch.func.grad(lambda x: f(x, None, 2.0, 3)[0].sum())(torch.ones(5))],
    "no formula": lambda f, b: b(*_leaves(), torch.ones(5), 2.0)[0].sum().backward(),
    "wrong arguments": lambda f, b: f(torch.ones(5)),
    "compile": lambda f, b: [torch.compile(lambda x: f(x, None, 2.0, 3)[0] * 2, fullgraph=True, backend="aot_eager")(
        torch.ones(5, requires_grad=True))],
}


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("check", CHECKS)
def test_gpu_op_behaves_like_custom_op(check):
    out = {}
    for kind, (f, b) in OPS.items():
        try:
            out[kind] = CHECKS[check](f, b)
        except Exception as e:  # noqa: BLE001  the refusals are compared as well
            out[kind] = type(e)
    got, ref = out["gpu_op"], out["custom_op"]
    if not isinstance(ref, list):
        assert got is ref
        return
    assert len(got) == len(ref)
    for a, r in zip(got, ref):
        assert torch.equal(a, r) if isinstance(r, Tensor) else a == r, (a, r)


@pytest.mark.parametrize("args,kw", [((), {}), (("y",), {}), ((None,), {"n": 2}), ((), {"c": 3.0}), ((), {"n": 5}),
                                     (("y", 4.0, 5), {}), ((None, 3.0), {"n": 7})])
def test_default_arguments(args, kw):
    """Arguments left at (or equal to) their defaults, in front of given ones or not, reach setup_context."""
    out = []
    for d in DEFAULTS.values():
        x, y = _leaves()
        r = d(x, *(y if a == "y" else a for a in args), **kw)
        r.sum().backward()
        out.append([r, x.grad] + [y.grad] * ("y" in args))
    for a, r in zip(*out):
        assert torch.equal(a, r)


def test_unsupported_signatures_are_refused():
    def kw_only(x: Tensor, *, c: float) -> Tensor:
        return x * c

    def tensor_list(xs: list[Tensor]) -> Tensor:
        return xs[0].clone()

    def optional_list(x: Tensor, ys: list[Optional[Tensor]]) -> Tensor:
        return x.clone()

    def returns_list(x: Tensor) -> list[Tensor]:
        return [x.clone()]

    for f in (kw_only, tensor_list, optional_list, returns_list):
        with pytest.raises(ValueError, match="custom_op"):
            gpu_op(f"archbench_test::{f.__name__}")(f)
