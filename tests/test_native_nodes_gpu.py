"""The C++ autograd nodes of the layers against their Python functions: same bits, same tensors saved, same refusals."""
import pytest
import torch

from savanna_amd import _lib, two_pass_chunked_gate_conv_gate
from savanna_amd.kernels.cgcg.src.kernel_utils import FwdKernelConfigRefactor
from savanna_amd.kernels.short_hyena import run_short_hyena
from savanna_amd.operators.hyena import CgcgConfig, HyenaMixer, HyenaMROperator

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not _lib.TORCH_OPS, reason="the torch extension is not loaded")]
DEV = "cuda:0"
CFG = FwdKernelConfigRefactor(CHUNK_SIZE=128, BLOCK_D=16, THREADBLOCK_SWIZZLE="row")


def _case(kind):
    """(callable, inputs) with the inputs requiring grad."""
    gen = torch.Generator(device=DEV).manual_seed(3)
    bs, L, g, dg = 2, 150, 4, 16
    r = lambda *s, t=torch.bfloat16: torch.randn(*s, generator=gen, device=DEV).to(t).requires_grad_()
    if kind in ("gated", "short", "strided"):
        xs = [r(bs, L, g, dg) if kind != "strided" else r(L, bs, g, dg) for _ in range(3)] + [r(g, 1, 7 if kind == "short" else 64)]
        view = (lambda t: t.transpose(0, 1)) if kind == "strided" else (lambda t: t)
        return lambda x, B, C, h: two_pass_chunked_gate_conv_gate(view(x), view(B), view(C), h, bs, L, g, dg, fwd_kernel_cfg=CFG), xs
    if kind == "time_major":
        return lambda q, k, v, w: run_short_hyena(q, k, v, w, autotune=True), [r(L, bs, g, dg) for _ in range(3)] + [r(g, 1, 7)]
    torch.manual_seed(0)
    op = HyenaMROperator(g * dg, g, 64, CgcgConfig(cgcg_dtype="float32" if kind == "module" else "bfloat16"), small_init=False,
                         device=DEV, fuse_filter=kind != "mixer_filter")
    if kind == "module":
        return lambda a, b, c, w: op(a, b, c), [r(bs, L, g, dg) for _ in range(3)] + [op.filter.h]
    mixer = HyenaMixer(op, 3, dtype=torch.bfloat16, device=DEV)
    return lambda f, *w: mixer(f), [r(bs, L, 3 * g * dg), *mixer.parameters()]


KINDS = ["gated", "short", "strided", "time_major", "module", "mixer", "mixer_filter"]


@pytest.mark.parametrize("kind", KINDS)
def test_same_bits_and_saved_tensors(kind, monkeypatch):
    f, xs = _case(kind)

    def step():
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append((t.shape, t.dtype)), t)[1], lambda t: t):
            y = f(*xs)
        dy = torch.ones_like(y)
        first = torch.autograd.grad(y, xs, dy, retain_graph=True)
        again = torch.autograd.grad(y, xs, dy)
        with pytest.raises(RuntimeError, match="second time"):
            torch.autograd.grad(y, xs, dy)
        assert all(torch.equal(a, b) for a, b in zip(first, again))
        with torch.no_grad():
            assert torch.equal(f(*xs), y)
        return [y.detach(), *first], packed

    native, saved = step()
    monkeypatch.setattr(_lib, "native_nodes", lambda t: False)
    python, saved_python = step()
    assert all(torch.equal(a, b) and a.stride() == b.stride() for a, b in zip(native, python))
    assert saved == saved_python


@pytest.mark.parametrize("kind", ["gated", "time_major", "mixer"])
def test_changed_inputs_are_noticed(kind):
    f, xs = _case(kind)
    leaf = xs[0]
    xs[0] = leaf * 1
    y = f(*xs)
    xs[0].mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


def test_transforms_and_dual_numbers_take_the_python_functions():
    f, xs = _case("gated")
    x = xs[0].detach()
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        with pytest.raises(NotImplementedError, match="jvp"):
            f(dual, *xs[1:])
    # (the C++ node would not refuse: vmap runs an operator without a batching rule sample by sample)
    with pytest.raises(RuntimeError, match="setup_context"):
        torch.func.vmap(lambda t: f(t, *(p.detach() for p in xs[1:])))(x[None])
    assert not torch.func.vmap(lambda t: t.new_full((), float(_lib.native_nodes(t))))(x[None]).any() and _lib.native_nodes(x)


def test_refusals_are_those_of_the_python_function():
    f, xs = _case("gated")
    x, B, C, h = (t.detach() for t in xs)
    bs, L, g, dg = x.shape
    call = lambda *t, **k: two_pass_chunked_gate_conv_gate(*t, bs, L, g, dg, **{"fwd_kernel_cfg": CFG, **k})
    for bad in ((x[:1], B, C, h), (x, B[:, :5], C, h), (x, B, C, h[:2]), (x, B.float(), C, h)):
        with pytest.raises(AssertionError):
            call(*bad)
    with pytest.raises(NotImplementedError):
        call(x, B, C, h, fwd_kernel_cfg=None, fwd_autotune=True, schedule="persistent")
    with pytest.raises(Exception, match="dtype"):
        call(x.double(), B.double(), C.double(), h.double())


def test_schemas_and_meta_results():
    from savanna_amd import _ops

    r = lambda *s, t=torch.bfloat16: torch.randn(*s, device=DEV).to(t)
    bs, L, g, dg = 1, 130, 2, 16
    x, w, decay, wf = r(bs, L, g, dg), r(g, 128, t=torch.float32), torch.rand(g, 128, device=DEV), r(3 * g * dg, 1, 3)
    args = {"gate_conv_gate": (x, x, x, r(g, 1, 33)), "short_hyena": (r(L, bs, g, dg),) * 3 + (r(g, 1, 7),),
            "gate_conv_gate_decay": (x, x, x, w, decay, 128, torch.bfloat16), "mixer_mr": (r(bs, L, g, dg, 3), wf, r(g, 1, 128)),
            "mixer_mr_decay": (r(bs, L, g, dg, 3), wf, w, decay, 128, torch.bfloat16)}
    assert set(args) == set(_ops.NODE_NAMES)
    for name, a in args.items():
        torch.library.opcheck(getattr(torch.ops.gcg, name), a, test_utils=("test_schema", "test_faketensor"))
