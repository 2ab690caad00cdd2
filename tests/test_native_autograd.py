"""theseus._native: the operator's autograd functions as native torch nodes against the Python
functions that they stand in for (the same kernels, so the same bits), their checks, and the
calls that stay with the Python functions."""
import warnings

import pytest
import torch

from theseus import gdn as G
from theseus import wkv7 as W
from theseus.synthetic import wkv7_inputs


def test_module_loads_here():
    assert W._native_module() is not None


def test_calls_that_stay_with_python():
    class Sub(torch.Tensor):
        pass

    x = torch.zeros(1, 2, 1, 4)
    assert W._native(x, torch.nn.Parameter(x)) is not None
    assert W._native(x, x.as_subclass(Sub)) is None
    seen = []
    torch.func.vmap(lambda t: (seen.append(W._native(t)), t)[1])(torch.zeros(2, 3))
    assert seen == [None]
    torch.jit.trace(lambda t: (seen.append(W._native(t)), t * 2)[1], torch.zeros(2), check_trace=False)
    with torch.autograd.forward_ad.dual_level():
        seen.append(W._native(x))
    assert seen == [None] * len(seen) and len(seen) >= 3
    assert W._native(x) is not None


def _case(B, T, H, N, dtype):
    inp = wkv7_inputs(B, T, H, N, seed=3, dtype=dtype, s0_std=.1, with_dsT=True)
    return [inp[n].cuda() for n in "rwkvab"] + [inp["s0"].cuda()], inp["dy"].cuda(), inp["dsT"].cuda()


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore::RuntimeWarning")
@pytest.mark.parametrize("N,dtype,T", [(64, torch.bfloat16, 40), (128, torch.bfloat16, 40), (64, torch.float32, 17),
                                       (40, torch.bfloat16, 5), (64, torch.bfloat16, 1)])
def test_same_bits_as_the_python_functions(N, dtype, T):
    xs, dy, dsT = _case(2, T, 3, N, dtype)
    # inputs as programs hold them: a strided view, a bf16 state, gradients wanted of some
    xs[2] = torch.stack([xs[2], xs[2]], -1)[..., 0]
    for state_dt in (torch.float32, torch.bfloat16):
        for outs in ((0,), (1,), (0, 1)):
            got = []
            for native in (False, True):
                a = [x.detach().clone(memory_format=torch.preserve_format) for x in xs]
                a[6] = a[6].to(state_dt)
                for i in (0, 1, 2, 3, 6):
                    a[i].requires_grad_()
                r = W._native_module().wkv7(*a) if native else W._WKV.apply(*a)
                torch.autograd.backward([r[i] for i in outs], [(dy, dsT)[i] for i in outs])
                got.append([t.detach() for t in r] + [t.grad for t in a])
            for p, q in zip(*got):
                assert (p is None) == (q is None)
                assert p is None or (torch.equal(p, q) and p.dtype == q.dtype)
    with torch.no_grad():
        a = [x.contiguous() for x in xs]
        y, end, _ = W.extension().forward(*a, False)
        yn, en = W.wkv7(*xs)
        assert torch.equal(y, yn) and torch.equal(end, en) and not yn.requires_grad


@pytest.mark.gpu
def test_gdn_same_bits():
    g = torch.Generator(device="cuda").manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    B, T, H, N = 1, 70, 2, 128
    xs = [rnd(B, T, H, N) * N ** -.5 for _ in range(3)] + [-rnd(B, T, H).exp(), rnd(B, T, H).sigmoid(), rnd(B, H, N, N)]
    grads = rnd(B, T, H, N), rnd(B, H, N, N)
    got = []
    for f in (G._GDN.apply, W._native_module().gdn):
        a = [x.clone().requires_grad_() for x in xs]
        r = f(*a)
        torch.autograd.backward(r, grads)
        got.append([t.detach() for t in r] + [t.grad for t in a])
    assert all(torch.equal(p, q) for p, q in zip(*got))


@pytest.mark.gpu
def test_checks_streams_hooks_and_family(monkeypatch):
    xs, dy, dsT = _case(1, 40, 2, 64, torch.bfloat16)
    with pytest.raises(RuntimeError, match="input mismatch"):
        W.wkv7(xs[0], xs[1].float(), *xs[2:])
    with pytest.raises(RuntimeError, match="invalid s0 shape"):
        W.wkv7(*xs[:6], xs[6][:, :1])
    with pytest.raises(RuntimeError, match="s0 must be contiguous CUDA FP32"):
        W.wkv7(*xs[:6], xs[6].cpu())
    with pytest.raises(RuntimeError, match="invalid T or head size"):
        W.wkv7(*[x[..., :1] for x in xs[:6]], xs[6])
    a = [x.clone().requires_grad_() for x in xs]
    ref = torch.autograd.grad(W.wkv7(*a)[0], a, dy)
    with pytest.warns(RuntimeWarning, match="float32 token tensors"):
        W.wkv7(*[x.float() for x in a[:6]], a[6])
    # saved tensors through hooks (activation offload), and a backward on another stream
    kept = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t) or t.cpu(), lambda t: t.cuda()):
        y, _ = W.wkv7(*a)
    assert len(kept) == 7
    for p, q in zip(torch.autograd.grad(y, a, dy), ref):
        assert torch.equal(p, q)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        y, _ = W.wkv7(*a)
        got = torch.autograd.grad(y, a, dy)
    torch.cuda.current_stream().wait_stream(s)
    assert all(torch.equal(p, q) for p, q in zip(got, ref))
    # the backward refuses the other family's saved states, strict mode the step-serial kernels
    y, _ = W.wkv7(*a)
    monkeypatch.setenv("THESEUS_WKV7_FAMILY", "seq")
    with pytest.raises(RuntimeError, match="other kernel family"):
        torch.autograd.grad(y, a, dy)
    monkeypatch.delenv("THESEUS_WKV7_FAMILY")
    monkeypatch.setenv("THESEUS_WKV7_STRICT", "1")
    with pytest.raises(RuntimeError, match="step-serial kernels"):
        W.wkv7(*[x.float() for x in a[:6]], a[6])


@pytest.mark.gpu
def test_traced_calls_run_the_kernels():
    """torch.jit.trace of calls with gradients: the traced function replays the operator."""
    xs, _, _ = _case(1, 40, 2, 64, torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    B, T, H, N = 1, 40, 2, 128
    gs = [rnd(B, T, H, N) * N ** -.5 for _ in range(3)] + [-rnd(B, T, H).exp(), rnd(B, T, H).sigmoid(), rnd(B, H, N, N)]

    def delta_rule(*a):
        return G.gated_delta_rule(*a, output_final_state=True, use_qk_l2norm_in_kernel=True)

    for f, args in ((lambda *a: W.wkv7(*a), xs), (delta_rule, gs)):
        args = tuple(a.requires_grad_() for a in args)
        traced = torch.jit.trace(f, args, check_trace=False)
        other = tuple((a.detach() * .5).requires_grad_() for a in args)
        for a in (args, other):
            assert all(torch.equal(p, q) for p, q in zip(traced(*a), f(*a)))


@pytest.mark.gpu
def test_forward_mode_is_refused_by_the_python_functions():
    xs, _, _ = _case(1, 40, 2, 64, torch.bfloat16)
    xs = [x.requires_grad_() for x in xs]
    with torch.autograd.forward_ad.dual_level():
        r = torch.autograd.forward_ad.make_dual(xs[0], torch.ones_like(xs[0]))
        with pytest.raises(NotImplementedError, match="jvp"):
            W.wkv7(r, *xs[1:])


@pytest.mark.gpu
def test_fallback_warning_names_the_caller(monkeypatch):
    """A float32 call warns once, at the line that calls the operator, with gradients and without;
    its backward does not warn again (strict mode still refuses there)."""
    xs, dy, _ = _case(1, 5, 2, 64, torch.float32)
    for grad in (True, False):
        a = [x.clone().requires_grad_(grad) for x in xs]
        with warnings.catch_warnings(record=True) as seen:
            warnings.simplefilter("always")
            y, _ = W.wkv7(*a)
        assert [w.filename for w in seen] == [__file__] and "step-serial" in str(seen[0].message)
        if grad:
            with warnings.catch_warnings():
                warnings.simplefilter("error")
                torch.autograd.grad(y, a, dy, retain_graph=True)
            monkeypatch.setenv("THESEUS_WKV7_STRICT", "1")
            with pytest.raises(RuntimeError, match="step-serial"):
                torch.autograd.grad(y, a, dy)
            monkeypatch.delenv("THESEUS_WKV7_STRICT")
