"""The fused TimeMix pieces of calls without gradients: the parameters in one launch, the decay
input in the kk kernel's launch, and the token shift at every number of tokens per thread,
against the separate launches (the same arithmetic, so the same bits) and the torch chain."""
import pytest
import torch

from theseus import fused
from theseus.timemix import TimeMix, _shift_lerp_ops

pytestmark = pytest.mark.gpu
bf = torch.bfloat16


@pytest.mark.parametrize("C", [64, 320, 5120])
def test_pack_params_is_the_conversions(C):
    g = torch.Generator(device="cuda").manual_seed(C)
    ps = [torch.randn(1, 1, C, generator=g, device="cuda").to(d) for d in (bf, torch.float32, torch.float16)]
    ps += [torch.randn(C // 64, 64, generator=g, device="cuda").to(bf), torch.randn(2 * C, generator=g, device="cuda")[::2]]
    out = fused.pack_params(ps, C)
    assert out.shape == (5, C) and out.dtype == torch.float32
    for row, p in zip(out, ps):
        assert torch.equal(row, p.float().reshape(C))


# below, at and above each line of the dispatch (512 workgroups of 256 threads at 2 and 8
# tokens per thread), odd token counts, a sequence start inside a thread's tokens
@pytest.mark.parametrize("B,T,C", [(1, 1, 64), (64, 1, 5120), (3, 5, 128), (2, 255, 5120), (1, 511, 5120),
                                   (1, 410, 5120), (2, 411, 2560), (3, 683, 5120), (1, 1639, 5120), (7, 235, 5120)])
def test_shift_lerp_forward_at_every_width(B, T, C):
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(B, T, C, generator=g, device="cuda").to(bf)
    shift = torch.randn(B, C, generator=g, device="cuda").to(bf)
    coefs = [torch.rand(1, 1, C, generator=g, device="cuda") for _ in range(6)]
    with torch.no_grad():
        got = fused.shift_lerp(x, shift, coefs)
        rows = fused.shift_lerp(x, shift, fused.pack_params(coefs, C))
        want = _shift_lerp_ops(x, shift, coefs)
    for a, b, c in zip(got, rows, want):
        # (torch rounds product and sum apart, 2^-23 of the mix's terms; the bf16 roundings of the
        # two are then equal or neighbours, 2^-7 apart)
        assert torch.equal(a, b)
        torch.testing.assert_close(a, c, rtol=2 ** -7, atol=1e-5)
        assert (a != c).float().mean() < 1e-3


@pytest.mark.parametrize("B,T,C", [(1, 1, 64), (3, 7, 320), (1, 4096, 128), (5, 821, 192)])
def test_decay_input_in_the_kk_launch(B, T, C):
    g = torch.Generator(device="cuda").manual_seed(T)
    k, za, zw = (torch.randn(B, T, C, generator=g, device="cuda").to(bf) for _ in range(3))
    a0, kk, ka, w0 = (torch.randn(1, 1, C, generator=g, device="cuda") for _ in range(4))
    with torch.no_grad():
        w, *got, _ = fused.kk_kmod_w(k, za, a0, kk, ka, zw, w0, 64, bf)
        *want, _ = fused.kk_kmod(k, za, a0, kk, ka, 64, bf)
        assert torch.equal(w.reshape(B, T, C), fused.add_param(zw, w0))
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("dtype", [bf, torch.float32])
def test_layer_without_gradients_equals_the_layer_with(dtype):
    """The no-grad layer (packed parameters, one kk launch) against the same call with autograd
    on, which converts each parameter: the same bits."""
    torch.manual_seed(0)
    m = TimeMix(256, 2, 6, backend="cuda")
    with torch.no_grad():
        for n, p in m.named_parameters():
            if n in ("w1", "a1", "g1", "output.weight"):
                p.normal_(0, .05)
    m = m.cuda().to(dtype)
    x = torch.randn(2, 100, 256, device="cuda", dtype=bf)
    with torch.autocast("cuda", dtype=bf):
        ref, st = m(x)
        with torch.no_grad():
            out, st2 = m(x)
    # (7 chunks: below the time split, which only calls without saved states take)
    assert torch.equal(out, ref) and not out.requires_grad
    assert torch.equal(st["wkv"], st2["wkv"])


def _shift_case(C=256):
    g = torch.Generator(device="cuda").manual_seed(2)
    x, shift = torch.randn(1, 40, C, generator=g, device="cuda").to(bf), torch.randn(1, C, generator=g, device="cuda").to(bf)
    return x, shift, torch.rand(6, C, generator=g, device="cuda")


@pytest.mark.parametrize("dtype", [torch.float32, bf, torch.float64])
def test_coefficient_tensor_keeps_its_gradients(dtype):
    """Six parameters or one [6, C] tensor of them, of any type: the same mixes and gradients."""
    x, shift, c = _shift_case()
    c = c.to(dtype).requires_grad_()
    rows = [r.detach().reshape(1, 1, -1).requires_grad_() for r in c]
    got, want = fused.shift_lerp(x, shift, c), fused.shift_lerp(x, shift, rows)
    dys = [torch.full_like(x, i + 1) for i in range(6)]
    gc, gr = torch.autograd.grad(got, c, dys)[0], torch.autograd.grad(want, rows, dys)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert torch.equal(gc, torch.cat(gr, 1)[0])
    with torch.no_grad():
        assert all(torch.equal(a, b) for a, b in zip(fused.shift_lerp(x, shift, c), want))


def test_shift_lerp_leaves_to_its_function_what_only_that_answers():
    x, shift, c = _shift_case()
    with torch.no_grad():
        traced = torch.jit.trace(lambda x, s, c: fused.shift_lerp(x, s, c), (x, shift, c), check_trace=False)
        assert all(torch.equal(a, b) for a, b in zip(traced(2 * x, shift, c), fused.shift_lerp(2 * x, shift, c)))
    with torch.autograd.forward_ad.dual_level(), pytest.raises(NotImplementedError, match="jvp"):
        fused.shift_lerp(torch.autograd.forward_ad.make_dual(x, x), shift, c)
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.vmap(lambda x, s: fused.shift_lerp(x, s, c))(x[None], shift[None])


@pytest.mark.parametrize("dtype", [bf, torch.float32])
def test_layer_refuses_a_tangent(dtype):
    m = TimeMix(256, 2, 6, backend="cuda").cuda().to(dtype).requires_grad_(False)
    x = torch.randn(1, 40, 256, device="cuda", dtype=bf)
    with torch.autocast("cuda", dtype=bf), torch.autograd.forward_ad.dual_level():
        with pytest.raises(NotImplementedError, match="jvp"):
            m(torch.autograd.forward_ad.make_dual(x, x))


@pytest.mark.parametrize("dtype", [bf, torch.float32])
@pytest.mark.parametrize("name", ["w0", "a0", "x_r", "k_k"])
def test_gradient_of_a_tensor_in_a_parameter_s_place(name, dtype):
    """A layer whose parameters need no gradient, one of them replaced by a tensor that does (a
    generated one): the gradient that the parameter itself would get."""
    torch.manual_seed(0)
    m = TimeMix(256, 2, 6, backend="cuda")
    with torch.no_grad():
        for n, p in m.named_parameters():
            if n in ("w1", "a1", "g1", "output.weight"):
                p.normal_(0, .05)
    m = m.cuda().to(dtype)
    x = torch.randn(2, 100, 256, device="cuda", dtype=bf)  # (200 rows: past the few-row products)

    def grad(of):
        with torch.autocast("cuda", dtype=bf):
            out, _ = m(x)
        return torch.autograd.grad(out, of, torch.ones_like(out))[0]

    want = grad(getattr(m, name))
    t = getattr(m, name).detach().clone().requires_grad_()
    delattr(m.requires_grad_(False), name)
    setattr(m, name, t)
    assert torch.equal(grad(t), want) and want.abs().max() > 0
