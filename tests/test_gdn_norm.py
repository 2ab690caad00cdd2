"""The gated delta rule's training pair with q and k normalised in the kernels
(theseus_gdn_forward_train_ex / _backward_ex): against a float64 torch loop, at tails of the
16-step chunks, with rows that are zero or tiny beside the 1e-6 of the normalisation.

Bars: float32 I/O rel-L2 1e-4 (the bar of the training pair without the normalisation, which
adds one rsqrt and two dot products of 128 terms, below 1e-6); dg, whose terms cancel by e^g
and more at strong decays, at most 1.25 times the error of that pair on q and k normalised by
torch in float32.  bf16 I/O: one rounding of each output, 2^-8 of its size at most, so rel-L2
5e-3 (1.7e-3 if evenly spread).
"""
import pytest
import torch

from conftest import rel_l2
from theseus import gdn as G

pytestmark = pytest.mark.gpu


def _loop64(q, k, v, g, beta, s0):
    n = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k = n(q) / q.shape[-1] ** .5, n(k)
    S, out = s0, []  # [B,H,K,V]
    for t in range(q.shape[1]):
        S = S * torch.exp(g[:, t])[..., None, None]
        u = beta[:, t][..., None] * (v[:, t] - (k[:, t][..., None] * S).sum(-2))
        S = S + k[:, t][..., None] * u[..., None, :]
        out.append((q[:, t][..., None] * S).sum(-2))
    return torch.stack(out, 1), S


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,H", [(1, 1, 1), (2, 15, 2), (1, 16, 3), (1, 17, 2), (2, 70, 2), (1, 333, 2)])
def test_training_pair_with_normalisation(B, T, H, dtype):
    N = 128
    gen = torch.Generator().manual_seed(T + H)
    rnd = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    q, k, v = (rnd(B, T, H, N).to(dtype) for _ in range(3))
    if T > 1:
        q[0, 0], k[0, T - 1, 0] = 0, 1e-5  # (norms 0 and 1e-4 against sqrt(1e-6))
    xs = [q, k, v, -torch.exp(rnd(B, T, H)), torch.sigmoid(rnd(B, T, H)), .1 * rnd(B, H, N, N)]
    do, dsT = rnd(B, T, H, N).to(dtype), rnd(B, H, N, N)
    gpu = [x.cuda().requires_grad_() for x in xs]
    o, sT = G.chunk_gated_delta_rule(*gpu[:5], initial_state=gpu[5], output_final_state=True,
                                     use_qk_l2norm_in_kernel=True)
    assert o.dtype == dtype and sT.dtype == torch.float32
    torch.autograd.backward((o, sT), (do.cuda(), dsT.cuda()))
    ref = [x.double().requires_grad_() for x in xs]
    ro, rs = _loop64(*ref)
    torch.autograd.backward((ro, rs), (do.double(), dsT.double()))
    got = [o, sT] + [x.grad for x in gpu]
    want = [ro, rs] + [x.grad for x in ref]
    plain = [x.detach().float().requires_grad_() for x in gpu]  # normalised by torch outside
    po, ps = G.chunk_gated_delta_rule(G.l2norm(plain[0]), G.l2norm(plain[1]), *plain[2:5], initial_state=plain[5],
                                      output_final_state=True)
    torch.autograd.backward((po, ps), (do.cuda().float(), dsT.cuda()))
    for name, a, b in zip(["o", "sT", "dq", "dk", "dv", "dg", "dbeta", "ds0"], got, want):
        bar = 5e-3 if a.dtype == torch.bfloat16 else 1e-4
        if name == "dg":
            bar = max(bar, 1.25 * rel_l2(plain[3].grad, b))
        assert a.dtype == (dtype if name in ("o", "dq", "dk", "dv") else torch.float32)
        assert rel_l2(a, b) <= bar, (name, rel_l2(a, b))


@pytest.mark.parametrize("dtype,norm,changed", [(torch.bfloat16, True, (0, 1, 2)), (torch.bfloat16, False, (0, 1, 2)),
                                                (torch.float32, True, (0, 1)), (torch.float16, True, (0, 1, 2))])
def test_inputs_changed_in_place_after_the_call(dtype, norm, changed):
    """What the call computed from copies before it normalised inside the kernels may still be
    changed between the call and its backward; the gradients are of the values at the call."""
    g = torch.Generator(device="cuda").manual_seed(4)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    B, T, H, N = 1, 33, 2, 128
    leaves = [rnd(B, T, H, N).to(dtype).requires_grad_() for _ in range(3)]
    rest, do, grads = [-rnd(B, T, H).exp(), rnd(B, T, H).sigmoid()], rnd(B, T, H, N).to(dtype), []
    for change in (False, True):
        qkv = [x * 1 for x in leaves]
        o, _ = G.chunk_gated_delta_rule(*qkv, *rest, use_qk_l2norm_in_kernel=norm)
        for i in changed if change else ():
            qkv[i].mul_(2)
        grads.append(torch.autograd.grad(o, leaves, do))
    assert all(torch.equal(a, b) for a, b in zip(*grads))
