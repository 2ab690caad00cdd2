"""Training with few heads at head size 64 on the chunk-record kernels (bf16, more than 28
chunks n a head, at most CUs / 4 heads, (3 CUs / 10 - B H) n > 760): against the float64
oracle, and against the chunked kernels where both take the call.
Bars as in test_wkv7_gpu.py (bf16 outputs one ULP, float32 states rel-L2 1e-4).
"""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import wkv7_oracle as O
from theseus import wkv7 as W
from theseus.synthetic import wkv7_inputs
from test_wkv7_gpu import NAMES, _check, _gpu_fwd_bwd, _oracle, _untile

pytestmark = pytest.mark.gpu


# 29 chunks and up: 5 .. 9 segments, uneven ones, partial last chunks; the smallest head
# count and the most that the rule admits at these lengths
@pytest.mark.parametrize("B,T,H,cus", [(1, 449, 1, 256), (1, 464, 2, 256), (2, 490, 3, 256), (1, 500, 4, 256),
                                       (3, 450, 2, 256), (1, 513, 5, 256), (1, 1021, 5, 256), (1, 464, 49, 256),
                                       (1, 1021, 6, 64), (2, 1021, 32, 256)])
def test_few_heads_against_oracle(B, T, H, cus, monkeypatch):
    monkeypatch.setenv("THESEUS_WKV7_CUS", str(cus))
    lib = W.extension().lib
    n, rec = -(-T // 16), 23552 - 768
    assert lib.theseus_wkv7_forward_best_workspace_size(B, T, H, 64, 0, 1) >= B * H * n * rec
    assert lib.theseus_wkv7_backward_workspace_size(B, T, H, 64, 0) >= B * H * n * 4 * 64 * 64
    inp = wkv7_inputs(B, T, H, 64, seed=T + H, dtype=torch.bfloat16, s0_std=.1, with_dsT=True)
    got = _gpu_fwd_bwd(inp, torch.bfloat16, inp["dsT"])
    for name, g, r in zip(NAMES, got, _oracle(inp, inp["dsT"])):
        _check(name, g, r, torch.bfloat16)
        if name in ("sT", "ds0"):
            assert rel_l2(g, r) <= 1e-4, name


def test_few_heads_rule_and_saved_states(monkeypatch):
    """Outside the rule (too many heads for the CUs, 28 chunks) the sizes are the chunked
    kernels'; inside it the saved states are in the same tiled order and either family's
    backward reads either forward's."""
    lib, ext = W.extension().lib, W.extension()
    monkeypatch.setenv("THESEUS_WKV7_CUS", "256")
    for B, T, H in [(1, 464, 50), (1, 512, 53), (1, 4096, 65), (1, 448, 2)]:
        assert lib.theseus_wkv7_backward_workspace_size(B, T, H, 64, 0) == 0
    inp = wkv7_inputs(1, 460, 3, 64, seed=5, dtype=torch.bfloat16, s0_std=.1, with_dsT=True)
    xs, s0, dy, dsT = [inp[n].cuda() for n in "rwkvab"], inp["s0"].cuda(), inp["dy"].cuda(), inp["dsT"].cuda()
    fwd, bwd = {}, {}
    for cus in ("256", "3"):  # records; chunked (3 heads on 3 CUs)
        monkeypatch.setenv("THESEUS_WKV7_CUS", cus)
        fwd[cus] = ext.forward(*xs, s0, True)
    for a, b in zip(fwd["256"], fwd["3"]):
        assert rel_l2(a, b) <= (1e-5 if a.dtype == torch.float32 else 3e-3)
    # the records in one pass (their bytes alone in the workspace): the same again
    rec = 3 * 29 * 22784
    y, sT, saved = (torch.empty_like(x) for x in fwd["256"])
    ws = torch.empty((rec,), dtype=torch.uint8, device="cuda")
    monkeypatch.setenv("THESEUS_WKV7_CUS", "256")
    p = lambda t: t.data_ptr()  # noqa: E731
    assert lib.theseus_wkv7_forward(1, 460, 3, 64, 0, *map(p, (*xs, s0, y, sT, saved, ws)), rec,
                                    torch.cuda.current_stream().cuda_stream) == 0
    for a, b in zip((y, sT, saved), fwd["256"]):
        assert rel_l2(a, b) <= (1e-5 if a.dtype == torch.float32 else 3e-3)
    saved = fwd["256"][2]
    assert torch.equal(_untile(saved[:, :, 0]), s0) and torch.equal(saved[:, :, -1], fwd["256"][1])
    for cus in ("256", "3"):
        monkeypatch.setenv("THESEUS_WKV7_CUS", cus)
        for other in ("256", "3"):
            bwd[cus, other] = ext.backward(*xs, fwd[other][2], dy, dsT)
    for key, grads in bwd.items():
        for name, a, b in zip(NAMES[2:], grads, bwd["3", "3"]):
            assert rel_l2(a, b) <= (1e-4 if name == "ds0" else 3e-3), (key, name)


@pytest.mark.parametrize("mode", ["wide", "max_decay", "no_decay"])
def test_few_heads_at_the_ends_of_the_decay_range(mode):
    inp = wkv7_inputs(1, 450, 3, 64, seed=8, dtype=torch.bfloat16, s0_std=.1, with_dsT=True)
    w = inp["w"].float()
    inp["w"] = {"wide": 8 * w, "max_decay": torch.full_like(w, 30.), "no_decay": torch.full_like(w, -30.)}[mode].to(
        torch.bfloat16).contiguous()
    got = _gpu_fwd_bwd(inp, torch.bfloat16, inp["dsT"])
    for name, g, r in zip(NAMES, got, _oracle(inp, inp["dsT"])):
        if mode == "no_decay":  # values in the thousands: one bf16 ULP of the neighbouring power of two and, from
            # 450 undamped steps of split-bf16 products (2^-17 each, 20 sigma), 2^-9 of the output's own size
            g = g.detach().double().cpu().numpy()
            assert rel_l2(g, r) <= 5e-3 and np.all(np.abs(g - r) <= 2e-2 + 2.0 ** -7 * np.abs(r) +
                                                   2.0 ** -9 * np.abs(r).mean()), name
        elif name == "dw" and mode == "max_decay":
            # dw = -e^{-1/2} s (1 - s) dlogd of a saturated sigmoid, s (1 - s) = 9e-14: in float32 1 - s is
            # zero or one rounding of s, 2^-24 of the gradient dlogd of the log decay
            s1s = np.exp(-30.) / (1 + np.exp(-30.)) ** 2
            dlogd = np.abs(r).max() / (np.exp(-.5) * s1s)
            assert dlogd > .1 and np.all(np.abs(g.detach().double().cpu().numpy() - r) <= 2.0 ** -24 * dlogd + 2.0 ** -8 * np.abs(r))
        else:
            _check(name, g, r, torch.bfloat16)


@pytest.mark.parametrize("N", [64, 128])
def test_backward_by_the_workspace_it_is_given(N, monkeypatch):
    """The backward takes what a call brings: nothing at N = 64 (the chunked kernels), the records
    and dL/dS alone (one pass), fewer segments than the most, all of them."""
    monkeypatch.setenv("THESEUS_WKV7_CUS", "256")
    B, T, H = 1, 600, 3
    lib, ext, n = W.extension().lib, W.extension(), 38
    inp = wkv7_inputs(B, T, H, N, seed=9, dtype=torch.bfloat16, s0_std=.1, with_dsT=True)
    xs, s0, dy, dsT = [inp[i].cuda() for i in "rwkvab"], inp["s0"].cuda(), inp["dy"].cuda(), inp["dsT"].cuda()
    saved = ext.forward(*xs, s0, True)[2]
    best = lib.theseus_wkv7_backward_workspace_size(B, T, H, N, 0)
    record = {64: 12544, 128: 25088}[N] + 4 * N * N + 6 * 1024
    least, state = B * H * n * record, B * H * N * N * 4
    assert best == least + 15 * state  # (9 segments)
    ref = ext.backward(*xs, saved, dy, dsT)
    p = lambda t: t.data_ptr()  # noqa: E731
    for size in ([0] if N == 64 else []) + [least, least + 5 * state, best]:
        grads = [torch.empty_like(x) for x in xs] + [torch.empty_like(s0)]
        ws = torch.empty((max(size, 1),), dtype=torch.uint8, device="cuda")
        assert lib.theseus_wkv7_backward(B, T, H, N, 0, *map(p, (*xs, saved, dy, dsT, *grads)), p(ws) if size else None,
                                         size, torch.cuda.current_stream().cuda_stream) == 0
        for name, a, b in zip(NAMES[2:], grads, ref):
            if size == best:
                assert torch.equal(a, b), name
            assert rel_l2(a, b) <= (1e-5 if name == "ds0" else 3e-3), (size, name)
    if N == 128:  # (nothing else reads its saved states)
        assert lib.theseus_wkv7_backward(B, T, H, N, 0, *map(p, (*xs, saved, dy, dsT, *grads)), p(ws), least - 1,
                                         torch.cuda.current_stream().cuda_stream) == 4
