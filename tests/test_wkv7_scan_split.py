"""The record scans' time split with saved states (head size 128): segments against one pass."""
import pytest
import torch

from conftest import rel_l2
from theseus import wkv7 as W
from theseus.synthetic import wkv7_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,B,T,H,cus", [(128, 1, 500, 2, 256), (128, 2, 333, 2, 24), (128, 1, 600, 8, 256),
                                           # four segments of both row groups; one group per segment,
                                           # the forward alone (65 chunks) and both (97, 130)
                                           (128, 1, 1030, 2, 12), (128, 1, 1030, 2, 8), (128, 1, 1550, 2, 8),
                                           (128, 2, 2070, 3, 48)])
def test_saved_state_split_against_one_pass(N, B, T, H, cus, monkeypatch):
    """The same records scanned in segments and in one pass: float32 states to rounding."""
    inp = wkv7_inputs(B, T, H, N, seed=N + T, dtype=torch.bfloat16, s0_std=.1, with_dsT=True)
    xs, s0, dy, dsT = [inp[n].cuda() for n in "rwkvab"], inp["s0"].cuda(), inp["dy"].cuda(), inp["dsT"].cuda()
    ext, out = W.extension(), {}
    for c in (cus, B * H):
        monkeypatch.setenv("THESEUS_WKV7_CUS", str(c))
        f = ext.forward(*xs, s0, True)
        out[c] = [*f, *ext.backward(*xs, f[2], dy, dsT)]
    for a, b in zip(*out.values()):
        assert rel_l2(a, b) <= (1e-5 if a.dtype == torch.float32 else 3e-3)


# both sides of the rules' lines on 256 CUs
@pytest.mark.parametrize("saved,N,H,n,split", [
    (True, 128, 8, 15, False), (True, 128, 8, 16, True), (True, 128, 17, 19, False), (True, 128, 17, 20, True),
    (True, 128, 33, 47, False), (True, 128, 33, 48, True), (True, 128, 43, 63, False), (True, 128, 43, 64, True),
    (True, 128, 86, 100, False), (True, 64, 20, 28, False), (True, 64, 20, 29, True), (True, 64, 86, 40, False)] + [
    (False, *case) for case in [(128, 8, 19, False), (128, 8, 20, True), (128, 33, 47, False), (128, 33, 48, True),
                                         (128, 43, 47, False), (128, 43, 48, True), (128, 65, 100, False),
                                         (64, 16, 15, False), (64, 16, 16, True), (64, 17, 19, False), (64, 17, 20, True),
                                         (64, 80, 47, False), (64, 80, 48, True), (64, 129, 50, False)]])
def test_forward_split_where_it_pays(saved, N, H, n, split, monkeypatch):
    """The forward, with saved states or without, given its best workspace, against the same
    records in one pass (a workspace of the records alone): the same bits where the rule keeps
    one pass, equal to rounding where it splits."""
    monkeypatch.setenv("THESEUS_WKV7_CUS", "256")
    lib, T = W.extension().lib, 16 * n - 3
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    p = lambda t: t.data_ptr()  # noqa: E731
    s0, stream = .1 * rnd(1, H, N, N), torch.cuda.current_stream().cuda_stream
    calls = []
    q, k, v = (rnd(1, T, H, N).bfloat16() for _ in range(3))
    decay, beta = -.002 * rnd(1, T, H).exp(), rnd(1, T, H).sigmoid()  # (weak: a segment's start reaches its end)
    states = torch.empty((1, H, n + 1, N, N), device="cuda") if saved else None
    kept = (states,) if saved else ()
    gdn = lib.theseus_gdn_forward_train_ex if saved else lib.theseus_gdn_forward
    calls.append((lambda o, sT, ws, b: gdn(1, T, H, N, 0, 1, *map(p, (q, k, v, decay, beta, s0, o, sT, *kept, ws)), b, stream),
                  {64: 22784, 128: 43264}[N], lib.theseus_gdn_forward_best_workspace_size(1, T, H, N, saved)))
    if N == 128:
        kk = torch.nn.functional.normalize(rnd(1, T, H, N), dim=-1)
        xs = [q, (rnd(1, T, H, N) - 6).bfloat16(), k, v, -kk.bfloat16(), (kk * rnd(1, T, H, N).sigmoid()).bfloat16()]
        calls.append((lambda o, sT, ws, b: lib.theseus_wkv7_forward(1, T, H, N, 0, *map(p, (*xs, s0, o, sT)),
                                                                    p(states) if saved else None, p(ws), b, stream),
                      43520, lib.theseus_wkv7_forward_best_workspace_size(1, T, H, N, 0, saved)))
    for f, rec, best in calls:
        out = []
        for size in (H * n * rec, best):
            o, sT, ws = torch.empty_like(q), torch.empty_like(s0), torch.empty((size,), dtype=torch.uint8, device="cuda")
            assert f(o, sT, ws, size) == 0
            out.append((o, sT, *(x.clone() for x in kept)))
        same = all(torch.equal(a, b) for a, b in zip(*out))
        assert same == (not split)
        for a, b in zip(*out):
            assert rel_l2(a, b) <= (1e-5 if a.dtype == torch.float32 else 3e-3)
