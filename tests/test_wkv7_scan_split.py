"""The record scans' time split with saved states (head size 128): segments against one pass."""
import pytest
import torch

from conftest import rel_l2
from theseus import wkv7 as W
from theseus.synthetic import wkv7_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,B,T,H,cus", [(128, 1, 500, 2, 256), (128, 2, 333, 2, 24), (128, 1, 600, 8, 256)])
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
