"""The step-serial kernels (float32 token tensors, head sizes other than 64 and 128, the
exp decay mode) at the edges of their padded head sizes (32, 64, 128), of the 16-step
segments, and of the backward's windows of segments, against the float64 oracle.

Bar for float32 I/O: rel-L2 <= 2e-6.  Every output is a sum of float32 products whose
longest chain of roundings is a tree over the head's keys or value rows (at most log2(128)
= 7 levels) after the state's own: a state element is rounded three times a step and
remembers about 1 / (1 - e^{-0.6 sigmoid}) < 8 steps, so some 30 roundings of 2^-24 = 6e-8
each, 1.8e-6 if they all fell the same way (measured: 1e-7 - 3e-7).
"""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from oracle import wkv7_oracle as O
from theseus import wkv7 as W
from theseus.synthetic import wkv7_inputs

pytestmark = pytest.mark.gpu
FP32_BAR = 2e-6
NAMES = ["y", "sT", "dr", "dw", "dk", "dv", "da", "db", "ds0"]


def _gpu(inp, flags=0):
    xs = [inp[n].cuda().requires_grad_() for n in "rwkvab"]
    s0 = inp["s0"].cuda().requires_grad_()
    y, sT = W.wkv7_ex(*xs, s0, flags=flags)
    torch.autograd.backward((y, sT), (inp["dy"].cuda(), inp["dsT"].cuda()))
    torch.cuda.synchronize()
    return [y.detach(), sT.detach()] + [x.grad for x in xs] + [s0.grad]


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
@pytest.mark.parametrize("T", [1, 15, 16, 17, 33])
@pytest.mark.parametrize("N", [2, 3, 31, 32, 33, 36, 63, 64, 65, 127, 128])
def test_edges_of_head_size_and_segments(N, T):
    inp = wkv7_inputs(2, T, 3, N, seed=100 * N + T, dtype=torch.float32, s0_std=.3, with_dsT=True)
    got = _gpu(inp)
    arr = [inp[n].double().numpy() for n in "rwkvab"]
    s0, dy, dsT = (inp[n].double().numpy() for n in ("s0", "dy", "dsT"))
    ref = [*O.forward_c(*arr, s0), *O.backward_c(*arr, s0, dy, dsT)]
    for name, g, r in zip(NAMES, got, ref):
        e = rel_l2(g, r)
        assert e <= FP32_BAR, (name, e)


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
@pytest.mark.parametrize("N,H", [(40, 3), (64, 3), (40, 300), (64, 300)])
def test_key_value_states_and_exp_decay(N, H):
    """[key][value] states and d = exp(w) (w <= 0), with few heads (256-lane workgroups) and
    many (1024 lanes): the same numbers as the transposed states, the oracle's as well."""
    inp = wkv7_inputs(1, 19, H, N, seed=N + H, dtype=torch.float32, s0_std=.3, with_dsT=True)
    inp["w"] = -inp["w"].exp()
    rows = _gpu(inp, W.DECAY_EXP)
    tr = dict(inp, s0=inp["s0"].transpose(-1, -2).contiguous(), dsT=inp["dsT"].transpose(-1, -2).contiguous())
    kv = _gpu(tr, W.DECAY_EXP | W.STATE_KEY_VALUE)
    for i, (a, b) in enumerate(zip(rows, kv)):
        assert torch.equal(a, b.transpose(-1, -2) if i in (1, 8) else b), NAMES[i]
    arr = [inp[n].double().numpy() for n in "rwkvab"]
    s0, dy, dsT = (inp[n].double().numpy() for n in ("s0", "dy", "dsT"))
    ref = [*O.forward_c(*arr, s0, mode="exp"), *O.backward_c(*arr, s0, dy, dsT, mode="exp")]
    for name, g, r in zip(NAMES, rows, ref):
        assert rel_l2(g, r) <= FP32_BAR, name


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
def test_backward_windows_equal_one_window():
    """512 heads of 128 keys over 33 segments keep 1.03 GiB of dL/dS: two windows.  Each half of the
    heads fits one window, has heads enough for workgroups of the same shape (256 and more run
    1024 lanes), and must give the same bits."""
    B, T, H, N = 4, 16 * 33, 128, 128
    ext = W.extension()
    assert ext.lib.theseus_wkv7_backward_workspace_size(B, T, H, N, 1) == 2 ** 30  # (32 of the 33 segments)
    assert ext.lib.theseus_wkv7_backward_workspace_size(B // 2, T, H, N, 1) == B // 2 * H * 33 * N * N * 4
    g = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    r, w, k, v = (rnd(B, T, H, N) for _ in range(4))
    kk = torch.nn.functional.normalize(rnd(B, T, H, N), dim=-1)
    xs = [r, w, k, v, -kk, kk * torch.sigmoid(rnd(B, T, H, N))]
    s0, dy, dsT = .1 * rnd(B, H, N, N), rnd(B, T, H, N), rnd(B, H, N, N)

    def run(b0, b1):
        part = [x[b0:b1].contiguous() for x in xs]
        _, _, saved = ext.forward(*part, s0[b0:b1].contiguous(), True)
        return ext.backward(*part, saved, dy[b0:b1].contiguous(), dsT[b0:b1].contiguous())

    whole, halves = run(0, 4), [run(0, 2), run(2, 4)]
    for name, a, *bs in zip(NAMES[2:], whole, *halves):
        assert torch.equal(a, torch.cat(bs)), name


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
def test_infinite_inputs_stay_in_their_columns():
    """A value row's infinity reaches that row's outputs alone, and a head size whose last
    wave has padded rows (zero times infinity there) gives the float64 oracle's pattern of
    finite values."""
    inp = wkv7_inputs(1, 5, 1, 30, seed=3, dtype=torch.float32, s0_std=.3, with_dsT=True)
    inp["r"][0, 4, 0, 7] = float("inf")
    got = _gpu(inp)
    arr = [inp[n].double().numpy() for n in "rwkvab"]
    s0, dy, dsT = (inp[n].double().numpy() for n in ("s0", "dy", "dsT"))
    with np.errstate(all="ignore"):
        ref = [*O.forward(*arr, s0), *O.backward(*arr, s0, dy, dsT)]
    for name, g, r in zip(NAMES, got, ref):
        assert np.array_equal(np.isfinite(g.double().cpu().numpy()), np.isfinite(r)), name


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
def test_more_heads_than_one_launch_takes():
    """16777296 heads at 256 lanes each are more lanes than a grid has (2^32 - 1): the same bits as
    from two calls of half the heads."""
    H, N, T, ext = 2 ** 23 + 40, 4, 2, W.extension()
    g = torch.Generator(device="cuda").manual_seed(6)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    xs, s0, dy, dsT = [rnd(2, T, H, N) for _ in range(6)], rnd(2, H, N, N), rnd(2, T, H, N), rnd(2, H, N, N)

    def run(b):
        y, sT, saved = ext.forward(*[x[b] for x in xs], s0[b], True)
        return y, sT, *ext.backward(*[x[b] for x in xs], saved, dy[b], dsT[b])

    whole, halves = run(slice(0, 2)), [run(slice(0, 1)), run(slice(1, 2))]
    for name, a, *bs in zip(NAMES, whole, *halves):
        assert all(torch.equal(a[i:i + 1], b) for i, b in enumerate(bs)), name


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
@pytest.mark.parametrize("T", [1, 3, 16, 17, 31])
@pytest.mark.parametrize("N", [32, 64, 128])
def test_infinities_in_the_last_segment(N, T):
    """The steps past the end of a sequence leave an infinite state (an infinite key at the last
    step) and an infinite dL/dsT as they are: the float64 oracle's pattern of finite values, and
    the finite ones at their usual bar."""
    ext = W.extension()
    inp = wkv7_inputs(1, T, 2, N, seed=3, dtype=torch.float32, s0_std=.3, with_dsT=True)
    inf = {n: x.clone() for n, x in inp.items() if torch.is_tensor(x)}
    inf["k"][0, T - 1, 0, 7] = float("inf")
    inf["dsT"][0, 0, 3, 5] = float("inf")

    def run(a, dsT):
        xs, s0, dy = [a[n] for n in "rwkvab"], a["s0"], inp["dy"]
        y, sT, saved = ext.forward(*[x.cuda() for x in (*xs, s0)], True)
        got = [y, sT, *ext.backward(*[x.cuda() for x in xs], saved, dy.cuda(), dsT.cuda())]
        arr = [x.double().numpy() for x in (*xs, s0)]
        with np.errstate(all="ignore"):
            ref = [*O.forward(*arr), *O.backward(*arr, dy.double().numpy(), dsT.double().numpy())]
        return [g.double().cpu().numpy() for g in got], ref

    for part, (got, ref) in ((slice(0, 2), run(inf, inp["dsT"])), (slice(2, 9), run(inp, inf["dsT"]))):
        for name, g, r in zip(NAMES[part], got[part], ref[part]):
            ok = np.isfinite(r)
            assert np.array_equal(np.isfinite(g), ok) and ok.any(), name
            assert rel_l2(g[ok], r[ok]) <= FP32_BAR, name
        assert not np.isfinite(ref[1 if part.start == 0 else 8]).all()
