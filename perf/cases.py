"""The calls this framework is measured by: what a training run, a prefill, a serving loop
and a conversion from a gated-delta-rule teacher have it do, through its public entry points.

Every case is a dict of plain values with a "kind":

* wkv7_train    -- the recurrence under autograd (theseus.wkv7.wkv7): y, the end state and the
                   gradients of r, w, k, v, a, b and the initial state.
* wkv7_infer    -- the same operator without gradients (a prefill chunk with a carried state).
* wkv7_decode   -- one token per lane without gradients (the serving step through the operator).
* gdn_infer     -- the gated delta rule of the teacher's layers, no gradients, state out.
* gdn_train     -- the same with gradients of q, k, v, g and beta.
* timemix_train -- a whole TimeMix layer forward and backward under bf16 autocast over float32
                   parameters: output, end state, gradients of x and of all 23 parameters.
* timemix_infer -- the layer with bf16 weights over a prompt, no gradients.
* timemix_step  -- the layer with bf16 weights on one token per lane in a serving loop that owns
                   its parameter store.
* adamw         -- the optimizer step after backward over one layer's parameters.

The value distributions are those of theseus.synthetic (r, w, k, v ~ N(0,1), a = -kk,
b = kk * sigmoid(N(0,1)), s0 ~ N(0, 0.1)), drawn on the GPU from the seed.
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "rwkv-theseus_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DECAY_SCALE = math.exp(-0.5)
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # the training shape of a 5120-wide layer's recurrence: 4 lanes of 2048 tokens
        dict(name="train_4x2048", kind="wkv7_train", B=4, T=2048, H=80, N=64, dtype="bf16"),
        # one lane of a 2560-wide layer, a length that is no multiple of anything
        dict(name="train_1x1021", kind="wkv7_train", B=1, T=1021, H=40, N=64, dtype="bf16"),
        # the smallest training call: float32, two heads, 64 tokens
        dict(name="train_fp32_small", kind="wkv7_train", B=1, T=64, H=2, N=64, dtype="fp32"),
        # the training shape at head size 128 (a 4096-wide layer)
        dict(name="train_n128", kind="wkv7_train", B=4, T=2048, H=32, N=128, dtype="bf16"),
        # one prefill chunk of 512 tokens, the state carried from chunk to chunk
        dict(name="prefill_512", kind="wkv7_infer", B=1, T=512, H=80, N=64, dtype="bf16"),
        # the serving step of 64 lanes through the operator
        dict(name="decode_64", kind="wkv7_decode", B=64, T=1, H=80, N=64, dtype="bf16"),
        # the teacher's gated delta rule over 2048 tokens, without and with gradients
        dict(name="gdn_infer", kind="gdn_infer", B=1, T=2048, H=32, N=128, dtype="bf16"),
        dict(name="gdn_train", kind="gdn_train", B=1, T=2048, H=32, N=128, dtype="bf16"),
        # one layer's training step at the full width: the largest work
        dict(name="layer_train", kind="timemix_train", B=2, T=4096, H=80, N=64, dtype="bf16"),
        # a ragged prompt through a 2048-wide layer
        dict(name="layer_prompt", kind="timemix_infer", B=1, T=777, H=32, N=64, dtype="bf16"),
        # the layer's serving step for 64 lanes
        dict(name="layer_step", kind="timemix_step", B=64, T=1, H=80, N=64, dtype="bf16"),
        # the optimizer step over the full-width layer's 112 M parameters
        dict(name="adamw_layer", kind="adamw", B=1, T=1, H=80, N=64, dtype="fp32"),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["wkv7_train", "wkv7_train", "wkv7_train_fp32", "wkv7_train_n128", "wkv7_infer", "wkv7_decode",
                       "gdn_infer", "gdn_train", "timemix_train", "timemix_infer", "timemix_step", "adamw"])
    B, T, H, N, dtype = 1, 1, 1, 64, "bf16"
    if kind == "wkv7_train":
        B, T, H = rng.randint(1, 4), _log(rng, 64, 2048), _log(rng, 8, 80)
    elif kind == "wkv7_train_fp32":
        kind, dtype = "wkv7_train", "fp32"
        B, T, H, N = rng.randint(1, 2), _log(rng, 16, 256), _log(rng, 2, 16), rng.choice([32, 64])
    elif kind == "wkv7_train_n128":
        kind, N = "wkv7_train", 128
        B, T, H = rng.randint(1, 4), _log(rng, 64, 2048), _log(rng, 4, 32)
    elif kind == "wkv7_infer":
        B, T, H = rng.randint(1, 4), _log(rng, 16, 2048), _log(rng, 8, 80)
    elif kind == "wkv7_decode":
        B, H = _log(rng, 1, 64), _log(rng, 8, 80)
    elif kind == "gdn_infer":
        B, T, H, N = rng.randint(1, 2), _log(rng, 64, 2048), _log(rng, 8, 32), rng.choice([64, 128, 128])
    elif kind == "gdn_train":
        B, T, H, N = rng.randint(1, 2), _log(rng, 64, 2048), _log(rng, 8, 32), 128
    elif kind == "timemix_train":
        B, T, H = rng.randint(1, 2), _log(rng, 128, 4096), rng.choice([12, 16, 32, 40, 64, 80])
    elif kind == "timemix_infer":
        B, T, H = rng.randint(1, 2), _log(rng, 16, 2048), rng.choice([12, 16, 32, 40, 64, 80])
    elif kind == "timemix_step":
        B, H = _log(rng, 1, 64), rng.choice([12, 16, 32, 40, 64, 80])
    elif kind == "adamw":
        H, dtype = rng.choice([12, 16, 32, 40, 64, 80]), "fp32"
    return dict(kind=kind, B=B, T=T, H=H, N=N, dtype=dtype)


# ---------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _wkv7_inputs(c, seed):
    """r, w, k, v, a, b in the case's type, the initial state and the output gradient."""
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    B, T, H, N = c["B"], c["T"], c["H"], c["N"]
    r, w, k, v = (_randn(g, B, T, H, N) for _ in range(4))
    kk = F.normalize(_randn(g, B, T, H, N), dim=-1, eps=1e-12)
    b = kk * torch.sigmoid(_randn(g, B, T, H, N))
    xs = [x.to(dt) for x in (r, w, k, v, -kk, b)]
    return xs, .1 * _randn(g, B, H, N, N), _randn(g, B, T, H, N).to(dt)


def _gdn_inputs(c, seed):
    """q, k, v, the log decay g, beta, the initial state and the output gradient."""
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    B, T, H, N = c["B"], c["T"], c["H"], c["N"]
    q, k, v = (_randn(g, B, T, H, N).to(dt) for _ in range(3))
    gg = -torch.exp(_randn(g, B, T, H))
    beta = torch.sigmoid(_randn(g, B, T, H))
    return q, k, v, gg, beta, .1 * _randn(g, B, H, N, N), _randn(g, B, T, H, N).to(dt)


def _ranks(C):
    return max(32, round(2.5 * math.sqrt(C) / 32) * 32), max(32, round(5 * math.sqrt(C) / 32) * 32)


def _layer_shapes(C, H, N):
    """A TimeMix layer's 23 parameters."""
    rank, grank = _ranks(C)
    s = {"x_" + n: (1, 1, C) for n in "rwkvag"}
    s.update(w1=(C, rank), w2=(rank, C), a1=(C, rank), a2=(rank, C), w0=(1, 1, C), a0=(1, 1, C), g1=(C, grank),
             g2=(grank, C), k_k=(1, 1, C), k_a=(1, 1, C), r_k=(H, N))
    s.update({n + ".weight": (C, C) for n in ("receptance", "key", "value", "output")})
    s.update({"ln_x.weight": (C,), "ln_x.bias": (C,)})
    return s


def _layer_params(c, g):
    """Parameters of a layer in training: projections and LoRAs N(0, 0.02), the vectors
    spread over the range that training moves them in."""
    C, H, N = c["H"] * c["N"], c["H"], c["N"]
    out = {}
    for n, s in _layer_shapes(C, H, N).items():
        z = torch.randn(*s, generator=g, device="cuda")
        if n.startswith("x_"):
            out[n] = torch.sigmoid(z)
        elif n == "w0":
            out[n] = z * 2 - 1
        elif n == "a0":
            out[n] = z * .3
        elif n == "k_k":
            out[n] = .7 + .1 * z
        elif n == "k_a":
            out[n] = 1 + .1 * z
        elif n == "ln_x.weight":
            out[n] = .6 + .05 * z
        else:
            out[n] = .02 * z
    return out


def _layer(c, params, dtype):
    """A TimeMix module holding ``params``, as a program with a checkpoint builds it: on the
    meta device, since the constructor's own initialisation is thrown away."""
    from theseus.timemix import TimeMix
    with torch.device("meta"):
        m = TimeMix(c["H"] * c["N"], 3, 8, head_size=c["N"], backend="cuda")
    m.load_state_dict({n: p.to(dtype) for n, p in params.items()}, assign=True)
    return m


def _layer_inputs(c, g):
    B, T, H, N = c["B"], c["T"], c["H"], c["N"]
    C, bf = H * N, torch.bfloat16
    x = _randn(g, B, T, C).to(bf)
    st = {"shift": _randn(g, B, C).to(bf), "wkv": .1 * _randn(g, B, H, N, N)}
    return x, st


GRAD_SCALE, CLIP = .5, 1.0
LR, WEIGHT_DECAY, BETAS, EPS = 1e-3, .01, (.9, .95), 1e-8


def _adamw_inputs(c, seed):
    """One layer's float32 parameters, gradients and moments (as after some hundred steps)."""
    g = _gen(seed)
    out = []
    for n, s in _layer_shapes(c["H"] * c["N"], c["H"], c["N"]).items():
        p, gr, m = .02 * _randn(g, *s), .01 * _randn(g, *s), .003 * _randn(g, *s)
        v = (.003 * _randn(g, *s)).square() + 1e-6
        out.append((n, p, gr, m, v))
    return out


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("wkv7_train", "wkv7_infer", "wkv7_decode"):
        xs, s0, dy = _wkv7_inputs(c, seed)
        if kind == "wkv7_train":
            xs, s0 = [x.requires_grad_() for x in xs], s0.requires_grad_()
        return dict(kind=kind, xs=xs, s0=s0, dy=dy)
    if kind in ("gdn_infer", "gdn_train"):
        q, k, v, g, beta, s0, do = _gdn_inputs(c, seed)
        xs = [q, k, v, g, beta]
        if kind == "gdn_train":
            xs = [x.requires_grad_() for x in xs]
        return dict(kind=kind, xs=xs, s0=s0, dy=do)
    if kind == "adamw":
        from theseus.optim import FusedAdamW
        ps, flat, matrices = [], [], []
        moments = {}
        for n, p, gr, m, v in _adamw_inputs(c, seed):
            p = torch.nn.Parameter(p)
            p.grad = gr
            ps.append(p)
            (matrices if p.dim() == 2 else flat).append(p)
            moments[p] = {"step": torch.tensor(100.0), "exp_avg": m, "exp_avg_sq": v}
        opt = FusedAdamW([dict(params=matrices, weight_decay=WEIGHT_DECAY), dict(params=flat, weight_decay=0.0)],
                         lr=LR, betas=BETAS, eps=EPS)
        for p, s in moments.items():
            opt.state[p] = s
        return dict(kind=kind, opt=opt, ps=ps)
    g = _gen(seed)
    params = _layer_params(c, g)
    x, st = _layer_inputs(c, g)
    if kind == "timemix_train":
        m = _layer(c, params, torch.float32)
        gy = _randn(g, *x.shape).to(x.dtype)
        leaves = [x.requires_grad_()] + [p.requires_grad_() for p in m.parameters()]
        return dict(kind=kind, m=m, x=x, st=st, gy=gy, leaves=leaves)
    m = _layer(c, params, torch.bfloat16).eval().requires_grad_(False)
    return dict(kind=kind, m=m, x=x, st=st, store={})


# ---------------------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "wkv7_train":
        from theseus.wkv7 import wkv7
        y, end = wkv7(*state["xs"], state["s0"])
        grads = torch.autograd.grad(y, state["xs"] + [state["s0"]], state["dy"])
        return [y.detach(), end.detach(), *grads]
    if kind in ("wkv7_infer", "wkv7_decode"):
        from theseus.wkv7 import wkv7
        with torch.no_grad():
            return list(wkv7(*state["xs"], state["s0"]))
    if kind == "gdn_infer":
        from theseus.gdn import chunk_gated_delta_rule
        with torch.no_grad():
            return list(chunk_gated_delta_rule(*state["xs"], initial_state=state["s0"], output_final_state=True,
                                               use_qk_l2norm_in_kernel=True))
    if kind == "gdn_train":
        from theseus.gdn import chunk_gated_delta_rule
        o, _ = chunk_gated_delta_rule(*state["xs"], use_qk_l2norm_in_kernel=True)
        return [o.detach(), *torch.autograd.grad(o, state["xs"], state["dy"])]
    if kind == "timemix_train":
        with torch.autocast("cuda", dtype=torch.bfloat16):
            out, end = state["m"](state["x"], state["st"])
        grads = torch.autograd.grad(out, state["leaves"], state["gy"])
        return [out.detach(), end["wkv"].detach(), *grads]
    if kind == "timemix_infer":
        with torch.no_grad():
            out, end = state["m"](state["x"], state["st"])
        return [out, end["wkv"]]
    if kind == "timemix_step":
        from theseus import fused
        with torch.no_grad(), fused.param_cache(state["store"]):
            out, end = state["m"](state["x"], state["st"])
        return [out, end["wkv"]]
    if kind == "adamw":
        norm = state["opt"].step_after_backward(grad_scale=GRAD_SCALE, max_norm=CLIP)
        return [norm, *[p.detach() for p in state["ps"]]]
    raise ValueError(kind)


# ---------------------------------------------------------------------------- what a pass needs
def work(case):
    c, kind = case, case["kind"]
    B, T, H, N = c["B"], c["T"], c["H"], c["N"]
    C, e = H * N, 2 if c["dtype"] == "bf16" else 4
    tok, state = B * T * C, B * H * N * N * 4
    # a step of the recurrence on an N x N state: S a, two rank-one updates, S r (2 N^2 each);
    # its adjoint: q, dr, dw, dk, dv, da, db and the two updates of dL/dS
    rec_f, rec_b = 8 * B * T * H * N * N, 18 * B * T * H * N * N
    if kind == "wkv7_train":  # six inputs and dy in, y and six gradients out; s0 in, end and ds0 out
        return {"bytes": 14 * tok * e + 3 * state, "flops": rec_f + rec_b}
    if kind in ("wkv7_infer", "wkv7_decode"):
        return {"bytes": 7 * tok * e + 2 * state, "flops": rec_f}
    if kind == "gdn_infer":
        return {"bytes": 4 * tok * e + 8 * B * T * H + 2 * state, "flops": rec_f}
    if kind == "gdn_train":  # q, k, v, do in, o, dq, dk, dv out; g, beta in, their gradients out
        return {"bytes": 8 * tok * e + 16 * B * T * H, "flops": rec_f + rec_b}
    numel = sum(math.prod(s) for s in _layer_shapes(C, H, N).values())
    mats = sum(math.prod(s) for n, s in _layer_shapes(C, H, N).items() if len(s) == 2 and n != "r_k")
    if kind == "adamw":  # parameter, gradient and both moments in; parameter and moments out
        return {"bytes": 28 * numel, "flops": 15 * numel}
    if kind == "timemix_train":  # float32 parameters in and their gradients out; x, gy in, out, dx out
        return {"bytes": 8 * numel + 4 * tok * 2 + 2 * state, "flops": 6 * B * T * mats + rec_f + rec_b}
    return {"bytes": 2 * numel + 2 * tok * 2 + 2 * state, "flops": 2 * B * T * mats + rec_f}


def tolerance(case):
    c, kind = case, case["kind"]
    if kind == "adamw":
        return {"rel": 1e-5}
    if c["dtype"] == "fp32":
        return {"rel": 1e-5}
    if kind.startswith("timemix"):
        return {"rel": 2.5e-2}
    return {"rel": 7e-3}


# ---------------------------------------------------------------------------- in 64 bits
class _Recurrence64(torch.autograd.Function):
    """S_t = S_{t-1} diag(d_t) + (S_{t-1} a_t) b_t^T + v_t k_t^T, y_t = S_t r_t step by step in
    float64 (S: [B,H,value,key]), with the adjoint written out the same way."""

    @staticmethod
    def forward(ctx, r, d, k, v, a, b, s0):
        T = r.shape[1]
        states = torch.empty((T + 1,) + tuple(s0.shape), dtype=torch.float64, device=s0.device)
        states[0] = s0
        y = torch.empty_like(r)
        for t in range(T):
            S = states[t]
            sa = (S * a[:, t].unsqueeze(-2)).sum(-1, keepdim=True)
            S = S * d[:, t].unsqueeze(-2)
            S.addcmul_(sa, b[:, t].unsqueeze(-2))
            S.addcmul_(v[:, t].unsqueeze(-1), k[:, t].unsqueeze(-2))
            states[t + 1] = S
            y[:, t] = (S * r[:, t].unsqueeze(-2)).sum(-1)
        ctx.save_for_backward(r, d, k, v, a, b, states)
        return y, states[T].clone()

    @staticmethod
    def backward(ctx, dy, dend):
        r, d, k, v, a, b, states = ctx.saved_tensors
        grads = [torch.empty_like(r) for _ in range(6)]
        dr, dd, dk, dv, da, db = grads
        G = dend.clone()
        for t in range(r.shape[1] - 1, -1, -1):
            S, dyt, vt = states[t], dy[:, t].unsqueeze(-1), v[:, t].unsqueeze(-1)
            dr[:, t] = (states[t + 1] * dyt).sum(-2)
            G = torch.addcmul(G, dyt, r[:, t].unsqueeze(-2))
            sa = (S * a[:, t].unsqueeze(-2)).sum(-1, keepdim=True)
            q = (G * b[:, t].unsqueeze(-2)).sum(-1, keepdim=True)
            dv[:, t] = (G * k[:, t].unsqueeze(-2)).sum(-1)
            dd[:, t] = (G * S).sum(-2)
            dk[:, t] = (G * vt).sum(-2)
            db[:, t] = (G * sa).sum(-2)
            da[:, t] = (S * q).sum(-2)
            G = torch.addcmul(G * d[:, t].unsqueeze(-2), q, a[:, t].unsqueeze(-2))
        return (*grads, G)


def _wkv7_64(r, w, k, v, a, b, s0):
    return _Recurrence64.apply(r, torch.exp(-DECAY_SCALE * torch.sigmoid(w)), k, v, a, b, s0)


def _gdn_64(q, k, v, g, beta, s0):
    """S_t = e^g (I - beta k k^T) S_{t-1} + beta k v^T, o = S^T q / sqrt(K), on S^T's layout."""
    N = q.shape[-1]
    q, k = (x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
    eg, be = torch.exp(g).unsqueeze(-1), beta.unsqueeze(-1)
    o, end = _Recurrence64.apply(q / math.sqrt(N), eg.expand_as(q).contiguous(), k, v * be, k, -eg * be * k,
                                 s0.transpose(-1, -2).contiguous())
    return o, end.transpose(-1, -2)


def _layer_64(p, x, shift, s0, H, N):
    B, T, C = x.shape
    delta = torch.cat([shift.unsqueeze(1), x[:, :-1]], 1) - x
    mix = {n: x + delta * p["x_" + n] for n in "rwkvag"}
    r, k, v = (mix[n[0]] @ p[n + ".weight"].t() for n in ("receptance", "key", "value"))
    w = p["w0"] + torch.tanh(mix["w"] @ p["w1"]) @ p["w2"]
    a = torch.sigmoid(p["a0"] + (mix["a"] @ p["a1"]) @ p["a2"])
    gate = torch.sigmoid(mix["g"] @ p["g1"]) @ p["g2"]
    heads = (B, T, H, N)
    kk = F.normalize((k * p["k_k"]).reshape(heads), dim=-1, eps=1e-12)
    k = (k * (1 + (a - 1) * p["k_a"])).reshape(heads)
    r, v = r.reshape(heads), v.reshape(heads)
    y, end = _wkv7_64(r, w.reshape(heads), k, v, -kk, kk * a.reshape(heads), s0)
    yn = (y - y.mean(-1, keepdim=True)) * torch.rsqrt(y.var(-1, unbiased=False, keepdim=True) + 64e-5)
    yn = yn.reshape(B, T, C) * p["ln_x.weight"] + p["ln_x.bias"]
    bonus = ((r * k * p["r_k"]).sum(-1, keepdim=True) * v).reshape(B, T, C)
    return ((yn + bonus) * gate) @ p["output.weight"].t(), end


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("wkv7_train", "wkv7_infer", "wkv7_decode"):
        xs, s0, dy = _wkv7_inputs(c, seed)
        xs, s0 = [x.double() for x in xs], s0.double()
        if kind != "wkv7_train":
            return list(_wkv7_64(*xs, s0))
        xs, s0 = [x.requires_grad_() for x in xs], s0.requires_grad_()
        y, end = _wkv7_64(*xs, s0)
        return [y.detach(), end.detach(), *torch.autograd.grad(y, xs + [s0], dy.double())]
    if kind in ("gdn_infer", "gdn_train"):
        q, k, v, g, beta, s0, do = _gdn_inputs(c, seed)
        xs = [x.double() for x in (q, k, v, g, beta)]
        if kind == "gdn_infer":
            return list(_gdn_64(*xs, s0.double()))
        xs = [x.requires_grad_() for x in xs]
        o, _ = _gdn_64(*xs, torch.zeros_like(s0, dtype=torch.float64))
        return [o.detach(), *torch.autograd.grad(o, xs, do.double())]
    if kind == "adamw":
        inp = _adamw_inputs(c, seed)
        total = math.sqrt(sum(float((gr.double() * GRAD_SCALE).square().sum()) for _, _, gr, _, _ in inp))
        factor = GRAD_SCALE * min(1.0, CLIP / (total + 1e-6))
        step, out = 101, []
        for n, p, gr, m, v in inp:
            p, gr, m, v = p.double(), gr.double() * factor, m.double(), v.double()
            m = m + (gr - m) * (1 - BETAS[0])
            v = v * BETAS[1] + gr * gr * (1 - BETAS[1])
            p = p * (1 - LR * (WEIGHT_DECAY if p.dim() == 2 else 0.0))
            denom = v.sqrt() / math.sqrt(1 - BETAS[1] ** step) + EPS
            out.append(p - LR / (1 - BETAS[0] ** step) * m / denom)
        return [torch.tensor(total, dtype=torch.float64, device="cuda"), *out]
    g = _gen(seed)
    params = _layer_params(c, g)
    x, st = _layer_inputs(c, g)
    if kind == "timemix_train":
        gy = _randn(g, *x.shape).to(x.dtype)
        names = [n for n, _ in _layer(c, params, torch.float32).named_parameters()]
        p = {n: params[n].double().requires_grad_() for n in names}
        x64 = x.double().requires_grad_()
        out, end = _layer_64(p, x64, st["shift"].double(), st["wkv"].double(), c["H"], c["N"])
        return [out.detach(), end.detach(), *torch.autograd.grad(out, [x64] + [p[n] for n in names], gy.double())]
    p = {n: t.to(torch.bfloat16).double() for n, t in params.items()}
    return list(_layer_64(p, x.double(), st["shift"].double(), st["wkv"].double(), c["H"], c["N"]))
