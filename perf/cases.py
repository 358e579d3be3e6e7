"""Performance cases of the kernel backend: the calls its users make, from one decoded token to the
largest prompt and training step, with the work each cannot do without and its result in 64 bits.

A case is a dict of plain values; ``kind`` names the entry point:

* ``step``        one decode step of the mLSTM state (``mlstm_recurrent_step__native``, or the
                  backend module in inference mode with one token)
* ``prefill``     a prompt through ``mLSTMBackend`` in inference mode (any length, initial state)
* ``chunkwise``   ``mlstm_chunkwise`` over whole chunks, last states returned
* ``train``       the chunkwise kernel forward and backward (gradients of q, k, v, i, f)
* ``slstm``       the sLSTM time loop over a whole sequence
* ``slstm_layer`` sLSTM layer: projection cell (conv + SiLU, gates, z), time loop, output cell
* ``mlstm_layer`` mLSTM layer: projection cell, backend, output cell (norm, gate, projection)
* ``decode``      one decode step of a whole stack, replayed from a HIP graph; returns logits

Inputs follow the backend's workloads (``xlstm_hip.workloads``): q scaled by 1/sqrt(DQK), k, v and
input gates N(0, 1), forget gates N(3, 1), drawn on the GPU from the seed.
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "xlstm-metal_amd"))

import xlstm_hip  # noqa: E402
from xlstm_hip.stack import StackConfig, xLSTMStack  # noqa: E402

DEV = "cuda:0"
EPS = 1e-6
GATE_CAP = 15.0
DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
ESZ = {"bf16": 2, "f16": 2, "f32": 4}


# ------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # a chat reply: one sequence, one token, the 7B head shape (latency, launches)
        dict(name="step_b1", kind="step", via="backend", B=1, NH=8, DQK=256, DV=512, dtype="bf16"),
        # batched serving: 16 sequences (the state's traffic)
        dict(name="step_b16", kind="step", via="op", B=16, NH=8, DQK=256, DV=512, dtype="bf16"),
        # the headline prefill: a batch of four 8k prompts
        dict(name="prefill_8k", kind="chunkwise", B=4, NH=8, S=8192, DQK=256, DV=512, dtype="bf16"),
        # a user's prompt: one sequence of no round length
        dict(name="prefill_prompt", kind="prefill", B=1, NH=8, S=2011, DQK=256, DV=512, dtype="bf16"),
        # short f16 prompts of a batch, the smaller model's head shape
        dict(name="prefill_f16", kind="prefill", B=8, NH=8, S=500, DQK=128, DV=256, dtype="f16"),
        # float32 evaluation
        dict(name="prefill_f32", kind="chunkwise", B=1, NH=8, S=1024, DQK=256, DV=512, dtype="f32"),
        # training at the 7B head shape: forward and backward
        dict(name="train_7b", kind="train", B=2, NH=8, S=4096, DQK=256, DV=512, dtype="bf16"),
        # training of the smaller model on short sequences
        dict(name="train_small", kind="train", B=2, NH=8, S=1024, DQK=128, DV=256, dtype="bf16"),
        # the sLSTM time loop of a batch of 4k prompts
        dict(name="slstm_4k", kind="slstm", B=8, S=4096, NH=4, H=512, dtype="bf16"),
        # a whole sLSTM layer on one prompt of odd length
        dict(name="slstm_layer", kind="slstm_layer", B=1, S=777, d=2048, NH=4, dtype="bf16"),
        # a whole mLSTM layer on one 2k prompt
        dict(name="mlstm_layer", kind="mlstm_layer", B=1, S=2048, d=4096, NH=8, dtype="bf16"),
        # serving a mixed stack (one sLSTM block in eight): a token for each of 8 sequences
        dict(name="decode_stack", kind="decode", B=8, d=2048, blocks=8, NH=8, every=8, vocab=50304, dtype="bf16"),
    ]


HEADS = ((64, 128), (96, 192), (128, 256), (256, 512))


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "step", "prefill", "prefill", "prefill", "chunkwise", "train", "train", "slstm",
                       "slstm_layer", "mlstm_layer", "decode"))
    DQK, DV = rng.choice(HEADS)
    NH = rng.choice((4, 8))
    if kind == "step":
        return dict(kind=kind, via=rng.choice(("backend", "op")), B=_log(rng, 1, 16), NH=NH, DQK=DQK, DV=DV,
                    dtype=rng.choice(("bf16", "bf16", "f16", "f32")))
    if kind == "prefill":
        B = rng.choice((1, 1, 2, 4, 8))
        return dict(kind=kind, B=B, NH=NH, S=_log(rng, 17, 8192 // B), DQK=DQK, DV=DV, dtype=rng.choice(("bf16", "bf16", "f16")))
    if kind == "chunkwise":
        dt = rng.choice(("bf16", "f32", "f32"))
        DQK, DV = rng.choice(((64, 128), (128, 256), (256, 512)))
        B = rng.choice((1, 1, 2))
        return dict(kind=kind, B=B, NH=NH, S=64 * _log(rng, 1, (16 if dt == "f32" else 128) // B), DQK=DQK, DV=DV, dtype=dt)
    if kind == "train":
        DQK, DV = rng.choice(((128, 256), (256, 512)))
        B = rng.choice((1, 2, 4))
        return dict(kind=kind, B=B, NH=NH, S=64 * _log(rng, 2, 128 // B), DQK=DQK, DV=DV, dtype="bf16")
    if kind == "slstm":
        B = _log(rng, 1, 8)
        return dict(kind=kind, B=B, S=_log(rng, 16, 4096), NH=4, H=rng.choice((192, 256, 512)),
                    dtype=rng.choice(("bf16", "bf16", "f32")))
    if kind == "slstm_layer":
        return dict(kind=kind, B=rng.choice((1, 2)), S=_log(rng, 16, 1024), d=rng.choice((1024, 2048)), NH=4, dtype="bf16")
    if kind == "mlstm_layer":
        return dict(kind=kind, B=1, S=_log(rng, 17, 2048), d=rng.choice((2048, 4096)), NH=8, dtype="bf16")
    return dict(kind=kind, B=_log(rng, 1, 16), d=rng.choice((1024, 2048)), blocks=rng.choice((4, 6, 8)), NH=8,
                every=4, vocab=50304, dtype="bf16")


# ------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _cap(x):
    return GATE_CAP * torch.tanh(x / GATE_CAP)


def _qkv_inputs(c, seed):
    """q, k, v, i, f of a sequence in the case's dtype."""
    g, dt = _gen(seed), DT[c["dtype"]]
    B, NH, S, DQK, DV = (c[x] for x in ("B", "NH", "S", "DQK", "DV"))
    q = _randn(g, B, NH, S, DQK) / math.sqrt(DQK)
    k, v = _randn(g, B, NH, S, DQK), _randn(g, B, NH, S, DV)
    i, f = _randn(g, B, NH, S), _randn(g, B, NH, S) + 3.0
    return g, tuple(t.to(dt) for t in (q, k, v, i, f))


def _step_inputs(c, seed):
    g, dt = _gen(seed), DT[c["dtype"]]
    B, NH, DQK, DV = (c[x] for x in ("B", "NH", "DQK", "DV"))
    q, k, v = _randn(g, B, NH, DQK).to(dt), _randn(g, B, NH, DQK).to(dt), _randn(g, B, NH, DV).to(dt)
    i, f = _cap(_randn(g, B, NH, 1)), _cap(_randn(g, B, NH, 1) + 3.0)
    C, n, m = 0.1 * _randn(g, B, NH, DQK, DV), _randn(g, B, NH, DQK).abs(), _randn(g, B, NH, 1)
    return q, k, v, i, f, C, n, m


def _module_weights(module, seed, g):
    """Linear and conv weights N(0, 1 / fan-in), biases 0 but the forget gate's 3, norm weights near 1."""
    for name, p in module.named_parameters():
        owner, what = name.split(".")[-2:]
        with torch.no_grad():
            if "norm" in owner:
                p.copy_(1.0 + 0.1 * _randn(g, *p.shape) if what == "weight" else 0.1 * _randn(g, *p.shape))
            elif what == "bias":
                p.fill_(3.0 if owner == "fgate_proj" else 0.0)
            else:
                p.copy_(_randn(g, *p.shape) / math.sqrt(p[0].numel()))
    return module


def _layer_modules(c, seed):
    g, dt, d, NH = _gen(seed), DT[c["dtype"]], c["d"], c["NH"]
    if c["kind"] == "slstm_layer":
        proj = xlstm_hip.sLSTMProjectionCell(d, NH, d // NH, gate_soft_cap=GATE_CAP)
        out = xlstm_hip.sLSTMOutputCell(d, NH, d // NH, eps=EPS)
    else:
        proj = xlstm_hip.mLSTMProjectionCell(d, NH, d // (2 * NH), d // NH, gate_soft_cap=GATE_CAP)
        out = xlstm_hip.mLSTMOutputCell(d, NH, d // NH, eps=EPS)
    proj, out = (_module_weights(m.to(DEV, dt), seed, g) for m in (proj, out))
    x = _randn(g, c["B"], c["S"], d).to(dt)  # a normalised residual stream
    return proj, out, x


def _backend():
    return xlstm_hip.mLSTMBackend(xlstm_hip.mLSTMBackendConfig(mode="inference"))


def _stack_inputs(c, seed):
    """The model, its states (as a prompt leaves them, contents drawn) and the tokens."""
    g, B = _gen(seed), c["B"]
    cfg = StackConfig("stack", d_model=c["d"], num_blocks=c["blocks"], mlstm_heads=c["NH"], slstm_every=c["every"],
                      vocab=c["vocab"], dtype=DT[c["dtype"]])
    model = xLSTMStack.random(cfg, DEV, seed=seed)
    with torch.no_grad():
        # a residual stream of unit scale and depth-scaled branches, as training starts from
        model.embedding.weight.div_(cfg.init_std)
        for blk in model.blocks:
            for lin in (blk.out.out_proj, blk.ffn.proj_down):
                lin.weight.div_(math.sqrt(2 * cfg.num_blocks))
    prompt = torch.randint(0, cfg.vocab, (B, 16), generator=g, device=DEV)
    _, states = model.prefill(prompt)
    for st in states:
        for key, t in vars(st).items():
            x = _randn(g, *t.shape)
            t.copy_(0.1 * x if key == "C" else x.abs() + 0.5 if key == "n" else x)
    return model, states, torch.randint(0, cfg.vocab, (B,), generator=g, device=DEV)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "step":
        return dict(case=c, x=_step_inputs(c, seed), backend=_backend() if c["via"] == "backend" else None)
    if kind in ("prefill", "chunkwise"):
        return dict(case=c, x=_qkv_inputs(c, seed)[1], backend=_backend())
    if kind == "train":
        g, x = _qkv_inputs(c, seed)
        dh = _randn(g, c["B"], c["NH"], c["S"], c["DV"]).to(DT[c["dtype"]])
        return dict(case=c, x=tuple(t.requires_grad_(True) for t in x), dh=dh,
                    kernel=xlstm_hip.get_mlstm_kernel("chunkwise--native_custbw"))
    if kind == "slstm":
        g, dt = _gen(seed), DT[c["dtype"]]
        B, S, NH = c["B"], c["S"], c["NH"]
        z = _randn(g, B, S, NH, c["H"]).to(dt)
        i, f, o = (_randn(g, B, S, NH).to(dt), (_randn(g, B, S, NH) + 3.0).to(dt), _randn(g, B, S, NH).to(dt))
        return dict(case=c, x=(z, i, f, o))
    if kind in ("slstm_layer", "mlstm_layer"):
        proj, out, x = _layer_modules(c, seed)
        return dict(case=c, proj=proj, out=out, x=x, backend=_backend())
    # decode: the step captured once, as a serving loop does
    model, states, token = _stack_inputs(c, seed)
    saved = [[t.clone() for t in vars(st).values()] for st in states]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        model.decode_step(token, states)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    for st, sv in zip(states, saved):
        for t, s in zip(vars(st).values(), sv):
            t.copy_(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = model.decode_step(token, states)
    return dict(case=c, model=model, states=states, token=token, graph=graph, logits=logits)


# ------------------------------------------------------------------------------------- one pass
def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "step":
        q, k, v, i, f, C, n, m = s["x"]
        if c["via"] == "backend":
            h, (C, n, m) = s["backend"](q[:, :, None], k[:, :, None], v[:, :, None], i, f, C, n, m)
        else:
            h, (C, n, m) = xlstm_hip.mlstm_recurrent_step__native(q, k, v, i, f, C, n, m, eps=EPS)
        return {"h": h.reshape(c["B"], c["NH"], c["DV"]), "C": C, "n": n, "m": m}
    if kind == "prefill":
        h, (C, n, m) = s["backend"](*s["x"])
        return {"h": h, "C": C, "n": n, "m": m}
    if kind == "chunkwise":
        h, (C, n, m) = xlstm_hip.mlstm_chunkwise(*s["x"], return_last_states=True, chunk_size=64, eps=EPS)
        return {"h": h, "C": C, "n": n, "m": m}
    if kind == "train":
        q, k, v, i, f = s["x"]
        h = s["kernel"](q=q, k=k, v=v, i=i, f=f, chunk_size=64, eps=EPS)
        dq, dk, dv, di, df = torch.autograd.grad(h, (q, k, v, i, f), s["dh"])
        return {"h": h.detach(), "dq": dq, "dk": dk, "dv": dv, "di": di, "df": df}
    if kind == "slstm":
        h, (cl, nl, ml) = xlstm_hip.slstm_sequence(*s["x"], eps=EPS)
        return {"h": h, "c": cl, "n": nl, "m": ml}
    if kind == "slstm_layer":
        with torch.no_grad():
            z, i, f, o, _ = s["proj"](s["x"])
            h, (cl, nl, ml) = xlstm_hip.slstm_sequence(z, i, f, o, eps=EPS)
            return {"y": s["out"](h), "c": cl, "n": nl, "m": ml}
    if kind == "mlstm_layer":
        with torch.no_grad():
            q, k, v, i, f = s["proj"](s["x"])
            h, (C, n, m) = s["backend"](q, k, v, i, f)
            return {"y": s["out"](h, s["x"]), "C": C, "n": n, "m": m}
    s["graph"].replay()
    return {"logits": s["logits"], "states": [dict(vars(st)) for st in s["states"]]}


# ------------------------------------------------------------------------------------- work
def _chunk_flops(c):
    L = min(64, c["S"])
    return c["B"] * c["NH"] * c["S"] * (4 * c["DQK"] * c["DV"] + 2 * L * (c["DQK"] + c["DV"]))


def _chunk_bytes(c):
    BNH, e = c["B"] * c["NH"], ESZ[c["dtype"]]
    return BNH * c["S"] * (2 * c["DQK"] + 2 * c["DV"] + 2) * e + BNH * (c["DQK"] * c["DV"] + c["DQK"] + 1) * 4


def work(case):
    c, kind = case, case["kind"]
    if kind == "step":
        BNH, e = c["B"] * c["NH"], ESZ[c["dtype"]]
        state = BNH * (c["DQK"] * c["DV"] + c["DQK"] + 1) * 4
        return {"bytes": 2 * state + BNH * (2 * c["DQK"] + 2 * c["DV"]) * e + 2 * BNH * 4,
                "flops": BNH * 6 * c["DQK"] * c["DV"]}
    if kind in ("prefill", "chunkwise"):
        return {"bytes": _chunk_bytes(c), "flops": _chunk_flops(c)}
    if kind == "train":
        # forward; backward: the states again, dC, and the three products with a state per token,
        # the four chunk-local products with DQK and the two with DV
        BNH, S, DQK, DV, e = c["B"] * c["NH"], c["S"], c["DQK"], c["DV"], ESZ[c["dtype"]]
        back = 2 * BNH * S * (5 * DQK * DV + 4 * 64 * DQK + 2 * 64 * DV)
        return {"bytes": BNH * S * e * ((2 * DQK + 2 * DV + 2) + (2 * DQK + 2 * DV + 2) + (2 * DQK + DV + 2)),
                "flops": _chunk_flops(c) + back}
    if kind == "slstm":
        B, S, NH, H, e = c["B"], c["S"], c["NH"], c["H"], ESZ[c["dtype"]]
        return {"bytes": e * (2 * B * S * NH * H + 3 * B * S * NH + 2 * B * NH * H + B * NH), "flops": 10 * B * S * NH * H}
    if kind == "slstm_layer":
        M, d, NH, e = c["B"] * c["S"], c["d"], c["NH"], ESZ[c["dtype"]]
        return {"bytes": e * (2 * M * d + 2 * d * d + 3 * NH * d + 8 * d), "flops": 2 * M * d * (2 * d + 3 * NH + 4)}
    if kind == "mlstm_layer":
        M, d, NH, e = c["B"] * c["S"], c["d"], c["NH"], ESZ[c["dtype"]]
        cc = dict(c, DQK=d // (2 * NH), DV=d // NH)
        return {"bytes": e * (2 * M * d + 4 * d * d + 2 * NH * d) + c["B"] * NH * (cc["DQK"] * cc["DV"] + cc["DQK"] + 1) * 4,
                "flops": 2 * M * d * (4 * d + 2 * NH) + _chunk_flops(cc)}
    B, d, e = c["B"], c["d"], ESZ[c["dtype"]]
    ffn = (int(d * 2.667) + 63) // 64 * 64
    ns = c["blocks"] // c["every"]
    nm = c["blocks"] - ns
    weights = c["vocab"] * d + c["blocks"] * 3 * d * ffn + nm * (4 * d * d + 2 * c["NH"] * d) + ns * (2 * d * d + 12 * d)
    states = nm * B * (d * d // 2 // c["NH"] + d // 2 + c["NH"]) * 4 + ns * B * 8 * d
    return {"bytes": weights * e + 2 * states + B * c["vocab"] * e, "flops": 2 * B * weights}


def tolerance(case):
    """About four times what the path is off its value in 64 bits (measured): float32 products as
    bf16 hi + lo pairs 6e-6, elementwise float32 2e-7; one bf16 rounding of an output 1.7e-3 (f16
    2e-4); the decode step's reference roundings 6e-3 (f16 7e-4); the layers' projections and
    roundings 5e-3; eight blocks in a row 1.5e-2."""
    kind, dt = case["kind"], case["dtype"]
    if dt == "f32":
        return {"rel": 3e-5 if kind == "chunkwise" else 1e-5}
    if kind == "decode":
        return {"rel": 3e-2}
    if kind in ("slstm_layer", "mlstm_layer"):
        return {"rel": 2e-2}
    if kind == "step":
        return {"rel": 3e-3 if dt == "f16" else 2e-2}
    return {"rel": 1e-3 if dt == "f16" else 7e-3}


# ------------------------------------------------------------------------------------- in 64 bits
def _d(*ts):
    return tuple(t.detach().double() for t in ts)


def _mlstm64(q, k, v, i, f, C, n, m, chunk=128):
    """h and the last (C, n, m) of the mLSTM over a sequence, the stabilisers and each token's divisor
    taken as constants by autograd (as the custom backward does)."""
    DQK, S = q.shape[-1], q.shape[2]
    q = q * DQK ** -0.5
    b = F.logsigmoid(f).cumsum(-1)
    M = (b + torch.maximum(m, torch.cummax(i - b, -1).values)).detach()
    hs, b0, ms = [], torch.zeros_like(b[..., :1]), m
    for s in range(0, S, chunk):
        e = min(S, s + chunk)
        qc, kc, vc, bc, ic, Mc = q[:, :, s:e], k[:, :, s:e], v[:, :, s:e], b[..., s:e], i[..., s:e], M[..., s:e]
        keep = torch.ones(e - s, e - s, dtype=torch.bool, device=q.device).tril()
        D = bc[..., :, None] - bc[..., None, :] + ic[..., None, :] - Mc[..., :, None]
        W = (qc @ kc.transpose(-1, -2).contiguous()) * torch.exp(D.masked_fill(~keep, -math.inf))
        qi = qc * torch.exp(bc - b0 + ms - Mc)[..., None]
        den = (qi * n[:, :, None]).sum(-1) + W.sum(-1)
        den = (torch.maximum(den.abs(), torch.exp(-Mc)) + EPS).detach()
        hs.append((qi @ C + W @ vc) / den[..., None])
        ka = kc * torch.exp(bc[..., -1:] - bc + ic - Mc[..., -1:])[..., None]
        g = torch.exp(bc[..., -1:] - b0 + ms - Mc[..., -1:])
        C = g[..., None] * C + ka.transpose(-1, -2).contiguous() @ vc
        n = g * n + ka.sum(2)
        b0, ms = bc[..., -1:], Mc[..., -1:]
    return torch.cat(hs, 2), C, n, ms


def _zero_state64(q, v):
    B, NH, _, DQK = q.shape
    return (q.new_zeros(B, NH, DQK, v.shape[-1]), q.new_zeros(B, NH, DQK), q.new_zeros(B, NH, 1))


def _slstm64(z, i, f, o, c, n, m):
    hs, lf, tz, og = [], F.logsigmoid(f), torch.tanh(z), torch.sigmoid(o)
    b = lf.cumsum(1)
    M = b + torch.maximum(m[:, None], torch.cummax(i - b, 1).values)
    fg = torch.exp(lf + torch.cat([m[:, None], M[:, :-1]], 1) - M)[..., None]
    ig = torch.exp(i - M)[..., None]
    u = ig * tz
    for t in range(z.shape[1]):
        c = torch.addcmul(u[:, t], fg[:, t], c)
        n = torch.addcmul(ig[:, t], fg[:, t], n)
        hs.append(c / (n.abs() + EPS))
    return og[..., None] * torch.stack(hs, 1), c, n, M[:, -1]


def _slstm_proj64(p, x, window=None):
    """z, i, f, o of x [B, S, d]; window: x preceded by the conv's earlier inputs."""
    K = p["conv1d.conv.weight"].shape[-1]
    if window is None:
        window = F.pad(x, (0, 0, K - 1, 0))
    S = x.shape[1]
    w = p["conv1d.conv.weight"][:, 0]
    xc = F.silu(sum(window[:, j:j + S] * w[:, j] for j in range(K)) + p["conv1d.conv.bias"])
    i, f = (_cap(xc @ p[g + ".weight"].T + p[g + ".bias"]) for g in ("igate_proj", "fgate_proj"))
    return x @ p["z_proj.weight"].T, i, f, _cap(x @ p["ogate_proj.weight"].T + p["ogate_proj.bias"])


def _slstm_out64(p, h):
    B, S, NH, H = h.shape
    y = F.group_norm(h.reshape(B * S, NH * H), NH, p["group_norm.weight"], p["group_norm.bias"], EPS)
    return y.view(B, S, NH * H) @ p["out_proj.weight"].T


def _mlstm_proj64(p, x, NH):
    q, k, v = ((x @ p[n + ".weight"].T).unflatten(-1, (NH, -1)).transpose(1, 2).contiguous()
               for n in ("q_proj", "k_proj", "v_proj"))
    i, f = (_cap(x @ p[g + ".weight"].T + p[g + ".bias"]).transpose(1, 2) for g in ("igate_proj", "fgate_proj"))
    return q, k, v, i, f


def _mlstm_out64(p, h, x):
    h = h.transpose(1, 2)
    y = (h * torch.rsqrt((h * h).mean(-1, keepdim=True) + EPS)).flatten(2) * p["norm.weight"]
    return (y * torch.sigmoid(x @ p["ogate_proj.weight"].T)) @ p["out_proj.weight"].T


def _params64(module):
    return {k: p.detach().double() for k, p in module.named_parameters()}


def _rms64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _stack64(c, seed):
    model, states, token = _stack_inputs(c, seed)
    x = model.embedding.weight.detach()[token].double()[:, None]
    new = []
    for b, (blk, st) in enumerate(zip(model.blocks, states)):
        p = _params64(blk)
        sub = lambda pre: {k[len(pre):]: v for k, v in p.items() if k.startswith(pre)}  # noqa: E731
        if c["every"] and (b + 1) % c["every"] == 0:
            xn = _rms64(x, p["norm_slstm.weight"])
            window = torch.cat([st.conv.double(), xn], 1)
            z, i, f, o = _slstm_proj64(sub("proj."), xn, window)
            h, cc, nn, mm = _slstm64(z.unflatten(-1, (i.shape[-1], -1)), i, f, o, *_d(st.c, st.n, st.m))
            x = x + _slstm_out64(sub("out."), h)
            new.append({"c": cc, "n": nn, "m": mm, "conv": window[:, 1:]})
        else:
            xn = _rms64(x, p["norm_mlstm.weight"])
            h, C, n, m = _mlstm64(*_mlstm_proj64(sub("proj."), xn, c["NH"]), *_d(st.C, st.n, st.m))
            x = x + _mlstm_out64(sub("out."), h, xn)
            new.append({"C": C, "n": n, "m": m})
        xn = _rms64(x, p["norm_ffn.weight"])
        up = F.silu(xn @ p["ffn.proj_up_gate.weight"].T) * (xn @ p["ffn.proj_up.weight"].T)
        x = x + up @ p["ffn.proj_down.weight"].T
    xn = _rms64(x, model.out_norm.weight.detach().double())[:, 0]
    logits = 30.0 * torch.tanh(xn @ model.lm_head.weight.detach().double().T / 30.0)
    return {"logits": logits, "states": new}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "step":
        q, k, v, i, f, C, n, m = _d(*_step_inputs(c, seed))
        h, C, n, m = _mlstm64(q[:, :, None], k[:, :, None], v[:, :, None], i, f, C, n, m)
        return {"h": h[:, :, 0], "C": C, "n": n, "m": m}
    if kind in ("prefill", "chunkwise"):
        x = _d(*_qkv_inputs(c, seed)[1])
        h, C, n, m = _mlstm64(*x, *_zero_state64(x[0], x[2]))
        return {"h": h, "C": C, "n": n, "m": m}
    if kind == "train":
        g, x = _qkv_inputs(c, seed)
        dh = _randn(g, c["B"], c["NH"], c["S"], c["DV"]).to(DT[c["dtype"]]).double()
        x = tuple(t.requires_grad_(True) for t in _d(*x))
        h = _mlstm64(*x, *_zero_state64(x[0], x[2]))[0]
        dq, dk, dv, di, df = torch.autograd.grad(h, x, dh)
        return {"h": h.detach(), "dq": dq, "dk": dk, "dv": dv, "di": di, "df": df}
    if kind == "slstm":
        z, i, f, o = _d(*prepare(c, seed)["x"])
        zero = z.new_zeros(z.shape[0], *z.shape[2:])
        h, cl, nl, ml = _slstm64(z, i, f, o, zero, zero, zero[..., 0])
        return {"h": h, "c": cl, "n": nl, "m": ml}
    with torch.no_grad():
        if kind == "decode":
            return _stack64(c, seed)
        proj, out, x = _layer_modules(c, seed)
        p, po, x = _params64(proj), _params64(out), x.double()
        if kind == "slstm_layer":
            z, i, f, o = _slstm_proj64(p, x)
            z = z.unflatten(-1, (c["NH"], -1))
            zero = z.new_zeros(z.shape[0], *z.shape[2:])
            h, cl, nl, ml = _slstm64(z, i, f, o, zero, zero, zero[..., 0])
            return {"y": _slstm_out64(po, h), "c": cl, "n": nl, "m": ml}
        q, k, v, i, f = _mlstm_proj64(p, x, c["NH"])
        h, C, n, m = _mlstm64(q, k, v, i, f, *_zero_state64(q, v))
        return {"y": _mlstm_out64(po, h, x), "C": C, "n": n, "m": m}
