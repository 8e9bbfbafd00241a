"""The work a user of this framework has it do, case by case, for timing.

Every case goes through a public entry point: the attention op
(``ops.chunk_cyfa``, ``ops.fused_recurrent_cyfa``), the attention layer and
the MLP of a decoder block, and the graphed greedy decode step of a model.
Sizes are those of the shipped configurations (hidden size 1024 / 1536 / 2048
with 4 / 6 / 8 heads of 256 channels and 128 slots), of the benchmark and of
the tests, with odd and ragged lengths beside the round ones.

``exact`` restates the math in float64 with plain torch: the op chunk by
chunk, differentiable, and the layer around it.
"""

import math
import sys
from pathlib import Path

import torch
import torch.nn.functional as F

_PKG = str(Path(__file__).resolve().parents[1] / "cyfa-jittor_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from cyclic_flow_attention import CyclicFlowAttention, CyclicFlowAttentionConfig, CyclicFlowAttentionForCausalLM  # noqa: E402
from cyclic_flow_attention.models.cyfa.modeling_cyfa import GatedMLP  # noqa: E402
from cyclic_flow_attention.ops import chunk_cyfa, fused_recurrent_cyfa  # noqa: E402
from cyclic_flow_attention.ops.utils import readout_table  # noqa: E402

DEV = "cuda"
EPS = 1e-6
MLP_WIDTH = {1024: 2816, 1536: 4096, 2048: 5632}  # the configurations' MLP widths
HEADS = {1024: 4, 1536: 6, 2048: 8}
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
MODEL_LAYERS = 8  # of a configuration's 24 equal layers


def listed():
    return [
        # One sequence's next token at the 1.4B model's heads: the smallest call, all latency.
        _decode("decode_one", B=1, H=8),
        # A serving batch's next token (the benchmark's 64 sequences at the 400M model's heads): a stream of fp32 states.
        _decode("decode_batch", B=64, H=4),
        # A short interactive prompt, two chunks with a ragged end.
        _prefill("prefill_short", B=1, T=97, H=4),
        # The benchmark's prefill batch.
        _prefill("prefill_batch", B=8, T=2048, H=4),
        # A long document continued from a carried state, one sequence, 1.4B heads.
        _prefill("prefill_long", B=1, T=16384, H=8, state=True),
        # A training step of the op at the benchmark's batch, bf16: forward, then every gradient.
        _train("train_batch", B=8, T=2048, H=4),
        # fp32 training, ragged, with carried states and their cotangents (sequence-chunked training).
        _train("train_fp32", B=2, T=1000, H=4, dtype="fp32", state=True),
        # A block's attention layer over a prefill batch, 400M.
        _layer("layer_prefill", hidden=1024, B=8, T=2048),
        # Batched prompts of unequal length, right-padded with a mask as generate_batch sends them.
        _layer("layer_padded", hidden=1024, B=8, T=576, padded=True),
        # A training step of one attention layer, bf16 parameters with fp32 norms and gates, odd length.
        _layer("layer_train", hidden=1024, B=2, T=1500, train=True),
        # A block's SwiGLU MLP over a prefill batch, 400M.
        dict(name="mlp_prefill", kind="mlp", hidden=1024, B=8, T=2048),
        # One greedy step of a serving loop: the graphed decode step of the 400M model (its lm_head and 8 of its layers).
        dict(name="model_decode", kind="model", hidden=1024, B=16),
    ]


def _decode(name, B, H, dtype="bf16"):
    return dict(name=name, kind="decode", B=B, H=H, dtype=dtype)


def _prefill(name, B, T, H, state=False):
    return dict(name=name, kind="prefill", B=B, T=T, H=H, dtype="bf16", D=256, M=128, state=state)


def _train(name, B, T, H, dtype="bf16", D=256, M=128, state=False):
    return dict(name=name, kind="train", B=B, T=T, H=H, dtype=dtype, D=D, M=M, state=state)


def _layer(name, hidden, B, T, padded=False, train=False):
    return dict(name=name, kind="layer", hidden=hidden, B=B, T=T, padded=padded, train=train)


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _batch_time(rng, tokens, t_lo, t_hi):
    """(B, T) with B * T at most ``tokens``, T over its range's logarithm."""
    T = _log_int(rng, t_lo, min(t_hi, tokens))
    return _log_int(rng, 1, max(1, min(16, tokens // T))), T


def draw(rng):
    kind = rng.choice(["decode", "prefill", "prefill", "train", "train", "layer", "layer", "mlp", "model"])
    if kind == "decode":
        c = _decode("", _log_int(rng, 1, 64), rng.choice([4, 6, 8]), rng.choice(["bf16", "bf16", "fp32"]))
        if c["H"] * c["B"] > 256:
            c["B"] = 256 // c["H"]
    elif kind == "prefill":
        H = rng.choice([4, 6, 8])
        B, T = _batch_time(rng, 131072 // H, 33, 16384)
        c = _prefill("", B, T, H, rng.random() < 0.3)
    elif kind == "train":
        H = rng.choice([4, 6, 8])
        if rng.random() < 0.6:
            B, T = _batch_time(rng, 65536 // H, 65, 4096)
            c = _train("", B, T, H)
        else:
            B, T = _batch_time(rng, 16384 // H, 65, 2048)
            c = _train("", B, T, H, "fp32", rng.choice([64, 128, 256]), rng.choice([64, 128]), rng.random() < 0.5)
    elif kind == "layer":
        mode = rng.choice(["prefill", "padded", "train"])
        hidden = rng.choice([1024, 1536, 2048])
        B, T = _batch_time(rng, {"prefill": 8192, "padded": 8192, "train": 3000}[mode], 65, 4096)
        if mode == "padded":
            T = (T + 63) // 64 * 64
        c = _layer("", hidden, B, T, mode == "padded", mode == "train")
    elif kind == "mlp":
        hidden = rng.choice([1024, 1536, 2048])
        B, T = _batch_time(rng, 8192, 1, 8192)
        c = dict(name="", kind="mlp", hidden=hidden, B=B, T=T)
    else:
        c = dict(name="", kind="model", hidden=rng.choice([1024, 1536, 2048]), B=_log_int(rng, 1, 64))
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, *shape):
    return torch.randn(*shape, device=DEV, generator=gen)


def _op_inputs(gen, B, T, H, D, M, dtype):
    """q, k, v as projections give them, gates as their activations do."""
    return dict(
        q=_randn(gen, B, T, H, D).to(dtype),
        k=_randn(gen, B, T, H, D).to(dtype),
        v=_randn(gen, B, T, H, D).to(dtype),
        g=F.logsigmoid(_randn(gen, B, T, H) + 3),
        delta=torch.sigmoid(_randn(gen, B, T, H)),
        beta=torch.sigmoid(_randn(gen, B, T, H)),
        readout=torch.eye(M - 1, device=DEV).expand(H, -1, -1) + 0.05 * _randn(gen, H, M - 1, M - 1),
        q_norm_weight=1 + 0.1 * _randn(gen, D),
        k_norm_weight=1 + 0.1 * _randn(gen, D),
    )


def _op_state(gen, B, H, D, M):
    return (0.3 * _randn(gen, B, H, D, M), 0.3 * _randn(gen, B, H, M, D),
            500.0 * torch.rand(B, H, device=DEV, generator=gen))


def _fill(module, gen):
    """Weights of a module as a checkpoint would hold them: N(0, 0.02)
    projections, short convolutions and norms of order one, the readout as
    initialised, decays of some tens of tokens; bf16 except norms, readout,
    A_log and dt_bias. (A readout far from its initial identity makes some
    outputs nearly vanish in front of the output norm, and the gradients of
    those few tokens, which no 16-bit path resolves, then outweigh the rest.)"""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if "norm" in name:
                p.copy_(1 + 0.1 * _randn(gen, *p.shape))
            elif "conv1d" in name:
                p.copy_(0.3 * _randn(gen, *p.shape))
            elif name.endswith("readout"):
                p.copy_(torch.eye(p.shape[-1], device=DEV).expand_as(p))
            elif name.endswith("A_log"):
                p.copy_(torch.log(1 + 15 * torch.rand(p.shape, device=DEV, generator=gen)))
            elif name.endswith("dt_bias"):
                p.copy_(-4 + _randn(gen, *p.shape))
            else:
                p.copy_((0.1 if name.endswith("bias") else 0.02) * _randn(gen, *p.shape))
            if not any(s in name for s in ("norm", "readout", "A_log", "dt_bias")):
                p.data = p.data.to(torch.bfloat16)
    return module


def prepare(case, seed):
    gen = _gen(seed)
    kind, B = case["kind"], case["B"]
    if kind == "decode":
        H = case["H"]
        x = _op_inputs(gen, B, 1, H, 256, 128, DTYPES[case["dtype"]])
        return dict(kind=kind, x=x, init=_op_state(gen, B, H, 256, 128), table=readout_table(x["readout"]))
    if kind in ("prefill", "train"):
        T, H, D, M, dt = case["T"], case["H"], case["D"], case["M"], DTYPES[case["dtype"]]
        x = _op_inputs(gen, B, T, H, D, M, dt)
        init = _op_state(gen, B, H, D, M) if case["state"] else None
        if kind == "prefill":
            return dict(kind=kind, x=x, init=init, table=readout_table(x["readout"]))
        cot = [_randn(gen, B, T, H, D).to(dt)]
        if init is not None:
            cot += [_randn(gen, *t.shape) for t in init]
        x = {n: t.requires_grad_(True) for n, t in x.items()}
        init = None if init is None else tuple(t.requires_grad_(True) for t in init)
        return dict(kind=kind, x=x, init=init, cot=cot)
    hidden = case["hidden"]
    if kind == "model":
        cfg = CyclicFlowAttentionConfig(hidden_size=hidden, num_heads=HEADS[hidden], num_hidden_layers=MODEL_LAYERS)
        with torch.device(DEV):
            model = CyclicFlowAttentionForCausalLM(cfg)
        _fill(model, gen).eval()
        ids = torch.randint(0, cfg.vocab_size, (B, 65), device=DEV, generator=gen)
        with torch.no_grad():
            cache = model(ids[:, :64], use_cache=True)["cache"]
        return dict(kind=kind, step=model.graphed_decoder(cache, ids[:, 64:]), token=ids[:, 64:].contiguous())
    T = case["T"]
    x = _randn(gen, B, T, hidden).bfloat16()
    if kind == "mlp":
        cfg = CyclicFlowAttentionConfig(hidden_size=hidden, num_heads=HEADS[hidden])
        with torch.device(DEV):
            mlp = GatedMLP(cfg)
        return dict(kind=kind, mlp=_fill(mlp, gen).eval(), x=x)
    with torch.device(DEV):
        layer = CyclicFlowAttention(hidden_size=hidden, num_heads=HEADS[hidden])
    _fill(layer, gen)
    mask = None
    if case["padded"]:
        lengths = torch.randint(T // 4, T + 1, (B,), device=DEV, generator=gen)
        lengths[0] = T
        mask = (torch.arange(T, device=DEV)[None, :] < lengths[:, None]).long()
    if not case["train"]:
        return dict(kind=kind, train=False, layer=layer.eval(), x=x, mask=mask)
    # the biases of the gates stay as they are: their gradients, a few sums over
    # all tokens that cancel to a percent of their terms, are noise in bf16
    layer.b_proj.bias.requires_grad_(False)
    layer.d_proj.bias.requires_grad_(False)
    return dict(kind=kind, train=True, layer=layer.train(), x=x.requires_grad_(True), mask=mask,
                cot=_randn(gen, B, T, hidden).bfloat16())


# ---------------------------------------------------------------- one pass


def run(state):
    kind = state["kind"]
    if kind == "decode":
        with torch.no_grad():
            return fused_recurrent_cyfa(**state["x"], initial_state=state["init"], output_final_state=True,
                                        table=state["table"])
    if kind == "prefill":
        with torch.no_grad():
            return chunk_cyfa(**state["x"], initial_state=state["init"], output_final_state=True,
                              table=state["table"])
    if kind == "train":
        x, init = state["x"], state["init"]
        o, final = chunk_cyfa(**x, initial_state=init, output_final_state=init is not None)
        outs = [o] if init is None else [o, *final]
        leaves = list(x.values()) + ([] if init is None else list(init))
        grads = torch.autograd.grad(outs, leaves, state["cot"])
        return dict(o=o.detach(), final=None if init is None else [t.detach() for t in final], grads=grads)
    if kind == "mlp":
        with torch.no_grad():
            return state["mlp"](state["x"])
    if kind == "model":
        step = state["step"]
        step.tokens.copy_(state["token"])  # the token the serving loop sampled
        tokens = step.step()
        return dict(tokens=tokens, logits=step.logits,
                    cache=[[list(c["recurrent_state"]), list(c["conv_state"])] for c in step.cache])
    layer = state["layer"]
    if not state["train"]:
        with torch.no_grad():
            y, cache = layer(state["x"], use_cache=True, attention_mask=state["mask"])
        return y, list(cache["recurrent_state"]), list(cache["conv_state"])
    y, _ = layer(state["x"])
    names, params = zip(*((n, p) for n, p in layer.named_parameters() if p.requires_grad))
    grads = torch.autograd.grad(y, [state["x"], *params], state["cot"])
    return dict(y=y.detach(), x=grads[0], params=dict(zip(names, grads[1:])))


# ---------------------------------------------------------------- what a pass cannot do without


def _op_flops(rows, D, M):
    """The recurrent form's products per token and head: both states updated
    and read (2 flops each per element), logits and weights of the slots."""
    return rows * (8 * D * M + 4 * (M - 1) * M)


def work(case):
    kind, B = case["kind"], case["B"]
    if kind == "decode":
        bh = B * case["H"]
        item = 2 if case["dtype"] == "bf16" else 4
        return dict(bytes=bh * (4 * 2 * (2 * 256 * 128) + 4 * 256 * item) + case["H"] * 127 * 128 * 4,
                    flops=_op_flops(bh, 256, 128))
    if kind in ("prefill", "train"):
        rows, D, M = B * case["T"] * case["H"], case["D"], case["M"]
        item = 2 if case["dtype"] == "bf16" else 4
        states = B * case["H"] * 2 * D * M * 4
        table = case["H"] * (M - 1) * M * 4
        nbytes = rows * (4 * D * item + 12) + table + states * (1 + case["state"])
        if kind == "prefill":
            return dict(bytes=nbytes, flops=_op_flops(rows, D, M))
        # q, k, v, the gates and o's cotangent read; o and the gradients written
        nbytes = rows * (8 * D * item + 24) + 2 * table + (4 * states if case["state"] else 0)
        return dict(bytes=nbytes, flops=3 * _op_flops(rows, D, M))
    hidden = case["hidden"]
    H = HEADS[hidden]
    attn_w = 4 * hidden * hidden + 2 * 256 * hidden + 3 * H * hidden
    mlp_w = 3 * hidden * MLP_WIDTH[hidden]
    if kind == "model":
        weights = MODEL_LAYERS * (attn_w + mlp_w) + 32000 * hidden
        states = MODEL_LAYERS * B * H * (2 * 256 * 128) * 4
        return dict(bytes=2 * weights + 2 * states + 2 * B * 32000,
                    flops=2 * B * weights + MODEL_LAYERS * _op_flops(B * H, 256, 128))
    tokens = B * case["T"]
    if kind == "mlp":
        return dict(bytes=2 * (mlp_w + 2 * tokens * hidden), flops=2 * tokens * mlp_w)
    states = B * H * 2 * 256 * 128 * 4
    flops = 2 * tokens * attn_w + _op_flops(tokens * H, 256, 128)
    if case["train"]:
        return dict(bytes=2 * (2 * attn_w + 4 * tokens * hidden), flops=3 * flops)
    return dict(bytes=2 * (attn_w + 2 * tokens * hidden) + states, flops=flops)


def tolerance(case):
    """Against ``exact`` the paths measure: bf16 op 0.0036 (decode 0.0019), and
    in a training step 0.007 at delta's gradient; layers 0.005 at the output,
    0.017 at states that a rounded a|b|d projection decays, 0.035 at the
    gates' gradients; the MLP 0.0035; fp32 ops 3e-6 (decode 6.4e-6)."""
    kind = case["kind"]
    if kind in ("decode", "prefill", "train"):
        if case["dtype"] == "fp32":
            return {"rel": 2.5e-5 if kind == "decode" else 1e-5}
        return {"rel": {"decode": 0.008, "prefill": 0.014, "train": 0.02}[kind]}
    if kind == "mlp":
        return {"rel": 0.014}
    return {"rel": 0.02} if kind == "layer" and not case["train"] else {"rel": 0.03, "differ": 0.01}


# ---------------------------------------------------------------- the same in float64


def _basis(M):
    R = M - 1
    r = torch.arange(R, device=DEV, dtype=torch.float64)[:, None]
    col = torch.arange(M, device=DEV)
    angle = (r * (col // 2)) % R * (2 * math.pi / R)
    phi = torch.where(col % 2 == 1, torch.sin(angle), torch.cos(angle))
    return phi * _pair_scale(M).repeat_interleave(2) * (col != 1)


def _pair_scale(M):
    s = torch.full((M // 2,), math.sqrt(2.0 / (M - 1)), device=DEV, dtype=torch.float64)
    s[0] = math.sqrt(1.0 / (M - 1))
    return s


def _turn(x, c, s):
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack([c * e - s * o, s * e + c * o], -1).flatten(-2)


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _sgla(q, k, v, g, S, scale):
    """o_t = scale q_t S_t with S_t = e^{g_t} S_{t-1} + k_t v_t^T, 64 tokens at a time."""
    out = []
    for t in range(0, q.shape[2], 64):
        qc, kc, vc = (x[:, :, t:t + 64] for x in (q, k, v))
        G = g[:, :, t:t + 64].cumsum(-1)
        n = G.shape[-1]
        keep = torch.ones(n, n, device=DEV, dtype=torch.bool).tril()
        decay = torch.exp((G[..., :, None] - G[..., None, :]).masked_fill(~keep, -math.inf))
        out.append(scale * ((qc @ kc.mT * decay) @ vc + torch.exp(G)[..., None] * (qc @ S)))
        last = G[..., -1:]
        S = torch.exp(last)[..., None] * S + (kc * torch.exp(last - G)[..., None]).mT @ vc
    return torch.cat(out, 2), S


def _op64(q, k, v, g, delta, beta, readout, q_norm_weight, k_norm_weight, init):
    """The op in float64, differentiable: (o [B, T, H, D], (hk, hv, clock))."""
    B, T, H, D = q.shape
    M = readout.shape[-1] + 1
    q, k = _norm(q, q_norm_weight).transpose(1, 2), _norm(k, k_norm_weight).transpose(1, 2)
    v, g, delta, beta = (x.transpose(1, 2) for x in (v, g, delta, beta))
    if init is None:
        zero = torch.zeros(B, H, D, M, device=DEV, dtype=torch.float64)
        init = (zero, zero.mT, zero[..., 0, 0])
    lam = delta.cumsum(-1) + init[2][..., None]
    angle = lam[..., None] * torch.arange(M // 2, device=DEV, dtype=torch.float64) * (2 * math.pi / (M - 1))
    c, s = torch.cos(angle), torch.sin(angle)
    w = beta[..., None] * torch.stack([_pair_scale(M) * c, -_pair_scale(M) * s], -1).flatten(-2)
    raw, hk = _sgla(q, k, w, g, init[0], D ** -0.5)
    table = readout @ _basis(M)
    p = torch.softmax(_turn(raw, c, s) @ table.mT, -1)
    o, hv = _sgla(_turn(p @ table, c, -s), w, v, g, init[1], 1.0)
    return o.transpose(1, 2), (hk, hv, lam[..., -1])


def _conv64(x, weight):
    W = weight.shape[-1]
    xp = F.pad(x, (0, 0, W - 1, 0))
    return sum(xp[:, i:i + x.shape[1]] * weight[:, 0, i] for i in range(W))


def _layer64(p, x, H, mask):
    """The attention layer in float64 on the parameters ``p``: (y, states, conv caches)."""
    B, T, _ = x.shape
    qkv = [x @ p[n + "_proj.weight"].mT for n in "qkv"]
    if mask is not None:
        qkv = [t * mask[..., None] for t in qkv]
    ends = torch.full((B,), T, device=DEV) if mask is None else mask.sum(1)
    rows = ends[:, None] + torch.arange(-3, 0, device=DEV)[None, :]  # (lengths here are at least 3)
    conv = [t[torch.arange(B, device=DEV)[:, None], rows] for t in qkv]
    q, k, v = (_conv64(t, p[n + "_conv1d.weight"]).view(B, T, H, 256) for n, t in zip("qkv", qkv))
    g = -torch.exp(p["A_log"]) * F.softplus(x @ p["a_proj.weight"].mT + p["dt_bias"])
    delta = torch.sigmoid(x.detach() @ p["d_proj.weight"].mT + p["d_proj.bias"])
    beta = torch.sigmoid(x @ p["b_proj.weight"].mT + p["b_proj.bias"])
    if mask is not None:
        g, delta, beta = (t * mask[..., None] for t in (g, delta, beta))
    o, states = _op64(q, k, v, g, delta, beta, p["readout"], p["q_norm.weight"], p["k_norm.weight"], None)
    gate = (x @ p["g_proj.0.weight"].mT) @ p["g_proj.1.weight"].mT + p["g_proj.1.bias"]
    o = _norm(o * 127, p["o_norm.weight"]).flatten(2) * torch.sigmoid(gate)
    return o @ p["o_proj.weight"].mT, states, conv


def exact(case, seed):
    kind = case["kind"]
    if kind == "model":  # a rounding of one layer travels through the others: no such value
        return None
    st = prepare(case, seed)
    if kind in ("decode", "prefill"):
        x = {n: t.double() for n, t in st["x"].items()}
        init = None if st["init"] is None else [t.double() for t in st["init"]]
        return _op64(**x, init=init)
    if kind == "train":
        x = {n: t.detach().double().requires_grad_(True) for n, t in st["x"].items()}
        init = None if st["init"] is None else [t.detach().double().requires_grad_(True) for t in st["init"]]
        o, final = _op64(**x, init=init)
        outs = [o] if init is None else [o, *final]
        leaves = list(x.values()) + ([] if init is None else init)
        grads = torch.autograd.grad(outs, leaves, [t.double() for t in st["cot"]])
        return dict(o=o.detach(), final=None if init is None else [t.detach() for t in final], grads=grads)
    if kind == "mlp":
        x = st["x"].double()
        w = {n: p.detach().double() for n, p in st["mlp"].named_parameters()}
        h = F.silu(x @ w["gate_proj.weight"].mT) * (x @ w["up_proj.weight"].mT)
        return h @ w["down_proj.weight"].mT
    p = {n: t.detach().double().requires_grad_(st["train"] and t.requires_grad)
         for n, t in st["layer"].named_parameters()}
    x = st["x"].detach().double().requires_grad_(st["train"])
    y, states, conv = _layer64(p, x, HEADS[case["hidden"]], st["mask"])
    if not st["train"]:
        return y, list(states), conv
    trained = {n: t for n, t in p.items() if t.requires_grad}
    grads = torch.autograd.grad(y, [x, *trained.values()], st["cot"].double())
    return dict(y=y.detach(), x=grads[0], params=dict(zip(trained, grads[1:])))
