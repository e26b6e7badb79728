"""The work a program has this framework do, as measurable cases.

Four kinds of case, each through the package's public entry points:

* ``linear``    one ``MixedLinear`` called eagerly (the module API without a graph);
* ``layer``     the four projections of decoder layers -- Q/K/V and Gate/Up stacked
                (``MixedLinearGroup``), O, Down -- each on an activation of its own.
                Decode row counts are replayed as a HIP graph, as a serving loop does;
                prompts are eager calls;
* ``attention`` ``decode_attention`` over a static KV cache;
* ``step``      one fused one-token step of a whole (shallow) Llama model, replayed as
                a HIP graph, to its logits.

Layer widths are those of Llama-3.2-3B, Qwen2.5-7B and Qwen2.5-14B (Qwen with Q/K/V
biases).  Weights are N(0, 0.02); activations N(0, 1) with 0.5% of the channels x 20.
16-bit tiles are spread uniformly or, ``clustered``, picked by the top-k rule on weights
with a few loud row and column blocks, which gives row tiles very uneven shares.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from tilequant_amd import MixedLinear, MixedLinearGroup, pack_weight_from_tile_ids
from tilequant_amd.attention import decode_attention, decode_attention_workspace
from tilequant_amd.fused_decode import FusedDecodeStep

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
# hidden, (q, k, v) widths, MLP width, biased Q/K/V
MODELS = {
    "llama3.2-3b": (3072, (3072, 1024, 1024), 8192, False),
    "qwen2.5-7b": (3584, (3584, 512, 512), 18944, True),
    "qwen2.5-14b": (5120, (5120, 1024, 1024), 13824, True),
}
GROUPS = ("qkv", "o", "gate_up", "down")
MOST_ROW_PARAMS = 8192 * 100_663_296   # rows x weights of the largest prompt: a Llama-3.2-3B layer at 8192 rows
STEP_VOCAB = 8192   # small beside the two layers, as a vocabulary is beside a whole model's


def listed():
    layer = dict(kind="layer", dtype="bf16", clustered=False)
    return [
        # one token through one attention-output projection, called eagerly: a module-level program's smallest call
        dict(name="linear_1", kind="linear", model="llama3.2-3b", group="o", rows=1, keep=0.01, dtype="bf16",
             clustered=False),
        # single-user decoding
        dict(layer, name="decode_1", model="llama3.2-3b", rows=1, keep=0.01, layers=4, graph=True),
        # a small decode batch, the quoted benchmark configuration
        dict(layer, name="decode_4", model="llama3.2-3b", rows=4, keep=0.01, layers=4, graph=True),
        # the same on a larger model whose 16-bit tiles cluster in a few row tiles
        dict(layer, name="decode_4_clustered", model="qwen2.5-7b", rows=4, keep=0.10, clustered=True, layers=2,
             graph=True),
        # a medium decode batch, many 16-bit tiles
        dict(layer, name="decode_16", model="qwen2.5-14b", rows=16, keep=0.20, clustered=True, layers=2, graph=True),
        # a full serving batch
        dict(layer, name="decode_64", model="llama3.2-3b", rows=64, keep=0.01, layers=4, graph=True),
        # a short chat prompt
        dict(layer, name="prompt_128", model="llama3.2-3b", rows=128, keep=0.05, layers=1, graph=False),
        # an ordinary prompt of ragged length, in fp16
        dict(layer, name="prompt_777", model="qwen2.5-7b", rows=777, keep=0.10, clustered=True, dtype="fp16",
             layers=1, graph=False),
        # a long prompt
        dict(layer, name="prompt_2048", model="llama3.2-3b", rows=2048, keep=0.05, layers=1, graph=False),
        # a batch of long prompts, the quoted prefill configuration
        dict(layer, name="prompt_8192", model="llama3.2-3b", rows=8192, keep=0.05, layers=1, graph=False),
        # attention of a small batch at the end of a long request
        dict(name="attention_4x2304", kind="attention", batch=4, q_heads=24, kv_heads=8, length=2304, used=2304,
             dtype="bf16"),
        # a whole decode step to its logits
        dict(name="step_4", kind="step", batch=4, layers=2, keep=0.01, length=2304, used=2200, dtype="bf16",
             clustered=False),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(("linear", "decode", "prompt", "attention", "step"), (2, 4, 5, 2, 1))[0]
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
    clustered = rng.random() < 0.5
    keep = rng.choice((0.01, 0.05, 0.10, 0.20))
    model = rng.choice(sorted(MODELS))
    if kind == "linear":
        return dict(kind="linear", model=model, group=rng.choice(GROUPS), rows=_log(rng, 1, 64), keep=keep,
                    dtype=dtype, clustered=clustered)
    if kind == "decode":
        return dict(kind="layer", model=model, rows=_log(rng, 1, 64), keep=keep, dtype=dtype, clustered=clustered,
                    layers=rng.choice((2, 3)), graph=True)
    if kind == "prompt":
        hidden, qkv, mlp, _ = MODELS[model]
        per_row = hidden * (sum(qkv) + hidden + 3 * mlp) * (1 + 2 * keep)   # 16-bit tiles cost more
        most = min(8192, int(MOST_ROW_PARAMS / per_row))
        return dict(kind="layer", model=model, rows=_log(rng, 65, most), keep=keep,
                    dtype=dtype, clustered=clustered, layers=1, graph=False)
    if kind == "attention":
        q_heads, kv_heads = rng.choice(((24, 8), (28, 4), (40, 8)))
        batch = _log(rng, 1, 16)
        length = _log(rng, 128, 65536 // batch)
        return dict(kind="attention", batch=batch, q_heads=q_heads, kv_heads=kv_heads, length=length,
                    used=rng.randint(max(1, length // 2), length), dtype=dtype)
    length = _log(rng, 128, 4096)
    return dict(kind="step", batch=_log(rng, 1, 8), layers=rng.choice((1, 2)), keep=keep, length=length,
                used=rng.randint(max(1, length // 2), length), dtype=dtype, clustered=clustered)


# ---- inputs ---------------------------------------------------------------------

class _Numbers:
    """A sequence of random tensors on the GPU, made from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return (torch.randn(shape, generator=self.gen, device=DEV, dtype=torch.float32) * std).to(dtype)

    def permutation(self, n):
        return torch.randperm(n, generator=self.gen, device=DEV)

    def activation(self, rows, k, dtype):
        x = self.normal(rows, k)
        x[:, self.permutation(k)[: round(0.005 * k)]] *= 20
        return x.to(dtype)

    def weight(self, m, k, case):
        """One projection's weight, and a [m / 64, k / 64] mask that is True for its 16-bit tiles."""
        n_tr, n_tc = m // 64, k // 64
        w = self.normal(m, k, std=0.02)
        take = max(1, math.ceil(case["keep"] * n_tr * n_tc))
        mask = torch.zeros(n_tr * n_tc, dtype=torch.bool, device=DEV)
        if case["clustered"]:
            tiles = w.view(n_tr, 64, n_tc, 64)
            tiles[:, :, self.permutation(n_tc)[: max(1, round(0.03 * n_tc))]] *= 4
            tiles[self.permutation(n_tr)[: max(1, round(0.03 * n_tr))]] *= 3
            w = w.to(DTYPES[case["dtype"]])
            score = w.float().abs().view(n_tr, 64, n_tc, 64).sum(dim=(1, 3)).view(-1)
            mask[score.topk(take).indices] = True
        else:
            w = w.to(DTYPES[case["dtype"]])
            mask[self.permutation(n_tr * n_tc)[:take]] = True
        return w, mask.view(n_tr, n_tc)


def _widths(model, group):
    """Input width and member output widths of a projection group."""
    hidden, qkv, mlp, _ = MODELS[model]
    return {"qkv": (hidden, qkv), "o": (hidden, (hidden,)), "gate_up": (hidden, (mlp, mlp)),
            "down": (mlp, (hidden,))}[group]


def _group_weights(num, case, model, group):
    """(weight, 16-bit mask, bias or None) of each member of a projection group."""
    k, widths = _widths(model, group)
    out = []
    for m in widths:
        w, mask = num.weight(m, k, case)
        biased = group == "qkv" and MODELS[model][3]
        out.append((w, mask, num.normal(m, std=0.5, dtype=w.dtype) if biased else None))
    return out


def _module(members, case):
    mods = []
    for w, mask, bias in members:
        flat = mask.view(-1).cpu()
        pack = pack_weight_from_tile_ids(
            w, n_tr=mask.shape[0], n_tc=mask.shape[1], int8_tile_ids=torch.nonzero(~flat).view(-1),
            fp16_tile_ids=torch.nonzero(flat).view(-1), cfg={})
        mods.append(MixedLinear(pack, bias, {"dtype_out": case["dtype"]}))
    return mods[0] if len(mods) == 1 else MixedLinearGroup(mods)


def _linear_of(module):
    return module.linear if isinstance(module, MixedLinearGroup) else module


def _projections(case):
    """(layer, group) of every projection of the case, in call order."""
    if case["kind"] == "linear":
        return [(0, case["group"])]
    return [(i, g) for i in range(case["layers"]) for g in GROUPS]


def _attention_inputs(case, seed):
    num = _Numbers(seed)
    dt = DTYPES[case["dtype"]]
    shape = (case["batch"], case["kv_heads"], case["length"], 128)
    return (num.normal(case["batch"], case["q_heads"], 128, dtype=dt), num.normal(*shape, dtype=dt),
            num.normal(*shape, dtype=dt))


def _step_inputs(case, seed):
    """Token ids, embedding and per-layer (norms, members by group, caches) of a shallow Llama, one by one."""
    num = _Numbers(seed)
    dt = DTYPES[case["dtype"]]
    hidden, qkv, _, _ = MODELS["llama3.2-3b"]
    token = torch.randint(0, STEP_VOCAB, (case["batch"], 1), generator=num.gen, device=DEV)
    yield token, num.normal(STEP_VOCAB, hidden, std=0.02, dtype=dt), 1 + num.normal(hidden, std=0.1, dtype=dt)
    shape = (case["batch"], qkv[1] // 128, case["length"], 128)
    for _ in range(case["layers"]):
        norms = [1 + num.normal(hidden, std=0.1, dtype=dt) for _ in range(2)]
        members = {g: _group_weights(num, case, "llama3.2-3b", g) for g in GROUPS}
        yield norms, members, num.normal(*shape, dtype=dt), num.normal(*shape, dtype=dt)


def _rope(positions, dtype):
    freq = 1.0 / (5e5 ** (torch.arange(0, 128, 2, device=DEV, dtype=torch.float32) / 128))
    angle = positions.float().unsqueeze(-1) * freq
    angle = torch.cat((angle, angle), dim=-1)
    return angle.cos().to(dtype), angle.sin().to(dtype)


class _Norm(torch.nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight = torch.nn.Parameter(weight, requires_grad=False)
        self.variance_epsilon = 1e-5


def _step_model(case, seed):
    """The model a decode step is bound to (Llama layout), its cache and the step's inputs."""
    parts = _step_inputs(case, seed)
    token, table, final = next(parts)
    hidden, qkv, mlp, _ = MODELS["llama3.2-3b"]
    layers, caches = [], []
    for norms, members, k, v in parts:
        mods = {g: _module(m, case) for g, m in members.items()}
        attn = torch.nn.Module()
        attn.tilequant_qkv, attn.o_proj, attn.scaling = mods["qkv"], mods["o"], 128 ** -0.5
        ffn = torch.nn.Module()
        ffn.tilequant_gate_up, ffn.down_proj = mods["gate_up"], mods["down"]
        layer = torch.nn.Module()
        layer.self_attn, layer.mlp = attn, ffn
        layer.input_layernorm, layer.post_attention_layernorm = (_Norm(w) for w in norms)
        layers.append(layer)
        caches.append(SimpleNamespace(keys=k, values=v))
    text = torch.nn.Module()
    text.embed_tokens = torch.nn.Embedding.from_pretrained(table)
    text.layers = torch.nn.ModuleList(layers)
    text.norm = _Norm(final)
    text.rotary_emb = lambda x, pos: _rope(pos, x.dtype)
    model = torch.nn.Module()
    model.model = text
    model.lm_head = torch.nn.Linear(hidden, STEP_VOCAB, bias=False, device="meta")
    model.lm_head.weight = torch.nn.Parameter(table, requires_grad=False)
    cfg = SimpleNamespace(model_type="llama", hidden_size=hidden, num_attention_heads=qkv[0] // 128,
                          num_key_value_heads=qkv[1] // 128, head_dim=128, intermediate_size=mlp)
    cfg.get_text_config = lambda decoder=True: cfg
    model.config = cfg
    return model, SimpleNamespace(layers=caches), token


def _captured(call):
    """``call`` as a HIP graph and its outputs, warmed up on the capturing stream."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = call()
    return graph, out


# ---- the cases ------------------------------------------------------------------

@torch.inference_mode()
def prepare(case, seed):
    dt = DTYPES[case["dtype"]]
    if case["kind"] == "attention":
        q, k, v = _attention_inputs(case, seed)
        used = torch.full((case["batch"],), case["used"], dtype=torch.int32, device=DEV)
        return {"q": q, "k": k, "v": v, "used": used,
                "ws": decode_attention_workspace(case["batch"], case["q_heads"], case["length"], q.device)}
    if case["kind"] == "step":
        model, cache, token = _step_model(case, seed)
        step = FusedDecodeStep(model, cache, case["batch"], case["length"], token.device)
        position = torch.full((1,), case["used"] - 1, dtype=torch.long, device=DEV)
        used = torch.full((case["batch"],), case["used"], dtype=torch.int32, device=DEV)
        graph, out = _captured(lambda: step(token, position, used))
        return {"graph": graph, "out": out, "keep": (model, cache, step, token, position, used)}
    num = _Numbers(seed)
    calls = []
    for _, group in _projections(case):
        mod = _linear_of(_module(_group_weights(num, case, case["model"], group), case))
        calls.append((mod, num.activation(case["rows"], _widths(case["model"], group)[0], dt)))
    if case["kind"] == "layer" and case["graph"]:
        graph, out = _captured(lambda: [mod(x) for mod, x in calls])
        return {"graph": graph, "out": out, "keep": calls}
    return {"calls": calls}


@torch.inference_mode()
def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if "calls" in state:
        return [mod(x) for mod, x in state["calls"]]
    return decode_attention(state["q"], state["k"], state["v"], state["used"], scale=128 ** -0.5,
                            workspace=state["ws"])


def _gemm_work(case, rows, group, model):
    k, widths = _widths(model, group)
    read = 0
    for m in widths:
        tiles = (m // 64) * (k // 64)
        t16 = max(1, math.ceil(case["keep"] * tiles))
        read += 4100 * (tiles - t16) + 8192 * t16
    m = sum(widths)
    return read + 2 * rows * (k + m), 2.0 * rows * m * k


def work(case):
    if case["kind"] == "attention":
        kv = 4 * case["batch"] * case["kv_heads"] * case["used"] * 128
        heads = case["batch"] * case["q_heads"]
        return {"bytes": kv + 4 * heads * 128, "flops": 4.0 * heads * case["used"] * 128}
    if case["kind"] == "step":
        n, hidden, kv = case["batch"], 3072, 8
        nbytes, flops = 2 * STEP_VOCAB * (hidden + n), 2.0 * n * STEP_VOCAB * hidden
        for g in GROUPS:
            b, f = _gemm_work(case, n, g, "llama3.2-3b")
            nbytes, flops = nbytes + case["layers"] * b, flops + case["layers"] * f
        nbytes += case["layers"] * 4 * n * kv * case["used"] * 128
        return {"bytes": nbytes, "flops": flops + case["layers"] * 4.0 * n * 24 * case["used"] * 128}
    nbytes = flops = 0
    for _, g in _projections(case):
        b, f = _gemm_work(case, case["rows"], g, case["model"])
        nbytes, flops = nbytes + b, flops + f
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Two correct implementations differ in the order of their fp32 sums, which
    moves an output by one step of its 16-bit type now and then."""
    if case["kind"] == "step":
        # one 16-bit rounding that falls the other way can move a column tile's scale, and with it a
        # tile's INT8 codes in every layer after: 0.7% per layer against 64-bit sums
        return {"rel": 0.03, "max": 0.3}
    return {"rel": 5e-3, "max": 0.03} if case["dtype"] == "bf16" else {"rel": 7e-4, "max": 4e-3}


# ---- plain torch in 64 bits -----------------------------------------------------

def _scale(absmax):
    """absmax / 127, and 1 where a tile is all zero.  The divisor is a tensor: torch multiplies by the
    reciprocal of a number, which is one step off often enough to move codes at ties."""
    return torch.where(absmax > 0, absmax / torch.full_like(absmax, 127.0), torch.ones_like(absmax))


def _codes64(x):
    """An activation as its INT8 codes times their scales: one scale per 64 columns over all rows."""
    n, k = x.shape
    t = x.float().view(n, k // 64, 64)
    a = t.abs().amax(dim=(0, 2))
    s = _scale(a).to(x.dtype).float()
    q = (t / s[:, None]).round().clamp(-127, 127)
    return (q.double() * s.double()[:, None]).view(n, k)


def _linear64(x, members):
    xq = _codes64(x)
    out = []
    for w, mask, bias in members:
        n_tr, n_tc = mask.shape
        t = w.float().view(n_tr, 64, n_tc, 64)
        a = t.abs().amax(dim=(1, 3), keepdim=True)
        s = _scale(a)
        q = (t / s).round().clamp(-127, 127).double() * s.double()
        kept = mask[:, None, :, None]
        y = xq @ torch.where(kept, 0.0, q).view(w.shape).t()
        y += x.double() @ torch.where(kept, t.double(), 0.0).view(w.shape).t()
        out.append(y if bias is None else y + bias.double())
    return torch.cat(out, dim=1)


def _attention64(q, k, v, used):
    batch, heads, _ = q.shape
    kv = k.shape[1]
    q = q.double().view(batch, kv, heads // kv, 128)
    score = torch.matmul(q, k[:, :, :used].double().transpose(2, 3).contiguous()) * 128 ** -0.5
    return torch.matmul(score.softmax(dim=-1), v[:, :, :used].double()).view(batch, heads, 128)


def _step64(case, seed):
    """The step with 64-bit sums, rounded to the model's type where its modules round."""
    dt = DTYPES[case["dtype"]]
    parts = _step_inputs(case, seed)
    token, table, final = next(parts)
    batch, used = case["batch"], case["used"]
    h = table[token.view(-1)]

    def norm(x, w):
        x64 = x.double()
        return w * (x64 * torch.rsqrt(x64.square().mean(dim=-1, keepdim=True) + 1e-5)).to(dt)

    def rotate(x, cos, sin):
        half = torch.cat((-x[..., 64:], x[..., :64]), dim=-1)
        return x * cos + half * sin

    cos, sin = _rope(torch.tensor(used - 1, device=DEV), dt)
    for norms, members, k, v in parts:
        qkv = _linear64(norm(h, norms[0]), members["qkv"]).to(dt).view(batch, -1, 128)
        k[:, :, used - 1], v[:, :, used - 1] = rotate(qkv[:, 24:32], cos, sin), qkv[:, 32:]
        att = _attention64(rotate(qkv[:, :24], cos, sin), k, v, used).to(dt).view(batch, -1)
        h = h + _linear64(att, members["o"]).to(dt)
        gate, up = _linear64(norm(h, norms[1]), members["gate_up"]).to(dt).chunk(2, dim=1)
        act = (gate.double() * torch.sigmoid(gate.double())).to(dt) * up
        h = h + _linear64(act, members["down"]).to(dt)
    return (norm(h, final).double() @ table.double().t()).view(batch, 1, STEP_VOCAB)


@torch.inference_mode()
def exact(case, seed):
    if case["kind"] == "attention":
        return _attention64(*_attention_inputs(case, seed), case["used"])
    if case["kind"] == "step":
        return _step64(case, seed)
    num = _Numbers(seed)
    out = []
    for _, group in _projections(case):
        members = _group_weights(num, case, case["model"], group)
        out.append(_linear64(num.activation(case["rows"], _widths(case["model"], group)[0], DTYPES[case["dtype"]]),
                             members))
    return out
