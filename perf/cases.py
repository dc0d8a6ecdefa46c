"""What a user of this package has it do, as cases that can be timed and compared.

Three kinds of work, each through the public entry points (``tritonllm_amd`` and its ``modules``):

``token``   one decode step of a batch: token gather, per layer {RMSNorm + QKV + bias + rotary with the new k / v written
            into the KV cache, attention over the cache, out-projection + bias + residual, the MLP block's RMSNorm, the
            clamped SwiGLU of the routed experts}, the final RMSNorm and the logits of the whole vocabulary. A serving
            loop captures the step in a HIP graph and replays it per token (``graph``); a program that does not, or a
            batch whose shape has just changed, runs it call by call.
``prompt``  the same layers over the tokens of one or several prompts, or of a chat's next turn behind ``past`` tokens
            that are already in the cache. Prompts are not captured: their lengths differ.
``load``    MXFP4 expert weights of a checkpoint expanded to bf16.

The expert GEMMs and the routing are not part of this package: the SwiGLU reads activations of the experts' size.
Layers alternate between sliding-window and full attention; sizes are those of the 2880-wide model this repository is
built for (24 layers, 64 query and 8 KV heads of 64, vocabulary 201 088), and once a 4096-wide model, which takes the
kernels for general shapes.
"""
from __future__ import annotations

import math

import torch

import tritonllm_amd as T
from tritonllm_amd import modules

N_Q, N_KV, HD = 64, 8, 64
VOCAB = 201088
WINDOW = 128
EXPERTS_PER_TOKEN = 4
EPS = 1e-5
SM_SCALE = 0.125
BF16 = torch.bfloat16

TOKEN_LAYERS = 24
PROMPT_LAYERS = 4          # two windowed and two full layers: a prompt's layers repeat, and none of it leaves the caches warm


def _token(batch, context, *, slots=None, fp8=False, graph=True, hidden=2880, layers=TOKEN_LAYERS):
    """``context``: visible tokens, the new one included; ``slots``: the size of the preallocated KV cache."""
    return {"kind": "token", "batch": batch, "context": context, "slots": slots or context, "fp8": fp8, "graph": graph,
            "hidden": hidden, "layers": layers}


def _prompt(seqs, tokens, *, past=0, layers=PROMPT_LAYERS):
    return {"kind": "prompt", "seqs": seqs, "tokens": tokens, "past": past, "layers": layers}


def listed():
    return [
        # one user, early in a conversation: the weight stream and ~120 launches are all there is
        {"name": "token_1x300", **_token(1, 300, slots=4096)},
        # two users, the step issued call by call from Python (no graph)
        {"name": "token_2x700_eager", **_token(2, 700, slots=1024, graph=False)},
        # the batch this repository's benchmark is quoted at, at the original context length
        {"name": "token_8x4096", **_token(8, 4096)},
        # long contexts: the KV cache is most of what is read
        {"name": "token_8x32768", **_token(8, 32768)},
        # a continuous batch of odd size
        {"name": "token_49x1111", **_token(49, 1111, slots=2048)},
        # fp8 weights (ATTN_FP8, UNEMBED_FP8)
        {"name": "token_fp8_5x2000", **_token(5, 2000, slots=4096, fp8=True)},
        # a model of another width
        {"name": "token_wide_8x2048", **_token(8, 2048, hidden=4096, layers=8)},
        # a chat's next turn: few new tokens behind a conversation
        {"name": "prompt_97_after_1500", **_prompt(1, 97, past=1500)},
        # three short prompts of one length together, an odd number of rows
        {"name": "prompt_3x333", **_prompt(3, 333)},
        # one prompt of the ordinary benchmark length
        {"name": "prompt_2048", **_prompt(1, 2048)},
        # a long document
        {"name": "prompt_8192", **_prompt(1, 8192)},
        # the up-projection of all 32 experts of a layer, as a checkpoint holds it
        {"name": "load_mlp1", "kind": "load", "experts": 32, "rows": 5760},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.random()
    if kind < 0.5:
        batch = _log_int(rng, 1, 128)
        context = _log_int(rng, 64, min(32768, 262144 // batch))
        wide = rng.random() < 0.12
        return _token(batch, context, slots=context + rng.choice((0, 0, rng.randrange(1, context + 1))), fp8=rng.random() < 0.25,
                      graph=rng.random() < 0.8, hidden=4096 if wide else 2880, layers=8 if wide else TOKEN_LAYERS)
    if kind < 0.9:
        seqs = rng.choice((1, 1, 1, 2, 3, 4))
        tokens = _log_int(rng, 16, 8192 // seqs)
        past = _log_int(rng, 16, 4096) if seqs == 1 and tokens <= 2048 and rng.random() < 0.35 else 0
        return _prompt(seqs, tokens, past=past)
    return {"kind": "load", "experts": rng.randrange(1, 33), "rows": rng.choice((2880, 5760))}


# ------------------------------------------------------------------------------------------------------- inputs
def _normal(gen, *shape, std=1.0):
    return torch.empty(*shape, dtype=BF16, device="cuda").normal_(0.0, std, generator=gen)


def _scale(gen, hidden):
    return 1.0 + 0.1 * torch.randn(hidden, device="cuda", generator=gen)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "load":
        shape = (case["experts"], case["rows"], 90)
        return {"case": case,
                "blocks": torch.randint(0, 256, (*shape, 16), dtype=torch.uint8, device="cuda", generator=gen),
                "scales": torch.randint(112, 128, shape, dtype=torch.uint8, device="cuda", generator=gen),
                "out": torch.empty(case["experts"], case["rows"], 2880, dtype=BF16, device="cuda")}
    n, hidden = case["layers"], case.get("hidden", 2880)
    qkv_dim = (N_Q + 2 * N_KV) * HD
    s = {"case": case, "yarn": T.gpt_oss_yarn(), "table": _normal(gen, VOCAB, hidden),
         "attn_scale": [_scale(gen, hidden) for _ in range(n)], "mlp_scale": [_scale(gen, hidden) for _ in range(n)],
         "final_scale": _scale(gen, hidden), "sinks": [_normal(gen, N_Q) for _ in range(n)],
         "qkv_b": [_normal(gen, qkv_dim, std=0.02) for _ in range(n)]}
    qkv_w = [_normal(gen, qkv_dim, hidden, std=0.02) for _ in range(n)]
    out_w = [_normal(gen, hidden, N_Q * HD, std=0.02) for _ in range(n)]
    out_b = [_normal(gen, hidden, std=0.02) for _ in range(n)]
    if case["kind"] == "prompt":
        seqs, tokens, past = case["seqs"], case["tokens"], case["past"]
        rows = seqs * tokens
        s["ids"] = torch.randint(0, VOCAB, (rows,), dtype=torch.int32, device="cuda", generator=gen)
        s["positions"] = (past + torch.arange(tokens, device="cuda")).repeat(seqs)
        s["offset"] = torch.full((1,), past, dtype=torch.int64, device="cuda")
        s["k"] = [_normal(gen, seqs, past + tokens, N_KV, HD) for _ in range(n)]
        s["v"] = [_normal(gen, seqs, past + tokens, N_KV, HD) for _ in range(n)]
        s["q"] = torch.empty(rows, N_Q * HD, dtype=BF16, device="cuda")
        s["qkv_w"] = qkv_w
        s["out"] = []
        for w, b in zip(out_w, out_b):
            m = modules.OUT(N_Q * HD, hidden, device="cuda").requires_grad_(False)
            m.weight.copy_(w)
            m.bias.copy_(b)
            s["out"].append(m)
        s["experts_in"] = [_normal(gen, EXPERTS_PER_TOKEN * rows, 2 * hidden, std=2.0) for _ in range(n)]
        s["normed"] = [torch.empty(rows, hidden, dtype=BF16, device="cuda") for _ in range(n)]
        return s
    batch, context = case["batch"], case["context"]
    unembed = _normal(gen, VOCAB, hidden, std=0.02)
    if case["fp8"]:
        s["qkv_w"], s["qkv_ws"] = zip(*(T.quantize_fp8_rows(w) for w in qkv_w))
        s["out_w"], s["out_ws"] = zip(*(T.quantize_fp8_rows(w) for w in out_w))
        s["unembed"] = T.quantize_fp8_rows(unembed)
    else:
        s["qkv_w"], s["qkv_ws"] = qkv_w, [None] * n
        s["out_w"], s["out_ws"] = out_w, [None] * n
        s["unembed"] = (unembed, None)
    s["out_b"] = out_b
    s["next_ids"] = torch.randint(0, VOCAB, (batch,), dtype=torch.int32, device="cuda", generator=gen)
    s["ids"] = torch.zeros_like(s["next_ids"])
    s["offset"] = torch.zeros(1, dtype=torch.int64, device="cuda")
    s["k"] = _normal(gen, n, batch, case["slots"], N_KV, HD)
    s["v"] = _normal(gen, n, batch, case["slots"], N_KV, HD)
    s["experts_in"] = [_normal(gen, EXPERTS_PER_TOKEN * batch, 2 * hidden, std=2.0) for _ in range(n)]
    s["x"] = torch.empty(batch, hidden, dtype=BF16, device="cuda")
    s["normed"] = torch.empty(n, batch, hidden, dtype=BF16, device="cuda")
    s["act"] = torch.empty(n, EXPERTS_PER_TOKEN * batch, hidden, dtype=BF16, device="cuda")
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _token_layers(s)
        torch.cuda.current_stream().wait_stream(side)
        s["captured"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["captured"]):
            s["logits"] = _token_layers(s)
    return s


# ------------------------------------------------------------------------------------------------------- passes
def _window(layer):
    return WINDOW if layer % 2 == 0 else None


def _token_layers(s):
    case = s["case"]
    batch = case["batch"]
    x = T.embedding_forward(s["ids"], s["table"], out=s["x"]).view(batch, 1, -1)
    for l in range(case["layers"]):
        q = T.qkv_rope_cache_decode_forward(x, s["qkv_w"][l], s["qkv_b"][l], None, None, 131072, s["k"][l], s["v"][l], s["offset"], N_Q, N_KV,
                                            HD, s["qkv_ws"][l], yarn=s["yarn"], norm_scale=s["attn_scale"][l], norm_eps=EPS)
        o = T.attention_decode(q.view(batch, 1, N_KV, N_Q // N_KV, HD), s["k"][l], s["v"][l], s["sinks"][l], SM_SCALE, _window(l), s["offset"])
        x = T.out_residual_decode_forward(o, s["out_w"][l], s["out_b"][l], x, s["out_ws"][l])
        T.rmsnorm_forward(x, s["mlp_scale"][l], EPS, out=s["normed"][l].view(batch, 1, -1))
        T.swiglu(s["experts_in"][l], out=s["act"][l])
    t = T.rmsnorm_forward(x, s["final_scale"], EPS)
    return T.unembedding_decode_forward(t, *s["unembed"])


def _run_token(s):
    case = s["case"]
    s["ids"].copy_(s["next_ids"])
    s["offset"].fill_(case["context"] - 1)
    if case["graph"]:
        s["captured"].replay()
        logits = s["logits"]
    else:
        logits = _token_layers(s)
    new = case["context"] - 1
    return {"logits": logits, "x": s["x"], "k": s["k"][:, :, new], "v": s["v"][:, :, new], "normed": s["normed"], "act": s["act"]}


def _run_prompt(s):
    case = s["case"]
    seqs, tokens, past = case["seqs"], case["tokens"], case["past"]
    rows = seqs * tokens
    acts = []
    for l in range(case["layers"]):
        # the new tokens' rows of the cache (one run of rows: several prompts start with an empty one)
        k_new, v_new = (c[l][:, past:].view(rows, N_KV * HD) for c in (s["k"], s["v"]))
        if l == 0:
            x, t = T.embedding_rmsnorm_forward(s["ids"], s["table"], s["attn_scale"][0], EPS)
            T.qkv_rope_forward(t, s["qkv_w"][0], s["qkv_b"][0], N_Q, N_KV, HD, yarn=s["yarn"], positions=s["positions"],
                               out=(s["q"], k_new, v_new))
        else:
            T.qkv_rope_forward(x, s["qkv_w"][l], s["qkv_b"][l], N_Q, N_KV, HD, yarn=s["yarn"], positions=s["positions"],
                               out=(s["q"], k_new, v_new), norm_scale=s["attn_scale"][l], norm_eps=EPS)
        o = T.attention(s["q"].view(seqs, tokens, N_KV, N_Q // N_KV, HD), s["k"][l], s["v"][l], s["sinks"][l], SM_SCALE, _window(l), s["offset"])
        x = x + s["out"][l](o).view(rows, -1)
        T.rmsnorm_forward(x, s["mlp_scale"][l], EPS, out=s["normed"][l])
        acts.append(T.swiglu(s["experts_in"][l]))
    t = T.rmsnorm_forward(x, s["final_scale"], EPS)
    return {"x": x, "final": t, "k": [k[:, past:] for k in s["k"]], "v": [v[:, past:] for v in s["v"]], "normed": s["normed"], "act": acts}


def run(state):
    kind = state["case"]["kind"]
    if kind == "load":
        return T.mxfp4_dequant(state["blocks"], state["scales"], out=state["out"])
    return _run_token(state) if kind == "token" else _run_prompt(state)


# ------------------------------------------------------------------------------------------------------- what a pass cannot do without
def _visible(past, tokens, window):
    """(query, key) pairs that attention of ``tokens`` queries behind ``past`` keys looks at, and the keys among them."""
    if window is None:
        return tokens * past + tokens * (tokens + 1) // 2, past + tokens
    return sum(min(past + i + 1, window) for i in range(tokens)), min(past + tokens, tokens + window - 1)


def work(case):
    if case["kind"] == "load":
        blocks = case["experts"] * case["rows"] * 90
        return {"bytes": blocks * (16 + 1 + 64), "flops": 0}
    token = case["kind"] == "token"
    n, hidden = case["layers"], case.get("hidden", 2880)
    seqs, tokens, past = (case["batch"], 1, case["context"] - 1) if token else (case["seqs"], case["tokens"], case["past"])
    rows, qkv_dim, q_dim = seqs * tokens, (N_Q + 2 * N_KV) * HD, N_Q * HD
    wb = 1 if token and case["fp8"] else 2
    nbytes = rows * (4 + 4 * hidden) + n * 4 * hidden * 2                       # ids, gathered rows, x, norm scales
    flops = 0
    for l in range(n):
        pairs, keys = _visible(past, tokens, _window(l))
        nbytes += qkv_dim * hidden * wb + q_dim * hidden * wb + 2 * (qkv_dim + hidden)      # the two weights and biases
        nbytes += seqs * keys * 2 * N_KV * HD * 2                                # k and v of the visible context (new ones among them)
        nbytes += rows * hidden * 2                                              # the MLP block's normed rows
        nbytes += rows * EXPERTS_PER_TOKEN * 3 * hidden * 2                      # SwiGLU in and out
        flops += 2 * rows * hidden * (qkv_dim + q_dim) + 4 * seqs * pairs * N_Q * HD
    if token:
        nbytes += VOCAB * hidden * wb + rows * VOCAB * 2
        flops += 2 * rows * VOCAB * hidden
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Outputs are bf16 and run through up to 24 layers, each rounding its operands to bf16: sums in another order move
    some of them by one place, and what follows by as much. With every projection and softmax summed another way (the
    norm as a launch of its own, other context splits, the other QKV kernel, out-projection and prompt attention in
    fp32) the outputs of 17 cases were off by 0.5 - 1.2e-2 (2-norm) and by at most 7.3e-2 (single values)."""
    if case["kind"] == "load":
        return "exact"
    return {"rel": 3e-2, "max": 0.25}
