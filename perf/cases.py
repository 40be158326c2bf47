"""The work that users of the quantized-linear library have it do, as timed cases.

A program that serves a model holds its weights resident (`Context.weights`)
and calls one linear layer after another: one activation row per token while it
decodes, a few rows when it batches sequences, tens to thousands of rows for a
prompt. So most cases here are a short stack of `layers` weights of one shape,
each with its own input and output, called in order; several layers, because a
model's weights are read from memory once per token and not from a cache.
Device calls (`Weights.linear_device`) run on a stream of the program, host
calls (`Weights.linear`) are the synchronous call of the `KernelBackend`
contract. The decoder case is a conversation on the device-resident Qwen3
decoder: a prompt, a generated reply, and the next turn's tokens up to their
logits.

Sizes: the Qwen3-8B projections (hidden 4096, k/v 1024, intermediate 12288) and
the 4096 x 14336 feed-forward shapes that bench.py measures, and for drawn cases
everything around them. Weights are N(0, 0.02^2), the K-quants' with 0.5 % of
N(0, 0.2^2) outliers, quantized here in plain torch to the formats' blocks with
f16 scales as files hold them; activations are N(0, 1).

The bit-identical EXACT mode and the dequantizer are checking aids and are not
timed.
"""
import math

import numpy as np
import torch

import quantinfer_amd as qa

QTYPE = {"f32": qa.F32, "q8_0": qa.Q8_0, "q4_0": qa.Q4_0, "q4_k": qa.Q4_K, "q5_k": qa.Q5_K, "q6_k": qa.Q6_K}
LAYOUT = {"row_major": qa.ROW_MAJOR, "output_rows": qa.OUTPUT_ROWS}
MODE = {"auto": qa.MODE_AUTO, "f32": qa.MODE_F32}
WIRE_BITS = {"f32": 32.0, "q8_0": 8.5, "q4_0": 4.5, "q4_k": 4.5, "q5_k": 5.5, "q6_k": 6.5625}
GEMM_ROWS = 128  # AUTO mode takes f16 operands from here (include/qi_hip.h)


def _linear(name, weight, m, k, n, layers, layout="output_rows", mode="f32", call="device"):
    return dict(name=name, kind="linear", call=call, weight=weight, layout=layout, mode=mode, m=m, k=k, n=n,
                layers=layers)


def listed():
    return [
        # k/v projection of one decoded token: the smallest call, a matter of latency
        _linear("decode_kv_q4_0", "q4_0", 1, 4096, 1024, 8),
        # feed-forward up projection of one decoded token: the headline shape
        _linear("decode_up_q4_k", "q4_k", 1, 4096, 14336, 3),
        # the same kind of call through the host contract: tensors in host memory, synchronous
        _linear("host_decode_q8_0", "q8_0", 1, 4096, 4096, 3, call="host"),
        # feed-forward down projection for a batch of sequences
        _linear("batch_down_q5_k", "q5_k", 8, 14336, 4096, 2),
        # gate projection for a larger batch or a speculated run of tokens
        _linear("batch_gate_q4_0", "q4_0", 16, 4096, 12288, 2),
        # prompts in the default mode: f16 operands on the matrix cores
        _linear("prompt_gate_q4_k", "q4_k", 512, 4096, 12288, 1, mode="auto"),
        _linear("prompt_down_q8_0", "q8_0", 2048, 12288, 4096, 1, mode="auto"),
        # a prompt of ragged length with f32 accuracy (what keeps greedy tokens those of the CPU)
        _linear("prompt_f32_q6_k", "q6_k", 333, 4096, 14336, 1),
        # QuantInfer's own layout, blocks along N: a decoded token and a short prompt
        _linear("row_major_decode_q4_k", "q4_k", 1, 4096, 14336, 2, layout="row_major"),
        _linear("row_major_prompt_q8_0", "q8_0", 130, 4096, 4096, 1, layout="row_major"),
        # dense f32 weights (a model that is not quantized): a prompt
        _linear("dense_prompt_f32", "f32", 300, 2048, 8192, 1, layout="row_major"),
        # a conversation on the decoder, four layers of the 8B shape
        dict(name="decoder_8b_width", kind="decoder", hidden=4096, intermediate=12288, heads=32, kv_heads=8,
             head_dim=128, model_layers=4, vocab=32768, prompt=300, new=48, turn=7, mode="f32"),
    ]


def _log(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _steps(v, step):
    return max(step, int(v / step + 0.5) * step)


def draw(rng):
    kind = rng.choice(["decode", "decode", "host", "batch", "batch", "few", "prompt", "prompt", "prompt_f32",
                       "row_major", "row_major", "dense", "decoder"])
    weight = rng.choice(["q8_0", "q4_0", "q4_k", "q5_k", "q6_k"])
    k = _steps(_log(rng, 512, 14336), 256)
    n = min(int(_log(rng, 512, 24576)), 4096 * 14336 // k)
    if rng.random() < 0.7:
        n = _steps(n, 64)  # model shapes; else a ragged output count
    if kind == "decoder":
        hd = rng.choice([64, 128])
        kv = rng.choice([2, 4, 8])
        heads = kv * rng.choice([2, 4])
        # hidden sizes and head counts as in the decoder's tests and up to the 8B width
        hidden = _steps(_log(rng, 512, 4096), 256)
        return dict(kind=kind, hidden=hidden, intermediate=3 * hidden, heads=heads, kv_heads=kv, head_dim=hd,
                    model_layers=rng.randint(1, 4), vocab=rng.randint(1000, 32768), prompt=int(_log(rng, 9, 400)),
                    new=rng.randint(8, 40), turn=rng.randint(1, 16), mode="f32")
    case = dict(kind="linear", call="device", weight=weight, layout="output_rows", mode="f32", m=1, k=k, n=n,
                layers=rng.randint(1, 4))
    if kind == "host":
        case.update(call="host", m=rng.choice([1, 1, 1, 2, 5, 16, 40]), mode="auto", layers=2)
    elif kind == "batch":
        case.update(m=rng.randint(2, 16), layers=2)
    elif kind == "few":
        case.update(m=rng.randint(17, GEMM_ROWS - 1), layers=1, mode=rng.choice(["f32", "auto"]))
    elif kind == "prompt":
        case.update(m=int(_log(rng, GEMM_ROWS, 2048)), layers=1, mode="auto")
    elif kind == "prompt_f32":
        case.update(m=int(_log(rng, GEMM_ROWS, 1024)), layers=1)
    elif kind == "row_major":
        m = rng.choice([1, 2, int(_log(rng, 3, 16)), int(_log(rng, 17, 512))])
        case.update(m=m, n=_steps(n, 256), layers=2 if m < 17 else 1, layout="row_major",
                    mode=rng.choice(["f32", "auto"]))
    elif kind == "dense":
        case.update(weight="f32", layout="row_major", m=rng.choice([1, int(_log(rng, 2, 16)), int(_log(rng, 17, 512))]),
                    k=_steps(k, 4), n=_steps(min(n, 14336), 4), layers=1)
    elif kind == "decode" and weight in ("q8_0", "q4_0") and rng.random() < 0.2:
        case.update(k=_steps(k + 96, 32))  # whole blocks, but not whole 256-element units
    return case


# ---------------------------------------------------------------- blocks
# The formats' logical blocks (include/qi_hip.h) made and read back in torch.
# A matrix is [rows, columns] with the blocks along the columns.

def _bytes(t):
    return t.contiguous().view(torch.uint8).reshape(t.shape[0], -1)


def _f16(t):
    return t.to(torch.float16).to(torch.float32)


def _div(a, b):
    return torch.where(b == 0, torch.zeros_like(a), a / torch.where(b == 0, torch.ones_like(b), b))


def _u8(t):
    return t.to(torch.int32).to(torch.uint8)


def _pack_6bit(sc, mn):
    sc, mn = sc.to(torch.int32), mn.to(torch.int32)
    return torch.cat([sc[:, :4] | (sc[:, 4:] >> 4 << 6), mn[:, :4] | (mn[:, 4:] >> 4 << 6),
                      (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1).to(torch.uint8)


def _quantize(weight, w):
    """(bytes [blocks, block size] u8, the weights they stand for in f64), both on w's device."""
    f64 = torch.float64
    if weight in ("q8_0", "q4_0"):
        b = w.reshape(-1, 32)
        top = 127 if weight == "q8_0" else 7
        d = _f16(b.abs().amax(1, keepdim=True) / top)
        q = torch.round(_div(b, d)).clamp_(-top - (weight == "q4_0"), top)
        codes = q.to(torch.int8) if weight == "q8_0" else _u8(q + 8)
        return torch.cat([_bytes(d), _bytes(codes)], 1), (d.to(f64) * q.to(f64)).reshape(w.shape)
    if weight == "q6_k":
        b = w.reshape(-1, 16, 16)
        step = b.abs().amax(2) / 31
        d = _f16(step.amax(1, keepdim=True) / 127)
        sc = torch.round(_div(step, d)).clamp_(1, 127)
        q = torch.round(_div(b, (d * sc)[:, :, None])).clamp_(-32, 31)
        u = (q + 32).to(torch.int32).reshape(-1, 2, 4, 32)
        low = torch.cat([(u[:, :, 0] & 15) | (u[:, :, 2] & 15) << 4, (u[:, :, 1] & 15) | (u[:, :, 3] & 15) << 4], 2)
        high = (u >> 4)[:, :, 0] | (u >> 4)[:, :, 1] << 2 | (u >> 4)[:, :, 2] << 4 | (u >> 4)[:, :, 3] << 6
        out = torch.cat([_bytes(d), _bytes(sc.to(torch.int8)), _bytes(low.to(torch.uint8)),
                         _bytes(high.to(torch.uint8))], 1)
        return out, ((d.to(f64) * sc.to(f64))[:, :, None] * q.to(f64)).reshape(w.shape)
    top = 15 if weight == "q4_k" else 31
    b = w.reshape(-1, 8, 32)
    low, high = b.amin(2).clamp_max(0), b.amax(2)
    step = (high - low).clamp_min(0) / top
    d, dmin = _f16(step.amax(1, keepdim=True) / 63), _f16(-low.amin(1, keepdim=True) / 63)
    sc, mn = torch.round(_div(step, d)).clamp_(0, 63), torch.round(_div(-low, dmin)).clamp_(0, 63)
    q = torch.round(_div(b + (dmin * mn)[:, :, None], (d * sc)[:, :, None])).clamp_(0, top)
    u = q.to(torch.int32)
    pairs = (u & 15).reshape(-1, 4, 2, 32)
    parts = [_bytes(d), _bytes(dmin), _pack_6bit(sc, mn)]
    if weight == "q5_k":
        parts.append(_bytes(((u >> 4) << torch.arange(8, device=w.device)[None, :, None]).sum(1).to(torch.uint8)))
    parts.append(_bytes((pairs[:, :, 0] | pairs[:, :, 1] << 4).to(torch.uint8)))
    value = (d.to(f64) * sc.to(f64))[:, :, None] * q.to(f64) - (dmin.to(f64) * mn.to(f64))[:, :, None]
    return torch.cat(parts, 1), value.reshape(w.shape)


def _blocks(weight, w):
    """Host blocks of a [rows, columns] matrix, as Context.weights takes them."""
    if weight == "f32":
        return w.reshape(-1).cpu().numpy()
    return _quantize(weight, w)[0].cpu().numpy().reshape(-1).view(qa.BLOCK_DTYPES[QTYPE[weight]])


def _normal(gen, rows, cols, std=1.0, outliers=False):
    w = torch.randn(rows, cols, generator=gen, device="cuda") * std
    if outliers:
        w = torch.where(torch.rand(rows, cols, generator=gen, device="cuda") < 0.005, w * 10, w)
    return w


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _layer(case, seed, index):
    """Weight matrix [rows, columns] in its layout's order and input [m, k] of one layer."""
    gen = _generator(1000 * seed + index)
    rows, cols = (case["n"], case["k"]) if case["layout"] == "output_rows" else (case["k"], case["n"])
    w = _normal(gen, rows, cols, 0.02, case["weight"] in ("q4_k", "q5_k", "q6_k"))
    return w, _normal(gen, case["m"], case["k"])


# ---------------------------------------------------------------- decoder
NORMS = ("input_layernorm", "q_norm", "k_norm", "post_attention_layernorm")


def _config(case):
    return dict(vocab_size=case["vocab"], hidden_size=case["hidden"], intermediate_size=case["intermediate"],
                num_hidden_layers=case["model_layers"], num_attention_heads=case["heads"],
                num_key_value_heads=case["kv_heads"], head_dim=case["head_dim"], max_position_embeddings=1024,
                rms_norm_eps=1e-6, rope_theta=1e6)


def _decoder_weights(case, seed):
    """Yields ("embedding", w), then each layer's parts, then ("final_norm", w) and ("head", w), on the GPU."""
    gen = _generator(seed)
    h, hd = case["hidden"], case["head_dim"]
    qs, ks, i = case["heads"] * hd, case["kv_heads"] * hd, case["intermediate"]
    norm = lambda d: 1 + 0.05 * torch.randn(d, generator=gen, device="cuda")  # noqa: E731
    yield "embedding", _normal(gen, case["vocab"], h, 0.02)
    for _ in range(case["model_layers"]):
        layer = dict(zip(NORMS, (norm(h), norm(hd), norm(hd), norm(h))))
        for name, n, k in (("q_proj", qs, h), ("k_proj", ks, h), ("v_proj", ks, h), ("o_proj", h, qs),
                           ("gate_proj", i, h), ("up_proj", i, h), ("down_proj", h, i)):
            layer[name] = _normal(gen, n, k, 0.02)
        yield "layer", layer
    yield "final_norm", norm(h)
    yield "head", _normal(gen, case["vocab"], h, 0.02)


def _tokens(case, seed, salt, count):
    return np.random.default_rng([seed, salt]).integers(0, case["vocab"], count).astype(np.int32)


def _prepare_decoder(case, seed):
    model = qa.Qwen3(_context(), _config(case))
    index, final_norm = 0, None
    for name, w in _decoder_weights(case, seed):
        if name == "embedding":
            model.set_embedding(w.cpu().numpy())
        elif name == "layer":
            # as GGUF files of the 8B shape: Q4_K projections
            model.set_layer(index, {p: w[p].cpu().numpy() if p in NORMS else
                                    (qa.Q4_K, qa.OUTPUT_ROWS, _blocks("q4_k", w[p])) for p in w})
            index += 1
        elif name == "final_norm":
            final_norm = w.cpu().numpy()
        else:
            model.set_output(final_norm, (qa.Q6_K, qa.OUTPUT_ROWS, _blocks("q6_k", w)))
    model.set_mode(MODE[case["mode"]])
    cache = model.kv_cache(case["prompt"] + case["new"] + case["turn"] + 1)
    return dict(model=model, cache=cache, new=case["new"], prompt=_tokens(case, seed, 1, case["prompt"]),
                turn=_tokens(case, seed, 2, case["turn"]))


def _exact_decoder(case, seed):
    f64 = torch.float64
    hq, hk, hd, eps = case["heads"], case["kv_heads"], case["head_dim"], 1e-6
    layers, part = [], {}
    for name, w in _decoder_weights(case, seed):
        if name == "layer":
            layers.append({p: w[p].to(f64) if p in NORMS else _quantize("q4_k", w[p])[1] for p in w})
        else:
            part[name] = _quantize("q6_k", w)[1] if name == "head" else w.to(f64)
    half = hd // 2
    # the model's rotation angles are f32 numbers
    inv = torch.tensor(1e6, dtype=torch.float32) ** -(2 * torch.arange(half, dtype=torch.float32) / hd)
    total = case["prompt"] + case["new"] + case["turn"]
    angle = (torch.arange(total, dtype=torch.float32)[:, None] * inv[None, :]).to(f64).cuda()
    keys = [torch.zeros(hk, total, hd, dtype=f64, device="cuda") for _ in layers]
    values = [torch.zeros(hk, total, hd, dtype=f64, device="cuda") for _ in layers]

    def rms(x, w):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w

    def rope(x, at):  # [t, heads, hd]
        c, s = torch.cos(angle[at:at + x.shape[0]])[:, None], torch.sin(angle[at:at + x.shape[0]])[:, None]
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * c - b * s, a * s + b * c], -1)

    def forward(tokens, at):
        t = len(tokens)
        h = part["embedding"][torch.as_tensor(np.asarray(tokens), device="cuda", dtype=torch.long)]
        mask = torch.arange(at + t, device="cuda")[None, :] > (at + torch.arange(t, device="cuda"))[:, None]
        for w, kc, vc in zip(layers, keys, values):
            x = rms(h, w["input_layernorm"])
            q = rope(rms((x @ w["q_proj"].T).reshape(t, hq, hd), w["q_norm"]), at)
            kc[:, at:at + t] = rope(rms((x @ w["k_proj"].T).reshape(t, hk, hd), w["k_norm"]), at).transpose(0, 1)
            vc[:, at:at + t] = (x @ w["v_proj"].T).reshape(t, hk, hd).transpose(0, 1)
            heads = []
            for j in range(hq):
                score = (q[:, j] @ kc[j * hk // hq, :at + t].T) / math.sqrt(hd)
                heads.append(torch.softmax(score.masked_fill(mask, -math.inf), -1) @ vc[j * hk // hq, :at + t])
            h = h + torch.cat(heads, -1) @ w["o_proj"].T
            x = rms(h, w["post_attention_layernorm"])
            h = h + (torch.nn.functional.silu(x @ w["gate_proj"].T) * (x @ w["up_proj"].T)) @ w["down_proj"].T
        return rms(h[-1:], part["final_norm"]) @ part["head"].T

    logits, at, ids = forward(_tokens(case, seed, 1, case["prompt"]), 0), case["prompt"], []
    for _ in range(case["new"]):
        ids.append(int(logits.argmax()))
        logits = forward(ids[-1:], at)
        at += 1
    logits = forward(_tokens(case, seed, 2, case["turn"]), at)
    return dict(ids=np.asarray(ids), logits=logits[0].cpu().numpy())


# ---------------------------------------------------------------- what is timed
_KEPT = {}


def _context():
    """The program's one open device, kept for its life."""
    if "context" not in _KEPT:
        _KEPT["context"] = qa.Context(0)
    return _KEPT["context"]


def _stream():
    if "stream" not in _KEPT:
        _KEPT["stream"] = torch.cuda.Stream()
    return _KEPT["stream"].cuda_stream


def prepare(case, seed):
    if case["kind"] == "decoder":
        return _prepare_decoder(case, seed)
    calls = []
    for index in range(case["layers"]):
        w, x = _layer(case, seed, index)
        held = _context().weights(QTYPE[case["weight"]], LAYOUT[case["layout"]], case["k"], case["n"],
                                  _blocks(case["weight"], w))
        if case["call"] == "host":
            calls.append((held, x.cpu().numpy(), None))
        else:
            calls.append((held, x, torch.zeros(case["m"], case["n"], device="cuda")))
    return dict(calls=calls, m=case["m"], mode=MODE[case["mode"]], stream=_stream())


def run(state):
    if "model" in state:
        model, cache = state["model"], state["cache"]
        cache.reset()
        ids = model.generate(cache, state["prompt"], state["new"])
        logits, _ = model.forward(cache, state["turn"])
        return dict(ids=np.asarray(ids), logits=logits)
    out = []
    for weights, x, y in state["calls"]:
        if y is None:
            out.append(weights.linear(x, state["mode"]))
        else:
            weights.linear_device(x.data_ptr(), state["m"], y.data_ptr(), state["mode"], state["stream"])
            out.append(y)
    return out


def exact(case, seed):
    if case["kind"] == "decoder":
        return _exact_decoder(case, seed)
    out = []
    for index in range(case["layers"]):
        w, x = _layer(case, seed, index)
        value = w.to(torch.float64) if case["weight"] == "f32" else _quantize(case["weight"], w)[1]
        out.append((x.to(torch.float64) @ (value.T if case["layout"] == "output_rows" else value)).cpu().numpy())
    return out


def work(case):
    if case["kind"] == "decoder":
        h, i, hd, total = case["hidden"], case["intermediate"], case["head_dim"], case["prompt"] + case["new"]
        qs, ks = case["heads"] * hd, case["kv_heads"] * hd
        layer = h * (qs + 2 * ks) + qs * h + 3 * h * i
        weights = (layer * case["model_layers"] * WIRE_BITS["q4_k"] + h * case["vocab"] * WIRE_BITS["q6_k"]) / 8
        steps = case["new"] + 2  # the prompt and the next turn read the weights once each
        # every step reads the cached keys and values before it
        cached = 2 * 4 * ks * case["model_layers"] * (case["new"] * (case["prompt"] + case["new"] / 2) + total)
        tokens = total + case["turn"]
        return dict(bytes=steps * weights + cached,
                    flops=2 * layer * case["model_layers"] * tokens + 2 * h * case["vocab"] * steps)
    m, k, n = case["m"], case["k"], case["n"]
    return dict(bytes=case["layers"] * (k * n * WIRE_BITS[case["weight"]] / 8 + 4 * m * (k + n)),
                flops=case["layers"] * 2 * m * k * n)


def tolerance(case):
    # Measured against exact(): the decoder's logits 1.5e-6, f16 operands 2.9e-4; f32 calls 1e-7 to 2.5e-7 in short
    # exact sums, where one f32 sum over k = 4096 to 14336 in another order shows 1e-6 to 2e-6.
    if case["kind"] == "decoder":
        return {"rel": 1e-5, "max": 1e-4}
    f16 = case["mode"] == "auto" and case["layout"] == "output_rows" and case["m"] >= GEMM_ROWS
    return {"rel": 1.2e-3, "max": 1e-2} if f16 else {"rel": 4e-6, "max": 4e-5}
