"""What is timed when this framework is measured: the linear work of the 8B backbone on packed GGUF weights.

Every case goes through the entry points a user's program calls: the module that a checkpoint's Linear becomes
(``GGUFLinear``), a decoder layer as the loader leaves it (q / k / v on one stacked weight, the fused MLP forward), the
helpers that fold norms and residual adds in, the launcher for mixed text and image rows, the greedy token step on the
vocabulary projection, and the standalone decoder.  Attention, rope and sampling belong to the model that uses the
framework and are not here; streaming layers from host memory is bound by the host link and is not here either.

Kinds of case
* ``linear``     one projection, ``rows`` activation rows, with or without bias;
* ``layers``     ``layers`` decoder layers one after the other, the seven projections of each as the loader leaves them;
* ``folded``     the same layers through the helpers that take the layer's norms and residual adds;
* ``mixed``      the seven projections of one layer with text rows routed to one weight set and image rows to another,
                 the text rows first (``text`` of them) or scattered;
* ``greedy``     the arg-max over the vocabulary projection;
* ``dequantize`` one packed matrix decoded.

Several layers (or several matrices) stand behind each pass with few rows, because a decoding model reads every layer
once per token: weights come from memory, not from a cache that the previous pass left warm.
"""
import math

import torch

from sensenova_u1_amd import GGUFLinear, GGUFParameter, dequantize_gguf_tensor, fuse_gated_mlps, gated_mlp, grouped_linear
from sensenova_u1_amd import set_gguf2meta_model, stack_shared_input_projections, synthetic
from sensenova_u1_amd.modality import FusedProjections
from sensenova_u1_amd.ops import GGML_QUANT_SIZES

TYPES = {"q4_0": 2, "q4_1": 3, "q5_0": 6, "q5_1": 7, "q8_0": 8, "q2_k": 10, "q3_k": 11, "q4_k": 12, "q5_k": 13, "q6_k": 14, "bf16": 30}
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
EPS = 1e-6


def listed():
    model = {"hidden": 4096, "inter": 12288, "kv": 1024}
    q8 = {"type": "q8_0", "down_type": "q8_0"}
    kq = {"type": "q4_k", "down_type": "q6_k"}
    return [
        # the smallest call: one square projection for one token (latency, host time)
        {"name": "linear_1row_q8_0", "kind": "linear", "rows": 1, "n": 4096, "k": 4096, "type": "q8_0", "bias": False},
        # text decode, one token: the think loop over an 8-bit checkpoint as the loader leaves it
        {"name": "decode_1row_q8_0", "kind": "layers", "rows": 1, "layers": 3, **model, **q8},
        # the same over a 4-bit checkpoint, by a program that folds norms and residual adds in
        {"name": "decode_1row_k_quants", "kind": "folded", "rows": 1, "layers": 6, **model, **kq},
        # batched decode: sixteen sequences
        {"name": "decode_16rows_q8_0", "kind": "layers", "rows": 16, "layers": 3, **model, **q8},
        # a short prompt
        {"name": "prompt_40rows_q8_0", "kind": "layers", "rows": 40, "layers": 3, **model, **q8},
        # an ordinary prompt, an odd number of tokens
        {"name": "prompt_203rows_k_quants", "kind": "layers", "rows": 203, "layers": 4, **model, **kq},
        # a long prompt
        {"name": "prompt_509rows_q8_0", "kind": "layers", "rows": 509, "layers": 3, **model, **q8},
        # image tokens of a 1024 x 1024 picture, one denoising step
        {"name": "image_1024rows_k_quants", "kind": "layers", "rows": 1024, "layers": 2, **model, **kq},
        # image tokens of a 2048 x 2048 picture
        {"name": "image_4096rows_q8_0", "kind": "layers", "rows": 4096, "layers": 1, **model, **q8},
        # a prompt and a picture in one pass, each on its own tower's weights
        {"name": "mixed_512_4096rows_q8_0", "kind": "mixed", "rows": 4608, "text": 512, "scattered": False, **model, **q8},
        # greedy next token over the vocabulary
        {"name": "greedy_1row_q6_k", "kind": "greedy", "rows": 1, "n": 151936, "k": 4096, "type": "q6_k"},
        # a program that wants the weights themselves
        {"name": "dequantize_q4_k", "kind": "dequantize", "n": 12288, "k": 4096, "count": 3, "type": "q4_k", "out": "fp16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    # the model's own widths in half of the draws, other widths of the same proportions in the rest
    hidden, inter, kv = rng.choice([(4096, 12288, 1024)] * 3 + [(2048, 6144, 512), (2560, 9728, 1024), (3584, 8960, 512)])
    # the mixes that checkpoints of this kind come in, each as (attention and gate / up, down)
    kind_t, down_t = rng.choice([("q8_0", "q8_0")] * 3 + [("q4_k", "q6_k")] * 3 + [("q5_k", "q6_k"), ("q6_k", "q6_k"), ("q4_k", "q4_k"),
                                 ("q4_0", "q4_0"), ("q5_0", "q5_0"), ("q3_k", "q4_k")])
    kind = rng.choice(["layers"] * 6 + ["folded", "linear", "linear", "mixed", "greedy", "dequantize"])
    one = rng.choice([kind_t, kind_t, "q4_1", "q5_1", "q2_k", "q3_k", "q6_k", "bf16"])
    if kind == "linear":
        n = rng.choice([hidden, inter, kv, rng.randrange(96, inter)])
        k = rng.choice([hidden, inter, 256 * rng.randrange(1, 48)])
        return {"kind": kind, "rows": _log_int(rng, 1, 4096), "n": n, "k": k, "type": one, "bias": rng.random() < 0.25}
    if kind == "dequantize":
        return {"kind": kind, "n": _log_int(rng, 512, inter), "k": rng.choice([hidden, inter]), "count": 3,
                "type": one if one != "bf16" else kind_t, "out": rng.choice(sorted(DTYPES))}
    if kind == "greedy":
        return {"kind": kind, "rows": _log_int(rng, 1, 16), "n": rng.choice([151936, rng.randrange(32000, 151936)]), "k": hidden,
                "type": one if one != "bf16" else kind_t}
    shape = {"hidden": hidden, "inter": inter, "kv": kv, "type": kind_t, "down_type": down_t}
    if kind == "mixed":
        rows = _log_int(rng, 128, 4608)
        return {"kind": kind, "rows": rows, "text": rng.randrange(1, rows), "scattered": rng.random() < 0.5, **shape}
    rows = _log_int(rng, 1, 16) if kind == "folded" else _log_int(rng, 1, 4096)
    return {"kind": kind, "rows": rows, "layers": 3 if rows <= 512 else 2 if rows <= 1024 else 1, **shape}


class _MLP(torch.nn.Module):
    def __init__(self, hidden, inter):
        super().__init__()
        self.gate_proj = torch.nn.Linear(hidden, inter, bias=False)
        self.up_proj = torch.nn.Linear(hidden, inter, bias=False)
        self.down_proj = torch.nn.Linear(inter, hidden, bias=False)
        self.act_fn = torch.nn.SiLU()

    def forward(self, x):
        return self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))


class _Layer(torch.nn.Module):
    def __init__(self, hidden, inter, kv):
        super().__init__()
        self.q_proj = torch.nn.Linear(hidden, hidden, bias=False)
        self.k_proj = torch.nn.Linear(hidden, kv, bias=False)
        self.v_proj = torch.nn.Linear(hidden, kv, bias=False)
        self.o_proj = torch.nn.Linear(hidden, hidden, bias=False)
        self.mlp = _MLP(hidden, inter)


def _parameter(qtype, n, k, seed):
    return GGUFParameter(synthetic.make_packed(TYPES[qtype], n, k, seed=seed, device="cuda"), quant_type=TYPES[qtype])


def _module(qtype, n, k, seed, bias=False):
    mod = GGUFLinear(k, n, bias=bias, compute_dtype=torch.bfloat16, device="meta")
    mod.weight = _parameter(qtype, n, k, seed)
    if bias:
        mod.bias = torch.nn.Parameter(synthetic.make_activations(1, n, seed=seed + 1, device="cuda")[0], requires_grad=False)
    return mod


def _layer_shapes(case):
    h, i, kv = case["hidden"], case["inter"], case["kv"]
    return {"q_proj": (h, h), "k_proj": (kv, h), "v_proj": (kv, h), "o_proj": (h, h),
            "mlp.gate_proj": (i, h), "mlp.up_proj": (i, h), "mlp.down_proj": (h, i)}


def _layers(case, count, seed):
    """``count`` layers built without storage and filled from packed weights, as a checkpoint's loading does."""
    with torch.device("meta"):
        model = torch.nn.ModuleList([_Layer(case["hidden"], case["inter"], case["kv"]) for _ in range(count)])
    weights = {}
    for i in range(count):
        for j, (name, (n, k)) in enumerate(_layer_shapes(case).items()):
            qtype = case["down_type"] if name == "mlp.down_proj" else case["type"]
            weights[f"{i}.{name}.weight"] = _parameter(qtype, n, k, seed * 1000 + i * 10 + j)
    return set_gguf2meta_model(model, weights, torch.bfloat16, torch.device("cuda")).eval()


def prepare(case, seed):
    kind = case["kind"]
    seed = seed * 7919 + 17
    state = {"case": case}
    if kind == "dequantize":
        state["weights"] = [_parameter(case["type"], case["n"], case["k"], seed + i) for i in range(case["count"])]
        return state
    rows = case["rows"]
    if kind in ("linear", "greedy"):
        state["module"] = _module(case["type"], case["n"], case["k"], seed, case.get("bias", False))
        state["x"] = synthetic.make_activations(rows, case["k"], seed=seed + 2, device="cuda")
        return state
    hidden = case["hidden"]
    state["x"] = synthetic.make_activations(rows, hidden, seed=seed + 2, device="cuda")
    state["context"] = synthetic.make_activations(rows, hidden, seed=seed + 3, device="cuda")
    if kind == "mixed":
        state["towers"] = list(_layers(case, 2, seed))
        state["wide"] = synthetic.make_activations(rows, case["inter"], seed=seed + 4, device="cuda")
        state["indicator"] = None
        if case["scattered"]:
            order = torch.randperm(rows, generator=torch.Generator().manual_seed(seed))
            state["indicator"] = (order >= case["text"]).to("cuda")
        return state
    model = _layers(case, case["layers"], seed)
    if kind == "layers":
        fuse_gated_mlps(model)
        stack_shared_input_projections(model)
        state["layers"] = list(model)
    else:
        gammas = synthetic.make_activations(2, hidden, seed=seed + 4, device="cuda") * 0.1 + 1.0
        state["norms"] = [gammas[0].contiguous(), gammas[1].contiguous()]
        state["layers"] = [(FusedProjections([m.q_proj, m.k_proj, m.v_proj], release_sources=True), m.o_proj, m.mlp) for m in model]
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    with torch.no_grad():
        if kind == "linear":
            return state["module"](state["x"])
        if kind == "greedy":
            return state["module"].forward_argmax(state["x"])
        if kind == "dequantize":
            return [dequantize_gguf_tensor(w, DTYPES[case["out"]]) for w in state["weights"]]
        x, context = state["x"], state["context"]
        out = []
        if kind == "layers":
            for layer in state["layers"]:
                out += [layer.q_proj(x), layer.k_proj(x), layer.v_proj(x), layer.o_proj(context), layer.mlp(x)]
            return out
        if kind == "folded":
            before, after = state["norms"]
            for qkv, o_proj, mlp in state["layers"]:
                out += qkv(x, before, EPS)
                h = o_proj.forward_residual(context, x)
                out += [h, gated_mlp(h, mlp.gate_proj, mlp.up_proj, mlp.down_proj, norm_weight=after, eps=EPS, residual=h)]
            return out
        und, gen = state["towers"]
        ind = state["indicator"]
        text = case["text"] if ind is None else None
        for name, rows in (("q_proj", x), ("k_proj", x), ("v_proj", x), ("o_proj", context), ("mlp.gate_proj", x),
                           ("mlp.up_proj", x), ("mlp.down_proj", state["wide"])):
            out.append(grouped_linear(rows, ind, und.get_submodule(name), gen.get_submodule(name), n_text=text))
        return out


def _packed_bytes(qtype, n, k):
    block, size = GGML_QUANT_SIZES[TYPES[qtype]]
    return n * (k // block) * size


def work(case):
    kind = case["kind"]
    if kind == "dequantize":
        item = torch.empty((), dtype=DTYPES[case["out"]]).element_size()
        n, k = case["n"], case["k"]
        return {"bytes": case["count"] * (_packed_bytes(case["type"], n, k) + item * n * k), "flops": case["count"] * n * k}
    rows = case["rows"]
    if kind in ("linear", "greedy"):
        n, k = case["n"], case["k"]
        out = 8 * rows if kind == "greedy" else 2 * rows * n
        return {"bytes": _packed_bytes(case["type"], n, k) + 2 * rows * k + out, "flops": 2 * rows * n * k}
    nbytes = flops = 0
    for name, (n, k) in _layer_shapes(case).items():
        qtype = case["down_type"] if name == "mlp.down_proj" else case["type"]
        nbytes += _packed_bytes(qtype, n, k)
        flops += 2 * rows * n * k
    h, i, kv = case["hidden"], case["inter"], case["kv"]
    if kind == "mixed":
        # both towers' weights; the hidden states, the context and the gated activations; seven outputs
        return {"bytes": 2 * nbytes + 2 * rows * (2 * h + i) + 2 * rows * (3 * h + 2 * kv + 2 * i), "flops": flops}
    # the hidden states and the context once per layer; q, k, v, o and the MLP's output (gate / up stay inside)
    nbytes += 2 * rows * (2 * h) + 2 * rows * (3 * h + 2 * kv)
    return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}


def tolerance(case):
    if case["kind"] in ("dequantize", "greedy"):
        return "exact"   # decoded values, and the place of the largest logit
    # The decoded weights are the same bits in any implementation at this precision; sums in another order move single
    # outputs by one bf16 step (against 64-bit sums: up to 9e-5 over an output of a few hundred values, 5e-5 over large
    # ones), and behind the MLP's inner values and the norms those steps pass on to the outputs (up to 3.6e-4).
    if case["kind"] in ("linear", "mixed"):
        return {"rel": 4e-4}
    return {"rel": 1.4e-3}


# What run() returns, in 64 bits from plain torch.  The decoded weights are part of the path's definition (every step of a
# type's decode rounds to fp16, the result to bf16), so the decode below keeps those steps; the sums, the norm and the
# gated product behind it are in 64 bits throughout.
def _fp16(blocks, at):
    return blocks[:, at:at + 2].contiguous().view(torch.float16)


def _bits(b, shifts, mask):
    """Bytes [n, groups, width] -> [n, groups * shifts, width]: the fields at each shift, lowest first."""
    s = torch.tensor(shifts, dtype=torch.uint8, device=b.device).reshape(1, 1, -1, 1)
    return ((b.unsqueeze(2) >> s) & mask).reshape(b.shape[0], -1, b.shape[2])


def _six_bit_pairs(s):
    low, high, top = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    return (torch.cat([low & 63, (top & 15) | ((low >> 2) & 48)], 1), torch.cat([high & 63, (top >> 4) | ((high >> 2) & 48)], 1))


def _decoded(qtype, packed):
    """Packed rows -> the fp16 weights [n, k] (bf16 weights: as they are)."""
    if qtype == "bf16":
        return packed.view(torch.bfloat16)
    n = packed.shape[0]
    b = packed.reshape(-1, GGML_QUANT_SIZES[TYPES[qtype]][1])
    if qtype == "q8_0":
        w = _fp16(b, 0) * b[:, 2:].contiguous().view(torch.int8)
    elif qtype in ("q4_0", "q4_1", "q5_0", "q5_1"):
        at = 4 if qtype[-1] == "1" else 2
        fifth = qtype[1] == "5"
        q = _bits(b[:, at + (4 if fifth else 0):].unsqueeze(1), [0, 4], 15).reshape(-1, 32)
        if fifth:
            q = q | (_bits(b[:, at:at + 4].unsqueeze(1), range(8), 1).transpose(1, 2).reshape(-1, 32) << 4)
        w = _fp16(b, 0) * q + _fp16(b, 2) if qtype[-1] == "1" else _fp16(b, 0) * (q.to(torch.int8) - (16 if fifth else 8))
    elif qtype == "q2_k":
        q = _bits(b[:, 16:80].reshape(-1, 2, 32), [0, 2, 4, 6], 3).reshape(-1, 16, 16)
        w = (_fp16(b, 80) * (b[:, :16] & 15)).unsqueeze(2) * q - (_fp16(b, 82) * (b[:, :16] >> 4)).unsqueeze(2)
    elif qtype == "q3_k":
        q = _bits(b[:, 32:96].reshape(-1, 2, 32), [0, 2, 4, 6], 3).reshape(-1, 16, 16).to(torch.int8)
        low = _bits(b[:, :32].unsqueeze(1), range(8), 1).reshape(-1, 16, 16).to(torch.int8)
        s = _bits(b[:, 96:104].unsqueeze(1), [0, 4], 15).reshape(-1, 16) | (_bits(b[:, 104:108].unsqueeze(1), [0, 2, 4, 6], 3).reshape(-1, 16) << 4)
        w = (_fp16(b, 108) * (s.to(torch.int8) - 32)).unsqueeze(2) * (q - 4 * (1 - low))
    elif qtype in ("q4_k", "q5_k"):
        scale, low = _six_bit_pairs(b[:, 4:16])
        q = _bits(b[:, -128:].reshape(-1, 4, 32), [0, 4], 15)
        if qtype == "q5_k":
            q = q | (_bits(b[:, 16:48].unsqueeze(1), range(8), 1) << 4)
        w = (_fp16(b, 0) * scale).unsqueeze(2) * q - (_fp16(b, 2) * low).unsqueeze(2)
    else:
        q = _bits(b[:, :128].reshape(-1, 2, 64), [0, 4], 15).reshape(-1, 16, 16)
        q = q | (_bits(b[:, 128:192].reshape(-1, 2, 32), [0, 2, 4, 6], 3).reshape(-1, 16, 16) << 4)
        w = (_fp16(b, 208) * b[:, 192:208].contiguous().view(torch.int8)).unsqueeze(2) * (q.to(torch.int8) - 32)
    return w.reshape(n, -1)


def exact(case, seed):
    kind = case["kind"]
    seed = seed * 7919 + 17

    def packed(qtype, n, k, s):
        return synthetic.make_packed(TYPES[qtype], n, k, seed=s, device="cuda")

    def weights(qtype, n, k, s):
        return _decoded(qtype, packed(qtype, n, k, s)).to(torch.bfloat16).double()

    def activations(rows, k, s):
        return synthetic.make_activations(rows, k, seed=s, device="cuda").double()

    if kind == "greedy":
        return None
    if kind == "dequantize":
        return [_decoded(case["type"], packed(case["type"], case["n"], case["k"], seed + i)).double() for i in range(case["count"])]
    rows = case["rows"]
    if kind == "linear":
        y = activations(rows, case["k"], seed + 2) @ weights(case["type"], case["n"], case["k"], seed).T
        return y + activations(1, case["n"], seed + 1)[0] if case["bias"] else y
    hidden = case["hidden"]
    x, context = activations(rows, hidden, seed + 2), activations(rows, hidden, seed + 3)
    shapes = _layer_shapes(case)

    def weight(i, name):
        qtype = case["down_type"] if name == "mlp.down_proj" else case["type"]
        return weights(qtype, *shapes[name], seed * 1000 + i * 10 + list(shapes).index(name)).T

    def mlp(i, rows):
        return (torch.nn.functional.silu(rows @ weight(i, "mlp.gate_proj")) * (rows @ weight(i, "mlp.up_proj"))) @ weight(i, "mlp.down_proj")

    out = []
    if kind == "mixed":
        image = torch.arange(rows, device="cuda") >= case["text"]
        if case["scattered"]:
            image = image[torch.randperm(rows, generator=torch.Generator().manual_seed(seed)).to("cuda")]
        wide = activations(rows, case["inter"], seed + 4)
        for name in shapes:
            a = wide if name == "mlp.down_proj" else context if name == "o_proj" else x
            y = torch.empty(rows, shapes[name][0], dtype=torch.float64, device="cuda")
            y[~image] = a[~image] @ weight(0, name)
            y[image] = a[image] @ weight(1, name)
            out.append(y)
        return out
    if kind == "folded":
        gammas = (synthetic.make_activations(2, hidden, seed=seed + 4, device="cuda") * 0.1 + 1.0).double()

        def norm(rows, gamma):
            return rows * torch.rsqrt(rows.square().mean(1, keepdim=True) + EPS) * gamma
    for i in range(case["layers"]):
        a = norm(x, gammas[0]) if kind == "folded" else x
        out += [a @ weight(i, name) for name in ("q_proj", "k_proj", "v_proj")]
        h = context @ weight(i, "o_proj")
        if kind == "folded":
            h = h + x
            out += [h, h + mlp(i, norm(h, gammas[1]))]
        else:
            out += [h, mlp(i, x)]
    return out
