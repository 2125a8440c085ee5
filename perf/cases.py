"""What a program has this library do, as cases that can be timed and checked.

A case is a dict of plain values. `kind` says which of the public entry points
it goes through:

  prefill    a prompt in 512-token steps (Model.step), the last one's logits
  turn       the chat tool's paired runs (Model.paired): a fresh prompt, its
             reply, then the reply under pins from the same seed
  decode     a reply's tokens after a long prompt that the caches hold
             (Model.step of the last prompt token, Model.decode)
  variants   one prompt's original and steered replies in one batch, the
             residuals captured (Model.generate_variants)
  inspect    a prompt read with the capture store on (Model.generate of no
             tokens, Model.capture)
  mlp        one feed-forward block of some rows (frz_op_gated, frz_op_gemv)
  attention  one decode token's rope, cache append and attention, in the
             entry point made for serving loops (frz_op_rope_attention_noalloc)
  head       one row's logits, selection and draw (frz_op_gemv, frz_op_topk,
             frz_op_draw)

Models are the full 26-layer Gemma-3-1B shape with seeded random weights,
either all Q4_0 or in the formats of the file the reference pins (Q8_0
embedding and head, Q4_1 downs in layers 0-2). A program keeps one model for
all its prompts, so the states of a case share theirs; the ids, pins, rows and
caches come from the seed.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import frizzle_amd as fz
from frizzle_amd import _lib

CONTEXT = 8192
BLOCK = 512                      # tokens of a step
HIDDEN, FFN, HEADS, DIM, LAYERS, VOCAB = 1152, 6912, 4, 256, 26, 262144
WINDOW, PATTERN = 512, 6         # five sliding layers, then a global one
QKV = (HEADS + 2) * DIM
ROLES = ["q", "k", "v", "o", "gate", "up", "down", "attn_norm", "q_norm", "k_norm",
         "post_attn_norm", "ffn_norm", "post_ffn_norm"]
WEIGHTS_SEED = 20240


def listed():
    return [
        # One decode token's attention over the keys of a global layer.
        {"name": "attention_global", "kind": "attention", "position": 5003, "window": 8192},
        # A prompt's rows through one feed-forward block, a neuron or two pinned.
        {"name": "mlp_29", "kind": "mlp", "tokens": 29},
        # The tied head's product, its 64 best and the draw.
        {"name": "head", "kind": "head"},
        # A one-line chat message: the time to its first token.
        {"name": "prefill_21", "kind": "prefill", "tokens": 21, "mode": "exact",
         "formats": "pinned"},
        # A few paragraphs, bit for bit the reference's arithmetic.
        {"name": "prefill_333", "kind": "prefill", "tokens": 333, "mode": "exact",
         "formats": "pinned"},
        # A document, bit for bit the reference's arithmetic.
        {"name": "prefill_2048", "kind": "prefill", "tokens": 2048, "mode": "exact",
         "formats": "q4_0"},
        # A message and a long document in the fast mode.
        {"name": "fast_prefill_150", "kind": "prefill", "tokens": 150, "mode": "bf16",
         "formats": "q4_0"},
        {"name": "fast_prefill_3001", "kind": "prefill", "tokens": 3001, "mode": "bf16",
         "formats": "q4_0"},
        # The chat tool's turn: the reply and the steered reply to one message.
        {"name": "paired_turn", "kind": "turn", "tokens": 61, "reply": 24, "pins": 8,
         "formats": "pinned"},
        # Replying late in a long conversation.
        {"name": "decode_7901", "kind": "decode", "tokens": 7901, "reply": 32},
        # A steering study: one original and 15 steered replies, with residuals.
        {"name": "variants_16", "kind": "variants", "tokens": 300, "variants": 16, "reply": 16},
        # An inspection: every layer's captures and readouts at a prompt's end.
        {"name": "inspect_45", "kind": "inspect", "tokens": 45},
    ]


def _between(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "prefill", "turn", "decode", "variants", "inspect",
                       "mlp", "attention"])
    if kind == "prefill":
        mode = rng.choice(["exact", "bf16"])
        return {"kind": kind, "tokens": _between(rng, 2, 2048 if mode == "exact" else 3000),
                "mode": mode, "formats": rng.choice(["q4_0", "pinned"])}
    if kind == "turn":
        return {"kind": kind, "tokens": _between(rng, 8, 500), "reply": rng.randint(4, 24),
                "pins": rng.randint(1, 32), "formats": rng.choice(["q4_0", "pinned"])}
    if kind == "decode":
        return {"kind": kind, "tokens": _between(rng, 40, 8000), "reply": rng.randint(8, 32)}
    if kind == "variants":
        return {"kind": kind, "tokens": _between(rng, 16, 700), "variants": rng.randint(2, 24),
                "reply": rng.randint(4, 16)}
    if kind == "inspect":
        return {"kind": kind, "tokens": _between(rng, 2, 400)}
    if kind == "mlp":
        return {"kind": kind, "tokens": _between(rng, 1, 512)}
    window = rng.choice([512, 8192])
    return {"kind": kind, "position": _between(rng, 1, 8191), "window": window}


# ---- the model and its weights ---------------------------------------------------


@functools.lru_cache(None)
def _device():
    return fz.Device(0)


def _blocks(rng, fmt, rows, cols):
    """Seeded GGUF blocks: half-normal scales, uniform codes, Q4_1's minimum
    such that weights lie about zero, Q8_0's codes 16 times wider."""
    n = rows * cols // 32
    d = np.abs(rng.normal(0.0, 0.02, n)).astype(np.float16)
    if fmt == fz.Q8_0:
        d = (d.astype(np.float32) / 16).astype(np.float16)
        out = np.empty((n, 34), dtype=np.uint8)
        out[:, 2:] = rng.integers(0, 256, size=(n, 32), dtype=np.uint8)
    else:
        head = 4 if fmt == fz.Q4_1 else 2
        out = np.empty((n, head + 16), dtype=np.uint8)
        if fmt == fz.Q4_1:
            m = (-d.astype(np.float32) * 8).astype(np.float16)
            out[:, 2:4] = m.view(np.uint8).reshape(n, 2)
        out[:, head:] = rng.integers(0, 256, size=(n, 16), dtype=np.uint8)
    out[:, 0:2] = d.view(np.uint8).reshape(n, 2)
    return out.reshape(-1)


@functools.lru_cache(None)
def _tensors(formats):
    """{(layer, role): (GGUF bytes or gains, format)} of the whole model."""
    cfg = fz.gemma3_1b_config(context=CONTEXT)
    out = {}
    for layer in range(LAYERS):
        for role in ROLES:
            fmt = fz.Q4_0 if role in ("q", "k", "v", "o", "gate", "up", "down") else None
            out[layer, role] = (fz.synth_tensor(cfg, WEIGHTS_SEED, layer, role), fmt)
    out[-1, "output_norm"] = (fz.synth_tensor(cfg, WEIGHTS_SEED, -1, "output_norm"), None)
    if formats == "pinned":
        rng = np.random.default_rng(WEIGHTS_SEED)
        out[-1, "embedding"] = (_blocks(rng, fz.Q8_0, VOCAB, HIDDEN), fz.Q8_0)
        for layer in range(3):
            out[layer, "down"] = (_blocks(rng, fz.Q4_1, HIDDEN, FFN), fz.Q4_1)
    else:
        out[-1, "embedding"] = (fz.synth_tensor(cfg, WEIGHTS_SEED, -1, "embedding"), fz.Q4_0)
    return out


def _new_model(formats):
    model = fz.Model(_device(), fz.gemma3_1b_config(context=CONTEXT))
    for (layer, role), (data, fmt) in _tensors(formats).items():
        model.set_tensor(layer, role, data, fmt if fmt != fz.Q4_0 else None)
    return model


@functools.lru_cache(None)
def _model(formats, mode="exact", capture=False):
    model = _new_model(formats)
    if mode == "bf16":
        model.set_prefill(fz.PREFILL_BF16)
    if capture:
        model.set_capture(True)
    return model


class _OwnModel:
    """A model of one state's own, for caches that a state keeps filled."""

    def __init__(self):
        self.model = _new_model("q4_0")

    def __del__(self):
        self.model.close()


def _prompt(model, ids, samp, logits=True):
    for p in range(0, len(ids), BLOCK):
        block = ids[p:p + BLOCK]
        model.step(p, block, logits=logits and p + len(block) == len(ids), samp=samp)


def _pins(rng, n):
    pins = {}
    while len(pins) < n:
        layer, neuron = int(rng.integers(0, LAYERS)), int(rng.integers(0, FFN))
        pins[layer, neuron] = fz.Edit(layer, neuron, fz.EditKind.SET,
                                      float(rng.uniform(-10, 10)))
    return list(pins.values())


# ---- the states --------------------------------------------------------------------


def _split(fmt, blocks):
    codes, scales = fz.block_split(fmt, blocks)
    return torch.from_numpy(codes).cuda(), torch.from_numpy(scales).cuda()


@functools.lru_cache(None)
def _block_weights():
    """Layer 0's feed-forward matrices and the Q4_0 head, on the device."""
    t = _tensors("q4_0")
    return {r: _split(fz.Q4_0, t[k][0])
            for r, k in (("gate", (0, "gate")), ("up", (0, "up")), ("down", (0, "down")),
                         ("head", (-1, "embedding")))}


def _mlp_inputs(case, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(0, 1, (case["tokens"], HIDDEN)).astype(np.float32)
    pins = [fz.Edit(0, int(n), fz.EditKind.SET, float(rng.uniform(-10, 10)))
            for n in sorted(rng.choice(FFN, 2, replace=False))]
    return x, pins


def _attention_inputs(case, seed):
    rng = np.random.default_rng(seed)
    slots = 5120 if case["window"] == WINDOW else CONTEXT
    qkv = rng.normal(0, 1.5, QKV).astype(np.float32)
    gains = (1 + 0.1 * rng.normal(0, 1, (2, DIM))).astype(np.float32)
    cache = rng.normal(0, 1, (2, slots, DIM)).astype(np.float32).astype(np.float16)
    return slots, qkv, gains, cache


def _sampling(seed):
    # The chat tool's settings.
    return fz.sampling(temperature=0.8, top_k=40, top_p=0.95, min_p=0.05, seed=seed)


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    s = {"case": case, "kind": kind, "samp": _sampling(seed)}
    if kind == "mlp":
        x, pins = _mlp_inputs(case, seed)
        t = case["tokens"]
        s.update(x=torch.from_numpy(x).cuda(), w=_block_weights(),
                 edits=torch.from_numpy(fz.edit_table(pins, 1).view(np.int32)).cuda(),
                 act=torch.empty(t, FFN, device="cuda"), y=torch.empty(t, HIDDEN, device="cuda"))
    elif kind == "attention":
        slots, qkv, gains, cache = _attention_inputs(case, seed)
        base = 10000.0 if case["window"] == WINDOW else 1000000.0
        s.update(slots=slots, qkv=torch.from_numpy(qkv).cuda(),
                 gains=torch.from_numpy(gains).cuda(), keys=torch.from_numpy(cache[0]).cuda(),
                 values=torch.from_numpy(cache[1]).cuda(),
                 turns=torch.from_numpy(fz.rope_turns(base, DIM)).cuda(),
                 out=torch.empty(HEADS, DIM, device="cuda"))
    elif kind == "head":
        x = rng.normal(0, 1, HIDDEN).astype(np.float32)
        s.update(x=torch.from_numpy(x).cuda(), w=_block_weights(),
                 logits=torch.empty(VOCAB, device="cuda"),
                 candidates=torch.empty(64, 2, dtype=torch.int32, device="cuda"),
                 record=torch.empty(4, dtype=torch.int32, device="cuda"))
    else:
        s["ids"] = rng.integers(0, VOCAB, case["tokens"]).astype(np.uint32)
        if kind == "prefill":
            s["model"] = _model(case["formats"], case["mode"])
        elif kind == "turn":
            s["model"] = _model(case["formats"])
            s["pins"] = _pins(rng, case["pins"])
        elif kind == "decode":
            own = _OwnModel()
            _prompt(own.model, s["ids"], fz.sampling())
            s.update(own=own, model=own.model)
        elif kind == "variants":
            s["model"] = _model("q4_0")
            s["sets"] = [[]] + [_pins(rng, int(rng.integers(1, 33)))
                                for _ in range(case["variants"] - 1)]
        elif kind == "inspect":
            s["model"] = _model("q4_0", capture=True)
            s["pins"] = _pins(rng, 2)
    if s.get("model") is None:
        s["lib"], s["device"] = fz.load(), _device().handle
        torch.cuda.synchronize()
    return s


def _gemv(s, w, rows, cols, x, y, tokens):
    _lib.check(s["lib"].frz_op_gemv(s["device"], w[0].data_ptr(), w[1].data_ptr(), rows, cols,
                                    x.data_ptr(), cols, y.data_ptr(), rows, tokens, 0))


def run(s):
    case, kind, model = s["case"], s["kind"], s.get("model")
    if kind == "mlp":
        t, (gate, up) = case["tokens"], (s["w"]["gate"], s["w"]["up"])
        _lib.check(s["lib"].frz_op_gated(
            s["device"], gate[0].data_ptr(), gate[1].data_ptr(), up[0].data_ptr(),
            up[1].data_ptr(), FFN, HIDDEN, s["x"].data_ptr(), s["act"].data_ptr(), t, 0,
            s["edits"].data_ptr(), 0))
        _gemv(s, s["w"]["down"], HIDDEN, FFN, s["act"], s["y"], t)
        return {"act": s["act"], "y": s["y"]}
    if kind == "attention":
        _lib.check(s["lib"].frz_op_rope_attention_noalloc(
            s["device"], s["qkv"].data_ptr(), s["turns"].data_ptr(), s["gains"][0].data_ptr(),
            s["gains"][1].data_ptr(), s["keys"].data_ptr(), s["values"].data_ptr(),
            s["out"].data_ptr(), s["slots"], case["window"], 1e-6, 0.0625, case["position"]))
        return {"out": s["out"], "keys": s["keys"], "values": s["values"]}
    if kind == "head":
        _gemv(s, s["w"]["head"], VOCAB, HIDDEN, s["x"], s["logits"], 1)
        _lib.check(s["lib"].frz_op_topk(s["device"], s["logits"].data_ptr(), VOCAB,
                                        s["candidates"].data_ptr()))
        _lib.check(s["lib"].frz_op_draw(s["device"], s["candidates"].data_ptr(),
                                        ctypes.byref(s["samp"]), 77, 1, s["record"].data_ptr()))
        best = s["candidates"]
        return {"logits": s["logits"], "best": best[:, 0].view(torch.float32),
                "tokens": best[:, 1], "record": s["record"]}
    if kind == "prefill":
        _prompt(model, s["ids"], s["samp"])
        return {"logits": model.logits(), "token": int(model.record()[0])}
    if kind == "turn":
        original, steered = model.paired(s["ids"], s["pins"], s["samp"], case["reply"])
        return {"original": original, "steered": steered, "logits": model.logits()}
    if kind == "decode":
        n = case["tokens"]
        model.step(n - 1, s["ids"][-1:], logits=True, samp=fz.sampling())
        first = int(model.record()[0])
        tokens, _ = model.decode(n, case["reply"], fz.sampling())
        return {"first": first, "tokens": tokens, "logits": model.logits()}
    if kind == "variants":
        replies, residuals = model.generate_variants(s["ids"], s["sets"], s["samp"],
                                                     case["reply"], residuals=True)
        return {"tokens": np.concatenate(replies), "residuals": residuals}
    model.generate(s["ids"], s["pins"], s["samp"], 0)
    return _captures(*model.capture())


def _captures(store, layout):
    """The store by slot: the layers' rows together, the weights over the keys
    each layer reads, the readouts as logits and tokens."""
    def rows(slot):
        return np.stack([store[first:first + width] for first, width in
                         (layer[slot] for layer in layout)])

    out = {name: rows(name).view(np.float32)
           for name in ("neurons", "residual", "attention_added", "mlp_added", "query", "stats")}
    out["weights"] = np.concatenate([store[layer["weights"][0]:][:layer["weights"][1]]
                                     for layer in layout]).view(np.float32)
    readout = rows("readout").reshape(LAYERS, 64, 2)
    out["readout_logits"] = np.ascontiguousarray(readout[:, :, 0]).view(np.float32)
    out["readout_tokens"] = readout[:, :, 1].astype(np.int64)
    return out


# ---- what a pass cannot do without --------------------------------------------------

_LAYER_WEIGHTS = QKV * HIDDEN + HIDDEN * HEADS * DIM + 3 * FFN * HIDDEN
_Q4 = 0.5625  # bytes a Q4_0 weight


def _weight_bytes(formats, head=True):
    b = LAYERS * _LAYER_WEIGHTS * _Q4
    if formats == "pinned":
        b += 3 * HIDDEN * FFN * 0.0625
    return b + (VOCAB * HIDDEN * (1.0625 if formats == "pinned" else _Q4) if head else 0)


def _keys_read(first, last):
    """Keys read by the rows at positions first..last, over all layers."""
    p = np.arange(first, last + 1, dtype=np.float64) + 1
    local = LAYERS - LAYERS // PATTERN
    return float(local * np.minimum(p, WINDOW).sum() + (LAYERS // PATTERN) * p.sum())


def _attention_flops(first, last):
    return _keys_read(first, last) * HEADS * DIM * 4


def _held_keys(n):
    local = LAYERS - LAYERS // PATTERN
    return local * min(n, WINDOW) + (LAYERS // PATTERN) * n


_KEY_BYTES = 2 * 2 * DIM  # a key and its value, F16
_HEAD_FLOPS = 2.0 * VOCAB * HIDDEN


def _prefill_work(tokens, formats, head=True):
    flops = 2.0 * tokens * LAYERS * _LAYER_WEIGHTS + _attention_flops(0, tokens - 1)
    return (_weight_bytes(formats, head) + tokens * (LAYERS * _KEY_BYTES + 4) + (4 * VOCAB if head else 0),
            flops + (_HEAD_FLOPS if head else 0))


def _decode_work(position, steps, formats, rows=1):
    """`steps` steps of `rows` rows each, rows after a shared prefix."""
    b = f = 0.0
    for i in range(steps):
        b += _weight_bytes(formats) + rows * (4 * VOCAB + LAYERS * _KEY_BYTES)
        b += _held_keys(position) * _KEY_BYTES + rows * i * LAYERS * _KEY_BYTES
        f += rows * (2.0 * LAYERS * _LAYER_WEIGHTS + _HEAD_FLOPS
                     + _attention_flops(position + i, position + i))
    return b, f


def work(case):
    kind, t = case["kind"], case.get("tokens", 1)
    if kind == "mlp":
        b = 3 * FFN * HIDDEN * _Q4 + 4.0 * t * (2 * HIDDEN + FFN)
        return {"bytes": b, "flops": 6.0 * t * FFN * HIDDEN}
    if kind == "attention":
        keys = min(case["position"] + 1, case["window"])
        return {"bytes": float(keys * _KEY_BYTES + 4 * (QKV + HEADS * DIM)),
                "flops": 4.0 * keys * HEADS * DIM}
    if kind == "head":
        return {"bytes": VOCAB * HIDDEN * _Q4 + 4.0 * (HIDDEN + VOCAB), "flops": _HEAD_FLOPS}
    if kind == "prefill":
        b, f = _prefill_work(t, case["formats"])
    elif kind == "turn":
        b, f = _prefill_work(t, case["formats"])
        # the reply's other steps, then the steered reply's, whose prompt is cached
        db, df = _decode_work(t, 2 * case["reply"] - 1, case["formats"])
        b, f = b + db, f + df
    elif kind == "decode":
        b, f = _decode_work(t, case["reply"] + 1, "q4_0")
    elif kind == "variants":
        b, f = _prefill_work(t - 1, "q4_0", head=False)
        db, df = _decode_work(t, case["reply"], "q4_0", case["variants"])
        b += db + 4.0 * case["reply"] * case["variants"] * LAYERS * HIDDEN
        f += df
    else:
        b, f = _prefill_work(t, "q4_0")
        f += (LAYERS - 1) * _HEAD_FLOPS
        b += 4.0 * fz.capture_words(fz.gemma3_1b_config(context=CONTEXT))
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    # About four times the largest error of each path against 64 bits: 5e-7
    # for the blocks (sums of up to 6,912 products in f32), 3e-7 for exact
    # steps' logits, 1.3e-6 for the fast mode's and 2.3e-6 for what a layer's
    # attention adds. A sampled reply has one value for its tokens.
    if case["kind"] in ("mlp", "attention", "head"):
        return {"rel": 2e-6, "max": 2e-5, "differ": 0.02}
    return {"rel": 1e-5, "max": 1e-4, "differ": 0.02}


# ---- the same in 64 bits -------------------------------------------------------------


def _dense(fmt, raw, rows, cols):
    """GGUF blocks as f64 weights on the device, by the formats' definitions."""
    b = torch.from_numpy(np.asarray(raw, dtype=np.uint8)).cuda()
    if fmt == fz.Q8_0:
        b = b.view(-1, 34)
        d = b[:, :2].contiguous().view(torch.float16).double()
        w = b[:, 2:].contiguous().view(torch.int8).double() * d
    else:
        head = 4 if fmt == fz.Q4_1 else 2
        b = b.view(-1, head + 16)
        d = b[:, :2].contiguous().view(torch.float16).double()
        q = torch.cat([b[:, head:] & 15, b[:, head:] >> 4], 1).double()
        if fmt == fz.Q4_1:
            w = q * d + b[:, 2:4].contiguous().view(torch.float16).double()
        else:
            w = (q - 8) * d
    return w.reshape(rows, cols)


def _gelu(g):
    return 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3)))


def _rms(x, gain):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * gain


def _rope(x, positions, turns):
    """Pairs (k, k + 128) turned by the position's turns, which the model
    defines in f32."""
    t = (positions.float()[:, None] * turns).double()
    angle = 2 * math.pi * (t - torch.round(t))
    c, s = torch.cos(angle)[:, None], torch.sin(angle)[:, None]
    a, b = x[..., :DIM // 2], x[..., DIM // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


class _Exact:
    """The model in f64, its keys and values rounded to the cache's F16."""

    def __init__(self, formats):
        self.t = _tensors(formats)
        self.shape = {"q": (HEADS * DIM, HIDDEN), "k": (DIM, HIDDEN), "v": (DIM, HIDDEN),
                      "o": (HIDDEN, HEADS * DIM), "gate": (FFN, HIDDEN), "up": (FFN, HIDDEN),
                      "down": (HIDDEN, FFN), "embedding": (VOCAB, HIDDEN)}
        self.held = {}
        self.keys = [torch.empty(0, DIM, device="cuda", dtype=torch.float64)] * LAYERS
        self.values = list(self.keys)
        self.seen = {}

    def w(self, layer, role):
        if (layer, role) not in self.held:
            data, fmt = self.t[layer, role]
            self.held[layer, role] = (
                _dense(fmt, data, *self.shape[role]) if fmt is not None
                else torch.from_numpy(np.array(data).view(np.float32)).cuda().double())
        return self.held[layer, role]

    def rows(self, position, ids, pins=(), keep=False):
        """The residual rows of a step's ids; with `keep`, the last row's captures."""
        ids = torch.from_numpy(np.asarray(ids).astype(np.int64)).cuda()
        at = position + torch.arange(len(ids), device="cuda")
        x = self.w(-1, "embedding")[ids] * math.sqrt(HIDDEN)
        for layer in range(LAYERS):
            w = functools.partial(self.w, layer)
            is_global = layer % PATTERN == PATTERN - 1
            turns = torch.from_numpy(fz.rope_turns(1e6 if is_global else 1e4, DIM)).cuda()
            if keep:
                self.keep("residual", x)
            h = _rms(x, w("attn_norm"))
            q = _rms((h @ w("q").T).view(-1, HEADS, DIM), w("q_norm"))
            k = _rms((h @ w("k").T).view(-1, 1, DIM), w("k_norm"))
            q, k = _rope(q, at, turns), _rope(k, at, turns)[:, 0]
            self.keys[layer] = torch.cat([self.keys[layer][:position], k.half().double()])
            self.values[layer] = torch.cat([self.values[layer][:position],
                                            (h @ w("v").T).half().double()])
            low = max(0, position + 1 - WINDOW) if not is_global else 0
            ks, vs = self.keys[layer][low:], self.values[layer][low:]
            j = low + torch.arange(len(ks), device="cuda")
            live = j[None] <= at[:, None]
            if not is_global:
                live &= j[None] > at[:, None] - WINDOW
            scores = torch.einsum("thd,sd->hts", q, ks) / math.sqrt(DIM)
            weights = torch.softmax(scores.masked_fill(~live, -math.inf), -1)
            a = (weights @ vs).transpose(0, 1).reshape(len(ids), HEADS * DIM)
            added = _rms(a @ w("o").T, w("post_attn_norm"))
            x = x + added
            h = _rms(x, w("ffn_norm"))
            act = _gelu(h @ w("gate").T) * (h @ w("up").T)
            for e in pins:
                if e.layer == layer:
                    act[-1, e.neuron] = e.value
            mlp = _rms(act @ w("down").T, w("post_ffn_norm"))
            x = x + mlp
            if keep:
                self.keep("query", q.reshape(len(ids), -1))
                self.keep("attention_added", added)
                self.keep("neurons", act)
                self.keep("mlp_added", mlp)
                self.keep("after", x)
        return x

    def keep(self, name, rows):
        self.seen.setdefault(name, []).append(rows[-1])

    def prompt(self, ids, pins=(), keep=False):
        for p in range(0, len(ids), BLOCK):
            last = p + BLOCK >= len(ids)
            x = self.rows(p, ids[p:p + BLOCK], pins if last else (), keep and last)
        return x

    def logits(self, rows):
        return _rms(rows, self.w(-1, "output_norm")) @ self.w(-1, "embedding").T


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        x, pins = _mlp_inputs(case, seed)
        t, x = _tensors("q4_0"), torch.from_numpy(x).cuda().double()
        act = (_gelu(x @ _dense(fz.Q4_0, t[0, "gate"][0], FFN, HIDDEN).T)
               * (x @ _dense(fz.Q4_0, t[0, "up"][0], FFN, HIDDEN).T))
        for e in pins:
            act[:, e.neuron] = e.value
        return {"act": act, "y": act @ _dense(fz.Q4_0, t[0, "down"][0], HIDDEN, FFN).T}
    if kind == "attention":
        slots, qkv, gains, cache = _attention_inputs(case, seed)
        p, window = case["position"], case["window"]
        turns = torch.from_numpy(fz.rope_turns(1e4 if window == WINDOW else 1e6, DIM)).cuda()
        qkv, gains = (torch.from_numpy(a).cuda().double() for a in (qkv, gains))
        at = torch.tensor([p], device="cuda")
        q = _rope(_rms(qkv[:HEADS * DIM].view(1, HEADS, DIM), gains[0]), at, turns)[0]
        k = _rope(_rms(qkv[HEADS * DIM:][:DIM].view(1, 1, DIM), gains[1]), at, turns)[0, 0]
        keys, values = (torch.from_numpy(c).cuda() for c in cache)
        keys[p % slots], values[p % slots] = k.half(), qkv[-DIM:].half()
        j = torch.arange(max(0, p + 1 - window), p + 1, device="cuda") % slots
        weights = torch.softmax(q @ keys[j].double().T / math.sqrt(DIM), -1)
        return {"out": weights @ values[j].double(), "keys": keys, "values": values}
    if kind == "head":
        x = np.random.default_rng(seed).normal(0, 1, HIDDEN).astype(np.float32)
        w = _dense(fz.Q4_0, _tensors("q4_0")[-1, "embedding"][0], VOCAB, HIDDEN)
        logits = w @ torch.from_numpy(x).cuda().double()
        return {"logits": logits, "best": logits.topk(64).values, "tokens": None, "record": None}
    s = _exact_inputs(case, seed)
    if kind == "prefill":
        m = _Exact(case["formats"])
        return {"logits": m.logits(m.prompt(s["ids"])[-1]), "token": None}
    if kind == "decode":
        # Greedy, so each step's token is the last one's best logit.
        m, n = _Exact("q4_0"), case["tokens"]
        logits = m.logits(m.prompt(s["ids"])[-1])
        for i in range(case["reply"]):
            logits = m.logits(m.rows(n + i, [int(logits.argmax())])[-1])
        return {"first": None, "tokens": None, "logits": logits}
    if kind == "inspect":
        m = _Exact("q4_0")
        m.prompt(s["ids"], s["pins"], keep=True)
        out = {name: torch.stack(m.seen[name])
               for name in ("neurons", "residual", "attention_added", "mlp_added", "query")}
        best = m.logits(torch.stack(m.seen["after"])).topk(64, dim=-1).values
        return dict(out, stats=None, weights=None, readout_logits=best, readout_tokens=None)
    return None  # sampled replies: their tokens have no 64-bit value


def _exact_inputs(case, seed):
    rng = np.random.default_rng(seed)
    ids = rng.integers(0, VOCAB, case["tokens"]).astype(np.uint32)
    return {"ids": ids, "pins": _pins(rng, 2)}
