"""Timed workloads of the forward path, through its public entry points.

What a program of this framework has the GPU do, by how it is used:

- one decode token through a decoder layer (lh_layer_forward, one launch
  sequence of a few tens of microseconds), shortly after a prompt and at a long
  context, for the compact FP8 and the resident FP32 weights;
- a block of tokens through a layer on the matrix cores (LH_PATH_MFMA, the
  default prefill mode): a short message, a turn's 64 tokens after a long
  conversation, a ragged chunk and a whole 256-token chunk of a long prompt;
- the same on the precise path (prefill mode CUSTOM, and every multi-token call
  of the resident strategy), whose results equal the chain of decode steps;
- whole calls of the 26-layer model through the runtime: decode steps after a
  restored checkpoint, and a prompt in two chunks.

A layer's weights are FP8 codes of normally distributed values with one scale
per tensor, its cache rows and residual rows are normal with a spread over the
channels, at the model's sizes (hidden 3072, 32 query and 8 KV heads of 128,
inner 9216). The calls run the seeded synthetic model of the runtime.
"""
import ctypes
import math

import numpy as np
import torch

import lunelette_amd as lh
from lunelette_amd import synthetic
from lunelette_amd.runtime import Runtime

HIDDEN, QUERY, KV, INNER, VOCAB, LAYERS = 3072, 4096, 1024, 9216, 131072, 26
HEADS, KV_HEADS, DIM = 32, 8, 128
LAYER_WEIGHTS = (QUERY + 2 * KV) * HIDDEN + HIDDEN * QUERY + 3 * HIDDEN * INNER
PATHS = {"fused": lh.PATH_FUSED, "lookup": lh.PATH_LOOKUP, "resident": lh.PATH_RESIDENT,
         "mfma": lh.PATH_MFMA}
STEPS = 4   # decode steps of a "decode" call


def _layer(name, path, count, length, context):
    return {"name": name, "kind": "layer", "path": path, "count": count, "length": length,
            "context": context}


def listed():
    return [
        # One generated token: soon after a prompt, and deep in a long session.
        _layer("decode_layer_550", "fused", 1, 549, 4352),
        _layer("decode_layer_16000", "fused", 1, 15999, 17920),
        # The resident FP32 strategy: its decode, and a short prompt's block.
        _layer("resident_decode_layer_1024", "resident", 1, 1023, 4352),
        _layer("resident_layer_48", "resident", 48, 517, 4352),
        # A short user message, and one turn's 64 tokens after a long session.
        _layer("append_layer_7", "mfma", 7, 1203, 4352),
        _layer("append_layer_64", "mfma", 64, 15872, 17920),
        # A prompt's ragged last chunk, and a whole chunk of a long prompt.
        _layer("prefill_layer_201", "mfma", 201, 256, 4352),
        _layer("prefill_layer_256", "mfma", 256, 4096, 4352),
        # The precise prefill mode: a message, and a whole chunk.
        _layer("precise_layer_37", "fused", 37, 777, 4352),
        _layer("precise_layer_256", "fused", 256, 4096, 4352),
        # The whole model: decode steps after a restored checkpoint, a prompt.
        {"name": "decode_call", "kind": "decode", "prefix": 1500},
        {"name": "prompt_call", "kind": "prompt", "count": 443},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    which = rng.random()
    context = rng.choice((4352, 17920))
    if which < 0.05:
        return {"kind": "decode", "prefix": _log_int(rng, 2, 4300)}
    if which < 0.10:
        return {"kind": "prompt", "count": _log_int(rng, 257, 512)}
    if which < 0.35:
        path, count = rng.choice(("fused", "fused", "lookup", "resident")), 1
    elif which < 0.70:
        path, count = "mfma", _log_int(rng, 2, 256)
    else:
        path, count = rng.choice(("fused", "fused", "lookup", "resident")), _log_int(rng, 2, 256)
        # No dearer than the listed whole chunk after 4096 positions.
        context = 4352
        if path != "fused":
            count = min(count, 96)
    length = _log_int(rng, 1, context - count)
    return {"kind": "layer", "path": path, "count": count, "length": length, "context": context}


# ---- inputs ---------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _codes(g, rows, cols):
    """E4M3 codes of normal values whose largest magnitudes reach the format's."""
    out = torch.empty(rows, cols, dtype=torch.uint8, device="cuda")
    for r in range(0, rows, 3072):
        n = min(3072, rows - r)
        v = torch.randn(n, cols, device="cuda", generator=g).mul_(80).clamp_(-448, 448)
        out[r:r + n] = v.to(torch.float8_e4m3fn).view(torch.uint8)
    return out


def _decode(codes):
    return codes.view(torch.float8_e4m3fn)


def _bf16(v):
    return float(torch.tensor(v).bfloat16())


def _layer_inputs(case, seed):
    g = _generator(seed)
    count, context = case["count"], case["context"]
    d = {"qkv": _codes(g, QUERY + 2 * KV, HIDDEN), "o": _codes(g, HIDDEN, QUERY),
         "gate": _codes(g, INNER, HIDDEN), "up": _codes(g, INNER, HIDDEN),
         "down": _codes(g, HIDDEN, INNER)}
    # Weights of about 0.02: one BF16-exact scale per tensor (q,k,v,o,gate,up,down).
    d["scale"] = [_bf16(s * 1e-4) for s in (2.5, 2.6, 2.3, 2.4, 2.5, 2.2, 2.1)]
    for n in ("input_norm", "post_norm"):
        d[n] = (1 + 0.1 * torch.randn(HIDDEN, device="cuda", generator=g)).bfloat16().float()
    spread = torch.exp(0.5 * torch.randn(HIDDEN, device="cuda", generator=g))
    d["x"] = torch.randn(count, HIDDEN, device="cuda", generator=g) * spread
    # Cache rows below `length`; [8][context][128], K's words permuted inside a
    # 64-position tile (normal values: the permutation of them is as good).
    for n, s in (("keys", 2.0), ("values", 1.0)):
        d[n] = s * torch.randn(KV_HEADS, context, DIM, device="cuda", generator=g)
    return d


class _Layer:
    """A program's layer: weights, cache, workspace with the step's tokens set."""

    def __init__(self, case, seed):
        self.case, self.lib = case, lh.lib()
        d = self.d = _layer_inputs(case, seed)
        w = self.weights = lh.LayerWeights()
        for n in ("qkv", "o", "gate", "up", "down"):
            if case["path"] == "resident":
                d[n] = _decode(d[n]).float()
                setattr(w, "f32_" + n, d[n].data_ptr())
            else:
                setattr(w, n, d[n].data_ptr())
        for i, s in enumerate(d["scale"]):
            w.scale[i] = s
        w.input_norm, w.post_norm = d["input_norm"].data_ptr(), d["post_norm"].data_ptr()
        self.x = torch.empty_like(d["x"])
        self.path = PATHS[case["path"]]
        torch.cuda.synchronize()
        self.workspace = self.lib.lh_workspace_create(case["context"], case["count"])
        if not self.workspace:
            raise RuntimeError(lh.last_error())
        ids = np.zeros(case["count"], np.int64)
        lh.check(self.lib.lh_workspace_set_tokens(
            self.workspace, ids.ctypes.data_as(lh.c_int64_p), case["length"], case["count"],
            self.stream()))
        first, last = case["length"], case["length"] + case["count"]
        self.tiles = (first // 64, (last + 63) // 64)
        self.rows = (first, last)

    @staticmethod
    def stream():
        return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def run(self):
        d = self.d
        self.x.copy_(d["x"])   # the layer works in place
        lh.check(self.lib.lh_layer_forward(
            ctypes.byref(self.weights), self.x.data_ptr(), d["keys"].data_ptr(),
            d["values"].data_ptr(), self.workspace, self.path, self.stream()))
        return _outputs(self.x, d["keys"], d["values"], self.tiles, self.rows)

    def __del__(self):
        if getattr(self, "workspace", None):
            torch.cuda.synchronize()
            self.lib.lh_workspace_destroy(self.workspace)
            self.workspace = None


def _outputs(x, keys, values, tiles, rows):
    """The layer's output rows and the cache it updated (K by whole tiles)."""
    k = keys.view(KV_HEADS, -1, 64 * DIM)
    return {"x": x, "keys": k[:, tiles[0]:tiles[1]], "values": values[:, rows[0]:rows[1]]}


class _Call:
    """A program's runtime of the 26-layer model."""

    def __init__(self, case, seed):
        self.case = case
        self.runtime = Runtime(seed=int(seed) + 1, layers=LAYERS, context=4352, block=256)
        prefix = case["prefix"] if case["kind"] == "decode" else 0
        n = prefix + STEPS if prefix else case["count"]
        self.ids = synthetic.tokens(int(seed) + 1, 3, n)
        self.checkpoint = None
        if prefix:
            self.runtime.prefill(self.ids[:min(256, prefix)], copy=False)
            for at in range(256, prefix, 256):
                self.runtime.append(self.ids[at:min(at + 256, prefix)], copy=False)
            self.checkpoint = self.runtime.checkpoint()

    def run(self):
        rt, ids = self.runtime, self.ids
        if self.checkpoint:
            rt.restore(self.checkpoint, copy=False)
            return [rt.decode(t) for t in ids[self.case["prefix"]:]]
        rt.reset()
        return [rt.prefill(ids[:256]), rt.append(ids[256:])]

    def __del__(self):
        if getattr(self, "checkpoint", None):
            self.runtime.destroy_checkpoint(self.checkpoint)
            self.checkpoint = None
        if getattr(self, "runtime", None):
            self.runtime.close()


def prepare(case, seed):
    return _Layer(case, seed) if case["kind"] == "layer" else _Call(case, seed)


def run(state):
    return state.run()


# ---- what a pass cannot do without ------------------------------------------

def _layer_work(count, length, weight_bytes):
    """Bytes and operations of one layer over `count` tokens after `length`."""
    pairs = count * length + count * (count + 1) // 2     # (token, visible position)
    nbytes = LAYER_WEIGHTS * weight_bytes + 2 * HIDDEN * 4 + \
        2 * KV * 4 * (length + count) + 2 * HIDDEN * 4 * count
    return nbytes, 2 * LAYER_WEIGHTS * count + 4 * HEADS * DIM * pairs


def work(case):
    if case["kind"] == "layer":
        nbytes, flops = _layer_work(case["count"], case["length"],
                                    4 if case["path"] == "resident" else 1)
        return {"bytes": nbytes, "flops": flops}
    chunks = [(1, case["prefix"] + i) for i in range(STEPS)] if case["kind"] == "decode" else \
        [(256, 0), (case["count"] - 256, 256)]
    nbytes = flops = 0
    for count, length in chunks:
        b, f = _layer_work(count, length, 1)
        nbytes += LAYERS * b + VOCAB * HIDDEN * 2 + VOCAB * 4 + count * HIDDEN * 2
        flops += LAYERS * f + 2 * VOCAB * HIDDEN
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # About four times what the paths differ by from 64 bits: 2.7e-7 for the precise
    # paths' 32-bit sums; 8.5e-6 for the matrix-core path, whose operands carry
    # 16 bits (P and V of the attention) to 24. The calls run a model whose
    # near-one-hot softmax amplifies rounding through 26 layers: the precise
    # and the matrix-core prefill, both right, give logits that differ by up
    # to 8e-3 (single ones by 4e-2 of their root mean square).
    if case["kind"] != "layer":
        return {"rel": 2e-2, "max": 0.15}
    return {"rel": 3.5e-5 if case["path"] == "mfma" else 1.2e-6}


# ---- the same layer in 64 bits ------------------------------------------------

def _rotation(positions):
    """YaRN cos and sin [n][128] (theta 1e6, factor 16, original context 16384,
    beta 32 and 1): the angle in 32 bits as the model defines it, its sine and
    cosine in 64."""
    f = np.float32
    denominator = 2 * math.log(1e6)
    low = f(math.floor(128 * math.log(16384 / (32 * 2 * math.pi)) / denominator))
    high = f(math.ceil(128 * math.log(16384 / (2 * math.pi)) / denominator))
    j = np.arange(64)
    frequency = np.power(1e6, 2 * j / 128).astype(f)
    ramp = np.clip((j.astype(f) - low) / (high - low), f(0), f(1))
    keep = f(1) - ramp
    inverse = (f(1) / (f(16) * frequency)) * (f(1) - keep) + (f(1) / frequency) * keep
    angle = (inverse[None, :] * positions.astype(f)[:, None]).astype(np.float64)
    angle = np.concatenate([angle, angle], axis=1)
    to = lambda v: torch.from_numpy(v).cuda()  # noqa: E731
    return to(np.cos(angle)), to(np.sin(angle))


def _untile(keys):
    t = keys.view(KV_HEADS, -1, 4, 8, 16, 4, 4)   # head, tile, p/16, i, p%16, quarter, 4 dims
    return t.permute(0, 1, 2, 4, 5, 3, 6).reshape(keys.shape)


def _tile(keys):
    t = keys.view(KV_HEADS, -1, 4, 16, 4, 8, 4)
    return t.permute(0, 1, 2, 5, 3, 4, 6).reshape(keys.shape)


def exact(case, seed):
    if case["kind"] != "layer":
        return None
    d = _layer_inputs(case, seed)
    n, length = case["count"], case["length"]
    scale = d["scale"]

    def project(x, codes, s):
        out = torch.empty(x.shape[0], codes.shape[0], dtype=torch.float64, device="cuda")
        for r in range(0, codes.shape[0], 3072):
            w = _decode(codes[r:r + 3072]).float().double()
            out[:, r:r + 3072] = x @ w.t()
        return out * s

    def norm(x, gamma):
        return gamma.double() * x * torch.rsqrt(x.square().mean(1, keepdim=True) + 1e-5)

    x = d["x"].double()
    h = norm(x, d["input_norm"])
    q = project(h, d["qkv"][:QUERY], scale[0]).view(n, HEADS, DIM)
    k = project(h, d["qkv"][QUERY:QUERY + KV], scale[1]).view(n, KV_HEADS, DIM)
    v = project(h, d["qkv"][QUERY + KV:], scale[2]).view(n, KV_HEADS, DIM)
    positions = np.arange(length, length + n)
    cos, sin = _rotation(positions)

    def rotate(u):
        half = torch.cat([-u[..., 64:], u[..., :64]], dim=-1)
        return u * cos[:, None] + half * sin[:, None]

    factor = 1 + 0.1 * np.log(1.0 + positions // 16384)
    q, k = rotate(q) * torch.from_numpy(factor).cuda()[:, None, None], rotate(k)
    keys, values = _untile(d["keys"]).double(), d["values"].double()
    keys[:, length:length + n] = k.transpose(0, 1)
    values[:, length:length + n] = v.transpose(0, 1)
    seen = length + n
    visible = torch.arange(seen, device="cuda")[None, :] <= \
        torch.arange(length, seen, device="cuda")[:, None]
    attended = torch.empty(n, HEADS, DIM, dtype=torch.float64, device="cuda")
    for head in range(HEADS):
        kv = head // (HEADS // KV_HEADS)
        s = (q[:, head] @ keys[kv, :seen].t()) / math.sqrt(DIM)
        p = torch.softmax(s.masked_fill(~visible, -math.inf), dim=1)
        attended[:, head] = p @ values[kv, :seen]
    x = x + project(attended.view(n, QUERY), d["o"], scale[3])
    h = norm(x, d["post_norm"])
    gate, up = project(h, d["gate"], scale[4]), project(h, d["up"], scale[5])
    x = x + project(gate / (1 + torch.exp(-gate)) * up, d["down"], scale[6])
    first = length
    return _outputs(x, _tile(keys), values, (first // 64, (seen + 63) // 64), (first, seen))
