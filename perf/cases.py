"""Timed workloads of the INT8 KV-cache path, with their exact results.

Each case is one step of the engine's work on the full-attention layers, through the calls that
the engine makes, in commands of the device (begin ... end) as it opens them:

* ``decode``  one generated token: per layer the fused RoPE, append and attention
  (``engine.decode_append``), every layer in one command;
* ``prompt``  a prompt or a turn after ``history`` cached tokens, in chunks of ``chunk`` rows, one
  command a chunk with every layer in it. ``path`` is "fused" (``prepare_fused``, then the
  workspace's ``encode_int8`` on the prepared query), "unfused" (``append_rows``, then
  ``encode_int8`` on the rotated query) or "fp16" (``prepare_fused_fp16`` and
  ``encode_online_fp16`` over FP16 storage);
* ``verify``  a speculative verify block of ``rows`` candidates: per layer ``append_rows`` and
  ``verify_attention_int8``, every layer in one command (one row of it is the engine's serial
  decode on the three-kernel reader).

The model has ten full-attention layers; a case holds as many as its ``layers`` says, each with a
cache and inputs of its own. Outputs are the attention rows, the appended cache bytes and their scales.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PACKAGE = os.path.join(_ROOT, "llm-bootstrap-qwen3.6-35b-dotnet-metal_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import ctypes  # noqa: E402

from bootstrap_hip import engine  # noqa: E402
from bootstrap_hip.native import Device  # noqa: E402

WINDOW = 262144
EPSILON = 1e-6
THETA = engine.ROPE_THETA
OUTLIERS = (30, 31, 62, 63)      # the K channels that carry outliers, in and outside the rotated dimensions


def listed():
    return [
        # the next token of a short chat: launches and latency count
        {"name": "decode_chat", "kind": "decode", "history": 777, "layers": 10},
        # the next token over a few files or a long chat, away from any power of two
        {"name": "decode_9k", "kind": "decode", "history": 9001, "layers": 10},
        # the next token after the 30K-token prompt that the reference profiles
        {"name": "decode_30k", "kind": "decode", "history": 30725, "layers": 10},
        # the next token at half the model's window, the repository's long-context decode
        {"name": "decode_128k", "kind": "decode", "history": 131072, "layers": 10},
        # a one-line prompt: the reference's (0, 33) shape
        {"name": "prompt_33", "kind": "prompt", "path": "fused", "history": 0, "tokens": 33, "chunk": 512, "layers": 10},
        # an ordinary prompt in three chunks, the last one ragged
        {"name": "prompt_1500", "kind": "prompt", "path": "fused", "history": 0, "tokens": 1500, "chunk": 512, "layers": 10},
        # a user's turn in a running conversation, less than a chunk long
        {"name": "turn_200", "kind": "prompt", "path": "fused", "history": 6000, "tokens": 200, "chunk": 512, "layers": 10},
        # the headline workload: a 30720-token prompt of one layer in 60 chunks
        {"name": "prompt_30k", "kind": "prompt", "path": "fused", "history": 0, "tokens": 30720, "chunk": 512, "layers": 1},
        # a chunk through the unfused preparation, as the engine runs it with fusion off
        {"name": "unfused_300", "kind": "prompt", "path": "unfused", "history": 2100, "tokens": 300, "chunk": 512, "layers": 10},
        # a chunk of the FP16-storage control
        {"name": "fp16_chunk", "kind": "prompt", "path": "fp16", "history": 7680, "tokens": 512, "chunk": 512, "layers": 10},
        # a full verify block after a short prompt
        {"name": "verify_8_1500", "kind": "verify", "history": 1500, "rows": 8, "layers": 10},
        # half a block after the 30K-token prompt
        {"name": "verify_4_30k", "kind": "verify", "history": 30000, "rows": 4, "layers": 10},
    ]


def _log(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "prompt", "prompt", "prompt", "verify", "verify"))
    if kind == "decode":
        return {"kind": kind, "history": _log(rng, 4, WINDOW - 1), "layers": 10}
    if kind == "verify":
        return {"kind": kind, "history": _log(rng, 16, 131072), "rows": rng.randint(1, 8), "layers": 10}
    history = rng.choice((0, _log(rng, 8, 60000)))
    tokens = _log(rng, 8, 2048)
    chunk = rng.choice((512, 512, 2048))
    # at most the key-row pairs of the largest listed case
    layers = max(1, min(10, int(2.5e8 / (tokens * (history + tokens)))))
    return {"kind": kind, "path": rng.choice(("fused", "fused", "unfused", "fp16")), "history": history,
            "tokens": tokens, "chunk": chunk, "layers": layers}


# ---------------------------------------------------------------- inputs

def _rows(case):
    return {"decode": 1, "verify": case.get("rows"), "prompt": case.get("tokens")}[case["kind"]]


def _generator(seed, *what):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + sum(p * x for p, x in zip((7919, 104729, 1299709), what))) & 0x7FFFFFFFFFFF)
    return g


def _unit(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPSILON)


def _key_rows(n, g):
    """K projections with outlier channels, [n][2][256]."""
    k = torch.randn(n, 2, 256, device="cuda", generator=g)
    k[:, :, list(OUTLIERS)] *= 20
    return k


def _history(case, seed, layer):
    """The cached tokens' K (normalized, as the cache holds it) and V, FP32."""
    g, n = _generator(seed, 1, layer), case["history"]
    return _unit(_key_rows(n, g)), torch.randn(n, 2, 256, device="cuda", generator=g)


def _weights(seed, layer):
    """Norm weights in bfloat16 (applied as w + 1): queries 2.3 times unit size give scores of that
    deviation, keys unit size."""
    g = _generator(seed, 2, layer)
    wq = 1.3 + 0.2 * torch.randn(256, device="cuda", generator=g)
    wk = 0.1 * torch.randn(256, device="cuda", generator=g)
    return wq.bfloat16(), wk.bfloat16()


def _fresh(case, seed, layer):
    """What the projections hand over for the new rows: ``qkv`` [n][16][q | gate][256] where the
    norms are part of the pass, else normalized ``q`` and ``gate`` [n][16][256]; k, v [n][2][256]."""
    g, n = _generator(seed, 3, layer), _rows(case)
    x = {"k": _key_rows(n, g), "v": torch.randn(n, 2, 256, device="cuda", generator=g)}
    if case.get("path") in ("fused", "fp16"):
        x["qkv"] = torch.randn(n, 16, 2, 256, device="cuda", generator=g)
        return x
    x["k"] = _unit(x["k"])
    x["q"] = 2.3 * _unit(torch.randn(n, 16, 256, device="cuda", generator=g))
    x["gate"] = torch.randn(n, 16, 256, device="cuda", generator=g)
    return x


# ---------------------------------------------------------------- device memory as tensors

class _Memory:
    """A device buffer that torch can see, released with the last tensor over it. The library hands
    out opaque handles ({context, device pointer, bytes}); the pointer is read from the handle so
    that inputs are made, and outputs looked at, where they are."""

    def __init__(self, buffer):
        self.buffer = buffer
        self.pointer = ctypes.c_uint64.from_address(buffer.handle + 8).value

    @property
    def __cuda_array_interface__(self):
        return {"shape": (self.buffer.length,), "typestr": "|u1", "data": (self.pointer, False), "version": 2}

    def __del__(self):
        if self.buffer is not None and self.buffer.device.handle:
            self.buffer.dispose()


def _tensor(buffer, dtype):
    return torch.as_tensor(_Memory(buffer), device="cuda").view(dtype)


_device = None


def _the_device():
    global _device
    if _device is None:
        _device = Device()
    return _device


class _State:
    def __init__(self, case):
        self.case = case
        self.device = _the_device()
        self.views = []          # keep every buffer of the state alive
        self.caches = []
        self.inputs = []
        self.results = []

    def put(self, tensor):
        buffer = self.device.allocate(tensor.numel() * tensor.element_size())
        view = _tensor(buffer, tensor.dtype)
        view.copy_(tensor.reshape(-1))
        self.views.append(view)
        return buffer

    def take(self, nbytes, dtype=torch.float32):
        buffer = self.device.allocate(nbytes)
        view = _tensor(buffer, dtype)
        self.views.append(view)
        return buffer, view

    def keep(self, layer):
        views = [_tensor(b, t) for b, t in zip(layer.buffers(), self.types)]
        self.views += views
        self.caches.append(layer)
        return views

    types = (torch.int8, torch.int8, torch.float32, torch.float32)


def _store(state, case, seed, layer, index):
    """The history into a layer's INT8 cache, through the framework's store."""
    n = case["history"]
    if n == 0:
        return
    k, v = _history(case, seed, index)
    device = state.device
    buffers = [device.allocate(n * 2048) for _ in range(2)]
    views = [_tensor(b, torch.float32) for b in buffers]
    for view, x in zip(views, (k, v)):
        view.copy_(x.reshape(-1))
    torch.cuda.synchronize()
    device.begin()
    engine.store_rows(device, layer, buffers[0], buffers[1], n, 0)
    device.end()


def prepare(case, seed):
    state = _State(case)
    device, n, first = state.device, _rows(case), case["history"]
    capacity = first + n
    fp16 = case.get("path") == "fp16"
    fused = case.get("path") in ("fused", "fp16")
    if fp16:
        state.types = (torch.float16, torch.float16)
    chunk = min(n, case.get("chunk", n))
    if case["kind"] == "verify":
        floats = min(engine.ATTENTION_WORKSPACE_FLOATS, n * 16 * capacity)
        state.scores = state.take(floats * 4)[0]
    if case["kind"] == "prompt":
        state.workspace = engine.DeviceAttentionWorkspace(device)
        state.workspace.prepare(chunk)
        state.views.append(_tensor(state.workspace.packed_query, torch.float16))
        if fused:
            state.gate = state.take(chunk * 16384)[0]
        else:
            state.rotated = state.take(chunk * 16384)[0]
    for index in range(case["layers"]):
        if fp16:
            layer = engine.Fp16KvLayer(device, capacity)
            key, value = state.keep(layer)
            if first:
                for view, x in zip((key, value), _history(case, seed, index)):
                    view[: first * 512].copy_(x.reshape(-1))
            result = {"key": key[first * 512:], "value": value[first * 512:]}
        else:
            layer = engine.Int8KvLayer(device, capacity)
            key, value, ks, vs = state.keep(layer)
            _store(state, case, seed, layer, index)
            result = {"key": key[first * 512:],
                      "value": value[first // 256 * 256 * 512:],      # whole pages from the first new token's
                      "key_scale": ks[first * 2:], "value_scale": vs[first * 2:]}
        x = {name: state.put(t) for name, t in _fresh(case, seed, index).items()}
        if fused:
            x["wq"], x["wk"] = (state.put(w) for w in _weights(seed, index))
        if case["kind"] != "prompt":
            x["rotated"], view = state.take(n * 16384)
            result["rotated" if case["kind"] == "decode" else "out"] = view.view(n, 16, 256)
        if case["kind"] != "verify":
            x["out"], view = state.take(n * 16384)
            result["out"] = view.view(n, 16, 256)
        state.inputs.append(x)
        state.results.append(result)
    torch.cuda.synchronize()
    return state


def _decode(state):
    device, position = state.device, state.case["history"]
    device.begin()
    for layer, x in zip(state.caches, state.inputs):
        engine.decode_append(device, layer, x["q"], x["k"], x["v"], x["rotated"], x["gate"], x["out"], position)
    device.end()


def _verify(state):
    device, rows, position = state.device, state.case["rows"], state.case["history"]
    device.begin()
    for layer, x in zip(state.caches, state.inputs):
        engine.append_rows(device, layer, x["q"], x["k"], x["v"], x["rotated"], rows, position)
        engine.verify_attention_int8(device, layer, x["rotated"], x["gate"], state.scores, rows, position)
    device.end()


def _prompt(state):
    device, case, workspace = state.device, state.case, state.workspace
    done, path = 0, state.case["path"]
    while done < case["tokens"]:
        rows, position = min(case["chunk"], case["tokens"] - done), case["history"] + done
        device.begin()
        for layer, x in zip(state.caches, state.inputs):
            k, v, out = x["k"].at(done * 2048), x["v"].at(done * 2048), x["out"].at(done * 16384)
            if path == "unfused":
                engine.append_rows(device, layer, x["q"].at(done * 16384), k, v, state.rotated, rows, position)
                workspace.encode_int8(state.rotated, layer.key, layer.value, layer.key_scale, layer.value_scale,
                                      x["gate"].at(done * 16384), out, rows, position)
                continue
            prepare_rows = engine.prepare_fused if path == "fused" else engine.prepare_fused_fp16
            prepare_rows(device, layer, x["qkv"].at(done * 32768), k, v, x["wq"], x["wk"], workspace.packed_query,
                         state.gate, rows, position, epsilon=EPSILON)
            if path == "fused":
                workspace.encode_int8(None, layer.key, layer.value, layer.key_scale, layer.value_scale, state.gate,
                                      out, rows, position, prepared_query=True)
            else:
                engine.encode_online_fp16(workspace, None, layer, state.gate, out, rows, position, prepared_query=True)
        device.end()
        done += rows


def run(state):
    {"decode": _decode, "verify": _verify, "prompt": _prompt}[state.case["kind"]](state)
    return state.results


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    """Per layer: the cached and new keys once (INT8: 1040 bytes a token, FP16: 2048), the new rows'
    inputs and outputs once; two products of 256 multiply-adds per visible key, row and head."""
    n, first = _rows(case), case["history"]
    token = 2048 if case.get("path") == "fp16" else 1040
    row = 4096 + 16384 * 3                              # K and V in; q, gate and the output
    if case["kind"] == "decode":
        row += 16384                                    # the rotated query is an output too
    pairs = n * first + n * (n + 1) // 2
    return {"bytes": float(case["layers"] * (token * (first + n) + row * n)),
            "flops": float(case["layers"] * pairs * 16 * 256 * 4)}


# ---------------------------------------------------------------- exact results

def _rotate(x, first):
    """Partial RoPE of [n][heads][256] from position ``first``: the path defines the angle as the
    FP32 product of the position and the FP32 frequency."""
    n = x.shape[0]
    freq = torch.tensor([THETA ** (-2.0 * j / 64.0) for j in range(32)], dtype=torch.float64).float().cuda()
    angle = (torch.arange(first, first + n, device="cuda").float()[:, None] * freq).double()[:, None, :]
    c, s = torch.cos(angle), torch.sin(angle)
    a, b = x[..., :32], x[..., 32:64]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., 64:]], -1)


def _norm(x, w):
    return x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + EPSILON) * (w.double() + 1)


def _codes(x):
    """(codes, scale) of FP32 vectors along the last axis: the quantizer that defines the cache."""
    x = x.float()
    top = x.abs().amax(-1, keepdim=True)
    # tensor by tensor: torch turns a division by or of a number into a product with a reciprocal
    full = torch.full_like(top, 127.0)
    code = torch.clamp(torch.round(x * torch.where(top > 0, full / top, torch.zeros_like(top))), -127, 127)
    return code, (top / full)[..., 0]


def _held(x, fp16):
    """What the cache gives back for the vectors, in 64 bits, and their scales."""
    if fp16:
        return x.half().double(), None
    code, scale = _codes(x)
    return code.double() * scale.double()[..., None], scale.double()


def _attend(q, k, v, first):
    """softmax(q k / 16) v of [n][16][256] queries, row r seeing keys 0 .. first + r."""
    n, keys = q.shape[0], k.shape[0]
    out = torch.empty_like(q)
    step = max(1, int(1 << 30) // (8 * 8 * keys))
    at = torch.arange(keys, device="cuda")
    for g in range(2):
        kt, vg = k[:, g].t().contiguous(), v[:, g].contiguous()
        for r in range(0, n, step):
            rows = min(step, n - r)
            seen = first + r + rows
            s = torch.mm(q[r:r + rows, 8 * g:8 * g + 8].reshape(rows * 8, 256), kt[:, :seen].contiguous()) / 16.0
            s = s.view(rows, 8, seen)
            s.masked_fill_((at[:seen] > first + r + torch.arange(rows, device="cuda")[:, None])[:, None, :], -math.inf)
            p = torch.softmax(s, -1).view(rows * 8, seen)
            out[r:r + rows, 8 * g:8 * g + 8] = torch.mm(p, vg[:seen]).view(rows, 8, 256)
    return out


def exact(case, seed):
    first, kind, path = case["history"], case["kind"], case.get("path")
    fp16 = path == "fp16"
    results = []
    for index in range(case["layers"]):
        x = _fresh(case, seed, index)
        if path in ("fused", "fp16"):
            wq, wk = _weights(seed, index)
            q, gate = _rotate(_norm(x["qkv"][:, :, 0], wq), first), x["qkv"][:, :, 1].double()
            k = _rotate(_norm(x["k"], wk), first)
        else:
            q, gate = _rotate(x["q"].double(), first), x["gate"].double()
            k = _rotate(x["k"].double(), first)
        new_k, ks = _held(k, fp16)
        new_v, vs = _held(x["v"], fp16)
        old_k, old_v = _history(case, seed, index)
        keys = torch.cat([_held(old_k, fp16)[0], new_k])
        values = torch.cat([_held(old_v, fp16)[0], new_v])
        del old_k, old_v
        # the prefill kernels take the query in FP16, which is the path's own layout for it
        asked = q if kind != "prompt" else q.float().half().double()
        out = _attend(asked, keys, values, first) * torch.sigmoid(gate)
        if fp16:
            results.append({"key": new_k.reshape(-1), "value": new_v.reshape(-1), "out": out})
            continue
        result = {"key": None, "value": None, "key_scale": ks.reshape(-1), "value_scale": vs.reshape(-1), "out": out}
        if kind == "decode":
            result["rotated"] = q
        results.append(result)
    return results


def tolerance(case):
    # Against exact() the FP16 operands of the chunk kernels measure 1.6e-4 to 2.9e-4, the 32-bit
    # paths of decode and verify 3.8e-7 to 6.7e-7; their sums in another order stay below these.
    if case["kind"] == "prompt":
        return {"rel": 1.2e-3, "max": 0.02}
    return {"rel": 5e-6, "max": 2e-4}
