"""The attention path's work as a program has it done, for timing.

Each case is one call, or one captured decode step, through the public entry
points of ``breezetoken_amd.backend.HipBackend``.  ``listed()`` names the
workloads, ``draw(rng)`` gives further ones of the same ranges, ``prepare``
makes what the program holds before the call (inputs from a seed, caches,
weights, plans, captured graphs), ``run`` is one pass, ``work`` the bytes and
operations a pass cannot do without, ``tolerance`` what another correct
implementation at the same precision may differ by, and ``exact`` the same
results in 64 bits from plain torch.

Kinds:

* ``decode``   eager single-token attention over ``seq`` cached keys;
* ``fixed``    one graph replay of the fixed-capacity decode of ``layers``
  attention layers, each on its own cache, at a device position;
* ``step``     the same behind each layer's preparation (q/k norm, RoPE, cache
  writes), as a decode step of a model's attention layers holds it;
* ``batch``    one decode call for sequences sharing a cache, device positions;
* ``ragged``   one decode call for sequences of very different lengths, split
  counts planned on the host (``plan = "host"``) or on the device;
* ``prefill``  causal prompt attention, all keys new;
* ``chunk``    one chunk of a long prompt behind ``offset`` cached keys, with
  the sequence's kept images;
* ``token``    a whole decode step of a small hybrid model in one graph: Gated
  DeltaNet layers, every fourth an attention layer, MLPs, vocabulary head.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from breezetoken_amd.backend import HipBackend, rope_tables
from breezetoken_amd.kvcache import KVCache

DEV = "cuda"
ROPE_DIM, THETA, EPS = 64, 1.0e7, 1e-6
GDN_HEADS, GDN_DIM = 16, 128

_shared: dict = {}


def _backend() -> HipBackend:
    """One backend per process, as a program holds it."""
    if "backend" not in _shared:
        _shared["backend"] = HipBackend(DEV)
    return _shared["backend"]


# ---------------------------------------------------------------------- cases
def listed() -> list[dict]:
    return [
        # The first tokens of a chat: one eager decode call over a few hundred
        # keys, where launches and the host path are the cost.
        dict(name="decode_short", kind="decode", heads=8, kv_heads=2, dim=256, seq=301, q="f32"),
        # The end of a very long context, 8 query heads per kv head, 1% of the
        # keys 8 times as large (they stress the softmax's running maximum).
        dict(name="decode_131k", kind="decode", heads=16, kv_heads=2, dim=256, seq=131072, q="f32"),
        # A decode step's attention layers in one graph at an ordinary context.
        dict(name="step_4k", kind="step", heads=8, kv_heads=2, dim=256, layers=6, cap=8192, valid=4099),
        # The benchmark's decode: six layer caches of 65,536 slots at 32k.
        dict(name="fixed_32k", kind="fixed", heads=8, kv_heads=2, dim=256, layers=6, cap=65536, valid=32768),
        # A small server's batch, similar lengths, head dimension 128, bf16 q.
        dict(name="batch_24", kind="batch", heads=32, kv_heads=8, dim=128, batch=24, longest=3000, q="bf16"),
        # The benchmark's ragged batch of 32, 256 to 32,768 tokens each.
        dict(name="ragged_32", kind="ragged", heads=8, kv_heads=2, dim=256, batch=32, shortest=256, longest=32768,
             lens=4, plan="host"),
        # A busy server's batch with the same spread; its plan is made on the
        # device, so that the lengths never leave it.
        dict(name="ragged_144", kind="ragged", heads=8, kv_heads=2, dim=256, batch=144, shortest=256, longest=32768,
             lens=11, plan="device"),
        # A short prompt; q in f32 as the model's projections leave it.
        dict(name="prefill_333", kind="prefill", heads=8, kv_heads=2, dim=256, steps=333, q="f32", out="f32"),
        # An ordinary long prompt of the larger model, q in f32.
        dict(name="prefill_3001", kind="prefill", heads=16, kv_heads=2, dim=256, steps=3001, q="f32", out="f32"),
        # The benchmark's longest prompt, all in bf16.
        dict(name="prefill_8192", kind="prefill", heads=8, kv_heads=2, dim=256, steps=8192, q="bf16", out="bf16"),
        # A later chunk of a long prompt of the larger model.
        dict(name="chunk_16k", kind="chunk", heads=16, kv_heads=2, dim=256, steps=512, offset=16384, q="bf16",
             out="bf16"),
        # A whole token of a model with the 0.8B model's layer sizes.
        dict(name="token_step", kind="token", heads=8, kv_heads=2, dim=256, layers=8, hidden=1024, ffn=3584,
             vocab=248320, cap=2048, valid=1001),
    ]


# (heads, kv heads, head dim): the 0.8B- and 35B-A3B-like attention layers and
# the head dimension 128 of other GQA models, group sizes 4 and 8.
SHAPES = ((8, 2, 256), (8, 2, 256), (16, 2, 256), (32, 8, 128), (16, 2, 128))


def _log(rng, lo: int, hi: int) -> int:
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))


def draw(rng) -> dict:
    kind = rng.choice(("decode", "decode", "step", "fixed", "batch", "ragged", "ragged", "prefill", "prefill",
                       "prefill", "chunk", "token"))
    heads, kv_heads, dim = rng.choice(SHAPES)
    case = dict(kind=kind, heads=heads, kv_heads=kv_heads, dim=dim)
    dtype = rng.choice(("f32", "bf16"))
    if kind == "decode":
        return dict(case, seq=_log(rng, 17, 131072), q=dtype)
    if kind == "step":
        valid = _log(rng, 64, 16384)
        return dict(case, layers=rng.choice((4, 6, 8)), cap=-(-(valid + rng.randrange(1, 2048)) // 32) * 32, valid=valid)
    if kind == "fixed":
        valid = _log(rng, 256, 32768)
        return dict(case, layers=rng.choice((2, 4, 6)), cap=rng.choice((32768, 40960, 65536)), valid=valid)
    if kind == "batch":
        return dict(case, batch=_log(rng, 2, 64), longest=_log(rng, 200, 8192), q=dtype)
    if kind == "ragged":
        batch = _log(rng, 4, 200)
        return dict(case, batch=batch, shortest=rng.choice((32, 256)), longest=_log(rng, 2000, 32768),
                    lens=rng.randrange(1 << 20), plan=rng.choice(("host", "device")))
    if kind == "prefill":
        return dict(case, steps=_log(rng, 17, 8192), q=dtype, out=rng.choice(("f32", dtype)))
    if kind == "chunk":
        return dict(case, steps=_log(rng, 48, 1024), offset=_log(rng, 500, 16384), q=dtype, out=dtype)
    return dict(case, heads=8, kv_heads=2, dim=256, layers=rng.choice((4, 8)), hidden=rng.choice((1024, 2048)),
                ffn=rng.choice((2048, 3584, 6144)), vocab=rng.choice((4096, 248320)), cap=4096,
                valid=_log(rng, 64, 4000))


# --------------------------------------------------------------------- inputs
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g: torch.Generator, *shape: int, dtype: str = "f32") -> torch.Tensor:
    x = torch.randn(*shape, generator=g, device=DEV)
    return x.to(torch.bfloat16) if dtype == "bf16" else x


def _bf16(g: torch.Generator, *shape: int) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.bfloat16)


def _out_dtype(case: dict) -> torch.dtype:
    return torch.bfloat16 if case["out"] == "bf16" else torch.float32


def _lens(case: dict) -> list[int]:
    """Log-uniform lengths in [shortest, longest], the same for every seed."""
    u = torch.rand(case["batch"], generator=torch.Generator().manual_seed(case["lens"]), dtype=torch.float64)
    lo, hi = math.log(case["shortest"]), math.log(case["longest"])
    return [int(math.exp(lo + float(x) * (hi - lo))) for x in u]


def _batch_lens(case: dict) -> list[int]:
    """Lengths of a batch that was filled together: 60% to 100% of the longest."""
    n, top = case["batch"], case["longest"]
    return [max(1, top - (top * 2 // 5) * i // n) for i in range(n)]


def _offsets(lens: list[int]) -> tuple[list[int], int]:
    """First slots of the sequences' regions, whole 32-slot tiles each."""
    first, total = [], 0
    for n in lens:
        first.append(total)
        total += -(-n // 32) * 32
    return first, total


def _inputs(case: dict, seed: int) -> dict:
    """The case's input tensors; the values a path meets: unit-variance q, K, V."""
    g = _gen(seed)
    kind, H, G, D = case["kind"], case["heads"], case["kv_heads"], case["dim"]
    if kind == "decode":
        q = _randn(g, H, D, dtype=case["q"])
        k, v = _bf16(g, case["seq"], G, D), _bf16(g, case["seq"], G, D)
        rows = torch.randperm(case["seq"] * G, generator=g, device=DEV)[: case["seq"] * G // 100]
        k.view(-1, D)[rows] *= 8.0
        return dict(q=q, k=k, v=v)
    if kind in ("fixed", "step"):
        layers = []
        for _ in range(case["layers"]):
            cache = KVCache(case["cap"], G, D, DEV)
            cache.k[: case["valid"]] = _bf16(g, case["valid"], G * D)
            cache.v[: case["valid"]] = _bf16(g, case["valid"], G * D)
            layer = dict(cache=cache)
            if kind == "fixed":
                layer["q"] = _randn(g, H, D)
            else:
                layer["qkv"] = _randn(g, 2 * H * D + 2 * G * D)
                layer["q_norm"] = 1.0 + 0.1 * _randn(g, D)
                layer["k_norm"] = 1.0 + 0.1 * _randn(g, D)
            layers.append(layer)
        return dict(layers=layers, pos=torch.tensor([case["valid"] - 1], dtype=torch.int32, device=DEV))
    if kind in ("batch", "ragged"):
        lens = _batch_lens(case) if kind == "batch" else _lens(case)
        first, total = _offsets(lens)
        return dict(q=_randn(g, case["batch"], H, D, dtype=case.get("q", "f32")), k=_bf16(g, total, G, D),
                    v=_bf16(g, total, G, D), lens=lens, first=first)
    if kind in ("prefill", "chunk"):
        keys = case["steps"] + case.get("offset", 0)
        return dict(q=_randn(g, case["steps"], H, D, dtype=case["q"]), k=_bf16(g, keys, G, D), v=_bf16(g, keys, G, D))
    return _token_inputs(case, g)


def _token_inputs(case: dict, g: torch.Generator) -> dict:
    H, G, D, N = case["heads"], case["kv_heads"], case["dim"], case["hidden"]
    Hg, Dg = GDN_HEADS, GDN_DIM

    def w(k: int, n: int) -> torch.Tensor:
        return (torch.randn(k, n, generator=g, device=DEV) / math.sqrt(k)).to(torch.bfloat16)

    layers = []
    for i in range(case["layers"]):
        layer = dict(norm=1.0 + 0.1 * _randn(g, N), norm2=1.0 + 0.1 * _randn(g, N),
                     w_gate_up=w(N, 2 * case["ffn"]), w_down=w(case["ffn"], N))
        if i % 4 == 3:
            cache = KVCache(case["cap"], G, D, DEV)
            cache.k[: case["valid"]] = _bf16(g, case["valid"], G * D)
            cache.v[: case["valid"]] = _bf16(g, case["valid"], G * D)
            layer.update(w_in=w(N, 2 * H * D + 2 * G * D), w_o=w(H * D, N), q_norm=1.0 + 0.1 * _randn(g, D),
                         k_norm=1.0 + 0.1 * _randn(g, D), cache=cache)
        else:
            layer.update(w_in=w(N, 3 * Hg * Dg + 2 * Hg), w_o=w(Hg * Dg, N), state=0.1 * _randn(g, Hg, Dg, Dg))
        layers.append(layer)
    return dict(x=_randn(g, N), layers=layers, norm=1.0 + 0.1 * _randn(g, N), w_head=w(N, case["vocab"]),
                pos=torch.tensor([case["valid"] - 1], dtype=torch.int32, device=DEV))


# -------------------------------------------------------------------- prepare
def _tables(cap: int):
    """RoPE tables, built once per capacity as a model does at load time."""
    if ("rope", cap) not in _shared:
        _shared["rope", cap] = rope_tables(cap, ROPE_DIM, THETA, DEV)
    return _shared["rope", cap]


def _captured(fn):
    """``fn`` run once eagerly (workspaces, handles), then captured in a graph."""
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def prepare(case: dict, seed: int) -> dict:
    be = _backend()
    s = _inputs(case, seed)
    s.update(case=case, scale=case["dim"] ** -0.5)
    kind, H, G, D = case["kind"], case["heads"], case["kv_heads"], case["dim"]
    if kind == "fixed":
        s["graph"], s["out"] = _captured(lambda: [
            be.attention_fixed(layer["q"], *layer["cache"].views(), s["pos"], s["scale"]) for layer in s["layers"]])
    elif kind == "step":
        cos, sin = _tables(case["cap"])

        def step():
            outs = []
            for layer in s["layers"]:
                k, v = layer["cache"].views()
                q, _ = be.attn_prep(layer["qkv"], layer["q_norm"], layer["k_norm"], EPS, cos, sin, s["pos"], ROPE_DIM,
                                    k, v, H, G, D)
                outs.append(be.attention_fixed(q, k, v, s["pos"], s["scale"]))
            return outs

        s["graph"], outs = _captured(step)
        s["out"] = dict(out=outs, k=[layer["cache"].k for layer in s["layers"]],
                        v=[layer["cache"].v for layer in s["layers"]])
    elif kind == "token":
        # The warm-up pass before the capture must not advance the states.
        states = [layer["state"] for layer in s["layers"] if "state" in layer]
        kept = [t.clone() for t in states]
        s["graph"], logits = _captured(lambda: _token_step(be, case, s))
        for t, t0 in zip(states, kept):
            t.copy_(t0)
        s["out"] = dict(logits=logits, states=states,
                        k=[layer["cache"].k for layer in s["layers"] if "cache" in layer],
                        v=[layer["cache"].v for layer in s["layers"] if "cache" in layer])
    elif kind in ("batch", "ragged"):
        s["first_slot"] = torch.tensor(s["first"], dtype=torch.int64, device=DEV)
        s["len"] = torch.tensor(s["lens"], dtype=torch.int32, device=DEV)
        s["pos"] = s["len"] - 1
    elif kind == "chunk":
        # The earlier chunks of this sequence left their keys in the images.
        off, top = case["offset"], case["offset"] + case["steps"]
        s["images"] = be.prefill_images(top, G, D)
        be.attention_prefill(s["q"][:1].expand(off, H, D).contiguous(), s["k"][:off], s["v"][:off], s["scale"],
                             _out_dtype(case), images=s["images"])
    return s


def _token_step(be: HipBackend, case: dict, s: dict) -> torch.Tensor:
    H, G, D = case["heads"], case["kv_heads"], case["dim"]
    Hg, Dg = GDN_HEADS, GDN_DIM
    cos, sin = _tables(case["cap"])
    x = s["x"]
    for layer in s["layers"]:
        p = be.linear(F.rms_norm(x, x.shape, layer["norm"], EPS), layer["w_in"])
        if "cache" in layer:
            k, v = layer["cache"].views()
            q, gate = be.attn_prep(p, layer["q_norm"], layer["k_norm"], EPS, cos, sin, s["pos"], ROPE_DIM, k, v, H, G, D)
            o = be.attention_fixed(q, k, v, s["pos"], s["scale"]) * torch.sigmoid(gate)
        else:
            q, k, v, g, beta = p.split((Hg * Dg, Hg * Dg, Hg * Dg, Hg, Hg))
            o = be.gdn_decode(q.view(Hg, Dg), k.view(Hg, Dg), v.view(Hg, Dg), -F.softplus(g), beta, layer["state"],
                              Dg**-0.5)
        x = x + be.linear(o.reshape(-1), layer["w_o"])
        gate, up = be.linear(F.rms_norm(x, x.shape, layer["norm2"], EPS), layer["w_gate_up"]).chunk(2)
        x = x + be.linear(F.silu(gate) * up, layer["w_down"])
    return be.linear(F.rms_norm(x, x.shape, s["norm"], EPS), s["w_head"])


# ------------------------------------------------------------------------ run
def run(s: dict):
    be, case = _backend(), s["case"]
    kind = case["kind"]
    if kind in ("fixed", "step", "token"):
        s["graph"].replay()
        return s["out"]
    if kind == "decode":
        return be.attention(s["q"], s["k"], s["v"], s["scale"])
    if kind == "batch":
        return be.attention_batched(s["q"], s["k"], s["v"], s["pos"], s["first_slot"], s["scale"], case["longest"])
    if kind == "ragged":
        return be.attention_ragged(s["q"], s["k"], s["v"], s["first_slot"], s["len"],
                                   s["lens"] if case["plan"] == "host" else None, s["scale"])
    if kind == "prefill":
        return be.attention_prefill(s["q"], s["k"], s["v"], s["scale"], _out_dtype(case))
    return be.attention_prefill(s["q"], s["k"], s["v"], s["scale"], _out_dtype(case), q_offset=case["offset"],
                                images=s["images"])


# ----------------------------------------------------------------------- work
def work(case: dict) -> dict:
    kind, H, G, D = case["kind"], case["heads"], case["kv_heads"], case["dim"]
    size = {"f32": 4, "bf16": 2}
    row = 2 * G * D * 2  # K and V of one token
    if kind == "decode":
        return {"bytes": case["seq"] * row + H * D * (size[case["q"]] + 4), "flops": 4 * H * D * case["seq"]}
    if kind == "fixed":
        return {"bytes": case["layers"] * (case["valid"] * row + H * D * 8),
                "flops": case["layers"] * 4 * H * D * case["valid"]}
    if kind == "step":
        io = (2 * H * D + 2 * G * D) * 4 + 2 * D * 4 + H * D * 4 + 2 * ROPE_DIM * 4
        return {"bytes": case["layers"] * (case["valid"] * row + io), "flops": case["layers"] * 4 * H * D * case["valid"]}
    if kind in ("batch", "ragged"):
        lens = _batch_lens(case) if kind == "batch" else _lens(case)
        io = case["batch"] * H * D * (size[case.get("q", "f32")] + 4)
        return {"bytes": sum(lens) * row + io, "flops": 4 * H * D * sum(lens)}
    if kind in ("prefill", "chunk"):
        S, off = case["steps"], case.get("offset", 0)
        return {"bytes": (S + off) * row + S * H * D * (size[case["q"]] + size[case["out"]]),
                "flops": 4 * H * D * (S * off + S * (S + 1) // 2)}
    N, Hg, Dg = case["hidden"], GDN_HEADS, GDN_DIM
    n_attn = case["layers"] // 4
    n_gdn = case["layers"] - n_attn
    weights = N * case["vocab"] + case["layers"] * 3 * N * case["ffn"]
    weights += n_attn * (N * (2 * H * D + 2 * G * D) + H * D * N) + n_gdn * (N * (3 * Hg * Dg + 2 * Hg) + Hg * Dg * N)
    state = n_gdn * Hg * Dg * Dg
    keys = n_attn * case["valid"]
    return {"bytes": weights * 2 + 2 * state * 4 + keys * row + (N + case["vocab"]) * 4,
            "flops": 2 * weights + 6 * state + 4 * H * D * keys}


# ------------------------------------------------------------------ tolerance
def tolerance(case: dict) -> dict:
    """About four times what was measured between the path and ``exact``."""
    kind = case["kind"]
    if kind in ("decode", "fixed", "batch", "ragged"):
        # q and P enter the matrix unit as two bf16 terms (about 16 bits), sums
        # in f32: 3e-6 measured, 6e-6 with the scaled keys.
        return {"rel": 2.4e-5, "max": 1e-3}
    if kind in ("prefill", "chunk"):
        # P and V in fp16 (11 bits), sums in f32: 1.7e-4 measured; a bf16 result
        # adds its own rounding: 1.7e-3 measured.
        return {"rel": 6e-3, "max": 3e-2} if case["out"] == "bf16" else {"rel": 7e-4, "max": 7e-3}
    # f32 activations (5e-7 measured in logits and states, 3e-6 behind the
    # attention); a written K value near a bf16 rounding boundary may fall to
    # either side, 2^-8 of itself and up to 2e-5 of a short cache's norm.
    return {"rel": 4e-5, "max": 1e-2}


# ---------------------------------------------------------------------- exact
def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: float) -> torch.Tensor:
    """(H, D) attention of one token over k, v (S, G, D), in float64."""
    H, G = q.shape[0], k.shape[1]
    out = torch.empty(H, q.shape[1], dtype=torch.float64, device=q.device)
    for g in range(G):
        kg, vg = k[:, g].double(), v[:, g].double()
        h = slice(g * H // G, (g + 1) * H // G)
        out[h] = torch.softmax(q[h].double() @ kg.T * scale, dim=-1) @ vg
    return out


def _rms64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x: torch.Tensor, pos: int) -> torch.Tensor:
    """Rotate-half RoPE over the first ROPE_DIM values, the tables' f32 angles."""
    cos, sin = _tables(pos + 1)
    c, s = cos[pos].double(), sin[pos].double()
    half = ROPE_DIM // 2
    rot = x[..., :ROPE_DIM]
    turned = torch.cat((-rot[..., half:], rot[..., :half]), dim=-1)
    return torch.cat((rot * c + turned * s, x[..., ROPE_DIM:]), dim=-1)


def _prep64(case: dict, layer: dict, qkv: torch.Tensor):
    """q, gate and the layer's caches with this token's K and V rows, which are
    stored in bf16."""
    H, G, D, pos = case["heads"], case["kv_heads"], case["dim"], case["valid"] - 1
    qg, k, v = qkv.split((2 * H * D, G * D, G * D))
    q, gate = qg.view(H, 2, D).unbind(1)
    q = _rope64(_rms64(q, layer["q_norm"]), pos)
    k = _rope64(_rms64(k.view(G, D), layer["k_norm"]), pos)
    kc, vc = layer["cache"].k.clone(), layer["cache"].v.clone()
    kc[pos], vc[pos] = k.reshape(-1).to(torch.bfloat16), v.to(torch.bfloat16)
    return q, gate, kc, vc


def exact(case: dict, seed: int):
    s = _inputs(case, seed)
    kind, H, G, D = case["kind"], case["heads"], case["kv_heads"], case["dim"]
    scale = D**-0.5
    if kind == "decode":
        return _attend(s["q"], s["k"], s["v"], scale)
    if kind in ("fixed", "step"):
        n, shape = case["valid"], (case["cap"], G, D)
        outs, ks, vs = [], [], []
        for layer in s["layers"]:
            if kind == "fixed":
                q, kc, vc = layer["q"], layer["cache"].k, layer["cache"].v
            else:
                q, _, kc, vc = _prep64(case, layer, layer["qkv"].double())
            outs.append(_attend(q, kc.view(shape)[:n], vc.view(shape)[:n], scale))
            ks.append(kc)
            vs.append(vc)
        return outs if kind == "fixed" else dict(out=outs, k=ks, v=vs)
    if kind in ("batch", "ragged"):
        return torch.stack([_attend(s["q"][b], s["k"][o : o + n], s["v"][o : o + n], scale)
                            for b, (n, o) in enumerate(zip(s["lens"], s["first"]))])
    if kind in ("prefill", "chunk"):
        S, off = case["steps"], case.get("offset", 0)
        out = torch.empty(S, H, D, dtype=torch.float64, device=DEV)
        key = torch.arange(S + off, device=DEV)
        for g in range(G):
            kt, vg = s["k"][:, g].double().T.contiguous(), s["v"][:, g].double()
            for h in range(g * H // G, (g + 1) * H // G):
                for r0 in range(0, S, 2048):
                    rows = torch.arange(r0, min(S, r0 + 2048), device=DEV)
                    x = s["q"][r0 : r0 + 2048, h].double() @ kt * scale
                    x.masked_fill_(key > off + rows[:, None], -math.inf)
                    out[r0 : r0 + 2048, h] = torch.softmax(x, dim=-1) @ vg
        return out
    return _token64(case, s)


def _token64(case: dict, s: dict) -> dict:
    G, D, n = case["kv_heads"], case["dim"], case["valid"]
    Hg, Dg = GDN_HEADS, GDN_DIM

    def lin(x, w):
        y = torch.empty(w.shape[1], dtype=torch.float64, device=DEV)
        for c in range(0, w.shape[1], 32768):
            y[c : c + 32768] = x @ w[:, c : c + 32768].double()
        return y

    x = s["x"].double()
    states, ks, vs = [], [], []
    for layer in s["layers"]:
        p = lin(_rms64(x, layer["norm"]), layer["w_in"])
        if "cache" in layer:
            q, gate, kc, vc = _prep64(case, layer, p)
            shape = (case["cap"], G, D)
            o = _attend(q, kc.view(shape)[:n], vc.view(shape)[:n], D**-0.5) * torch.sigmoid(gate)
            ks.append(kc)
            vs.append(vc)
        else:
            q, k, v, g, beta = p.split((Hg * Dg, Hg * Dg, Hg * Dg, Hg, Hg))
            q, k, v = (t.view(Hg, Dg) for t in (q, k, v))
            q = q * torch.rsqrt(q.square().sum(-1, keepdim=True) + 1e-6) * Dg**-0.5
            k = k * torch.rsqrt(k.square().sum(-1, keepdim=True) + 1e-6)
            st = layer["state"].double() * torch.exp(-F.softplus(g))[:, None, None]
            delta = (v - (st * k[:, :, None]).sum(1)) * torch.sigmoid(beta)[:, None]
            st = st + k[:, :, None] * delta[:, None, :]
            o = (st * q[:, :, None]).sum(1)
            states.append(st)
        x = x + lin(o.reshape(-1), layer["w_o"])
        gate, up = lin(_rms64(x, layer["norm2"]), layer["w_gate_up"]).chunk(2)
        x = x + lin(F.silu(gate) * up, layer["w_down"])
    return dict(logits=lin(_rms64(x, s["norm"]), s["w_head"]), states=states, k=ks, v=vs)
