"""The work a program has this library do, as cases that can be timed and checked.

Each case is one pass through the public entry points of webllm_amd.qlinear: single quantized linears, whole sequences of
them (decode and prefill), decoder layers with attention over the KV cache, the tied lm_head, prefill attention, and the
load-time unpack. Inputs are made on the GPU from a seed with plain torch; `prepare` puts them into the library's arenas
with the plans a program would keep, `run` is the pass, `exact` the same result in 64-bit torch arithmetic.
"""
import math

import torch

from webllm_amd import qlinear as ql

# (C, intermediate, heads, kv heads, head dim) of the two model shapes the benchmark and the tests use.
MODELS = {"05b": (896, 4864, 14, 2, 64), "7b": (3584, 18944, 28, 4, 128)}
EPS = 1e-6
VOCAB = 151936


def listed():
    return [
        # One q/o projection for one token: the smallest call, launch latency.
        {"name": "linear_05b_m1", "kind": "linear", "M": 1, "K": 896, "N": 896, "count": 1, "x": "f32", "bias": True,
         "asym": False},
        # The benchmark's decode step: the 168 linears of a 24-layer model, each on an input of its own.
        {"name": "step_05b_m1", "kind": "step", "model": "05b", "layers": 24, "M": 1},
        # The same linears as a decode step has them: chained through RMSNorm, SiLU-mul and residuals.
        {"name": "chain_05b_m1", "kind": "chain", "model": "05b", "layers": 24, "M": 1},
        # Batched decode (8 rows) of the large model's layers, chained.
        {"name": "chain_7b_m8", "kind": "chain", "model": "7b", "layers": 4, "M": 8},
        # One decoder layer of token generation at a long context: cache store, attention, then o, gate, up, down and the
        # next layer's q, k, v as one sequence.
        {"name": "layer_7b_t4000", "kind": "layer", "model": "7b", "M": 1, "past": 4000},
        # A prompt of 512 tokens through the whole model's linears in their order.
        {"name": "prefill_chain_05b_m512", "kind": "chain", "model": "05b", "layers": 24, "M": 512},
        # A short ragged prompt, one linear per call, fp32 activations, asymmetric zero points.
        {"name": "prefill_linear_m77", "kind": "linear", "M": 77, "K": 3584, "N": 3584, "count": 1, "x": "f32",
         "bias": False, "asym": True},
        # gate and up of the large model on a 512-token prompt with fp16 activations: matrix-core bound.
        {"name": "prefill_gate_up_7b_m512", "kind": "linear", "M": 512, "K": 3584, "N": 18944, "count": 2, "x": "f16",
         "bias": False, "asym": False},
        # The tied lm_head of one decoded token: the largest single read of a step.
        {"name": "lm_head_m1", "kind": "head", "M": 1, "K": 896, "N": VOCAB},
        # Logits of every position of a 256-token prompt, as a forward over a prompt returns them.
        {"name": "lm_head_m256", "kind": "head", "M": 256, "K": 896, "N": VOCAB},
        # Prefill attention: the second 1024-token chunk of a 2048-token prompt.
        {"name": "attn_7b_m1024", "kind": "attn", "model": "7b", "M": 1024, "past": 1024},
        # Load-time dequantization of the small model's weights into the fp16 arena.
        {"name": "unpack_05b", "kind": "unpack", "model": "05b", "layers": 24},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "prefill", "prefill", "step", "chain", "chain", "prefill_chain", "layer",
                       "head", "attn", "unpack"])
    model = rng.choice(["05b", "7b"])
    C, I = MODELS[model][:2]
    if kind in ("linear", "prefill"):
        M = _log(rng, 1, 16) if kind == "linear" else _log(rng, 17, 1024)
        if rng.random() < 0.5:
            K, N = rng.choice([(C, C), (C, I), (I, C)])
        else:
            K, N = 128 * _log(rng, 4, 148), 8 * _log(rng, 16, 2368)
        count = rng.choice([1, 1, 2, 3])
        while M * K * N * count > 512 * 3584 * 18944 * 2:
            M = max(17, M // 2 + rng.randrange(8))
            count = 1
        return {"kind": "linear", "M": M, "K": K, "N": N, "count": count, "x": rng.choice(["f32", "f16"]),
                "bias": rng.random() < 0.4, "asym": rng.random() < 0.3}
    if kind in ("step", "chain"):
        layers = rng.randint(8, 24) if model == "05b" else rng.randint(2, 6)
        return {"kind": kind, "model": model, "layers": layers, "M": _log(rng, 1, 16)}
    if kind == "prefill_chain":
        layers = rng.randint(4, 24) if model == "05b" else rng.randint(1, 2)
        return {"kind": "chain", "model": model, "layers": layers, "M": _log(rng, 17, 512)}
    if kind == "layer":
        return {"kind": "layer", "model": model, "M": rng.choice([1, 1, 1, 2, 3, 4, 5]), "past": _log(rng, 16, 8000)}
    if kind == "head":
        K = rng.choice([512, 896, 896, 2048, 3584])
        return {"kind": "head", "M": _log(rng, 1, 256), "K": K,
                "N": VOCAB if K <= 896 and rng.random() < 0.6 else 16 * _log(rng, 500, 4096) + rng.choice([0, 0, 1, 5])}
    if kind == "attn":
        M = _log(rng, 17, 1024)
        past = 0 if rng.random() < 0.5 else _log(rng, 16, 4000)
        while M * (past + M // 2) > 1024 * 1536:
            past //= 2
        return {"kind": "attn", "model": model, "M": M, "past": past}
    layers = rng.randint(4, 24) if model == "05b" else rng.randint(1, 2)
    return {"kind": "unpack", "model": model, "layers": layers}


# ------------------------------------------------------------------ inputs, from the seed alone, in plain torch

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * scale


def _linear(g, K, N, bias=False, asym=False):
    """One GPTQ linear of group 128: random nibbles, stored zeros 7 (symmetric checkpoints) or any, fp16 scales."""
    def words(*shape):
        return torch.randint(-2**31, 2**31, shape, generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
    G = K // 128
    return {"K": K, "N": N, "qw": words(K // 8, N),
            "qz": words(G, N // 8) if asym else torch.full((G, N // 8), 0x77777777, dtype=torch.int32, device="cuda"),
            "sc": (_normal(g, G, N).abs() * 0.01).to(torch.float16),
            "bias": _normal(g, N, scale=0.1) if bias else None}


def _layer_shapes(model, kind):
    """(name, K, N) of a layer's linears in execution order: the benchmark's step of the large model leaves k and v out."""
    C, I, _, KV, D = MODELS[model]
    kv = [("k", C, KV * D), ("v", C, KV * D)] if model == "05b" or kind == "layer" else []
    return [("q", C, C)] + kv + [("o", C, C), ("gate", C, I), ("up", C, I), ("down", I, C)]


def _inputs(case, seed):
    g, kind, M = _gen(seed), case["kind"], case.get("M", 0)
    if kind == "linear":
        x = _normal(g, M, case["K"])
        return {"x": x.to(torch.float16) if case["x"] == "f16" else x,
                "lin": [_linear(g, case["K"], case["N"], case["bias"], case["asym"]) for _ in range(case["count"])]}
    if kind == "head":
        return {"x": _normal(g, M, case["K"]), "w": _normal(g, case["N"], case["K"], scale=0.02).to(torch.float16)}
    C, I, H, KV, D = MODELS[case["model"]]
    if kind in ("attn", "layer"):
        T = case["past"] + M
        d = {"q": _normal(g, M, H * D), "k": _normal(g, T, KV * D), "v": _normal(g, T, KV * D)}
        if kind == "layer":
            d["h"] = _normal(g, M, C)
            d["lin"] = {n: _linear(g, k, N, bias=n in ("q", "k", "v")) for n, k, N in _layer_shapes(case["model"], kind)}
            d["norm"] = [1 + _normal(g, C, scale=0.1) for _ in range(2)]
        return d
    d = {"lin": [{n: _linear(g, k, N, bias=n in ("q", "k", "v")) for n, k, N in _layer_shapes(case["model"], kind)}
                 for _ in range(case["layers"])]}
    if kind == "step":
        d["x"] = [{n: _normal(g, M, l["K"]) for n, l in layer.items()} for layer in d["lin"]]
    if kind == "chain":
        d["h"] = _normal(g, M, C)
        d["norm"] = [[1 + _normal(g, C, scale=0.1) for _ in range(2)] for _ in range(case["layers"])]
    return d


# ------------------------------------------------------------------ the library's side

_context = None


def _ctx():
    """One context (device, stream) per process, as a program keeps it."""
    global _context
    if _context is None:
        _context = ql.Context(0)
    return _context


class _Bytes:
    def __init__(self, arena, off, shape, kind):
        self.arena = arena
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "version": 3,
                                         "data": (arena.device_ptr + off, False)}


_KINDS = {torch.float32: "<f4", torch.float16: "<f2", torch.int32: "<i4"}


class _Arena:
    """Tensors laid out in one device arena: take() reserves, place() copies in, view() is the memory as a tensor."""

    def __init__(self):
        self.lay, self.todo, self.arena = ql.ArenaLayout(), [], None

    def take(self, *shape, dtype=torch.float32):
        return self.lay.take(math.prod(shape) * torch.empty((), dtype=dtype).element_size())

    def put(self, t):
        off = self.take(*t.shape, dtype=t.dtype)
        self.todo.append((off, t))
        return off

    def linear(self, l):
        return ql.make_desc(self.put(l["qw"]), self.put(l["qz"]), self.put(l["sc"]), l["K"], l["N"], 128,
                            None if l["bias"] is None else self.put(l["bias"]))

    def place(self):
        self.arena = _ctx().arena(self.lay.used)
        for off, t in self.todo:
            self.view(off, t.shape, t.dtype).copy_(t)
        self.todo = []
        return self.arena

    def view(self, off, shape, dtype=torch.float32):
        return torch.as_tensor(_Bytes(self.arena, off, shape, _KINDS[dtype]), device="cuda")


class _State:
    """A program's handles: call() is the pass, outputs the arena memory it fills. A sequence holds its arenas by address
    only, so the state keeps them, and ends the sequence first."""

    def __init__(self, *arenas):
        self.arenas, self.seq = arenas, None

    def __del__(self):
        if self.seq is not None:
            self.seq.destroy()


def _by_layer(arena, offs, counts, layers, dtype):
    """One tensor per layer over its linears' outputs, which lie one after the other (their sizes are whole 256 bytes)."""
    per = len(offs) // layers
    return [arena.view(offs[i], (sum(counts[i:i + per]),), dtype) for i in range(0, len(offs), per)]


def _prepare_layer(case, d, w, a, cache, s):
    C, I, H, KV, D = MODELS[case["model"]]
    M, past, ctx = case["M"], case["past"], _ctx()
    T, row = past + M, KV * D
    q, new_k, new_v, h = a.put(d["q"]), a.put(d["k"][past:]), a.put(d["v"][past:]), a.put(d["h"])
    at = a.take(M, H * D)
    norm = [w.put(t) for t in d["norm"]]
    desc = {n: w.linear(l) for n, l in d["lin"].items()}
    order = ["o", "gate", "up", "down", "q", "k", "v"]
    y = {n: a.take(M, d["lin"][n]["N"]) for n in order}
    xs = [at, y["o"], y["o"], y["gate"]] + [y["down"]] * 3
    fuse = [ql.make_fuse(res_off=h)] + [ql.make_fuse(norm_w_off=norm[0], norm_eps=EPS)] * 2 + \
        [ql.make_fuse(x2_off=y["up"], res_off=y["o"])] + [ql.make_fuse(norm_w_off=norm[1], norm_eps=EPS)] * 3
    zero = torch.zeros(M, row, device="cuda")
    kc, vc = (cache.put(torch.cat([d[n][:past], zero])) for n in ("k", "v"))
    W, A, S = w.place(), a.place(), cache.place()
    s.seq = seq = ctx.seq([desc[n] for n in order], W, A, xs, ql.DTYPE_F32, M, [y[n] for n in order], fuse=fuse)

    def call():
        ctx.kv_store(A, new_k, S, kc, T, M, row, past)
        ctx.kv_store(A, new_v, S, vc, T, M, row, past)
        ctx.attention_decode(A, q, S, kc, vc, T, M, H, KV, D, past, at)
        seq.run()

    s.call = call
    s.outputs = [a.view(at, (M, H * D))] + [a.view(y[n], (M, d["lin"][n]["N"])) for n in ("down", "q", "k", "v")] + \
        [cache.view(c + past * row * 4, (M, row)) for c in (kc, vc)]


def prepare(case, seed):
    kind, M, d, ctx = case["kind"], case.get("M", 0), _inputs(case, seed), _ctx()
    w, a, cache = _Arena(), _Arena(), _Arena()
    s = _State(w, a, cache)
    if kind == "linear":
        descs = [w.linear(l) for l in d["lin"]]
        x, n = a.put(d["x"]), len(descs)
        ys = [a.take(M, case["N"]) for _ in descs]
        scratch = a.lay.take(max(16, ql.plan_linear(M, case["N"], case["K"], 128).scratch_bytes if n == 1 else
                                 ql.plan_batch(descs, M)))
        W, A, dt = w.place(), a.place(), ql.DTYPE_F16 if case["x"] == "f16" else ql.DTYPE_F32
        if n == 1:
            s.call = lambda: ctx.linear(descs[0], W, A, x, dt, M, ys[0], scratch)
        else:
            s.call = lambda: ctx.linear_batch(descs, W, A, [x] * n, dt, M, ys, scratch)
        s.outputs = [a.view(y, (M, case["N"])) for y in ys]
    elif kind == "head":
        wo, x, y = w.put(d["w"]), a.put(d["x"]), a.take(M, case["N"])
        W, A = w.place(), a.place()
        s.call = lambda: ctx.gemv_f16w(W, wo, None, A, x, M, case["N"], case["K"], y)
        s.outputs = [a.view(y, (M, case["N"]))]
    elif kind == "attn":
        C, I, H, KV, D = MODELS[case["model"]]
        past = case["past"]
        T = past + M
        k, v, q, o = w.put(d["k"]), w.put(d["v"]), a.put(d["q"]), a.take(M, H * D)
        W, A = w.place(), a.place()
        s.call = lambda: ctx.attention_decode(A, q, W, k, v, T, M, H, KV, D, past, o)
        s.outputs = [a.view(o, (M, H * D))]
    elif kind == "layer":
        _prepare_layer(case, d, w, a, cache, s)
    elif kind == "step":
        flat = [(n, l, x[n]) for layer, x in zip(d["lin"], d["x"]) for n, l in layer.items()]
        descs, xs = [w.linear(l) for _, l, _ in flat], [a.put(x) for _, _, x in flat]
        ys = [a.take(M, l["N"]) for _, l, _ in flat]
        W, A = w.place(), a.place()
        s.seq = ctx.seq(descs, W, A, xs, ql.DTYPE_F32, M, ys)
        s.call = s.seq.run
        s.outputs = _by_layer(a, ys, [M * t.N for t in descs], case["layers"], torch.float32)
    elif kind == "chain":
        descs, xs, ys, fuse, h, keep = [], [], [], [], a.put(d["h"]), []
        for i, (layer, norm) in enumerate(zip(d["lin"], d["norm"])):
            nw, y = [w.put(t) for t in norm], {}
            for n, l in layer.items():
                descs.append(w.linear(l))
                y[n] = a.take(M, l["N"])
                ys.append(y[n])
                if n in ("q", "k", "v"):
                    xs.append(h)
                    fuse.append(ql.make_fuse(norm_w_off=nw[0], norm_eps=EPS))
                elif n == "o":
                    xs.append(y["q"])
                    fuse.append(ql.make_fuse(res_off=h))
                elif n in ("gate", "up"):
                    xs.append(y["o"])
                    fuse.append(ql.make_fuse(norm_w_off=nw[1], norm_eps=EPS))
                else:
                    xs.append(y["gate"])
                    fuse.append(ql.make_fuse(x2_off=y["up"], res_off=y["o"]))
                if n in ("k", "v"):
                    keep.append((y[n], (M, l["N"])))
            h = y["down"]
        keep.append((h, d["h"].shape))
        W, A = w.place(), a.place()
        s.seq = ctx.seq(descs, W, A, xs, ql.DTYPE_F32, M, ys, fuse=fuse)
        s.call = s.seq.run
        s.outputs = [a.view(off, shape) for off, shape in keep]
    elif kind == "unpack":
        descs = [w.linear(l) for layer in d["lin"] for l in layer.values()]
        offs = [a.take(l["N"], l["K"], dtype=torch.float16) for layer in d["lin"] for l in layer.values()]
        W, A = w.place(), a.place()
        s.call = lambda: ctx.unpack_f16_batch(descs, W, A, offs)
        s.outputs = _by_layer(a, offs, [t.N * t.K for t in descs], case["layers"], torch.float16)
    else:
        raise ValueError(kind)
    torch.cuda.synchronize()
    return s


def run(state):
    state.call()
    return state.outputs


# ------------------------------------------------------------------ what a pass cannot do without

def _linear_work(M, K, N, x_bytes=4, bias=False):
    """Packed weights, zeros, scales once; x once, y once."""
    return K * N // 2 + K * N // 256 + K * N // 64 + M * K * x_bytes + M * N * 4 + (N * 4 if bias else 0), 2 * M * K * N


def work(case):
    kind, M = case["kind"], case.get("M", 0)
    if kind == "linear":
        K, N, n = case["K"], case["N"], case["count"]
        xb = 2 if case["x"] == "f16" else 4
        b, f = _linear_work(M, K, N, xb, case["bias"])
        return {"bytes": n * b - (n - 1) * M * K * xb, "flops": n * f}
    if kind == "head":
        K, N = case["K"], case["N"]
        return {"bytes": 2 * K * N + 4 * M * (K + N), "flops": 2 * M * K * N}
    C, I, H, KV, D = MODELS[case["model"]]
    if kind == "unpack":
        kn = sum(K * N for _, K, N in _layer_shapes(case["model"], kind))
        return {"bytes": case["layers"] * (kn // 2 + kn // 256 + kn // 64 + 2 * kn), "flops": 0}
    total = {"bytes": 0, "flops": 0}
    if kind in ("attn", "layer"):
        T = case["past"] + M
        total = {"bytes": 8 * T * KV * D + 8 * M * H * D, "flops": 4 * H * D * sum(case["past"] + m + 1 for m in range(M))}
    if kind == "attn":
        return total
    layers = case.get("layers", 1)
    for n, K, N in _layer_shapes(case["model"], kind):
        b, f = _linear_work(M, K, N, 4, n in ("q", "k", "v"))
        if kind != "step":      # chained: only the weights, and what goes in and out of the chain, have to pass through memory
            b -= 4 * M * (K + N)
        total["bytes"] += layers * b
        total["flops"] += layers * f
    if kind == "chain":
        total["bytes"] += 8 * M * C + (layers * 8 * M * KV * D if case["model"] == "05b" else 0) + layers * 8 * C
    if kind == "layer":
        total["bytes"] += 4 * M * (3 * C + 4 * KV * D) + 8 * C
    return total


def tolerance(case):
    """What another correct implementation of the same precision may show: fp32 sums in another order (decode, attention,
    the fp16-weight head, and fp16 operands with fp32 sums); for a layer, whose RMSNorm'd outputs are up to 7e-6 from the
    64-bit result, four times that; for a chain of prefill layers, where an activation that crosses an fp16 rounding moves
    all that follow (up to 3e-3 from the 64-bit result over 24 layers), about four times that; exact bits for the unpack."""
    kind = case["kind"]
    if kind == "unpack":
        return "exact"
    if kind == "chain" and case["M"] > 16:
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 3e-5 if kind == "layer" else 1e-5}


# ------------------------------------------------------------------ the same in 64 bits

def _weight(l):
    """fp64 [K, N] of a packed linear: (q - (z + 1)) * s."""
    shift = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    q = ((l["qw"][:, None, :] >> shift[None, :, None]) & 15).reshape(l["K"], l["N"])
    z = ((l["qz"][:, :, None] >> shift) & 15).reshape(l["K"] // 128, l["N"]) + 1
    return (q - z.repeat_interleave(128, 0)).double() * l["sc"].double().repeat_interleave(128, 0)


def _mul(x, l):
    y = x.double() @ _weight(l)
    return y if l["bias"] is None else y + l["bias"].double()


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _glu(g, u):
    return g / (1 + torch.exp(-g)) * u


def _attend(q, k, v, case):
    C, I, H, KV, D = MODELS[case["model"]]
    M, T = q.shape[0], k.shape[0]
    q, k, v = (t.double().reshape(t.shape[0], -1, D) for t in (q, k, v))
    seen = torch.arange(T, device="cuda")[None, :] <= case["past"] + torch.arange(M, device="cuda")[:, None]
    out = []
    for h in range(H):
        kv = h // (H // KV)
        score = (q[:, h] @ k[:, kv].T.contiguous()) / math.sqrt(D)
        out.append(torch.softmax(score.masked_fill(~seen, -math.inf), -1) @ v[:, kv].contiguous())
    return torch.stack(out, 1).reshape(M, H * D)


def exact(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        return [_mul(d["x"], l) for l in d["lin"]]
    if kind == "head":
        rows = 16384
        return [torch.cat([d["x"].double() @ d["w"][i:i + rows].double().T.contiguous()
                           for i in range(0, case["N"], rows)], 1)]
    if kind == "attn":
        return [_attend(d["q"], d["k"], d["v"], case)]
    if kind == "step":
        return [torch.cat([_mul(x[n], l).reshape(-1) for n, l in layer.items()]) for layer, x in zip(d["lin"], d["x"])]
    if kind == "unpack":
        return [torch.cat([_weight(l).T.reshape(-1) for l in layer.values()]) for layer in d["lin"]]
    if kind == "layer":
        L, past = d["lin"], case["past"]
        at = _attend(d["q"], d["k"], d["v"], case)
        o = _mul(at, L["o"]) + d["h"].double()
        n = _norm(o, d["norm"][0])
        h = _mul(_glu(_mul(n, L["gate"]), _mul(n, L["up"])), L["down"]) + o
        n = _norm(h, d["norm"][1])
        return [at, h] + [_mul(n, L[p]) for p in ("q", "k", "v")] + [d["k"][past:].double(), d["v"][past:].double()]
    h, keep = d["h"].double(), []
    for L, norm in zip(d["lin"], d["norm"]):
        n = _norm(h, norm[0])
        keep += [_mul(n, L[p]) for p in ("k", "v") if p in L]
        o = _mul(_mul(n, L["q"]), L["o"]) + h
        n = _norm(o, norm[1])
        h = _mul(_glu(_mul(n, L["gate"]), _mul(n, L["up"])), L["down"]) + o
    return keep + [h]
