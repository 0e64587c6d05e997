"""The work a user of this package gives it, as cases that can be timed and compared.

Four families, each through the public entry point that a program calls:
  linear  BC_LinearEXL3.run_alloc (one projection), or linear() over fused projections that share the input (q|k|v)
  mlp     BC_GatedMLP.forward (a dense gated MLP)
  moe     BlockSparseMLP.forward (routing from router logits or from a router weight, routed experts, shared expert)
  blobs   moe_forward_blobs (experts as contiguous blobs in PLANAR4 word order)
Weights are uniformly random trellis words (every word is a valid weight), random +-1 input signs and +-1 / sqrt(k)
output signs, which keeps layer outputs O(1); activations are N(0, 1) fp16 rows, as after a norm.
"""
import importlib
import math

import torch

exl3 = importlib.import_module("b70-inference_amd")


# ------------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # one decode token through one projection of a 4-bit dense model: the smallest call, latency and host path
        dict(name="linear_decode", kind="linear", k=4096, n=4096, shards=1, K=4, rows=1, out32=False),
        # a verify block of 6 tokens through the widest projection of a 31B-class dense model
        dict(name="linear_verify", kind="linear", k=5376, n=21504, shards=1, K=4, rows=6, out32=False),
        # a short prompt (ragged row count) through a fused q|k|v projection at 5 bits
        dict(name="qkv_short_prompt", kind="linear", k=4096, n=6144, shards=3, K=5, rows=77, out32=False),
        # an ordinary prefill chunk through a square projection, fp32 output
        dict(name="linear_chunk", kind="linear", k=4096, n=4096, shards=1, K=3, rows=512, out32=True),
        # a full 2048-token prefill chunk through the widest projection: the largest dense call
        dict(name="linear_prefill", kind="linear", k=5376, n=21504, shards=1, K=4, rows=2048, out32=False),
        # one decode token through the dense MLP
        dict(name="mlp_decode", kind="mlp", H=5376, I=21504, K=4, rows=1, act="gelu_tanh"),
        # a ragged prompt through the dense MLP
        dict(name="mlp_prefill", kind="mlp", H=5376, I=21504, K=4, rows=397, act="gelu_tanh"),
        # one decode token through a sparse layer of many small experts, router included
        dict(name="moe_decode", kind="moe", H=2048, I=512, E=512, topk=10, Kgu=3, Kd=3, shared=False, rows=1, router=True,
             zipf=False),
        # a batch of 8 sequences decoding through the same layer
        dict(name="moe_decode_batch", kind="moe", H=2048, I=512, E=512, topk=10, Kgu=3, Kd=3, shared=False, rows=8,
             router=True, zipf=False),
        # a 512-token prefill chunk over 160 wide experts with a skewed (Zipf) expert load
        dict(name="moe_prefill", kind="moe", H=5120, I=1536, E=160, topk=8, Kgu=2, Kd=3, shared=False, rows=512,
             router=False, zipf=True),
        # 4 decode rows and a 256-row prefill chunk together, per-tile 1/2-bit experts and a shared expert
        dict(name="moe_mixed_bits", kind="moe", H=7168, I=2048, E=256, topk=8, Kgu=0, Kd=0, shared=True, rows=260,
             router=False, zipf=False),
        # a 1024-token prefill chunk over expert blobs as the reference packs them
        dict(name="blobs_prefill", kind="blobs", H=2560, I=640, E=512, topk=10, K=3, rows=1024, bf16=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo, hi):
    return 128 * max(1, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 128)))


def draw(rng):
    while True:
        kind = rng.choice(("linear", "linear", "mlp", "moe", "moe", "blobs"))
        if kind == "linear":
            shards = rng.choice((1, 1, 3))
            c = dict(kind=kind, k=_dim(rng, 1024, 8192), n=_dim(rng, 1024, 21504), shards=shards,
                     K=rng.choice((2, 3, 4, 4, 5, 6, 8)), rows=_log(rng, 1, 2048), out32=rng.random() < 0.5)
            if shards > 1 and c["n"] < 128 * shards:
                continue
        elif kind == "mlp":
            c = dict(kind=kind, H=_dim(rng, 1024, 5376), I=_dim(rng, 1024, 21504), K=rng.choice((2, 3, 4, 5, 6)),
                     rows=_log(rng, 1, 1024), act=rng.choice(("silu", "gelu_tanh")))
        elif kind == "moe":
            E = rng.choice((8, 32, 64, 128, 160, 256, 512))
            mixed = rng.random() < 0.2
            K = rng.choice((2, 3, 4))
            c = dict(kind=kind, H=_dim(rng, 1024, 7168), I=_dim(rng, 512, 4096 if E <= 64 else 2048), E=E,
                     topk=2 if E == 8 else rng.choice((4, 8, 10)), Kgu=0 if mixed else K,
                     Kd=0 if mixed else rng.choice((K, 3)), shared=rng.random() < 0.4, rows=_log(rng, 1, 1024),
                     router=rng.random() < 0.5, zipf=rng.random() < 0.3)
        else:
            c = dict(kind=kind, H=_dim(rng, 1024, 4096), I=_dim(rng, 512, 1536), E=rng.choice((64, 128, 256, 512)),
                     topk=rng.choice((4, 8, 10)), K=rng.choice((2, 3, 4)), rows=_log(rng, 1, 1024),
                     bf16=rng.random() < 0.5)
        # no dearer than the largest listed ones: weights to generate and read, operations, expert row blocks
        if _weights(c) > 3.8e9 or _flops(c) > 2.1e11 * (2.2 if kind == "linear" else 1.0):
            continue
        return c


# ------------------------------------------------------------------------------------------------ work
def _weights(c):
    if c["kind"] == "linear":
        return c["k"] * c["n"]
    if c["kind"] == "mlp":
        return 3 * c["H"] * c["I"]
    return 3 * c["H"] * c["I"] * (c["E"] + (1 if c.get("shared") else 0))


def _flops(c):
    if c["kind"] == "linear":
        return 2.0 * c["rows"] * c["k"] * c["n"]
    if c["kind"] == "mlp":
        return 6.0 * c["rows"] * c["H"] * c["I"]
    return 6.0 * c["rows"] * (c["topk"] + (1 if c.get("shared") else 0)) * c["H"] * c["I"]


def work(case):
    """Bytes: the trellis words and signs of every matrix touched once (routed experts: those that a uniform routing is
    expected to touch), the rows in and out once. Operations: the matrix products."""
    c = case
    r = c["rows"]
    if c["kind"] == "linear":
        b = c["k"] * c["n"] * c["K"] / 8 + 2 * c["k"] * c["shards"] + 2 * c["n"] + 2 * r * c["k"] \
            + (4 if c["out32"] else 2) * r * c["n"]
    elif c["kind"] == "mlp":
        b = 3 * c["H"] * c["I"] * c["K"] / 8 + 6 * (c["H"] + c["I"]) + 6 * r * c["H"]
    else:
        E, k = c["E"], c["topk"]
        touched = E * (1 - (1 - k / E) ** r)
        bits = (c["K"], c["K"]) if c["kind"] == "blobs" else tuple(1.62 if v == 0 else v for v in (c["Kgu"], c["Kd"]))
        per = c["H"] * c["I"] * (2 * bits[0] + bits[1]) / 8 + 6 * (c["H"] + c["I"])
        b = (touched + (1 if c.get("shared") else 0)) * per + (4 if c["kind"] == "blobs" else 6) * r * c["H"]
        b += 8 * r * k if c["kind"] == "blobs" else 2 * E * c["H"] if c["router"] else 4 * r * E
    return {"bytes": float(b), "flops": float(_flops(c))}


def tolerance(case):
    # Each rounding to fp16 (the transformed input; in an MLP also gate, up, activation and down input) leaves about
    # 2e-4 of the result's norm: single projections measure 3.0e-4 (fp32 rows) and 3.6e-4 (fp16 rows) against 64 bits,
    # gated layers 6.4e-4. About four times that.
    if case["kind"] == "linear":
        return {"rel": 1.2e-3}
    if case["kind"] == "blobs" and case["bf16"]:
        return {"rel": 8e-3}                    # rows out in bf16: its own rounding is 1.7e-3
    return {"rel": 2.5e-3}


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _signs(shape, g, scale=1.0):
    return ((torch.randint(0, 2, shape, device="cuda", generator=g).float() * 2 - 1) * scale).half()


def _isqrt(k):
    return float(torch.tensor(1.0 / math.sqrt(k)).half())


def _packed(E, k, n, K, g):
    """E projections k -> n in one allocation per tensor kind, as a loader lays them out."""
    tr = torch.randint(-32768, 32768, (E, k // 16, n // 16, 16 * K), dtype=torch.int16, device="cuda", generator=g)
    su, sv = _signs((E, k), g), _signs((E, n), g, _isqrt(k))
    return [exl3.BC_LinearEXL3(tr[e], su[e], sv[e], K, None, False, True, None) for e in range(E)]


def _mixed(k, n, g):
    """A projection whose tiles hold 1 or 2 bits a weight (38 / 62)."""
    nt = (k // 16) * (n // 16)
    kmap = (1 + (torch.rand(nt, device="cuda", generator=g) >= 0.38)).to(torch.uint8)
    woff = torch.zeros(nt + 1, dtype=torch.int64, device="cuda")
    woff[1:] = torch.cumsum(kmap.to(torch.int64) * 8, 0)
    words = torch.randint(-(2 ** 31), 2 ** 31, (int(woff[-1]),), dtype=torch.int64, device="cuda",
                          generator=g).to(torch.int32)
    return exl3.MixedEXL3(words, kmap, woff.to(torch.int32), _signs((k,), g), _signs((n,), g, _isqrt(k)))


def _experts(E, k, n, K, g):
    return [_mixed(k, n, g) for _ in range(E)] if K == 0 else _packed(E, k, n, K, g)


def _shard_widths(n, shards):
    """A query projection and equally wide key and value projections, in whole 128-column blocks."""
    kv = max(1, n // 128 // 6)
    return [n] if shards == 1 else [n - 128 * kv * (shards - 1)] + [128 * kv] * (shards - 1)


def _blob_layout(H, I, K):
    """Word and byte sizes of an expert blob: gate|up trellis, down trellis, the six sign vectors."""
    gu, dn = (H // 16) * (2 * I // 16) * 8 * K, (I // 16) * (H // 16) * 8 * K
    return gu, dn, 4 * (gu + dn) + 2 * 3 * (H + I)


def prepare(case, seed):
    c, g = case, _gen(seed)
    r = c["rows"]
    if c["kind"] == "linear":
        lins = [_packed(1, c["k"], w, c["K"], g)[0] for w in _shard_widths(c["n"], c["shards"])]
        x = torch.randn(r, c["k"], device="cuda", generator=g).half()
        s = {"kind": "linear", "x": x, "lins": lins, "n": c["n"], "out32": c["out32"], "fused": None}
        if c["shards"] > 1:
            s["fused"] = exl3.fuse_linears(lins)
            if c["out32"]:
                s["y"] = torch.empty(r, c["n"], dtype=torch.float32, device="cuda")
        return s
    H, I = c["H"], c["I"]
    x = torch.randn(r, H, device="cuda", generator=g).half()
    if c["kind"] == "mlp":
        gt, up, dn = (_packed(1, a, b, c["K"], g)[0] for a, b in ((H, I), (H, I), (I, H)))
        silu = c["act"] == "silu"
        mlp = exl3.BC_GatedMLP(None, None, None, None, None, None, None, c["K"], False, True, silu, not silu, False, gt,
                               up, dn, 0.0)
        return {"kind": "mlp", "x": x, "mlp": mlp, "projs": (gt, up, dn)}
    E, k = c["E"], c["topk"]
    logits = torch.randn(r, E, device="cuda", generator=g)
    if c["kind"] == "blobs":
        gu, dn, size = _blob_layout(H, I, c["K"])
        stride = (size + 4095) // 4096 * 4096
        arena = torch.randint(-32768, 32768, (E, stride // 2), dtype=torch.int16, device="cuda", generator=g)
        at = 2 * (gu + dn)
        for n, scale in ((H, 1.0), (H, 1.0), (I, _isqrt(H)), (I, _isqrt(H)), (I, 1.0), (H, _isqrt(I))):
            arena[:, at:at + n] = _signs((E, n), g, scale).view(torch.int16)
            at += n
        ptrs = torch.arange(E, dtype=torch.int64, device="cuda") * stride + arena.data_ptr()
        w, ids = torch.softmax(logits, 1).topk(k, 1)
        w = (w / w.sum(1, keepdim=True)).float().contiguous()
        return {"kind": "blobs", "x": x.bfloat16() if c["bf16"] else x, "arena": arena, "ptrs": ptrs,
                "ids": ids.to(torch.int32).contiguous(), "w": w, "I": I, "K": c["K"], "E": E}
    n_tab = E + (1 if c["shared"] else 0)
    projs = (_experts(n_tab, H, I, c["Kgu"], g), _experts(n_tab, H, I, c["Kgu"], g), _experts(n_tab, I, H, c["Kd"], g))
    bias = None
    if c["zipf"]:
        bias = -1.1 * torch.log(torch.randperm(E, device="cuda", generator=g).float() + 1)
    gate = (torch.randn(H, E, device="cuda", generator=g) / math.sqrt(H)).half() if c["router"] else None
    layer = exl3.BlockSparseMLP(exl3.ExpertTables(*projs), k, c["shared"], "silu", 0.0, gate, bias)
    return {"kind": "moe", "x": x, "layer": layer, "projs": projs, "gate": gate, "bias": bias, "k": k,
            "params": None if c["router"] else {"router_logits": logits}, "shared": c["shared"], "E": E}


def run(state):
    s = state
    if s["kind"] == "linear":
        if s["fused"] is None:
            return s["lins"][0].run_alloc(s["x"], s["n"], s["out32"])
        tr, suh, svh, sonb, bounds, K = s["fused"]
        return exl3.linear(s["x"], tr, suh, svh, sonb, bounds, K, out=s.get("y"))
    if s["kind"] == "mlp":
        return s["mlp"].forward(s["x"])
    if s["kind"] == "moe":
        return s["layer"].forward(s["x"], s["params"])
    return exl3.moe_forward_blobs(s["x"], s["ids"], s["w"], s["ptrs"], s["I"], s["K"], s["E"])


# ------------------------------------------------------------------------------------------------ 64-bit results
def _codebook():
    """The mul1 codebook: fp16(fma(1024 + byte sum of s * 0x83DCD12D mod 2^32, 0x1EEE, 0xC931)) for every state s."""
    s = torch.arange(65536, dtype=torch.int64, device="cuda")
    p = (s * 0x83DCD12D) & 0xFFFFFFFF
    h = 1024 + (p & 255) + ((p >> 8) & 255) + ((p >> 16) & 255) + (p >> 24)
    return (h.double() * 0.00676727294921875 - 10.3828125).half().double()


def _tiles(words, K, book):
    """Weights [T, 16, 16] of tiles [T, 8K] of ring words (int64): position t takes the 16 ring bits before bit
    (t + 1) K and lies at row 8 ((t >> 1) & 1) + 2 ((t >> 3) & 3) + (t & 1), column (t >> 5) + 8 ((t >> 2) & 1)."""
    t = torch.arange(256, device="cuda")
    bit = ((t + 1) * K - 16) % (256 * K)
    i, off = bit >> 5, bit & 31
    pair = (words[:, i] << 32) | words[:, (i + 1) % (8 * K)]
    v = book[(pair >> (48 - off)) & 0xFFFF]
    out = torch.empty(words.shape[0], 16, 16, dtype=torch.float64, device="cuda")
    out[:, 8 * ((t >> 1) & 1) + 2 * ((t >> 3) & 3) + (t & 1), (t >> 5) + 8 * ((t >> 2) & 1)] = v
    return out


def _words(int16, K):
    return int16.contiguous().view(torch.int32).reshape(-1, 8 * K).to(torch.int64) & 0xFFFFFFFF


def _matrix(p, book):
    """Hadamard-domain weights [k, n] of a projection, in strips of tile-rows to bound memory."""
    if isinstance(p, exl3.MixedEXL3):
        k, n = p.suh.numel(), p.svh.numel()
        w = p.words.view(torch.int32).to(torch.int64) & 0xFFFFFFFF
        t = torch.empty(p.kmap.numel(), 16, 16, dtype=torch.float64, device="cuda")
        for K in range(1, 9):
            sel = (p.kmap == K).nonzero()[:, 0]
            if sel.numel():
                at = p.woff[sel].to(torch.int64)[:, None] + torch.arange(8 * K, device="cuda")
                t[sel] = _tiles(w[at], K, book)
    else:
        tk, tn, K = p.trellis.shape[0], p.trellis.shape[1], p.trellis.shape[2] // 16
        k, n = 16 * tk, 16 * tn
        out = torch.empty(k, n, dtype=torch.float64, device="cuda")
        for a in range(0, tk, 32):
            b = min(tk, a + 32)
            s = _tiles(_words(p.trellis[a:b], K), K, book).view(b - a, tn, 16, 16)
            out[16 * a:16 * b] = s.permute(0, 2, 1, 3).reshape(16 * (b - a), n)
        return out
    return t.view(k // 16, n // 16, 16, 16).permute(0, 2, 1, 3).reshape(k, n)


def _had(x):
    """Blockwise 128-point Hadamard transform / sqrt(128)."""
    H = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    for _ in range(7):
        H = torch.cat([torch.cat([H, H], 1), torch.cat([H, -H], 1)], 0)
    return (x.reshape(-1, 128) @ (H / math.sqrt(128))).reshape(x.shape)


def _proj(x, p, book):
    return _had(_had(x * p.suh.double()) @ _matrix(p, book)) * p.svh.double()


def _gated(x, gate, up, down, silu, book):
    a, b = _proj(x, gate, book), _proj(x, up, book)
    if silu:
        h = a * torch.sigmoid(a) * b
    else:
        h = 0.5 * a * (1 + torch.tanh(math.sqrt(2 / math.pi) * (a + 0.044715 * a ** 3))) * b
    return _proj(h, down, book)


class _Blob:
    """One projection of an expert blob, its words in PLANAR4 order: within each group of 4 tiles of a tile-row, word
    (tile t, period g, plane i) lies at 4 G i + G t + g, with D = K / gcd(K, 32) planes and G = 8K / D periods."""

    def __init__(self, words, K, suh, svh):
        tk, tn = words.shape[0], words.shape[1] // (8 * K)
        D = K // math.gcd(K, 32)
        G = 8 * K // D
        idx = [[4 * G * i + G * t + q for q in range(G) for i in range(D)] for t in range(4)]
        idx = torch.tensor(idx, device="cuda").reshape(-1)
        w = words.reshape(tk, tn // 4, 32 * K)[:, :, idx].reshape(tk, tn, 8 * K)
        self.trellis = w.contiguous().view(torch.int16).reshape(tk, tn, 16 * K)
        self.suh, self.svh = suh, svh


def _blob_expert(rec, H, I, K):
    gu, dn, _ = _blob_layout(H, I, K)
    words = rec[:2 * (gu + dn)].view(torch.int32)
    wgu = words[:gu].reshape(H // 16, -1)
    at, v = 2 * (gu + dn), []
    for n in (H, H, I, I, I, H):
        v.append(rec[at:at + n].view(torch.float16))
        at += n
    half = (I // 16) * 8 * K
    return (_Blob(wgu[:, :half], K, v[0], v[2]), _Blob(wgu[:, half:], K, v[1], v[3]),
            _Blob(words[gu:gu + dn].reshape(I // 16, -1), K, v[4], v[5]))


def exact(case, seed):
    c, s, book = case, prepare(case, seed), _codebook()
    x = s["x"].double()
    if c["kind"] == "linear":
        return torch.cat([_proj(x, p, book) for p in s["lins"]], 1)
    if c["kind"] == "mlp":
        return _gated(x, *s["projs"], c["act"] == "silu", book)
    if c["kind"] == "blobs":
        ids, w = s["ids"].long(), s["w"].double()
        experts = lambda e: _blob_expert(s["arena"][e], c["H"], c["I"], c["K"])  # noqa: E731
    else:
        lg = x @ s["gate"].double() if s["gate"] is not None else s["params"]["router_logits"].double()
        p, ids = torch.softmax(lg if s["bias"] is None else lg + s["bias"].double(), 1).topk(s["k"], 1)
        w = p / p.sum(1, keepdim=True)
        experts = lambda e: tuple(q[e] for q in s["projs"])  # noqa: E731
    out = torch.zeros_like(x)
    for e in range(c["E"]):
        row, slot = (ids == e).nonzero(as_tuple=True)
        if row.numel():
            out.index_add_(0, row, _gated(x[row], *experts(e), True, book) * w[row, slot][:, None])
    if c.get("shared"):
        out += _gated(x, *experts(c["E"]), True, book)
    return out
