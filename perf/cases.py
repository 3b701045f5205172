"""The workloads this framework's speed is measured on: the calls a program
that serves a DeepSeek-R1 shaped model makes, through the package's public
entry points, from one matrix-vector product to a 512-token prefill.

A case is a dict of plain values with a "kind":

  matvec   n products y = W x of Q4_K or Q6_K rows (out x in), one after the
           other, as a host program walks the matrices of a layer
  expert   n SwiGLU experts of one token, one call each
  decode   one token through n4 Q4_K-down and n6 Q6_K-down MoE layers, the
           rms_norm fused in, the hidden state updated in place
  dense    one token through `layers` dense layers: rms_norm, then the FFN
  batch    T tokens of a serving step through one MoE layer
  prefill  T prompt tokens through `layers` MoE layers, in place
  attn     a sequence of S tokens through one attention layer, token by
           token, the cache growing from empty

Weights are synthetic: random quants and scales whose block scales give the
weights of one matrix a standard deviation of about 0.02 around zero, the
router N(0, 0.01) with a bias N(0, 0.1), attention matrices N(0, 1 / fan in),
activations N(0, 1).
"""
import functools
import math
import weakref

import torch

import flash_deepseek_amd as fd

HIDDEN, FFN, EXPERTS, GROUPS, TOP_GROUPS, ROUTED_SCALE = 7168, 2048, 256, 8, 4, 2.5
GATE = 57344 * 144  # bytes of a 2048 x 7168 Q4_K matrix
BLOCK = {"q4": 144, "q6": 210}
NH, QA, KVL, NOPE, ROPE, VH = 128, 1536, 512, 128, 64, 128


def listed():
    return [
        # the smallest call: a host program's gate / up products, bound by latency and launches
        {"name": "matvec_q4k", "kind": "matvec", "fmt": "q4", "out": 2048, "in": 7168, "n": 4},
        # a token's routed experts one by one, as a host that routes for itself runs them (Q6_K down)
        {"name": "expert_q6k", "kind": "expert", "q6": True, "n": 8},
        # batch-1 decode through a model file that mixes Q4_K and Q6_K down matrices
        {"name": "decode_mixed", "kind": "decode", "n4": 2, "n6": 2, "K": 8},
        # batch-1 decode through the model's three dense layers
        {"name": "dense_r1", "kind": "dense", "layers": 3, "inter": 18432},
        # serving steps: a few sequences, a small and an ordinary batch, a large one
        {"name": "batch_t5", "kind": "batch", "q6": False, "T": 5, "K": 8},
        {"name": "batch_t16", "kind": "batch", "q6": False, "T": 16, "K": 8},
        {"name": "batch_t64_q6k", "kind": "batch", "q6": True, "T": 64, "K": 8},
        {"name": "batch_t256", "kind": "batch", "q6": False, "T": 256, "K": 8},
        # prompts: the largest call, and a ragged one through a layer with Q6_K down matrices
        {"name": "prefill_t512", "kind": "prefill", "q6": False, "T": 512, "K": 8, "layers": 1},
        {"name": "prefill_t150_q6k", "kind": "prefill", "q6": True, "T": 150, "K": 8, "layers": 1},
        # attention of a short exchange and of a long document
        {"name": "attn_s48", "kind": "attn", "S": 48},
        {"name": "attn_s2048", "kind": "attn", "S": 2048},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    plain = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        case = _draw(rng)
        if case not in plain:
            return case


def _draw(rng):
    kind = rng.choice(["matvec", "expert", "decode", "dense", "batch", "batch", "batch", "prefill", "prefill", "attn"])
    K = rng.choice([2, 4, 5, 6, 7, 8, 8, 8, 10, 12, 16])
    if kind == "matvec":
        return {"kind": kind, "fmt": rng.choice(["q4", "q6"]), "out": _log(rng, 256, 18432), "in": 256 * _log(rng, 2, 28),
                "n": rng.randint(2, 6)}
    if kind == "expert":
        return {"kind": kind, "q6": rng.random() < 0.5, "n": rng.randint(2, 32)}
    if kind == "decode":
        n4 = rng.randint(0, 3)
        return {"kind": kind, "n4": n4, "n6": rng.randint(0 if n4 else 1, 4 - n4), "K": K}
    if kind == "dense":
        return {"kind": kind, "layers": rng.randint(1, 3), "inter": 512 * _log(rng, 4, 36)}
    if kind == "batch":
        return {"kind": kind, "q6": rng.random() < 0.5, "T": _log(rng, 2, 512), "K": K}
    if kind == "prefill":
        return {"kind": kind, "q6": rng.random() < 0.5, "T": _log(rng, 16, 512), "K": K, "layers": 1}
    return {"kind": "attn", "S": _log(rng, 4, 2048)}


# ---- seeded inputs -------------------------------------------------------------------
def _gen(seed, *salt):
    g = torch.Generator(device="cuda")
    h = seed & 0x7FFFFFFF
    for s in salt:
        h = (h * 1000003 + s + 1) & 0x7FFFFFFFFFFFFFF
    return g.manual_seed(h)


def _normal(g, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).add_(mean)


def _norm_w(g, n):
    return _normal(g, n, std=0.1, mean=1.0)


def _halves(g, shape, unit):
    """fp16 block scales between 0.5 and 1.5 units."""
    return (torch.rand(shape, generator=g, device="cuda") + 0.5).mul_(unit).half()


def _fill_q4(blocks, g):
    """Block scales of uint8 Q4_K blocks [..., 144] whose other bytes are random."""
    d = _halves(g, blocks.shape[:-1], 8e-5)
    blocks[..., 0:4] = torch.stack([d, (d.float() * 7.5).half()], -1).view(torch.uint8)


def _fill_q6(blocks, g):
    blocks[..., 208:210] = _halves(g, blocks.shape[:-1], 1.5e-5).unsqueeze(-1).view(torch.uint8)


def _matrix(g, fmt, rows, cols):
    """Packed rows of one matrix: uint8 [rows, cols / 256, block bytes]."""
    b = torch.empty(rows, cols // 256, BLOCK[fmt], dtype=torch.uint8, device="cuda").random_(0, 256, generator=g)
    (_fill_q4 if fmt == "q4" else _fill_q6)(b, g)
    return b


def _blobs(g, n, q6):
    """n packed experts [gate | up | down]: uint8 [n, expert bytes]."""
    size = fd.EXPERT_Q6K_BYTES if q6 else fd.EXPERT_Q4K_BYTES
    e = torch.empty(n, size, dtype=torch.uint8, device="cuda")
    e.view(-1).random_(0, 256, generator=g)
    _fill_q4(e[:, :2 * GATE].view(n, -1, 144), g)
    down = e[:, 2 * GATE:]
    (_fill_q6(down.view(n, -1, 210), g) if q6 else _fill_q4(down.view(n, -1, 144), g))
    return e


def _moe_weights(seed, layer, q6):
    """(experts [257, bytes], the last one the shared expert; router; bias; norm weights)"""
    g = _gen(seed, 11, layer)
    Wg, bias, nw = _normal(g, EXPERTS, HIDDEN, std=0.01), _normal(g, EXPERTS, std=0.1), _norm_w(g, HIDDEN)
    return _blobs(g, EXPERTS + 1, q6), Wg, bias, nw


def _attn_weights(seed):
    g = _gen(seed, 12)

    def mat(fan_in, *shape):
        return _normal(g, *shape, std=fan_in ** -0.5).half()

    return {"attn_norm": _norm_w(g, HIDDEN), "q_a": mat(HIDDEN, QA, HIDDEN), "q_a_norm": _norm_w(g, QA),
            "q_b": mat(QA, NH * (NOPE + ROPE), QA), "kv_a": mat(HIDDEN, KVL + ROPE, HIDDEN),
            "kv_a_norm": _norm_w(g, KVL), "k_b": mat(NOPE, NH, KVL, NOPE), "v_b": mat(KVL, NH, VH, KVL),
            "o_proj": mat(NH * VH, HIDDEN, NH * VH)}


def _dense_weights(seed, layer, inter):
    g = _gen(seed, 13, layer)
    return ([_normal(g, *s, std=s[1] ** -0.5).half() for s in ((inter, HIDDEN), (inter, HIDDEN), (HIDDEN, inter))],
            _norm_w(g, HIDDEN))


def _tokens(seed, n):
    return _normal(_gen(seed, 14), n, HIDDEN)


def _residual(seed, n):
    return _normal(_gen(seed, 15), n, HIDDEN)


def _is_q6(case, layer):
    return layer >= case["n4"] if case["kind"] == "decode" else case["q6"]


def _n_layers(case):
    return {"decode": lambda: case["n4"] + case["n6"], "batch": lambda: 1}.get(case["kind"], lambda: case["layers"])()


# ---- states --------------------------------------------------------------------------
_free_ids = list(range(fd.MAX_LAYERS))


class _State:
    """Layer ids held by a program, given back with it."""

    def __init__(self, n_layers, release):
        self.layers = [_free_ids.pop() for _ in range(n_layers)]
        weakref.finalize(self, _State._give_back, self.layers, release).atexit = False

    @staticmethod
    def _give_back(layers, release):
        for L in layers:
            release(L)
            _free_ids.append(L)


def prepare(case, seed):
    fd.init(torch.cuda.current_device())
    kind = case["kind"]
    if kind in ("decode", "batch", "prefill"):
        s = _State(_n_layers(case), fd.release_layer)
        s.keep, s.norm = [], []
        for i, L in enumerate(s.layers):
            blobs, Wg, bias, nw = _moe_weights(seed, i, _is_q6(case, i))
            fd.attach_layer(L, blobs[:EXPERTS], blobs.shape[1], Wg, bias, shared=blobs[EXPERTS:])
            s.keep.append((Wg, bias))
            s.norm.append(nw)
        T, K = case.get("T", 1), case["K"]
        s.x = _tokens(seed, T)
        s.out = torch.empty_like(s.x)
        s.idx = torch.empty(len(s.layers), T, K, dtype=torch.int32, device="cuda")
        s.w = torch.empty(len(s.layers), T, K, device="cuda")
        s.h_in = _residual(seed, T) if kind == "batch" else None
    elif kind == "matvec":
        s = _State(0, None)
        g = _gen(seed, 16)
        s.W = [_matrix(g, case["fmt"], case["out"], case["in"]) for _ in range(case["n"])]
        s.x = _normal(g, case["in"])
        s.y = torch.empty(case["n"], case["out"], device="cuda")
    elif kind == "expert":
        s = _State(0, None)
        s.blobs = _blobs(_gen(seed, 17), case["n"], case["q6"])
        s.x = _tokens(seed, 1)[0]
        s.y = torch.empty(case["n"], HIDDEN, device="cuda")
    elif kind == "dense":
        s = _State(case["layers"], fd.release_dense)
        s.norm = []
        for i, L in enumerate(s.layers):
            (gate, up, down), nw = _dense_weights(seed, i, case["inter"])
            fd.attach_dense(L, gate, up, down, case["inter"])
            s.norm.append(nw)
        s.x = _tokens(seed, 1)
        s.out, s.h_post = torch.empty_like(s.x), torch.empty_like(s.x)
    else:
        s = _State(1, fd.attn_release)
        fd.attn_upload(s.layers[0], {k: v.cpu().numpy() for k, v in _attn_weights(seed).items()}, max_seq=case["S"])
        s.x = _tokens(seed, case["S"])
        s.out = torch.empty_like(s.x)
    s.case = case
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "matvec":
        f = fd.matvec_q4k if s.case["fmt"] == "q4" else fd.matvec_q6k
        for W, y in zip(s.W, s.y):
            f(W, s.x, y, s.case["out"], s.case["in"])
        return s.y
    if kind == "expert":
        for blob, y in zip(s.blobs, s.y):
            fd.expert_ffn(blob, s.blobs.shape[1], s.x, y)
        return s.y
    if kind == "decode":
        h = s.x
        for i, L in enumerate(s.layers):
            fd.moe_layer_norm(L, h, s.norm[i], s.case["K"], s.out, idx=s.idx[i], w=s.w[i])
            h = s.out
        return {"hidden": s.out, "idx": s.idx, "w": s.w}
    if kind == "batch":
        fd.moe_forward_batched(s.layers[0], s.x, s.h_in, s.case["T"], s.case["K"], s.out, idx=s.idx[0], w=s.w[0])
        return {"hidden": s.out, "idx": s.idx, "w": s.w}
    if kind == "prefill":
        s.out.copy_(s.x)  # the prompt's embeddings
        fd.moe_prefill(s.layers, s.out, s.case["T"], s.case["K"], s.norm, idx=s.idx)
        return {"hidden": s.out, "idx": s.idx}
    if kind == "dense":
        h = s.x
        for L, nw in zip(s.layers, s.norm):
            fd.rms_norm(h, nw, s.h_post, 1)
            fd.dense_ffn(L, s.h_post, h, s.out)
            h = s.out
        return s.out
    L = s.layers[0]
    fd.attn_reset(L)
    s.out.copy_(s.x)
    for t, h in enumerate(s.out):
        fd.attn_forward(L, h, t)
    return s.out


# ---- what a pass cannot do without -----------------------------------------------------
@functools.lru_cache(None)
def _distinct(T, K):
    """Distinct routed experts of T tokens whose logits have the workload's distribution."""
    g = torch.Generator().manual_seed(T * 100 + K)
    score = torch.sigmoid(torch.randn(T, EXPERTS, generator=g) * 0.01 * math.sqrt(HIDDEN))
    return int(torch.unique(_route(score, torch.randn(EXPERTS, generator=g) * 0.1, K)).numel())


def work(case):
    kind, vec = case["kind"], 4 * HIDDEN
    if kind == "matvec":
        w = case["out"] * case["in"]
        n = case["n"]
        return {"bytes": n * (w // 256 * BLOCK[case["fmt"]] + 4 * case["out"]) + 4 * case["in"], "flops": 2 * w * n}
    if kind == "expert":
        size = fd.EXPERT_Q6K_BYTES if case["q6"] else fd.EXPERT_Q4K_BYTES
        return {"bytes": case["n"] * (size + vec) + vec, "flops": case["n"] * 6 * HIDDEN * FFN}
    if kind == "dense":
        w = 3 * case["inter"] * HIDDEN * case["layers"]
        return {"bytes": 2 * w + (case["layers"] + 2) * vec, "flops": 2 * w}
    if kind == "attn":
        # every token of a sequence is a call of its own: the layer's weights and the cache so far, once per token
        S = case["S"]
        w = HIDDEN * (QA + KVL + ROPE) + QA * NH * (NOPE + ROPE) + NH * KVL * (NOPE + VH) + HIDDEN * NH * VH
        pairs = S * (S + 1) // 2
        return {"bytes": S * (2 * w + 2 * vec) + pairs * 4 * (KVL + ROPE),
                "flops": 2 * w * S + pairs * NH * 2 * (2 * KVL + ROPE)}
    T, K, b = case.get("T", 1), case["K"], 0
    for i in range(_n_layers(case)):
        size = fd.EXPERT_Q6K_BYTES if _is_q6(case, i) else fd.EXPERT_Q4K_BYTES
        b += (_distinct(T, K) + 1) * size + 4 * EXPERTS * (HIDDEN + 1)
    b += T * vec * (3 if kind == "batch" else 2)
    return {"bytes": b, "flops": _n_layers(case) * T * ((K + 1) * 6 * HIDDEN * FFN + 2 * EXPERTS * HIDDEN)}


def tolerance(case):
    """Four times what the paths differ by from the same in 64 bits, or a little more."""
    if case["kind"] == "prefill":  # one fp16 plane of the activations: 2.9e-4 .. 3.4e-4, largest 1.9e-3
        return {"rel": 1.5e-3, "max": 8e-3}
    if case["kind"] in ("decode", "dense"):  # layers in a chain, each carrying on the rounding of those before: 2.4e-6, 9.7e-6
        return {"rel": 1e-5, "max": 4e-5}
    return {"rel": 3e-6, "max": 2e-5}  # fp32 grade: 1.6e-7 .. 6.4e-7, largest 4.2e-6


# ---- the same in 64 bits ---------------------------------------------------------------
def _deq_q4(b):
    """Q4_K blocks uint8 [rows, n, 144] -> float64 [rows, 256 n]."""
    d, dmin = b[..., 0:4].contiguous().view(torch.float16).double().unbind(-1)
    s = b[..., 4:16].int()
    lo, hi = s[..., 0:4], s[..., 4:8]
    sc = torch.cat([lo & 63, (s[..., 8:12] & 15) | (lo >> 6 << 4)], -1)
    m = torch.cat([hi & 63, (s[..., 8:12] >> 4) | (hi >> 6 << 4)], -1)
    qs = b[..., 16:].reshape(*b.shape[:-1], 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], -2).reshape(*b.shape[:-1], 8, 32).double()
    w = q * (d.unsqueeze(-1) * sc).unsqueeze(-1) - (dmin.unsqueeze(-1) * m).unsqueeze(-1)
    return w.reshape(b.shape[0], -1)


def _deq_q6(b):
    d = b[..., 208:210].contiguous().view(torch.float16).double()
    ql, qh = b[..., :128].reshape(*b.shape[:-1], 2, 2, 32), b[..., 128:192].reshape(*b.shape[:-1], 2, 1, 32)
    q = torch.cat([ql & 15, ql >> 4], -2) | torch.cat([(qh >> 2 * k & 3) << 4 for k in range(4)], -2)
    sc = b[..., 192:208].contiguous().view(torch.int8).double() * d
    return ((q.double() - 32).reshape(*b.shape[:-1], 16, 16) * sc.unsqueeze(-1)).reshape(b.shape[0], -1)


def _ffn(blob, q6, x):
    """One expert on float64 rows x."""
    gate, up = (_deq_q4(m.view(FFN, -1, 144)) for m in (blob[:GATE], blob[GATE:2 * GATE]))
    down = blob[2 * GATE:]
    down = _deq_q6(down.view(HIDDEN, -1, 210)) if q6 else _deq_q4(down.view(HIDDEN, -1, 144))
    g = x @ gate.T
    return (g * torch.sigmoid(g) * (x @ up.T)) @ down.T


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w.double()


def _route(score, bias, K):
    """The K experts of each row of scores: the best of the four groups whose two best experts are best."""
    c = score + bias
    per = EXPERTS // GROUPS
    top = c.view(-1, GROUPS, per).topk(2, -1).values.sum(-1).topk(TOP_GROUPS, -1).indices
    keep = torch.zeros(c.shape[0], GROUPS, dtype=torch.bool, device=c.device).scatter_(1, top, True)
    return c.masked_fill(~keep.repeat_interleave(per, 1), -math.inf).topk(K, -1).indices


def _moe(weights, q6, x, K):
    blobs, Wg, bias, _ = weights
    score = torch.sigmoid(x @ Wg.double().T)
    idx = _route(score, bias.double(), K)
    w = score.gather(1, idx)
    w = w * (ROUTED_SCALE / w.sum(-1, keepdim=True))
    y = _ffn(blobs[EXPERTS], q6, x)
    for e in torch.unique(idx).tolist():
        t, k = (idx == e).nonzero(as_tuple=True)
        y.index_add_(0, t, _ffn(blobs[e], q6, x[t]) * w[t, k].unsqueeze(-1))
    return y


def _yarn():
    """Rotation frequencies of the 32 pairs, in float32 as the model defines them."""
    f32 = lambda v: torch.tensor(v, dtype=torch.float32)  # noqa: E731
    edge = [64 * math.log(4096 / (r * 2 * math.pi)) / (2 * math.log(10000)) for r in (32, 1)]
    lo, hi = math.floor(edge[0]), math.ceil(edge[1])
    i = torch.arange(32, dtype=torch.float32)
    extra = 1.0 / torch.pow(f32(10000.0), 2 * i / 64)
    mask = 1.0 - ((i - lo) / (hi - lo)).clamp(0, 1)
    return extra / 40.0 * (1.0 - mask) + extra * mask


def _rotate(x, cos, sin):
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)


def _attention(case, seed):
    w = {k: v.double() for k, v in _attn_weights(seed).items()}
    S = case["S"]
    h = _tokens(seed, S).double()
    x = _rms(h, w["attn_norm"])
    q = (_rms(x @ w["q_a"].T, w["q_a_norm"]) @ w["q_b"].T).view(S, NH, NOPE + ROPE)
    kv = x @ w["kv_a"].T
    c = _rms(kv[:, :KVL], w["kv_a_norm"])
    ang = (torch.arange(S, dtype=torch.float32)[:, None] * _yarn()[None]).double().cuda()  # the angle is a float
    cos, sin = ang.cos(), ang.sin()
    k_rope = _rotate(kv[:, KVL:], cos, sin)
    q_rope = _rotate(q[..., NOPE:], cos[:, None], sin[:, None])
    scale = (0.1 * math.log(40) + 1) ** 2 / math.sqrt(NOPE + ROPE)
    past = torch.ones(S, S, dtype=torch.bool, device="cuda").tril()
    out = torch.empty(S, NH, VH, dtype=torch.float64, device="cuda")
    for i in range(NH):
        s = (q[:, i, :NOPE] @ (c @ w["k_b"][i]).T + q_rope[:, i] @ k_rope.T) * scale
        out[:, i] = torch.softmax(s.masked_fill(~past, -math.inf), -1) @ (c @ w["v_b"][i].T)
    return h + out.flatten(1) @ w["o_proj"].T


def exact(case, seed):
    kind = case["kind"]
    if kind == "matvec":
        g = _gen(seed, 16)
        W = [_matrix(g, case["fmt"], case["out"], case["in"]) for _ in range(case["n"])]
        x = _normal(g, case["in"]).double()
        return torch.stack([(_deq_q4(m) if case["fmt"] == "q4" else _deq_q6(m)) @ x for m in W])
    if kind == "expert":
        x = _tokens(seed, 1).double()
        return torch.cat([_ffn(b, case["q6"], x) for b in _blobs(_gen(seed, 17), case["n"], case["q6"])])
    if kind == "attn":
        return _attention(case, seed)
    if kind == "dense":
        h = _tokens(seed, 1).double()
        for i in range(case["layers"]):
            (gate, up, down), nw = _dense_weights(seed, i, case["inter"])
            x = _rms(h, nw)
            a = x @ gate.double().T
            h = h + (a * torch.sigmoid(a) * (x @ up.double().T)) @ down.double().T
        return h
    x = _tokens(seed, case.get("T", 1)).double()
    if kind == "batch":
        y = _residual(seed, case["T"]).double() + _moe(_moe_weights(seed, 0, case["q6"]), case["q6"], x, case["K"])
        return {"hidden": y, "idx": None, "w": None}
    for i in range(_n_layers(case)):
        weights = _moe_weights(seed, i, _is_q6(case, i))
        x = x + _moe(weights, _is_q6(case, i), _rms(x, weights[3]), case["K"])
    return {"hidden": x, "idx": None, "w": None} if kind == "decode" else {"hidden": x, "idx": None}
