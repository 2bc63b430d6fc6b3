"""The measured workloads of the library: what a host program built on it has
it do, each through a public entry point of `biv_amd.hip`.

Two layer kinds, the two feed-forward layers of the models it serves:

  moe    the qwen35moe mixture-of-experts block (256 experts of which 8 are
         used, width 2048, expert width 512, a shared expert), from one token
         of a chat to a 4096-token prefill chunk;
  dense  the qwen35 dense SwiGLU FFN, from one token to a 512-token chunk.

Weights are ~N(0, 0.02) quantised to the ggml types, hidden states ~N(0, 1);
both come from the seed alone and are made on the GPU.
"""
import ctypes
import math

import numpy as np
import torch

from biv_amd import hip, synth

Q8_0, Q4K, Q6K, BF16 = synth.Q8_0, synth.Q4K, synth.Q6K, synth.BF16
# (gate and up, down) matrix types by name
TYPES = {"q8": (Q8_0, Q8_0), "kq": (Q4K, Q6K), "bf16": (BF16, BF16)}
BPW = {Q8_0: 34 / 32, Q4K: 144 / 256, Q6K: 210 / 256, BF16: 2.0}  # bytes per weight
EPS = 1e-6


def _moe(name, types, tokens, layers=1, entry="device", skew=0.0, n_embd=2048, n_expert=256, k=8, n_ff=512,
         shared=True):
    c = dict(kind="moe", types=types, tokens=tokens, layers=layers, entry=entry, skew=skew, n_embd=n_embd,
             n_expert=n_expert, k=k, n_ff=n_ff, shared=shared)
    return dict(name=name, **c) if name else c


def _dense(name, types, tokens, n_embd=4096, n_ff=12288, add=False):
    c = dict(kind="dense", types=types, tokens=tokens, n_embd=n_embd, n_ff=n_ff, add=add)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one chat, one token at a time: the FFN halves of 8 consecutive layers
        _moe("decode_q8_1", "q8", 1, layers=8, entry="step"),
        # the same chat with 4 drafted tokens verified at once
        _moe("verify_q8_5", "q8", 5, layers=4, entry="step"),
        # Model::ffn on host arrays, as a CPU engine that offloads the block
        # calls it, for a small batch
        _moe("host_q8_9", "q8", 9, entry="host"),
        # 8 chats batched continuously, 5 tokens each
        _moe("batch_q8_40", "q8", 40, layers=2),
        # a prefill chunk whose expert loads are skewed, as real text's are
        _moe("prefill_q8_512", "q8", 512, skew=1.1),
        # the 4-bit quantisation of the same model: one chat, and a long prompt
        _moe("decode_kq_1", "kq", 1, layers=8),
        _moe("prefill_kq_2048", "kq", 2048),
        # the unquantised model's prefill: norm, block and residual of a layer
        _moe("prefill_bf16_4096", "bf16", 4096, entry="step"),
        # a 9B dense model: decoding, draft verification, a prefill chunk
        _dense("dense_q8_1", "q8", 1),
        _dense("dense_q8_5", "q8", 5),
        _dense("dense_q8_512", "q8", 512),
        # a ragged last prefill chunk of the 4-bit dense model
        _dense("dense_kq_130", "kq", 130),
    ]


def draw(rng):
    def logint(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))

    types = rng.choice(["q8", "q8", "kq", "bf16"])
    if rng.random() < 0.4:
        n_embd, n_ff = 512 * rng.randint(2, 8), 512 * rng.randint(3, 24)
        return _dense(None, types, logint(1, 512), n_embd, n_ff, add=rng.random() < 0.5)
    if rng.random() < 0.6:
        n_embd, n_expert, k, n_ff, shared = 2048, 256, 8, 512, True
    else:
        n_embd, n_ff = rng.choice([512, 1024, 2048]), rng.choice([512, 1024])
        n_expert, k, shared = rng.randint(16, 128), rng.randint(2, 8), rng.random() < 0.7
    if rng.random() < 0.5:  # decode sizes
        return _moe(None, types, logint(1, 48), rng.choice([1, 2]), rng.choice(["device", "step", "step", "host"]),
                    0.0, n_embd, n_expert, k, n_ff, shared)
    tokens = logint(49, 4096 if types == "bf16" and n_expert == 256 else 2048)
    return _moe(None, types, tokens, 1, rng.choice(["device", "device", "step"]), rng.choice([0.0, 1.1]), n_embd,
                n_expert, k, n_ff, shared)


# ---------------------------------------------------------------------------
# Seeded weights.  Each matrix has a generator of its own, so a matrix is the
# same whether the others are made or not.


def _gen(seed, tag):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1009 + tag) % (1 << 62))
    return g


def _normal(g, shape, std):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std


def _blocks(ty, w):
    """Rows of float32 weights [rows, cols] as ggml blocks, [rows, bytes] uint8."""
    rows, cols = w.shape
    if ty == BF16:
        return w.to(torch.bfloat16).view(torch.uint8).reshape(rows, -1)
    if ty == Q8_0:
        x = w.reshape(rows, cols // 32, 32)
        d = x.abs().amax(-1) / 127
        q = torch.round(x / torch.where(d > 0, d, torch.ones_like(d))[..., None]).clamp_(-127, 127).to(torch.int8)
        return torch.cat([d.half()[..., None].view(torch.uint8), q.view(torch.uint8)], -1).reshape(rows, -1)
    if ty == Q4K:
        x = w.reshape(rows, cols // 256, 8, 32)
        lo = -x.amin(-1).clamp(max=0)
        sc = (x.amax(-1) + lo) / 15
        d, dm = (sc.amax(-1) / 63).half(), (lo.amax(-1) / 63).half()
        s6 = torch.round(sc / d.float().clamp(min=1e-8)[..., None]).clamp_(0, 63)
        m6 = torch.round(lo / dm.float().clamp(min=1e-8)[..., None]).clamp_(0, 63)
        eff = (d.float()[..., None] * s6).clamp(min=1e-8)[..., None]
        q = torch.round((x + (dm.float()[..., None] * m6)[..., None]) / eff).clamp_(0, 15).to(torch.uint8)
        s, m = s6.to(torch.uint8), m6.to(torch.uint8)
        sc_bytes = torch.cat([s[..., :4] | ((s[..., 4:] >> 4) << 6), m[..., :4] | ((m[..., 4:] >> 4) << 6),
                              (s[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)], -1)
        nib = q[..., 0::2, :] | (q[..., 1::2, :] << 4)
        return torch.cat([d[..., None].view(torch.uint8), dm[..., None].view(torch.uint8), sc_bytes, nib.flatten(-2)],
                         -1).reshape(rows, -1)
    x = w.reshape(rows, cols // 256, 16, 16)  # Q6_K
    sc = x.abs().amax(-1) / 31
    d = (sc.amax(-1) / 127).half()
    s8 = torch.round(sc / d.float().clamp(min=1e-8)[..., None]).clamp_(-128, 127)
    eff = (d.float()[..., None] * s8).clamp(min=1e-8)[..., None]
    q = (torch.round(x / eff).clamp_(-32, 31) + 32).to(torch.uint8).reshape(rows, cols // 256, 2, 4, 32)
    a, b, c, e = (q[..., i, :] for i in range(4))
    ql = torch.cat([(a & 15) | ((c & 15) << 4), (b & 15) | ((e & 15) << 4)], -1).flatten(-2)
    qh = ((a >> 4) | ((b >> 4) << 2) | ((c >> 4) << 4) | ((e >> 4) << 6)).flatten(-2)
    return torch.cat([ql, qh, s8.to(torch.int8).view(torch.uint8), d[..., None].view(torch.uint8)], -1).reshape(rows, -1)


def _values(ty, blk, cols):
    """The float64 weights that ggml blocks [rows, bytes] hold, [rows, cols]."""
    rows = blk.shape[0]

    def f16(b):
        return b.contiguous().view(torch.float16).double()

    if ty == BF16:
        return blk.contiguous().view(torch.bfloat16).double()
    if ty == Q8_0:
        b = blk.reshape(rows, cols // 32, 34)
        return (f16(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8).double()).reshape(rows, cols)
    if ty == Q4K:
        b = blk.reshape(rows, cols // 256, 144)
        d, dm, s = f16(b[..., 0:2]), f16(b[..., 2:4]), b[..., 4:16]
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1).double()
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
        nib = b[..., 16:].reshape(rows, cols // 256, 4, 1, 32)
        q = torch.cat([nib & 15, nib >> 4], -2).reshape(rows, cols // 256, 8, 32).double()
        return ((d * sc)[..., None] * q - (dm * mn)[..., None]).reshape(rows, cols)
    b = blk.reshape(rows, cols // 256, 210)
    ql, qh = b[..., :128].reshape(rows, -1, 2, 2, 32), b[..., 128:192].reshape(rows, -1, 2, 1, 32)
    low = torch.cat([ql & 15, ql >> 4], -2)
    high = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], -2)
    q = (low | (high << 4)).to(torch.int16).sub_(32).double().reshape(rows, cols // 256, 16, 16)
    sc = b[..., 192:208].contiguous().view(torch.int8).double()
    return (f16(b[..., 208:210])[..., None] * sc[..., None] * q).reshape(rows, cols)


def _matrix(seed, tag, ty, rows, cols):
    """A matrix's ggml blocks on the GPU, made 2^26 weights at a time."""
    g = _gen(seed, tag)
    step = max(1, (1 << 26) // cols)
    parts = [_blocks(ty, _normal(g, (min(step, rows - r), cols), 0.02)) for r in range(0, rows, step)]
    return parts[0] if len(parts) == 1 else torch.cat(parts)


def _host(t):
    return t.reshape(-1).cpu().numpy()


def _routers(case, seed):
    return [_normal(_gen(seed, 100 + i), (case["n_expert"], case["n_embd"]), 0.02) for i in range(case["layers"])]


def _norms(case, seed):
    return [1 + _normal(_gen(seed, 200 + i), (case["n_embd"],), 0.02) for i in range(case["layers"])]


def _gate_inp(case, seed):
    return _normal(_gen(seed, 10), (1, case["n_embd"]), 0.02)


def _tokens(case, seed):
    """Hidden states [tokens, n_embd]; with skew s, every token's logits in
    the first layer's router share a bias of -0.13 s ln(rank) per expert, a
    popularity that falls with the expert's rank (about 60 of 512 tokens reach
    the hottest expert of 256 at s = 1.1)."""
    h = _normal(_gen(seed, 300), (case["tokens"], case["n_embd"]), 1.0)
    if case.get("skew"):
        ne = case["n_expert"]
        rank = torch.randperm(ne, generator=_gen(seed, 301), device="cuda") + 1
        b = -0.13 * case["skew"] * torch.log(rank.double())
        w = _routers(case, seed)[0].double()
        mu = w.T @ torch.linalg.solve(w @ w.T, b - b.mean())  # the least-norm solution of w mu = b
        h = h + mu.float()
    return h


# (tag, rows, cols) of a layer's gate, up and down matrices
def _shape(case):
    e, f = case["n_embd"], case["n_ff"]
    n = case.get("n_expert", 1)
    return ((1, n * f, e), (2, n * f, e), (3, n * e, f))


# ---------------------------------------------------------------------------


_stream = None


def _engine():
    """A context on the stream the program uses for all of its GPU work."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    torch.cuda.set_stream(_stream)
    eng = hip.HipEngine(0)
    eng.set_stream(_stream.cuda_stream)
    return eng


def prepare(case, seed):
    eng = _engine()
    gu, dn = TYPES[case["types"]]
    tys = (gu, gu, dn)
    e = case["n_embd"]
    state = dict(case=case, eng=eng)
    if case["kind"] == "dense":
        mats = [synth.Weight(ty, cols, rows, _host(_matrix(seed, tag, ty, rows, cols)))
                for ty, (tag, rows, cols) in zip(tys, _shape(case))]
        state["ffn"] = eng.dense(synth.DenseLayer(e, case["n_ff"], *mats))
    else:
        ne, ff = case["n_expert"], case["n_ff"]
        ups = []
        for ty, (tag, rows, cols) in zip(tys, _shape(case)):
            data = _host(_matrix(seed, tag, ty, rows, cols))
            ups.append(eng.upload_experts(synth.Experts(ty, cols, rows // ne, ne, data, len(data) // ne)))
        sh = [None] * 4
        if case["shared"]:
            sh = [eng.upload_weight(synth.Weight(ty, cols, rows // ne, _host(_matrix(seed, tag + 3, ty, rows // ne, cols))))
                  for ty, (tag, rows, cols) in zip(tys, _shape(case))]
            sh.append(eng.upload_weight(synth.Weight(synth.F32, e, 1, _host(_gate_inp(case, seed)).view(np.uint8))))
        # the layers share the expert matrices' memory and each has a router
        # of its own, so that each reads other experts, as distinct layers do
        state["layers"] = []
        for r in _routers(case, seed):
            router = eng.upload_weight(synth.Weight(synth.F32, e, ne, _host(r).view(np.uint8)))
            state["layers"].append(_moe_block(eng, router, ups, sh, case))
        state["norms"] = _norms(case, seed)
    h = _tokens(case, seed)
    if case.get("entry") == "host":
        h = h.cpu().numpy()
        out = np.zeros_like(h)
    else:
        out = torch.zeros((case.get("layers", 1),) + tuple(h.shape), device="cuda")
    state["h"], state["out"] = h, out
    torch.cuda.synchronize()
    return state


class _Shape:
    """What HipMoe reads of a layer."""

    def __init__(self, case):
        self.n_embd, self.n_expert, self.k, self.n_ff = case["n_embd"], case["n_expert"], case["k"], case["n_ff"]
        self.shared = True if case["shared"] else None


def _moe_block(eng, router, experts, shared, case):
    out = ctypes.c_void_p()
    eng._check(eng.L.biv_hip_moe_create(eng.h, router, *experts, *shared, case["k"], ctypes.byref(out)))
    return hip.HipMoe(eng, out, _Shape(case))


def run(state):
    case, h, out = state["case"], state["h"], state["out"]
    n = case["tokens"]
    if case["kind"] == "dense":
        if case["add"]:  # into the residual, which is the hidden state itself here
            out[0].copy_(h)
        state["ffn"].forward_device(h.data_ptr(), n, out.data_ptr(), add=case["add"])
        return out[0]
    if case["entry"] == "host":
        return state["layers"][0].ffn(h, out=out)
    if case["entry"] == "step":  # the residual goes through the layers in place
        x = out[0]
        x.copy_(h)
        for moe, w in zip(state["layers"], state["norms"]):
            moe.ffn_step_device(x.data_ptr(), w.data_ptr(), EPS, n)
        return x
    for i, moe in enumerate(state["layers"]):
        moe.forward_device(h.data_ptr(), n, out[i].data_ptr())
    return out


def work(case):
    gu, dn = TYPES[case["types"]]
    t, e, f = case["tokens"], case["n_embd"], case["n_ff"]
    expert = (2 * BPW[gu] + BPW[dn]) * e * f
    if case["kind"] == "dense":
        return dict(bytes=expert + (3 if case["add"] else 2) * 4 * t * e, flops=6.0 * t * e * f)
    ne, k, sh = case["n_expert"], case["k"], 1 if case["shared"] else 0
    used = ne * (1 - (1 - k / ne) ** t)  # distinct experts of t tokens
    io = (3 if case["entry"] == "step" else 2) * 4 * t * e
    layer = (used + sh) * expert + 4 * e * (ne + sh) + io
    return dict(bytes=case["layers"] * layer,
                flops=case["layers"] * t * (6.0 * e * f * (k + sh) + 2.0 * e * (ne + sh)))


def tolerance(case):
    # The quantised activations decide: another order of a 32-bit sum moves a
    # value over a rounding boundary here and there, one step of its block.
    # BF16 layers have no such step, only 32-bit sums (and at prefill the
    # two-part split of the activations).
    # Measured against 64 bits: quantised 1e-7 to 7e-4, bf16 3e-7 to 2.8e-5;
    # in a step the residual, about ten times the block, hides most of it.
    step = case.get("entry") == "step"
    if case["types"] == "bf16":
        return {"rel": 1e-5, "max": 2e-4} if step else {"rel": 1e-4, "max": 2e-3}
    return {"rel": 2e-3, "max": 3e-2}


# ---------------------------------------------------------------------------
# The same in 64 bits.


def _q8(x):
    """The activations' 8-bit blocks of 32 (amax / 127 steps, halves away
    from zero), as values."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    r = b / torch.where(d > 0, d, torch.ones_like(d))
    return (torch.trunc(r + torch.copysign(torch.full_like(r, 0.5), r)) * d).reshape(x.shape)


def _mm(x, w, ty):
    return (x if ty == BF16 else _q8(x)) @ w.T


def _swiglu(x, gate, up, down, gu, dn):
    g = _mm(x, gate, gu)
    return _mm(g * torch.sigmoid(g) * _mm(x, up, gu), down, dn)


def exact(case, seed):
    gu, dn = TYPES[case["types"]]
    tys = (gu, gu, dn)
    h = _tokens(case, seed).double()
    mats = [_matrix(seed, tag, ty, rows, cols) for ty, (tag, rows, cols) in zip(tys, _shape(case))]
    if case["kind"] == "dense":
        w = [_values(ty, m, cols) for ty, m, (_, _, cols) in zip(tys, mats, _shape(case))]
        y = _swiglu(h, *w, gu, dn)
        return h + y if case["add"] else y
    ne, k = case["n_expert"], case["k"]

    def expert(i):
        return [_values(ty, m[i * (rows // ne):(i + 1) * (rows // ne)], cols)
                for ty, m, (_, rows, cols) in zip(tys, mats, _shape(case))]

    shared = None
    if case["shared"]:
        shared = [_values(ty, _matrix(seed, tag + 3, ty, rows // ne, cols), cols)
                  for ty, (tag, rows, cols) in zip(tys, _shape(case))]

    def block(x, router):
        p = torch.softmax(x @ router.double().T, -1)
        w, ids = torch.topk(p, k, -1)
        w = w / w.sum(-1, keepdim=True)
        y = torch.zeros_like(x)
        for i in torch.unique(ids).tolist():
            tok, slot = (ids == i).nonzero(as_tuple=True)
            y.index_add_(0, tok, w[tok, slot, None] * _swiglu(x[tok], *expert(i), gu, dn))
        if shared is not None:
            g = torch.sigmoid(x @ _gate_inp(case, seed).double().T)
            y = y + g * _swiglu(x, *shared, gu, dn)
        return y

    routers = _routers(case, seed)
    if case["entry"] != "step":
        ys = [block(h, r) for r in routers]
        return ys[0].cpu().numpy() if case["entry"] == "host" else torch.stack(ys)
    x = h
    for r, nw in zip(routers, _norms(case, seed)):
        x = x + block(x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * nw.double(), r)
    return x
