"""Performance cases: the calls a program makes through qq_hip (the C ABI's
Python binding), at the sizes it makes them.

A case is one of four kinds of call on device pointers:

  layer   MoeLayer.forward_dev / forward_norm_dev: one MoE feed-forward block
          over T token rows (decode T = 1, decode batches, prompt chunks)
  stack   MoeStack.forward_dev: one token through n MoE blocks
  rows    Tensor.matvec_dev: a Q8_0 matrix times `rows` input rows
  lfm2    Lfm2Model.reset + forward_dev: the first tokens of a sequence through
          a whole (short) LFM2-MoE model, logits of every token

Two layer shapes are in use: LFM2-8B-A1B's (H 2048, F 1792, 32 experts, top-4,
sigmoid + bias) and Qwen3-30B-A3B's (H 2048, F 768, 128 experts, top-8,
softmax).  Weights and activations follow the benchmark's distributions: int8
uniform in [-127, 127], fp16 scales |N(0,1)| * 0.002, router N(0, 0.02),
activations N(0, 1).
"""
import math
import os
import struct
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwenqwen3.js_amd"))
import qq_hip  # noqa: E402

QK, QBLK = 32, 34
EPS = 1e-5
# H, F, E, K, softmax gating
SHAPES = {"lfm2": (2048, 1792, 32, 4, False), "qwen3": (2048, 768, 128, 8, True)}
HEAD_DIM, N_HEADS, N_KV, VOCAB, N_FF = 64, 32, 8, 65536, 7168
ROPE_BASE = 5000000.0
# the short LFM2 model: block kinds in order ("a" attention, else short-conv), 2 leading dense FFNs
LFM2_BLOCKS, LFM2_DENSE = "ccacca", 2


# ---------------------------------------------------------------- the cases

def _layer(name, T, shape="lfm2", norm=False, bias="uniform", router="f32", masked=0):
    c = {"kind": "layer", "shape": shape, "T": T, "norm": norm, "bias": bias, "router": router, "masked": masked}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one Q8_0 product of a dense FFN, as a decode step calls it
        {"name": "matvec_1024x3072", "kind": "rows", "in": 1024, "out": 3072, "rows": 1},
        # the same product over the rows of a prompt (LFM2's dense FFN)
        {"name": "rows_200_2048x7168", "kind": "rows", "in": 2048, "out": 7168, "rows": 200},
        # interactive decode: one token, one block
        _layer("decode_1", 1),
        # a handful of concurrent sequences
        _layer("batch_6", 6),
        # a serving batch, uniform routing
        _layer("batch_64", 64),
        # a short prompt (or a prompt's last chunk), ffn_norm folded in
        _layer("prompt_251", 251, norm=True),
        # a prompt chunk with skewed routing: hot and nearly idle experts
        _layer("prefill_2048_zipf", 2048, bias="zipf"),
        # the largest chunk
        _layer("prefill_4096", 4096, norm=True),
        # many small experts: a batch and a prompt
        _layer("qwen3_batch_16", 16, shape="qwen3"),
        _layer("qwen3_prompt_700", 700, shape="qwen3", norm=True),
        # one token through the 22 MoE blocks of the model
        {"name": "stack22_decode", "kind": "stack", "shape": "lfm2", "layers": 22},
        # a whole model: the first tokens of a sequence, logits of each
        {"name": "lfm2_tokens_8", "kind": "lfm2", "tokens": 8},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choices(["layer", "rows", "stack", "lfm2"], [10, 4, 1, 1])[0]
    if kind == "layer":
        shape = rng.choice(["lfm2", "lfm2", "qwen3"])
        return _layer(None, _log_int(rng, 1, 4096), shape=shape, norm=rng.random() < 0.5,
                      bias="uniform" if shape == "qwen3" else rng.choice(["uniform", "zipf"]),
                      router="q8_0" if rng.random() < 0.15 else "f32", masked=3 if rng.random() < 0.15 else 0)
    if kind == "rows":
        i, o = rng.choice([(1024, 3072), (3072, 1024), (2048, 2048), (2048, 512), (2048, 6144), (2048, 7168),
                           (7168, 2048), (2048, 65536), (1792, 2048), (2048, 1792), (1000, 1501), (2080, 777)])
        return {"kind": "rows", "in": i, "out": o, "rows": _log_int(rng, 1, min(2048, int(30e9 / (2.0 * i * o))))}
    if kind == "stack":
        return {"kind": "stack", "shape": rng.choice(["lfm2", "qwen3"]), "layers": rng.randint(2, 22)}
    return {"kind": "lfm2", "tokens": rng.randint(2, 8)}


# ---------------------------------------------------------------- seeded inputs

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gen(seed, salt):
    g = torch.Generator(device=_device())
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)
    return g


def _q8_0(g, in_dim, out_dim, n_mats=1, scale=0.002):
    """GGUF bytes [blocks, 34] of n_mats Q8_0 matrices (weights past in_dim zero)."""
    nb = (in_dim + QK - 1) // QK
    n = n_mats * out_dim * nb
    blocks = torch.empty((n, QBLK), dtype=torch.uint8, device=_device())
    qs = torch.randint(-127, 128, (n, QK), generator=g, device=_device(), dtype=torch.int8)
    if in_dim % QK:
        qs.view(-1, nb, QK)[:, -1, in_dim % QK:] = 0
    blocks[:, 2:] = qs.view(torch.uint8)
    d = (torch.randn(n, generator=g, device=_device()).abs() * scale).to(torch.float16)
    blocks[:, :2] = d.view(torch.uint8).view(n, 2)
    return blocks


def _dense(blocks, in_dim, out_dim):
    """float64 [out_dim, in_dim] of one matrix's GGUF blocks."""
    nb = (in_dim + QK - 1) // QK
    d = blocks[:, :2].contiguous().view(torch.float16).double()
    w = blocks[:, 2:].contiguous().view(torch.int8).double() * d
    return w.view(out_dim, nb * QK)[:, :in_dim]


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=_device(), dtype=torch.float32)


def _moe_inputs(case, seed, salt):
    """Everything of one MoE block: GGUF tensors, router, bias, norm weight, mask."""
    H, F, E, K, softmax = SHAPES[case["shape"]]
    g = _gen(seed, salt)
    rng = np.random.default_rng([int(seed), salt])
    w = {"gate": _q8_0(g, H, F, E), "up": _q8_0(g, H, F, E), "down": _q8_0(g, F, H, E)}
    w["router_q8"] = case.get("router") == "q8_0"
    w["router"] = _q8_0(g, H, E, 1, 0.02 / 64) if w["router_q8"] else _randn(g, E, H) * 0.02
    w["norm"] = torch.rand(H, generator=g, device=_device()) + 0.5
    w["bias"] = None
    if not softmax:
        if case.get("bias") == "zipf":    # expert popularity by Zipf's law (s = 1.1)
            pmf = np.arange(1, E + 1, dtype=np.float64) ** -1.1
            w["bias"] = (0.17 * np.log(pmf[rng.permutation(E)] / pmf.sum())).astype(np.float32)
        else:
            w["bias"] = rng.uniform(-0.01, 0.01, E).astype(np.float32)
    n = case.get("masked", 0)
    w["mask"] = sorted(int(e) for e in rng.choice(E, n, replace=False)) if n else None
    return w


def _layer_rows(case, seed):
    g = _gen(seed, 77)
    H, T = SHAPES[case["shape"]][0], case["T"]
    return _randn(g, T, H), _randn(g, T, H)


def _stack_row(case, seed):
    return _randn(_gen(seed, 78), 1, SHAPES[case["shape"]][0])


def _tokens(case, seed):
    return [int(t) for t in np.random.default_rng([int(seed), 79]).integers(0, VOCAB, case["tokens"])]


def _lfm2_tensors(seed):
    """[(GGUF name, shape, type, tensor)] of the short LFM2-MoE model."""
    H, F, E, _, _ = SHAPES["lfm2"]
    g = _gen(seed, 80)
    nq, nkv = N_HEADS * HEAD_DIM, N_KV * HEAD_DIM
    out = []

    def q8(name, i, o, n=1, scale=0.005):
        out.append((name, [i, o] + ([n] if n > 1 else []), 8, _q8_0(g, i, o, n, scale)))

    def f32(name, t, shape=None):
        out.append((name, shape or [t.numel()], 0, t.contiguous()))

    def norm(name, n):
        f32(name, torch.rand(n, generator=g, device=_device()) + 0.5)

    q8("token_embd.weight", H, VOCAB, scale=0.01)
    norm("token_embd_norm.weight", H)
    for i, kind in enumerate(LFM2_BLOCKS):
        p = "blk.%d." % i
        norm(p + "attn_norm.weight", H)
        norm(p + "ffn_norm.weight", H)
        if kind == "a":
            q8(p + "attn_q.weight", H, nq)
            q8(p + "attn_k.weight", H, nkv)
            q8(p + "attn_v.weight", H, nkv)
            q8(p + "attn_output.weight", nq, H)
            norm(p + "attn_q_norm.weight", HEAD_DIM)
            norm(p + "attn_k_norm.weight", HEAD_DIM)
        else:
            f32(p + "shortconv.conv.weight", _randn(g, H, 3) * 0.5, [3, H])
            q8(p + "shortconv.in_proj.weight", H, 3 * H)
            q8(p + "shortconv.out_proj.weight", H, H)
        if i < LFM2_DENSE:
            q8(p + "ffn_gate.weight", H, N_FF)
            q8(p + "ffn_up.weight", H, N_FF)
            q8(p + "ffn_down.weight", N_FF, H)
        else:
            f32(p + "ffn_gate_inp.weight", _randn(g, E, H) * 0.05, [H, E])
            f32(p + "exp_probs_b.bias", (torch.rand(E, generator=g, device=_device()) - 0.5) * 0.02)
            q8(p + "ffn_gate_exps.weight", H, F, E)
            q8(p + "ffn_up_exps.weight", H, F, E)
            q8(p + "ffn_down_exps.weight", F, H, E)
    return out


def _gguf_bytes(tensors):
    """A GGUF v3 file of the model as one uint8 array."""
    def s(text):
        return struct.pack("<Q", len(text)) + text.encode()

    H, F, E, K, _ = SHAPES["lfm2"]
    p, n = "lfm2moe.", len(LFM2_BLOCKS)
    kvs = [s("general.architecture") + struct.pack("<I", 8) + s("lfm2moe")]
    kvs += [s(p + k) + struct.pack("<II", 4, v) for k, v in (
        ("block_count", n), ("embedding_length", H), ("attention.head_count", N_HEADS), ("expert_count", E),
        ("expert_used_count", K), ("expert_feed_forward_length", F), ("leading_dense_block_count", LFM2_DENSE),
        ("shortconv.l_cache", 3), ("context_length", 4096))]
    kvs += [s(p + k) + struct.pack("<If", 6, v) for k, v in (
        ("attention.layer_norm_rms_epsilon", EPS), ("rope.freq_base", ROPE_BASE))]
    kvs.append(s(p + "attention.head_count_kv") + struct.pack("<IIQ", 9, 5, n) +
               b"".join(struct.pack("<i", N_KV if b == "a" else 0) for b in LFM2_BLOCKS))
    head = b"GGUF" + struct.pack("<IQQ", 3, len(tensors), len(kvs)) + b"".join(kvs)
    rel, pos = [], 0
    for name, shape, typ, t in tensors:
        pos = -(-pos // 32) * 32
        rel.append(pos)
        head += s(name) + struct.pack("<I", len(shape)) + b"".join(struct.pack("<Q", d) for d in shape)
        head += struct.pack("<IQ", typ, pos)
        pos += t.numel() * t.element_size()
    start = -(-len(head) // 32) * 32
    data = np.zeros(start + pos, np.uint8)
    data[:len(head)] = np.frombuffer(head, np.uint8)
    for (_, _, _, t), r in zip(tensors, rel):
        raw = t.reshape(-1).view(torch.uint8).cpu().numpy()
        data[start + r:start + r + raw.size] = raw
    return data


# ---------------------------------------------------------------- states

_CTX = None


def _ctx():
    """The program's one context."""
    global _CTX
    if _CTX is None:
        _CTX = qq_hip.Context(0)
    return _CTX


class State:
    """What a program holds for one case; the library handles are given back with it."""

    def __init__(self, case):
        self.case = case
        self.handles = []      # released in reverse order

    def keep(self, h):
        self.handles.append(h)
        return h

    def __del__(self):
        for h in reversed(self.handles):
            h.release()


def _moe_layer(st, case, w):
    H, F, E, K, softmax = SHAPES[case["shape"]]
    ctx = _ctx()
    torch.cuda.synchronize()
    t = [st.keep(ctx.upload_q8_0_dev(w[n].data_ptr(), w[n].numel(), i, o, E))
         for n, i, o in (("gate", H, F), ("up", H, F), ("down", F, H))]
    typ = qq_hip.TYPE_Q8_0 if w["router_q8"] else qq_hip.TYPE_F32
    layer = st.keep(ctx.moe_create(w["router"].cpu().numpy(), typ, w["bias"], *t, H, F, E, K))
    if softmax:
        layer.set_gating(qq_hip.GATING_SOFTMAX)
    return layer


def _routing(case, n):
    """Device arrays for the selected experts, weights and probabilities of n rows."""
    _, _, E, K, _ = SHAPES[case["shape"]]
    return (torch.zeros((n, K), dtype=torch.int32, device="cuda"), torch.zeros((n, K), dtype=torch.float64, device="cuda"),
            torch.zeros((n, E), dtype=torch.float32, device="cuda"))


def prepare(case, seed):
    st = State(case)
    kind = case["kind"]
    if kind == "layer":
        w = _moe_inputs(case, seed, 1)
        st.layer = _moe_layer(st, case, w)
        st.mask, st.norm = w["mask"], w["norm"]
        st.x, st.hidden = _layer_rows(case, seed)
        st.routing = _routing(case, case["T"])
    elif kind == "stack":
        layers, st.norms = [], []
        for l in range(case["layers"]):
            w = _moe_inputs(case, seed, 1 + l)
            layers.append(_moe_layer(st, case, w))
            st.norms.append(w["norm"])
        st.stack = st.keep(_ctx().moe_stack(layers, [n.data_ptr() for n in st.norms]))
        st.hidden = _stack_row(case, seed)
        st.routing = _routing(case, case["layers"])
    elif kind == "rows":
        w = _q8_0(_gen(seed, 1), case["in"], case["out"])
        torch.cuda.synchronize()
        st.tensor = st.keep(_ctx().upload_q8_0_dev(w.data_ptr(), w.numel(), case["in"], case["out"]))
        st.x = _randn(_gen(seed, 77), case["rows"], case["in"])
        st.y = torch.zeros((case["rows"], case["out"]), dtype=torch.float32, device="cuda")
    else:
        file = qq_hip.Gguf(data=_gguf_bytes(_lfm2_tensors(seed)))
        st.model = st.keep(qq_hip.Lfm2Model(_ctx(), file))
        file.close()
        st.tokens = _tokens(case, seed)
        st.logits = torch.zeros((case["tokens"], VOCAB), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    return st


def run(st):
    case, kind = st.case, st.case["kind"]
    if kind == "layer":
        idx, w, probs = st.routing
        if case["norm"]:
            st.layer.forward_norm_dev(st.hidden.data_ptr(), case["T"], st.norm.data_ptr(), EPS, mask=st.mask,
                                      idx_ptr=idx.data_ptr(), w_ptr=w.data_ptr(), probs_ptr=probs.data_ptr())
        else:
            st.layer.forward_dev(st.x.data_ptr(), st.hidden.data_ptr(), case["T"], mask=st.mask,
                                 idx_ptr=idx.data_ptr(), w_ptr=w.data_ptr(), probs_ptr=probs.data_ptr())
        return {"hidden": st.hidden, "idx": idx, "w": w, "probs": probs}
    if kind == "stack":
        idx, w, probs = st.routing
        st.stack.forward_dev(st.hidden.data_ptr(), 1, EPS, idx_ptr=idx.data_ptr(), w_ptr=w.data_ptr(),
                             probs_ptr=probs.data_ptr())
        return {"hidden": st.hidden, "idx": idx, "w": w, "probs": probs}
    if kind == "rows":
        st.tensor.matvec_dev(st.x.data_ptr(), st.y.data_ptr(), case["rows"])
        return st.y
    st.model.reset()
    for i, t in enumerate(st.tokens):
        st.model.forward_dev(t, i, st.logits[i].data_ptr())
    return st.logits


# ---------------------------------------------------------------- work and tolerance

def _q8_bytes(i, o):
    return o * ((i + QK - 1) // QK) * QBLK


def _moe_work(shape, T):
    """Bytes and operations of one block over T rows; experts touched under even routing."""
    H, F, E, K, _ = SHAPES[shape]
    touched = E * (1.0 - (1.0 - K / E) ** T)
    b = touched * (2 * _q8_bytes(H, F) + _q8_bytes(F, H)) + E * H * 4 + T * H * 4 * 2
    return b, 2.0 * T * K * 3 * H * F + 2.0 * T * H * E


def work(case):
    kind = case["kind"]
    if kind == "layer":
        b, f = _moe_work(case["shape"], case["T"])
        H, _, E, K, _ = SHAPES[case["shape"]]
        return {"bytes": b + case["T"] * (K * 12 + E * 4 + (0 if case["norm"] else H * 4)), "flops": f}
    if kind == "stack":
        b, f = _moe_work(case["shape"], 1)
        return {"bytes": b * case["layers"], "flops": f * case["layers"]}
    if kind == "rows":
        i, o, n = case["in"], case["out"], case["rows"]
        return {"bytes": _q8_bytes(i, o) + 4.0 * n * (i + o), "flops": 2.0 * n * i * o}
    H = SHAPES["lfm2"][0]
    nq, nkv = N_HEADS * HEAD_DIM, N_KV * HEAD_DIM
    n_moe, n_attn = len(LFM2_BLOCKS) - LFM2_DENSE, LFM2_BLOCKS.count("a")
    b, f = _moe_work("lfm2", 1)
    q8 = (len(LFM2_BLOCKS) - n_attn) * (_q8_bytes(H, 3 * H) + _q8_bytes(H, H))
    q8 += n_attn * (_q8_bytes(H, nq + 2 * nkv) + _q8_bytes(nq, H))
    q8 += LFM2_DENSE * 3 * _q8_bytes(H, N_FF) + _q8_bytes(H, VOCAB)
    n = case["tokens"]
    return {"bytes": n * (n_moe * b + q8 + 4.0 * VOCAB), "flops": n * (n_moe * f + 2.0 * q8 * QK / QBLK)}


def tolerance(case):
    # about four times the measured error against the 64-bit values
    if case["kind"] == "layer" and case["T"] >= 512:
        return {"rel": 2e-3, "max": 2e-2}     # fp16 operands and expert outputs, fp32 sums: 5.5e-4
    if case["kind"] == "lfm2":
        return {"rel": 5e-6}                  # fp32 sums through a whole model: 1.2e-6
    if case["kind"] == "stack":
        return {"rel": 5e-6, "differ": 0.01}  # fp32 sums through n blocks: 1.2e-6
    return {"rel": 1.5e-6}                    # fp32 sums: 2e-7 .. 4e-7


# ---------------------------------------------------------------- the values in 64 bits

def _f32(t):
    return t.float().double()


def _norm64(x, w):
    return w.double() * x / (x.square().mean(-1, keepdim=True) + EPS).sqrt()


def _silu64(v):
    return v / (1.0 + torch.exp(-v))


def _moe64(w, case, x):
    """MoE(x) in float64.  The routing is defined on stored fp32 values: logits,
    probabilities and selection scores are rounded where they are stored."""
    H, F, E, K, softmax = SHAPES[case["shape"]]
    x = x.double()
    router = _dense(w["router"], H, E) if w["router_q8"] else w["router"].double()
    logit = _f32(x @ router.t())
    if softmax:
        e = _f32(torch.exp(logit - logit.max(-1, keepdim=True).values))
        probs = _f32(e / e.sum(-1, keepdim=True))
        score = probs
    else:
        probs = _f32(1.0 / (1.0 + torch.exp(-logit)))
        score = _f32(probs + torch.from_numpy(w["bias"]).to(x.device).double())
    idx = torch.sort(score, dim=-1, descending=True, stable=True).indices[:, :K]
    p = torch.gather(probs, 1, idx)
    wk = p / (p.sum(-1, keepdim=True) + (0.0 if softmax else 1e-6))
    out = torch.zeros_like(x)
    nbH, nbF = F * (H // QK), H * (F // QK)
    for e in range(E):
        if w["mask"] and e in w["mask"]:
            continue
        t, k = torch.nonzero(idx == e, as_tuple=True)
        if not t.numel():
            continue
        xe = x[t]
        g = xe @ _dense(w["gate"][e * nbH:(e + 1) * nbH], H, F).t()
        u = xe @ _dense(w["up"][e * nbH:(e + 1) * nbH], H, F).t()
        y = (_silu64(g) * u) @ _dense(w["down"][e * nbF:(e + 1) * nbF], F, H).t()
        out.index_add_(0, t, wk[t, k].unsqueeze(1) * y)
    return out, idx.to(torch.int32), wk, probs


def _lfm264(case, seed):
    """Logits of the sequence in float64."""
    H, F, E, K, _ = SHAPES["lfm2"]
    T = {name: (shape, typ, t) for name, shape, typ, t in _lfm2_tensors(seed)}

    def mat(name):
        shape, _, t = T[name]
        return _dense(t, shape[0], shape[1])

    def vec(name):
        return T[name][2].double()

    def rope(v, pos):
        half = HEAD_DIM // 2
        th = pos / np.float64(np.float32(ROPE_BASE)) ** (torch.arange(half, device=v.device).double() / half)
        a, b = v[:, :half], v[:, half:]
        return torch.cat([a * th.cos() - b * th.sin(), a * th.sin() + b * th.cos()], 1)

    toks = _tokens(case, seed)
    embd = T["token_embd.weight"][2].view(VOCAB, H // QK, QBLK)
    h = torch.stack([_dense(embd[t], H, 1)[0] for t in toks])
    n = len(toks)
    for i, kind in enumerate(LFM2_BLOCKS):
        p = "blk.%d." % i
        x = _norm64(h, vec(p + "attn_norm.weight"))
        if kind == "a":
            q = (x @ mat(p + "attn_q.weight").t()).view(n, N_HEADS, HEAD_DIM)
            k = (x @ mat(p + "attn_k.weight").t()).view(n, N_KV, HEAD_DIM)
            v = (x @ mat(p + "attn_v.weight").t()).view(n, N_KV, HEAD_DIM)
            q = torch.stack([rope(_norm64(q[j], vec(p + "attn_q_norm.weight")), j) for j in range(n)])
            k = torch.stack([rope(_norm64(k[j], vec(p + "attn_k_norm.weight")), j) for j in range(n)])
            o = torch.empty_like(q)
            for hh in range(N_HEADS):
                gk = hh // (N_HEADS // N_KV)
                s = (q[:, hh] @ k[:, gk].t()) / math.sqrt(HEAD_DIM)
                s = s.masked_fill(torch.ones(n, n, device=s.device).triu(1).bool(), -math.inf)
                o[:, hh] = torch.softmax(s, -1) @ v[:, gk]
            h = h + o.reshape(n, -1) @ mat(p + "attn_output.weight").t()
        else:
            b, c, xx = (x @ mat(p + "shortconv.in_proj.weight").t()).split(H, 1)
            bx = torch.cat([torch.zeros(2, H, device=h.device).double(), b * xx])
            kern = T[p + "shortconv.conv.weight"][2].double()          # [H][3], oldest first
            conv = sum(bx[j:j + n] * kern[:, j] for j in range(3))
            h = h + (c * conv) @ mat(p + "shortconv.out_proj.weight").t()
        x = _norm64(h, vec(p + "ffn_norm.weight"))
        if i < LFM2_DENSE:
            a = _silu64(x @ mat(p + "ffn_gate.weight").t()) * (x @ mat(p + "ffn_up.weight").t())
            h = h + a @ mat(p + "ffn_down.weight").t()
        else:
            w = {"router_q8": False, "mask": None, "router": T[p + "ffn_gate_inp.weight"][2],
                 "bias": T[p + "exp_probs_b.bias"][2].cpu().numpy(), "gate": T[p + "ffn_gate_exps.weight"][2],
                 "up": T[p + "ffn_up_exps.weight"][2], "down": T[p + "ffn_down_exps.weight"][2]}
            h = h + _moe64(w, {"shape": "lfm2"}, x)[0]
    return _norm64(h, vec("token_embd_norm.weight")) @ mat("token_embd.weight").t()


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        w = _moe_inputs(case, seed, 1)
        x, hidden = _layer_rows(case, seed)
        hidden = hidden.double()
        xin = _f32(_norm64(hidden, w["norm"])) if case["norm"] else x
        out, idx, wk, probs = _moe64(w, case, xin)
        return {"hidden": hidden + out, "idx": idx, "w": wk, "probs": probs}
    if kind == "stack":
        h = _stack_row(case, seed).double()
        route = []
        for l in range(case["layers"]):
            w = _moe_inputs(case, seed, 1 + l)
            out, *r = _moe64(w, case, _norm64(h, w["norm"]))
            h = h + out
            route.append(r)
        idx, wk, probs = (torch.cat(r) for r in zip(*route))
        return {"hidden": h, "idx": idx, "w": wk, "probs": probs}
    if kind == "rows":
        w = _dense(_q8_0(_gen(seed, 1), case["in"], case["out"]), case["in"], case["out"])
        return _randn(_gen(seed, 77), case["rows"], case["in"]).double() @ w.t()
    return _lfm264(case, seed)
