"""What a user of this framework has it do, as cases that can be timed and compared.

Two models stand for the work.  "full" is the LFM2.5-8B-A1B shape that bench.py
measures (24 layers: 18 short convs and 6 attentions; dense FFNs in layers 0-1, 32
experts top-4 after that).  "block" holds one of each kind of its layers at their real
widths (conv + dense, conv + MoE, attention + MoE, conv + MoE) under the same head, so
that a pass through it can be checked against 64-bit arithmetic.  Weights are seeded
Q6_K blocks; `scales` 1 gives them sub-block scales over the whole int8 range, the form
quantizers write into model files, 0 the narrower ones of the benchmark's model.

Sessions that start past position 0 resume a seeded state of the values such a state
holds (K normalised per head; V and the conv state as large as the projections make
them), as a server that keeps sessions does.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "lfm2-w9100-rust_amd"))
import lfm_hip  # noqa: E402

CTX = 4096
MODELS = {
    "block": dict(n_layers=4, attention_layers=(2,), dense_lead=1),
    "full": dict(n_layers=24, attention_layers=lfm_hip.LFM2_ATTENTION_LAYERS, dense_lead=2),
}


def listed():
    return [
        # One token with its logits at a position deep in a chat: the step of a program
        # that samples on the host, the smallest call of a model.
        {"name": "sample_step", "kind": "forward", "model": "block", "scales": 1, "start": 2900, "tokens": 1},
        # The greedy loop on the device at the end of a full context: the benchmark's
        # headline, on the whole model.
        {"name": "decode_full", "kind": "decode", "model": "full", "scales": 0, "start": 3840, "tokens": 32},
        # A short user turn appended to a running chat.
        {"name": "turn_7", "kind": "forward", "model": "block", "scales": 1, "start": 731, "tokens": 7},
        # A first message of ordinary length in an empty session.
        {"name": "message_37", "kind": "forward", "model": "block", "scales": 0, "start": 0, "tokens": 37},
        # One 64-token chunk of a long prompt, the api_stream driver's prefill step.
        {"name": "chunk_64", "kind": "chunk", "model": "block", "scales": 1, "start": 1984, "tokens": 64},
        # Prompts between a message and a document, through one call each: a system
        # prompt with a question (an odd length), a page, several pages.
        {"name": "prompt_203", "kind": "forward", "model": "block", "scales": 0, "start": 0, "tokens": 203},
        {"name": "prompt_512", "kind": "forward", "model": "block", "scales": 1, "start": 0, "tokens": 512},
        {"name": "prompt_1500", "kind": "forward", "model": "block", "scales": 1, "start": 0, "tokens": 1500},
        # The benchmark's prompt on the whole model: the largest call.
        {"name": "prompt_3840_full", "kind": "forward", "model": "full", "scales": 0, "start": 0, "tokens": 3840},
        # A server that keeps more sessions than engines: the resident one is parked, a
        # parked one resumed and continued by a token.
        {"name": "session_switch", "kind": "session", "model": "block", "scales": 0, "start": 1900, "tokens": 1},
        # The operator API on device buffers: one row of activations through the dense
        # down projection, and a prompt's rows through the short conv's input projection.
        {"name": "matvec_down", "kind": "matvec", "rows": 2048, "in_dim": 7168, "scales": 1},
        {"name": "gemm_in_proj", "kind": "gemm", "rows": 6144, "in_dim": 2048, "tokens": 300, "scales": 0},
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choices(["prompt", "turn", "chunk", "step", "decode", "session", "matvec", "gemm"],
                       [32, 14, 10, 8, 12, 8, 8, 8])[0]
    scales = rng.randint(0, 1)
    if kind == "prompt":  # up to a whole context in one call
        return {"kind": "forward", "model": "block", "scales": scales, "start": 0,
                "tokens": _log_uniform(rng, 2, CTX)}
    if kind == "turn":
        return {"kind": "forward", "model": "block", "scales": scales, "start": _log_uniform(rng, 16, 3000),
                "tokens": _log_uniform(rng, 2, 600)}
    if kind == "chunk":
        return {"kind": "chunk", "model": "block", "scales": scales, "start": 64 * rng.randint(1, 60),
                "tokens": rng.choice([64, 64, rng.randint(1, 63)])}
    if kind == "step":
        return {"kind": "forward", "model": "block", "scales": scales, "start": _log_uniform(rng, 8, CTX - 2),
                "tokens": 1}
    if kind == "decode":
        full = rng.random() < 0.2
        n = rng.randint(8, 32)
        return {"kind": "decode", "model": "full" if full else "block", "scales": scales,
                "start": _log_uniform(rng, 32, CTX - n - 1), "tokens": n}
    if kind == "session":
        return {"kind": "session", "model": "block", "scales": scales, "start": _log_uniform(rng, 64, CTX - 2),
                "tokens": 1}
    in_dim = 256 * rng.choice([8, 8, 7, 28, rng.randint(1, 32)])
    rows = _log_uniform(rng, 200, 16384)
    if kind == "matvec":
        return {"kind": "matvec", "rows": rows, "in_dim": in_dim, "scales": scales}
    return {"kind": "gemm", "rows": rows, "in_dim": in_dim, "tokens": _log_uniform(rng, 2, 1024), "scales": scales}


# ------------------------------------------------------------------ inputs
def _hparams(case):
    return lfm_hip.make_hparams(**MODELS[case["model"]])


def _opts(case, seed):
    return lfm_hip.synth_opts(seed=0x5EED0000 + seed, full_scales=case["scales"])


def _ids(hp, n, seed):
    return np.random.default_rng([seed, 1]).integers(0, hp.vocab, n, dtype=np.uint32)


def _session(case, hp, valid, seed, which=0):
    """A session's state at `valid` tokens in the snapshot's byte order: per attention
    layer K then V [valid][kv * 64], per conv layer [dim][2]; K and V are binary16
    values, as every snapshot's are."""
    g = torch.Generator().manual_seed(1000003 * which + seed)
    big = 4.0 if case["scales"] else 1.0
    out = []
    for layer in range(hp.n_layers):
        kv = hp.kv_heads[layer]
        if kv:
            out.append(torch.randn(valid * kv * 64, generator=g).half().float())
            out.append((15.0 * big * torch.randn(valid * kv * 64, generator=g)).half().float())
        else:
            out.append(225.0 * big * big * torch.randn(hp.dim * 2, generator=g))
    return torch.cat(out).numpy()


def _weight(case, seed):
    return lfm_hip.synth_q6k_blocks(0x5EED0000 + seed, "op.weight", case["rows"] * case["in_dim"] // 256,
                                    threads=16, full_scales=bool(case["scales"]))


def _activations(case, seed):
    n = case.get("tokens", 1)
    g = torch.Generator().manual_seed(seed)
    return torch.randn(n, case["in_dim"], generator=g)


def prepare(case, seed):
    if case["kind"] in ("matvec", "gemm"):
        rows, n = case["rows"], case.get("tokens", 1)
        return {"case": case, "w": lfm_hip.Q6Weight(_weight(case, seed), rows, case["in_dim"]),
                "x": _activations(case, seed).cuda(), "y": torch.empty(n, rows, device="cuda")}
    hp = _hparams(case)
    e = lfm_hip.GpuEngine.load_synthetic(hp, _opts(case, seed), ctx=CTX, threads=16)
    state = {"case": case, "engine": e, "ids": _ids(hp, case["tokens"], seed)}
    if case["start"]:
        e.restore_session(case["start"], _session(case, hp, case["start"], seed).tobytes())
    if case["kind"] == "session":
        state["parked"] = _session(case, hp, case["start"], seed, which=1).tobytes()
    return state


# ------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("matvec", "gemm"):
        w, x, y, lib = state["w"], state["x"], state["y"], lfm_hip.lib()
        if kind == "matvec":
            rc = lib.lfm_q6k_matvec(w.buf.ptr, w.rows, w.in_dim,
                                    ctypes.cast(x.data_ptr(), ctypes.c_void_p),
                                    ctypes.cast(y.data_ptr(), ctypes.c_void_p), None)
        else:
            rc = lib.lfm_q6k_gemm(w.buf.ptr, w.rows, w.in_dim,
                                  ctypes.cast(x.data_ptr(), ctypes.c_void_p), x.shape[0],
                                  ctypes.cast(y.data_ptr(), ctypes.c_void_p), None)
        if rc:
            raise RuntimeError(lib.lfm_last_error().decode())
        return y
    e, ids, start = state["engine"], state["ids"], case["start"]
    if kind == "forward":
        if start == 0:
            e.reset_session()
        return e.forward(ids, start)
    if kind == "chunk":
        e.forward_token(ids, start)
        return {"max": e.last_max_logit, "logits": e.snapshot_resident_logits()}
    if kind == "decode":
        tokens = e.decode_run(int(ids[0]), start, case["tokens"], eos=0xFFFFFFFF)
        return {"tokens": np.array(tokens, dtype=np.int64), "logits": e.snapshot_resident_logits()}
    resumed = state["parked"]
    parked = state["parked"] = e.snapshot_resident_cache(start)
    e.restore_session(start, resumed)
    return {"parked": np.frombuffer(parked, dtype=np.float32), "logits": e.forward(ids, start)}


# ------------------------------------------------------------------ work
def work(case):
    if case["kind"] in ("matvec", "gemm"):
        rows, k, n = case["rows"], case["in_dim"], case.get("tokens", 1)
        return {"bytes": lfm_hip.q6k_nbytes(rows, k) + 4 * n * (k + rows), "flops": 2 * n * rows * k}
    hp = _hparams(case)
    dim, steps = hp.dim, 1
    n, start = case["tokens"], case["start"]
    if case["kind"] == "decode":
        n, steps = 1, case["tokens"]
    per = lfm_hip.Q6_K_BYTES / lfm_hip.QK_K
    weights = flops = kv_bytes = 0.0
    for layer in range(hp.n_layers):
        rows = n if layer + 1 < hp.n_layers else 1  # the last layer's FFN runs for the last token
        kv = hp.kv_heads[layer]
        if kv:
            w = 2 * dim * dim + 2 * 64 * kv * dim
            pairs = n * start + n * (n + 1) // 2
            flops += 2 * n * w + 4 * 64 * hp.heads * pairs
            kv_bytes += 2 * 64 * kv * 2 * (start + n)
            weights += w * per
        else:
            w = 4 * dim * dim
            flops += 2 * n * w
            weights += w * per
        if layer < hp.dense_lead:
            flops += 2 * rows * 3 * hp.n_ff * dim
            weights += 3 * hp.n_ff * dim * per
        else:
            touched = hp.n_expert * (1 - (1 - hp.n_used / hp.n_expert) ** rows)
            flops += 2 * rows * (hp.n_expert * dim + hp.n_used * 3 * hp.expert_ff * dim)
            weights += touched * 3 * hp.expert_ff * dim * per + 4 * hp.n_expert * dim
    flops += 2 * hp.vocab * dim
    weights += hp.vocab * dim * per + n * dim * per
    total = steps * (weights + kv_bytes) + 4 * hp.vocab
    if case["kind"] == "session":  # the cache read and written in binary16, both blobs in fp32
        total += 6 * 2 * sum(2 * 64 * hp.kv_heads[l] * start for l in range(hp.n_layers))
    return {"bytes": total, "flops": steps * flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("matvec", "gemm"):  # 4 x the 4.1e-7 that fp32 sums over 2048 inputs show
        return {"rel": 2e-6, "max": 2e-5}
    if case["model"] == "full":
        # 1.1e-5 between the batched and the token-by-token forward; 22 layers choose
        # experts, and where two scores nearly tie a difference in rounding chooses
        # another one, which every later layer and position sees
        return {"rel": 1e-3, "max": 0.01, "differ": 0.0}
    return {"rel": 1e-5, "max": 6e-5, "differ": 0.0}  # 4 x the 2.5e-6 that prompts show


# ------------------------------------------------------------------ 64 bits
def _dequant(raw, dev):
    """Raw Q6_K bytes -> float64 weights, 256 per 210-byte block."""
    b = torch.from_numpy(np.ascontiguousarray(raw)).to(dev).view(-1, 210)
    n = b.shape[0]
    ql = b[:, :128].view(n, 2, 2, 32).int()
    qh = b[:, 128:192].view(n, 2, 32).int()
    sc = b[:, 192:208].contiguous().view(torch.int8).view(n, 2, 4, 2).double()
    d = b[:, 208:210].contiguous().view(torch.float16).double().view(n, 1, 1, 1)
    q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4),
                     (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                     (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4),
                     (ql[:, :, 1] >> 4) | (((qh >> 6) & 3) << 4)], dim=2) - 32
    return ((d * sc).unsqueeze(-1) * q.view(n, 2, 4, 2, 16).double()).reshape(-1)


class _Exact:
    """The model in 64 bits.  Kept from the format: weights, K and V as binary16, rotary
    angles as 32-bit numbers."""

    def __init__(self, case, seed, dev):
        self.hp, self.opts, self.dev = _hparams(case), _opts(case, seed), dev
        self.descs = {d.name.decode(): d for d in lfm_hip.model_tensor_descs(self.hp, self.opts)}
        self.raw, self.k, self.v, self.conv = {}, {}, {}, {}
        for layer in range(self.hp.n_layers):
            kv = self.hp.kv_heads[layer]
            if kv:
                self.k[layer] = torch.zeros(0, kv, 64, dtype=torch.float64, device=dev)
                self.v[layer] = torch.zeros(0, kv, 64, dtype=torch.float64, device=dev)
            else:
                self.conv[layer] = torch.zeros(self.hp.dim, 2, dtype=torch.float64, device=dev)

    def restore(self, flat, valid):
        at = 0
        flat = torch.from_numpy(flat).to(self.dev).double()
        for layer in range(self.hp.n_layers):
            kv = self.hp.kv_heads[layer]
            if kv:
                n = valid * kv * 64
                self.k[layer] = flat[at:at + n].view(valid, kv, 64)
                self.v[layer] = flat[at + n:at + 2 * n].view(valid, kv, 64)
                at += 2 * n
            else:
                n = self.hp.dim * 2
                self.conv[layer] = flat[at:at + n].view(self.hp.dim, 2)
                at += n

    def tensor(self, name, expert=None):
        d = self.descs[name]
        if name not in self.raw:
            self.raw[name] = lfm_hip.synth_tensor(d, self.opts, threads=16)
        raw = self.raw[name]
        if d.ggml_type != lfm_hip.GGML_TYPE_Q6_K:
            return torch.from_numpy(raw).to(self.dev).double().view(*reversed(d.shape))
        if expert is None:
            return _dequant(raw, self.dev).view(d.shape[1], d.shape[0])
        size = raw.size // d.shape[2]
        return _dequant(raw[expert * size:(expert + 1) * size], self.dev).view(d.shape[1], d.shape[0])

    def norm(self, x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + float(np.float32(self.hp.eps))) * w

    def angles(self, start, n):
        scale = np.power(np.float32(self.hp.rope_theta), np.float32(-2.0 / 64))
        th = np.zeros((n, 32), dtype=np.float32)
        for p in range(32):
            r, a, b = np.float32(1), np.float32(scale), p
            while True:
                if b & 1:
                    r = np.float32(r * a)
                b //= 2
                if b == 0:
                    break
                a = np.float32(a * a)
            th[:, p] = np.arange(start, start + n, dtype=np.float32) * r
        th = torch.from_numpy(th).to(self.dev).double()
        return th.cos().unsqueeze(1), th.sin().unsqueeze(1)

    def attention(self, layer, h, start):
        hp, n, kv = self.hp, h.shape[0], self.hp.kv_heads[layer]
        p = "blk.%d." % layer
        c, s = self.angles(start, n)

        def rotated(x):
            a, b = x[..., :32], x[..., 32:]
            return torch.cat([a * c - b * s, a * s + b * c], -1)

        q = rotated(self.norm((h @ self.tensor(p + "attn_q.weight").T).view(n, hp.heads, 64),
                              self.tensor(p + "attn_q_norm.weight")))
        k = rotated(self.norm((h @ self.tensor(p + "attn_k.weight").T).view(n, kv, 64),
                              self.tensor(p + "attn_k_norm.weight")))
        v = (h @ self.tensor(p + "attn_v.weight").T).view(n, kv, 64)
        self.k[layer] = torch.cat([self.k[layer], k.half().double()])
        self.v[layer] = torch.cat([self.v[layer], v.half().double()])
        keys = torch.arange(start + n, device=self.dev)
        mask = keys[None, :] > torch.arange(start, start + n, device=self.dev)[:, None]
        out = torch.empty(n, hp.heads, 64, dtype=torch.float64, device=self.dev)
        for head in range(hp.heads):
            g = head * kv // hp.heads
            score = (q[:, head] @ self.k[layer][:, g].T) / 8.0
            out[:, head] = torch.softmax(score.masked_fill(mask, -math.inf), -1) @ self.v[layer][:, g]
        return out.view(n, -1) @ self.tensor(p + "attn_output.weight").T

    def short_conv(self, layer, h):
        p = "blk.%d.shortconv." % layer
        b, c, x = (h @ self.tensor(p + "in_proj.weight").T).chunk(3, -1)
        taps = self.tensor(p + "conv.weight")  # [dim][3]
        seq = torch.cat([self.conv[layer].T, b * x])
        self.conv[layer] = seq[-2:].T.contiguous()
        n = h.shape[0]
        y = c * sum(seq[i:i + n] * taps[:, i] for i in range(3))
        return y @ self.tensor(p + "out_proj.weight").T

    def ffn(self, layer, x):
        hp, p = self.hp, "blk.%d." % layer
        h = self.norm(x, self.tensor(p + "ffn_norm.weight"))
        if layer < hp.dense_lead:
            g = torch.nn.functional.silu(h @ self.tensor(p + "ffn_gate.weight").T)
            return (g * (h @ self.tensor(p + "ffn_up.weight").T)) @ self.tensor(p + "ffn_down.weight").T
        prob = torch.sigmoid(h @ self.tensor(p + "ffn_gate_inp.weight").T)
        top = (prob + self.tensor(p + "exp_probs_b.bias")).topk(hp.n_used, -1).indices
        w = prob.gather(-1, top)
        w = w / w.sum(-1, keepdim=True).clamp(min=6.103515625e-5)
        out = torch.zeros_like(x)
        for ex in range(hp.n_expert):
            row, rank = (top == ex).nonzero(as_tuple=True)
            if row.numel():
                a = h[row]
                g = torch.nn.functional.silu(a @ self.tensor(p + "ffn_gate_exps.weight", ex).T)
                g = g * (a @ self.tensor(p + "ffn_up_exps.weight", ex).T)
                out.index_add_(0, row, w[row, rank, None] * (g @ self.tensor(p + "ffn_down_exps.weight", ex).T))
        return out

    def forward(self, ids, start):
        hp = self.hp
        emb = self.tensor("token_embd.weight")
        x = emb[torch.from_numpy(np.asarray(ids, dtype=np.int64)).to(self.dev)]
        for layer in range(hp.n_layers):
            h = self.norm(x, self.tensor("blk.%d.attn_norm.weight" % layer))
            x = x + (self.attention(layer, h, start) if hp.kv_heads[layer] else self.short_conv(layer, h))
            if layer + 1 == hp.n_layers:
                x = x[-1:]
            x = x + self.ffn(layer, x)
        return (self.norm(x, self.tensor("token_embd_norm.weight")) @ emb.T).view(-1)


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] in ("matvec", "gemm"):
        w = _dequant(_weight(case, seed), dev).view(case["rows"], case["in_dim"])
        return _activations(case, seed).to(dev).double() @ w.T
    if case["model"] == "full":
        # Over 22 layers of expert choices the distance from a 64-bit answer says which
        # near ties fell the other way, not how exact the sums are: the same layers are
        # compared in the block model.
        return None
    hp = _hparams(case)
    start, ids = case["start"], _ids(hp, case["tokens"], seed)
    m = _Exact(case, seed, dev)
    if case["kind"] == "session":
        m.restore(_session(case, hp, start, seed, which=1), start)
        return {"parked": _session(case, hp, start, seed).astype(np.float64), "logits": m.forward(ids, start)}
    if start:
        m.restore(_session(case, hp, start, seed), start)
    if case["kind"] == "decode":
        token, tokens = int(ids[0]), []
        for i in range(case["tokens"]):
            logits = m.forward([token], start + i)
            token = int(logits.argmax())
            tokens.append(token)
        return {"tokens": np.array(tokens, dtype=np.int64), "logits": logits}
    logits = m.forward(ids, start)
    if case["kind"] == "chunk":
        return {"max": float(logits.max()), "logits": logits}
    return logits
