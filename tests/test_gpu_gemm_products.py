"""The engine's GEMM kernels against 64 bits, seen through a short conv's state.

The products of the two-part weights (scales outside [-64, 64]) in full:

A weight of odd magnitude above 2048 is not a binary16 number: the kernels hold it as
w + r (r = +-1) and the activation as hi + lo.  The inputs here make lo decide the
result, so a weight that met lo rounded to w is off by 1 / 3937 and more.

And super-block scales at their edges: lfm_q6k_gemm reads the planes up to 1024 tokens,
so the kernels over the tile copies, which every call of a model runs, are reached
through a model here.
"""
import numpy as np
import pytest

from model_util import gpu_engine, model_tensors
from test_gpu_kernels import blocks, edge_scales, encode_q6k

pytestmark = pytest.mark.gpu

DIM = 512


@pytest.mark.parametrize("T", [1, 33, 1024, 1280])
def test_odd_weight_times_low_half(gpu, T):
    """One-hot tokens 1 + 2^-12 (hi 1, lo 2^-12) against weights sc (q - 32) of every
    magnitude up to 4096: the product has 24 bits or fewer, as has every partial sum, so
    it comes out exactly.  T <= 1024 reads the planes, 1280 the copies."""
    rows, in_dim = 256, 512
    codes = (np.arange(in_dim)[None, :] + np.arange(rows)[:, None]) % 64
    scales = np.repeat((-128 + np.arange(rows))[:, None], in_dim // 16, axis=1)
    raw = encode_q6k(codes.reshape(-1, 256), scales.reshape(-1, 16), np.ones(rows * in_dim // 256))
    k = (7 * np.arange(T)) % in_dim
    x = np.zeros((T, in_dim), dtype=np.float32)
    x[np.arange(T), k] = 1 + 2.0 ** -12
    y = gpu.q6k_gemm(gpu.Q6Weight(raw.reshape(-1), rows, in_dim), x)
    want = (scales[:, k // 16] * (codes[:, k] - 32)).T * (1 + 2.0 ** -12)
    assert np.array_equal(want, want.astype(np.float32))
    bad = np.argwhere(y != want)
    assert bad.size == 0, [(int(t), int(r), float(y[t, r]), float(want[t, r])) for t, r in bad[:8]]


def q6k(weights, scale):
    """Raw blocks of a [rows][k] matrix scale * (-32 .. 31), with d = 1."""
    rows, k = weights.shape
    q = (weights // scale + 32).astype(int)
    assert np.array_equal((q - 32) * scale, weights) and q.min() >= 0 and q.max() <= 63
    n = rows * k // 256
    sc = np.broadcast_to(np.broadcast_to(scale, weights.shape)[:, ::16], (rows, k // 16)).reshape(n, 16)
    return encode_q6k(q.reshape(n, 256), sc, np.ones(n)).reshape(-1)


def one_hot(rows, cols, k):
    m = np.zeros((rows, k), dtype=int)
    m[np.arange(rows), cols] = 1
    return m


def conv_model(gpu, emb, nw, raws):
    """Three short-conv layers with dense FFNs over the embedding emb (whole numbers), the
    norms of layer 0 with weights nw; every matrix that `raws` leaves out is zero.
    Returns the rows that layer 0's norms make, too."""
    dim = emb.shape[1]
    hp = gpu.make_hparams(dim=dim, heads=dim // 64, n_layers=3, attention_layers=(), kv=dim // 256, vocab=len(emb),
                          eos=1 << 30, n_expert=8, n_used=2, expert_ff=256, n_ff=512, dense_lead=3)
    own = {"token_embd.weight": q6k(emb, 1), "blk.0.attn_norm.weight": nw, "blk.0.ffn_norm.weight": nw, **raws}
    tensors = []
    for name, t, shape, data in model_tensors(hp):
        zero = np.ones_like(data) if t == 0 else np.zeros_like(data)
        tensors.append((name, t, shape, own.get(name, zero)))
    inv = 1 / np.sqrt(np.mean(emb * emb.astype(np.float64), axis=1) + np.float64(np.float32(hp.eps)))
    return hp, tensors, emb * inv[:, None] * nw.astype(np.float64)


def probe_model(gpu, delta, raws):
    """Token 0's embedding is +1, -1, +1, .., token 1's the negative; the norms weigh
    column 2i by 1 + delta_i, so a row of equal weights sums delta: the hi halves (1 in
    every column) cancel and the lo halves stay."""
    nw = np.ones(DIM, np.float32)
    nw[::2] += delta
    emb = np.ones((300, DIM), dtype=int)
    emb[0, 1::2] = emb[1, ::2] = -1
    return conv_model(gpu, emb, nw, raws)


def conv_states(g, n):
    return np.frombuffer(g.snapshot_resident_cache(n), np.float32).reshape(3, -1, 2).astype(np.float64)


def near(got, want):
    """Relative error 5e-5: an element of the normalised row is rounded to 2^-24 of
    itself, 2^-12 of delta, which the 256 terms of a sum average to 1e-5; a weight
    rounded to binary16 for the lo halves is off by 2.5e-4."""
    err = np.abs(got - want) / np.abs(want)
    assert err.max() <= 5e-5, (np.unravel_index(err.argmax(), err.shape), err.max())


DELTA = np.float32(2.0 ** -12) * (1 + np.random.default_rng(5).integers(0, 2 ** 10, DIM // 2).astype(np.float32) / 2 ** 11)


@pytest.mark.parametrize("n", [2, 33, 130, 704, 705, 830])
def test_single_weight_sums_low_halves(gpu, n):
    """Layer 0's in_proj: rows of 3937 (B) and one column each (X); the conv state is
    B X of the last two tokens.  705 tokens and more run the large-call kernel."""
    in_proj = np.zeros((3 * DIM, DIM), dtype=int)
    scale = np.ones((3 * DIM, DIM), dtype=int)
    in_proj[:DIM], scale[:DIM] = 127 * 31, 127
    col = np.random.default_rng(1).integers(0, DIM, DIM)
    in_proj[2 * DIM:] = one_hot(DIM, col, DIM)
    hp, tensors, h = probe_model(gpu, DELTA, {"blk.0.shortconv.in_proj.weight": q6k(in_proj, scale)})
    g = gpu_engine(hp, tensors, ctx=1024)
    g.forward([0, 1] * (n // 2) + [0] * (n % 2), 0)
    state = conv_states(g, n)[0]
    g.close()
    last = [(n - 2) % 2, (n - 1) % 2]
    near(state, np.stack([h[t].sum() * 3937 * h[t][col] for t in last], axis=1))


@pytest.mark.parametrize("n", [2, 33, 130, 704, 705, 830])
def test_gate_up_pair_sums_low_halves(gpu, n):
    """Layer 0's FFN adds silu(gate) up to the residual, with up rows of 3937 (even) and
    -2048 (odd: exact in binary16); layer 1's conv state shows the residual's rows, whose
    ratio changes if only the even ones lose their remainder."""
    gate = 20 * one_hot(DIM, np.zeros(DIM, dtype=int), DIM)
    up = np.full((DIM, DIM), 127 * 31)
    scale = np.full((DIM, DIM), 127)
    up[1::2], scale[1::2] = -2048, 64
    eye = one_hot(DIM, np.arange(DIM), DIM)
    in_proj = np.concatenate([eye, 0 * eye, one_hot(DIM, np.full(DIM, 3), DIM)])
    hp, tensors, h = probe_model(gpu, DELTA, {
        "blk.0.ffn_gate.weight": q6k(gate, 1), "blk.0.ffn_up.weight": q6k(up, scale),
        "blk.0.ffn_down.weight": q6k(eye, 1), "blk.1.shortconv.in_proj.weight": q6k(in_proj, 1)})
    g = gpu_engine(hp, tensors, ctx=1024)
    g.forward([0] * n, 0)  # (token 0: its gate, 20 h[0], is positive)
    state = conv_states(g, n)[1]
    g.close()
    gt = gate @ h[0]
    x = np.where(np.arange(DIM) % 2, -1.0, 1.0) + gt / (1 + np.exp(-gt)) * (up @ h[0])
    hx = x / np.sqrt(np.mean(x * x) + np.float64(np.float32(hp.eps)))
    near(state, np.stack([hx * hx[3]] * 2, axis=1))


@pytest.mark.parametrize("n,h16", [(2, "1"), (31, "1"), (33, "1"), (130, "1"), (704, "1"), (705, "1"), (705, "0"), (1000, "1"),
                                   (1000, "0")])
@pytest.mark.parametrize("sc_lim", [32, 128])
def test_block_scale_edges(gpu, oracle, monkeypatch, n, h16, sc_lim):
    """in_proj with B rows whose super-block scales are zero, -0.0, subnormal or eleven
    decades apart within the row, X rows of one column each: the conv state's B X of the
    last two tokens against float64, for the tile-copy kernels of small calls and, from
    705 tokens, the binary16 copies or (h16 0) the Q6_K weights; sc_lim 128: the two-part
    weights.  Relative to |row| |h| / sqrt(dim) |X|, the size of such a product: 1e-5, the
    bar of the GEMMs."""
    monkeypatch.setenv("LFM_PREFILL_H16", h16)
    dim, nb = 2048, 8
    rng = np.random.default_rng(n)
    raw = blocks(3 * dim * nb, 7, sc_lim=sc_lim).reshape(3 * dim, nb, 210)
    d, kind = edge_scales(dim, nb, rng)
    raw[:dim, :, 208:210] = d.view(np.uint8).reshape(dim, nb, 2)
    col = rng.integers(0, dim, dim)
    raw[2 * dim:] = q6k(one_hot(dim, col, dim), 1).reshape(dim, nb, 210)
    emb = rng.integers(1, 32, (300, dim)) * rng.choice([-1, 1], (300, dim))
    hp, tensors, h = conv_model(gpu, emb, rng.uniform(0.5, 2, dim).astype(np.float32),
                                {"blk.0.shortconv.in_proj.weight": raw.reshape(-1)})
    ids = rng.integers(0, 300, n)
    g = gpu_engine(hp, tensors, ctx=1024)
    g.forward([int(t) for t in ids], 0)
    state = conv_states(g, n)[0]
    g.close()
    w = oracle.dequant_rows(raw[:dim].reshape(-1), dim, dim).astype(np.float64).reshape(dim, dim)
    ht = h[ids[-2:]].T
    want = (w @ ht) * ht[col]
    size = np.linalg.norm(w, axis=1)[:, None] * np.linalg.norm(ht, axis=0) / np.sqrt(dim) * np.abs(ht[col])
    assert not state[kind == 0].any()
    err = np.abs(state - want)[kind != 0] / size[kind != 0]
    assert err.max() <= 1e-5, (np.unravel_index(err.argmax(), err.shape), err.max())
