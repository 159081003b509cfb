"""Multi-token forwards around the line between the small-call and the large-call kernels.

Bars: logits and resident state rel-L2 <= 1e-3 against the oracle (the bar of the layer
outputs).  Between two paths of the engine, whose sums differ in order only: 2e-5 for
logits and conv states (fp32 sums and 22-bit activations, ~1e-6 per layer); a token's K
and V are binary16, so an element next to a rounding boundary moves by 2^-11 of itself
(a few in a thousand do: ~3e-5), and a token whose expert choice is a near tie within
that rounding may choose another expert (~1e-5 of the decisions), so 1 % of the tokens
may be further off than 2e-4.
"""
import numpy as np
import pytest

from conftest import rel_l2
from model_util import gpu_engine, model_tensors, oracle_engine

pytestmark = pytest.mark.gpu


def ids(n, vocab, seed):
    return [int(t) for t in np.random.default_rng(seed).integers(0, vocab, n)]


def state(g, n):
    return np.frombuffer(g.snapshot_resident_cache(n), np.float32)


def check_same(hp, n, a, b):
    """Snapshots a and b of two paths (see the bars above)."""
    at = 0
    for layer in range(hp.n_layers):
        kv = hp.kv_heads[layer]
        size = n * kv * 64 if kv else hp.dim * 2
        for _ in range(2 if kv else 1):
            x, y = a[at:at + size].astype(np.float64), b[at:at + size].astype(np.float64)
            at += size
            if kv:
                x, y = x.reshape(n, -1), y.reshape(n, -1)
                off = np.linalg.norm(x - y, axis=1) / np.linalg.norm(y, axis=1)
                assert (off > 2e-4).sum() <= max(1, n // 100), (layer, np.sort(off)[-5:])
            else:
                assert rel_l2(x, y) <= 2e-5, layer
    assert at == a.size == b.size


@pytest.mark.parametrize("n", [255, 257, 511, 704, 705])
def test_boundary_matches_oracle(gpu, oracle, n):
    """8 experts top-2, so that an expert's list spans several token tiles on both
    sides of the line (704 tokens), lists of more than 256 tokens among them."""
    hp = gpu.make_hparams(dim=512, heads=8, n_layers=4, attention_layers=(1, 3), kv=2, vocab=1000,
                          eos=1 << 30, n_expert=8, n_used=2, expert_ff=512, n_ff=1024, dense_lead=1)
    tensors = model_tensors(hp, gpu.synth_opts(0x9E3779B97F4A7C15, bias_sigma=0.1))
    prompt = ids(n, hp.vocab, n)
    g = gpu_engine(hp, tensors, ctx=768)
    o = oracle_engine(oracle, hp, tensors, ctx=768)
    lg, lo = g.forward(prompt, 0), o.forward(prompt, 0)
    e = rel_l2(lg, lo), rel_l2(state(g, n), np.frombuffer(o.snapshot(n), np.float32))
    print(f"T={n}: logits / state rel-L2 {e[0]:.2e} / {e[1]:.2e}")
    assert e[0] <= 1e-3 and e[1] <= 1e-3
    g.close()
    o.close()


@pytest.fixture(scope="module", params=[0, 1], ids=["narrow", "full_scales"])
def real(gpu, request):
    """Real widths, one layer of each kind, sub-block scales within [-32, 31] or over
    the whole int8 range (the two-part kernels)."""
    hp = gpu.make_hparams(dim=2048, heads=32, n_layers=4, attention_layers=(2,), kv=8, vocab=4096,
                          eos=1 << 30, n_expert=32, n_used=4, expert_ff=1792, n_ff=7168, dense_lead=1)
    e = gpu.GpuEngine.load_synthetic(hp, gpu.synth_opts(0x5EED, full_scales=request.param), ctx=1024)
    yield hp, e
    e.close()


@pytest.mark.parametrize("n", [129, 203, 416, 704, 705, 1000])
def test_real_width_whole_equals_chunks(real, n):
    """One call of n tokens against the same prompt in 64-token calls."""
    hp, e = real
    prompt = ids(n, hp.vocab, 7 * n)
    e.reset_session()
    lw = e.forward(prompt, 0)
    sw = state(e, n).copy()
    e.reset_session()
    for s in range(0, n, 64):
        e.forward_token(prompt[s:s + 64], s)
    lc, sc = e.snapshot_resident_logits(), state(e, n)
    assert rel_l2(lw, lc) <= 2e-5
    check_same(hp, n, sw, sc)


@pytest.mark.parametrize("n", [2, 33, 200, 257, 704, 750])
@pytest.mark.parametrize("sigma", [0.0, 4.0])
def test_expert_lists_of_any_length(gpu, oracle, n, sigma):
    """64 experts top-4: a spread of 4 in the selection bias sends every token to the
    same few experts (lists of n tokens beside empty ones), 0 spreads them; either way
    every list's tiles are found, on both sides of the line between the call sizes."""
    hp = gpu.make_hparams(dim=512, heads=8, n_layers=4, attention_layers=(1,), kv=2, vocab=1000,
                          eos=1 << 30, n_expert=64, n_used=4, expert_ff=256, n_ff=512, dense_lead=1)
    tensors = model_tensors(hp, gpu.synth_opts(0x2545F4914F6CDD1D, bias_sigma=sigma))
    prompt = ids(n, hp.vocab, n)
    g = gpu_engine(hp, tensors, ctx=768)
    o = oracle_engine(oracle, hp, tensors, ctx=768)
    g.set_route_log(True)
    lg, lo = g.forward(prompt, 0), o.forward(prompt, 0)
    counts = np.bincount(g.prefill_routes(1)[1].reshape(-1), minlength=64)
    assert counts.sum() == 4 * n and (sigma == 0.0 or counts.max() == n)
    assert rel_l2(lg, lo) <= 1e-3
    assert rel_l2(state(g, n), np.frombuffer(o.snapshot(n), np.float32)) <= 1e-3
    g.close()


@pytest.mark.parametrize("full_scales,h16", [(0, "1"), (0, "0"), (1, "1")])
@pytest.mark.parametrize("n", [129, 160, 161, 193, 225, 256])
def test_last_columns_of_large_calls(gpu, oracle, monkeypatch, n, full_scales, h16):
    """Large-call kernels (a model narrower than 512 runs them from 129 tokens) with 1, 32,
    33, 65, 97 and 128 columns in the last 128-token tile: each form of the last tile, and
    the experts' own list ends, for the binary16 copies, the Q6_K weights (bit for bit what
    the copies give) and the two-part weights."""
    monkeypatch.setenv("LFM_PREFILL_H16", h16)
    hp = gpu.make_hparams(dim=256, heads=4, n_layers=4, attention_layers=(1,), kv=2, vocab=1000,
                          eos=1 << 30, n_expert=8, n_used=4, expert_ff=256, n_ff=512, dense_lead=1)
    tensors = model_tensors(hp, gpu.synth_opts(0x9E3779B97F4A7C15, bias_sigma=0.1, full_scales=full_scales))
    prompt = ids(n, hp.vocab, n)
    g = gpu_engine(hp, tensors, ctx=256)
    o = oracle_engine(oracle, hp, tensors, ctx=256)
    lg, lo = g.forward(prompt, 0), o.forward(prompt, 0)
    sg = state(g, n)
    assert rel_l2(lg, lo) <= 1e-3
    assert rel_l2(sg, np.frombuffer(o.snapshot(n), np.float32)) <= 1e-3
    g.close()
    if h16 == "0":
        monkeypatch.setenv("LFM_PREFILL_H16", "1")
        g = gpu_engine(hp, tensors, ctx=256)
        assert g.h16_bytes() > 0
        assert g.forward(prompt, 0).tobytes() == lg.tobytes() and state(g, n).tobytes() == sg.tobytes()
        g.close()
