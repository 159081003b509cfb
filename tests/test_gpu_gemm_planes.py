"""lfm_q6k_gemm on the weight's row-major planes (up to 1024 tokens) and over its copies.

Each wave of the planes kernel decides by itself, per half block, whether its scales need
the two-part weights, so rows and blocks of every kind are mixed: scales within [-64, 64],
the edges -64, 64 and -65, the whole int8 range, super-block scales of zero and -0.0.
Against float64 per token: an error of 1e-5, the bar of the prefill GEMM."""
import numpy as np
import pytest

from test_gpu_kernels import blocks, encode_q6k

pytestmark = pytest.mark.gpu


def mixed_blocks(rows, nb, seed):
    rng = np.random.default_rng(seed)
    raw = blocks(rows * nb, seed, sc_lim=64).reshape(rows * nb, 210)
    kind = rng.integers(0, 6, rows * nb)
    sc = raw[:, 192:208].view(np.int8)
    sc[kind == 1] = rng.integers(-128, 128, (int((kind == 1).sum()), 16))
    sc[kind == 2, 5] = -65
    sc[kind == 3, 3] = 64
    raw[kind == 4, 208:210] = 0
    raw[kind == 5, 208:210] = np.frombuffer(np.float16(-0.0).tobytes(), np.uint8)
    return raw.reshape(-1)


@pytest.mark.parametrize("rows,in_dim", [(1, 256), (31, 512), (33, 8192), (128, 1792), (129, 2048), (700, 768)])
@pytest.mark.parametrize("T", [1, 2, 32, 33, 1024, 1025])
def test_matches_f64(gpu, oracle, rows, in_dim, T):
    raw = mixed_blocks(rows, in_dim // 256, rows + T)
    w64 = oracle.dequant_rows(raw, rows, in_dim).astype(np.float64).reshape(rows, in_dim)
    x = np.random.default_rng(T).standard_normal((T, in_dim)).astype(np.float32)
    x[0] *= 1000.0
    x[T // 2] *= 1e-20
    y = gpu.q6k_gemm(gpu.Q6Weight(raw, rows, in_dim), x)
    want = x.astype(np.float64) @ w64.T
    zero = ~w64.any(axis=1)
    assert not y[:, zero].any()
    if not zero.all():
        # relative to |W| |x| / sqrt(in_dim), what |want| is for random x: one row's dot
        # product alone may cancel (of 1025, the smallest is a thousandth of that)
        size = np.linalg.norm(w64) * np.linalg.norm(x.astype(np.float64), axis=1) / np.sqrt(in_dim)
        err = np.linalg.norm(y - want, axis=1) / size
        assert err.max() <= 1e-5, (int(err.argmax()), err.max())


@pytest.mark.parametrize("T", [1024, 1280])
@pytest.mark.parametrize("lo,hi", [(-128, 128), (-64, 65)])
def test_every_weight_bit_for_bit(gpu, lo, hi, T):
    """One-hot tokens pick every (scale, code) pair from the planes and from the copies."""
    rows, in_dim = 256, 256
    codes = (np.arange(in_dim)[None, :] + np.arange(rows)[:, None]) % 64
    scales = np.repeat((lo + np.arange(rows) % (hi - lo))[:, None], 16, axis=1)
    x = np.zeros((T, in_dim), dtype=np.float32)
    x[np.arange(T), np.arange(T) % in_dim] = 1.0
    y = gpu.q6k_gemm(gpu.Q6Weight(encode_q6k(codes, scales, np.ones(rows)).reshape(-1), rows, in_dim), x)
    want = (scales[:, np.arange(in_dim) // 16] * (codes - 32)).T.astype(np.float32)
    assert np.array_equal(y, want[np.arange(T) % in_dim])
