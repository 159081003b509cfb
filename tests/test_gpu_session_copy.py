"""Session snapshot and restore against the library's own binary16 conversions.

The bytes are whole numbers here: every float of a restored state must come back as
f16(f32) for K and V and unchanged for the conv state, bit for bit, for any bit pattern
(NaN, infinities, subnormals), and positions past the restored ones must keep theirs.
"""
import numpy as np
import pytest

from model_util import gpu_engine, model_tensors, small_hparams

import lfm_hip

pytestmark = pytest.mark.gpu

CTX = 1600


@pytest.fixture(scope="module")
def engine(gpu):
    hp = small_hparams(dim=512, heads=8, kinds=("conv", "attn", "conv", "attn"), kv=8, vocab=300)
    hp.kv_heads[3] = 2
    e = gpu_engine(hp, model_tensors(hp), ctx=CTX)
    yield hp, e
    e.close()


def through_f16(bits):
    """f32 -> binary16 -> f32 of each bit pattern, by the library's host conversions."""
    f = bits.view(np.float32)
    with np.errstate(over="ignore", invalid="ignore"):
        h = f.astype(np.float16).view(np.uint16)
    nan = np.isnan(f)
    h[nan] = [lfm_hip.lib().lfm_f32_to_f16(float(x)) for x in f[nan]] if nan.sum() < 2000 else h[nan]
    e = h & 0x7C00
    out = h.view(np.float16).astype(np.float32).view(np.uint32)
    special = e == 0x7C00
    out[special] = ((h[special].astype(np.uint32) & 0x8000) << 16) | 0x7F800000 \
        | ((h[special].astype(np.uint32) & 0x3FF) << 13)
    return out


def layers(hp, valid):
    at = 0
    for layer in range(hp.n_layers):
        kv = hp.kv_heads[layer]
        n = 2 * valid * kv * 64 if kv else 2 * hp.dim
        yield kv, at, at + n
        at += n


# a short chunk, the chunk edge on either side of 1 MB, several chunks
@pytest.mark.parametrize("valid", [0, 1, 77, 203, 204, 1599, CTX])
def test_round_trip_bits(engine, valid):
    hp, e = engine
    n = e.snapshot_bytes(valid) // 4
    r = np.random.default_rng(valid)
    bits = r.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    tame = r.random(n) < 0.9  # mostly finite values of binary16's range, its edges among them
    f = (r.standard_normal(n) * 2.0 ** r.integers(-26, 17, n)).astype(np.float32)
    bits = np.where(tame, f.view(np.uint32), bits)
    bits = np.where(np.isnan(bits.view(np.float32)) & (r.random(n) < 0.9), np.uint32(0x7FC00000), bits)
    nan = np.flatnonzero(np.isnan(bits.view(np.float32)))
    bits[nan[1500:]] = 0x7F800000
    e.restore_session(valid, bits.tobytes())
    got = np.frombuffer(e.snapshot_resident_cache(valid), np.uint32)
    assert got.size == n
    for kv, a, b in layers(hp, valid):
        want = through_f16(bits[a:b]) if kv else bits[a:b]
        assert np.array_equal(got[a:b], want), (kv, np.flatnonzero(got[a:b] != want)[:5])


def test_positions_past_the_restored_ones_are_kept(engine):
    hp, e = engine
    r = np.random.default_rng(5)
    full = r.standard_normal(e.snapshot_bytes(CTX) // 4).astype(np.float16).astype(np.float32)
    e.restore_session(CTX, full.tobytes())
    part = r.standard_normal(e.snapshot_bytes(100) // 4).astype(np.float16).astype(np.float32)
    e.restore_session(100, part.tobytes())
    got = np.frombuffer(e.snapshot_resident_cache(CTX), np.float32)
    for (kv, a, b), (_, c, d) in zip(layers(hp, CTX), layers(hp, 100)):
        if not kv:
            assert np.array_equal(got[a:b], part[c:d])
            continue
        g, f, p = got[a:b].reshape(2, CTX, -1), full[a:b].reshape(2, CTX, -1), part[c:d].reshape(2, 100, -1)
        assert np.array_equal(g[:, :100], p) and np.array_equal(g[:, 100:], f[:, 100:])


def test_large_snapshot_in_threads(gpu):
    """More than 32 MB: four threads, the last chunk short and not every thread's."""
    hp = small_hparams(dim=512, heads=8, kinds=("attn",) * 6, kv=8, vocab=300)
    e = gpu_engine(hp, model_tensors(hp), ctx=CTX)
    for valid in (1400, 1597):
        full = np.random.default_rng(valid).standard_normal(e.snapshot_bytes(valid) // 4, dtype=np.float32)
        full = full.astype(np.float16).astype(np.float32)
        assert full.nbytes > 32 << 20
        e.restore_session(valid, full.tobytes())
        assert np.array_equal(np.frombuffer(e.snapshot_resident_cache(valid), np.float32), full)
    e.close()
