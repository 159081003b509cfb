"""What calls return through pinned host memory: logits, decode tokens, and the ids and
the state that a call starts with."""
import numpy as np
import pytest

from conftest import rel_l2
from model_util import gpu_engine, model_tensors, oracle_engine, small_hparams

pytestmark = pytest.mark.gpu


# vocabularies around the 16-byte units and the 1024 words of a workgroup
@pytest.mark.parametrize("vocab", [66, 301, 1023, 1024, 4097])
def test_logits_reach_the_host(gpu, oracle, vocab):
    """Forward calls on each way the ids travel (1: state only, up to 64 in the launch's
    arguments, more in host memory) against the oracle (logits rel-L2 <= 1e-3, the bar
    of the model tests); the returned logits are the resident ones bit for bit."""
    hp = small_hparams(vocab=vocab)
    tensors = model_tensors(hp)
    g, o = gpu_engine(hp, tensors, ctx=256), oracle_engine(oracle, hp, tensors, ctx=256)
    rng = np.random.default_rng(vocab)
    at = 0
    for n in (65, 1, 64, 2):
        ids = rng.integers(0, vocab, n)
        got, want = g.forward(ids, at), o.forward(ids, at)
        assert got.size == vocab and rel_l2(got, want) <= 1e-3
        assert np.array_equal(got, g.snapshot_resident_logits())
        at += n
    # a decode run's tokens and logits, then the same greedy steps one call at a time
    first = int(np.argmax(got))
    cache = g.snapshot_resident_cache(at)
    run = g.decode_run(first, at, 9)
    last = g.snapshot_resident_logits()
    g.restore_session(at, cache)
    token, steps = first, []
    for s in range(9):
        lg = g.forward([token], at + s)
        token = int(np.argmax(lg))
        steps.append(token)
    assert run == steps and np.array_equal(last, lg)
    g.close()


def test_reset_clears_every_conv_state(gpu):
    hp = small_hparams(kinds=("conv", "attn", "conv", "conv"))
    g = gpu_engine(hp, model_tensors(hp), ctx=64)
    first = g.forward([3, 5, 7], 0)
    g.forward([11, 13], 3)
    g.reset_session()
    assert np.frombuffer(g.snapshot_resident_cache(0), np.float32).size == 3 * 2 * hp.dim
    assert not np.frombuffer(g.snapshot_resident_cache(0), np.float32).any()
    assert np.array_equal(g.forward([3, 5, 7], 0), first)
    g.close()
