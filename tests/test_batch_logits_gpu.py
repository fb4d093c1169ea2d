"""Logits of a static-batched decode step on their way to the caller: in one pinned piece, in several, in more than are in flight at once, with a last
piece of odd length, into memory that was never touched and into memory that was.  Every row is the single-sequence step's, bit for bit
(position 0: a row depends on its token alone)."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,n", [(512, 1), (33008, 31), (33008, 32), (50000, 43), (70000, 64)])
def test_every_row_arrives(vocab, n):
    from importlib import import_module
    import __graft_entry__ as ge
    pkg = ge.load_package()
    plans = import_module(ge.PKG_NAME + ".plan")
    cfg = dataclasses.replace(pkg.synth.CONFIGS["tiny-llama"], vocab=vocab)
    plan = plans.HipMasterPlan.initializeTornadoVMPlan(pkg.synth.make_numpy(cfg, seed=3), prefill_batch_size=64, n_seqs=64)
    rng = np.random.default_rng(n)
    for _ in range(2):
        toks = rng.integers(0, vocab, n)
        logits, ids = plan.forward_decode_batch(toks, np.arange(n), np.zeros(n))
        only, ids2 = plan.forward_decode_batch(toks, np.arange(n), np.zeros(n), want_logits=False)
        assert only is None and np.array_equal(ids, ids2)
        for i in (range(n) if n < 5 else (0, 1, n // 3, n // 2, n - 2, n - 1)):
            row = plan.forward_decode(int(toks[i]), 0)
            assert np.array_equal(logits[i], row) and ids[i] == row.argmax(), i
        assert np.array_equal(logits.argmax(axis=1), ids)
    plan.freeTornadoExecutionPlan()


@pytest.mark.parametrize("vocab,n", [(4096, 64), (4112, 64), (4096, 33), (8192, 63), (8224, 64), (12288, 64), (12304, 64)])
def test_around_whole_pieces(vocab, n):
    """Steps whose logits end at, in front of or behind one, two and three pieces of 1 MB; destinations that do not start on a page."""
    from importlib import import_module
    import __graft_entry__ as ge
    pkg = ge.load_package()
    plans, hip = import_module(ge.PKG_NAME + ".plan"), import_module(ge.PKG_NAME + ".hip")
    cfg = dataclasses.replace(pkg.synth.CONFIGS["tiny-llama"], vocab=vocab)
    plan = plans.HipMasterPlan.initializeTornadoVMPlan(pkg.synth.make_numpy(cfg, seed=3), prefill_batch_size=64, n_seqs=64)
    rng = np.random.default_rng(n)
    t, s, p, ids = rng.integers(0, vocab, n).astype(np.int32), np.arange(n, dtype=np.int32), np.zeros(n, np.int32), np.empty(n, np.int32)
    want = np.stack([plan.forward_decode(int(x), 0) for x in t])
    for off in (0, 1, 1023):
        mem = np.full(n * vocab + 2048, 7.0, np.float32)
        out = mem[off:off + n * vocab]
        hip.check(hip.lib().gl3_forward_decode_batch(plan._ctx, plans._p(t), plans._p(s), plans._p(p), n, plans._p(out), plans._p(ids)), plan._ctx)
        assert np.array_equal(out.reshape(n, vocab), want) and np.array_equal(ids, want.argmax(axis=1))
        assert (mem[:off] == 7).all() and (mem[off + n * vocab:] == 7).all()
    plan.freeTornadoExecutionPlan()


def test_page_locked_destination():
    """The caller's page-locked memory is written by the device itself: 64 x 70000 floats arrive in well under the time that a copy through the plan's own takes."""
    import time
    from importlib import import_module
    import __graft_entry__ as ge
    import torch
    pkg = ge.load_package()
    plans, hip = import_module(ge.PKG_NAME + ".plan"), import_module(ge.PKG_NAME + ".hip")
    vocab, n = 70000, 64
    plan = plans.HipMasterPlan.initializeTornadoVMPlan(pkg.synth.make_numpy(dataclasses.replace(pkg.synth.CONFIGS["tiny-llama"], vocab=vocab), seed=3), prefill_batch_size=64, n_seqs=64)
    t, s, p, ids = np.arange(n, dtype=np.int32), np.arange(n, dtype=np.int32), np.zeros(n, np.int32), np.empty(n, np.int32)
    plain, locked = np.zeros((n, vocab), np.float32), torch.zeros((n, vocab), pin_memory=True).numpy()

    def best(out):
        times = []
        for _ in range(12):
            a = time.perf_counter()
            hip.check(hip.lib().gl3_forward_decode_batch(plan._ctx, plans._p(t), plans._p(s), plans._p(p), n, plans._p(out), plans._p(ids)), plan._ctx)
            times.append(time.perf_counter() - a)
        return min(times)
    through, direct = best(plain), best(locked)
    assert np.array_equal(plain, locked) and np.array_equal(plain[5], plan.forward_decode(5, 0))
    assert direct < 0.85 * through, (direct, through)
    plan.freeTornadoExecutionPlan()
