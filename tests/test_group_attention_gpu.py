"""Static-batched decode where a workgroup serves a group of query heads (attn_head_kernel on 512 threads): head sizes 32, 64, 96 and 128, groups of 2 to 8 heads,
positions around whole quads, wavefronts and the launch's last one (127); and the norm in front of the products at the widest row that stays in registers (5120), beyond it, and where the last quad
of a thread is missing.  Yardstick: the CPU oracle, bit for bit."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGES = (0, 1, 3, 4, 31, 62, 63, 64, 65, 125, 126, 127)


def check(base, positions, **sizes):
    from importlib import import_module
    import __graft_entry__ as ge
    from oracle import oracle_c
    pkg = ge.load_package()
    plans = import_module(ge.PKG_NAME + ".plan")
    model = pkg.synth.make_numpy(dataclasses.replace(pkg.synth.CONFIGS[base], ctx=136, **sizes), seed=5)
    toks = np.random.default_rng(sizes["dim"]).integers(0, model.cfg.vocab, max(positions) + 1)
    oracle, want = oracle_c.COracle(model), {}
    for i, t in enumerate(toks):
        row = oracle.forward(int(t), i)
        if i in positions:
            want[i] = row.copy()
    n = len(positions)
    plan = plans.HipMasterPlan.initializeTornadoVMPlan(model, prefill_batch_size=64, n_seqs=n)
    for s, p in enumerate(positions):
        if p:
            plan.prefill_seq(s, toks[:p], 0)
    logits, ids = plan.forward_decode_batch(np.array([toks[p] for p in positions]), np.arange(n), np.array(positions))
    for s, p in enumerate(positions):
        assert np.array_equal(logits[s], want[p]), p
        assert ids[s] == want[p].argmax(), p
    plan.freeTornadoExecutionPlan()


@pytest.mark.parametrize("base,heads,kv,hs", [("tiny-llama", 8, 2, 32), ("tiny-llama", 6, 3, 64), ("tiny-llama", 8, 1, 64), ("tiny-llama", 4, 1, 128), ("tiny-llama", 6, 1, 96), ("tiny-qwen3", 8, 2, 128)])
def test_groups(base, heads, kv, hs):
    check(base, EDGES, n_heads=heads, n_kv_heads=kv, head_size=hs, dim=heads * hs)


@pytest.mark.parametrize("dim", [1056, 5088, 5120, 5152])
def test_rows(dim):
    check("tiny-qwen3", (0, 5), n_heads=4, n_kv_heads=1, head_size=64, dim=dim)
