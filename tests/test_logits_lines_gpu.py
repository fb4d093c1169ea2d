"""Logits of a single step on either side of the lines between a kernel behind the head and results that the head's kernel writes to the host itself (logits_leave, csrc/gl3_api.hip): 65536 rows, and per
weight type the columns from which more rows leave too.  Steps that hand logits out, keep them on the device (greedy id) and hand them out again take turns on one captured step.  Yardstick: the CPU
oracle, bit for bit."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F16, Q4_0, Q8_0 = 1, 2, 8


@pytest.mark.parametrize("wtype,dim,vocab", [(Q8_0, 256, 65536), (Q8_0, 256, 65552), (Q8_0, 2528, 65552), (Q8_0, 2560, 65552), (Q4_0, 256, 65536), (Q4_0, 256, 65552), (Q4_0, 2048, 65552),
                                             (F16, 256, 65552), (F16, 1024, 65552)])
def test_steps_take_turns(wtype, dim, vocab):
    from importlib import import_module
    import __graft_entry__ as ge
    from oracle import oracle_c
    pkg = ge.load_package()
    plans = import_module(ge.PKG_NAME + ".plan")
    cfg = dataclasses.replace(pkg.synth.CONFIGS["tiny-qwen3"], dim=dim, hidden=256, n_layers=1, n_heads=8, n_kv_heads=2, head_size=32, vocab=vocab, ctx=16)
    model = pkg.synth.make_numpy(cfg, wtype=wtype, seed=11)
    plan = plans.HipMasterPlan(model)
    oracle = oracle_c.COracle(model, vector_bits=0 if wtype == Q8_0 else 256)
    toks = np.random.default_rng(dim).integers(0, vocab, 6)
    for pos, t in enumerate(toks):
        want = oracle.forward(int(t), pos)
        if pos % 3 == 1:
            assert plan.forward_decode_argmax(int(t), pos) == want.argmax()
        else:
            assert np.array_equal(plan.tornadoVMForwardDecode(int(t), pos), want), pos
    plan.freeTornadoExecutionPlan()
