"""Attention of one token behind fewer than 128 positions (attn_head_kernel) at head sizes of 32 and 96.  Their bits are held by test_gpu_decode.py and test_group_attention_gpu.py; here they may not
take longer than the next larger size, whose chains, rows and reads are longer.  A loop over the head that waits for every read it makes took 1.13 - 1.45 times as long (32: 6.3 - 9.0 us beside 5.6 - 7.3
of 64, 96: 7.9 - 12.5 beside 6.1 - 8.6 of 128).  Bound: 1.1, for the spread of the smallest of seven averages (1 %) and the clock."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def attention_us(hs, positions):
    from importlib import import_module
    import __graft_entry__ as ge
    pkg = ge.load_package()
    plans = import_module(ge.PKG_NAME + ".plan")
    model = pkg.synth.make_numpy(dataclasses.replace(pkg.synth.CONFIGS["tiny-llama"], ctx=136, n_heads=32, n_kv_heads=32, head_size=hs, dim=32 * hs, n_layers=4), seed=5)
    plan = plans.HipMasterPlan.initializeTornadoVMPlan(model, prefill_batch_size=128)
    toks = np.random.default_rng(hs).integers(0, model.cfg.vocab, 128)
    plan.prefill_seq(0, toks, 0)
    out = []
    for p in positions:
        plan.forward_decode(int(toks[p]), p)
        out.append(min(plan.profile_kernel("attention", 40)["avg_us"] for _ in range(7)))
    plan.freeTornadoExecutionPlan()
    return out


@pytest.mark.parametrize("hs,next_size", [(32, 64), (96, 128)])
def test_no_slower_than_the_next_larger_head(hs, next_size):
    positions = (20, 60, 126)
    for p, us, longer in zip(positions, attention_us(hs, positions), attention_us(next_size, positions)):
        print("head of %d behind %d: %.2f us, of %d %.2f" % (hs, p, us, next_size, longer))
        assert us < 1.1 * longer, (p, us, longer)
