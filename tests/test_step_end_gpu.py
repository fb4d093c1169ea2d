"""The end of a step: results are whole when the call returns, whatever stands behind them on the stream; steps with logits and with the greedy id alternate, vocabularies
take one workgroup of the kernel that hands logits out, several and more than it has, and prompts of several portions hand their records on in turn."""
import dataclasses

import numpy as np
import pytest

import __graft_entry__ as ge
import test_noditar_gpu as N

pytestmark = pytest.mark.gpu


def mods():
    from importlib import import_module
    pkg = ge.load_package()
    return pkg, import_module(ge.PKG_NAME + ".plan"), import_module(ge.PKG_NAME + ".hybrid")


@pytest.mark.parametrize("vocab", [16, 1024, 1040, 262208])
def test_logits_and_ids_of_single_steps(vocab):
    pkg, plans, _ = mods()
    cfg = dataclasses.replace(pkg.synth.CONFIGS["tiny-llama"], vocab=vocab, n_layers=1, ctx=80)
    plan = plans.HipMasterPlan(pkg.synth.make_numpy(cfg, seed=3))
    toks = np.random.default_rng(0).integers(0, vocab, 60)
    first = [plan.forward_decode(int(t), i).copy() for i, t in enumerate(toks)]
    for i, t in enumerate(toks):          # a result read too early would show the step before
        if i % 3 == 0:
            assert np.array_equal(plan.forward_decode(int(t), i), first[i])
        else:
            assert plan.forward_decode_argmax(int(t), i) == int(np.argmax(first[i]))
    plan.freeTornadoExecutionPlan()


@pytest.mark.parametrize("batch", [3, 4, 5, 16])
def test_portions_in_turn(tmp_path, batch):
    """Portions of up to four tokens are read from page-locked memory by their first kernel, longer ones are copied; every want of a call, in the first, a middle and the last portion."""
    _, _, hybrid = mods()
    cfg = N.config([N.att(heads=2, kv_heads=1, dim=8, vdim=8), N.ssm(heads=2, vdim=8, state=8)])
    m = N.Model(hybrid, tmp_path, cfg, 4)
    toks = N.tokens_for(cfg, 61)
    want = m.ref(toks)
    p = m.plan("float32", ctx=80, max_batch=batch)
    s = p.acquire()
    for rows in ([60], [0, 60], [30], []):
        got = p.step(s, toks, 0, rows)
        if rows:
            assert N.err(got, want[rows]) < 3e-5
        assert N.err(p.step(s, toks[:1], 0, [0]), want[:1]) < 3e-5
    p.close()
