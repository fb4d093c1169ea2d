"""A step's inputs and outputs cross the link to the host in kernels of the step: steps of up to four tokens whose first kernel reads them in page-locked memory,
longer ones that take a copy, vocabularies that are no multiple of four, and records that change from step to step.

GGUF plans: bit for bit the token-by-token steps.  Layer-list plans: the float64 restatements (float32 sums of a few hundred terms: some 1e-6 of the logits'
root mean square; a token, its neighbour, a position or a wanted row read from the step before is an error of order one)."""
import dataclasses

import numpy as np
import pytest

import __graft_entry__ as ge
import test_noditar_gpu as N
import test_tutedra_gpu as T

pytestmark = pytest.mark.gpu
SIZES = [1, 3, 4, 5, 1, 4, 2, 6, 1]          # four tokens are read over the link, five take a copy


@pytest.mark.parametrize("weights", ["q8_0", "f16", "q4_0"])
def test_batched_steps_and_prompts(weights):
    from importlib import import_module
    pkg = ge.load_package()
    plans = import_module(ge.PKG_NAME + ".plan")
    cfg = dataclasses.replace(pkg.synth.CONFIGS["tiny-llama"], ctx=64)
    model = pkg.synth.make_numpy(cfg, seed=3, wtype={"f16": 1, "q4_0": 2, "q8_0": 8}[weights])
    one, many = plans.HipMasterPlan(model), plans.HipMasterPlan.initializeTornadoVMPlan(model, prefill_batch_size=8, n_seqs=8)
    toks = np.random.default_rng(1).integers(0, cfg.vocab, (8, sum(SIZES) + 2)).astype(np.int32)
    want = [[one.forward_decode(int(t), p) for p, t in enumerate(row)] for row in toks[:6]]
    pos = 0
    for c in SIZES:
        many.prefill(toks[0, pos:pos + c], pos)
        pos += c
    assert np.array_equal(many.forward_decode(int(toks[0, pos]), pos), want[0][pos])
    many.reset_kv()
    pos = np.zeros(6, int)
    for c in SIZES:
        at = np.arange(6)[::-1][:c]
        logits, ids = many.forward_decode_batch(toks[at, pos[at]], at, pos[at])
        for i, b in enumerate(at):
            assert np.array_equal(logits[i], want[b][pos[b]]) and ids[i] == want[b][pos[b]].argmax(), (c, b)
        pos[at] += 1
    one.reset_kv()
    assert [one.forward_decode_argmax(int(t), p) for p, t in enumerate(toks[0, :5])] == [int(w.argmax()) for w in want[0][:5]]
    one.freeTornadoExecutionPlan()
    many.freeTornadoExecutionPlan()


@pytest.mark.parametrize("vocab", [131, 132, 133, 134])
@pytest.mark.parametrize("design", ["noditar", "tutedra"])
def test_layer_list_portions(tmp_path, design, vocab):
    from importlib import import_module
    ge.load_package()
    hy = import_module(ge.PKG_NAME + ".hybrid")
    mod, layer = (N, N.ssm(heads=2, vdim=24, state=16, conv=3)) if design == "noditar" else (T, T.hgrn(heads=3, dim=19, vdim=20))          # (Tutedra: rows of token pairs)
    cfg, total = dict(mod.config([layer]), vocab=vocab), sum(SIZES)
    m = mod.Model(hy, tmp_path, cfg, 5)
    toks = [np.random.default_rng(s).integers(0, vocab, total).astype(np.int32) for s in range(2)]
    p = m.plan("float32", ctx=total + 8, max_batch=8, n_seqs=2)
    slots, got, pos = [p.acquire(), p.acquire()], [[], []], 0
    for c in SIZES:
        for i in range(2):
            got[i].append(p.step(slots[i], toks[i][pos:pos + c], pos, list(range(c - 1, -1, -2))[::-1]))
        pos += c
    p.close()
    rows = [a + k for a, c in zip(np.cumsum([0] + SIZES), SIZES) for k in list(range(c - 1, -1, -2))[::-1]]
    for i in range(2):
        assert N.err(np.concatenate(got[i]), m.ref(toks[i])[rows]) < 3e-5
