"""The small-batch Q8_0 GEMM (csrc/gl3_bd_gemm.h), whose scale products come from the matrix cores, against the token-by-token steps bit for bit: rows of blocks that fill the last tile of
four to every degree, one to 64 tokens around the tiles of 16 and 32, and weight scales that are zero, subnormal, the smallest normal and large in 16 bits."""
import dataclasses

import numpy as np
import pytest

import __graft_entry__ as ge

pytestmark = pytest.mark.gpu
ODD = np.array([0x0000, 0x8000, 0x0001, 0x03FF, 0x0400, 0x2E66, 0x3C00, 0xBC00], np.uint16)          # 0, -0, 2^-24, the largest subnormal, 2^-14, 0.1, 1, -1


@pytest.mark.parametrize("dim,hidden", [(256, 512), (288, 544), (320, 576), (352, 608)])
def test_batched_steps_are_the_single_steps(dim, hidden):
    from importlib import import_module
    pkg = ge.load_package()
    plans = import_module(ge.PKG_NAME + ".plan")
    cfg = dataclasses.replace(pkg.synth.CONFIGS["tiny-llama"], dim=dim, hidden=hidden, n_heads=dim // 32, n_kv_heads=dim // 32, vocab=544, ctx=16)
    model = pkg.synth.make_numpy(cfg, seed=dim)
    rng = np.random.default_rng(dim)
    for name, (raw, ty, rows, cols) in model.tensors.items():
        if ty == pkg.synth.GGML_Q8_0:
            blocks = raw.reshape(-1, 34)
            at = rng.choice(len(blocks), len(blocks) // 8, replace=False)
            blocks[at, :2] = rng.choice(ODD, len(at)).view(np.uint8).reshape(-1, 2)
    one, many = plans.HipMasterPlan(model), plans.HipMasterPlan.initializeTornadoVMPlan(model, prefill_batch_size=64, n_seqs=64)
    toks = rng.integers(0, cfg.vocab, (2, 64)).astype(np.int32)
    want = []
    for b in range(64):
        one.forward_decode(int(toks[0, b]), 0)
        want.append(one.forward_decode(int(toks[1, b]), 1).copy())
    assert np.isfinite(want).all() and len({w.tobytes() for w in want}) > 60
    for n in (1, 2, 15, 16, 17, 31, 32, 33, 48, 64):
        at = rng.permutation(64)[:n]
        many.forward_decode_batch(toks[0, at], at, np.zeros(n, int))
        logits, _ = many.forward_decode_batch(toks[1, at], at, np.ones(n, int))
        for i, b in enumerate(at):
            assert np.array_equal(logits[i], want[b]), (n, b)
    one.freeTornadoExecutionPlan()
    many.freeTornadoExecutionPlan()
