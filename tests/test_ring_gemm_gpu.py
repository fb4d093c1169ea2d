"""The layer-list family's ring GEMM (csrc/gl3_hy_gemm.h) at the edges of its tiles, through plans of one attention layer: the head's product
(vocabulary rows), the fused projection, the gate / up product (activation in the epilogue) and the K-split output and down products, with row
counts around 32, 64, 128 and 256, column counts that leave remainders in every tile size, and K of fewer stages than the rings hold.  The last case's
width is no multiple of a stage and stays with the other kernel.

Yardstick: tests/noditar_ref.py in float64.  Bound: float32 products of K terms and the sums behind them err by a few 1e-6 of the logits'
root mean square, bfloat16 plans by 2^-9 per rounded operand over the products on a path, some 1e-2; an element that is read or written
in the wrong place is an error of order one."""
import numpy as np
import pytest

import __graft_entry__ as ge
import noditar_ref as R
import test_kugadra_gpu as U
from test_noditar_gpu import Model, att, config, err, tokens_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hy():
    from importlib import import_module
    ge.load_package()
    return import_module(ge.PKG_NAME + ".hybrid")


# (tokens, width, vocabulary, feed-forward): tiles of the head's product bf16 / f32 behind each
CASES = [(9, 64, 211, 96), (33, 192, 1003, 160), (64, 128, 20001, 64), (65, 128, 20003, 288), (129, 128, 20005, 416), (130, 64, 29999, 96),
         (257, 128, 20007, 7008), (300, 64, 30001, 15008), (255, 704, 451, 608), (191, 1024, 333, 1056), (256, 128, 33001, 64), (70, 104, 515, 72),
         (65, 128, 451, 8208), (300, 192, 333, 16392), (300, 192, 21856, 64), (300, 128, 24592, 64), (300, 64, 32840, 64), (129, 192, 21763, 64), (129, 192, 20485, 64),
         (5, 1024, 333, 9024), (8, 704, 12001, 608), (6, 1024, 12003, 9056)]          # 5 to 8 tokens: where the tiles cost less than the dot products


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,width,vocab,ff", CASES)
def test_tiles_and_remainders(hy, tmp_path, n, width, vocab, ff, dtype):
    cfg = config([att(heads=4, kv_heads=2, dim=16, vdim=24, ff=ff)], width=width, vocab=vocab, streams=1)
    m = Model(hy, tmp_path, cfg, seed=n)
    toks = tokens_for(cfg, n)
    p = m.plan(dtype, ctx=n + 8, max_batch=320)
    s = p.acquire()
    got = p.step(s, toks, 0, list(range(n)))
    p.close()
    want = m.ref(toks)
    assert err(got, want) < (2e-5 if dtype == "float32" else 3e-2)
    # every entry, not only the rows' norms: one wrong element of a row of 30000 disappears in its norm
    assert np.abs(got - want).max() < (2e-4 if dtype == "float32" else 2.5e-1) * np.sqrt((want ** 2).mean())


# the up product of a feed-forward without a gate (squared ReLU in the epilogue): (tokens, width, feed-forward)
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,width,ff", [(33, 192, 160), (65, 128, 8328), (65, 192, 8208), (129, 64, 16488), (300, 192, 28976), (33, 64, 32800)])
def test_up_product_without_a_gate(hy, tmp_path, n, width, ff, dtype):
    m = U.Model(hy, tmp_path, U.config([U.lig(heads=2, dim=16, vdim=16, mlp=U.dense(ff))], width=width), seed=n)
    toks, want = m.tokens(n)
    p = m.plan(dtype, ctx=n + 8, max_batch=320)
    got = U.whole(p, toks)
    p.close()
    assert err(got, want) < (2e-5 if dtype == "float32" else 3e-2)
