"""One wanted row of a layer-list step: the head's kernel writes it to page-locked memory itself, two rows take a copy behind it.  Vocabularies that end in a lone row, leave workgroups without rows
or stand beside 16384 rows, where a pair of rows has four wavefronts or one; one token (the product that makes its own norm) and the end of a prompt.
Yardsticks: the same row among two wanted ones (the same normed row and weights: float32 sums of 72 or 2048 terms in another order, some 1e-6 of the logits' root mean square, in both types), the token
as the last row of the prompt with it (bfloat16: rows that the kernels for one and for many tokens round apart now and then, 2^-9 of an operand) and the float64 restatement."""
import numpy as np
import pytest

import __graft_entry__ as ge
import test_noditar_gpu as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width,vocab", [(72, 3), (72, 515), (2048, 513), (2048, 16383), (2048, 16387)])
def test_one_row_and_two(tmp_path, width, vocab, dtype):
    from importlib import import_module
    ge.load_package()
    hy = import_module(ge.PKG_NAME + ".hybrid")
    cfg = N.config([N.att(heads=4, kv_heads=2, dim=16, vdim=16, ff=72)], width=width, vocab=vocab, streams=2)
    m = N.Model(hy, tmp_path, cfg, seed=3)
    plan = m.plan(dtype, ctx=32, max_batch=16)
    toks = np.random.default_rng(vocab).integers(0, vocab, 9).astype(np.int32)
    s = plan.acquire()
    two = plan.step(s, toks[:8], 0, want=[6, 7])
    one = plan.step(s, toks[:8], 0, want=[7])
    token = plan.step(s, toks[8:], 8, want=[0])
    last = plan.step(s, toks, 0, want=[7, 8])
    plan.close()
    want = m.ref(toks)

    def off(got, ref):
        d = got.astype(np.float64) - ref
        return np.sqrt((d ** 2).mean() / (ref.astype(np.float64) ** 2).mean())
    f32 = dtype == "float32"
    print("one/two %.2e token/last %.2e one/exact %.2e token/exact %.2e" % (off(one[0], two[1]), off(token[0], last[1]), off(one[0], want[7]), off(token[0], want[8])))
    assert off(one[0], two[1]) < 4e-6
    assert off(token[0], last[1]) < (4e-6 if f32 else 1e-2)
    assert off(one[0], want[7]) < (2e-5 if f32 else 2e-2) and off(token[0], want[8]) < (2e-5 if f32 else 2e-2)
