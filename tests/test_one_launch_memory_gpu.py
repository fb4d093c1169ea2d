"""Matrix memories of one token in one launch (csrc/gl3_hy_one_kernels.h, hy_scan_out and hy_pair_one) where a head's columns take several passes, at the edges of a pass and of the
gate, and beside an attention in every pairing of head size and states.  Each case says whether the gate admits it, so none can pass on the other kernels unnoticed.

Yardstick: the float64 restatement.  Bound: float32 sums of a few hundred terms err by some 1e-6 of the logits' root mean square, 3e-5 for whole models as in the other single-step
tests (bfloat16 plans round every product's input: 6e-2; an mLSTM divides by a sum that may come near zero, which leaves rounded inputs without a bound: float32 alone); a
lost row, column or pass is an error of order one."""
import os
import re

import numpy as np
import pytest

import __graft_entry__ as ge
import test_kosusun_gpu as K

pytestmark = pytest.mark.gpu


def par(dim, right):
    return K.par(left=K.attn(heads=4, kv_heads=2, dim=dim, vdim=dim, size=200, pool=0, rot_dims=16), right=right, ff=0)


# layer, states, columns, columns a pass, taken by the one launch
CASES = {
    "mlstm_64x600": (K.mls(heads=2, dim=64, vdim=599, ff=0), 64, 600, 256, True), "mlstm_40x257": (K.mls(heads=3, dim=40, vdim=256, ff=0), 40, 257, 256, True),
    "mlstm_40x256": (K.mls(heads=2, dim=40, vdim=255, ff=0), 40, 256, 256, True), "mlstm_16x1024": (K.mls(heads=2, dim=16, vdim=1023, ff=0), 16, 1024, 256, True),
    "mlstm_80x500": (K.mls(heads=2, dim=80, vdim=499, ff=0), 80, 500, 384, True), "mlstm_100x385": (K.mls(heads=2, dim=100, vdim=384, ff=0), 100, 385, 384, True),
    "mlstm_129x300": (K.mls(heads=2, dim=129, vdim=299, ff=0), 129, 300, 192, True), "mlstm_200x193": (K.mls(heads=2, dim=200, vdim=192, ff=0), 200, 193, 192, True),
    "mlstm_256x160": (K.mls(heads=2, dim=256, vdim=159, ff=0), 256, 160, 192, True), "mlstm_256x161": (K.mls(heads=2, dim=256, vdim=160, ff=0), 256, 161, 192, False),
    "retention_64x600": (par(132, K.ret(heads=2, dim=64, vdim=600)), 64, 600, 256, True), "retention_129x300": (par(64, K.ret(heads=2, dim=129, vdim=300)), 129, 300, 192, True),
    "pair_64_64x600": (par(64, K.ret(heads=2, dim=64, vdim=600)), 64, 600, 256, True), "pair_64_80x500": (par(64, K.ret(heads=3, dim=80, vdim=500)), 80, 500, 384, True),
    "pair_128_40x257": (par(128, K.ret(heads=2, dim=40, vdim=257)), 40, 257, 256, True), "pair_128_128x256": (par(128, K.ret(heads=2, dim=128, vdim=256)), 128, 256, 384, True),
    "pair_72_100x400": (par(72, K.ret(heads=2, dim=100, vdim=400)), 100, 400, 384, True),
}


def gate():
    with open(os.path.join(ge.PKG_DIR, "csrc", "gl3_hy_one_kernels.h")) as f:
        text = f.read()
    return [eval(re.search(r"constexpr int %s = ([0-9 *]+);" % name, text).group(1)) for name in ("HY_SCAN_OUT", "HY_SCAN_OUT_P")]


@pytest.mark.parametrize("name,dtype", [(n, d) for n in CASES for d in (["float32"] if n.startswith("mlstm") else ["float32", "bfloat16"])])
def test_tokens_one_by_one(tmp_path, name, dtype):
    from importlib import import_module
    ge.load_package()
    hy = import_module(ge.PKG_NAME + ".hybrid")
    layer, states, columns, per_pass, taken = CASES[name]
    elements, widest = gate()
    assert taken == (states <= 256 and columns <= widest and states * columns <= elements) and per_pass == (256 if states <= 64 else 384 if states <= 128 else 192)
    cfg = K.config([layer])
    m = K.Model(hy, tmp_path, cfg, 5)
    sizes = [1] * 8 + [9, 1, 1] + [1] * 12
    total = sum(sizes)
    toks = [np.random.default_rng(i).integers(0, cfg["vocab"], total).astype(np.int32) for i in range(2)]
    p = m.plan(dtype, ctx=total + 8, max_batch=32, n_seqs=2)
    slots, got, pos = [p.acquire(), p.acquire()], [[], []], 0
    for c in sizes:
        for i in range(2):
            got[i].append(p.step(slots[i], toks[i][pos:pos + c], pos, list(range(c))))
        pos += c
    p.close()
    for i in range(2):
        assert K.err(np.concatenate(got[i]), m.ref(toks[i])) < (3e-5 if dtype == "float32" else 6e-2)
