"""Launches of one token that share one (csrc/gl3_hy_beside_kernels.h) at the edges of their rules: mixers with and without a one-launch form beside the gate / up rows, head and
state sizes on either side of a kernel's, K on either side of the split over wavefronts, output and down projections that split alike and not, odd row counts, a choice of experts over one
and several rows per lane, positions that leave the one-launch form.  Two sequences alternate, so a state written to the wrong slot shows.

Yardstick: the designs' float64 restatements.  Bound: float32 sums of a few hundred to a thousand terms err by some 1e-6 of the logits' root mean square (3e-5 holds for the launches apart); a lost
row, expert or part is an error of order one.  bfloat16 plans round every product's input, and what a design makes of that (a normaliser near zero, a choice of experts that flips) differs from model to
model: the same tokens in portions of 16, which the kernels for many tokens make with the same roundings, say how much, and sums in another order move some of them by one place: twice as much, and at
least the design's own bound."""
import numpy as np
import pytest

import __graft_entry__ as ge
import test_kosusun_gpu as K
import test_kugadra_gpu as U
import test_noditar_gpu as N

pytestmark = pytest.mark.gpu
SIZES = [1, 1, 3, 1, 1, 9, 1, 1, 2, 1]


@pytest.fixture(scope="module")
def hy():
    from importlib import import_module
    ge.load_package()
    return import_module(ge.PKG_NAME + ".hybrid")


A, R = K.attn, K.ret
CASES = {
    "pair_64_64": (K, [K.par(left=A(dim=64, vdim=64), right=R(heads=3, dim=64, vdim=66), ff=70)], {}),
    "pair_128_128": (K, [K.par(left=A(heads=2, kv_heads=1, dim=128, vdim=72), right=R(heads=2, dim=128, vdim=130), ff=33)], {}),
    "pair_64_128": (K, [K.par(left=A(dim=40, vdim=64), right=R(heads=1, dim=100, vdim=31), ff=32)], {}),
    "pair_heads_of_200": (K, [K.par(left=A(heads=2, kv_heads=1, dim=200, vdim=24, rot_dims=64), ff=65)], {}),
    "pair_of_136_states": (K, [K.par(right=R(heads=1, dim=136, vdim=72), ff=40)], {}),
    "leaves_the_window": (K, [K.par(left=A(size=7, pool=3), ff=40)], {}),
    "pools_completed": (K, [K.par(left=A(size=500, pool=2), ff=40)], {}),
    "mlstm_64": (K, [K.mls(heads=3, dim=64, vdim=64, ff=100)], {}),
    "mlstm_128": (K, [K.mls(heads=2, dim=127, vdim=200, ff=31)], {}),
    "mlstm_260": (K, [K.mls(heads=1, dim=260, vdim=40, ff=64)], {}),
    "split_k": (K, [K.par(ff=1100), K.mls(ff=96)], {"width": 1024, "vocab": 61}),
    "splits_differ": (K, [K.par(ff=1056)], {"width": 1032, "vocab": 61}),
    "odd_width": (K, [K.par(ff=35), K.mls(ff=33)], {"width": 91}),
    "experts_and_shared": (U, [U.lig(mlp=U.moe(experts=6, top=2, ff=24, shared=40)), U.lat(mlp=U.moe(experts=5, top=5, ff=33, shared=90))], {}),
    "experts_alone": (U, [U.lig(mlp=U.moe(experts=6, top=2, ff=24, shared=0))], {}),
    "experts_64_rows": (U, [U.lig(mlp=U.moe(experts=64, top=3, ff=8, shared=40))], {}),
    "experts_65_rows": (U, [U.lig(mlp=U.moe(experts=65, top=3, ff=8, shared=31))], {}),
    "experts_300_rows": (U, [U.lig(mlp=U.moe(experts=300, top=4, ff=8, shared=32))], {}),
    "experts_split_k": (U, [U.lig(mlp=U.moe(experts=3, top=2, ff=1030, shared=1100))], {"width": 1024, "vocab": 61}),
    "experts_split_apart": (U, [U.lig(mlp=U.moe(experts=3, top=2, ff=40, shared=1100))], {"width": 1024, "vocab": 61}),
}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(CASES))
def test_single_tokens(hy, tmp_path, name, dtype):
    mod, layers, kw = CASES[name]
    cfg, total = mod.config(layers, **kw), sum(SIZES)
    m = mod.Model(hy, tmp_path, cfg, 3)
    rng = np.random.default_rng(4)
    toks = [rng.integers(0, cfg["vocab"], total).astype(np.int32) for _ in range(2)]
    p = m.plan(dtype, ctx=total + 8, max_batch=16, n_seqs=2)
    if dtype == "bfloat16":
        whole = [mod.whole(p, t) for t in toks]
    slots, got, pos = [p.acquire(), p.acquire()], [[], []], 0
    for c in SIZES:
        for i in range(2):
            got[i].append(p.step(slots[i], toks[i][pos:pos + c], pos, list(range(c))))
        pos += c
    p.close()
    for i in range(2):
        want = m.ref(toks[i])
        bound = 3e-5 if dtype == "float32" else max(mod.BF16_TOL, 2 * N.err(whole[i], want))
        assert N.err(np.concatenate(got[i]), want) < bound
