"""Single tokens whose residual updates and norms the next product makes (csrc/gl3_hy_pre_kernels.h): widths around what a wavefront's places and a workgroup's threads cover (8 ... 4096, and 4104,
which keeps the launch of its own), rows that leave pairs and wavefronts over, four wavefronts a pair and one, one, two and four streams, post norms, gates, squared ReLU,
capped logits, and a step that hands no logits out between two that do.

Yardstick: the same steps in a plan with layer taps, whose updates stay launches of their own, and the designs' float64 restatements.  Bound: float32 sums of K terms in another
order, some 1e-6 of the logits' root mean square; bfloat16 plans round rows that differ so far apart now and then, 2^-9 of an operand."""
import numpy as np
import pytest

import __graft_entry__ as ge
import test_kosusun_gpu as K
import test_kugadra_gpu as U
import test_noditar_gpu as N

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hy():
    from importlib import import_module
    ge.load_package()
    return import_module(ge.PKG_NAME + ".hybrid")


def noditar(width, vocab, streams=2, ff=72):
    return N, N.config([N.att(heads=4, kv_heads=2, dim=16, vdim=16, ff=ff), N.ssm(heads=2, vdim=16, state=16), N.lat(heads=2, dim=16, vdim=16, kv_rank=32, ff=ff)], width=width, vocab=vocab, streams=streams)


def kosusun(width, vocab, ff=56):
    return K, K.config([K.par(ff=ff), K.mls(heads=2, dim=16, vdim=16, ff=ff)], width=width, vocab=vocab)


def kugadra(width, vocab, ff=56):
    return U, U.config([U.lig(heads=2, dim=16, vdim=16, mlp=U.dense(ff)), U.lat(mlp=U.moe())], width=width, vocab=vocab)


CASES = [(noditar, 8, 3, 1, 40), (noditar, 104, 211, 2, 72), (noditar, 264, 2051, 4, 2050), (noditar, 2048, 2047, 1, 8200), (noditar, 4096, 1025, 2, 300), (noditar, 4104, 257, 2, 72),
         (kosusun, 88, 131, None, 56), (kosusun, 520, 4099, None, 8200), (kosusun, 2056, 515, None, 1030), (kugadra, 96, 131, None, 56), (kugadra, 1032, 2055, None, 4100), (kugadra, 4096, 259, None, 96)]


def both_ways(hy, path, make, width, vocab, streams, ff, dtype):
    """Logits of twelve tokens, the first three at once: updates deferred, and launches of their own."""
    mod, cfg = make(width, vocab, streams, ff) if streams else make(width, vocab, ff)
    return both_plans(mod.Model(hy, path, cfg, seed=width % 97 + 1).plan, width, vocab, dtype)


def both_plans(plan, width, vocab, dtype):
    toks = np.random.default_rng(width).integers(0, vocab, 12).astype(np.int32)
    out = []
    for taps in (False, True):
        p = plan(dtype, ctx=32, max_batch=16, layer_taps=taps)
        s = p.acquire()
        rows = [p.step(s, toks[:3], 0, want=[2])]
        for i in range(3, 12):
            r = p.step(s, toks[i:i + 1], i, want=[] if i == 6 else [0])
            if i != 6:
                rows.append(r)
        out.append(np.concatenate(rows).astype(np.float64))
        p.close()
    return out


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("make,width,vocab,streams,ff", CASES)
def test_same_as_updates_of_their_own(hy, tmp_path, make, width, vocab, streams, ff, dtype):
    got, own = both_ways(hy, tmp_path, make, width, vocab, streams, ff, dtype)
    scale = np.sqrt((own ** 2).mean())
    assert np.sqrt(((got - own) ** 2).mean()) < (4e-6 if dtype == "float32" else 2e-2) * scale
    assert np.abs(got - own).max() < (4e-5 if dtype == "float32" else 2e-1) * scale


# widths around where a wavefront's places are one or two (1024, 2048), both sides of 16384 rows, and up to 32 pairs a workgroup
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("make,width,vocab,streams,ff", CASES + [(noditar, 1016, 4099, 1, 72), (noditar, 1024, 16381, 4, 8160), (noditar, 1032, 16387, 2, 8200), (kosusun, 2048, 12001, None, 2100),
                                                                 (kugadra, 2056, 9001, None, 96)])
def test_same_bits(hy, tmp_path, make, width, vocab, streams, ff, dtype):
    """The sums are those of the launches that a deferred update stands for, term by term."""
    got, own = both_ways(hy, tmp_path, make, width, vocab, streams, ff, dtype)
    assert np.array_equal(got, own)


@pytest.mark.parametrize("vocab", [24575, 24577])          # 384 MB: the last head whose product makes the update, the first behind a launch
def test_heads_of_many_bytes(hy, tmp_path, vocab):
    _, cfg = noditar(4096, vocab, 2)
    w = N.R.random_weights(dict(cfg, vocab=64), 5)
    for k in ("embed", "head"):
        w[k] = np.ascontiguousarray(np.resize(w[k], (vocab, 4096)))
    hy.save_model_dir(str(tmp_path), cfg, w)
    got, own = both_plans(lambda dtype, **kw: hy.HybridPlan.from_dir(str(tmp_path), dtype=dtype, **kw), 4096, vocab, "float32")
    assert np.array_equal(got, own) and np.abs(got).max() > 0


def test_against_the_restatement(hy, tmp_path):
    cfg = N.config([N.att(ff=72), N.ssm(), N.lat(ff=72)], width=136, vocab=211, streams=4)
    m = N.Model(hy, tmp_path, cfg, seed=3)
    toks = N.tokens_for(cfg, 14)
    p = m.plan("float32", ctx=32, max_batch=16)
    s = p.acquire()
    got = np.concatenate([p.step(s, toks[i:i + 1], i, want=[0]) for i in range(14)])
    p.close()
    assert N.err(got, m.ref(toks)) < 2e-5
