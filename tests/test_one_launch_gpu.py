"""Steps of one token whose mixers run in one launch each (csrc/gl3_hy_one_kernels.h) at the edges of the kernels: head sizes around the pieces of 64
entries, one to eight query heads per key / value head, every norm, bias, sink, gate and turn, strips of sixteen wavefronts that are not full, windows about
to be passed, cached rows shared by layers, state rows and value columns around their blocks; and the positions at which a step goes over to the kernels of many workgroups and back
(a slot that restarts).  Two sequences alternate, so a row or state written to the wrong slot shows.

Yardstick: the designs' float64 restatements.  Bound: float32 sums of a few hundred terms err by some 1e-6 of the logits' root mean
square, 3e-5 for whole models as in the single-step tests; a lost row, key or column is an error of order one."""
import numpy as np
import pytest

import __graft_entry__ as ge
import test_kosusun_gpu as K
import test_kugadra_gpu as U
import test_noditar_gpu as N
import test_vonulix_gpu as V

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hy():
    from importlib import import_module
    ge.load_package()
    return import_module(ge.PKG_NAME + ".hybrid")


def par(left, right=None, **kw):
    return K.par(left=K.attn(**left), right=right or K.ret(heads=2, dim=8, vdim=8, rot_dims=4), ff=0, **kw)


LAYERS = {
    "heads_64": (N, N.att(heads=8, kv_heads=1, dim=64, vdim=64, ff=0)), "heads_4_and_68": (N, N.att(heads=3, kv_heads=3, dim=4, vdim=68, ff=0)),
    "heads_128": (N, N.att(heads=6, kv_heads=2, dim=128, vdim=64, ff=0)), "heads_132_and_256": (N, N.att(heads=4, kv_heads=2, dim=132, vdim=256, ff=0)),
    "heads_65": (N, N.att(heads=4, kv_heads=2, dim=65, vdim=64, ff=0)),          # (rows that do not start on 16 bytes: the kernels of many workgroups)
    "whole_norm_bias_sink_turn": (K, par(dict(heads=6, kv_heads=2, dim=72, vdim=32, size=400, pool=0, rot_dims=48))),
    "window_passed": (K, par(dict(heads=4, kv_heads=2, dim=64, vdim=64, size=37, pool=5, rot_dims=64))),
    "window_of_the_sequence": (K, par(dict(heads=4, kv_heads=2, dim=32, vdim=32, size=90, pool=8, rot_dims=32))),
    "turned_values": (V, V.layer(heads=4, kv_heads=2, dim=64, vdim=40, size=60, keep=3, rot_dims=32, experts=0)),
    "latent_4": (N, N.lat(heads=3, dim=20, vdim=4, kv_rank=4, ff=0)), "latent_260": (N, N.lat(heads=3, dim=33, vdim=132, kv_rank=260, ff=0)),
    "latent_512": (N, N.lat(heads=2, dim=128, vdim=512, kv_rank=512, ff=0)), "latent_30": (N, N.lat(heads=3, dim=20, vdim=28, kv_rank=30, ff=0)),
    "latent_turned": (U, U.lat(heads=3, dim=64, rot_dim=32, vdim=64, kv_rank=224, q_rank=36, mlp=None)),
    "retention_64": (K, K.par(right=K.ret(heads=3, dim=64, vdim=128, rot_dims=64), ff=0)), "retention_65": (K, K.par(right=K.ret(heads=3, dim=65, vdim=63, rot_dims=32), ff=0)),
    "retention_129": (K, K.par(right=K.ret(heads=2, dim=129, vdim=500, rot_dims=0), ff=0)), "mlstm_20": (K, K.mls(heads=3, dim=20, vdim=255, ff=0)),
    "mlstm_128": (K, K.mls(heads=2, dim=128, vdim=127, ff=0)), "mlstm_256": (K, K.mls(heads=2, dim=256, vdim=256, ff=0)), "mlstm_63": (K, K.mls(heads=2, dim=63, vdim=64, ff=0)),
}
MORE = {"latent_turned": [U.lat(heads=2, dim=16, rot_dim=32, vdim=20, kv_rank=224, q_rank=24, kv_from=0, mlp=None)]}          # (a layer that reads another one's rows)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(LAYERS))
def test_tokens_one_by_one(hy, tmp_path, name, dtype):
    mod, layer = LAYERS[name]
    layers = [layer] + MORE.get(name, [])
    kw = {"side": 0} if mod is V else {}
    cfg, total = mod.config(layers, **kw), 100
    m = mod.Model(hy, tmp_path, cfg, 5)
    rng = np.random.default_rng(9)
    toks = [rng.integers(0, cfg["vocab"], total).astype(np.int32) for _ in range(2)]
    p = m.plan(dtype, ctx=total + 8, max_batch=32, n_seqs=2)
    slots, got, pos = [p.acquire(), p.acquire()], [[], []], 0
    sizes = [1] * 20 + [17, 1, 1, 25] + [1] * 36          # from the first token on, and behind longer portions
    assert sum(sizes) == total
    for c in sizes:
        for i in range(2):
            got[i].append(p.step(slots[i], toks[i][pos:pos + c], pos, list(range(c))))
        pos += c
    p.close()
    for i in range(2):
        assert N.err(np.concatenate(got[i]), m.ref(toks[i])) < (3e-5 if dtype == "float32" else 6e-2)


@pytest.mark.parametrize("name,positions", [("heads_64", 768), ("heads_132_and_256", 253), ("latent_512", 204), ("latent_260", 640)])
def test_where_steps_go_over_to_many_workgroups(hy, tmp_path, name, positions):
    mod, layer = LAYERS[name]
    cfg = mod.config([layer])
    m = mod.Model(hy, tmp_path, cfg, 6)
    n = positions + 4
    toks = np.random.default_rng(3).integers(0, cfg["vocab"], n).astype(np.int32)
    want = m.ref(toks)
    p = m.plan("float32", ctx=n + 4, max_batch=512)
    s = p.acquire()
    p.step(s, toks[:positions - 4], 0, [])
    got = [p.step(s, toks[i:i + 1], i, [0])[0] for i in range(positions - 4, n)]
    again = [p.step(s, toks[i:i + 1], i, [0])[0] for i in range(3)]          # the slot restarts
    p.close()
    assert N.err(np.array(got), want[positions - 4:]) < 3e-5 and N.err(np.array(again), want[:3]) < 3e-5


@pytest.mark.parametrize("width", [6, 1022, 8196])
@pytest.mark.parametrize("design", ["streams", "plain"])
def test_embedding_with_the_first_norm(hy, tmp_path, design, width):
    """One to four tokens: the embedding makes the first norm, a single token's last update the final one; rows around a thread's registers, five tokens beside them."""
    mod = N if design == "streams" else K
    cfg = mod.config([N.att(heads=2, kv_heads=1, dim=8, vdim=8, ff=0)] if design == "streams" else [K.mls(heads=2, dim=8, vdim=8, ff=8)], width=width, vocab=37)
    m = mod.Model(hy, tmp_path, cfg, 7)
    toks = np.random.default_rng(1).integers(0, 37, 24).astype(np.int32)
    p = m.plan("float32", ctx=32, max_batch=32)
    s, got, pos = p.acquire(), [], 0
    for c in [1, 2, 4, 5, 3, 1, 1, 7]:
        got.append(p.step(s, toks[pos:pos + c], pos, list(range(c))))
        pos += c
    again = p.step(s, toks[:3], 0, [2])          # (one wanted row of several)
    p.close()
    want = m.ref(toks)
    assert N.err(np.concatenate(got), want) < 3e-5 and N.err(again, want[2:3]) < 3e-5
