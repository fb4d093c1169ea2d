"""Launches of one token that share one (csrc/gl3_hy_beside_kernels.h) take every sum in the order of the launches they stand for: the same steps in a plan whose launches stay apart (GL3_HY_APART=1)
give the same bits.  The forms of test_side_by_side_gpu.py, and the gate / up rows that walk (hy_walk_glu) with several chunks of a row and several pairs of rows per wavefront: widths of one to six
chunks, with whole and ragged last ones, and past the longest row that walks, feed-forwards of less than a pair per wavefront up to five, beside attention with retention and beside mLSTM, and beside more mixer workgroups than it takes (129)."""
import os

import numpy as np
import pytest

import __graft_entry__ as ge
import test_kosusun_gpu as K
import test_side_by_side_gpu as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hy():
    from importlib import import_module
    ge.load_package()
    return import_module(ge.PKG_NAME + ".hybrid")


def both(hy, path, cfg, dtype):
    """Logits of two sequences that take turns, in steps of several tokens and one, launches together and apart."""
    total = sum(S.SIZES)
    rng = np.random.default_rng(4)
    toks = [rng.integers(0, cfg["vocab"], total).astype(np.int32) for _ in range(2)]
    out = []
    for apart in ("0", "1"):
        os.environ["GL3_HY_APART"] = apart
        try:
            p = hy.HybridPlan.from_dir(str(path), dtype=dtype, ctx=total + 8, max_batch=16, n_seqs=2)
        finally:
            del os.environ["GL3_HY_APART"]
        slots, got, pos = [p.acquire(), p.acquire()], [], 0
        for c in S.SIZES:
            got += [p.step(slots[i], toks[i][pos:pos + c], pos, list(range(c))) for i in range(2)]
            pos += c
        p.close()
        out.append(np.concatenate(got))
    assert np.isfinite(out[0]).all() and out[0].std() > 0
    return out


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(S.CASES))
def test_forms(hy, tmp_path, name, dtype):
    mod, layers, kw = S.CASES[name]
    cfg = mod.config(layers, **kw)
    mod.Model(hy, tmp_path, cfg, 3)
    got, own = both(hy, tmp_path / "m3", cfg, dtype)
    assert np.array_equal(got.view(np.uint32), own.view(np.uint32))


WIDE = K.par(left=K.attn(heads=96, kv_heads=2, dim=8, vdim=8, rot_dims=8), right=K.ret(heads=33, dim=8, vdim=8), ff=700)


# 16 x 249 and 253 wavefronts: a pair each up to 3984 / 4048 features
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width,ff", [(8, 96), (256, 3968), (264, 4096), (512, 4128), (520, 12000), (1000, 8000), (1016, 4100), (1016, 7900), (1536, 8192), (1540, 8200), (2048, 8192), (2056, 8200), (2048, 20000), (3072, 8200), (3080, 8192), (4096, 8224)])
def test_rows_that_walk(hy, tmp_path, width, ff, dtype):
    cfg = K.config([K.par(ff=ff), K.mls(ff=ff)], width=width, vocab=600)          # (random_model_dir: matrices of fewer than 4096 entries are constant)
    hy.random_model_dir(str(tmp_path), cfg, seed=width + ff)
    got, own = both(hy, tmp_path, cfg, dtype)
    assert np.array_equal(got.view(np.uint32), own.view(np.uint32))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_more_mixers_than_the_walk_takes(hy, tmp_path, dtype):
    cfg = K.config([WIDE], width=264, vocab=61)
    hy.random_model_dir(str(tmp_path), cfg, seed=9)
    got, own = both(hy, tmp_path, cfg, dtype)
    assert np.array_equal(got.view(np.uint32), own.view(np.uint32))
