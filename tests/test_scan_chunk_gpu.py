"""The recurrences 32 tokens at a time (csrc/gl3_hy_scan_chunk.h): every kind that takes them (state-space layers, exponential gates with their
normaliser column, retention with turned keys, a fixed decay behind silu) at the key sizes 64 / 128 / 256, value columns that do not fill a column
block, portions whose last chunk is full, holds one token or is cut behind an earlier portion, decays near one and decays that underflow; the same kinds with
so many heads or values that there are more than 256 blocks of 16 value columns (128 and 256 states then go 32 columns at a time, 64 stay with 16).

Yardstick: the designs' float64 restatements, which walk token by token.  Bound: float32 products and sums of a few hundred terms err by some
1e-6 of the logits' root mean square (heads are normed to size one behind the memory); a lost token or a wrong decay is an error of order one."""
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


def decays(lo, hi):
    def tweak(w):
        for k in w:
            if k.endswith("A_log"):
                w[k][:] = np.linspace(lo, hi, w[k].size)
    return tweak


LAYERS = {
    "ssm128": (N, N.ssm(heads=6, vdim=64, state=128, groups=2, norm_groups=3, conv=4), None),
    "ssm64_odd_columns": (N, N.ssm(heads=4, vdim=25, state=64, groups=4, norm_groups=2), None),
    "ssm128_underflow": (N, N.ssm(heads=8, vdim=32, state=128), decays(-9.0, 6.0)),
    "mlstm64": (K, K.mls(heads=4, dim=64, vdim=40, ff=0), None), "mlstm256": (K, K.mls(heads=2, dim=256, vdim=64, ff=0), None),
    "retention128": (K, K.par(right=K.ret(heads=4, dim=128, vdim=34, rot_dims=128), ff=0), None),
    "retention64_part": (K, K.par(right=K.ret(heads=6, dim=64, vdim=50, rot_dims=24), ff=0), None),
    "lightning64": (U, U.lig(heads=4, dim=64, vdim=56, mlp=None), None), "lightning128": (U, U.lig(heads=2, dim=128, vdim=16, mlp=None), None),
}


@pytest.mark.parametrize("n,batch", [(17, 64), (32, 64), (65, 128), (160, 160), (230, 97)])
@pytest.mark.parametrize("name", list(LAYERS))
def test_chunks_and_portions(hy, tmp_path, name, n, batch):
    mod, layer, tweak = LAYERS[name]
    cfg = mod.config([layer])
    m = mod.Model(hy, tmp_path, cfg, n, tweak) if tweak else mod.Model(hy, tmp_path, cfg, n)
    toks = np.random.default_rng(n).integers(0, cfg["vocab"], n + 3).astype(np.int32)
    p = m.plan("float32", ctx=n + 8, max_batch=batch)
    s = p.acquire()
    got = [p.step(s, toks[:n], 0, list(range(n)))]
    for i in range(3):                        # the state goes on token by token
        got.append(p.step(s, toks[n + i:n + i + 1], n + i, [0]))
    p.close()
    got, want = np.concatenate(got), m.ref(toks)
    assert N.err(got, want) < 3e-5, N.err(got, want)


SLOW = [1.0 - 2.0 ** (-1.0 - 0.4 * i) for i in range(24)]


# more than 256 blocks of 16 value columns; 56, 72, 209 (208 and the normaliser) and 170 columns leave 24, 8, 17 and 10 in the last block of 32
WIDE = {
    "ssm64": (N, N.ssm(heads=64, vdim=80, state=64, groups=4, norm_groups=4)), "ssm128": (N, N.ssm(heads=70, vdim=56, state=128, groups=2, norm_groups=2)),
    "ssm256": (N, N.ssm(heads=52, vdim=72, state=256)),
    "mlstm64": (K, K.mls(heads=32, dim=64, vdim=128, ff=0)), "mlstm256": (K, K.mls(heads=20, dim=256, vdim=208, ff=0)),
    "retention64": (K, K.par(right=K.ret(heads=24, dim=64, vdim=170, rot_dims=24, decay=SLOW), ff=0)), "lightning64": (U, U.lig(heads=24, dim=64, vdim=170, decay=SLOW, mlp=None)),
    "lightning128": (U, U.lig(heads=24, dim=128, vdim=170, decay=SLOW, mlp=None)),
}


@pytest.mark.parametrize("n,batch", [(17, 64), (33, 64), (65, 128), (130, 97)])
@pytest.mark.parametrize("name", list(WIDE))
def test_many_column_blocks(hy, tmp_path, name, n, batch):
    mod, layer = WIDE[name]
    mix = layer["mixer"].get("right") or layer["mixer"]
    assert mix["heads"] * ((mix["vdim"] + (layer["type"] == "mlstm") + 15) // 16) > 256
    cfg = mod.config([layer])
    m = mod.Model(hy, tmp_path, cfg, n)
    toks = np.random.default_rng(n).integers(0, cfg["vocab"], n + 2).astype(np.int32)
    p = m.plan("float32", ctx=n + 8, max_batch=batch)
    s = p.acquire()
    got = [p.step(s, toks[:n], 0, list(range(n)))]
    for i in range(2):
        got.append(p.step(s, toks[n + i:n + i + 1], n + i, [0]))
    p.close()
    got, want = np.concatenate(got), m.ref(toks)
    assert N.err(got, want) < 3e-5, N.err(got, want)


@pytest.mark.parametrize("bad", [5, 40, 79])
@pytest.mark.parametrize("name", ["ssm128", "ssm64_odd_columns", "mlstm64", "mlstm256", "lightning64", "lightning128"])
def test_a_token_that_is_not_finite(hy, tmp_path, name, bad):
    """It is its own row's and the later ones' concern: the rows in front of it are the restatement's of the tokens in front of it."""
    mod, layer, _ = LAYERS[name]
    cfg = mod.config([layer])
    odd = cfg["vocab"] - 1

    def tweak(*a):
        a[-1]["embed"][odd] = np.nan
    m = mod.Model(hy, tmp_path, cfg, bad, tweak)
    toks = np.random.default_rng(bad).integers(0, odd, 80).astype(np.int32)
    toks[bad] = odd
    p = m.plan("float32", ctx=88, max_batch=128)
    got = p.step(p.acquire(), toks, 0, list(range(80)))[:, :odd]          # (a tied head has a column of the odd token)
    p.close()
    want = m.ref(toks[:bad])[:, :odd]
    assert N.err(got[:bad], want) < 3e-5
    assert np.isnan(got[bad:]).all()


def test_forced_walk(hy, tmp_path):
    """GL3_HY_SCAN_NL: the token-by-token walk with that many states per lane, for a portion and for single tokens.  Its sums are added in another order for each value
    (so the bits differ), and every one is the restatement's."""
    import os
    import subprocess
    import sys
    cfg = N.config([N.ssm(heads=4, vdim=64, state=128)])
    m = N.Model(hy, tmp_path, cfg, 3)
    toks = np.random.default_rng(3).integers(0, cfg["vocab"], 43).astype(np.int32)
    code = ("import sys, numpy as np; from importlib import import_module; import __graft_entry__ as ge; ge.load_package(); hy = import_module(ge.PKG_NAME + '.hybrid')\n"
            "toks = np.array(%r, np.int32); p = hy.HybridPlan.from_dir(%r, dtype='float32', ctx=64, max_batch=64); s = p.acquire()\n"
            "out = [p.step(s, toks[:40], 0, list(range(40)))] + [p.step(s, toks[i:i + 1], i, [0]) for i in range(40, 43)]\n"
            "np.save(sys.argv[1], np.concatenate(out)); p.close()" % (toks.tolist(), m.dir))
    got = {}
    for nl in ("", "8", "32"):
        path = str(tmp_path / ("out%s.npy" % nl))
        env = {k: v for k, v in os.environ.items() if k != "GL3_HY_SCAN_NL"}
        subprocess.run([sys.executable, "-c", code, path], env=dict(env, GL3_HY_SCAN_NL=nl) if nl else env, cwd=ge.ROOT, check=True, timeout=100)
        got[nl] = np.load(path)
        assert N.err(got[nl], m.ref(toks)) < 3e-5
    for a, b in (("", "8"), ("", "32"), ("8", "32")):
        assert not np.array_equal(got[a][:40], got[b][:40]), (a, b)
