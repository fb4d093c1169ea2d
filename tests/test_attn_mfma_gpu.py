"""The attention core on the matrix cores (csrc/gl3_hy_attn_mfma.h): the head sizes it is built for, whole prompts and portions behind earlier
positions, key splits of short portions and single tokens far from the start, row blocks and key tiles of 32 with remainders, groups of 1, 3 and 4 query heads, windows with kept first keys and with pooled
blocks, latent attention's expanded keys with and without a rotated part, a distance penalty with the extra unit; the short portions at
the end of a cut prompt go through the key-split kernel.

Yardstick: the designs' float64 restatements.  Bound: float32 scores of up to 192 terms, a softmax and sums over the keys err by some 1e-6 of the
logits' root mean square (queries and keys of size one); a lost or extra key of a few hundred is an error of 1e-3 and more."""
import time

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


LAYERS = {
    "64_gqa2": (N, N.att(heads=4, kv_heads=2, dim=64, vdim=64, ff=0)), "128_gqa3": (N, N.att(heads=6, kv_heads=2, dim=128, vdim=128, ff=0, scale=0.1)),
    "128_mha": (N, N.att(heads=3, kv_heads=3, dim=128, vdim=128, ff=0, scale=0.1)), "latent64": (N, N.lat(heads=4, dim=64, vdim=64, kv_rank=96, ff=0)),
    "window_pool64": (K, K.par(left=K.attn(heads=4, kv_heads=1, dim=64, vdim=64, size=37, pool=5), ff=0)),
    "window_pool128": (K, K.par(left=K.attn(heads=4, kv_heads=2, dim=128, vdim=128, size=100, pool=16, scale=0.1), ff=0)),
    "window_keep64": (V, V.layer(size=29, keep=3, experts=0, heads=4, kv_heads=2, dim=64, vdim=64)),
    "latent96": (U, U.lat(heads=4, dim=64, rot_dim=32, vdim=64, kv_rank=60, mlp=None)), "latent192": (U, U.lat(heads=2, dim=128, rot_dim=64, vdim=128, kv_rank=60, mlp=None, scale=0.1)),
}


@pytest.mark.parametrize("n,batch", [(17, 64), (33, 64), (200, 256), (333, 128), (300, 97)])
@pytest.mark.parametrize("name", list(LAYERS))
def test_portions_and_tiles(hy, tmp_path, name, n, batch):
    mod, layer = LAYERS[name]
    cfg = mod.config([layer])
    m = mod.Model(hy, tmp_path, cfg, seed=n)
    toks = np.random.default_rng(n).integers(0, cfg["vocab"], n).astype(np.int32)
    p = m.plan("float32", ctx=n + 8, max_batch=batch)
    s = p.acquire()
    got = p.step(s, toks, 0, list(range(n)))
    p.close()
    want = m.ref(toks)
    assert N.err(got, want) < 2e-5, N.err(got, want)


# a few tokens at a time (hy_attn_few_kernel): the head sizes above and latents of 128 / 256 / 512 cached entries scored in the latent's space
FEW = {k: LAYERS[k] for k in ("64_gqa2", "128_gqa3", "128_mha", "window_pool64", "window_pool128", "window_keep64")}
FEW.update({"latent_direct128": (U, U.lat(heads=5, dim=24, rot_dim=32, vdim=20, kv_rank=96, mlp=None)), "latent_direct256": (N, N.lat(heads=3, dim=16, vdim=24, kv_rank=256, ff=0)),
            "latent_direct512": (N, N.lat(heads=40, dim=16, vdim=16, kv_rank=512, ff=0))})


@pytest.mark.parametrize("n", [0, 31, 130])
@pytest.mark.parametrize("name", list(FEW))
def test_a_few_tokens(hy, tmp_path, name, n):
    mod, layer = FEW[name]
    cfg = mod.config([layer])
    m = mod.Model(hy, tmp_path, cfg, seed=n)
    steps = [1, 1, 3, 8, 16, 1, 5]
    toks = np.random.default_rng(n).integers(0, cfg["vocab"], n + sum(steps)).astype(np.int32)
    p = m.plan("float32", ctx=len(toks) + 8, max_batch=64)
    s, got, pos = p.acquire(), [], n
    if n:
        got.append(p.step(s, toks[:n], 0, list(range(n))))
    for k in steps:
        got.append(p.step(s, toks[pos:pos + k], pos, list(range(k))))
        pos += k
    p.close()
    want = m.ref(toks)
    assert N.err(np.concatenate(got), want) < 2e-5


def odd_model(hy, tmp_path, mod, layer, seed):
    """A model whose last token embeds as not-a-number: its key and its value are none."""
    cfg = mod.config([layer])
    odd = cfg["vocab"] - 1

    def tweak(*a):
        a[-1]["embed"][odd] = np.nan
    return mod.Model(hy, tmp_path, cfg, seed, tweak), odd


@pytest.mark.parametrize("bad", [3, 50, 99])
@pytest.mark.parametrize("name", list(LAYERS))
def test_rows_that_do_not_see_a_bad_key(hy, tmp_path, name, bad):
    """Rows in front of a key and value that are not numbers, and rows whose window has left them behind, are the restatement's."""
    mod, layer = LAYERS[name]
    m, odd = odd_model(hy, tmp_path, mod, layer, bad)
    toks = np.random.default_rng(bad).integers(0, odd, 100).astype(np.int32)
    good = toks.copy()
    toks[bad] = odd
    p = m.plan("float32", ctx=108, max_batch=128)
    got = p.step(p.acquire(), toks, 0, list(range(100)))[:, :odd]
    p.close()
    want = m.ref(good)[:, :odd]
    assert N.err(got[:bad], want[:bad]) < 2e-5
    assert np.isnan(got[bad]).all()
    if name == "window_keep64" and bad >= 3:          # 29 keys and the first three
        assert N.err(got[bad + 29:], want[bad + 29:]) < 2e-5 if bad + 29 < 100 else True
        assert np.isnan(got[bad:bad + 29]).all()


@pytest.mark.parametrize("name", list(FEW))
def test_few_rows_that_do_not_see_a_bad_key(hy, tmp_path, name):
    mod, layer = FEW[name]
    m, odd = odd_model(hy, tmp_path, mod, layer, 7)
    toks = np.random.default_rng(7).integers(0, odd, 61).astype(np.int32)
    good = toks.copy()
    p = m.plan("float32", ctx=80, max_batch=64)
    s = p.acquire()
    first = 10 if name == "window_keep64" else 35          # (out of the window by the next step, or inside it)
    toks[first] = odd
    p.step(s, toks[:31], 0, [])
    got = [p.step(s, toks[31:39], 31, list(range(8))), p.step(s, toks[39:55], 39, list(range(16)))]
    got += [p.step(s, toks[i:i + 1], i, [0]) for i in range(55, 61)]
    p.close()
    got, want = np.concatenate(got)[:, :odd], m.ref(good)[31:, :odd]
    if name == "window_keep64":
        assert np.isnan(got[:8]).all() and N.err(got[8:], want[8:]) < 2e-5
    else:
        assert N.err(got[:4], want[:4]) < 2e-5 and np.isnan(got[4]).all()


# Key splits: a short portion behind more than 512 positions is dealt out to up to eight workgroups per row block, single tokens to up to 128 (more tiles than
# splits from 4097 positions on).  A split without a key, and rows that see none of a split's keys, leave partial sums that the merge must pass over.
@pytest.mark.parametrize("fill,n", [(600, 17), (1100, 40), (1500, 33), (2100, 18)])
@pytest.mark.parametrize("name", ["64_gqa2", "128_gqa3", "window_pool64", "window_pool128", "window_keep64", "latent64", "latent192"])
def test_key_splits(hy, tmp_path, name, fill, n):
    mod, layer = LAYERS[name]
    cfg = mod.config([layer])
    m = mod.Model(hy, tmp_path, cfg, seed=n)
    toks = np.random.default_rng(n).integers(0, cfg["vocab"], fill + n).astype(np.int32)
    p = m.plan("float32", ctx=fill + n + 8, max_batch=512)
    s = p.acquire()
    p.step(s, toks[:fill], 0, [])
    got = p.step(s, toks[fill:], fill, list(range(n)))
    p.close()
    assert N.err(got, m.ref(toks)[fill:]) < 2e-5


@pytest.mark.parametrize("dim", [64, 128])
def test_more_tiles_than_splits(hy, tmp_path, dim):
    cfg = N.config([N.att(heads=2, kv_heads=1, dim=dim, vdim=dim, ff=0)])
    m = N.Model(hy, tmp_path, cfg, seed=dim)
    fill, steps = 4180, [1, 5, 1]
    toks = np.random.default_rng(dim).integers(0, cfg["vocab"], fill + sum(steps)).astype(np.int32)
    p = m.plan("float32", ctx=len(toks) + 8, max_batch=512)
    s, got, pos = p.acquire(), [], fill
    p.step(s, toks[:fill], 0, [])
    for k in steps:
        got.append(p.step(s, toks[pos:pos + k], pos, list(range(k))))
        pos += k
    p.close()
    assert N.err(np.concatenate(got), m.ref(toks)[fill:]) < 2e-5


@pytest.mark.parametrize("heads,kv_heads", [(16, 16), (32, 16)])
def test_few_rows_of_many_tiles(hy, tmp_path, heads, kv_heads):
    """Heads of 64 whose tiles are more than run side by side: up to 8 rows a key / value head through the vector kernel, more through the few-token kernel."""
    cfg = N.config([N.att(heads=heads, kv_heads=kv_heads, dim=64, vdim=64, ff=0)])
    m = N.Model(hy, tmp_path, cfg, seed=heads)
    fill, steps = 1530, [1, 1, 4, 5, 1, 8, 9, 2]          # 768 tiles end at position 1536
    toks = np.random.default_rng(heads).integers(0, cfg["vocab"], fill + sum(steps)).astype(np.int32)
    p = m.plan("float32", ctx=len(toks) + 8, max_batch=512)
    s, got, pos = p.acquire(), [], fill
    p.step(s, toks[:fill], 0, [])
    for k in steps:
        got.append(p.step(s, toks[pos:pos + k], pos, list(range(k))))
        pos += k
    p.close()
    assert N.err(np.concatenate(got), m.ref(toks)[fill:]) < 2e-5


@pytest.mark.parametrize("size", [64, 128])
def test_infinite_key_entries(hy, tmp_path, size):
    """Three tokens whose keys hold an infinity (a latent entry that only they have, past the largest float when expanded): a row with a score of plus infinity is not a number, one
    with minus infinity leaves the key out.  One portion against portions of 16, whose kernel multiplies in float32."""
    def tweak(w):
        w["embed"][:, 0], w["embed"][3, 0], w["embed"][4, 0] = 0.0, 30.0, -30.0
        w["l0.mix.dkv"][5] = 0.0
        w["l0.mix.dkv"][5, 0] = 1.0
        w["l0.mix.uk"][:, 5] = 0.0
        w["l0.mix.uk"][7, 5] = 3e38
        w["l0.mix.uv"][:, 5] = 0.0
    cfg = N.config([N.lat(heads=1, dim=size, vdim=size, kv_rank=96, ff=0, scale=0.05)])
    m = N.Model(hy, tmp_path, cfg, seed=size, tweak=tweak)
    toks = N.tokens_for(cfg, 192)
    toks[(toks == 3) | (toks == 4)] = 5
    toks[[20, 90, 150]] = 3, 4, 3
    out = []
    for batch in (256, 16):
        p = m.plan("float32", ctx=200, max_batch=batch)
        out.append(p.step(p.acquire(), toks, 0, list(range(192))))
        p.close()
    whole, short = out
    bad = np.isnan(short).any(axis=1)
    assert 20 < bad.sum() < 180 and not bad[:20].any() and np.array_equal(np.isnan(whole).any(axis=1), bad)
    assert np.abs(whole[~bad] - short[~bad]).max() < 1e-4 * np.sqrt((short[~bad] ** 2).mean())


def exact_rows(size, seed, spread=4.0):
    """One latent attention layer whose queries, keys and values are matrix columns picked by the token, to the bit (every norm is of one entry, its mean square 1), and whose outputs are the logits but
    for a factor per row.  Scores of about `spread`."""
    W, R, heads = 1024, 256, 512 // size
    cfg = N.config([N.lat(heads=heads, dim=size, vdim=size, kv_rank=R, ff=0, scale=size ** -0.5)], width=W, vocab=512, streams=1, eps=1e-30)
    rng = np.random.default_rng(seed)
    w = {k: np.zeros_like(v, dtype=np.float32) for k, v in N.R.random_weights(cfg, 1).items()}
    w["embed"][np.arange(512), np.arange(512)] = 32.0
    w["l0.mix.dkv"][np.arange(512) % R, np.arange(512)] = 0.5
    for k in ("l0.norm1", "final.norm", "l0.mix.dkv.norm", "l0.hc1.in", "l0.hc1.mix", "l0.hc1.out"):
        w[k][...] = 1.0
    for k, scale in (("q", spread / 32), ("uk", 1 / 16), ("uv", 1 / 16)):
        w["l0.mix." + k][...] = scale * rng.standard_normal(w["l0.mix." + k].shape)
    w["l0.mix.o"][512 + np.arange(512), np.arange(512)] = 1.0
    w["head"][np.arange(512), 512 + np.arange(512)] = 1.0
    return cfg, w


@pytest.mark.parametrize("size,n,bound", [(64, 100, 2.5e-7), (64, 400, 3.1e-7), (128, 100, 3.2e-7), (128, 400, 4.0e-7)])
def test_error_of_the_attention_alone(hy, tmp_path, size, n, bound):
    """Scores of four, against float64.  The small plane products in front of the largest ones err by 1.8e-7, 2.3e-7, 2.2e-7 and 2.8e-7, float32 MFMAs by 2.9e-7, 3.6e-7, 3.8e-7 and 4.7e-7, and one chain
    in which every product is rounded to the size of the score by 3.3e-7, 4.4e-7, 5.0e-7 and 6.3e-7: the bounds lie between the first two."""
    cfg, w = exact_rows(size, n)
    hy.save_model_dir(str(tmp_path), cfg, w, dtype="F32")
    toks = np.random.default_rng(n).integers(0, 512, n).astype(np.int32)
    p = hy.HybridPlan.from_dir(str(tmp_path), dtype="float32", ctx=n + 8, max_batch=512)
    got = p.step(p.acquire(), toks, 0, list(range(n))).astype(np.float64)
    p.close()
    want = N.R.forward(cfg, N.R.to_f64(w), toks)
    got *= ((got * want).sum(axis=1) / (got * got).sum(axis=1))[:, None]          # (the last norm's factor)
    assert np.linalg.norm(got - want) < bound * np.linalg.norm(want)


@pytest.mark.parametrize("size", [64, 128])
def test_time_of_queries_that_are_not_numbers(hy, tmp_path, size):
    """Prompts of 512 tokens with such keys and queries in their second half, from the first token on, and throughout, take about as long as any other (0.15 ms against 0.12; scores made again one by one in the
    loop, 1.0 to 4.9 ms)."""
    cfg, w = exact_rows(size, 1)
    w["embed"][511] = np.nan
    hy.save_model_dir(str(tmp_path), cfg, w, dtype="F32")
    p = hy.HybridPlan.from_dir(str(tmp_path), dtype="float32", ctx=520, max_batch=512)
    toks = np.random.default_rng(1).integers(0, 511, 512).astype(np.int32)
    last, early = toks.copy(), toks.copy()
    last[256:], early[0] = 511, 511
    best = []
    for t in (toks, last, early, np.full_like(toks, 511)):
        took = []
        for _ in range(6):
            s = p.acquire()
            t0 = time.perf_counter()
            got = p.step(s, t, 0, [511])
            took.append(time.perf_counter() - t0)
            p.release(s)
        best.append(min(took))
        assert np.isnan(got).all() == (t is not toks)
    p.close()
    assert max(best[1:]) < 3 * best[0]


@pytest.mark.parametrize("batch", [128, 16])
def test_a_bad_key_alone_in_its_tile(hy, tmp_path, batch):
    """Row 91 sees keys 63 .. 91 and the first three: of the second tile of 32 the last key only, which is not a number."""
    m, odd = odd_model(hy, tmp_path, V, LAYERS["window_keep64"][1], 63)
    toks = np.random.default_rng(63).integers(0, odd, 100).astype(np.int32)
    good = toks.copy()
    toks[63] = odd
    p = m.plan("float32", ctx=108, max_batch=batch)
    got = p.step(p.acquire(), toks, 0, list(range(100)))[:, :odd]
    p.close()
    want = m.ref(good)[:, :odd]
    assert N.err(got[:63], want[:63]) < 2e-5 and N.err(got[92:], want[92:]) < 2e-5
    assert np.isnan(got[63:92]).all()


@pytest.mark.parametrize("dim,rot_dim,vdim", [(64, 32, 64), (128, 64, 128)])
def test_infinite_key_entries_beside_rotated_ones(hy, tmp_path, dim, rot_dim, vdim):
    """The same with keys of 96 and 192 entries."""
    def tweak(cfg, w):
        w["embed"][:, 0], w["embed"][3, 0], w["embed"][4, 0] = 0.0, 30.0, -30.0
        w["l0.mix.dkv"][5] = 0.0
        w["l0.mix.dkv"][5, 0] = 1.0
        w["l0.mix.uk"][:, 5] = 0.0
        w["l0.mix.uk"][7, 5] = 3e38
        w["l0.mix.uv"][:, 5] = 0.0
    cfg = U.config([U.lat(heads=1, dim=dim, rot_dim=rot_dim, vdim=vdim, kv_rank=60, mlp=None, scale=0.05)])
    m = U.Model(hy, tmp_path, cfg, seed=dim, tweak=tweak)
    toks = N.tokens_for(cfg, 192)
    toks[(toks == 3) | (toks == 4)] = 5
    toks[[20, 90, 150]] = 3, 4, 3
    out = []
    for batch in (256, 16):
        p = m.plan("float32", ctx=200, max_batch=batch)
        out.append(p.step(p.acquire(), toks, 0, list(range(192))))
        p.close()
    whole, short = out
    bad = np.isnan(short).any(axis=1)
    assert 20 < bad.sum() < 180 and not bad[:20].any() and np.array_equal(np.isnan(whole).any(axis=1), bad)
    assert np.abs(whole[~bad] - short[~bad]).max() < 1e-4 * np.sqrt((short[~bad] ** 2).mean())
