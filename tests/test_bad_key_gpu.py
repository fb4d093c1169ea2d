"""Single tokens whose attention runs in one launch (csrc/gl3_hy_one_kernels.h) and a key whose scores are not numbers while its value is one: every row that sees the key is not a number
either, as its own key, as a cached key that stands alone in its sixteen lanes and as one among others; rows in front of it, and a sequence that starts again, are the float64
restatement's (float32 sums of a few hundred terms: some 1e-6 of the logits' root mean square, bound 3e-5)."""
import numpy as np
import pytest

import __graft_entry__ as ge
import test_noditar_gpu as N

pytestmark = pytest.mark.gpu


def attention_key(w):
    """The key projection overflows: infinite entries times an inverse norm of zero."""
    w["l0.mix.k"][:, 0] = 3e38
    for other in ("q", "v", "g"):
        w["l0.mix." + other][:, 0] = 0.0


def latent_key(w):
    """Two finite entries of the latent, in different lanes' shares, whose products with the query are infinities of both signs."""
    two = [0, 8]
    w["l0.mix.dkv"][:, 0] = 0.0
    w["l0.mix.dkv"][two] = 0.0
    w["l0.mix.dkv"][two, 0] = 1.0, -1.0
    w["l0.mix.dkv.norm"][two] = 1e30
    w["l0.mix.uk"][:, two] = 1e12
    w["l0.mix.uv"][:, two] = 0.0
    for other in ("q", "g"):
        w["l0.mix." + other][:, 0] = 0.0


LAYERS = {"heads_64": (N.att(heads=4, kv_heads=2, dim=64, vdim=64, ff=0), attention_key), "heads_128": (N.att(heads=6, kv_heads=2, dim=128, vdim=64, ff=0), attention_key),
          "heads_132": (N.att(heads=2, kv_heads=1, dim=132, vdim=64, ff=0), attention_key), "latent": (N.lat(heads=3, dim=20, vdim=28, kv_rank=64, ff=0), latent_key)}


@pytest.mark.parametrize("bad,total", [(0, 4), (2, 6), (70, 75), (200, 203)])
@pytest.mark.parametrize("name", list(LAYERS))
def test_rows_that_see_a_key_that_is_not_a_number(tmp_path, name, bad, total):
    from importlib import import_module
    ge.load_package()
    hy = import_module(ge.PKG_NAME + ".hybrid")
    layer, spoil = LAYERS[name]
    cfg = N.config([layer])
    odd = cfg["vocab"] - 1

    def tweak(w):          # the last token alone has an entry in channel 0
        w["embed"][:, 0] = 0.0
        w["embed"][odd, 0] = 3.0
        spoil(w)
    m = N.Model(hy, tmp_path, cfg, 11, tweak)
    toks = np.random.default_rng(bad).integers(0, odd, total).astype(np.int32)
    good = toks.copy()
    toks[bad] = odd
    want = m.ref(good)
    p = m.plan("float32", ctx=total + 8, max_batch=32)
    s = p.acquire()
    got = np.concatenate([p.step(s, toks[i:i + 1], i, [0]) for i in range(total)])
    again = np.concatenate([p.step(s, good[i:i + 1], i, [0]) for i in range(3)])
    p.close()
    assert np.isnan(got[bad:]).all()
    assert bad == 0 or N.err(got[:bad], want[:bad]) < 3e-5
    assert N.err(again, want[:3]) < 3e-5
