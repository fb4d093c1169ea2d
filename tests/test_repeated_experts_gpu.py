"""A few tokens of a mixture of experts (hy_gemm_grouped, one launch of a dot product per token and choice) around the line from which an expert's weights come through the caches, two pairs an expert:
steps of several tokens against the same tokens one at a time, which stay below the line.  Bound: float32 sums in another order err by some 1e-6 of the row's root mean square; bfloat16 plans round each
product's input and may move it by 2^-8.

And tokens that all choose the same experts read their weights once from memory and take less time than tokens that do not: past the caches eight tokens on 2 of 8 experts took 0.94 of the time of eight
that choose differently, through them 0.85."""
import time

import numpy as np
import pytest

import __graft_entry__ as ge

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hy():
    from importlib import import_module
    ge.load_package()
    return import_module(ge.PKG_NAME + ".hybrid")


def config(experts, top, width=256, ff=96, vocab=500):
    moe = {"kind": "moe", "expert": {"ff": ff}, "router": {"experts": experts, "top": top, "scale": 1.7}, "shared": None}
    return {"architecture": "Kugadra", "vocab": vocab, "width": width, "embedding": {"scale": 2.5}, "norm": {"eps": 1e-5},
            "layers": [{"type": "lightning", "mixer": {"heads": 2, "dim": 16, "vdim": 16, "decay": [0.5, 0.75]}, "mlp": moe}]}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("experts,top", [(4, 4), (8, 2), (2, 1)])
@pytest.mark.parametrize("width,ff", [(256, 96), (1024, 40), (2048, 1032)])          # K split over wavefronts in neither, the first and both products
def test_steps_and_tokens(hy, tmp_path, experts, top, width, ff, dtype):
    cfg = config(experts, top, width, ff)
    hy.random_model_dir(str(tmp_path), cfg, seed=experts)
    p = hy.HybridPlan.from_dir(str(tmp_path), dtype=dtype, ctx=16, max_batch=8)
    s = p.acquire()
    toks = np.random.default_rng(5).integers(0, cfg["vocab"], 8).astype(np.int32)
    want = np.concatenate([p.step(s, toks[i:i + 1], i, [0]) for i in range(8)])
    for n in (2, 3, 4, 5, 8):
        got = p.step(s, toks[:n], 0, list(range(n)))
        err = np.sqrt(((got - want[:n]).astype(np.float64) ** 2).mean() / (want[:n].astype(np.float64) ** 2).mean())
        assert err < (1e-5 if dtype == "float32" else 2.0 ** -8 * 4), (n, err)
    p.close()


def test_tokens_that_choose_the_same(hy, tmp_path):
    hy.random_model_dir(str(tmp_path), config(8, 2, 2048, 1024), seed=3)
    p = hy.HybridPlan.from_dir(str(tmp_path), dtype="float32", ctx=16, max_batch=8)
    s = p.acquire()
    sets = {"same": np.full(8, 7, np.int32), "different": np.random.default_rng(1).integers(0, 500, 8).astype(np.int32)}
    times = {k: [] for k in sets}
    for _ in range(5):
        for k, toks in sets.items():
            for i in range(40):
                t0 = time.perf_counter()
                p.step(s, toks, 0)
                if i > 4:
                    times[k].append(time.perf_counter() - t0)
    p.close()
    us = {k: float(np.median(v)) * 1e6 for k, v in times.items()}
    print(us)
    assert us["same"] < 0.9 * us["different"], us
