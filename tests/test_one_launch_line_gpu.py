"""Latent attention of one token around the position at which steps leave the one-launch kernel (csrc/gl3_hybrid.hip, hy_latent_one_line), for ranks with and without a matrix-core kernel behind
it, wide expansions and few heads, and ranks that never use it.  Yardstick: the float64 restatement; float32 sums of a few hundred terms err by some 1e-6 of the logits' root mean square
(bound 3e-5), a lost row is an error of order one."""
import numpy as np
import pytest

import __graft_entry__ as ge
import test_noditar_gpu as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,rank,dim,vdim,line", [(2, 512, 128, 512, 204), (3, 64, 20, 28, 121), (2, 256, 64, 64, 366), (2, 128, 100, 60, 246), (3, 40, 20, 28, 242), (3, 16, 20, 28, 0),
                                                      (2, 31, 16, 16, 0), (2, 36, 16, 16, 216), (3, 32, 20, 28, 218), (2, 512, 256, 512, 58), (1, 512, 512, 512, 0)])
def test_latent_steps_around_the_line(tmp_path, heads, rank, dim, vdim, line):
    from importlib import import_module
    ge.load_package()
    hy = import_module(ge.PKG_NAME + ".hybrid")
    cfg = N.config([N.lat(heads=heads, dim=dim, vdim=vdim, kv_rank=rank, ff=0)])
    m = N.Model(hy, tmp_path, cfg, 8)
    first = max(0, line - 3)
    toks = np.random.default_rng(line).integers(0, cfg["vocab"], first + 7).astype(np.int32)
    p = m.plan("float32", ctx=len(toks) + 4, max_batch=512)
    s = p.acquire()
    if first:
        p.step(s, toks[:first], 0, [])
    got = [p.step(s, toks[i:i + 1], i, [0])[0] for i in range(first, len(toks))]
    p.close()
    assert N.err(np.array(got), m.ref(toks)[first:]) < 3e-5
