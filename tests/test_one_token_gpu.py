"""Steps of one token in the layer-list family at the edges of their kernels (csrc/gl3_hy_kernels.h): the recurrences' single step (every kind of decay,
state rows that do not fill sixteen wavefronts or pass them, value columns around a wavefront, the normaliser's column), the convolution's
blocks of eight tokens (portions shorter and longer than its taps and than a block, the tail handed from portion to portion by either kernel) and the
head products of long latents on sixteen wavefronts.  Two sequences alternate, so a state or tail written to the wrong slot shows.

Yardstick: the designs' float64 restatements.  Bound: float32 sums of a few hundred terms err by some 1e-6 of the logits' root mean
square; a lost row, column or token is an error of order one."""
import numpy as np
import pytest

import __graft_entry__ as ge
import test_kosusun_gpu as K
import test_kugadra_gpu as U
import test_noditar_gpu as N
import test_tutedra_gpu as T

pytestmark = pytest.mark.gpu
SIZES = [1, 1, 2, 1, 7, 1, 8, 1, 9, 1, 16, 1, 3, 17, 1, 1]


@pytest.fixture(scope="module")
def hy():
    from importlib import import_module
    ge.load_package()
    return import_module(ge.PKG_NAME + ".hybrid")


LAYERS = {
    "ssm_one_state": (N, N.ssm(heads=3, vdim=63, state=1, conv=1)), "ssm_17_states": (N, N.ssm(heads=4, vdim=65, state=17, groups=2, norm_groups=2, conv=2)),
    "ssm_300_states": (N, N.ssm(heads=2, vdim=130, state=300, conv=4)), "ssm_taps_5": (N, N.ssm(heads=6, vdim=64, state=64, groups=3, conv=5)),
    "ssm_taps_23": (N, N.ssm(heads=4, vdim=64, state=24, conv=23)),
    "mlstm_normaliser_column_64": (K, K.mls(heads=3, dim=20, vdim=63, ff=0)), "mlstm_normaliser_column_65": (K, K.mls(heads=2, dim=260, vdim=64, ff=0)),
    "retention_turned": (K, K.par(right=K.ret(heads=4, dim=64, vdim=66, rot_dims=32), ff=0)), "lightning": (U, U.lig(heads=3, dim=15, vdim=70, mlp=None)),
    "hgrn_odd": (T, T.hgrn(heads=3, dim=19, vdim=65)), "hgrn_272": (T, T.hgrn(heads=2, dim=272, vdim=24)),
    "latent_256": (N, N.lat(heads=3, dim=20, vdim=65, kv_rank=256, ff=0)), "latent_500": (N, N.lat(heads=2, dim=20, vdim=130, kv_rank=500, ff=0)),
    "latent_512": (U, U.lat(heads=3, dim=32, vdim=64, kv_rank=512, mlp=None)),
}


@pytest.mark.parametrize("name", list(LAYERS))
def test_single_steps_and_short_portions(hy, tmp_path, name):
    mod, layer = LAYERS[name]
    cfg, total = mod.config([layer]), sum(SIZES)
    m = mod.Model(hy, tmp_path, cfg, 5)
    rng = np.random.default_rng(9)
    toks = [rng.integers(0, cfg["vocab"], total).astype(np.int32) for _ in range(2)]
    p = m.plan("float32", ctx=total + 8, max_batch=32, n_seqs=2)
    slots, got, pos = [p.acquire(), p.acquire()], [[], []], 0
    for c in SIZES:
        for i in range(2):
            got[i].append(p.step(slots[i], toks[i][pos:pos + c], pos, list(range(c))))
        pos += c
    p.close()
    for i in range(2):
        assert N.err(np.concatenate(got[i]), m.ref(toks[i])) < 3e-5


def test_many_taps_do_not_queue(hy, tmp_path):
    """Eight tokens of a convolution with 64 taps: a thread that walks them one after the other takes 512 loads in a row, three times the step with 4 taps."""
    import time
    best = {}
    for conv in (4, 64):
        cfg = N.config([N.ssm(heads=32, vdim=64, state=128, conv=conv)] * 3)
        p = N.Model(hy, tmp_path, cfg, conv).plan("float32", ctx=40, max_batch=32)
        s, toks, times = p.acquire(), np.arange(8, dtype=np.int32), []
        for _ in range(30):
            a = time.perf_counter()
            p.step(s, toks, 0, [7])
            times.append(time.perf_counter() - a)
        p.close()
        best[conv] = min(times)
    assert best[64] < 2.0 * best[4], best
