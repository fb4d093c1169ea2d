"""float32 products of many tokens as products of bfloat16 planes (csrc/gl3_hy_gemm.h): matrices whose entries need all 24 bits (three planes, six products; the other tests'
weights are bfloat16 values and take one plane), at the edges of the tiles and of the rings, and values the planes cannot hold.

Yardstick: float64.  Bound of whole models: a float32 sum of K terms errs by a few 1e-6 of the logits' root mean square (measured up to 1.1e-6), the second plane left out is 2^-9 of every product (4e-3).  The
third is 2^-18 at most and 2e-6 on average, which a whole model's error does not show for one matrix (0.7e-6 to 2.5e-6 of the logits): test_the_smallest_plane looks for it in the direction in which its loss would move them."""
import time

import numpy as np
import pytest

import __graft_entry__ as ge
import kugadra_ref as KR
import noditar_ref as R
import test_kugadra_gpu as U
from test_noditar_gpu import att, config, err, lat, ssm, tokens_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hy():
    from importlib import import_module
    ge.load_package()
    return import_module(ge.PKG_NAME + ".hybrid")


def full_bits(ref, cfg, seed):
    """The design's random weights with every matrix entry moved by up to a part in 200: float32 values with all their bits."""
    rng = np.random.default_rng(seed)
    return {k: (v * (1.0 + 0.005 * rng.standard_normal(v.shape))).astype(np.float32) if v.ndim == 2 else v.astype(np.float32) for k, v in ref.random_weights(cfg, seed).items()}


def logits(hy, path, cfg, w, toks):
    hy.save_model_dir(str(path), cfg, w, dtype="F32")
    p = hy.HybridPlan.from_dir(str(path), dtype="float32", ctx=len(toks) + 8, max_batch=512)
    got = p.step(p.acquire(), toks, 0, list(range(len(toks))))
    p.close()
    return got


# stages of 32 k: fewer than a ring (64), the ring (96 - 160), behind it, across the 8-stage sums (544, 1056); rows and columns around 32, 64 and 128
@pytest.mark.parametrize("n,width,vocab,ff", [(9, 64, 211, 96), (33, 96, 1003, 160), (65, 128, 8195, 544), (130, 160, 451, 1056), (300, 192, 20003, 96)])
def test_all_bits_of_the_weights(hy, tmp_path, n, width, vocab, ff):
    cfg = config([att(heads=4, kv_heads=2, dim=16, vdim=24, ff=ff), lat(heads=2, dim=16, vdim=32, kv_rank=64, ff=ff)], width=width, vocab=vocab, streams=1)
    w = full_bits(R, cfg, n)
    toks = tokens_for(cfg, n)
    got, want = logits(hy, tmp_path / "m", cfg, w, toks), R.forward(cfg, R.to_f64(w), toks, None)
    assert err(got, want) < 3e-6
    assert np.abs(got - want).max() < 3e-5 * np.sqrt((want ** 2).mean())


@pytest.mark.parametrize("n,experts,top", [(40, 6, 2), (200, 3, 2)])          # tiles of 32 and of 64 rows
def test_all_bits_of_the_experts(hy, tmp_path, n, experts, top):
    cfg = U.config([U.lig(heads=2, dim=16, vdim=16, mlp=U.moe(experts=experts, top=top, ff=96, shared=64))], width=128)
    w = full_bits(KR, cfg, n)
    toks = tokens_for(cfg, n)
    got, want = logits(hy, tmp_path / "m", cfg, w, toks), KR.forward(cfg, KR.to_f64(w), toks)
    assert np.median(np.sqrt(((got - want) ** 2).mean(axis=1)) / np.sqrt((want ** 2).mean())) < 3e-6          # (a near tie of two experts may fall the other way)


ONE = {"head": None, "mlp.gate": None, "mlp.down": None, "mix.o": None, "mix.uk": None, "mix.uv": None, "mlp.e1.gate": 40, "mlp.e2.up": 200, "mlp.e1.down": 40, "mlp.e2.down": 200}


@pytest.mark.parametrize("name", ONE)
def test_the_smallest_plane(hy, tmp_path, name):
    """One matrix alone holds 24 bits (of the experts' one of one expert).  What is left between the logits and float64's must not point where the loss of its third plane points: the share is 1 if it
    is lost, 0 if not."""
    if ONE[name]:          # tiles of 32 and of 64 rows
        ref, n, cfg = KR, ONE[name], U.config([U.lig(heads=2, dim=16, vdim=16, mlp=U.moe(experts=3, top=2, ff=96, shared=64))], width=128)
    else:
        ref, n, cfg = R, 130, config([lat(heads=2, dim=16, vdim=32, kv_rank=64, ff=96)], width=128, vocab=451, streams=1)
    name = name if name == "head" else "l0." + name
    w = {k: R.bf16_round(v) for k, v in ref.random_weights(cfg, 11).items()}
    w[name] = (w[name] * (1.0 + 0.005 * np.random.default_rng(1).standard_normal(w[name].shape))).astype(np.float32)
    p0 = R.bf16_round(w[name])
    two = p0.astype(np.float64) + R.bf16_round(w[name] - p0)
    toks = tokens_for(cfg, n)
    got, full = logits(hy, tmp_path, cfg, w, toks).astype(np.float64), ref.forward(cfg, ref.to_f64(w), toks)
    lost = ref.forward(cfg, dict(ref.to_f64(w), **{name: two}), toks) - full
    left = got - full
    same = np.abs(left).max(axis=1) < 1e-4 * np.abs(full).max()          # (a near tie of two experts may fall the other way)
    assert same.mean() > 0.9
    left, lost = left[same], lost[same]
    share = (left * lost).sum() / (lost * lost).sum()
    assert abs(share) < 0.25


@pytest.mark.parametrize("bits", [16, 24])
@pytest.mark.parametrize("n,k", [(181, 2048), (64, 512)])
def test_error_of_one_product(hy, tmp_path, n, k, bits):
    """The head's product alone: with an identity in its place the logits are its operand, to the bit.  Float32 MFMAs err by 2.1e-7 here, a chain that rounds every plane's product to the sum's
    size by 1.7e-7 (bfloat16 values) and 2.3e-7; one rounding of 2^-24 per 16 k in blocks of 128 k by 0.8e-7 to 1.0e-7."""
    cfg = config([att(heads=2, kv_heads=2, dim=16, vdim=16, ff=32)], width=k, vocab=k, streams=1)
    rng = np.random.default_rng(k + bits)
    w = dict(R.random_weights(cfg, 7), head=np.eye(k, dtype=np.float32))
    toks = tokens_for(cfg, n)
    rows = logits(hy, tmp_path / "a", cfg, w, toks).astype(np.float64)
    head = (0.02 * rng.standard_normal((k, k))).astype(np.float32)
    head = head if bits == 24 else R.bf16_round(head)
    got, want = logits(hy, tmp_path / "b", cfg, dict(w, head=head), toks), rows @ head.astype(np.float64).T
    assert np.linalg.norm(got - want) < 1.4e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("log2,bound", [(100, 1.4e-7), (-108, 1.4e-7), (-116, 4e-6)])
def test_planes_of_large_and_tiny_values(hy, tmp_path, log2, bound):
    """Planes hold all bits of values above 2^-108; below, they run out of bfloat16's range (2.2e-6 at 2^-116, float32 MFMAs 2.1e-7)."""
    cfg = config([att(heads=2, kv_heads=2, dim=16, vdim=16, ff=32)], width=512, vocab=512, streams=1)
    w, toks = dict(R.random_weights(cfg, 7), head=np.eye(512, dtype=np.float32)), tokens_for(cfg, 64)
    rows = logits(hy, tmp_path / "a", cfg, w, toks).astype(np.float64)
    head = (np.random.default_rng(3).standard_normal((512, 512)) * 2.0 ** log2).astype(np.float32)
    got, want = logits(hy, tmp_path / "b", cfg, dict(w, head=head), toks), rows @ head.astype(np.float64).T
    assert np.linalg.norm(got * 2.0 ** -log2 - want * 2.0 ** -log2) < bound * np.linalg.norm(want * 2.0 ** -log2)


@pytest.mark.parametrize("bits", [16, 24])
def test_values_that_planes_do_not_hold(hy, tmp_path, bits):
    """Head rows of 3.395e38 (finite, rounds to infinity in bfloat16), of infinity and of mixed signs: every logit is what float32 products give."""
    cfg = config([att(heads=2, kv_heads=2, dim=16, vdim=16, ff=32)], width=64, vocab=300, streams=1)
    w = full_bits(R, cfg, 5) if bits == 24 else {k: R.bf16_round(v) for k, v in R.random_weights(cfg, 5).items()}
    toks = tokens_for(cfg, 40)
    base = logits(hy, tmp_path / "a", cfg, w, toks)
    head = w["head"].copy()
    head[7] = 0.0
    head[7, 3] = np.float32(3.395e38) * np.float32(1e-3 if bits == 16 else 1.0)
    head[11, 5] = np.inf
    head[12] = 0.0
    head[12, 5], head[12, 6] = np.inf, -np.inf
    got = logits(hy, tmp_path / "b", cfg, dict(w, head=head), toks)
    h = R.forward(cfg, R.to_f64(dict(w, head=np.eye(64)[np.arange(300) % 64])), toks, None)          # the normed rows themselves
    with np.errstate(over="ignore"):
        want7 = (h[:, 3] * np.float64(head[7, 3])).astype(np.float32)
    ok = np.abs(h[:, 3]) < 0.99 if bits == 24 else np.ones(40, bool)
    assert ok.sum() > 10 and np.all(np.abs(got[ok, 7] - want7[ok]) <= 2e-5 * np.abs(want7[ok]) + 1e-6 * np.abs(head[7, 3]))
    assert np.array_equal(got[:, 11], np.where(h[:, 5] > 0, np.inf, -np.inf))
    assert np.isnan(got[np.sign(h[:, 5]) == np.sign(h[:, 6]), 12]).all()
    rest = np.setdiff1d(np.arange(300), [7, 11, 12])
    assert np.abs(got[:, rest] - base[:, rest]).max() <= 1e-5 * np.abs(base).max()


@pytest.mark.parametrize("bits", [16, 24])
def test_time_of_a_prompt_that_is_not_a_number(hy, tmp_path, bits):
    """A result that is not a number because an operand is not is what it has to be: a prompt of such rows takes about as long as any other (0.25 ms against 0.21; a serial
    float32 chain per result, 6.1 ms)."""
    cfg = config([ssm(heads=4, vdim=64, state=16, ff=2048)], width=1024, vocab=4096, streams=1)
    w = {k: v.copy() for k, v in (full_bits(R, cfg, 3) if bits == 24 else R.random_weights(cfg, 3)).items()}
    w["embed"][7] = np.nan
    hy.save_model_dir(str(tmp_path), cfg, w, dtype="F32")
    p = hy.HybridPlan.from_dir(str(tmp_path), dtype="float32", ctx=256, max_batch=256)
    toks = tokens_for(cfg, 181)
    toks[toks == 7] = 8
    best = []
    for t in (toks, np.full_like(toks, 7)):
        took = []
        for _ in range(6):
            s = p.acquire()
            t0 = time.perf_counter()
            got = p.step(s, t, 0, [0, 180])
            took.append(time.perf_counter() - t0)
            p.release(s)
        best.append(min(took))
    p.close()
    assert np.isnan(got).all()
    assert best[1] < 3 * best[0]


def test_infinite_rows(hy, tmp_path):
    """Rows that hold an infinity among rows that are numbers and rows that are not: float32's results for each, and nobody else's change."""
    cfg = config([ssm(heads=2, vdim=16, state=16, ff=0)], width=256, vocab=300, streams=1)
    w = full_bits(R, cfg, 5)
    w["l0.mix.o"][:] = 0.0
    w["final.norm"][9], w["final.norm"][10] = 0.0, 3.0e38          # the operand's entry 10 is past the largest float where the row's is more than 1.13
    w["embed"][:, 10] = 0.01
    w["embed"][[3, 4], 10] = 4.0, -4.0
    w["embed"][5] = np.nan
    w["head"][:, 10] = np.random.default_rng(2).choice([0.0, 0.25, -0.25], 300) * 1e-30
    toks = tokens_for(cfg, 70) % 200 + 6
    toks[[2, 40]], toks[[9, 33]], toks[60] = 3, 4, 5          # (the recurrence carries the last one on)
    x = w["embed"][toks].astype(np.float64)
    x[60:] = np.nan
    got = logits(hy, tmp_path, cfg, w, toks)
    with np.errstate(all="ignore"):
        h = (x / np.sqrt((x ** 2).mean(axis=1, keepdims=True) + cfg["norm"]["eps"]) * w["final.norm"].astype(np.float64)).astype(np.float32)
        want = h.astype(np.float64) @ w["head"].astype(np.float64).T
    assert np.isinf(h).any(axis=1).sum() == 4 and np.isfinite(h).all(axis=1).sum() == 56
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
    ok = np.isfinite(want)
    assert np.abs(got[ok] - want[ok]).max() < 1e-5 * np.sqrt((want[ok] ** 2).mean())
