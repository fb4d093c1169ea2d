"""The exact parallel evaluation of the sequential f32 sum of squares (csrc/gl3_seqsum.h) against the plain
left-to-right chain, on random and adversarial inputs (ties, binade crossings, zeros, outliers)."""
import ctypes as C

import numpy as np
import pytest

import __graft_entry__ as ge

pytestmark = pytest.mark.gpu


def seq_sumsq(x):
    a = (x.astype(np.float32) * x.astype(np.float32)).astype(np.float32)
    return np.add.accumulate(a, dtype=np.float32)[-1]


def cases():
    rng = np.random.default_rng(5)
    for n in (1024, 2048, 2560, 4096, 5120):
        yield "normal", (rng.standard_normal(n) * 0.02).astype(np.float32)
        yield "uniform", (rng.random(n) * 2 - 1).astype(np.float32)
        yield "small-ints", rng.integers(0, 8, n).astype(np.float32)               # exact adds and ties
        yield "pow2", np.ldexp(1.0, rng.integers(-6, 6, n)).astype(np.float32)
        yield "const", np.ones(n, np.float32)
        yield "quarters", (rng.integers(1, 5, n) * 0.25).astype(np.float32)        # many exact ties
        x = (rng.random(n) * 1e-3).astype(np.float32); x[rng.integers(0, n, n // 50)] = 100.0
        yield "outliers", x
        x = rng.random(n).astype(np.float32); x[:5] = 1e-12
        yield "tiny-head", x
        yield "wide", np.ldexp(rng.random(n), rng.integers(-20, 20, n)).astype(np.float32)
        x = (rng.random(n) * 0.01).astype(np.float32); x[n // 2] = 3000.0
        yield "one-huge", x
        yield "zeros", np.zeros(n, np.float32)


def test_exact_sumsq_matches_sequential_chain(pkg):
    from importlib import import_module
    hip = import_module(ge.PKG_NAME + ".hip")
    L = hip.lib()
    out = C.c_float()
    for name, x in cases():
        x = np.ascontiguousarray(x, np.float32)
        assert L.gl3_debug_sumsq(0, x.ctypes.data_as(C.c_void_p), x.size, C.byref(out)) == 0
        ref = seq_sumsq(x)
        assert np.float32(out.value).view(np.uint32) == np.float32(ref).view(np.uint32), (name, x.size, out.value, float(ref))


@pytest.mark.parametrize("n", [1024, 1028, 2560, 4092, 5120])
def test_passes_of_the_replay(pkg, n):
    """Segments with a rounding tie are replayed one after the other, 61 in a pass: counts around one, two and three passes, spread over the wavefronts' spans or side by side.  5000^2 starts the sum in
    the middle of a binade with ulp 2: a term of 4 is easy, a term of 1 a tie."""
    from importlib import import_module
    L = import_module(ge.PKG_NAME + ".hip").lib()
    out = C.c_float()
    for hard in (0, 1, 59, 60, 61, 62, 121, 122, 123, 183, 184):
        for at in (np.linspace(1, n // 4 - 1, hard).astype(int), n // 4 - hard + np.arange(hard)):
            x = np.full(n, 2.0, np.float32)
            x[0] = 5000.0
            x[4 * at + hard % 4] = 1.0
            assert L.gl3_debug_sumsq(0, x.ctypes.data_as(C.c_void_p), n, C.byref(out)) == 0
            assert np.float32(out.value) == seq_sumsq(x), (hard, at[:4])
