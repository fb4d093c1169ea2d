"""The grouped expert products of the layer-list family (csrc/gl3_hy_gemm.h) at the edges of their tiles: experts of 1 - 32, 33 - 64 and more rows in
tiles of 32 (up to 48 rows on average) and 64 rows, hidden widths that leave remainders in the column tiles, gated (Vonulix) and
ungated (Kugadra) experts.  Widths are multiples of a 64-entry stage, what the ring kernel asks for.

Where every expert is chosen (top = experts) each has exactly as many rows as there are tokens and no choice can flip; the case with a choice makes
experts of different sizes in one launch and runs in float32, where the plan chooses as the restatement does (for Vonulix the tokens are drawn with a margin).

Bounds: the products' sums err by a few 1e-6 (float32) and some 1e-2 (bfloat16, 2^-9 per rounded operand over a path) of the logits' root mean square; a row
that misses its expert's product, or takes another's, moves its logits by order one."""
import pytest

import __graft_entry__ as ge
import test_kugadra_gpu as KU
import test_vonulix_gpu as VO

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hy():
    from importlib import import_module
    ge.load_package()
    return import_module(ge.PKG_NAME + ".hybrid")


# (tokens, width, experts, chosen, expert's hidden width)
ALL = [(9, 64, 1, 1, 64), (32, 128, 3, 3, 192), (33, 64, 2, 2, 128), (64, 192, 1, 1, 320), (65, 64, 3, 3, 64), (96, 320, 2, 2, 192), (129, 128, 1, 1, 448)]
SOME = [(70, 128, 5, 2, 192), (181, 64, 9, 4, 128)]


def check(m, n, dtype):
    toks, want = m.tokens(n)
    p = m.plan(dtype, ctx=n + 8, max_batch=256)
    got = KU.whole(p, toks)
    p.close()
    assert KU.err(got, want) < (2e-5 if dtype == "float32" else 3e-2)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,width,experts,top,ff", ALL)
def test_rows_of_an_expert(hy, tmp_path, n, width, experts, top, ff, dtype):
    check(KU.Model(hy, tmp_path, KU.config([KU.lig(mlp=KU.moe(experts=experts, top=top, ff=ff, shared=0))], width=width), seed=n), n, dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,width,experts,top,ff", ALL)
def test_rows_of_a_gated_expert(hy, tmp_path, n, width, experts, top, ff, dtype):
    check(VO.Model(hy, tmp_path, VO.config([VO.layer(experts=experts, top=top, ff=ff, shared=None)], width=width), seed=n), n, dtype)


@pytest.mark.parametrize("n,width,experts,top,ff", SOME)
@pytest.mark.parametrize("family", [KU, VO])
def test_experts_of_different_sizes(hy, tmp_path, n, width, experts, top, ff, family):
    layer = family.lig(mlp=family.moe(experts=experts, top=top, ff=ff, shared=0)) if family is KU else family.layer(experts=experts, top=top, ff=ff, shared=None)
    check(family.Model(hy, tmp_path, family.config([layer], width=width), seed=n), n, "float32")
