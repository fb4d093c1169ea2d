"""Page-locked memory that kernels of a step read or write is allocated coherent: what a kernel stores is the host's without a copy of the runtime's in between, whatever the runtime's default is."""
import os
import re

import pytest

import __graft_entry__ as ge

CSRC = os.path.join(ge.PKG_DIR, "csrc")
# pointer -> the file whose allocation kernels touch (gl3_hybrid.hip's h_dyn is the samplers' copy target alone)
TOUCHED = {"ctx->h_dyn": "gl3_api.hip", "ctx->h_logits": "gl3_api.hip", "ctx->h_argmax": "gl3_api.hip", "p->h_log[i]": "gl3_prefill.hip", "h->h_rec": "gl3_hybrid.hip",
           "h->h_logits": "gl3_hybrid.hip"}


@pytest.mark.parametrize("pointer", list(TOUCHED))
def test_memory_that_kernels_touch_is_coherent(pointer):
    with open(os.path.join(CSRC, TOUCHED[pointer])) as f:
        calls = re.findall(r"hipHostMalloc\(\(void\*\*\)&" + re.escape(pointer) + r",[^;]*;", f.read())
    assert len(calls) == 1 and "hipHostMallocCoherent" in calls[0], calls
