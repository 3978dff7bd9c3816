"""Rows in the experts' order where the experts fill a wavefront, just do not, or fill sixteen, and rows more than one workgroup, called
again and again (the counters are cleared behind a call)."""
import numpy as np
import pytest

import zabutar_model as zm
from test_gpu_zabutar import Pair, close, hip  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts,identity,top,groups,n", [(1, 0, 1, 1, 260), (64, 0, 5, 4, 260), (65, 1, 9, 3, 260), (600, 40, 9, 8, 116)])
def test_rows_of_experts(hip, tmp_path, experts, identity, top, groups, n):  # noqa: F811
    moe = zm.moe(ff=8, experts=experts, identity=identity, top=top, groups=groups, keep=groups, shared=0)
    p = Pair(hip, tmp_path, zm.config([zm.layer(zm.hgrn2(heads=1, dim=4, vdim=4), moe)], width=32, vocab=16))
    x = np.random.default_rng(0).standard_normal((n, 32)).astype(np.float32)
    want, b = p.layer(0, x), p.model.blocks[0]
    for cut in (n, 115, 17):  # 2340 rows of nine each, 1035, 153
        b.clear_cache()
        close(np.concatenate([b.forward_cached(x[a:a + cut]) for a in range(0, n, cut)]), want, 2e-5)
