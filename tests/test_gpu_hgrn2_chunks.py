"""Gated states over the row counts at which the chunks get longer, for one and several tiles of value columns, against 64 bits."""
import numpy as np
import pytest

import zabutar_model as zm
from test_gpu_zabutar import Pair, close, hip  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [17, 256, 257, 1024, 1025])  # chunks of 16, 16, 32, 32 and 64 rows of eight heads
@pytest.mark.parametrize("dim,vdim", [(20, 28), (128, 128), (36, 300)])
def test_chunks_of_every_length(hip, tmp_path, T, dim, vdim):  # noqa: F811
    """The gates' products fall off within a few hundred rows: a row is a sum of about as many products of dim terms, (300 x 128)^0.5
    2^-24 apart at random, 1.2e-5, in the state and in the result."""
    p = Pair(hip, tmp_path, zm.config([zm.layer(zm.hgrn2(heads=8, dim=dim, vdim=vdim), None)], width=32, vocab=16))
    x = np.random.default_rng(T).standard_normal((T + 3, 32)).astype(np.float32)
    want, b = p.layer(0, x), p.model.blocks[0]
    got = np.concatenate([b.forward_cached(x[:T]), b.forward_cached(x[T:])])  # (the state behind the chunks, too)
    close(got, want, 2.5e-5)
