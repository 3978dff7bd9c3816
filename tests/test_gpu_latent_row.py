"""One row of latent attention in a launch of its own, against 64 bits: the widths of its two forms and the first one behind them,
sizes that fill no round of keys, rows or pieces, sequences from their first token on, with and without a window, and the
number of keys from which on the three launches take over."""
import pytest

import tutilorn_model as tm
from test_gpu_tutilorn import Pair, close, hip, run_cut, tokens  # noqa: F401

pytestmark = pytest.mark.gpu


# TOL: sums of at most 592 products and 1064 keys round by 1700^0.5 times 2^-24 at random, 2.5e-6, once in each of five steps of a layer,
# and a score's error, of as much of its size (up to ten), comes through the exponential.
@pytest.mark.parametrize("n,cuts,m", [
    (135, (1,), dict(heads=2, dim=64, rot_dim=32, vdim=64, kv_rank=256, q_rank=48, window=0)),
    (70, (1,), dict(heads=3, dim=33, rot_dim=16, vdim=97, kv_rank=304, q_rank=28, window=50)),
    (40, (1,), dict(heads=2, dim=7, rot_dim=16, vdim=129, kv_rank=308, q_rank=28, window=0, rot_dims=6)),
    (35, (1,), dict(heads=1, dim=70, rot_dim=64, vdim=3, kv_rank=516, q_rank=28, window=33)),
    (35, (1,), dict(heads=9, dim=1, rot_dim=0, vdim=1, kv_rank=4, q_rank=8, window=0)),
    (1064, (1057, 1, 1, 1, 1, 1, 1, 1), dict(heads=2, dim=16, rot_dim=8, vdim=16, kv_rank=64, q_rank=32, window=0)),
    (420, (340, 1, 1, 1, 70, 1, 1), dict(heads=2, dim=96, rot_dim=32, vdim=96, kv_rank=320, q_rank=32, window=0)),
    (300, (255, 1, 1, 13, 1), dict(heads=2, dim=128, rot_dim=64, vdim=128, kv_rank=512, q_rank=32, window=0))])
def test_one_row_of_latent_attention(hip, tmp_path, n, cuts, m):  # noqa: F811
    p = Pair(hip, tmp_path, tm.config([tm.layer(tm.mixer(**m))], width=64))
    ids = tokens(n, p.cfg["vocab"])
    want = p.logits(ids)
    close(run_cut(p.model, ids, cuts), want, 2e-5)
    p.model.clear_cache()
    close(p.model.run_full(ids[:1]), want[0], 2e-5)  # a row that leaves nothing behind
