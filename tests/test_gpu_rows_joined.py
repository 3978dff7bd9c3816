"""One row between two sublayers of a Zabutar block inside the launch that reads it, against 64 bits: the widths, taps and first
products that take it along, those next to them that do not, and rows before and behind larger calls."""
import pytest

import zabutar_model as zm
from test_gpu_zabutar import Pair, close, hip, run_cut, tokens  # noqa: F401

pytestmark = pytest.mark.gpu

# Six sublayers of sums of at most 2048 products each, sqrt(2048) 2^-24 of a sum's size apart from 64 bits: 1.6e-5 added up, and as
# much again for norms, gates and the experts' weights.
TOL = 4e-5


@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("width", [1024, 1028, 2048])
def test_rows_joined_where_they_are_read(hip, tmp_path, width, taps):  # noqa: F811
    # prepared attention and a dense feed-forward, borrowed keys and experts, a state and nothing behind it
    a = dict(heads=4, kv_heads=2, dim=32, vdim=32, bias_max=9)
    cfg = zm.config([zm.layer(zm.attention(**a), zm.dense(1024)), zm.layer(zm.attention(**a, kv_from=0), zm.moe(ff=32, shared=32)),
                     zm.layer(zm.hgrn2(heads=2, dim=16, vdim=32), None)], 60, width, taps=taps, max_positions=16)
    p = Pair(hip, tmp_path, cfg, rel_rows=6)
    ids = tokens(9, cfg["vocab"])
    want = p.logits(ids)
    for cuts in ((1,), (1, 6, 1), (4, 1, 3, 1)):
        close(run_cut(p.model, ids, cuts), want, TOL)
    p.model.clear_cache()
    close(p.model.run_full(ids[:1]), want[0], TOL)  # a row that leaves no state behind
    close(run_cut(p.model, ids, (1,)), want, TOL)


@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("width", [8, 1024, 1028, 2048, 2052])
def test_rows_joined_many_at_a_time(hip, tmp_path, width, taps):  # noqa: F811
    """Whole workgroups of rows, one more and one less, the first of them behind a short call's: widths of one and two pieces and the
    next one, which takes two launches."""
    cfg = zm.config([zm.layer(zm.hgrn2(heads=2, dim=16, vdim=32), zm.dense(64)), zm.layer(zm.hgrn2(heads=2, dim=16, vdim=32), zm.dense(64))],
                    60, width, taps=taps, max_positions=40)
    p = Pair(hip, tmp_path, cfg)
    rows = 9 - taps
    ids = tokens(4 * rows + 4, cfg["vocab"])
    want = p.logits(ids)
    for cuts in ((4 * rows + 4,), (2, rows + 1, 2 * rows - 1, 2), (rows, 3 * rows, 4)):
        close(run_cut(p.model, ids, cuts), want, TOL)
