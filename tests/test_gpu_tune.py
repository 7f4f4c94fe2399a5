"""The autotuner against the defaults it replaces."""
import pytest

import zyklop_amd as zk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [5000, 11000, 40000])
def test_tuning_keeps_the_parts_of_few_buckets(tmp_path, m):
    """Over window tables, where the default takes more parts per bucket than a
    table can name, tuning leaves it (split 0): the proof's buffers are the same
    after zk_autotune and after loading the table it saved. With more buckets
    the splits are tuned, 1 to 4."""
    ctx = zk.Context(0)
    ctx.set_window_tables(1)
    circ = ctx.synth_circuit(95, m, 8)
    before = ctx.slot_bytes_check(circ)
    ctx.autotune(circ)
    path = tmp_path / "t.txt"
    ctx.tune_save(path)
    rows = [ln.split() for ln in path.read_text().splitlines() if not ln.startswith("#")]
    assert [int(r[1]) for r in rows] == [2, 3]
    few = m <= 11000
    splits = [int(s) for s in rows[0][4:6] + rows[1][4:5]]
    assert splits == [0, 0, 0] if few else all(1 <= s <= 4 for s in splits)
    if few:
        assert ctx.slot_bytes_check(circ) == before
        other = zk.Context(0)
        assert other.tune_load(path) == 2
        assert other.slot_bytes_check(circ) == before
        other.close()
    circ.free()
    ctx.close()
