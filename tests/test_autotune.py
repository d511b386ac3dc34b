"""The tile tuner compares fixed tiles with the library's rule (items cut by
load): it sets a tile only where one is faster, and reports gains over the
rule.  Launch times come from a model here; no GPU."""
import os

import pytest

from byteqc_amd.scf import autotune

S, P, W = 0, 1010, 2221   # (ss|ss), (ps|ps) row classes; (dd|dp) wave class


@pytest.fixture
def lib(monkeypatch):
    from byteqc_amd.lib import library_path, load_library
    if not os.path.exists(library_path()):
        pytest.skip('libbqcjk.so not built')
    lib = load_library()

    def timed(run, reps):
        # ms: by the rule S 1, P 3, W 4; a tile t costs S 2, P 1 at 64 (else
        # 5), W as much as by the rule
        out = []
        for cls, kind in ((S, 1), (P, 1), (W, 4)):
            t = lib.BQCget_set_tile(kind, cls, 0)
            ms = {S: 2.0 if t else 1.0, P: {0: 3.0, 64: 1.0}.get(t, 5.0), W: 4.0}[cls]
            out.append(dict(kind=17 if kind == 1 else 4, cls=cls, ms=ms, flops=1.0, nquart=1.0))
        return out * reps

    monkeypatch.setattr(autotune, '_timed', timed)
    yield lib
    autotune.reset()


def test_tiles_only_where_they_beat_the_rule(lib, tmp_path):
    table = autotune.tune(None, reps=2)
    assert {k: r['ck'] for k, r in table.items()} == {
        (1, S, 0): autotune.RULE, (1, P, 0): 64, (4, W, 0): autotune.RULE}
    assert autotune.current_tile(1, P, 0, 500) == 64
    assert autotune.current_tile(1, S, 0, 500) == autotune.current_tile(4, W, 0, 500) == 0
    assert autotune.gain(table) == (8.0, 6.0)
    path = str(tmp_path / 'tiles.json')
    autotune.save(table, path)
    autotune.reset()
    assert autotune.current_tile(1, P, 0, 500) == 0
    again = autotune.load(path)
    assert again == table
    autotune.install(again)
    assert autotune.current_tile(1, P, 0, 500) == 64


def test_set_tile_query(lib):
    assert lib.BQCget_set_tile(1, S, 0) == 0 and lib.BQCget_set_tile(2, S, 0) == -1
    lib.BQCset_tile(1, -1, 0, 32)
    lib.BQCset_tile(1, P, 0, 8)
    assert lib.BQCget_set_tile(1, S, 0) == 32 and lib.BQCget_set_tile(1, P, 0) == 8
    assert lib.BQCget_set_tile(4, W, 0) == 0
