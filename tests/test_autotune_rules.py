"""Which variants load_variants hands out: a choice tuned just now or taken
from a table without counts as it is; a shipped one for 65..128 rows by the
number of systems. Runs without a GPU (the timings are given)."""
import json

import numpy as np
import pytest

pytest.importorskip("torch")

from magma_amd import autotune as at  # noqa: E402

TILE, BLOCKED, WG = 1, 2, 6


@pytest.fixture(autouse=True)
def device(monkeypatch):
    monkeypatch.setattr(at, "device_key", lambda: "dev")


def table(path, entries):
    path.write_text(json.dumps({"dev": {str(b): e for b, e in entries.items()}}))
    return path


@pytest.mark.parametrize("variant", [TILE, WG])
def test_a_fresh_choice_is_returned(tmp_path, monkeypatch, variant):
    monkeypatch.setattr(at, "tune_buckets", lambda n, nrhs, buckets=None: {b: (variant, {TILE: 2.0, WG: 1.0}) for b in buckets})
    path = tmp_path / "t.json"
    n = np.full(27, 100)
    assert at.load_variants(n, path=path) == {6: variant}
    assert json.loads(path.read_text())["dev"]["6"]["systems"] == 27
    assert at.load_variants(n, path=path) == {6: variant}                   # and read back
    line = at.WG_OVER_TILE_SYSTEMS
    assert at.load_variants(np.full(line, 100), path=path) == {6: WG}       # on the other side of the line


def test_a_table_without_counts_stands(tmp_path):
    path = table(tmp_path / "t.json", {5: {"variant": WG}, 6: {"variant": TILE}, 7: {"variant": BLOCKED}})
    for count in (3, at.WG_OVER_TILE_SYSTEMS):
        n = np.concatenate([np.full(count, k) for k in (96, 112, 128)])
        assert at.load_variants(n, path=path) == {5: WG, 6: TILE, 7: BLOCKED}


@pytest.mark.parametrize("count,want", [(27, TILE), (at.WG_OVER_TILE_SYSTEMS - 1, TILE), (at.WG_OVER_TILE_SYSTEMS, WG)])
def test_a_count_on_the_other_side_of_the_line(tmp_path, count, want):
    path = table(tmp_path / "t.json", {4: {"variant": WG, "systems": 1600}, 5: {"variant": TILE, "systems": 20},
                                       6: {"variant": BLOCKED, "systems": 20}, 8: {"variant": WG, "systems": 6000}})
    n = np.concatenate([np.full(count, k) for k in (80, 96, 112, 192)])
    assert at.load_variants(n, path=path) == {4: want, 5: want, 6: BLOCKED, 8: WG}


def test_shipped_table_has_counts():
    for entries in json.loads(at.CACHE.read_text()).values():
        assert all(e["systems"] > 0 for e in entries.values())
