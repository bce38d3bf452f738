"""The autotuner's cache: a choice is taken only under the key it was stored
with, which names the version of the kernels' shapes. Runs without a GPU, on a
stand-in for the library."""
import json

from tgmm_amd import em


class _Lib:
    """tgmm_batch_autotune that picks eight fixed numbers."""
    tuned = 0

    def tgmm_batch_autotune(self, h, reps, tiles, buf, cap):
        self.tuned += 1
        for i, (n, _) in enumerate(em.Tiles._fields_):
            setattr(tiles._obj, n, 40 + i)
        buf.value = b"knn 1.0"
        return 0


def _batch(monkeypatch, sig="K5_S10"):
    b = em.Batch.__new__(em.Batch)
    b.L, b.h = _Lib(), None
    b.set = []
    monkeypatch.setattr(em.Batch, "signature", lambda self: sig)
    monkeypatch.setattr(em.Batch, "set_tiles", lambda self, t: self.set.append(t))
    monkeypatch.setattr(em.Batch, "reset", lambda self: None)
    return b


def test_choice_of_other_kernels_is_not_taken(tmp_path, monkeypatch):
    path = tmp_path / "tiles.json"
    monkeypatch.setenv("TGMM_TILES_CACHE", str(path))
    old = dict(em.DEFAULT_TILES, knn_cell=2)
    path.write_text(json.dumps({"K5_S10": old, "t1_K5_S10": old}))  # without and with a version
    b = _batch(monkeypatch)
    tiles, report = b.autotune(reps=1)
    assert b.L.tuned == 1 and b.set == [] and report == "knn 1.0"
    assert tiles != old
    again, report = b.autotune(reps=1)  # now from the cache
    assert b.L.tuned == 1 and again == tiles and b.set == [tiles] and report is None
    assert json.loads(path.read_text())["K5_S10"] == old  # an older library's entry stays its own
