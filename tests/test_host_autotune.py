"""What the autotuner times and what it takes from its cache (no kernels)."""
import json

import pytest

from jrystal_amd import autotune, workloads as W


class _Plan:
  row_path = True
  made = []

  @classmethod
  def from_workload(cls, wl, device=None, **opt):
    cls.made.append(opt)
    return cls()

  def close(self):
    pass


@pytest.fixture
def tune(monkeypatch, tmp_path):
  """Tunes a small workload with a given library and path; the last timed
  option is the fastest."""
  path = str(tmp_path / "tune.json")
  monkeypatch.setattr(autotune, "EnergyPlan", _Plan)
  monkeypatch.setattr(autotune, "_time",
                      lambda *a: 1.0 / len(_Plan.made))

  def run(library, row_path=True):
    monkeypatch.setattr(autotune, "library_digest", lambda: library)
    _Plan.row_path = row_path
    _Plan.made = []
    best = autotune.tune(W.tiny(), cache_path=path, device="cpu")
    return best, list(_Plan.made), json.load(open(path))

  return run


def test_choices_of_another_library_are_timed_again(tune):
  best, first, _ = tune("a")
  assert first and best == first[-1]
  assert tune("a")[:2] == (best, [])
  best, again, cache = tune("b")
  assert again == first and best == again[-1]
  assert [e["library"] for e in cache.values()] == ["b"]


def test_entries_without_a_library_are_timed_again(tune, tmp_path):
  key = autotune.shape_key(W.tiny())
  (tmp_path / "tune.json").write_text(json.dumps(
    {key: {"options": {"chunk_states": 7}, "ms": 1.0, "tried": []}}))
  best, made, _ = tune("a")
  assert made and best == made[-1]


def test_x_line_targets_are_timed_where_there_are_x_lines(tune):
  _, row, _ = tune("a")
  _, plane, _ = tune("b", row_path=False)
  assert not any(o["xline_blocks"] for o in row)
  assert plane == autotune.candidates(W.tiny())
