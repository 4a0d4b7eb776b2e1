"""The tuners' default candidates: no two of them are the same launch."""
import itertools

from mocassin_amd import autotune as AT


def test_single_model_candidates_are_different_launches():
    # auto and pool name one kernel
    shapes = [tuple(sorted(dict(c, kernel="auto").items())) for c in AT.candidates()]
    assert len(set(shapes)) == len(shapes)
    assert {c["kernel"] for c in AT.candidates()} == {"auto", "pool"}


def test_batch_candidates_are_different_launches():
    # chunk does not change the launch
    keys = [k for k in AT.BATCH_GRID if k != "chunk"]
    assert len(AT.BATCH_GRID["chunk"]) == 1
    shapes = list(itertools.product(*(AT.BATCH_GRID[k] for k in keys)))
    assert len(set(shapes)) == len(shapes) == 18
