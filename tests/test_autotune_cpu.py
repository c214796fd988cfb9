"""The tuner weighs every tile that a solver chooses by itself."""
from lbfs_amd import autotune


def test_candidates_hold_the_default_tiles():
    assert {(8, 8, 8, 512), (8, 8, 4, 256), (8, 4, 4, 256), (4, 4, 4, 256)} <= set(autotune.CANDIDATES)
    assert len(set(autotune.CANDIDATES)) == len(autotune.CANDIDATES)
