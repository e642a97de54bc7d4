"""The autotuner's second stage keeps the built-in launch shapes among its candidates, so that a
draw the defaults suit is refined around them (no GPU needed)."""
import pytest

pytest.importorskip("torch")


def test_refinement_tries_the_built_in_defaults():
    from softwarerenderer_amd import autotune as T
    # knobs whose 0 stands for a rule and not for one of the listed values
    for knob in ("raster_group", "expand_chunk"):
        assert 0 in T.REFINE[knob], knob
