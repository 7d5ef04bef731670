"""The autotuner tries the schedule that the ensemble came with."""
import pytest

pytestmark = pytest.mark.gpu


def test_autotune_keeps_the_short_tiles_of_small_ensembles():
    """Four small basins: the default of 4 rows takes 39 us a step, 8 rows 59."""
    from rakali_amd import scenarios as S
    from rakali_amd.ensemble import from_scenarios
    with from_scenarios(S.tidal_ensemble(n=4, seed=4, size=(64, 200))) as e:
        assert e.schedule["tile_rows"] == 4
        e.step(2)
        e.autotune(steps=20)
        assert e.schedule["schedule"] == "flat" and e.schedule["tile_rows"] < 8


def test_autotune_leaves_the_workgroups_and_graph_of_the_schedule():
    from rakali_amd import scenarios as S
    from rakali_amd.ensemble import from_scenarios
    with from_scenarios(S.tidal_ensemble(n=3, seed=5, size=(64, 120))) as e:
        e.set_schedule("flat", tile_rows=5, persistent_blocks=640, use_graph=True)
        e.autotune(steps=5)
        assert e.schedule["schedule"] == "flat" and e.schedule["persistent_blocks"] == 640 and e.schedule["use_graph"]
