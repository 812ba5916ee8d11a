"""The default schedule of a batch of temperatures: no more lanes per sample than the persistent grid
needs (each further wave costs the fetch of a tile), and tiles of the size its beads are worth."""
import numpy as np
import pytest

from helpers import make_data, random_model, stage_dict_models
from pibronic_amd import pimc
from pibronic_amd.batch import TemperatureBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A,pm,B,lanes,tile", [(2, False, 8192, [32, 16], 4), (4, False, 8192, [32, 16], 4),
                                               (4, True, 8192, [16, 8], 1), (6, False, 8192, [16, 8], 1),
                                               (2, False, 100, [64, 32], 1), (6, False, 100, [64, 32], 1)])
def test_lanes_and_tiles(tmp_path, A, pm, B, lanes, tile):
    print(f"[gpu-case] batch defaults A={A} pm={pm} B={B}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(A, 4, seed=A))
    tb = TemperatureBatch([make_data(FS, T, P, B, B, pm=pm) for T, P in [(100.0, 128), (236.0, 55)]], B)
    s = tb.schedule()
    assert (s["family"], s["lanes"], s["tile"]) == ("lanes", lanes, tile)


@pytest.mark.parametrize("A,pm", [(5, True), (6, True), (7, False)])
def test_lanes_set_for_one_launch_per_problem(tmp_path, A, pm):
    """Lanes given to the schedule run in the lanes kernel, bit for bit as set in the context; without
    them each problem runs as a single evaluation does."""
    print(f"[gpu-case] batch lanes A={A} pm={pm}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(A, 3, seed=A, quad="diag"))
    B, lanes = 300, [4, 2]
    datas = [make_data(FS, T, P, B, B, pm=pm) for T, P in [(200.0, 21), (400.0, 10)]]
    qs = [d.draw_host_sample(np.random.default_rng(i), B)[0] for i, d in enumerate(datas)]
    single = [pimc.evaluate_samples(d, q, pm=pm) for d, q in zip(datas, qs)]
    tb = TemperatureBatch(datas, B)
    tb.set_schedule("sequential")
    auto = tb.evaluate(qs)
    tb.set_schedule("sequential", lanes)
    given = tb.evaluate(qs)
    for i, d in enumerate(datas):
        d.context().set_lanes_per_sample(lanes[i])
        kept = pimc.evaluate_samples(d, qs[i], pm=pm)
        assert not np.array_equal(kept["s_g"], single[i]["s_g"])
        for k in ["s_rho", "s_g", "log_scale"] + (["s_gP", "s_gM"] if pm else []):
            assert np.array_equal(auto[i][k], single[i][k]) and np.array_equal(given[i][k], kept[k]), (i, k)
