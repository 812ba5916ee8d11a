"""The default schedule of a batch of temperatures: no more lanes per sample than the persistent grid
needs (each further wave costs the fetch of a tile), and tiles of the size its beads are worth."""
import pytest

from helpers import make_data, random_model, stage_dict_models
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
