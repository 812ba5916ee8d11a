"""Either side of each line at which sizes change between the block kernel and their other one: the
outputs are those of the one-wave-per-sample kernel (1e-11, as between any two FP64 kernels)."""
import numpy as np
import pytest

from helpers import make_data, random_model, rel_err, stage_dict_models
from pibronic_amd import pimc

pytestmark = pytest.mark.gpu
CU = 256


@pytest.mark.parametrize("A,pm,N,P,Bs", [
    (5, True, 2, 8, [187 * CU // 8, 187 * CU // 8 + 1]), (5, True, 12, 9, [6000, 128 * CU - 1, 128 * CU]),
    (5, True, 2, 65, [8 * CU - 1, 8 * CU]), (5, True, 2, 113, [5000]),
    (6, True, 2, 4, [250 * CU // 4, 250 * CU // 4 + 1]), (6, True, 2, 47, [256 * CU, 256 * CU + 1]),
    (6, True, 2, 64, [256 * CU - 1, 256 * CU]), (6, True, 2, 225, [8 * CU - 1, 8 * CU]), (6, True, 2, 257, [3000]),
    (7, False, 2, 7, [187 * CU // 7, 187 * CU // 7 + 1]), (7, False, 2, 12, [160 * CU, 160 * CU + 1]),
    (7, False, 2, 48, [128 * CU - 1, 128 * CU]), (7, False, 2, 113, [8 * CU - 1, 8 * CU, 64 * CU]),
    (7, False, 20, 230, [1, 300]), (7, False, 14, 257, [3000]),
    (12, True, 2, 4, [3 * CU - 1, 3 * CU]), (13, True, 8, 11, [8 * CU - 1, 8 * CU]),
    (16, True, 2, 12, [4 * CU, 4 * CU + 1, 40 * CU]), (14, True, 2, 32, [2000]), (11, False, 2, 6, [11 * CU, 20 * CU]),
])
def test_either_side(tmp_path, A, pm, N, P, Bs):
    print(f"[gpu-case] routes A={A} pm={pm} N={N} P={P}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(A, N, seed=A))
    data = make_data(FS, 300.0, P, 64, 64, pm=pm)
    q64, _ = data.draw_host_sample(np.random.default_rng(P), 64)
    data.force_wide = True
    want = pimc.evaluate_samples(data, q64, pm=pm)
    data.force_wide = False
    keys = ["s_rho", "s_g"] + (["s_gP", "s_gM"] if pm else [])
    for B in Bs:
        k = np.arange(B) % 64
        got = pimc.evaluate_samples(data, q64[k], pm=pm)
        for key in keys:
            assert rel_err(got[key], want[key][k], floor=1e-3 * np.mean(np.abs(want[key]))) < 1e-11, (B, key)
        assert np.max(np.abs(got["log_scale"] - want["log_scale"][k])) < 1e-9 * max(1.0, np.max(np.abs(want["log_scale"])))
