"""Samples share a wave of the block kernel (and of the four-sample kernel, 10 surfaces), and each keeps its own scaling of the exponential: a sample
far out (finite coordinates, a large |tau V|) changes no bit of another's outputs. Against the
one-wave-per-sample kernel on the same coordinates 1e-11, as between any two FP64 kernels."""
import numpy as np
import pytest

from helpers import make_data, random_model, rel_err, stage_dict_models
from pibronic_amd import pimc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A,pm", [(7, True), (8, False), (8, True), (11, True), (15, True), (10, False)])
@pytest.mark.parametrize("far", [1e2, 1e3, 1e5, 1e7, 1e12])
def test_an_outlier_stays_alone(tmp_path, A, pm, far):
    print(f"[gpu-case] block outlier A={A} pm={pm} far={far:g}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(A, 3, seed=4, quad="full"))
    B = 20000  # one stream per sample: four samples share a wave
    data = make_data(FS, 300.0, 6, B, B, pm=pm)
    q, _ = data.draw_host_sample(np.random.default_rng(2), B)
    clean = pimc.evaluate_samples(data, q, pm=pm)
    out = [5, 1002, 10003, 16000]  # every place of a wave
    bad = q.copy()
    bad[out] *= far
    r = pimc.evaluate_samples(data, bad, pm=pm)
    keep = np.ones(B, dtype=bool)
    keep[out] = False
    beside = np.unique([4 * (o // 4) + k for o in out for k in range(4) if 4 * (o // 4) + k not in out])
    data.force_wide = True
    w = pimc.evaluate_samples(data, q[beside], pm=pm)
    keys = ["s_rho", "s_g"] + (["s_gP", "s_gM"] if pm else [])
    for k in keys:
        assert rel_err(r[k][beside], w[k], floor=1e-3 * np.mean(np.abs(clean[k]))) < 1e-11, k
    for k in keys + ["log_scale"]:
        assert np.array_equal(r[k][keep], clean[k][keep]), k
