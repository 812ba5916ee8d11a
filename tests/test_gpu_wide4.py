"""Four samples per wave for 9 to 12 surfaces: the results of the one-wave-per-sample kernel
(PIB_EVAL_WIDE) bit for bit, from the batch where it is taken."""
import numpy as np
import pytest

from helpers import make_data, oracle_setup, random_model, rel_err, stage_dict_models
from oracle import pimc_oracle as po
from pibronic_amd import pimc
from pibronic_amd.vibronic_model_keys import VibronicModelKeys as VMK

pytestmark = pytest.mark.gpu


def _both(data, q, **kw):
    a = pimc.evaluate_samples(data, q, **kw)
    data.force_wide = True
    b = pimc.evaluate_samples(data, q, **kw)
    data.force_wide = False
    return a, b


@pytest.mark.parametrize("quad", [None, "diag", "full"])
@pytest.mark.parametrize("A,P", [(9, 13), (10, 3), (11, 4), (12, 17)])
def test_bit_for_bit(tmp_path, A, P, quad):
    """Every size; beads that fill no step of four, samples that fill no wave, mode pairs."""
    print(f"[gpu-case] wide4 A={A} P={P} quad={quad}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(A, 3, seed=A, quad=quad, off=0.2))
    B = 2821
    data = make_data(FS, 250.0, P, B, B)
    q, _ = data.draw_host_sample(np.random.default_rng(A), B)
    q *= np.linspace(0.2, 6.0, B)[:, None, None]  # counts that differ in a wave, up to overflow
    a, b = _both(data, q)
    for k in ("s_rho", "s_g", "log_scale"):
        assert np.array_equal(a[k], b[k], equal_nan=True), k
    o = po.evaluate(oracle_setup(FS, 250.0, P), q[:40])
    assert rel_err(a["s_g"][:40], o["s_g"], floor=1e-3 * np.mean(np.abs(o["s_g"]))) < 1e-10


@pytest.mark.parametrize("A,A_rho", [(9, 12), (12, 2), (5, 11)])
def test_other_sampling_surfaces(tmp_path, A, A_rho):
    print(f"[gpu-case] wide4 A={A} A_rho={A_rho}", flush=True)
    m, rng = random_model(A, 3, seed=A), np.random.default_rng(A_rho)
    rho = {VMK.N: 3, VMK.A: A_rho, VMK.w: m[VMK.w].copy(), VMK.E: rng.uniform(0, 0.3, A_rho),
           VMK.G1: rng.normal(0, 0.05, (3, A_rho))}
    FS = stage_dict_models(tmp_path, m, rho)
    data = make_data(FS, 300.0, 10, 2816, 2816)
    q, _ = data.draw_host_sample(np.random.default_rng(A), 2816)
    a, b = _both(data, q)
    for k in ("s_rho", "s_g", "log_scale"):
        assert np.array_equal(a[k], b[k], equal_nan=True), k
