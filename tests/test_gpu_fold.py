"""The lanes kernels' folded form (rho the coupled model's own surface diagonal, no linear coupling
with a diagonal: each O-exponent formed once) against the general form, which the debug run takes:
bit for bit, and the general form still taken for any other rho or coupling."""
import numpy as np
import pytest

from helpers import make_data, random_model, rel_err, stage_dict_models
from pibronic_amd import _native, pimc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A,pm", [(A, pm) for A in range(1, 8) for pm in (False, True) if not (pm and A > 6)])
def test_folded_equals_general_bit_for_bit(tmp_path, A, pm):
    print(f"[gpu-case] fold A={A} pm={pm}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(A, 5, seed=50 + A, quad="diag"))
    data = make_data(FS, 300.0, 13, 100, 100, pm=pm)
    q, _ = data.draw_host_sample(np.random.default_rng(A), 100)
    a, b = pimc.evaluate_samples(data, q, pm=pm), pimc.evaluate_samples(data, q, pm=pm, debug=True)
    for k in ["s_rho", "s_g", "log_scale"] + (["s_gP", "s_gM"] if pm else []):
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("change", ["rho displacement", "linear diagonal"])
@pytest.mark.parametrize("fp32", [False, True])
def test_other_constants_take_the_general_form(tmp_path, change, fp32):
    """One displaced surface of rho, or one diagonal linear coupling, changes the results as the
    one-wave-per-sample kernel says, and only the quantity it belongs to."""
    print(f"[gpu-case] fold {change} fp32={fp32}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(4, 3, seed=9))
    data = make_data(FS, 300.0, 11, 50, 50)
    data.fp32 = fp32
    ctx, rho, vib = data.context(), data.rho, data.vib
    q, _ = data.draw_host_sample(np.random.default_rng(1), 50)
    before = pimc.evaluate_samples(data, q)
    if change == "rho displacement":
        shift = rho.state_shift.copy()
        shift[2, 1] += 0.3
        ctx.set_omatrix_set(_native.SET_RHO, rho.const.cothAN[0], rho.const.cschAN[0], rho.const.omatrix_prefactor, shift)
    else:
        L = vib.linear.copy()
        L[1, 2, 2] += 0.05
        ctx.set_coupling(vib.energy, L, vib.quadratic)
    after = pimc.evaluate_samples(data, q)
    key, other = ("s_rho", "s_g") if change == "rho displacement" else ("s_g", "s_rho")
    scale = np.exp(after["log_scale"] - before["log_scale"])
    assert np.max(np.abs(after[key] * scale / before[key] - 1)) > 1e-3
    assert rel_err(after[other] * scale, before[other]) < (1e-3 if fp32 else 1e-11)
    if not fp32:
        data.force_wide = True
        w = pimc.evaluate_samples(data, q)
        for k in ("s_rho", "s_g"):
            assert rel_err(after[k], w[k]) < 1e-11, k
