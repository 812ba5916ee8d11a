"""The folded instances that test_gpu_fold.py cannot reach (FP32 and the persistent batched kernel, at
every surface count) against the general ones, bit for bit. A diagonal linear coupling of 1e-300, which no
sum beside ordinary terms feels, makes a problem take the general form."""
import numpy as np
import pytest

from helpers import make_data, random_model, stage_dict_models
from pibronic_amd import pimc
from pibronic_amd.batch import TemperatureBatch

pytestmark = pytest.mark.gpu


def _general(data):
    vib = data.vib
    L = vib.linear + 1e-300 * np.eye(data.states)
    data.context().set_coupling(vib.energy, L, vib.quadratic)
    return data


def _keys(pm):
    return ["s_rho", "s_g", "log_scale"] + (["s_gP", "s_gM"] if pm else [])


@pytest.mark.parametrize("pm", [False, True])
@pytest.mark.parametrize("A", range(1, 9))
def test_fp32(tmp_path, A, pm):
    print(f"[gpu-case] folded FP32 A={A} pm={pm}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(A, 5, seed=60 + A, quad="diag"))
    a, b = (make_data(FS, 300.0, 13, 100, 100, pm=pm) for _ in range(2))
    a.fp32 = b.fp32 = True
    q, _ = a.draw_host_sample(np.random.default_rng(A), 100)
    folded, general = pimc.evaluate_samples(a, q, pm=pm), pimc.evaluate_samples(_general(b), q, pm=pm)
    for k in _keys(pm):
        assert np.array_equal(folded[k], general[k]), k


@pytest.mark.parametrize("pm", [False, True])
@pytest.mark.parametrize("A", range(2, 9))
def test_batched(tmp_path, A, pm):
    print(f"[gpu-case] folded batch A={A} pm={pm}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(A, 5, seed=70 + A, quad="diag"))
    B, TP = 70, [(200.0, 21), (400.0, 10)]
    res = []
    for general in (False, True):
        datas = [make_data(FS, T, P, B, B, pm=pm) for T, P in TP]
        if general:
            datas = [_general(d) for d in datas]
        tb = TemperatureBatch(datas, B)
        tb.set_schedule("lanes", [4, 2])
        res.append(tb.evaluate([d.draw_host_sample(np.random.default_rng(i), B)[0] for i, d in enumerate(datas)]))
    for folded, general in zip(*res):
        for k in _keys(pm):
            assert np.array_equal(folded[k], general[k]), k
