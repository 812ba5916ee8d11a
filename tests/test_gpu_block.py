"""The block kernel (4 x 4 matrix blocks, four bead streams per wave), which pib_eval_block takes
at A = 8, from A = 7 on with +-dbeta and for surface counts without a lanes kernel: every compiled
size against the oracle, and against the one-wave-per-sample kernel (PIB_EVAL_WIDE) over everything
both accept. Tolerances are those of the other FP64 kernels: 1e-10 relative to the oracle, 1e-11
between two FP64 kernels on the same coordinates."""
import numpy as np
import pytest
import torch

from helpers import make_data, oracle_setup, random_model, rel_err, stage_dict_models
from oracle import pimc_oracle as po
from pibronic_amd import _native, pimc
from pibronic_amd.batch import TemperatureBatch
from pibronic_amd.vibronic_model_keys import VibronicModelKeys as VMK

pytestmark = pytest.mark.gpu

KEYS = ["s_rho", "s_g"]
KEYS_PM = KEYS + ["s_gP", "s_gM"]


def _announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


def _wide(data, q, **kw):
    data.force_wide = True
    try:
        return pimc.evaluate_samples(data, q, **kw)
    finally:
        data.force_wide = False


def _close(a, b, keys, tol):
    # relative to each sample, down to a thousandth of the mean (a trace that cancels says nothing)
    for k in keys:
        assert rel_err(a[k], b[k], floor=1e-3 * np.mean(np.abs(b[k]))) < tol, k
    assert np.max(np.abs(a["log_scale"] - b["log_scale"])) < 1e-9 * max(1.0, np.max(np.abs(b["log_scale"])))


@pytest.mark.parametrize("pm", [False, True])
@pytest.mark.parametrize("A", [7, 8, 9, 10, 11, 12, 13, 14, 15, 16])
def test_sizes_against_oracle(tmp_path, A, pm):
    """Every size, with modes, beads and samples that fill no tile (N = 3, P = 9, B = 7) and full
    (j != k) quadratic couplings; the debug run gives the same outputs bit for bit."""
    _announce(f"block A={A} pm={pm}")
    FS = stage_dict_models(tmp_path, random_model(A, 3, seed=40 + A, quad="full"))
    data = make_data(FS, 300.0, 9, 7, 7, pm=pm)
    q, _ = data.draw_host_sample(np.random.default_rng(A), 7)
    r = pimc.evaluate_samples(data, q, pm=pm)
    o = po.evaluate(oracle_setup(FS, 300.0, 9), q, pm=pm, keep=True)
    keys = KEYS_PM if pm else KEYS
    _close(r, o, keys, 1e-10)
    d = pimc.evaluate_samples(data, q, pm=pm, debug=True)
    for k in keys + ["log_scale"]:
        assert np.array_equal(d[k], r[k]), k
    err = np.max(np.abs(d["M"] - o["M"]), axis=(2, 3)) / np.max(np.abs(o["M"]), axis=(2, 3))
    assert err.max() < 1e-12
    S = d["S"][..., None]
    assert rel_err(d["O_vib"] / S, np.diagonal(o["O_vib"], axis1=2, axis2=3)) < 1e-11
    assert rel_err(d["O_rho"] / S, np.diagonal(o["O_rho"], axis1=2, axis2=3)) < 1e-11


@pytest.mark.parametrize("A,AR", [(5, 7), (3, 7), (8, 3), (6, 16), (9, 12), (16, 1)])
def test_other_surface_count_of_the_sampling_model(tmp_path, A, AR):
    _announce(f"block A={A} A_rho={AR}")
    m = random_model(A, 3, seed=7)
    rng = np.random.default_rng(AR)
    rho = {VMK.N: 3, VMK.A: AR, VMK.w: m[VMK.w].copy(), VMK.E: rng.uniform(0, 0.3, AR),
           VMK.G1: rng.normal(0, 0.05, (3, AR))}
    FS = stage_dict_models(tmp_path, m, rho)
    data = make_data(FS, 300.0, 10, 30, 30, pm=True)
    q, _ = data.draw_host_sample(np.random.default_rng(3), 30)
    _close(pimc.evaluate_samples(data, q, pm=True), po.evaluate(oracle_setup(FS, 300.0, 10), q, pm=True), KEYS_PM, 1e-10)


@pytest.mark.parametrize("A,pm", [(8, False), (9, True), (13, True)])
@pytest.mark.parametrize("B,P", [(1, 3), (5, 4), (9001, 5), (40003, 6)])
def test_streams_per_sample(tmp_path, A, pm, B, P):
    """From the smallest launch (four streams per sample) to one stream per sample, with a last
    wave that is not full, fewer beads than streams' steps, and no quadratic couplings."""
    _announce(f"block streams A={A} B={B} P={P}")
    FS = stage_dict_models(tmp_path, random_model(A, 2, seed=A, quad=None))
    data = make_data(FS, 300.0, P, B, B, pm=pm)
    q, _ = data.draw_host_sample(np.random.default_rng(B), B)
    keys = KEYS_PM if pm else KEYS
    _close(pimc.evaluate_samples(data, q, pm=pm), _wide(data, q, pm=pm), keys, 1e-11)
    a = pimc.evaluate_samples(data, q, pm=pm, noscale=True)
    _close(a, _wide(data, q, pm=pm, noscale=True), keys, 1e-11)
    assert np.all(a["log_scale"] == 0.0)


@pytest.mark.parametrize("A", [8, 12, 16])
def test_linear_couplings_with_a_diagonal(tmp_path, A):
    """Constants given straight to the context, with diagonal linear couplings (folded models have
    none), six modes and a coupling with off-diagonal mode pairs."""
    _announce(f"block linear diagonal A={A}")
    FS = stage_dict_models(tmp_path, random_model(A, 6, seed=A, quad="full"))
    data = make_data(FS, 300.0, 7, 20, 20, pm=True)
    ctx = data.context()
    vib = data.vib
    L = vib.linear + np.random.default_rng(1).normal(0.0, 0.05, (6, A))[:, :, None] * np.eye(A)
    ctx.set_coupling(vib.energy, L, vib.quadratic)
    q, _ = data.draw_host_sample(np.random.default_rng(2), 20)
    _close(pimc.evaluate_samples(data, q, pm=True), _wide(data, q, pm=True), KEYS_PM, 1e-11)


def test_sets_given_after_the_beads(tmp_path):
    """The +-dbeta sets (or new couplings) may come after the beads: constants follow the last
    call, and a plain evaluation does not need the +-dbeta sets."""
    _announce("block order of setters")
    FS = stage_dict_models(tmp_path, random_model(9, 3, seed=2))
    data = make_data(FS, 300.0, 8, 10, 10, pm=True)
    q, _ = data.draw_host_sample(np.random.default_rng(2), 10)
    want = pimc.evaluate_samples(data, q, pm=True)
    vib, rho = data.vib, data.rho
    ctx = _native.Context(0)
    out = torch.full((_native.NUM_OUT, 10), float("nan"), dtype=torch.float64, device="cuda")
    qd = torch.from_numpy(q).cuda()
    ctx.set_beads(8, data.tau)
    for slot, c, m in ((_native.SET_VIB, vib.const, vib), (_native.SET_RHO, rho.const, rho)):
        ctx.set_omatrix_set(slot, c.cothAN[0], c.cschAN[0], c.omatrix_prefactor, m.state_shift)
    ctx.set_coupling(vib.energy, vib.linear, vib.quadratic)
    ctx.eval_block(qd, 10, 0, out, 10)
    torch.cuda.synchronize()
    assert np.array_equal(out[_native.OUT_G].cpu().numpy(), pimc.evaluate_samples(data, q, pm=False)["s_g"])
    with pytest.raises(_native.NativeError, match="not set"):
        ctx.eval_block(qd, 10, _native.EVAL_PM, out, 10)
    for slot, c in ((_native.SET_VIB_PLUS, vib.const_plus), (_native.SET_VIB_MINUS, vib.const_minus)):
        ctx.set_omatrix_set(slot, c.cothAN[0], c.cschAN[0], c.omatrix_prefactor, vib.state_shift)
    ctx.eval_block(qd, 10, _native.EVAL_PM, out, 10)
    torch.cuda.synchronize()
    for k, row in (("s_g", _native.OUT_G), ("s_gP", _native.OUT_GP), ("s_gM", _native.OUT_GM)):
        assert np.array_equal(out[row].cpu().numpy(), want[k]), k


def test_zero_prefactor_keeps_its_kernel(tmp_path):
    """An O-matrix prefactor of exactly 0 (underflow) has no logarithm: the one-wave-per-sample
    kernel, which works with the factors themselves, still takes it."""
    _announce("block zero prefactor")
    FS = stage_dict_models(tmp_path, random_model(9, 3, seed=2))
    data = make_data(FS, 300.0, 8, 10, 10, pm=True)
    pref = data.vib.const.omatrix_prefactor.copy()
    pref[4] = 0.0
    data.context().set_omatrix_set(_native.SET_VIB, data.vib.const.cothAN[0], data.vib.const.cschAN[0], pref,
                                   data.vib.state_shift)
    q, _ = data.draw_host_sample(np.random.default_rng(2), 10)
    a, b = pimc.evaluate_samples(data, q, pm=True), _wide(data, q, pm=True)
    assert np.all(np.isfinite(a["s_g"]))
    for k in KEYS_PM + ["log_scale"]:
        assert np.array_equal(a[k], b[k]), k


def test_a_bad_sample_stays_alone(tmp_path):
    """Samples share a wave: NaN and infinite coordinates of one reach no other's outputs."""
    _announce("block NaN coordinates")
    FS = stage_dict_models(tmp_path, random_model(10, 3, seed=4))
    B = 20000  # one stream per sample
    data = make_data(FS, 300.0, 6, B, B, pm=True)
    q, _ = data.draw_host_sample(np.random.default_rng(2), B)
    clean = pimc.evaluate_samples(data, q, pm=True)
    bad = q.copy()
    bad[5, 2, 3] = np.nan
    bad[11, 0, 0] = np.inf
    r = pimc.evaluate_samples(data, bad, pm=True)
    keep = np.ones(B, dtype=bool)
    keep[[5, 11]] = False
    for k in KEYS_PM + ["log_scale"]:
        assert np.array_equal(r[k][keep], clean[k][keep]), k
    assert np.isnan(r["s_g"][5])


def test_batch_runs_them_one_launch_each(tmp_path):
    """Temperatures of a model of this kernel: the batch's schedule is one launch per problem, with
    the outputs of single evaluations bit for bit."""
    _announce("block batch")
    FS = stage_dict_models(tmp_path, random_model(8, 3, seed=6, quad="diag"))
    B = 96
    datas = [make_data(FS, T, P, B, B, pm=True) for T, P in [(200.0, 21), (400.0, 10)]]
    tb = TemperatureBatch(datas, B)
    assert tb.schedule()["family"] == "sequential"
    qs = [d.draw_host_sample(np.random.default_rng(i), B)[0] for i, d in enumerate(datas)]
    for res, d, q in zip(tb.evaluate(qs), datas, qs):
        single = pimc.evaluate_samples(d, q, pm=True)
        for k in KEYS_PM + ["log_scale"]:
            assert np.array_equal(res[k], single[k]), k


@pytest.mark.parametrize("A,pm,P", [(5, True, 7), (6, True, 9), (7, False, 6)])
def test_small_batches_of_lanes_sizes(tmp_path, A, pm, P):
    """Sizes with a lanes kernel that small batches take to the block kernel: both against each other
    on the same samples (set lanes per sample keep the lanes kernel), and the larger batch that stays
    with the lanes kernel, bit for bit what its own lanes give."""
    _announce(f"block small batches A={A} pm={pm}")
    FS = stage_dict_models(tmp_path, random_model(A, 2, seed=A, quad="full"))
    data = make_data(FS, 300.0, P, 300, 300, pm=pm)
    q, _ = data.draw_host_sample(np.random.default_rng(A), 300)
    keys = KEYS_PM if pm else KEYS
    block = pimc.evaluate_samples(data, q, pm=pm)
    _close(block, po.evaluate(oracle_setup(FS, 300.0, P), q, pm=pm), keys, 1e-10)
    ctx = data.context()
    ctx.set_lanes_per_sample(4)
    lanes = pimc.evaluate_samples(data, q, pm=pm)
    _close(block, lanes, keys, 1e-11)
    big = np.concatenate([q] * 220)  # 66,000 samples
    a = pimc.evaluate_samples(data, big, pm=pm)
    ctx.set_lanes_per_sample(ctx.lanes_per_sample(len(big)))
    b = pimc.evaluate_samples(data, big, pm=pm)
    for k in keys:
        assert np.array_equal(a[k], b[k]), k
        assert np.array_equal(a[k][:300], lanes[k]), k
