"""pib_eval_block_flow_offsets gives pib_eval_block's outputs on the same coordinates bit for bit, at
every surface count and on both sides of the batch size at which seven surfaces change their kernel."""
import numpy as np
import pytest
import torch

from helpers import make_data, random_model, stage_dict_models
from pibronic_amd import _native, flow

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A", range(1, 9))
@pytest.mark.parametrize("B", [3, 500, 45000])
@pytest.mark.parametrize("lanes", [0, 4])
def test_offsets_equal_coordinates(tmp_path, A, B, lanes):
    print(f"[gpu-case] offsets A={A} B={B} lanes={lanes}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(A, 2, seed=A, quad="full"))
    data = make_data(FS, 300.0, 64, B, B)
    flow.Flow(data, layers=2, hidden=64)  # sets the basis and its centre
    data.context().set_lanes_per_sample(lanes)
    m = torch.as_tensor(data.rho.state_weight @ data.rho.state_shift, device="cuda")
    q, _ = data.draw_host_sample(np.random.default_rng(A), B)
    dq = (torch.as_tensor(q, device="cuda") - m[:, None]).float()
    out = torch.full((2, _native.NUM_OUT, B), float("nan"), dtype=torch.float64, device="cuda")
    data.evaluate_offsets_device(dq, B, out[0], B)
    data.evaluate_device(m[:, None] + dq.double(), B, False, out[1], B)
    torch.cuda.synchronize()
    rows = [_native.OUT_RHO, _native.OUT_G, _native.OUT_LOGS]
    assert torch.isfinite(out[1, rows]).all()
    assert torch.equal(out[0, rows], out[1, rows])
