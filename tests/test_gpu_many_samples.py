"""More samples in one call than one launch of the block kernel has threads for (2^32, 16 per sample)."""
import numpy as np
import pytest
import torch

from helpers import make_data, random_model, stage_dict_models
from pibronic_amd import _native

pytestmark = pytest.mark.gpu


def test_more_samples_than_one_launch(tmp_path):
    print("[gpu-case] 2^28 samples of eight surfaces", flush=True)
    FS = stage_dict_models(tmp_path, random_model(8, 1, seed=8))
    n = 1 << 16
    B = (1 << 28) + 3 * 4 + 1
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 40 GB of device memory")
    data = make_data(FS, 300.0, 3, n, n)
    base = torch.as_tensor(data.draw_host_sample(np.random.default_rng(1), n)[0], device="cuda")
    want = torch.empty((_native.NUM_OUT, n), dtype=torch.float64, device="cuda")
    data.evaluate_device(base, n, False, want, n)
    q = torch.empty((B, 1, 3), dtype=torch.float64, device="cuda")
    for k in range(0, B, n):
        q[k:k + n] = base[:min(n, B - k)]
    out = torch.full((_native.NUM_OUT, B), float("nan"), dtype=torch.float64, device="cuda")
    data.evaluate_device(q, B, False, out, B)
    torch.cuda.synchronize()
    for r in (_native.OUT_RHO, _native.OUT_G, _native.OUT_LOGS):
        for k in range(0, B, n):
            assert torch.equal(out[r, k:k + n], want[r, :min(n, B - k)]), (r, k)
