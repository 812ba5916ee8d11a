"""The training pass sums weight gradients over the samples in parts of 256, as the plain products it
replaces do at least: the rounding of long sums must not grow with the batch."""
import numpy as np
import pytest
import torch

from helpers import make_data, random_model, stage_dict_models
from flow_helpers import random_params, ref_for
from pibronic_amd import flow

pytestmark = pytest.mark.gpu


def _split(x):
    hi = x.bfloat16()
    return hi.double(), (x - hi.float()).bfloat16().double()


@pytest.mark.parametrize("B", [64, 320, 2048, 32768])
def test_rounding_of_long_sums(tmp_path, B):
    """The same sample B times: every partial sum grows by equal terms, whose rounding errors add up.
    Against the three bf16 products of each term summed in float64, relative to the terms' sizes: the
    24 matrix instructions of a part, four sums in each, every one rounded by up to 2^-23, and B / 256
    FP32 additions of parts."""
    print(f"[gpu-case] weight gradient sums B={B}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(3, 8, seed=8))
    data = make_data(FS, 300.0, 64, 64, 64)
    L, h = 4, 256
    fl = flow.Flow(data, layers=L, hidden=h, smax=2.0, gemm="bf16x3")
    fl.set_params(random_params(ref_for(data, L, h, 2.0), 5))
    R = torch.as_tensor(data.draw_host_sample(np.random.default_rng(1), 1)[0], device="cuda").expand(B, -1, -1).contiguous()
    assert fl._train_ok(B)
    fl.loss_and_grad(R, torch.full((B,), 1.0 / B, dtype=torch.float64, device="cuda"))
    bufs = lambda name, n: fl._buf(name, (L, B, n))  # noqa: E731
    bound = 24 * 4 * 2.0 ** -23 + max(1, B // 256) * 2.0 ** -24
    for l in range(L):
        for name, x, y in (("W3", "h2s", ("os", fl.D)), ("W2", "h1s", ("dh2s", h))):
            xh, xl = _split(bufs(x, h)[l])
            yh, yl = _split(bufs(*y)[l])
            want = xl.T @ yh + xh.T @ yl + xh.T @ yh
            size = xh.abs().T @ yh.abs()
            err = (fl.p(l, name, fl.grad).double() - want).abs()
            print(name, l, float((err / size.clamp_min(1e-300))[size > 0].max()), bound, flush=True)
            assert torch.all(err <= bound * size), (l, name)
