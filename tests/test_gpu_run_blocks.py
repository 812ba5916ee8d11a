"""block_compute's results come back while the next block is evaluated: blocks drawn by the caller's own
code (a subclass, an attribute) are complete before it draws the next, and what was finished before
an exception is in the result."""
import types

import numpy as np
import pytest
import torch

from helpers import make_data, random_model, stage_dict_models
from pibronic_amd import pimc

pytestmark = pytest.mark.gpu
B, BLOCKS = 20000, 5


def _data(tmp_path, A=8):
    FS = stage_dict_models(tmp_path, random_model(A, 2 * A, seed=A))
    return make_data(FS, 300.0, 32, B * BLOCKS, B)


def test_own_draw_on_another_stream(tmp_path):
    """Coordinates put in place on a stream of the caller's, which waits for that stream alone."""
    print("[gpu-case] block loop, own draw", flush=True)
    data = _data(tmp_path)
    q = [torch.as_tensor(data.draw_host_sample(np.random.default_rng(k), B)[0], device="cuda") for k in range(BLOCKS)]
    want = [pimc.evaluate_samples(data, x.cpu().numpy()) for x in q]
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    result = pimc.BoxResult(data=data)

    def draw(self, view):
        k = view.start // B
        assert not np.isnan(result.scaled_g[:view.start]).any() and np.isnan(result.scaled_g[view.start:]).all()
        with torch.cuda.stream(side):
            self.device_buffers(B)["q"].copy_(q[k])
        side.synchronize()

    data.draw_sample = types.MethodType(draw, data)
    pimc.block_compute(data, result)
    for k, w in enumerate(want):
        rows = slice(k * B, (k + 1) * B)
        assert np.array_equal(result.scaled_g[rows], w["s_g"]) and np.array_equal(result.scaled_rho[rows], w["s_rho"])


@pytest.mark.parametrize("sampler", ["device", "host"])
def test_finished_blocks_survive_an_exception(tmp_path, sampler):
    print(f"[gpu-case] block loop, exception, {sampler}", flush=True)
    data = _data(tmp_path, A=3)
    data.sampler = sampler
    whole = pimc.block_compute(data, pimc.BoxResult(data=data))

    class Stop(Exception):
        pass

    def seed(self=data):
        if seed.calls == 3:
            raise Stop
        seed.calls += 1
        return 1234

    seed.calls = -1  # one call before the first block
    data.resolve_seed = seed
    result = pimc.BoxResult(data=data)
    with pytest.raises(Stop):
        pimc.block_compute(data, result)
    assert np.array_equal(result.scaled_g[:3 * B], whole.scaled_g[:3 * B])
    assert np.isnan(result.scaled_g[3 * B:]).all()
