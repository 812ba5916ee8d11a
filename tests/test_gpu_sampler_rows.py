"""The sampler's row write-out (8 or 16 beads staged per lane) and the one-launch samplers and block
sums of a batch. Draws are counter-based, so equality is bit for bit."""
import numpy as np
import pytest
import torch

from helpers import make_data, random_model, stage_dict_models
from pibronic_amd import _native
from pibronic_amd.batch import TemperatureBatch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("P", [3, 8, 16, 24, 25, 31, 32, 33, 48, 64, 77])
def test_rows_do_not_depend_on_the_block(tmp_path, P):
    """A block that fills no group of 64, at a destination off the line, equals the draws made one
    sample at a time; nothing beside it is written."""
    print(f"[gpu-case] sampler rows P={P}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(3, 3, seed=P))
    ctx = make_data(FS, 300.0, P, 100, 100).context()
    B, N = 67, 3
    buf = torch.full((B * N * P + 32,), -7.0, dtype=torch.float64, device=DEV)
    one = torch.empty((4, N, P), dtype=torch.float64, device=DEV)
    for lead in (3, 16):
        buf.fill_(-7.0)
        ctx.sample_block(9, 5, B, buf[lead:lead + B * N * P])
        got = buf[lead:lead + B * N * P].view(B, N, P)
        for i, b in enumerate((0, 15, 64, 66)):
            ctx.sample_block(9, 5 + b, 1, one[i])
            assert torch.equal(one[i], got[b]), (lead, b)
        assert torch.all(got != -7.0) and len(torch.unique(got)) > 0.99 * got.numel()
        assert torch.all(buf[:lead] == -7.0) and torch.all(buf[lead + B * N * P:] == -7.0)


@pytest.mark.parametrize("P", [48, 61, 96, 129])
def test_long_runs_off_the_line(tmp_path, P):
    """More than 256 MB of rows off the line (32 beads staged): the draws of smaller launches."""
    print(f"[gpu-case] sampler long runs P={P}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(2, 3, seed=P))
    ctx = make_data(FS, 300.0, P, 100, 100).context()
    N, lead = 3, 1
    B = (270 << 20) // (8 * N * P) + 5
    buf = torch.full((B * N * P + 8,), -7.0, dtype=torch.float64, device=DEV)
    got = buf[lead:lead + B * N * P].view(B, N, P)
    ctx.sample_block(9, 5, B, got)
    part = torch.empty((100, N, P), dtype=torch.float64, device=DEV)
    for first in (0, 63, B - 100):
        ctx.sample_block(9, 5 + first, 100, part)
        assert torch.equal(part, got[first:first + 100]), first
    assert torch.all(got != -7.0) and buf[0] == -7.0 and torch.all(buf[lead + B * N * P:] == -7.0)


@pytest.mark.parametrize("n", [1, 3, 18])
def test_batched_samplers_and_sums_are_the_single_ones(tmp_path, n):
    """Problems of rising P (one and two launches' worth): draws and sums of every problem and
    block equal its own launches'."""
    print(f"[gpu-case] batched samplers n={n}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(3, 4, seed=2))
    B, seed = 130, 11
    datas = [make_data(FS, 300.0 + 10 * i, 9 + 5 * i, B, B) for i in range(n)]
    tb = TemperatureBatch(datas, B, max_blocks=2)
    tb.run(seed, first_block=0, nblocks=2)
    got = tb.block_sums()
    sched = tb.schedule()
    for i, d in enumerate(datas):
        ctx = d.context()
        if sched["family"] == "wide":
            d.force_wide = True
        else:
            ctx.set_lanes_per_sample(sched["lanes"][i])
        q = torch.empty((B, d.modes, d.beads), dtype=torch.float64, device=DEV)
        out = torch.empty((_native.NUM_OUT, B), dtype=torch.float64, device=DEV)
        sums = torch.zeros(_native.NUM_SUMS, dtype=torch.float64, device=DEV)
        for k in range(2):
            ctx.sample_block(seed, k * B, B, q)
            d.evaluate_device(q, B, False, out, B)
            ctx.block_sums(out, B, B, False, 1.0, sums)
            torch.cuda.synchronize()
            assert np.allclose(got[k, i], sums.cpu().numpy(), rtol=1e-12, atol=0), (i, k)
