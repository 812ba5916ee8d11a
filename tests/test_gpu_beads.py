"""pib_set_beads stores two numbers: it neither waits for the device nor allocates, so it may be called
while evaluations are queued and inside a stream capture, for every kernel family."""
import numpy as np
import pytest
import torch

from helpers import make_data, random_model, stage_dict_models
from pibronic_amd import _native

pytestmark = pytest.mark.gpu


def _problem(tmp_path, A, pm):
    FS = stage_dict_models(tmp_path, random_model(A, 3, seed=A, quad="full"))
    B = 40000
    data = make_data(FS, 300.0, 8, B, B, pm=pm)
    q, _ = data.draw_host_sample(np.random.default_rng(A), B)
    q = torch.as_tensor(q, device="cuda")
    flags = _native.EVAL_PM if pm else 0

    def evaluate(P, tau):
        """P beads of the same rows (their first ones), at tau."""
        ctx.set_beads(P, tau)
        out = torch.zeros((_native.NUM_OUT, B), dtype=torch.float64, device="cuda")
        ctx.eval_block(q[:, :, :P].contiguous(), B, flags, out, B, None, torch.cuda.current_stream())
        return out

    ctx = data.context()
    return data, evaluate


@pytest.mark.parametrize("A,pm", [(4, False), (7, False), (7, True), (8, False), (8, True), (11, True), (12, False)])
def test_beads_set_while_evaluations_are_queued(tmp_path, A, pm):
    print(f"[gpu-case] beads A={A} pm={pm}", flush=True)
    data, evaluate = _problem(tmp_path, A, pm)
    tau = data.tau
    want = [evaluate(8, tau), evaluate(5, 0.4 * tau), evaluate(8, 1.5 * tau)]
    torch.cuda.synchronize()
    assert not torch.equal(want[0], want[2])
    torch.cuda._sleep(200_000_000)  # about 0.1 s
    done = torch.cuda.Event()
    done.record()
    got = [evaluate(8, tau), evaluate(5, 0.4 * tau), evaluate(8, 1.5 * tau)]
    assert not done.query()
    for g, w in zip(got, want):
        assert torch.equal(g, w)


@pytest.mark.parametrize("A,pm", [(4, False), (8, True), (12, False)])
def test_beads_set_inside_a_capture(tmp_path, A, pm):
    print(f"[gpu-case] beads in a capture A={A} pm={pm}", flush=True)
    data, evaluate = _problem(tmp_path, A, pm)
    tau = data.tau
    want = [evaluate(8, tau), evaluate(5, 0.4 * tau)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = [evaluate(8, tau), evaluate(5, 0.4 * tau)]
    for _ in range(3):
        for g in got:
            g.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for g, w in zip(got, want):
            assert torch.equal(g, w)
