"""The training pass in three launches per layer and direction against the layer-by-layer path, and
the FP32-accurate product tiles at the edges of their stages."""
import numpy as np
import pytest
import torch

from helpers import make_data, random_model, stage_dict_models
from flow_helpers import random_params, ref_for
from pibronic_amd import flow

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("N,hidden,layers,B", [(2, 64, 2, 64), (4, 128, 3, 192), (8, 512, 2, 128), (16, 256, 9, 64),
                                               (6, 192, 4, 1024), (16, 256, 8, 2048)])
def test_training_pass_matches_layer_by_layer(tmp_path, N, hidden, layers, B):
    """The forward makes the same products in the same order: the loss to 1e-12. The gradients' sums
    over samples are regrouped: to 64 roundings of FP32 (4e-6) in norm, each parameter block."""
    print(f"[gpu-case] training pass N={N} hidden={hidden} L={layers} B={B}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(3, N, seed=N))
    data = make_data(FS, 300.0, 64, B, B)
    fl = flow.Flow(data, layers=layers, hidden=hidden, smax=2.0, gemm="bf16x3")
    fl.set_params(random_params(ref_for(data, layers, hidden, 2.0), 5))
    R = torch.as_tensor(data.draw_host_sample(np.random.default_rng(1), B)[0], device=DEV)
    c = torch.softmax(torch.linspace(-1.0, 1.0, B, dtype=torch.float64, device=DEV), dim=0)
    assert fl._train_ok(B)
    fl.grad.fill_(float("nan"))
    loss, grad = float(fl.loss_and_grad(R, c)), fl.grad.clone()
    assert float(fl.loss_and_grad(R, c)) == loss and torch.equal(grad, fl.grad)
    fl._train_ok = lambda B: False
    want = float(fl.loss_and_grad(R, c))
    assert abs(loss - want) <= 1e-12 * abs(want)
    for l in range(layers):
        for name, _ in fl.shapes:
            g, w = fl.p(l, name, grad).double(), fl.p(l, name, fl.grad).double()
            assert torch.linalg.norm(g - w) <= 4e-6 * torch.linalg.norm(w), (l, name)


@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("K", [32, 64, 96, 160, 512])
def test_product_stages(tmp_path, ta, tb, K):
    """Half stages, one stage, and the two-way split of K, every operand order, inside wider rows.
    Per product term 3 x 2^-16 of the operands' split and K roundings of the sum."""
    print(f"[gpu-case] product ta={ta} tb={tb} K={K}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(2, 3, seed=1))
    ctx = make_data(FS, 300.0, 16, 10, 10).context()
    M, N = 128, 192
    g = torch.Generator().manual_seed(K)
    A = torch.randn((K, M + 4) if ta else (M, K + 4), generator=g)
    Bm = torch.randn((N, K + 8) if tb else (K, N + 8), generator=g)
    Ad, Bd = A.to(DEV), Bm.to(DEV)
    C = torch.full((M, N), float("nan"), device=DEV)
    ctx.gemm_bf16x3(Ad, Bd, C, M, N, K, A.shape[1], Bm.shape[1], N, trans_a=ta, trans_b=tb)
    torch.cuda.synchronize()
    a = (A[:, :M].T if ta else A[:, :K]).double()
    b = (Bm[:, :K].T if tb else Bm[:, :N]).double()
    tol = (3 * 2.0 ** -16 + K * 2.0 ** -24) * (a.abs() @ b.abs())
    assert torch.all((C.cpu().double() - a @ b).abs() <= tol)


@pytest.mark.parametrize("N,B", [(16, 82048), (8, 164096)])
def test_pieces_of_a_large_draw(tmp_path, N, B):
    """Just beyond the size from which draws are taken in pieces, with a last piece that is no whole
    launch: draws and offsets are those of the whole batch bit for bit."""
    print(f"[gpu-case] pieces N={N} B={B}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(2, N, seed=N))
    data = make_data(FS, 300.0, 64, 128, 128)
    fl = flow.Flow(data, layers=3, hidden=256, smax=2.0, gemm="bf16x3")
    fl.set_params(random_params(ref_for(data, 3, 256, 2.0), 5))
    fl.draw_precision = "bf16"
    assert len(fl._chunks(B)) > 1
    got = [fl.draw(B, 7, 3, offsets=True), fl.draw(B, 7, 3)]
    fl._chunks = lambda B: [slice(0, B)]
    want = [fl.draw(B, 7, 3, offsets=True), fl.draw(B, 7, 3)]
    for g, w in zip(got, want):
        assert torch.equal(g[0], w[0]) and torch.equal(g[1], w[1])
