"""The ring-summed log rho of the learned proposal and its gradient, over surface counts (each
compiled size and its edges) and bead counts around the wave."""
import numpy as np
import pytest
import torch

from flow_helpers import ref_for
from helpers import make_data, random_model, stage_dict_models

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("A", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("P", [3, 64, 65, 130])
def test_log_rho_and_gradient(tmp_path, A, P):
    """log rho to 1e-10; the gradient, stored in float32, to two of its roundings (1.2e-7) down to
    1e-9 of the sample's largest component."""
    print(f"[gpu-case] log rho A={A} P={P}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(A, 5, seed=A))
    data = make_data(FS, 300.0, P, 7, 7)
    ctx, ref = data.context(), ref_for(data, 1, 8, 2.0)
    q = torch.as_tensor(data.draw_host_sample(np.random.default_rng(P), 7)[0])
    c = torch.linspace(0.5, 2.0, 7, dtype=torch.float64)
    R, cd = q.to(DEV), c.to(DEV)
    lr = torch.empty(7, dtype=torch.float64, device=DEV)
    lr2 = torch.empty_like(lr)
    dR = torch.empty(q.shape, dtype=torch.float32, device=DEV)
    ctx.flow_logrho(7, R, logrho=lr)
    ctx.flow_logrho(7, R, c=cd, dR=dR, logrho=lr2)
    torch.cuda.synchronize()
    x = q.clone().requires_grad_(True)
    want = ref.log_rho(x)
    grad = torch.autograd.grad(-(c * want).sum(), x)[0]
    assert torch.equal(lr, lr2)
    assert torch.allclose(lr.cpu(), want.detach(), rtol=1e-13, atol=1e-10)
    err = (dR.cpu().double() - grad).abs()
    tol = 1.2e-7 * grad.abs() + 1e-9 * grad.abs().amax(dim=(1, 2), keepdim=True)
    assert torch.all(err <= tol), float((err / tol).max())
