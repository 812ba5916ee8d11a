"""BF16x3 products with more tiles than two work-groups per CU (one LDS stage), every operand order,
half stages and several stages, epilogues included: the same as few tiles at a time, bit for bit."""
import pytest
import torch

from helpers import make_data, random_model, stage_dict_models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("K", [32, 64, 96, 224])
def test_many_tiles_equal_few(tmp_path, ta, tb, K):
    print(f"[gpu-case] many product tiles ta={ta} tb={tb} K={K}", flush=True)
    FS = stage_dict_models(tmp_path, random_model(2, 3, seed=1))
    ctx = make_data(FS, 300.0, 16, 10, 10).context()
    M, N, part = 8192, 320, 1024  # 640 tiles; 80 at a time
    g = torch.Generator(device="cuda").manual_seed(K)
    rand = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    A, B = rand(K, M) if ta else rand(M, K), rand(N, K) if tb else rand(K, N)
    bias, mask, C0 = rand(N), rand(M, N), rand(M, N)
    for kw in (dict(), dict(bias=bias, relu=True), dict(accumulate=True), dict(mask=mask, ldmask=N)):
        got, want = C0.clone(), C0.clone()
        ctx.gemm_bf16x3(A, B, got, M, N, K, A.shape[1], B.shape[1], N, trans_a=ta, trans_b=tb, **kw)
        for m in range(0, M, part):
            a = A[:, m:] if ta else A[m:]
            sub = dict(kw, mask=mask[m:]) if "mask" in kw else kw
            ctx.gemm_bf16x3(a, B, want[m:], part, N, K, A.shape[1], B.shape[1], N, trans_a=ta, trans_b=tb, **sub)
        torch.cuda.synchronize()
        assert torch.equal(got, want), kw
