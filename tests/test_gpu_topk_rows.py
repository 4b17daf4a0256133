"""Top-k over rows whose first element is at every 2- or 4-byte offset of a
16-byte line, and rows shorter than one batch of loads, against a stable
float64 sort."""
import pytest
import torch

from cast_amd import topk_marginals

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("V,k", [(50257, 8), (32000, 16), (32003, 8), (4095, 8), (4103, 5), (17, 16), (3, 3),
                                 (131073, 8)])
def test_topk_rows(gpu, V, k, dtype):
    print(f"case topk-rows V={V} k={k} {dtype}", flush=True)
    g = torch.Generator(gpu).manual_seed(V)
    x = torch.randn(19, V, generator=g, device=gpu).mul_(5).to(dtype)
    x[1, 0], x[1, V - 1] = 60.0, 60.0               # the best at both ends, tied
    x[2] = 1.0                                      # ties everywhere: the first k
    x[3, :] = -torch.inf
    x[3, V // 2] = 0.0
    for splits in (0, 1):
        idx, lp = topk_marginals(x, k, on_device=True, splits=splits)
        val, want = torch.sort(x.double(), dim=1, descending=True, stable=True)
        assert torch.equal(idx, want[:, :k])
        ref = val[:, :k] - torch.logsumexp(x.double(), dim=1, keepdim=True)
        # 32-bit x - max - log(sum): each rounding within 2^-24 of up to 60
        ok = torch.isfinite(ref)
        assert torch.equal(torch.isfinite(lp), ok)
        assert ((lp.double() - ref).abs()[ok] <= 2e-5).all()
