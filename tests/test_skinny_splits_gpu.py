"""GPU tier: cfa_gemm_bf16_skinny at split counts that are not a multiple of
the splits summed at once (four, two above 64 rows), against a float64
product: one bf16 rounding of the output (2^-8 relative) plus 2^-14 of
|a| @ |w| for the fp32 order of the sums."""
import pytest
import torch

from cudaforge_amd.spec_step import skinny_gemm, skinny_gemm_workspace_bytes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [7, 30, 64, 65, 128])
@pytest.mark.parametrize("splits", [3, 5, 6, 10, 30])
def test_split_remainders(device, M, splits):
    N, K = 128, 30 * 128
    g = torch.Generator().manual_seed(M + splits)
    a = torch.randn(M, K, generator=g).bfloat16()
    w = (torch.randn(K, N, generator=g) / K ** 0.5).bfloat16()
    ws = torch.zeros(skinny_gemm_workspace_bytes(M, N, K, splits), dtype=torch.uint8, device=device)
    out = skinny_gemm(a.to(device), w.to(device), ws, splits=splits).double().cpu()
    ref = a.double() @ w.double()
    bound = ref.abs() * 2.0 ** -8 + (a.double().abs() @ w.double().abs()) * 2.0 ** -14
    assert bool(((out - ref).abs() <= bound).all())
