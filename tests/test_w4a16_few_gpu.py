"""GPU tier: the few-row W4A16 GEMM (cfa_w4a16_gemm_few, reached through
int4_gemm_dequant and cfa_w4a16_gemm_zp) against a float64 product of the
bit-exact dequantised weights.  Tolerance: fp32 accumulation in another
order, K * 2^-24 of sum |a| |w|, plus one rounding to the output type."""
import pytest
import torch

from cudaforge_amd import _lib
from cudaforge_amd.w4a16 import int4_gemm_dequant, w4a16_dequant, w4a16_gemm_zp

pytestmark = pytest.mark.gpu


def _problem(M, N, K, group, dtype, zeros, device, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(M, K, generator=g).to(dtype).to(device)
    q = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 8, N), generator=g, dtype=torch.int32).to(device)
    s = ((torch.rand(K // group, N, generator=g) + 0.5) / K ** 0.5).half().to(device)
    z = (torch.rand(K // group, N, generator=g) * 15).half().to(device) if zeros else None
    return a, q, s, z


def _check(c, a, q, s, z, group):
    w = w4a16_dequant(q, s, z, group_size=group, dtype=a.dtype).double()
    ref, mag = a.double() @ w, a.double().abs() @ w.abs()
    ulp = 2.0 ** -11 if a.dtype == torch.float16 else 2.0 ** -8
    tol = a.shape[1] * 2.0 ** -24 * mag + ulp * ref.abs() + 1e-6
    err = (c.double() - ref).abs()
    assert (err <= tol).all(), (err - tol).max().item()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,group,zeros", [
    (1, 128, 128, 128, False), (1, 14336, 4096, 128, True), (15, 256, 384, 32, True),
    (16, 1152, 2048, 64, False), (17, 128, 128, 32, True), (32, 384, 1152, 128, True),
    (33, 256, 640, 64, True), (63, 4096, 4096, 128, False), (64, 512, 14336, 256, True),
    (65, 128, 256, 128, True), (127, 640, 3200, 128, False), (128, 6144, 4096, 128, True)])
def test_few_rows_vs_float64(device, dtype, M, N, K, group, zeros):
    """Edges of the row tiles (16, 32, 64, 128), one column tile and counts
    not a multiple of 8, one pipeline step, odd step counts, split K, every
    group size in steps of 32."""
    a, q, s, z = _problem(M, N, K, group, dtype, zeros, device, M + N + K)
    c = int4_gemm_dequant(a, q, s, z, group_size=group)
    _check(c, a, q, s, z, group)
    assert torch.equal(c, int4_gemm_dequant(a, q, s, z, group_size=group))


@pytest.mark.parametrize("M,N,K", [(7, 512, 1024), (40, 28672, 4096), (100, 768, 2048),
                                   (9, 256, 96), (50, 256, 160)])
def test_zp_entry_same_weights(device, M, N, K):
    """cfa_w4a16_gemm_zp's route for few rows (and, K % 128 != 0, not)."""
    a, q, s, z = _problem(M, N, K, 32, torch.bfloat16, True, device, K)
    _check(w4a16_gemm_zp(a, q, s, z, group_size=32), a, q, s, z, 32)


def test_other_calls_keep_their_path(device):
    """Rows that need a gradient, strided rows, mapped and autocast calls go
    through dequantise + GEMM, and give the same product."""
    a, q, s, z = _problem(8, 256, 256, 128, torch.float16, True, device, 1)
    want = int4_gemm_dequant(a, q, s, z)
    x = a.clone().requires_grad_()
    y = int4_gemm_dequant(x, q, s, z)
    y.float().sum().backward()
    assert y.requires_grad and x.grad is not None
    assert torch.allclose(y.detach(), want, atol=2e-3, rtol=2e-3)
    wide = torch.zeros(8, 512, dtype=torch.float16, device=device)
    wide[:, ::2] = a
    assert torch.allclose(int4_gemm_dequant(wide[:, ::2], q, s, z), want, atol=2e-3, rtol=2e-3)
    v = torch.func.vmap(lambda r: int4_gemm_dequant(r, q, s, z))(a.view(2, 4, 256))
    assert torch.allclose(v.reshape(8, 256), want, atol=2e-3, rtol=2e-3)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert int4_gemm_dequant(a, q, s, z).dtype == torch.bfloat16
    with pytest.raises(ValueError):
        int4_gemm_dequant(a, q, s.float(), z)
    lib = _lib.load()
    assert lib.cfa_w4a16_gemm_few_workspace_size(129, 256, 256) == 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(128, 256, 256), (129, 256, 256), (5, 192, 256), (130, 192, 256), (5, 256, 192)])
def test_both_sides_of_the_row_and_column_rules(device, dtype, M, N, K):
    """128 and 129 rows, column counts and depths that are no multiple of 128
    (the dequantised product): the same tolerance on every route, the library
    product's sums included."""
    a, q, s, z = _problem(M, N, K, 64, dtype, True, device, M + N)
    _check(int4_gemm_dequant(a, q, s, z, group_size=64), a, q, s, z, 64)


def test_traces_and_function_modes_see_the_product(device):
    """A recorded trace holds the product of its input (an opaque kernel's
    output would be left out), and a function mode is called for it; a device
    context is no such mode."""
    from torch.overrides import TorchFunctionMode

    a, q, s, z = _problem(4, 256, 256, 128, torch.float16, True, device, 2)
    want = int4_gemm_dequant(a, q, s, z)
    traced = torch.jit.trace(lambda x: int4_gemm_dequant(x, q, s, z), (a,), check_trace=False)
    assert "aten::matmul" in str(traced.graph) or "aten::mm" in str(traced.graph)

    class Seen(TorchFunctionMode):
        names = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.names.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))

    with Seen():
        got = int4_gemm_dequant(a, q, s, z)
    assert any("matmul" in n for n in Seen.names), Seen.names
    assert torch.allclose(got, want, atol=2e-3, rtol=2e-3)
    with torch.device(device):
        assert torch.equal(int4_gemm_dequant(a, q, s, z), want)
