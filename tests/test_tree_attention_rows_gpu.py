"""GPU tier: tree attention at the edges of its query-row tiles (1, 15, 16,
64, 65, 128, 129 and 256 rows per KV head: one or two 16-row tiles a wave) and
of its split plan (1 to 40 key tiles), against the fp32 oracle (1e-2 abs)."""
import pytest
import torch

from cudaforge_amd import _lib, tree as T
from cudaforge_amd.verify import tree_attention, tree_attention_workspace_bytes
from tests.test_tree_attention_gpu import ATOL, _case, _oracle, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("N,Hq,Hkv", [(1, 1, 1), (15, 2, 2), (16, 4, 1), (13, 5, 1), (16, 2, 2), (32, 4, 1),
                                      (43, 3, 1), (64, 8, 2)])
@pytest.mark.parametrize("ctx", [[50, 3], [460, 301], [2500, 40]])
def test_row_and_split_edges(device, D, N, Hq, Hkv, ctx):
    q, kp, vp, bt, masks = _case(2, N, Hq, Hkv, ctx, 16, lambda b: T.binary_tree_parents(N),
                                 seed=N + Hq, D=D)
    got = _run(device, q, kp, vp, bt, ctx, masks, 16)
    want = _oracle(q, kp, vp, bt, ctx, masks, 16)
    assert (got - want).abs().max().item() <= ATOL


@pytest.mark.parametrize("ctx", [383, 447, 511])
def test_two_splits_or_one(device, ctx):
    """128 (sequence, KV head) items at 7, 8 and 9 tiles: 8 tiles and fewer
    stay in one split, 9 go to two."""
    B, N = 16, 1
    q, kp, vp, bt, masks = _case(B, N, 16, 8, [ctx] * B, 16, lambda b: T.binary_tree_parents(N), seed=ctx)
    got = _run(device, q, kp, vp, bt, [ctx] * B, masks, 16)
    want = _oracle(q, kp, vp, bt, [ctx] * B, masks, 16)
    assert (got - want).abs().max().item() <= ATOL


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("B,N,ctx", [(3, 31, [1500, 700, 1100]), (1, 8, [1080]), (2, 8, [1000, 900])])
def test_merge_of_few_splits_adds_no_error(device, D, B, N, ctx):
    """Where the automatic plan takes fewer splits than one work-group per CU,
    the partials are fp32, so the result is as close to the oracle as one split's
    (one rounding of the output), to within the sampling error of two rms
    values over n outputs, about 1 / sqrt(n) relative.  A bf16 rounding of
    four partials adds 3% to the rms."""
    q, kp, vp, bt, masks = _case(B, N, 32, 8, ctx, 16, lambda b: T.binary_tree_parents(N), seed=D + B, D=D)
    want = _oracle(q, kp, vp, bt, ctx, masks, 16).double()
    err = [(_run(device, q, kp, vp, bt, ctx, masks, 16, splits=s).double() - want).norm().item()
           for s in (0, 1)]
    assert err[0] <= err[1] * (1 + 4 / want.numel() ** 0.5), (err, want.norm().item())


@pytest.mark.parametrize("B,ctx", [(1, 312), (3, 760), (6, 1700)])
def test_smaller_workspace_takes_one_split_per_cu(device, B, ctx):
    """A workspace that holds the bf16 partials of one work-group per CU and
    not the fp32 ones gives what that split count gives, bit for bit."""
    N, D = 8, 128
    q, kp, vp, bt, masks = (x.to(device) if torch.is_tensor(x) else x for x in _case(
        B, N, 32, 8, [ctx] * B, 16, lambda b: T.binary_tree_parents(N), seed=B, D=D))
    tiles = -(-(ctx + N) // 64)
    s = -(-tiles // -(-tiles // min(tiles, -(-256 // (8 * B)))))
    need = tree_attention_workspace_bytes(B, N, 32, 8, D, ctx + N, s)
    assert need < tree_attention_workspace_bytes(B, N, 32, 8, D, ctx + N)
    lens = torch.full((B,), ctx, dtype=torch.int32, device=device)
    m = T.mask_tensor(masks, device)
    kw = dict(max_keys=ctx + N)
    want = tree_attention(q, kp, vp, bt, lens, m, num_splits=s, **kw)
    ws = torch.empty(need, dtype=torch.uint8, device=device)
    got = torch.empty_like(q)
    lib = _lib.load()
    args = (q.data_ptr(), kp.data_ptr(), vp.data_ptr(), bt.data_ptr(), bt.shape[1], lens.data_ptr(),
            kp.shape[0], 1, 0, 16, m.data_ptr(), 0, B, N, 0, 32, 8, D, D ** -0.5, ctx + N, 0,
            got.data_ptr(), ws.data_ptr())
    _lib.check(lib.cfa_tree_attention(*args, need, None), "cfa_tree_attention")
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    assert lib.cfa_tree_attention(*args, need - 256, None) == _lib.CFA_ERR_ARG
