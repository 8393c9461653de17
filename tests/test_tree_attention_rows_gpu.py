"""GPU tier: tree attention at the edges of its query-row tiles (1, 15, 16,
64, 65, 128, 129 and 256 rows per KV head: one or two 16-row tiles a wave) and
of its split plan (1 to 40 key tiles), against the fp32 oracle (1e-2 abs)."""
import pytest

from cudaforge_amd import tree as T
from tests.test_tree_attention_gpu import ATOL, _case, _oracle, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("N,Hq,Hkv", [(1, 1, 1), (15, 2, 2), (16, 4, 1), (13, 5, 1), (32, 4, 1),
                                      (43, 3, 1), (64, 8, 2)])
@pytest.mark.parametrize("ctx", [[50, 3], [460, 301], [2500, 40]])
def test_row_and_split_edges(device, D, N, Hq, Hkv, ctx):
    q, kp, vp, bt, masks = _case(2, N, Hq, Hkv, ctx, 16, lambda b: T.binary_tree_parents(N),
                                 seed=N + Hq, D=D)
    got = _run(device, q, kp, vp, bt, ctx, masks, 16)
    want = _oracle(q, kp, vp, bt, ctx, masks, 16)
    assert (got - want).abs().max().item() <= ATOL
