"""GPU tier: the kept probabilities of the filtered sampler (hist_kernel,
select_kernel and the draw over kept entries) against the oracle, token by
token: row lengths on both sides of the one-work-group path (24 chunks of
1024), more keys in one histogram bin than a row's list holds, probabilities
of 2 and above (the open last bin), zeros, and rules at their extremes."""
import numpy as np
import pytest
import torch

from cudaforge_amd.sampling import sample
from oracle import oracle as O

pytestmark = pytest.mark.gpu

LAST = float(np.float32(1.0) - np.float32(2.0 ** -24))


def _rows(kind, R, V):
    g = torch.Generator().manual_seed(R * 131 + V)
    if kind == "normal":
        return 2.0 * torch.randn(R, V, generator=g)
    if kind == "levels":                    # four probabilities, V / 4 entries each
        return 0.1 * torch.randint(0, 4, (R, V), generator=g).float()
    if kind == "peaked":
        x = torch.randn(R, V, generator=g)
        x[:, V // 2] += 30.0
        return x
    assert kind == "probs"                  # not normalised, some zero, some above 2
    x = torch.rand(R, V, generator=g) * 4.0
    x[:, ::3] = 0.0
    return x / V if V > 2000 else x


@pytest.mark.parametrize("top_p,top_k", [(0.9, 0), (0.9, 50), (1.0, 1), (1e-6, 0), (0.99999, 0),
                                         (0.5, -1), (1.0, 10 ** 6), (0.999, 3000)])
@pytest.mark.parametrize("kind,R,V", [("normal", 2, 1), ("normal", 3, 1000), ("normal", 2, 23552),
                                      ("normal", 2, 23553), ("normal", 2, 128256),
                                      ("levels", 2, 128256), ("levels", 2, 20000),
                                      ("peaked", 2, 32000), ("probs", 2, 1500),
                                      ("probs", 2, 50001)])
def test_filtered_draws(device, kind, R, V, top_p, top_k):
    x = _rows(kind, R, V).float()
    u = torch.rand(R, 4, generator=torch.Generator().manual_seed(V))
    u[:, 0], u[:, 1] = 0.0, LAST            # the first and the last kept entry
    tok, p = sample(x.to(device), mode="filtered", temperature=0.8, top_p=top_p, top_k=top_k,
                    draws=4, uniforms=u.to(device), return_probs=True,
                    input_kind="probs" if kind == "probs" else "logits")
    tok, p = tok.cpu().numpy(), p.cpu().numpy()
    for r in range(R):
        for d in range(4):
            want = O.sample_filtered(p[r], float(u[r, d]), top_p, top_k)
            assert tok[r, d] == want, (r, d, tok[r, d], want)


def test_filtered_many_rows_repeat(device):
    """More rows than histogram work-groups share out, twice the same."""
    x = _rows("normal", 300, 30011).to(device)
    u = torch.rand(300, 1, device=device)
    a = sample(x, mode="filtered", top_p=0.9, uniforms=u)
    b, p = sample(x, mode="filtered", top_p=0.9, uniforms=u, return_probs=True)
    assert torch.equal(a, b)
    for r in (0, 137, 299):
        assert a[r, 0].item() == O.sample_filtered(p[r].cpu().numpy(), float(u[r, 0]), 0.9, 0)


@pytest.mark.parametrize("V", [1500, 50001])
@pytest.mark.parametrize("top_p,top_k", [(0.9, 0), (0.9, 3), (1.0, 1), (1.0, 0)])
def test_infinite_and_nan_probabilities(device, V, top_p, top_k):
    """An infinite probability is the largest one; NaN is never kept (the
    oracle, which sorts, gets a zero in its place)."""
    g = torch.Generator().manual_seed(V)
    x = torch.rand(6, V, generator=g) * 4.0 / V
    x[0, V // 3] = float("inf")
    x[1, V // 3] = x[1, V - 2] = float("inf")
    x[2, 5] = float("nan")
    x[3, ::7] = float("nan")
    x[4] = float("nan")
    x[5, 7], x[5, 9] = float("inf"), float("nan")
    u = torch.rand(6, 3, generator=g)
    u[:, 0], u[:, 1] = 0.0, LAST
    tok = sample(x.to(device), mode="filtered", top_p=top_p, top_k=top_k, draws=3,
                 uniforms=u.to(device), input_kind="probs").cpu().numpy()
    for r in range(6):
        p = torch.nan_to_num(x[r], nan=0.0, posinf=float("inf")).numpy()
        for d in range(3):
            assert tok[r, d] == O.sample_filtered(p, float(u[r, d]), top_p, top_k), (r, d)


@pytest.mark.parametrize("V", [1500, 50001])
def test_masked_and_broken_logits(device, V):
    """-inf masks entries out; a row whose softmax is undefined (NaN, +inf,
    or nothing but -inf) keeps nothing and falls to its last index."""
    g = torch.Generator().manual_seed(V)
    x = 2.0 * torch.randn(5, V, generator=g)
    x[0, ::2] = float("-inf")
    x[1] = float("-inf")
    x[1, V // 2] = -3.0
    x[2, 11] = float("nan")
    x[3, 11] = float("inf")
    x[4] = float("-inf")
    u = torch.rand(5, 1, generator=g)
    tok, p = sample(x.to(device), mode="filtered", top_p=0.9, top_k=50, uniforms=u.to(device),
                    return_probs=True)
    tok, p = tok.cpu().numpy(), p.cpu().numpy()
    assert tok[0, 0] == O.sample_filtered(p[0], float(u[0, 0]), 0.9, 50) and tok[0, 0] % 2 == 1
    assert tok[1, 0] == V // 2
    assert (tok[2:, 0] == V - 1).all()
