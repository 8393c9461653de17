"""Workloads of the verification path, as a speculative-decoding server meets
them, for timing and for comparing two builds' outputs.

A case is a dict of plain values; ``kind`` names its entry point:

  chain    ``verify.chain_verify``: verification of B drafted chains
  sample   ``sampling.sample`` / ``expand_tree_level``: plain decode and the
           children of draft-tree nodes
  attn     ``verify.tree_attention``: draft-tree queries over the paged cache
  accept   ``verify.tree_verify``: the accepted path of a draft tree
  ffn      ``w4a16.W4A16Linear``: a Llama layer's SiLU-gated FFN, W4A16
  int4     ``w4a16.int4_gemm_dequant``: the INT4 GEMM on its own
  target   ``spec_step.TargetModel.forward_tree``: layers + head of the target
  draft    ``spec_step.DraftModel.forward_level``: one tree level of the draft

Logits follow the repository's benchmark: target 2 N(0, 1), draft = target +
N(0, 0.5), drafts drawn from the draft's softmax, seeded U(0, 1) uniforms.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cudaforge_amd import tree as T
from cudaforge_amd.kv_cache import KVCacheConfig, PagedKVCache
from cudaforge_amd.sampling import expand_tree_level, sample
from cudaforge_amd.spec_step import DRAFT_1B, TARGET_8B, DraftModel, LlamaShape, TargetModel
from cudaforge_amd.verify import chain_verify, tree_attention, tree_verify
from cudaforge_amd.w4a16 import W4A16Linear, int4_gemm_dequant

PAGE = 16
# mean per-position acceptance of a draft whose logits are the target's plus
# N(0, 0.5), at temperature 0.7
ACCEPT = 0.7


def listed():
    return [
        # one user's stream through the drop-in engine: its python-mode rules
        # and default top-p at the small test models' vocabulary
        dict(name="chain_python_b1", kind="chain", mode="python", B=1, K=4, V=32000,
             temperature=1.0, top_p=0.9),
        # the engine's defaults (K = 5, top-p 0.9) for a small batch at the
        # Llama-3 vocabulary
        dict(name="chain_python_b8", kind="chain", mode="python", B=8, K=5, V=128256,
             temperature=1.0, top_p=0.9),
        # the benchmark's headline: a full batch under per-sequence rules
        dict(name="chain_cpp_b64", kind="chain", mode="cpp", B=64, K=8, V=128256,
             temperature=0.7, top_p=1.0),
        # plain decode of a batch with the sampler's default filters
        # (SamplingParams: top-k 50, top-p 0.9)
        dict(name="sample_filtered_r32", kind="sample", mode="filtered", R=32, V=128256, draws=1,
             temperature=0.8, top_k=50, top_p=0.9),
        # the children of a tree level: 8 sequences x 16 nodes, two each
        dict(name="expand_level_r128", kind="sample", mode="expand", R=128, V=128256, draws=2,
             temperature=1.0, top_k=-1, top_p=1.0),
        # tree attention at the benchmark's batch and context
        dict(name="attn_b16_ctx4096", kind="attn", B=16, N=63, Hq=32, Hkv=8, D=128, ctx=4096,
             ragged=False),
        # a few users at different points of their conversations, small trees
        dict(name="attn_b3_ragged", kind="attn", B=3, N=31, Hq=32, Hkv=8, D=128, ctx=1500,
             ragged=True),
        # tree acceptance at the benchmark's batch
        dict(name="accept_b32", kind="accept", B=32, depth=5, V=128256, temperature=0.7),
        # the target's FFN for one user's 63-node tree
        dict(name="ffn_m63", kind="ffn", M=63, d=4096, ffn=14336),
        # plain decode of four users through the INT4 GEMM (fp16, as the
        # reference's own test calls it), at the 8B FFN's up projection
        dict(name="int4_m4", kind="int4", M=4, K=4096, N=14336, dtype="float16", zeros=False),
        # the verify step's target forward at 8B width, batch and context; 8
        # of the 32 layers, so that several copies of the state fit
        dict(name="target_b8_ctx2048", kind="target", layers=8, B=8, N=63, ctx=2048),
        # one level (8 nodes) of the 1B-shape draft's proposal, replayed from
        # a graph as the tree speculator does
        dict(name="draft_b8_level3", kind="draft", B=8, level=3, ctx=1024),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["chain", "sample", "attn", "accept", "ffn", "int4", "target", "draft"])
    if kind == "chain":
        return dict(kind=kind, mode=rng.choice(["python", "python", "cpp", "cpp", "greedy"]),
                    B=_log_int(rng, 1, 64), K=rng.randint(1, 8), V=_log_int(rng, 8000, 128256),
                    temperature=rng.choice([0.7, 1.0]), top_p=rng.choice([0.5, 0.9, 1.0]))
    if kind == "sample":
        mode = rng.choice(["filtered", "expand", "multinomial", "greedy"])
        draws = {"expand": 2, "greedy": rng.choice([1, 2])}.get(mode, 1)
        return dict(kind=kind, mode=mode, R=_log_int(rng, 1, 128), V=_log_int(rng, 8000, 128256),
                    draws=draws, temperature=rng.choice([0.7, 0.8, 1.0]),
                    top_k=rng.choice([-1, 50]) if mode == "filtered" else -1,
                    top_p=rng.choice([0.9, 0.95]) if mode == "filtered" else 1.0)
    if kind == "attn":
        return dict(kind=kind, B=_log_int(rng, 1, 16), N=rng.randint(1, 63),
                    Hq=rng.choice([32, 32, 16]), Hkv=8, D=rng.choice([128, 128, 64]),
                    ctx=_log_int(rng, 128, 4096), ragged=rng.choice([True, False]))
    if kind == "accept":
        return dict(kind=kind, B=_log_int(rng, 1, 32), depth=rng.randint(2, 5),
                    V=_log_int(rng, 8000, 128256), temperature=rng.choice([0.7, 1.0]))
    if kind == "ffn":
        d, ffn = rng.choice([(2048, 8192), (4096, 14336)])
        return dict(kind=kind, M=_log_int(rng, 1, 504), d=d, ffn=ffn)
    if kind == "int4":
        K, N = rng.choice([(4096, 6144), (4096, 4096), (4096, 14336), (14336, 4096),
                           (2048, 8192)])
        return dict(kind=kind, M=_log_int(rng, 1, 64), K=K, N=N,
                    dtype=rng.choice(["float16", "bfloat16"]), zeros=rng.choice([True, False]))
    if kind == "target":
        return dict(kind=kind, layers=8, B=rng.randint(1, 8), N=rng.choice([7, 15, 31, 63]),
                    ctx=_log_int(rng, 256, 2048))
    return dict(kind=kind, B=_log_int(rng, 1, 8), level=rng.randint(0, 4),
                ctx=_log_int(rng, 256, 1024))


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _ragged(case, g):
    """Context lengths [B] int32: the case's, or between a quarter of it and it."""
    B, ctx = case["B"], case["ctx"]
    if not case.get("ragged"):
        return torch.full((B,), ctx, dtype=torch.int32, device="cuda")
    lens = torch.randint(max(1, ctx // 4), ctx + 1, (B,), device="cuda", generator=g)
    lens[0] = ctx
    return lens.int()


def prepare(case, seed):
    g = _gen(seed)
    return _PREPARE[case["kind"]](case, g, seed)


def run(state):
    return _RUN[state["kind"]](state)


def work(case):
    return _WORK[case["kind"]](case)


def tolerance(case):
    return _TOLERANCE[case.get("dtype", case["kind"])]


def exact(case, seed):
    fn = _EXACT.get(case["kind"])
    return None if fn is None else fn(case, prepare(case, seed))


# Tokens, counts and paths are whole numbers: the same for every correct build
# of the same fp32 rules.  The others: three to four times the distance from
# 64 bits measured on MI355X (attention 0.0033, FFN 0.0049, INT4 GEMM 0.0004
# in fp16 and 0.0028 in bf16), which is what two correct builds can differ by;
# the models' logits are 0.013 to 0.017 off, so two builds stay within 0.03.
_TOLERANCE = {
    "chain": "exact",
    "sample": "exact",
    "accept": "exact",
    "attn": {"rel": 1e-2, "max": 0.1},
    "ffn": {"rel": 1e-2, "max": 0.1},
    "float16": {"rel": 1.5e-3, "max": 0.01},
    "bfloat16": {"rel": 1e-2, "max": 0.05},
    "target": {"rel": 3e-2, "max": 0.5},
    "draft": {"rel": 3e-2, "max": 0.5},
}


# -- chain ------------------------------------------------------------------

def _prepare_chain(case, g, seed):
    B, K, V, temp = case["B"], case["K"], case["V"], case["temperature"]
    tl = torch.randn(B, K + 1, V, device="cuda", generator=g) * 2.0
    dl = tl[:, :K] + 0.5 * torch.randn(B, K, V, device="cuda", generator=g)
    probs = torch.softmax(dl / temp, dim=-1).reshape(B * K, V)
    tok = torch.multinomial(probs, 1, generator=g).reshape(B, K).int()
    greedy = case["mode"] == "greedy"
    nu = K + 2 if case["mode"] == "python" else K + 1
    u = torch.rand(B, nu, device="cuda", generator=g)
    return dict(kind="chain", target=tl, draft=None if greedy else dl.contiguous(), tokens=tok,
                uniforms=None if greedy else u,
                kw=dict(temperature=temp, top_p=case["top_p"], mode=case["mode"]))


def _run_chain(s):
    o = chain_verify(s["target"], s["draft"], s["tokens"], s["uniforms"], **s["kw"])
    return dict(accept_len=o.accept_len, tokens=o.tokens, num_emitted=o.num_emitted,
                final=o.final, eos=o.eos)


def _work_chain(case):
    # the rows of every position that is tested (both windows), and the
    # target's last row when every draft is accepted; python mode keeps the
    # batch in lock step
    B, K, V = case["B"], case["K"], case["V"]
    if case["mode"] == "greedy":
        rows = B * (K + 1)
    else:
        a = ACCEPT ** B if case["mode"] == "python" else ACCEPT
        rows = B * (sum(2 * a ** i for i in range(K)) + a ** K)
    n = rows * V
    return {"bytes": 4 * n + 4 * B * (3 * K + 6), "flops": 4 * n}


# -- sampling ---------------------------------------------------------------

def _prepare_sample(case, g, seed):
    R, V = case["R"], case["V"]
    rows = torch.randn(R, V, device="cuda", generator=g) * 2.0
    # multinomial draws take u in (0, 1], filtered ones [0, 1)
    u = torch.rand(R, case["draws"], device="cuda", generator=g)
    if case["mode"] in ("expand", "multinomial"):
        u = 1.0 - u
    return dict(kind="sample", rows=rows, uniforms=u, **{k: case[k] for k in (
        "mode", "draws", "temperature", "top_k", "top_p")})


def _run_sample(s):
    if s["mode"] == "expand":
        return expand_tree_level(s["rows"], children=s["draws"], temperature=s["temperature"],
                                 uniforms=s["uniforms"])
    if s["mode"] == "greedy":
        return sample(s["rows"], mode="greedy", draws=s["draws"])
    return sample(s["rows"], mode=s["mode"], temperature=s["temperature"], top_k=s["top_k"],
                  top_p=s["top_p"], draws=s["draws"], uniforms=s["uniforms"])


def _work_sample(case):
    n = case["R"] * case["V"]
    return {"bytes": 4 * n + 8 * case["R"] * case["draws"], "flops": 4 * n}


# -- tree attention ---------------------------------------------------------

def _prepare_attn(case, g, seed):
    B, N, Hq, Hkv, D, ctx = (case[k] for k in ("B", "N", "Hq", "Hkv", "D", "ctx"))
    pages = (ctx + N + PAGE - 1) // PAGE
    nblk = B * pages + 8
    kp = torch.randn(nblk, 1, Hkv, PAGE, D, device="cuda", generator=g).bfloat16()
    vp = torch.randn(nblk, 1, Hkv, PAGE, D, device="cuda", generator=g).bfloat16()
    tables = torch.randperm(nblk, device="cuda", generator=g)[: B * pages].int().view(B, pages)
    q = torch.randn(B, N, Hq, D, device="cuda", generator=g).bfloat16()
    masks = T.ancestor_masks(T.binary_tree_parents(N))
    return dict(kind="attn", q=q, kp=kp, vp=vp, tables=tables.contiguous(), lens=_ragged(case, g),
                masks=T.mask_tensor(masks, "cuda"), max_keys=ctx + N)


def _run_attn(s):
    return tree_attention(s["q"], s["kp"], s["vp"], s["tables"], s["lens"], s["masks"],
                          max_keys=s["max_keys"])


def _work_attn(case):
    B, N, Hq, Hkv, D, ctx = (case[k] for k in ("B", "N", "Hq", "Hkv", "D", "ctx"))
    anc = sum(bin(int(x)).count("1") for x in T.ancestor_masks(T.binary_tree_parents(N)))
    keys = ctx if not case["ragged"] or B == 1 else (ctx + (B - 1) * 0.625 * ctx) / B
    return {"bytes": B * Hkv * (keys + N) * D * 4 + 4 * B * N * Hq * D,
            "flops": 4 * B * Hq * D * (N * keys + anc)}


def _tree_mask(N, lo=0):
    """[N - lo, N] bool: which tree nodes the nodes lo .. N - 1 see."""
    anc = T.ancestor_masks(T.binary_tree_parents(N))
    return torch.tensor([[bool((int(anc[i]) >> j) & 1) for j in range(N)] for i in range(lo, N)],
                        device="cuda")


def _pages(pool, layer, table, n):
    """The first n slots of one sequence in fp64: [Hkv, n, D]."""
    x = pool[table[: (n + PAGE - 1) // PAGE].long(), layer]      # [pages, Hkv, PAGE, D]
    return x.transpose(0, 1).reshape(pool.shape[2], -1, pool.shape[4])[:, :n].double()


def _attend(q, k, v, mask):
    """q [n, Hq, D], k / v [Hkv, S, D], mask [n, tree]: the last `tree` keys
    are the tree's; fp64 attention [n, Hq, D]."""
    n, Hq, D = q.shape
    Hkv, S, _ = k.shape
    qh = q.view(n, Hkv, Hq // Hkv, D).permute(1, 2, 0, 3).reshape(Hkv, -1, D).contiguous()
    sc = torch.bmm(qh, k.transpose(1, 2).contiguous()) / math.sqrt(D)
    see = torch.ones(n, S, dtype=torch.bool, device=q.device)
    see[:, S - mask.shape[1]:] = mask
    sc = sc.view(Hkv, Hq // Hkv, n, S).masked_fill(~see, float("-inf"))
    p = torch.softmax(sc, dim=-1).view(Hkv, -1, S)
    o = torch.bmm(p, v.contiguous()).view(Hkv, Hq // Hkv, n, D)
    return o.permute(2, 0, 1, 3).reshape(n, Hq, D)


def _exact_attn(case, s):
    N = case["N"]
    mask = _tree_mask(N)
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    for b, n in enumerate(s["lens"].tolist()):
        k = _pages(s["kp"], 0, s["tables"][b], n + N)
        v = _pages(s["vp"], 0, s["tables"][b], n + N)
        out[b] = _attend(s["q"][b].double(), k, v, mask)
    return out


# -- tree acceptance --------------------------------------------------------

def _prepare_accept(case, g, seed):
    B, V, temp = case["B"], case["V"], case["temperature"]
    N = 2 ** (case["depth"] + 1) - 1
    parents = torch.from_numpy(T.binary_tree_parents(N)).cuda()
    tl = torch.randn(B, N, V, device="cuda", generator=g) * 2.0
    dl = tl + 0.5 * torch.randn(B, N, V, device="cuda", generator=g)
    tok = torch.zeros(B, N, dtype=torch.int32, device="cuda")
    inner = (N - 1) // 2                                        # nodes with two children
    probs = torch.softmax(dl[:, :inner] / temp, dim=-1).reshape(B * inner, V)
    tok[:, 1:] = torch.multinomial(probs, 2, replacement=True, generator=g).view(B, N - 1).int()
    u = 1.0 - torch.rand(B, 4 * case["depth"] + 2, device="cuda", generator=g)
    return dict(kind="accept", target=tl, draft=dl, parents=parents, tokens=tok, uniforms=u,
                temperature=temp)


def _run_accept(s):
    o = tree_verify(s["target"], s["draft"], s["parents"], s["tokens"], s["uniforms"],
                    temperature=s["temperature"])
    return dict(path=o.path, path_len=o.path_len, tokens=o.tokens, num_emitted=o.num_emitted,
                final=o.final, eos=o.eos, status=o.status)


def _work_accept(case):
    # a node is left through a child with about the probability that one of
    # two candidates is accepted; its target and draft rows are read
    a = 1 - (1 - ACCEPT) ** 2
    rows = sum(2 * a ** i for i in range(case["depth"])) + a ** case["depth"]
    n = case["B"] * rows * case["V"]
    return {"bytes": 4 * n, "flops": 4 * n}


# -- W4A16 ------------------------------------------------------------------

def _weights64(lin):
    """The packed weights as fp64 [K, N]: (nibble - zero point) * scale."""
    q, K = lin.qweight, lin.K
    nib = torch.stack([(q >> (4 * i)) & 15 for i in range(8)], dim=1).view(K, lin.N)
    grp = torch.arange(K, device=q.device) // lin.group
    w = nib.double()
    if lin.zeros is not None:
        w -= lin.zeros.double()[grp]
    return w.mul_(lin.scales.double()[grp])


def _gate_up(y):
    """The gate and up halves of a product in the 64-column interleaved layout."""
    t = y.view(y.shape[0], -1, 2, 32)
    return t[:, :, 0].reshape(y.shape[0], -1), t[:, :, 1].reshape(y.shape[0], -1)


def _prepare_ffn(case, g, seed):
    M, d, ffn = case["M"], case["d"], case["ffn"]
    return dict(kind="ffn", x=torch.randn(M, d, device="cuda", generator=g).bfloat16(),
                up=W4A16Linear(d, 2 * ffn, "cuda", g), down=W4A16Linear(ffn, d, "cuda", g),
                scratch=torch.empty(2 * d * ffn, dtype=torch.bfloat16, device="cuda"))


def _run_ffn(s):
    act = s["up"].silu_gated(s["x"], s["scratch"])
    return dict(act=act, out=s["down"](act, s["scratch"]))


def _weight_bytes(K, N, zeros=True, group=128):
    return K * N // 2 + (4 if zeros else 2) * (K // group) * N


def _work_ffn(case):
    M, d, ffn = case["M"], case["d"], case["ffn"]
    return {"bytes": _weight_bytes(d, 2 * ffn) + _weight_bytes(ffn, d) + 2 * M * (2 * d + 2 * ffn),
            "flops": 2 * M * 3 * d * ffn}


def _exact_ffn(case, s):
    gate, up = _gate_up(s["x"].double() @ _weights64(s["up"]))
    act = torch.nn.functional.silu(gate) * up
    return dict(act=act, out=act @ _weights64(s["down"]))


class _Packed:
    """The weights of one INT4 GEMM call."""


def _prepare_int4(case, g, seed):
    K, N = case["K"], case["N"]
    w = _Packed()
    w.K, w.N, w.group = K, N, 128
    w.qweight = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 8, N), dtype=torch.int32,
                              device="cuda", generator=g)
    w.scales = ((0.5 + torch.rand(K // 128, N, device="cuda", generator=g))
                / math.sqrt(85.0 * K)).half()
    w.zeros = torch.randint(0, 16, (K // 128, N), device="cuda",
                            generator=g).half() if case["zeros"] else None
    a = torch.randn(case["M"], K, device="cuda", generator=g).to(getattr(torch, case["dtype"]))
    return dict(kind="int4", a=a, w=w)


def _run_int4(s):
    w = s["w"]
    return int4_gemm_dequant(s["a"], w.qweight, w.scales, w.zeros, group_size=w.group)


def _work_int4(case):
    M, K, N = case["M"], case["K"], case["N"]
    return {"bytes": _weight_bytes(K, N, case["zeros"]) + 2 * M * (K + N), "flops": 2 * M * K * N}


def _exact_int4(case, s):
    return s["a"].double() @ _weights64(s["w"])


# -- the models -------------------------------------------------------------

def _rms64(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, pos, theta):
    """Rotate-half embedding of x [B, n, H, D] at positions [B, n]."""
    D = x.shape[-1]
    inv = theta ** (-torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D)
    ang = pos.double()[..., None] * inv
    cos = torch.cat([ang.cos(), ang.cos()], -1)[..., None, :]
    sin = torch.cat([ang.sin(), ang.sin()], -1)[..., None, :]
    rot = torch.cat([-x[..., D // 2:], x[..., : D // 2]], -1)
    return x * cos + rot * sin


def _exact_model(shape, embed, layers, norm, head, weight, tokens, pos, tables, lens, lo, kp, vp):
    """Logits and pools after the forward of tree nodes lo .. lo + n - 1 (K/V
    at slots len + node), in fp64; `weight` gives a projection's matrix."""
    B, n = tokens.shape
    Hq, Hkv, D = shape.n_heads, shape.n_kv_heads, shape.head_dim
    kp, vp = kp.double(), vp.double()
    mask = _tree_mask(lo + n, lo)
    h = embed[tokens.long().reshape(-1)].double()
    for li, L in enumerate(layers):
        x = _rms64(h, L["attn_norm"], shape.eps)
        qkv = (x @ weight(L["wqkv"])).view(B, n, Hq + 2 * Hkv, D)
        q = _rope64(qkv[:, :, :Hq], pos, shape.rope_theta)
        k = _rope64(qkv[:, :, Hq:Hq + Hkv], pos, shape.rope_theta)
        o = torch.empty(B, n, Hq, D, dtype=torch.float64, device=h.device)
        for b, ctx in enumerate(lens):
            slot = ctx + lo + torch.arange(n, device=h.device)
            blk = tables[b].long()[slot // PAGE]
            kp[blk, li, :, slot % PAGE] = k[b]
            vp[blk, li, :, slot % PAGE] = qkv[b, :, Hq + Hkv:]
            o[b] = _attend(q[b], _pages(kp, li, tables[b], ctx + lo + n),
                           _pages(vp, li, tables[b], ctx + lo + n), mask)
        h = h + o.view(B * n, Hq * D) @ weight(L["wo"])
        gate, up = _gate_up(_rms64(h, L["ffn_norm"], shape.eps) @ weight(L["wgu"]))
        h = h + (torch.nn.functional.silu(gate) * up) @ weight(L["wdown"])
    h = _rms64(h, norm, shape.eps)
    logits = torch.cat([h @ head[:, c:c + 16384].double()
                        for c in range(0, head.shape[1], 16384)], dim=1)
    return dict(logits=logits.view(B, n, -1), keys=kp, values=vp)


def _prepare_target(case, g, seed):
    B, N, ctx = case["B"], case["N"], case["ctx"]
    t = TARGET_8B
    shape = LlamaShape(case["layers"], t.d_model, t.n_heads, t.n_kv_heads, t.head_dim, t.ffn,
                       t.vocab, t.rope_theta, t.eps)
    model = TargetModel(shape, torch.device("cuda"), seed=seed)
    pages = (ctx + N + PAGE - 1) // PAGE
    kv = PagedKVCache(KVCacheConfig(
        num_layers=shape.n_layers, num_kv_heads=shape.n_kv_heads, head_dim=shape.head_dim,
        block_size=PAGE, total_gpu_blocks=B * pages + 8, enable_prefix_caching=False,
        max_supported_batch_size=B, max_blocks_per_sequence=pages), device=torch.device("cuda"))
    rng = np.random.default_rng(seed)
    for b in range(B):
        kv.register_sequence_with_prefix(b, rng.integers(0, shape.vocab, ctx).tolist())
        kv.append_tokens(b, N)
    kv.key_pool.normal_(generator=g)
    kv.value_pool.normal_(generator=g)
    parents = T.binary_tree_parents(N)
    base = torch.full((B,), ctx, dtype=torch.int32, device="cuda")
    tokens = torch.randint(0, shape.vocab, (B, N), device="cuda", generator=g, dtype=torch.int32)
    pos = base[:, None] + torch.from_numpy(T.depths(parents)).cuda()[None, :]
    return dict(kind="target", model=model, kv=kv, tables=kv.prepare_batch_metadata(
        list(range(B))).block_tables, tokens=tokens, pos=pos, base=base,
        masks=T.mask_tensor(T.ancestor_masks(parents), "cuda"), max_keys=ctx + N)


def _run_target(s):
    logits = s["model"].forward_tree(s["tokens"], s["pos"], s["kv"], s["tables"], s["base"],
                                     s["masks"], s["max_keys"])
    return dict(logits=logits, keys=s["kv"].key_pool, values=s["kv"].value_pool)


def _layer_params(shape):
    d, hd = shape.d_model, shape.head_dim
    return [(d, (shape.n_heads + 2 * shape.n_kv_heads) * hd), (shape.n_heads * hd, d),
            (d, 2 * shape.ffn), (shape.ffn, d)]


def _work_model(shape, layers, B, n, keys, weight_bytes):
    M = B * n
    mats = _layer_params(shape)
    kv = B * shape.n_kv_heads * keys * shape.head_dim * 4
    flops = layers * (sum(2 * M * K * N for K, N in mats)
                      + 4 * M * shape.n_heads * shape.head_dim * keys)
    head = shape.d_model * shape.vocab
    return {"bytes": layers * (sum(weight_bytes(K, N) for K, N in mats) + kv) + 2 * head
            + 4 * M * shape.vocab, "flops": flops + 2 * M * head}


def _work_target(case):
    return _work_model(TARGET_8B, case["layers"], case["B"], case["N"], case["ctx"] + case["N"],
                       _weight_bytes)


def _exact_target(case, s):
    m, kv = s["model"], s["kv"]
    return _exact_model(m.shape, m.embed, m.layers, m.norm, m.lm_head, _weights64, s["tokens"],
                        s["pos"], s["tables"], s["base"].tolist(), 0, kv.key_pool, kv.value_pool)


def _prepare_draft(case, g, seed):
    B, ctx = case["B"], case["ctx"]
    lo, hi = 2 ** case["level"] - 1, 2 ** (case["level"] + 1) - 1
    model = DraftModel(DRAFT_1B, torch.device("cuda"), B, max_slots=ctx + 64, seed=seed)
    model.k_pool.normal_(generator=g)
    model.v_pool.normal_(generator=g)
    parents = T.binary_tree_parents(63)
    base = torch.full((B,), ctx, dtype=torch.int32, device="cuda")
    tokens = torch.randint(0, DRAFT_1B.vocab, (B, hi - lo), device="cuda", generator=g,
                           dtype=torch.int32)
    depths = torch.from_numpy(T.depths(parents)).cuda()
    pos = base[:, None] + depths[lo:hi][None, :]
    masks = T.mask_tensor(T.ancestor_masks(parents), "cuda")

    def level():
        return model.forward_level(tokens, pos, base, lo, masks)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        level()                                                 # outside the capture
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = level()
    return dict(kind="draft", model=model, graph=graph, logits=logits, tokens=tokens, pos=pos,
                base=base, masks=masks, lo=lo)


def _run_draft(s):
    s["graph"].replay()
    return dict(logits=s["logits"], keys=s["model"].k_pool, values=s["model"].v_pool)


def _work_draft(case):
    return _work_model(DRAFT_1B, DRAFT_1B.n_layers, case["B"], 2 ** case["level"],
                       case["ctx"] + 2 ** (case["level"] + 1) - 1, lambda K, N: 2 * K * N)


def _exact_draft(case, s):
    m = s["model"]
    return _exact_model(m.shape, m.embed, m.layers, m.norm, m.lm_head, lambda w: w.double(),
                        s["tokens"], s["pos"], m.block_tables, s["base"].tolist(), s["lo"],
                        m.k_pool, m.v_pool)


_PREPARE = {"chain": _prepare_chain, "sample": _prepare_sample, "attn": _prepare_attn,
            "accept": _prepare_accept, "ffn": _prepare_ffn, "int4": _prepare_int4,
            "target": _prepare_target, "draft": _prepare_draft}
_RUN = {"chain": _run_chain, "sample": _run_sample, "attn": _run_attn, "accept": _run_accept,
        "ffn": _run_ffn, "int4": _run_int4, "target": _run_target, "draft": _run_draft}
_WORK = {"chain": _work_chain, "sample": _work_sample, "attn": _work_attn,
         "accept": _work_accept, "ffn": _work_ffn, "int4": _work_int4, "target": _work_target,
         "draft": _work_draft}
_EXACT = {"attn": _exact_attn, "ffn": _exact_ffn, "int4": _exact_int4, "target": _exact_target,
          "draft": _exact_draft}
