"""Kernels that a dispatch picks by size: at the edges of their tiles and of the rule, against plain fp32 products."""
import math

import numpy as np
import pytest
import torch

from localai_amd import ops
from localai_amd.gguf import GGMLType, quantize

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _pages(ctx, Hkv, Dh, BS, seed):
    """Shuffled pages of random keys and values; places that hold no key of the sequence are NaN."""
    g = torch.Generator().manual_seed(seed)
    need = [-(-n // BS) for n in ctx]
    order = torch.randperm(sum(need), generator=g).tolist()
    kc = torch.full((sum(need), Hkv, BS, Dh), math.nan, dtype=torch.bfloat16)
    vc = torch.full((sum(need), Hkv, BS // 8, Dh, 8), math.nan, dtype=torch.bfloat16)
    bt = torch.zeros(len(ctx), max(need), dtype=torch.int32)
    keys, values = [], []
    for s, n in enumerate(ctx):
        k, v = torch.randn(2, n, Hkv, Dh, generator=g).to(torch.bfloat16)
        for b in range(need[s]):
            p = bt[s, b] = order.pop()
            rows = slice(b * BS, min(n, (b + 1) * BS))
            w = rows.stop - rows.start
            kc[p, :, :w] = k[rows].transpose(0, 1)
            pad = torch.full((BS, Hkv, Dh), math.nan, dtype=torch.bfloat16)
            pad[:w] = v[rows]
            vc[p] = pad.view(BS // 8, 8, Hkv, Dh).permute(2, 0, 3, 1)
        keys.append(k.float())
        values.append(v.float())
    return kc, vc, bt, keys, values


@pytest.mark.parametrize("Hq,Hkv,Dh,BS", [(32, 8, 128, 32), (4, 2, 128, 16), (6, 6, 128, 64), (12, 4, 64, 32), (8, 2, 64, 128)])
@pytest.mark.parametrize("qlens,ctx", [([1, 64, 65], [1, 64, 65]), ([3, 63, 32, 129], [64, 130, 33, 1000]),
                                       ([700] * 5, [701, 707, 700, 765, 1023])])
def test_prefill_flash(Hq, Hkv, Dh, BS, qlens, ctx):
    """Prompt portions that begin and end inside tiles and pages, alone and behind cached keys; the last lists give
    launches of more than 256 workgroups.  The weights are rounded to bf16 beside an fp32 sum and so is the result:
    each is off by at most 2^-9 of the largest value, twice that is allowed."""
    kc, vc, bt, keys, values = _pages(ctx, Hkv, Dh, BS, seed=Hq + len(ctx))
    q = torch.randn(sum(qlens), Hq, Dh, generator=torch.Generator().manual_seed(5)).to(torch.bfloat16)
    cu = torch.tensor([0] + list(np.cumsum(qlens)), dtype=torch.int32)
    cl = torch.tensor(ctx, dtype=torch.int32)
    scale = 1 / math.sqrt(Dh)
    out = ops.attn_prefill(q.to(DEV), kc.to(DEV), vc.to(DEV), cu.to(DEV), cl.to(DEV), bt.to(DEV), scale).float().cpu()
    at = 0
    for s, n in enumerate(qlens):
        k, v = (x[s].repeat_interleave(Hq // Hkv, 1) for x in (keys, values))
        sc = torch.einsum("qhd,khd->hqk", q[at:at + n].float(), k) * scale
        late = torch.arange(ctx[s])[None, :] > torch.arange(ctx[s] - n, ctx[s])[:, None]
        ref = torch.einsum("hqk,khd->qhd", torch.softmax(sc.masked_fill(late, -math.inf), -1), v)
        assert (out[at:at + n] - ref).abs().max().item() <= 2 ** -7 * v.abs().max().item()
        at += n


@pytest.mark.parametrize("Hq,Hkv,Dh,BS", [(32, 8, 128, 32), (6, 6, 128, 16), (8, 2, 64, 128)])
@pytest.mark.parametrize("qlens,ctx,shares", [([16], [2016], 7), ([5, 70], [1500, 130], 5), ([65, 1], [65, 4100], 15)])
def test_prefill_shares(Hq, Hkv, Dh, BS, qlens, ctx, shares):
    """The same behind long contexts, a tile's keys shared by several workgroups, some of them without keys (the short
    sequences), with empty and with partly masked shares."""
    blocks = max(-(-c // BS) for c in ctx)
    assert ops._prefill_splits(sum(-(-n // 64) for n in qlens), Hq, Hkv, Dh, BS, blocks * BS, sum(qlens) // len(qlens)) >= min(shares, 8)
    test_prefill_flash(Hq, Hkv, Dh, BS, qlens, ctx)


def _weight(N, K, t, seed):
    w = np.random.default_rng(seed).standard_normal((N, K)).astype(np.float32) * 0.05
    return ops.QWeight.from_raw(quantize(w, t), t, (N, K), DEV, keep_ref=True)


SKINNY = [(GGMLType.Q4_K, 64, 256), (GGMLType.Q4_K, 200, 2816), (GGMLType.Q6_K, 130, 768), (GGMLType.Q6_K, 321, 1024),
          (GGMLType.Q8_0, 72, 1280), (GGMLType.F16, 80, 512)]


@pytest.mark.parametrize("t,N,K", SKINNY)
@pytest.mark.parametrize("M", [3, 16, 17, 33, 64])
def test_skinny_products(t, N, K, M):
    """Fewer stages than ring slots, rows and columns past the last tile, an odd number of super-blocks, scales that
    straddle dwords.  The weights are rounded to bf16 (2^-9 of each), the sums are fp32."""
    w = _weight(N, K, t, N + K)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16)
    y = ops.linear(x.to(DEV), w, force="skinny").dense().cpu()
    bound = 2 ** -9 * (x.float().abs() @ w.ref.abs().t())
    assert ((y - x.float() @ w.ref.t()).abs() <= bound + 1e-5).all()


@pytest.mark.parametrize("t,N,K", SKINNY)
@pytest.mark.parametrize("M,mode", [(3, ops.ACT_SWIGLU), (16, ops.ACT_GEGLU), (31, ops.ACT_SWIGLU), (64, ops.ACT_GEGLU)])
def test_skinny_gated(t, N, K, M, mode):
    """act(gate) * up in the product's epilogue, of two weights and of the halves of one: each product is off by at most
    2^-9 of the sum of its terms' sizes, both activations' slopes stay below 1.2, the result is rounded to bf16."""
    N &= ~15
    a, b = _weight(N, K, t, 1), _weight(N, K, t, 2)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16)
    g, u = x.float() @ a.ref.t(), x.float() @ b.ref.t()
    eg, eu = (2 ** -9 * (x.float().abs() @ w.ref.abs().t()) for w in (a, b))
    s = torch.nn.functional.silu(g) if mode == ops.ACT_SWIGLU else torch.nn.functional.gelu(g, approximate="tanh")
    bound = 1.2 * eg * (u.abs() + eu) + s.abs() * eu + 2 ** -8 * (s * u).abs() + 1e-5
    for ws in ([a, b], [ops.concat_rows([a, b])]):
        h = ops.glu_linear(x.to(DEV), ws, N, mode)
        assert h is not None and ((h.float().cpu() - s * u).abs() <= bound).all()


@pytest.mark.parametrize("Hq,Hkv,Dh,BS,lens,bound", [(32, 8, 128, 32, [8001], 16384), (8, 8, 128, 16, [1, 128, 129, 256, 257, 385, 2049], 4096),
                                                     (16, 1, 64, 64, [255, 700, 5000], 5000), (12, 4, 80, 32, [1000] * 20, 4096)])
def test_decode_shares(Hq, Hkv, Dh, BS, lens, bound):
    """Partitions are equal shares of each sequence's own keys: one, up to all 64, and lengths at the edges of a round
    of the waves; twice in a row, as the tickets reset themselves.  Weights and result are rounded to bf16 as in the
    prompt kernel.  (Places without a key are zero: this kernel multiplies them by a weight of 0.)"""
    kc, vc, bt, keys, values = _pages(lens, Hkv, Dh, BS, seed=len(lens))
    kc, vc = kc.nan_to_num(), vc.nan_to_num()
    q = torch.randn(len(lens), Hq, Dh, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
    args = [t.to(DEV) for t in (q, kc, vc, bt, torch.tensor(lens, dtype=torch.int32))]
    ws = ops.decode_workspace(len(lens), Hq, Hkv, Dh, bound, DEV, BS)
    first = ops.attn_decode(*args, 1 / math.sqrt(Dh), bound, workspace=ws).cpu()
    again = ops.attn_decode(*args, 1 / math.sqrt(Dh), bound, workspace=ws).cpu()
    assert torch.equal(first, again)
    for s, n in enumerate(lens):
        k, v = (x[s].repeat_interleave(Hq // Hkv, 1) for x in (keys, values))
        w = torch.softmax(torch.einsum("hd,khd->hk", q[s].float(), k) / math.sqrt(Dh), -1)
        ref = torch.einsum("hk,khd->hd", w, v)
        assert (first[s].float() - ref).abs().max().item() <= 2 ** -7 * v.abs().max().item()


@pytest.mark.parametrize("M", [3, 17, 64])
@pytest.mark.parametrize("Na,Nb,K", [(320, 64, 1024), (130, 71, 512), (64, 200, 2816)])
def test_skinny_pair(M, Na, Nb, K):
    """A Q4_K and a Q6_K weight side by side in one launch against each alone: the same sums, bit for bit."""
    ws = [_weight(Na, K, GGMLType.Q4_K, 1), _weight(Nb, K, GGMLType.Q6_K, 2)]
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(DEV)
    y = ops.linear_multi(x, ws, force="skinny")
    S = y.S
    alone = [ops.linear(x, w, force="skinny", out_slabs=torch.empty(S, M, w.N, device=DEV)) for w in ws]
    if all(p.S == S for p in alone):
        assert torch.equal(y.t, torch.cat([p.t for p in alone], -1))
    else:
        assert torch.allclose(y.dense(), torch.cat([p.dense() for p in alone], -1), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("t,N,K,S", [(GGMLType.Q4_K, 256, 256, 1), (GGMLType.Q4_K, 200, 2816, 3), (GGMLType.Q6_K, 130, 768, 1),
                                     (GGMLType.Q6_K, 321, 1024, 2), (GGMLType.Q8_0, 72, 1280, 5), (GGMLType.Q8_0, 384, 4352, 4)])
@pytest.mark.parametrize("M,rb", [(65, 2), (128, 2), (129, 4), (256, 4), (300, 4), (300, 2)])
def test_wide_products(t, N, K, S, M, rb):
    """Rows and columns past the last tile, splits that begin inside a quad of scales, a shorter last split, an odd
    number of super-blocks; fp32 slabs and the bf16 matrix.  Bounds as for the skinny products, plus the result's
    rounding."""
    w = _weight(N, K, t, N + K)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16)
    ref = x.float() @ w.ref.t()
    bound = 2 ** -9 * (x.float().abs() @ w.ref.abs().t()) + 1e-5
    slabs = torch.empty(S, M, N, device=DEV)
    y = ops.linear(x.to(DEV), w, force=f"tile:{20 + rb}:{S}", out_slabs=slabs).dense().cpu()
    assert ((y - ref).abs() <= bound).all()
    y = ops.linear(x.to(DEV), w, force=f"tile:{20 + rb}:1").dense().cpu()
    assert ((y - ref).abs() <= bound + 2 ** -8 * ref.abs()).all()


@pytest.mark.parametrize("t", [GGMLType.Q4_K, GGMLType.Q6_K, GGMLType.Q8_0])
@pytest.mark.parametrize("F,K,M,rb", [(64, 512, 65, 2), (80, 2816, 256, 4), (144, 256, 200, 4), (208, 1024, 128, 2)])
def test_wide_gated(t, F, K, M, rb):
    """The gated form against the plain products; bounds as for the skinny one."""
    a, b = _weight(F, K, t, 1), _weight(F, K, t, 2)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16)
    g, u = x.float() @ a.ref.t(), x.float() @ b.ref.t()
    eg, eu = (2 ** -9 * (x.float().abs() @ w.ref.abs().t()) for w in (a, b))
    s = torch.nn.functional.silu(g)
    bound = 1.2 * eg * (u.abs() + eu) + s.abs() * eu + 2 ** -8 * (s * u).abs() + 1e-5
    for pair in ((a, 0, b, 0), (ops.concat_rows([a, b]), 0, ops.concat_rows([a, b]), F)):
        h = torch.empty(M, F, dtype=torch.bfloat16, device=DEV)
        ops._run_glu(x.to(DEV), pair, F, ops.ACT_SWIGLU, 20 + rb, h)
        assert ((h.float().cpu() - s * u).abs() <= bound).all()


@pytest.mark.parametrize("M,rb,S", [(70, 2, 2), (256, 4, 3), (256, 4, 1)])
def test_wide_pair(M, rb, S):
    """Q4_K and Q6_K side by side against each alone."""
    ws = [_weight(200, 1536, GGMLType.Q4_K, 1), _weight(72, 1536, GGMLType.Q6_K, 2)]
    x = torch.randn(M, 1536, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(DEV)
    y = ops.linear_multi(x, ws, force=f"tile:{20 + rb}:{S}", out_slabs=torch.empty(S, M, 272, device=DEV))
    alone = [ops.linear(x, w, force=f"tile:{20 + rb}:{S}", out_slabs=torch.empty(S, M, w.N, device=DEV)) for w in ws]
    assert torch.equal(y.t, torch.cat([p.t for p in alone], -1))


@pytest.mark.parametrize("t,N,K,M,tile", [(GGMLType.Q4_K, 2048, 8192, 257, 24), (GGMLType.Q4_K, 2050, 8192, 512, 24), (GGMLType.Q6_K, 4096, 14336, 701, 6),
                                          (GGMLType.Q8_0, 4096, 14336, 1024, 6), (GGMLType.Q4_K, 4096, 4096, 1280, None)])
def test_prompt_plan(t, N, K, M, tile):
    """Either side of the line between the quantised products and the copy with the library's: same sums, and the gated
    form through its entry.  Every path rounds a weight to bf16 and sums in fp32; the copy's result is rounded once more."""
    w = _weight(N, K, t, N + K)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16).to(DEV)
    plan = ops._plan_quant(M, K, [w])
    assert (plan[1] if plan else None) == tile
    wf = w.ref.to(DEV)
    ref, bound = x.float() @ wf.t(), 2 ** -9 * (x.float().abs() @ wf.abs().t()) + 1e-4
    assert ((ops.linear(x, w).dense() - ref).abs() <= bound + 2 ** -8 * ref.abs()).all()
    h = ops.glu_linear(x, [w], N // 2, ops.ACT_SWIGLU)
    if h is not None:
        s, u = torch.nn.functional.silu(ref[:, :N // 2]), ref[:, N // 2:]
        eg, eu = bound[:, :N // 2], bound[:, N // 2:]
        assert ((h.float() - s * u).abs() <= 1.2 * eg * (u.abs() + eu) + s.abs() * eu + 2 ** -8 * (s * u).abs() + 1e-5).all()


@pytest.mark.parametrize("T,BS,Dh,S", [(37, 16, 128, 0), (64, 8, 64, 0), (200, 64, 128, 3), (9, 32, 64, 1), (1501, 16, 128, 0)])
def test_rope_rows_of_a_prompt(T, BS, Dh, S):
    """Rows that fill groups of eight keys, with runs that begin inside one, end inside one, skip a row or are not stored:
    bit for bit what each row alone writes."""
    Hq, Hkv = 4, 2
    W, g = (Hq + 2 * Hkv) * Dh, torch.Generator().manual_seed(T)
    x = torch.randn(max(S, 1), T, W, generator=g).to(DEV)
    x = x if S else x[0].to(torch.bfloat16)
    slots, at = torch.empty(T, dtype=torch.int32), 3
    for t in range(T):                       # a new run of slots every 23 rows, a row of padding now and then
        at = at + 1 if t % 23 else at + 5
        slots[t] = -1 if t % 19 == 17 else at
    nb = at // BS + 2
    pos = torch.arange(T, dtype=torch.int32)
    cs = torch.randn(T, Dh, generator=g).to(DEV)
    kc = torch.zeros(nb, Hkv, BS, Dh, dtype=torch.bfloat16, device=DEV)
    one = [kc, torch.zeros(nb, Hkv, BS // 8, Dh, 8, dtype=torch.bfloat16, device=DEV)]
    many = [c.clone() for c in one]
    q1 = [ops.rope_kv(ops.Partial(x[..., t:t + 1, :].contiguous()), pos[t:t + 1].to(DEV), slots[t:t + 1].to(DEV), cs, Hq, Hkv, Dh, Dh, 0,
                      *one, BS) for t in range(T)]
    q = ops.rope_kv(ops.Partial(x), pos.to(DEV), slots.to(DEV), cs, Hq, Hkv, Dh, Dh, 0, *many, BS)
    assert torch.equal(q.view(T, -1), torch.cat([a.view(1, -1) for a in q1]))
    assert torch.equal(one[0], many[0]) and torch.equal(one[1], many[1])
    assert one[1].abs().sum() > 0
