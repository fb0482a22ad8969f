"""Kernels that a dispatch picks by size: at the edges of their tiles and of the rule, against plain fp32 products."""
import math

import numpy as np
import pytest
import torch

from localai_amd import ops

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
