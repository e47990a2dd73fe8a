"""Stage-2 forward without a mask: tiles of 256 query rows (16 tokens of 16 heads, 32 of 8).  Sizes around the ends of tiles, of
wavefronts and of key blocks, queries fewer and more than the keys, causal and not, as many tiles as the path asks for and fewer; the same
attention with a mask of everything takes the other walk.  Against fp32 softmax attention; tolerances of the forward tests: 2e-2 on a
16-bit output of order one, 1e-3 on average, 2e-3 on the log-sum-exp."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # query lengths, key lengths, KV heads, group, mask
    ([1000, 37, 2060], [1000, 37, 2060], 2, 16, "none"),
    ([1000, 37, 2060], [1000, 37, 2060], 2, 16, "all"),
    ([1000, 37, 2060], [1000, 37, 2060], 2, 16, "acausal"),
    ([2049, 15, 17, 1], [2049, 15, 17, 1], 2, 16, "none"),
    ([1030, 33], [2100, 4161], 4, 16, "none"),                # a chunk of a longer prompt
    ([1030, 33], [2100, 0], 4, 16, "acausal"),                # a sequence without keys
    ([2100, 90], [1030, 33], 2, 16, "none"),                  # the first queries see no key
    ([2070, 700], [2070, 700], 4, 8, "none"),
    ([2070, 700], [2070, 700], 4, 4, "none"),
    ([1920], [1920], 2, 16, "none"),
    ([1904], [1904], 2, 16, "none"),
    ([1000] + [16] * 30, [1000] + [16] * 30, 4, 16, "none"),  # one long, many short: most workgroups return at once
    ([2100], [2100], 2, 8, "none"),
]
GROUP_CASES = [  # the same without a mask, walked by groups of eight tokens
    ([1700], [1700], 2, 16, "none"),
    ([1000] + [16] * 3, [1000] + [16] * 3, 2, 16, "none"),
    ([24] * 80, [24] * 80, 2, 16, "none"),
    ([130] * 15, [1130] * 15, 2, 16, "acausal"),
]


def make_mask(kind, Hk, sq, sk):
    """bool (Hk, sum sq, blocks) with every causal block, or None."""
    if kind != "all":
        return None
    nblk = (max(sk) + 63) // 64
    rows = [torch.arange(nblk)[None] <= ((torch.arange(n) + m - n).clamp(min=0) // 64)[:, None] for n, m in zip(sq, sk)]
    return torch.cat(rows)[None].expand(Hk, -1, -1)


def reference(q, k, v, sq, sk, Hk, group, causal):
    outs, lses, q0, k0 = [], [], 0, 0
    for n, m in zip(sq, sk):
        qq = q[q0:q0 + n].float().view(n, Hk, group, 128)
        kk, vv = k[k0:k0 + m].float(), v[k0:k0 + m].float()
        last = torch.arange(n, device=q.device) + m - n if causal else torch.full((n,), m, device=q.device)
        ok = torch.arange(m, device=q.device)[None] <= last[:, None]
        o, ls = [], []
        for h in range(Hk):
            s = (qq[:, h].reshape(n * group, 128) @ kk[:, h].t().contiguous()) * 128 ** -0.5
            s = s.masked_fill(~ok.repeat_interleave(group, 0), float("-inf"))
            lse = torch.logsumexp(s, 1)
            o.append(torch.nan_to_num(torch.exp(s - lse[:, None])).matmul(vv[:, h].contiguous()).view(n, group, 128))
            ls.append(torch.where(torch.isinf(lse), torch.full_like(lse, float("inf")), lse).view(n, group))
        outs.append(torch.stack(o, 1).reshape(n, Hk * group, 128))
        lses.append(torch.stack(ls, 1).reshape(n, Hk * group))
        q0, k0 = q0 + n, k0 + m
    return torch.cat(outs), torch.cat(lses).t()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sq, sk, Hk, group, kind", CASES + GROUP_CASES)
def test_tile_walk(sq, sk, Hk, group, kind, dtype):
    import infllmv2_cuda_impl_amd as ops
    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(7)
    cu = lambda ns: torch.from_numpy(np.cumsum([0] + ns).astype(np.int32)).to(dev)
    q = torch.randn(sum(sq), Hk * group, 128, generator=g).to(dtype).to(dev)
    k = torch.randn(sum(sk), Hk, 128, generator=g).to(dtype).to(dev)
    v = torch.randn(sum(sk), Hk, 128, generator=g).to(dtype).to(dev)
    mask = make_mask(kind, Hk, sq, sk)
    idx = None
    if mask is not None:
        nblk = mask.shape[2]
        idx = torch.where(mask, torch.arange(nblk)[None, None], nblk).sort(2).values
        idx = torch.where(idx == nblk, -1, idx).to(torch.int32).to(dev)
    out, lse, _ = ops.infllmv2_attn_varlen_func(q, k, v, cu(sq), cu(sk), max(sq), max(sk), causal=kind != "acausal", topk_idx=idx,
                                                return_attn_probs=True)
    ref, ref_lse = reference(q, k, v, sq, sk, Hk, group, kind != "acausal")
    err = (out.float() - ref).abs()
    assert err.max() <= 2e-2 and err.mean() <= 1e-3, (err.max().item(), err.mean().item())
    if mask is not None:                                       # (KV heads, tokens x group) -> (heads, tokens)
        lse = lse.view(Hk, sum(sq), group).transpose(1, 2).reshape(Hk * group, sum(sq))
    both = torch.isinf(ref_lse) == torch.isinf(lse)
    assert both.all() and (torch.nan_to_num(lse - ref_lse, nan=0.0).abs() <= 2e-3).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group", [16, 8])
@pytest.mark.parametrize("gain", [1.0, 6.0])
def test_tile_walk_with_a_reference_exponent_that_moves(dtype, group, gain):
    """Rows whose largest score arrives late: a key that is a multiple of one query head's vector, in the row's first, a middle and its last
    block, with a logit far above the rest, so that the block's scores are formed again with sums and outputs that are not zero; with gain 6 the
    running maxima of all rows move on top of that.  Tokens at the ends of wavefronts and tiles."""
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    S, Hk = 2203, 2
    assert _lib.lib.infllmv2_varlen_fwd_dense_tiles(1, S, S, Hk * group, Hk, S, S, 1) == 1
    g = torch.Generator(device="cpu").manual_seed(11)
    q = (torch.randn(S, Hk * group, 128, generator=g) * gain).to(dtype)
    k, v = torch.randn(S, Hk, 128, generator=g).to(dtype), torch.randn(S, Hk, 128, generator=g).to(dtype)
    planted = []
    for i, t in enumerate((S - 1, 2202 - 70, 2047, 2048, 1601, 1600, 1599, 1057, 700, 335, 97, 64, 63)):
        for j, key in enumerate((t, 64 * (t // 128) + 11, 5 + i)):                # last, middle and first block of the token
            h, head = (i + j) % Hk, (5 * i + 3 * j) % group
            row = q[t, h * group + head].float()
            k[key, h] = (row / row.norm() * 60.0).to(dtype)
            planted.append((t, h * group + head, h, key))
    cu = torch.tensor([0, S], dtype=torch.int32).cuda()
    q, k, v = q.cuda(), k.cuda(), v.cuda()
    out, lse, _ = ops.infllmv2_attn_varlen_func(q, k, v, cu, cu, S, S, causal=True, return_attn_probs=True)
    ref, ref_lse = reference(q, k, v, [S], [S], Hk, group, True)
    err = (out.float() - ref).abs()
    # outputs are convex combinations of rows of v whatever the logits: the tolerance of the file.  A logit is a sum of 128 products in fp32,
    # good to 128 2^-24 of its size: that much more on the log-sum-exp.
    assert err.max() <= 2e-2 and err.mean() <= 1e-3, (err.max().item(), err.mean().item())
    assert ((lse - ref_lse).abs() <= 2e-3 + 128 * 2.0 ** -24 * ref_lse.abs()).all()
    # the planted keys do dominate: most of them are their row's largest logit, by far more than the walk lets pass without a new reference
    late = 0
    for t, head, h, key in planted:
        logits = (k[:t + 1, h].float() @ q[t, head].float()) * 128 ** -0.5
        before = logits[:key // 64 * 64]
        late += bool(key >= 64 and logits[key] > before.max() + 5 * math.log(2.0) + 2)
    assert late >= 10, late
