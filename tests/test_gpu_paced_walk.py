"""Stage-2 forward of rows far enough in their sequence to be walked at a pace (behind key block 512): the pace changes the order of a row's blocks, so
rows are checked against fp32 attention, and bit for bit across launches that hold them differently (alone, as a chunk of fewer queries, one KV head,
packed behind another sequence, images packed earlier, causal or not where that is the same), with rows on both sides of the line in one launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # keys, queries, group, window blocks, blocks anywhere, blocks near the end only
    (32768 + 72, 144, 16, 4, 9, 0),                            # the line runs through the queries; 5 blocks in common: steps of every kind
    (70011, 35, 16, 31, 40, 0),                                # more own blocks than common ones; the last group is shared out
    (70011, 64, 8, 31, 0, 70),                                 # all own blocks behind where the front is for most of the walk: more than there are steps
    (48000, 24, 16, 0, 20, 0),                                 # only the first block in common
    (48000, 24, 16, -1, 20, 0),                                # nothing in common: no clock
    (300011, 20, 16, 2, 0, 40),                                # 74 mask words, most of them empty
    (300011, 20, 16, -1, 30, 0),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S, C, group, window, anywhere, late", CASES)
def test_paced_rows(S, C, group, window, anywhere, late, dtype):
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    Hk, nblk = 2, (S + 63) // 64
    gen = torch.Generator(device="cuda").manual_seed(S + C)
    rand = lambda n, heads: torch.randn(n, heads, 128, generator=gen, device="cuda").to(dtype)
    q, k, v = rand(C, Hk * group), rand(S, Hk), rand(S, Hk)
    pos = torch.arange(S - C, S, device="cuda")
    last, at = pos // 64, torch.arange(nblk, device="cuda")
    chosen = ((at[None] <= last[:, None]) & (at[None] > last[:, None] - window) | (at[None] == 0) & (window >= 0))[None].repeat(Hk, 1, 1)
    for n, first in ((anywhere, 0), (late, nblk - 200)):
        if n:
            score = torch.rand(Hk, C, nblk, generator=gen, device="cuda").masked_fill((at[None, None] > last[None, :, None]) | (at < first), -1.0)
            chosen.scatter_(2, score.topk(n, 2).indices, True)
    chosen &= at[None, None] <= last[None, :, None]
    mask = ops.blockmask_to_uint64(chosen.contiguous())[0]

    def run(rows, heads=slice(0, Hk), before=0):
        """The rows of the queries against the keys before their end; `before` tokens of another sequence in front."""
        a, b = rows
        end = S - C + b
        qh = slice(heads.start * group, heads.stop * group)
        qs, ks, vs = q[a:b, qh], k[:end, heads], v[:end, heads]
        m = mask[heads, a:b, :(end + 4095) // 4096]
        if before:
            other = torch.zeros(m.shape[0], before, m.shape[2], dtype=m.dtype, device="cuda")
            other[:, :, 0] = 1
            qs, ks, vs, m = (
                torch.cat([qs[:1].expand(before, -1, -1), qs]), torch.cat([ks[:before], ks]), torch.cat([vs[:before], vs]), torch.cat([other, m], 1))
        cu = lambda *ns: torch.tensor([0] + [sum(ns[:i + 1]) for i in range(len(ns))], dtype=torch.int32, device="cuda")
        cu_q, cu_k = (cu(before, b - a), cu(before, end)) if before else (cu(b - a), cu(end))
        idx = torch.zeros(m.shape[0], m.shape[1], 64, dtype=torch.int32, device="cuda")
        with torch.no_grad():
            out = attend_varlen(qs, ks, vs, cu_q, cu_k, max(b - a, before), end, causal=True, topk_idx=idx, block_mask=m.contiguous())
        return out[before:]

    full = run((0, C))
    assert torch.equal(run((8, C)), full[8:]), "later queries alone"
    assert torch.equal(run((0, 16)), full[:16]), "earlier queries alone"
    assert torch.equal(run((0, C), slice(1, 2)), full[:, group:]), "a head alone"
    assert torch.equal(run((0, C), before=100), full), "packed behind another sequence"
    for t in range(0, C, max(1, C // 6)):
        for h in range(Hk):
            keys = (torch.nonzero(chosen[h, t])[:, 0][:, None] * 64 + torch.arange(64, device="cuda")[None]).reshape(-1)
            keys = keys[keys <= int(pos[t])]
            s = q[t, group * h:group * (h + 1)].float() @ k[keys, h].float().t() * 128 ** -0.5
            err = (full[t, group * h:group * (h + 1)].float() - torch.softmax(s, 1) @ v[keys, h].float()).abs()
            assert err.max() <= 2e-2 and err.mean() <= 1e-3, (t, h)
