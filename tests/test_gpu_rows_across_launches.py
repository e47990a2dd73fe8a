"""A masked row is the same bit for bit whatever else its launch holds: a chunk of queries against the keys before it, a KV head on its own, a sequence
alone or packed with others.  Forward, dQ and (deterministic mode) dK / dV, at sizes where tiles of 256 query rows and groups of 8 tokens take turns
in being the faster walk.  Chunks start at multiples of 8 tokens, which is half a tile for groups of 16 and a quarter for groups of 8."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # tokens, queries of the chunk, KV heads, group, blocks selected (negative: a window of so many, the layer's own walk)
    (4096, 512, 2, 16, 64), (2000, 776, 2, 16, 64), (3000, 1000, 4, 8, 32), (2500, 1492, 4, 16, 16),
    (4096, 504, 2, 16, -20), (2000, 776, 2, 16, -6), (3000, 1000, 4, 8, -9), (9000, 1008, 2, 8, -33),
]


def packed_mask(S, Hk, blocks, gen):
    """(Hk, S, words) int64, and the index list's width: random blocks of what a token sees with the first and its own, or a window."""
    nblk = (S + 63) // 64
    last = torch.arange(S, device="cuda") // 64
    at = torch.arange(nblk, device="cuda")
    if blocks < 0:
        near = (at[None] <= last[:, None]) & (at[None] > last[:, None] + blocks + 1)
        chosen = (near | (at[None] == 0))[None].expand(Hk, S, nblk)
    else:
        score = torch.rand(Hk, S, nblk, generator=gen, device="cuda").masked_fill(at[None, None] > last[None, :, None], -1.0)
        score[..., 0] = 2.0
        score.scatter_(2, last[None, :, None].expand(Hk, S, 1), 2.0)
        best = score.topk(min(blocks, nblk), 2)
        chosen = torch.zeros(Hk, S, nblk, dtype=torch.bool, device="cuda").scatter_(2, best.indices, best.values > 0)
    import infllmv2_cuda_impl_amd as ops
    return ops.blockmask_to_uint64(chosen.contiguous())[0], abs(blocks)


@pytest.mark.parametrize("S, C, Hk, group, blocks", CASES)
def test_rows_do_not_depend_on_the_launch(S, C, Hk, group, blocks):
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    gen = torch.Generator(device="cuda").manual_seed(91)
    rand = lambda heads: torch.randn(S, heads, 128, generator=gen, device="cuda").to(torch.bfloat16)
    q, k, v, dout = rand(Hk * group), rand(Hk), rand(Hk), rand(Hk * group)
    mask, width = packed_mask(S, Hk, blocks, gen)

    def run(q, k, v, dout, mask, q_lens, k_lens):
        cu = lambda ns: torch.tensor([sum(ns[:i]) for i in range(len(ns) + 1)], dtype=torch.int32, device="cuda")
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        idx = torch.zeros(k.shape[1], q.shape[0], width, dtype=torch.int32, device="cuda")     # with a mask at hand only its width counts
        out = attend_varlen(*leaves, cu(q_lens), cu(k_lens), max(q_lens), max(k_lens), causal=True, deterministic=True, topk_idx=idx,
                            block_mask=mask, alike=blocks < 0)
        return [out.detach()] + list(torch.autograd.grad(out, leaves, dout))

    full = run(q, k, v, dout, mask, [S], [S])
    chunk = run(q[S - C:], k, v, dout[S - C:], mask[:, S - C:].contiguous(), [C], [S])
    for name, a, b in zip(("out", "dq"), chunk, full):
        assert torch.equal(a, b[S - C:]), ("chunk", name)
    a0, a1 = S - C, S - C + 264                                # a chunk that later ones follow: those tokens as queries, what comes before their end as keys
    inner = run(q[a0:a1], k[:a1], v[:a1], dout[a0:a1], mask[:, a0:a1].contiguous(), [a1 - a0], [a1])
    for name, a, b in zip(("out", "dq"), inner, full):
        assert torch.equal(a, b[a0:a1]), ("inner chunk", name)
    for h in range(Hk):
        hs = slice(group * h, group * (h + 1))
        one = run(q[:, hs], k[:, h:h + 1], v[:, h:h + 1], dout[:, hs], mask[h:h + 1].contiguous(), [S], [S])
        for name, a, b in zip(("out", "dq", "dk", "dv"), one, (full[0][:, hs], full[1][:, hs], full[2][:, h:h + 1], full[3][:, h:h + 1])):
            assert torch.equal(a, b), ("head", h, name)
    again = lambda t, dim=0: torch.cat([t, t], dim)
    twice = run(again(q), again(k), again(v), again(dout), again(mask, 1), [S, S], [S, S])
    for name, a, b in zip(("out", "dq"), twice, full):
        assert torch.equal(a, again(b)), ("packed", name)
