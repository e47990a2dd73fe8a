"""dK/dV with a group's tokens dealt out evenly: items of 64 to 256 tokens, sequences that start and end inside a group of 2048 tokens and inside a word
of 64, and inputs one token longer than the rule serves.  dout is 1 in column t % 128 of token t and 0 elsewhere, and rows of P add up to one: column d
of dv, summed over a sequence's keys, is the number of (token, head) rows of the tokens with t % 128 = d.  A token that one block leaves out, or counts
twice, moves the sum by the block's share of 16 rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # lengths, KV heads, blocks selected (0: no mask)
    ([65], 1, 16), ([2047], 1, 16), ([2049, 63, 1], 2, 16), ([130, 3000, 700], 1, 32), ([1500, 2600], 2, 0), ([6145], 2, 32),
    ([28672], 1, 16), ([28673], 1, 16), ([14000, 14672], 1, 32), ([5000] * 6, 1, 32),
]


def random_blocks(lens, Hk, topk, g):
    """Each token's own block, the sequence's first, and random ones among those it can see."""
    out = []
    for n in lens:
        blocks = (n + 63) // 64
        own = torch.arange(n, device="cuda") // 64
        score = torch.rand(Hk, n, max(blocks, topk), generator=g, device="cuda")
        col = torch.arange(score.shape[-1], device="cuda")
        score += 2.0 * ((col == own[:, None]) | (col == 0))
        score.masked_fill_(col > own[:, None], -1.0)
        val, idx = score.topk(topk, dim=-1)
        idx = idx.masked_fill(val < 0, 1 << 30).sort(dim=-1).values
        out.append(idx.masked_fill(idx == 1 << 30, -1).int())
    return torch.cat(out, dim=1).contiguous()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens, Hk, topk", CASES)
def test_every_token_is_dealt_out_once(lens, Hk, topk, dtype):
    import infllmv2_cuda_impl_amd as ops
    g = torch.Generator(device="cuda").manual_seed(len(lens))
    total, mx = sum(lens), max(lens)
    q, k, v = (torch.randn(total, h, 128, generator=g, device="cuda").to(dtype).requires_grad_(True) for h in (16 * Hk, Hk, Hk))
    cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device="cuda")
    idx = random_blocks(lens, Hk, topk, g) if topk else None
    dout = torch.nn.functional.one_hot(torch.arange(total, device="cuda") % 128, 128).to(dtype)[:, None].expand(-1, 16 * Hk, -1).contiguous()
    dk = {}
    for deterministic in (False, True):
        out = ops.infllmv2_attn_varlen_func(q, k, v, cu, cu, mx, mx, causal=True, topk_idx=idx, deterministic=deterministic)
        dk[deterministic], dv = torch.autograd.grad(out, (k, v), dout)
        for i in range(len(lens)):
            a, b = sum(lens[:i]), sum(lens[:i + 1])
            want = 16.0 * dout[a:b, 0].double().sum(0)
            got = dv[a:b].double()
            # dv and P are rounded to 16 bits: a relative error of at most 2^-9 each, independent from element to element (four deviations)
            bound = 2.0 ** -9 * (4 * got.norm(dim=0) + 4 * want.sqrt()) + 1e-3
            worst = ((got.sum(0) - want).abs() - bound).max().item()
            assert worst <= 0, (deterministic, i, worst)
    a, b = dk[False].float(), dk[True].float()
    # the same products summed in float in another order, then rounded once to 16 bits
    assert ((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-4 * b.abs().max()).all()
