"""The order of a launch's token groups, in which heads take turns or not: every token of every head and sequence is walked once, forward and backward, for
1 to 35 groups to a sequence, a number of heads that is no power of two, empty sequences, and launches on either side of the line.  Against the
same tokens of one (sequence, KV head) at a time, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens, hk", [([5], 3), ([8, 0, 17], 3), ([128, 130], 2), ([136], 5), ([273, 1, 64], 3), ([600] * 7, 8), ([512] * 8, 8), ([520] * 8, 8)])
def test_every_group_once(lens, hk):
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    import infllmv2_cuda_impl_amd as ops
    gen = torch.Generator(device="cuda").manual_seed(sum(lens) + hk)
    total, most = sum(lens), max(lens)
    rand = lambda heads: torch.randn(total, heads, 128, generator=gen, device="cuda").to(torch.bfloat16)
    q, k, v, dout = rand(4 * hk), rand(hk), rand(hk), rand(4 * hk)
    nblk = (most + 63) // 64
    last = torch.cat([torch.arange(n, device="cuda") // 64 for n in lens])
    chosen = (torch.rand(hk, total, nblk, generator=gen, device="cuda") < 0.6) | (torch.arange(nblk, device="cuda")[None] == last[:, None])[None]
    mask = ops.blockmask_to_uint64(chosen.contiguous())[0]

    def run(q, k, v, dout, mask, ns):
        cu = torch.tensor([sum(ns[:i]) for i in range(len(ns) + 1)], dtype=torch.int32, device="cuda")
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        idx = torch.zeros(k.shape[1], q.shape[0], nblk, dtype=torch.int32, device="cuda")
        out = attend_varlen(*leaves, cu, cu, max(ns), max(ns), causal=True, topk_idx=idx, block_mask=mask)
        return out.detach(), torch.autograd.grad(out, leaves, dout)[0]

    out, dq = run(q, k, v, dout, mask, lens)
    start = 0
    for n in lens:
        for h in range(hk):
            if n == 0 or (len(lens) > 3 and (start // n + h) % 3 != 0):
                continue
            rows, heads = slice(start, start + n), slice(4 * h, 4 * h + 4)
            one, one_dq = run(q[rows, heads], k[rows, h:h + 1], v[rows, h:h + 1], dout[rows, heads], mask[h:h + 1, rows].contiguous(), [n])
            assert torch.equal(out[rows, heads], one) and torch.equal(dq[rows, heads], one_dq), (n, h)
        start += n
