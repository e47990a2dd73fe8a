"""A chunk's short groups, which go last in the launch where many keys lie before it: every row is, bit for bit, that of the run over all queries, with one to
five tokens in the last group, one and several sequences, and on either side of the line."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C, held, batch, hk", [(513, 4096, 1, 2), (516, 2048, 1, 2), (1025, 2040, 1, 1), (522, 4096, 1, 2), (525, 4096, 1, 2), (172, 3000, 3, 2), (1026, 33000, 1, 1)])
def test_rows_of_the_full_run(C, held, batch, hk):
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    import infllmv2_cuda_impl_amd as ops
    S, topk = C + held, 16
    gen = torch.Generator(device="cuda").manual_seed(C + held)
    rand = lambda heads: torch.randn(batch * S, heads, 128, generator=gen, device="cuda").to(torch.bfloat16)
    q, k, v = rand(hk * 16), rand(hk), rand(hk)
    nblk = (S + 63) // 64
    last = torch.arange(S, device="cuda").repeat(batch) // 64
    score = torch.rand(hk, batch * S, nblk, generator=gen, device="cuda").masked_fill(torch.arange(nblk, device="cuda")[None, None] > last[None, :, None], -1.0)
    score.scatter_(2, last[None, :, None].expand(hk, batch * S, 1), 2.0)
    best = score.topk(topk, 2)
    idx = torch.where(best.values > 0, best.indices, -1).to(torch.int32)
    cu = lambda n: torch.arange(0, n * batch + 1, n, dtype=torch.int32, device="cuda")
    tail = lambda t: t.view(batch, S, *t.shape[1:])[:, held:].reshape(batch * C, *t.shape[1:])
    run = lambda q, idx, n: attend_varlen(q, k, v, cu(n), cu(S), n, S, causal=True, topk_idx=idx)
    full = run(q, idx, S)
    chunk = run(tail(q), idx.view(hk, batch, S, topk)[:, :, held:].reshape(hk, batch * C, topk).contiguous(), C)
    assert torch.equal(chunk, tail(full))
