"""Stage 1 of few queries against many compressed keys, where workgroups share a block of tokens: scores and pooled scores of the last queries of a sequence are,
bit for bit, the rows of all its queries (which no one shares), with one and several sequences, tile counts that do not divide, and early
queries that see few tiles or none, and groups of up to 8 heads, of which two tokens share the rows of a product."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("n, m, group", [(n, m, 16) for n, m in ((9000, 104), (9000, 808), (20016, 112), (20016, 304), (40000, 1600), (8200, 1800))] +      # n - m a multiple of 64: the same visible keys
                         [(9000, 104, 8), (9000, 808, 1), (20016, 304, 8), (20016, 112, 2), (40000, 1600, 4), (8200, 1800, 8)])
def test_last_queries_are_rows_of_all(n, m, group, causal, dtype):
    import infllmv2_cuda_impl_amd as ops
    gen = torch.Generator(device="cuda").manual_seed(n + m)
    hk = 1
    r = lambda rows, heads: torch.randn(rows, heads, 128, generator=gen, device="cuda").to(dtype)
    q, k = r(n, group * hk), r(n, hk)
    cu = lambda *ns: torch.tensor(np.cumsum((0,) + ns), dtype=torch.int32, device="cuda")
    (fine, cu_f), (coarse, cu_c) = ops.compress_keys(k, cu(n), n, 32, 16), ops.compress_keys(k, cu(n), n, 128, 64)
    most = (n - 32) // 16 + 1
    whole = lambda f, *more: f(q, fine, coarse, cu(n), cu_f, cu_c, n, most, *more, causal=causal)
    part = lambda f, *more: f(q[-m:], fine, coarse, cu(m), cu_f, cu_c, m, most, *more, causal=causal)
    assert torch.equal(part(ops.infllmv2_attn_stage1), whole(ops.infllmv2_attn_stage1)[:, -m:])
    # pooled: behind n - m cached tokens, at the same positions
    a = ops.infllmv2_attn_stage1_pooled(q[-m:], fine, coarse, cu(m), cu_f, cu_c, m, most, 3, 1, cache_len=n - m, causal=causal)
    b = ops.infllmv2_attn_stage1_pooled(q, fine, coarse, cu(n), cu_f, cu_c, n, most, 3, 1, cache_len=0, causal=causal)
    assert torch.equal(a, b[:, -m:])


@pytest.mark.parametrize("group", [16, 8, 4, 1])
@pytest.mark.parametrize("causal", [True, False])
def test_packed_sequences(causal, group):
    import infllmv2_cuda_impl_amd as ops
    gen = torch.Generator(device="cuda").manual_seed(2)
    hk, sq, sk = 2, [40, 0, 3, 130, 17], [5000, 900, 70, 12000, 20]
    r = lambda rows, heads: torch.randn(rows, heads, 128, generator=gen, device="cuda").to(torch.bfloat16)
    cu = lambda ns: torch.tensor(np.cumsum([0] + list(ns)), dtype=torch.int32, device="cuda")
    q, k = r(sum(sq), group * hk), r(sum(sk), hk)
    (fine, cu_f), (coarse, cu_c) = ops.compress_keys(k, cu(sk), max(sk), 32, 16), ops.compress_keys(k, cu(sk), max(sk), 128, 64)
    most = (max(sk) - 32) // 16 + 1
    got = ops.infllmv2_attn_stage1(q, fine, coarse, cu(sq), cu_f, cu_c, max(sq), most, causal=causal)
    # the same rows among many others, so that the launch fills the chip: every sequence 30 times
    rep = lambda x, ns, c: torch.cat([x[c[b]:c[b + 1]] for b in range(len(ns))] * 30)
    cq, cf, cc = np.cumsum([0] + sq), cu_f.tolist(), cu_c.tolist()
    lens = lambda c: [c[b + 1] - c[b] for b in range(len(c) - 1)]
    many = ops.infllmv2_attn_stage1(rep(q, sq, cq), rep(fine, sq, cf), rep(coarse, sq, cc), cu(sq * 30), cu(lens(cf) * 30), cu(lens(cc) * 30), max(sq), most,
                                    causal=causal)
    assert torch.equal(got, many[:, :sum(sq)])
