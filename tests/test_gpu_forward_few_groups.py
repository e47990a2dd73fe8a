"""The forward of few tokens, where two, four or eight workgroups share the 8 tokens of a group: output and LSE of the last queries of a sequence are, bit for
bit, the rows of all its queries (which no one shares), around 32, 64 and 128 groups, with a last group of up to 4 tokens (whose rows several
wavefronts share), short and long sequences, masked and dense; and a caller may still have the output written over Q."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def random_mask(S, Hk, blocks, gen):
    """(Hk, S, words) int64: so many random blocks for each token, future ones among them, with the first and the token's own."""
    nblk = (S + 63) // 64
    chosen = torch.zeros(Hk, S, (nblk + 63) // 64 * 64, dtype=torch.bool, device="cuda")
    chosen.scatter_(2, torch.randint(0, nblk, (Hk, S, blocks), generator=gen, device="cuda"), True)
    chosen[..., 0] = True
    chosen.scatter_(2, (torch.arange(S, device="cuda") // 64)[None, :, None].expand(Hk, S, 1), True)
    import infllmv2_cuda_impl_amd as ops
    return ops.blockmask_to_uint64(chosen.contiguous())[0].contiguous()


def forward(q, k, v, mask, S, causal, over_q=False):
    from infllmv2_cuda_impl_amd import C
    out = q.clone() if over_q else torch.full_like(q, float("nan"))
    cu = lambda n: torch.tensor([0, n], dtype=torch.int32, device="cuda")
    out, lse, _, _ = C.varlen_fwd(out if over_q else q, k, v, out, cu(q.shape[0]), cu(S), None, None, None, None, q.shape[0], S, 0.0, 128 ** -0.5, False, causal,
                                  -1, -1, 0.0, False, None, mask)
    return out, lse


CASES = [(2100, 1, 9), (2100, 1, 252), (2100, 1, 260), (2100, 1, 508), (2100, 1, 516), (2049, 1, 513), (2051, 1, 515), (2053, 1, 1029), (2100, 1, 1020), (2100, 1, 1028), (2100, 2, 252), (2100, 2, 516),
         (2100, 4, 108), (33010, 1, 18), (33010, 1, 1018), (9000, 2, 200)]


@pytest.mark.parametrize("dtype, causal, masked", [(torch.bfloat16, True, True), (torch.float16, True, True), (torch.bfloat16, False, True), (torch.bfloat16, True, False)])
@pytest.mark.parametrize("S, Hk, m", CASES)
def test_last_queries_are_rows_of_all(S, Hk, m, dtype, causal, masked):
    gen = torch.Generator(device="cuda").manual_seed(S + m)
    r = lambda heads: torch.randn(S, heads, 128, generator=gen, device="cuda").to(dtype)
    q, k, v = r(16 * Hk), r(Hk), r(Hk)
    mask = random_mask(S, Hk, 20, gen) if masked else None
    first = (S - m) // 8 * 8                                   # chunks start at groups
    whole, lse = (t.clone() for t in forward(q, k, v, mask, S, causal))
    chunk = q[first:].contiguous(), k, v, mask[:, first:].contiguous() if masked else None, S, causal
    part, part_lse = forward(*chunk)
    whole, lse = whole[first:], lse.view(-1, S)[:, first:]
    if masked:
        assert torch.equal(part, whole) and torch.equal(part_lse, lse)
    else:                                                      # the two may take different walks: P and the output are each rounded to 8 bits, twice
        assert (part.float() - whole.float()).abs().max().item() <= 2.0 ** -7 * v.float().abs().max().item()
        torch.testing.assert_close(part_lse, lse, rtol=0, atol=1e-4)
    over, over_lse = forward(*chunk, over_q=True)
    assert torch.equal(over, part) and torch.equal(over_lse, part_lse)
