"""Calls with more work than one dispatch holds (fewer than 2^32 work-items in a dimension; the runtime starts too few workgroups for more, without an error): they
go out in parts.  Against the same call where it fits, or the definition, at the end of the output."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_thousands_of_sequences_beside_a_long_one():
    """20 000 sequences and a longest of 8192 tokens are 41 million groups of 8 tokens; nearly all of them are empty."""
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    B, Hk = 20000, 2
    gen = torch.Generator(device="cuda").manual_seed(1)
    lens = torch.randint(0, 12, (B,), generator=gen, device="cuda")
    cu = torch.cat([lens.new_zeros(1), lens.cumsum(0)]).to(torch.int32)
    T = int(cu[-1])
    q, k, v, dout = (torch.randn(T, Hk, 128, generator=gen, device="cuda").to(torch.bfloat16) for _ in range(4))
    idx = torch.zeros(Hk, T, 4, dtype=torch.int32, device="cuda")
    mask = torch.ones(Hk, T, 1, dtype=torch.int64, device="cuda")

    def run(longest):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        out = attend_varlen(*leaves, cu, cu, longest, 64, causal=True, topk_idx=idx, block_mask=mask)
        return (out,) + torch.autograd.grad(out, leaves, dout)
    want, got = run(11), run(8192)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])                                    # output and dQ
    for a, b in zip(got[2:], want[2:]):                          # dK, dV: sums of at most 11 tokens in fp32 in any order, rounded once
        assert (a.float() - b.float()).abs().max() <= 2.0 ** -7 * b.float().abs().max()


def test_mask_words_of_many_rows():
    from infllmv2_cuda_impl_amd import _lib
    rows, stream = (1 << 26) + 5, torch.cuda.current_stream().cuda_stream
    want = torch.arange(rows, device="cuda") & 1
    words = torch.full((rows,), -1, dtype=torch.int64, device="cuda")
    _lib.call("infllmv2_blockmask_to_uint64", stream, want.to(torch.uint8).data_ptr(), words.data_ptr(), rows, 1, 1)
    assert torch.equal(words, want)
    words.fill_(-1)
    idx = (want - 1).to(torch.int32)                             # -1: none, 0: the first block
    _lib.call("infllmv2_topk_to_uint64", stream, idx.data_ptr(), words.data_ptr(), rows, 1, 1, 1)
    assert torch.equal(words, want)


def test_mask_bytes_of_many_rows():
    from infllmv2_cuda_impl_amd import _lib
    rows = (1 << 29) + 5                                         # 8 bytes a thread, 64 a row: 34 GB
    words = torch.full((rows,), 5, dtype=torch.int64, device="cuda")
    words[-3:] = -2
    out = torch.full((rows, 64), 7, dtype=torch.uint8, device="cuda")
    _lib.call("infllmv2_uint64_to_bool", torch.cuda.current_stream().cuda_stream, words.data_ptr(), out.data_ptr(), rows, 64, 1)
    for at in (0, rows // 2, rows - 4):
        assert out[at].tolist() == [1, 0, 1] + [0] * 61
    assert out[-1].tolist() == out[-3].tolist() == [0] + [1] * 63
