"""The blocks of a window, written directly, are those that pooling marks +inf on a score tensor without columns and the selection then takes: bit for
bit, indices and mask, over batches, positions, rows at the edges of blocks and of mask words, and windows longer than the sequence."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # lengths, positions (None: prefill), heads, local, init, block
    ([1], None, 1, 4, 1, 64), ([64, 65, 1, 4096], None, 2, 0, 0, 64), ([4097], None, 4, 70, 3, 64), ([300, 5000], None, 1, 31, 1, 64), ([130], None, 2, 2, 5, 64),
    ([1, 1, 1], [0, 4095, 4096], 2, 8, 1, 64), ([1], [100000], 1, 31, 1, 64), ([700, 33], [64, 129], 2, 3, 2, 32), ([2000], None, 1, -1, 2, 64),
]


@pytest.mark.parametrize("lens, positions, heads, local, init, block", CASES)
def test_window_blocks(lens, positions, heads, local, init, block):
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    cu = ints([sum(lens[:i]) for i in range(len(lens) + 1)])
    held, most = (ints([0] * len(lens)), 0) if positions is None else (ints(positions), max(positions))
    idx, mask = _lib.host.window_blocks(heads, sum(lens), cu, None if positions is None else held, max(lens), most, local, init, block)
    scores = torch.empty((heads, sum(lens), 0), dtype=torch.bfloat16, device="cuda")
    pooled = ops.max_pooling_1d_varlen(scores, cu, torch.zeros_like(cu), held, max(lens), 0, local, init, block_size=block, stride=16, max_cache_len=most)
    want_idx, want_mask = ops.topk_blocks(pooled, init + local + 1, return_mask=True, by_index=True, drop_unreachable=True)
    assert torch.equal(idx, want_idx) and torch.equal(mask, want_mask)


WINDOWS = [([40000], 1, 16, 4, 1), ([66000, 33], 1, 8, 2, 0), ([700, 9000, 65], 2, 16, 31, 1), ([5000], 2, 8, 80, 66)]   # lengths, KV heads, group, local, init


@pytest.mark.parametrize("lens, Hk, group, local, init", WINDOWS)
def test_windows_by_tiles(lens, Hk, group, local, init):
    """Told that neighbouring rows are alike, forward and dQ go by tiles, whose walk jumps over the words between the first blocks and the window (more than
    eight of them in the first two cases): against the walk per token on the same mask."""
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    g = torch.Generator(device="cuda").manual_seed(5)
    total, mx = sum(lens), max(lens)
    q, k, v = (torch.randn(total, h, 128, generator=g, device="cuda").to(torch.bfloat16).requires_grad_(True) for h in (group * Hk, Hk, Hk))
    dout = torch.randn(total, group * Hk, 128, generator=g, device="cuda").to(torch.bfloat16)
    cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device="cuda")
    idx, mask = _lib.host.window_blocks(Hk, total, cu, None, mx, 0, local, init, 64)
    most = -(init + local + 1)
    assert _lib.lib.infllmv2_varlen_fwd_masked_tiles(len(lens), total, total, group * Hk, Hk, mx, mx, 1, most) == 1
    got, want = [], []
    for alike, result in ((True, got), (False, want)):
        out = attend_varlen(q, k, v, cu, cu, mx, mx, causal=True, topk_idx=idx if alike else None, block_mask=mask, alike=alike)
        result += [out] + list(torch.autograd.grad(out, (q, k, v), dout))
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
        # P, dS and the results are rounded to 8 bits of mantissa on either side, in other orders of summation: 2^-9 each
        assert (a.float() - b.float()).norm() <= 2.0 ** -7 * b.float().norm(), name
        rows = (a.float() - b.float()).norm(dim=-1) - 2.0 ** -4 * b.float().norm(dim=-1)
        assert rows.max() <= 1e-2, (name, rows.max().item())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens, Hk, group, local, init", WINDOWS)
def test_layer_window_against_fp32_attention(lens, Hk, group, local, init, dtype):
    """Output and dQ of the layer's window branch on sampled tokens (the edges of sequences, of the first blocks, of mask words, of tiles and some at random) against
    fp32 softmax attention over exactly the window's keys; tolerances of the forward and backward tests: 2e-2 and 1e-3 of values of order one."""
    import infllmv2_cuda_impl_amd as ops
    gen = torch.Generator(device="cuda").manual_seed(8)
    total, mx = sum(lens), max(lens)
    rand = lambda h: torch.randn(total, h, 128, generator=gen, device="cuda").to(dtype)
    q, k, v, dout = rand(group * Hk).requires_grad_(True), rand(Hk), rand(Hk), rand(group * Hk)
    cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device="cuda")
    out = ops.InfLLMv2Attention(local_blocks=local, init_blocks=init, selection="window")(q, k, v, cu, mx)
    dq, = torch.autograd.grad(out, q, dout)
    start, worst = 0, []
    for n in lens:
        near = [0, 1, 15, 16, 31, 63, 64, 65, 64 * (local + 1) - 1, 64 * (local + 1), 64 * (local + init + 1), 64 * (local + init + 1) + 15, 4095, 4096, n - 17, n - 2, n - 1]
        tokens = sorted({t for t in near if 0 <= t < n} | set(torch.randint(0, n, (24,), generator=torch.Generator().manual_seed(n)).tolist()))
        for t in tokens:
            at = torch.arange(t + 1, device="cuda")
            at = at[(at // 64 < init) | (at // 64 >= t // 64 - local)]
            kk, vv = k[start + at].float().transpose(0, 1).contiguous(), v[start + at].float().transpose(0, 1).contiguous()        # (Hk, keys, 128)
            qq, do = (x[start + t].detach().float().view(Hk, group, 128) for x in (q, dout))
            p = torch.softmax(qq @ kk.transpose(1, 2).contiguous() * 128 ** -0.5, 2)
            ref = p @ vv
            dp = do @ vv.transpose(1, 2).contiguous()
            ref_dq = (p * (dp - (p * dp).sum(2, keepdim=True)) * 128 ** -0.5) @ kk
            worst.append(torch.stack([x for a, b in ((out, ref), (dq, ref_dq)) for e in [(a[start + t].detach().float().view(Hk, group, 128) - b).abs()]
                                      for x in (e.max(), e.mean())]))
        start += n
    worst = torch.stack(worst)
    assert worst[:, 0].max() <= 2e-2 and worst[:, 1].mean() <= 1e-3, worst.max(0).values.tolist()
    assert worst[:, 2].max() <= 2e-2 and worst[:, 3].mean() <= 1e-3, worst.max(0).values.tolist()
