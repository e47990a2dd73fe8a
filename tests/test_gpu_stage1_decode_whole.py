"""Stage 1 of a decode step in one launch (few and short sequences) against the two launches that others take: the same bits, at the lengths where
coarse and fine tiles begin, where a token completes windows, and on either side of the rule.  A batch that holds the same sequences several times over has too
many workgroups for the one launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# coarse tiles begin at 128 + 64 * 64 k tokens, fine ones at 32 + 16 * 64 k; the rule's five coarse tiles are full from 20 544 to 20 607
LENS = [1, 31, 32, 127, 128, 1039, 1040, 1055, 1056, 1057, 4159, 4160, 4223, 4224, 4287, 8192, 16447, 16448, 20479, 20542, 20543, 20606, 20607]
COPIES = 16


def caches(ops, lens, cap, Hk, dtype, gen):
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(dtype)
    B = len(lens)
    k, v = mk(B, cap, Hk, 128), mk(B, cap, Hk, 128)
    L = torch.tensor(lens, dtype=torch.int32, device="cuda")
    fine, coarse = mk(B, cap // 16 + 1, Hk, 128), mk(B, cap // 64 + 1, Hk, 128)     # garbage behind the valid rows
    fl, cl = ops.compress_keys_cache_pair(k, L, (32, 16, fine), (128, 64, coarse))
    return k, v, L, fine, coarse, fl, cl


@pytest.mark.parametrize("dtype, Hk, G", [(torch.bfloat16, 2, 16), (torch.float16, 1, 8), (torch.bfloat16, 3, 1)])
def test_step(dtype, Hk, G):
    """Append, lengths, compressed keys, scores and selection; what the fine and coarse caches held in the new rows does not matter (NaN)."""
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(3)
    for n in LENS:
        cap = (n + 64) // 64 * 64 + 64
        k, v, L, fine, coarse, fl, cl = caches(ops, [n, max(1, n // 2)], cap, Hk, dtype, gen)
        for cache, rows in ((fine, fl), (coarse, cl), (k, L), (v, L)):
            for b in range(2):
                cache[b, int(rows[b]):] = float("nan")
        mk = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(dtype)
        q, kn, vn = mk(2, 1, Hk * G, 128), mk(2, 1, Hk, 128), mk(2, 1, Hk, 128)

        def step(times):
            many = lambda t: t.repeat(times, *[1] * (t.dim() - 1)).contiguous()
            args = [many(t) for t in (q, kn, vn, k, v, fine, coarse)]
            lens, fine_lens, coarse_lens = many(L), many(fl), many(cl)
            new, mask = _lib.host.decode_step(*args, lens, 0, fine_lens, coarse_lens, n + 1, 32, 16, 64, 8, 2, 1, 128 ** -0.5)
            return [mask, new, fine_lens, coarse_lens] + args[3:]
        times = max(1, 257 // (2 * Hk * max(1, ((n + 1 - 32) // 16 + 64) // 64)) + 1)
        for got, want in zip(step(1), step(times)):
            for c in range(0, times, max(1, times - 1)):
                a, b = got, want[2 * c:2 * c + 2]
                assert torch.equal(a.view(torch.int16) if a.is_floating_point() else a, b.view(torch.int16) if b.is_floating_point() else b), n
        # one sequence, its length on the host
        one = [t[:1].clone() for t in (q, kn, vn, k, v, fine, coarse)]
        new, mask = _lib.host.decode_step(*one, None, n, None, None, n + 1, 32, 16, 64, 8, 2, 1, 128 ** -0.5)
        ref = step(1)
        assert int(new) == n + 1 and torch.equal(mask, ref[0][:1])
        for a, b in zip(one[3:], ref[4:]):
            assert torch.equal(a.view(torch.int16), b[:1].view(torch.int16)), n


@pytest.mark.parametrize("kernel, stride", [(16, 8), (48, 16), (20, 16)])          # a coarse window of 192 rows is more than the one launch holds
def test_step_with_other_windows(kernel, stride):
    from infllmv2_cuda_impl_amd import _lib
    import infllmv2_cuda_impl_amd as ops
    gen = torch.Generator(device="cuda").manual_seed(4)
    Hk, block, cap = 2, 4 * stride, 3072
    for n in (4 * kernel - 1, 4 * kernel + 4 * stride - 1, 1500, 2047):
        mk = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(torch.bfloat16)
        k, v, L = mk(1, cap, Hk, 128), mk(1, cap, Hk, 128), torch.tensor([n], dtype=torch.int32, device="cuda")
        fine, coarse = mk(1, cap // stride + 1, Hk, 128), mk(1, cap // (4 * stride) + 1, Hk, 128)
        fl, cl = ops.compress_keys_cache_pair(k, L, (kernel, stride, fine), (4 * kernel, 4 * stride, coarse))
        q, kn, vn = mk(1, 1, 32, 128), mk(1, 1, Hk, 128), mk(1, 1, Hk, 128)
        res = []
        for times in (1, 257):
            many = lambda t: t.repeat(times, *[1] * (t.dim() - 1)).contiguous()
            args = [many(t) for t in (q, kn, vn, k, v, fine, coarse)]
            lens = [many(L), many(fl), many(cl)]
            topk = 8 if block == 64 else 0                     # the pooling is fused for blocks of 64 only
            _, mask = _lib.host.decode_step(*args, lens[0], 0, lens[1], lens[2], n + 1, kernel, stride, block, topk, 2, 1, 128 ** -0.5)
            res.append(([mask] if topk else []) + lens[1:] + args[3:])
        for a, b in zip(*res):
            assert torch.equal(a, b[:1]) and torch.equal(a, b[-1:])


@pytest.mark.parametrize("dtype, Hk, G", [(torch.bfloat16, 2, 16), (torch.float16, 1, 4)])
def test_scores_of_one_query(dtype, Hk, G):
    """Pooled and as rows of scores, caches and packed keys, causal or not, coarse keys or the fine ones again for the log-sum-exp."""
    import infllmv2_cuda_impl_amd as ops
    gen = torch.Generator(device="cuda").manual_seed(5)
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(dtype)
    for n in LENS:
        cap = (n + 64) // 64 * 64 + 64
        k, v, L, fine, coarse, fl, cl = caches(ops, [n], cap, Hk, dtype, gen)
        q = mk(1, 1, Hk * G, 128)
        times = 257 // (Hk * max(1, (int(fl) + 63) // 64)) + 1
        many = lambda t: t.repeat(times, *[1] * (t.dim() - 1)).contiguous()
        if int(fl) == 0:
            continue
        one = ops.infllmv2_attn_stage1_kvcache(q, fine, coarse, fl, cl, L, 2, 1, max_cache_len=n)
        two = ops.infllmv2_attn_stage1_kvcache(many(q), many(fine), many(coarse), many(fl), many(cl), many(L), 2, 1, max_cache_len=n)
        assert torch.equal(one[0].view(torch.int16), two[0].view(torch.int16)) and torch.equal(one[0].view(torch.int16), two[-1].view(torch.int16)), n
        if int(cl) == 0:
            continue
        cu = lambda ns: torch.tensor([0] + list(torch.tensor(ns).cumsum(0)), dtype=torch.int32, device="cuda")
        for c_rows in (coarse[0, :int(cl)], fine[0, :int(fl)]):
            for causal in (False, True):
                def scores(t):
                    return ops.infllmv2_attn_stage1(q[0].repeat(t, 1, 1), fine[0, :int(fl)].repeat(t, 1, 1), c_rows.repeat(t, 1, 1), cu([1] * t),
                                                    cu([int(fl)] * t), cu([len(c_rows)] * t), 1, int(fl), causal=causal)
                a, b = scores(1), scores(times)
                assert torch.equal(a[:, 0].view(torch.int16), b[:, -1].view(torch.int16)), (n, causal)
