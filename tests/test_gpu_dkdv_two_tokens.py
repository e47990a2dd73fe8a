"""dK/dV of groups of up to 8 query heads, two tokens to a tile of 16 rows and four to a step: items whose tokens are one, two, three or four more than a multiple of
four, tokens of a tile in different words of 64, partial last blocks, short and long slices, the deterministic mode, and tokens too far apart for the tiles to be shared."""
import pytest
import torch

from test_gpu_dkdv_even import random_blocks
from test_gpu_shared_by_some import attend, inputs, reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens, Hk, group, topk", [([1], 1, 8, 16), ([3], 2, 8, 0), ([65, 2, 66, 67], 1, 4, 16), ([2049, 63, 1], 2, 8, 16), ([130, 3000, 700], 1, 1, 32),
                                                   ([28672], 1, 8, 16), ([28673], 1, 8, 16), ([5000] * 6, 1, 2, 32), ([9001, 2050], 2, 8, 0)])
def test_every_token_counts_once(lens, Hk, group, topk, dtype):
    """dout is 1 in column t % 128 of token t: summed over a sequence's keys, column d of dv is the number of rows of the tokens with t % 128 = d."""
    import infllmv2_cuda_impl_amd as ops
    g = torch.Generator(device="cuda").manual_seed(len(lens))
    total, mx = sum(lens), max(lens)
    q, k, v = (torch.randn(total, h, 128, generator=g, device="cuda").to(dtype).requires_grad_(True) for h in (group * Hk, Hk, Hk))
    cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device="cuda")
    idx = random_blocks(lens, Hk, topk, g) if topk else None
    dout = torch.nn.functional.one_hot(torch.arange(total, device="cuda") % 128, 128).to(dtype)[:, None].expand(-1, group * Hk, -1).contiguous()
    dk = {}
    for deterministic in (False, True):
        out = ops.infllmv2_attn_varlen_func(q, k, v, cu, cu, mx, mx, causal=True, topk_idx=idx, deterministic=deterministic)
        dk[deterministic], dv = torch.autograd.grad(out, (k, v), dout)
        for i in range(len(lens)):
            a, b = sum(lens[:i]), sum(lens[:i + 1])
            want = float(group) * dout[a:b, 0].double().sum(0)
            got = dv[a:b].double()
            # dv and P are rounded to 16 bits: a relative error of at most 2^-9 each, independent from element to element (four deviations)
            bound = 2.0 ** -9 * (4 * got.norm(dim=0) + 4 * want.sqrt()) + 1e-3
            assert ((got.sum(0) - want).abs() - bound).max() <= 0, (deterministic, i)
    a, b = dk[False].float(), dk[True].float()
    # the same products summed in float in another order, then rounded once to 16 bits
    assert ((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-4 * b.abs().max()).all()


@pytest.mark.parametrize("far", [False, True])
@pytest.mark.parametrize("S, group, tail", [(700, 8, 0), (64 * 65, 8, 61), (333, 4, 0), (64 * 70 + 3, 2, 200)])
def test_gradients(S, group, tail, far):
    q, k, v, dout, pos, chosen, mask = inputs(S, group, tail, torch.bfloat16)
    C = q.shape[0]
    if far:                                                    # the tokens' rows of q lie 2.1 MiB apart
        if C > 350:
            C = 350                                            # the last queries are enough
            q, dout, pos, chosen, mask = q[-C:], dout[-C:].contiguous(), pos[-C:], chosen[:, -C:], mask[:, -C:].contiguous()
        wide = torch.empty(C, (1 << 20) + 4096, dtype=q.dtype, device="cuda")
        q = wide[:, :q.shape[1] * 128].unflatten(1, (q.shape[1], 128)).copy_(q)
    leaves = [q.detach().requires_grad_(True)] + [t.clone().requires_grad_(True) for t in (k, v)]
    dk, dv = torch.autograd.grad(attend(*leaves, mask), leaves, dout)[1:]
    for h in range(k.shape[1]):
        wide = [t.detach().float().requires_grad_(True) for t in (q, k, v)]
        ref = torch.cat([reference(*wide, pos, chosen, h, slice(a, min(C, a + 512))) for a in range(0, C, 512)])
        want = torch.autograd.grad(ref, wide, dout[:, group * h:group * (h + 1)].float())[1:]
        for got, w in zip((dk, dv), want):
            err, scale = (got[:, h].float() - w[:, h]).abs(), max(1.0, float(w.abs().max()))
            assert err.max() <= 2e-2 * scale and err.mean() <= 1e-3 * scale
