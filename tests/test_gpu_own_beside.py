"""Stage-2 forward and dQ where a row's own blocks are walked beside ring blocks: rows with fewer blocks than the ring, as many, up to eight over and more, rows that
miss some of the ring's blocks, more own blocks than ring blocks and none.  Against fp32 attention."""
import pytest
import torch

from test_gpu_shared_by_some import attend, reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S, group, ring, missed, own", [(2500, 16, 12, 3, 0), (2500, 16, 12, 3, 3), (2500, 16, 12, 2, 10), (2500, 8, 12, 2, 11), (2500, 16, 3, 1, 30), (2500, 16, 0, 0, 7),
                                                          (64 * 70, 16, 40, 9, 17), (64 * 70, 16, 40, 9, 18)])
def test_forward_and_backward(S, group, ring, missed, own):
    import infllmv2_cuda_impl_amd as ops
    Hk, C, nblk = 1, 132, (S + 63) // 64                       # 16 whole groups and a half
    gen = torch.Generator(device="cuda").manual_seed(S + own)
    rand = lambda n, heads: torch.randn(n, heads, 128, generator=gen, device="cuda").to(torch.bfloat16)
    q, k, v, dout = rand(C, group), rand(S, Hk), rand(S, Hk), rand(C, group)
    pos, rows = torch.arange(S - C, S, device="cuda"), torch.arange(C, device="cuda")
    chosen = torch.zeros(Hk, C, nblk, dtype=torch.bool, device="cuda")
    # the first blocks are the ring's, of which row r of a group misses every eighth from r on, at most so many; behind them own blocks, others for every row
    for j in range(ring):
        chosen[0, :, j] = (rows % 8 != j % 8) | (rows % 8 * 0 + j // 8 >= missed)
    span = nblk - 3 - ring
    for i in range(own):
        chosen[0, rows, ring + (rows % 8 * 5 + i * 2) % span] = True
    chosen &= (torch.arange(nblk, device="cuda")[None] <= pos[:, None] // 64)[None]
    chosen[0, rows, pos // 64] = True
    mask = ops.blockmask_to_uint64(chosen.contiguous())[0]
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
    out = attend(*leaves, mask)
    dq = torch.autograd.grad(out, leaves, dout)[0]
    wide = [t.float().requires_grad_(True) for t in (q, k, v)]
    ref = reference(*wide, pos, chosen, 0, slice(0, C))
    err = (out.float() - ref).abs()
    assert err.max() <= 2e-2 and err.mean() <= 1e-3
    want = torch.autograd.grad(ref, wide, dout.float())[0]
    err, scale = (dq.float() - want).abs(), max(1.0, float(want.abs().max()))
    assert err.max() <= 2e-2 * scale and err.mean() <= 1e-3 * scale
