"""Infinities and NaN in keys and values that causality hides from a row: a block that begins behind a row's last key does not reach it, where tiles of 256 query
rows straddle the beginning of a block (Sk - Sq is not a multiple of a tile's tokens) and walk it for some of their rows.  Without a mask, under a mask that lists blocks
wholly in the row's future, and for a window.  Forward and dQ, against the same launch with finite keys."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Sq, Sk, Hk, group, masked", [(2100, 2137, 4, 16, False), (2100, 2137, 4, 8, False), (2100, 2137, 4, 16, True), (2100, 2137, 4, 8, True),
                                                       (1999, 1990, 8, 16, False), (700, 2101, 8, 8, True)])
def test_blocks_behind_a_rows_last_key_do_not_reach_it(Sq, Sk, Hk, group, masked, dtype):
    from infllmv2_cuda_impl_amd import _lib
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    gen = torch.Generator(device="cuda").manual_seed(17)
    rand = lambda n, heads: torch.randn(n, heads, 128, generator=gen, device="cuda").to(dtype)
    q, k, v, dout = rand(Sq, Hk * group), rand(Sk, Hk), rand(Sk, Hk), rand(Sq, Hk * group)
    nblk = (Sk + 63) // 64
    mask = torch.full((Hk, Sq, (nblk + 63) // 64), -1, dtype=torch.int64, device="cuda") if masked else None       # every block, the future ones too
    idx = torch.zeros(Hk, Sq, nblk, dtype=torch.int32, device="cuda") if masked else None                    # with a mask at hand only its width counts
    sizes = (1, Sq, Sk, Hk * group, Hk, Sq, Sk, 1)
    if masked:
        assert _lib.lib.infllmv2_varlen_fwd_masked_tiles(*sizes, -nblk) == 1
    else:
        assert _lib.lib.infllmv2_varlen_fwd_dense_tiles(*sizes) == 1
    assert _lib.lib.infllmv2_varlen_bwd_dq_tiles(*sizes, -nblk if masked else 2 ** 31 - 1) == 1
    cu = lambda n: torch.tensor([0, n], dtype=torch.int32, device="cuda")

    def run():
        leaves = [t.detach().clone().requires_grad_(True) for t in (q, k, v)]
        out = attend_varlen(*leaves, cu(Sq), cu(Sk), Sq, Sk, causal=True, topk_idx=idx, block_mask=mask, alike=masked)
        return out.detach().float(), torch.autograd.grad(out, leaves[0], dout)[0].float()

    clean = run()
    first = 64 * (max(Sk - Sq, 0) // 64 + 5)                   # the block that holds what must not be seen
    sees = torch.arange(Sq, device="cuda") + Sk - Sq >= first
    assert (first - (Sk - Sq)) % (256 // group) != 0           # some tile straddles its beginning
    k[first + 9, :, 7], v[first + 30, :, 100], v[first + 63, :, 3] = float("nan"), float("inf"), float("-inf")
    for name, got, want in zip(("out", "dq"), run(), clean):
        assert torch.isfinite(got[~sees]).all(), name
        # the rows are walked once more in another order: P, dS and the result are rounded to the element type on either side
        assert (got[~sees] - want[~sees]).norm() <= 2.0 ** -7 * want[~sees].norm(), name
        assert (got[~sees] - want[~sees]).abs().max() <= 1e-2 * max(1.0, want.abs().max().item()), name
        assert not torch.isfinite(got[sees]).all()
