"""dQ by tiles of 256 query rows, under masks and without: blocks that some tokens of a tile or wavefront selected and others did not, rows that
selected nothing, masks of two words, ends of tiles, queries behind cached keys and before the first key, groups of 16, 8 and 4.  Under a mask it is the walk
of callers that say that neighbouring rows are alike, and holds for any mask.  All gradients (dK and
dV read the row scalars that this kernel leaves) against fp32 attention's; tolerances of the backward tests: 2e-2 and 1e-3 of the largest value."""
import pytest
import torch

from test_gpu_masked_tiles import inputs, selection

pytestmark = pytest.mark.gpu

CASES = [  # query lengths, key lengths, KV heads, group, blocks selected (0: no mask), causal
    ([1000, 37, 130], [1000, 37, 130], 4, 8, 16, True),
    ([1025], [1025], 8, 16, 16, True),
    ([4500], [4500], 4, 16, 64, True),                        # two mask words
    ([700, 256], [2100, 900], 8, 16, 32, True),               # behind cached keys
    ([1023], [1500], 8, 8, 16, False),
    ([1500, 1], [1500, 1], 8, 4, 16, True),
    ([2049, 15, 17, 1], [2049, 15, 17, 1], 4, 16, 0, True),
    ([2100, 90], [1030, 33], 4, 16, 0, True),                 # the first queries see no key
]


def gradients(q, k, v, dout, sq, sk, Hk, group, causal, idx):
    dq, dk, dv = (torch.zeros(t.shape, device=t.device) for t in (q, k, v))
    q0 = k0 = 0
    for n, m in zip(sq, sk):
        last = torch.arange(n, device=q.device) + m - n if causal else torch.full((n,), m, device=q.device)
        for h in range(Hk):
            ok = torch.arange(m, device=q.device)[None] <= last[:, None]
            if idx is not None:
                chosen = torch.zeros(n, (m + 63) // 64 + 1, dtype=torch.bool, device=q.device)
                ii = idx[h, q0:q0 + n].long().to(q.device)
                chosen.scatter_(1, torch.where(ii < 0, chosen.shape[1] - 1, ii), True)
                ok = ok & chosen[:, :-1].repeat_interleave(64, 1)[:, :m]
            kh, vh = k[k0:k0 + m, h].float(), v[k0:k0 + m, h].float()
            for g in range(group):
                qh, do = q[q0:q0 + n, h * group + g].float(), dout[q0:q0 + n, h * group + g].float()
                p = torch.nan_to_num(torch.softmax((qh @ kh.t() * 128 ** -0.5).masked_fill(~ok, float("-inf")), 1))
                dp = do @ vh.t()
                ds = p * (dp - (p * dp).sum(1, keepdim=True)) * 128 ** -0.5
                dq[q0:q0 + n, h * group + g] = ds @ kh
                dv[k0:k0 + m, h] += p.t() @ do
                dk[k0:k0 + m, h] += ds.t() @ qh
        q0, k0 = q0 + n, k0 + m
    return dq, dk, dv


def by_tiles(sq, sk, Hk, group, k, causal):
    from infllmv2_cuda_impl_amd import _lib
    return _lib.lib.infllmv2_varlen_bwd_dq_tiles(len(sq), sum(sq), sum(sk), Hk * group, Hk, max(sq), max(sk), int(causal), -k or 2 ** 31 - 1)


def backward(q, k, v, dout, cu_q, cu_k, sq, sk, causal, idx):
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    leaves = [t.detach().clone().requires_grad_(True) for t in (q, k, v)]
    out = attend_varlen(*leaves, cu_q, cu_k, max(sq), max(sk), causal=causal, topk_idx=idx, alike=idx is not None)
    return torch.autograd.grad(out, leaves, dout)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sq, sk, Hk, group, k, causal", CASES)
def test_dq_tiles(sq, sk, Hk, group, k, causal, dtype):
    assert by_tiles(sq, sk, Hk, group, k, causal) == 1
    gen = torch.Generator(device="cpu").manual_seed(6)
    q, kk, v, cu_q, cu_k = inputs(sq, sk, Hk, group, dtype, gen)
    dout = torch.randn(q.shape, generator=gen).to(dtype).cuda()
    idx = selection(sq, sk, Hk, k, causal, gen) if k else None
    grads = backward(q, kk, v, dout, cu_q, cu_k, sq, sk, causal, idx.cuda() if k else None)
    for name, got, ref in zip(("dq", "dk", "dv"), grads, gradients(q, kk, v, dout, sq, sk, Hk, group, causal, idx)):
        err, top = (got.float() - ref).abs(), ref.abs().max().item()
        assert err.max() <= 2e-2 * top and err.mean() <= 1e-3 * top, (name, err.max().item(), err.mean().item(), top)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group", [16, 8])
def test_infinities_stay_with_the_rows_that_selected_them(group, dtype):
    """Blocks that hold infinities and NaN, each selected by one token of a tile: every other row of dq is what it is without them."""
    S, Hk, k = 1100, 8, 16
    assert by_tiles([S], [S], Hk, group, k, True) == 1
    gen = torch.Generator(device="cpu").manual_seed(4)
    q, kk, v, cu, _ = inputs([S], [S], Hk, group, dtype, gen)
    dout = torch.randn(q.shape, generator=gen).to(dtype).cuda()
    idx = selection([S], [S], Hk, k, True, gen)
    bad = {3: 700, 7: 901, 9: 1099}                            # block -> the one token that selects it
    for block, token in bad.items():
        idx = torch.where(idx == block, -1, idx)
        idx[:, token, 1] = block
    clean = backward(q, kk, v, dout, cu, cu, [S], [S], True, idx.cuda())[0]
    kk[3 * 64 + 5, :, 7], v[7 * 64 + 40, :, 100], kk[9 * 64, :, 3] = float("nan"), float("inf"), float("-inf")
    dq = backward(q, kk, v, dout, cu, cu, [S], [S], True, idx.cuda())[0]
    touched = (idx[..., None] == torch.tensor(list(bad))).flatten(2).any(2).any(0).to(dq.device)
    assert torch.isfinite(dq[~touched].float()).all()
    top = clean.float().abs().max().item()                     # D comes from an output that may be rounded apart: a unit in the last place of it
    assert (dq[~touched].float() - clean[~touched].float()).abs().max() <= 1e-2 * top
    assert not torch.isfinite(dq[700].float()).all()


def test_which_backward_passes_form_dq_by_tiles():
    f = lambda lens, Hk, group, k: by_tiles(lens, lens, Hk, group, k, True)
    assert f([6000], 4, 8, 0) and f([16384], 2, 16, 0) and not f([300], 2, 16, 0)            # without a mask
    for lens, Hk in (([1000], 2), ([8000], 2), ([777, 5003, 1291, 9173], 2), ([3000], 4)):
        assert f(lens, Hk, 16, 33) and f(lens, Hk, 8, 6) and not f(lens, Hk, 16, 6)        # windows, whatever the sizes
        for k in (16, 64):                                     # blocks chosen by score
            assert not f(lens, Hk, 16, -k) and not f(lens, Hk, 8, -k)
    from infllmv2_cuda_impl_amd import _lib
    assert _lib.lib.infllmv2_varlen_bwd_dq_tiles(1, 3000, 3000, 32, 4, 3000, 3000, 1, 0) == 0     # how many blocks a row selects is not known
    for n in (0, 1, 2 ** 31 - 1):
        assert _lib.lib.infllmv2_varlen_bwd_dq_tiles(1, n, n, 32, 2, n, n, 1, 64) in (0, 1)
