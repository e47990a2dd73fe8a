"""Stage-2 forward by tiles of 256 query rows under a mask: blocks that some tokens of a tile or wavefront selected and others did not, rows that
selected nothing, masks of two words, ends of tiles, queries behind cached keys, groups of 16, 8 and 4.  It is the walk of callers that say that neighbouring
rows are alike, and holds for any mask.  Against fp32 softmax attention over the selected
blocks; tolerances of the forward tests: 2e-2 on a 16-bit output of order one, 1e-3 on average, 2e-3 on the log-sum-exp."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # query lengths, key lengths, KV heads, group, blocks selected, causal
    ([1000, 37, 130], [1000, 37, 130], 4, 8, 16, True),
    ([1025], [1025], 8, 16, 16, True),
    ([4500], [4500], 4, 16, 64, True),                        # two mask words
    ([700, 256], [2100, 900], 8, 16, 32, True),               # behind cached keys
    ([1023], [1500], 8, 8, 16, False),
    ([1500, 1], [1500, 1], 8, 4, 16, True),
]


def selection(sq, sk, Hk, k, causal, gen):
    """int32 (Hk, sum sq, k): random blocks of what a token sees (and a few it does not), the first and its own among them; some rows empty."""
    rows = []
    for n, m in zip(sq, sk):
        nblk = (m + 63) // 64
        last = (torch.arange(n) + m - n).clamp(min=0) // 64 if causal else torch.full((n,), nblk - 1)
        score = torch.rand(Hk, n, nblk, generator=gen)
        score[..., 0] = 2.0
        score.scatter_(2, last[None, :, None].expand(Hk, n, 1), 2.0)
        idx = score.topk(min(k, nblk), dim=2).indices
        idx = torch.nn.functional.pad(idx, (0, k - idx.shape[2]), value=-1)
        idx[:, 5::97] = -1
        rows.append(idx)
    return torch.cat(rows, 1).to(torch.int32)


def reference(q, k, v, sq, sk, Hk, group, causal, idx):
    outs, lses, q0, k0 = [], [], 0, 0
    for n, m in zip(sq, sk):
        qq = q[q0:q0 + n].float().view(n, Hk, group, 128)
        kk, vv = k[k0:k0 + m].float(), v[k0:k0 + m].float()
        last = torch.arange(n, device=q.device) + m - n if causal else torch.full((n,), m, device=q.device)
        o, ls = [], []
        for h in range(Hk):
            chosen = torch.zeros(n, (m + 63) // 64 + 1, dtype=torch.bool, device=q.device)
            ii = idx[h, q0:q0 + n].long().to(q.device)
            chosen.scatter_(1, torch.where(ii < 0, chosen.shape[1] - 1, ii), True)
            ok = chosen[:, :-1].repeat_interleave(64, 1)[:, :m] & (torch.arange(m, device=q.device)[None] <= last[:, None])
            ok = ok.repeat_interleave(group, 0)
            s = (qq[:, h].reshape(n * group, 128) @ kk[:, h].t().contiguous()) * 128 ** -0.5
            s = s.masked_fill(~ok, float("-inf"))
            lse = torch.logsumexp(s, 1)
            p = torch.nan_to_num(torch.exp(s - lse[:, None])).masked_fill(~ok, 0.0)
            o.append(p.matmul(vv[:, h].contiguous()).view(n, group, 128))
            ls.append(torch.where(torch.isinf(lse), torch.full_like(lse, float("inf")), lse).view(n, group))
        outs.append(torch.stack(o, 1).reshape(n, Hk * group, 128))
        lses.append(torch.stack(ls, 0))
        q0, k0 = q0 + n, k0 + m
    return torch.cat(outs), torch.cat(lses, 1)


def inputs(sq, sk, Hk, group, dtype, gen):
    dev = torch.device("cuda:0")
    cu = lambda ns: torch.from_numpy(np.cumsum([0] + ns).astype(np.int32)).to(dev)
    make = lambda n, heads: torch.randn(n, heads, 128, generator=gen).to(dtype).to(dev)
    return make(sum(sq), Hk * group), make(sum(sk), Hk), make(sum(sk), Hk), cu(sq), cu(sk)


def by_tiles(sq, sk, Hk, group, k, causal):
    from infllmv2_cuda_impl_amd import _lib
    return _lib.lib.infllmv2_varlen_fwd_masked_tiles(len(sq), sum(sq), sum(sk), Hk * group, Hk, max(sq), max(sk), int(causal), -k)


def attend(*args, **more):
    from infllmv2_cuda_impl_amd.attention import attend_varlen
    return attend_varlen(*args, causal=more.pop("causal", True), alike=True, **more)


def check(out, lse, ref, ref_lse, Hk, group):
    err = (out.float() - ref).abs()
    assert err.max() <= 2e-2 and err.mean() <= 1e-3, (err.max().item(), err.mean().item())
    lse = lse.view(Hk, -1, group)
    assert (torch.isinf(ref_lse) == torch.isinf(lse)).all()
    assert (torch.nan_to_num(lse - ref_lse, nan=0.0).abs() <= 2e-3).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sq, sk, Hk, group, k, causal", CASES)
def test_masked_tiles(sq, sk, Hk, group, k, causal, dtype):
    assert by_tiles(sq, sk, Hk, group, k, causal) == 1
    gen = torch.Generator(device="cpu").manual_seed(3)
    q, kk, v, cu_q, cu_k = inputs(sq, sk, Hk, group, dtype, gen)
    idx = selection(sq, sk, Hk, k, causal, gen)
    out, lse, _ = attend(q, kk, v, cu_q, cu_k, max(sq), max(sk), causal=causal, topk_idx=idx.cuda(), return_attn_probs=True)
    check(out, lse, *reference(q, kk, v, sq, sk, Hk, group, causal, idx), Hk, group)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group", [16, 8])
def test_infinities_stay_with_the_rows_that_selected_them(group, dtype):
    """Blocks that hold infinities and NaN, each selected by one token of a tile: every other row is what it is without them."""
    S, Hk, k = 1100, 8, 16
    assert by_tiles([S], [S], Hk, group, k, True) == 1
    gen = torch.Generator(device="cpu").manual_seed(4)
    q, kk, v, cu, _ = inputs([S], [S], Hk, group, dtype, gen)
    idx = selection([S], [S], Hk, k, True, gen)
    bad = {3: 700, 7: 901, 9: 1099}                            # block -> the one token that selects it
    for block, token in bad.items():
        idx = torch.where(idx == block, -1, idx)
        idx[:, token, 1] = block
    clean = attend(q, kk, v, cu, cu, S, S, topk_idx=idx.cuda())
    kk[3 * 64 + 5, :, 7], v[7 * 64 + 40, :, 100], v[9 * 64, :, 3] = float("nan"), float("inf"), float("-inf")
    out = attend(q, kk, v, cu, cu, S, S, topk_idx=idx.cuda())
    touched = torch.zeros(S, dtype=torch.bool, device=out.device)
    touched[list(bad.values())] = True
    touched[[t for t in range(S) if t // 64 in bad]] = True   # a block's own tokens select it whatever the indices above say
    touched |= (idx[..., None] == torch.tensor(list(bad))).flatten(2).any(2).any(0).to(out.device)
    assert torch.isfinite(out[~touched].float()).all()
    assert (out[~touched].float() - clean[~touched].float()).abs().max() <= 1e-2          # a unit in the last place of an output of order one
    assert not torch.isfinite(out[700].float()).all() and not torch.isfinite(out[901].float()).all()


def test_which_masked_launches_go_by_tiles():
    f = lambda lens, Hk, group, k: by_tiles(lens, lens, Hk, group, k, True)
    for lens, Hk, group in (([1000], 2, 16), ([3000], 2, 16), ([777, 5003, 1291, 9173], 2, 16), ([4000], 4, 8), ([131072], 2, 16)):
        assert f(lens, Hk, group, 16) == 1                     # a window, whatever the sizes
        for k in (0, 16, 64, 2 ** 31 - 1):                     # blocks chosen by score, or how many is not known
            assert f(lens, Hk, group, -k) == 0
    for n in (0, 1, 2 ** 31 - 1):
        assert f([n], 2, 16, 2 ** 31 - 1) in (0, 1)
