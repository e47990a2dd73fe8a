"""dK/dV of short inputs: slices of 128 tokens in which few tokens selected a block are put together to items of about 128 tokens, and 2, 4
or 8 XCDs share a group of 2048 tokens.  Densities on both sides of a light slice (32 of 128 tokens) and of a full item, sequences that
start inside a slice and a group, token counts on both sides of the rules for the sharing.  dK and dV against fp32 attention's gradients
per KV head (tolerances of the backward tests: 2e-2 and 1e-3 of the largest value); the deterministic mode, whose slices are longer,
agrees to the order of its fp32 sums and the rounding of the output."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # lengths, KV heads, share of the tokens that select a block
    ([2047], 1, 0.03),
    ([2500, 1], 1, 0.12),
    ([1000, 100, 1900], 2, 0.24),
    ([6144], 1, 0.20),                                         # 3 groups
    ([6145], 1, 0.26),                                         # 4
    ([3000] * 8, 1, 0.10),                                     # 12 groups of short sequences
]


def causal_reference(q, k, v, dout, mask, lens, Hk):
    """fp32 gradients (dq is not needed) of softmax attention over the selected blocks, one KV head of one sequence at a time."""
    dk, dv, t0 = torch.zeros(k.shape, device=k.device), torch.zeros(k.shape, device=k.device), 0
    for n in lens:
        rows = slice(t0, t0 + n)
        ok = mask[:, rows, :(n + 63) // 64].to(k.device).repeat_interleave(64, 2)[:, :, :n]
        ok = ok & (torch.arange(n, device=k.device)[None, None] <= torch.arange(n, device=k.device)[None, :, None])
        for h in range(Hk):
            kh, vh = k[rows, h].float(), v[rows, h].float()
            for g in range(16):
                qh, do = q[rows, 16 * h + g].float(), dout[rows, 16 * h + g].float()
                p = torch.softmax((qh @ kh.t() * 128 ** -0.5).masked_fill(~ok[h], float("-inf")), 1)
                dp = do @ vh.t()
                ds = p * (dp - (p * dp).sum(1, keepdim=True))
                dv[rows, h] += p.t() @ do
                dk[rows, h] += ds.t() @ qh * 128 ** -0.5
        t0 += n
    return dk, dv


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens, Hk, density", CASES)
def test_items(lens, Hk, density, dtype):
    import infllmv2_cuda_impl_amd as ops
    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(5)
    T, nblk = sum(lens), (max(lens) + 63) // 64
    cu = torch.from_numpy(np.cumsum([0] + lens).astype(np.int32)).to(dev)
    q, dout = (torch.randn(T, Hk * 16, 128, generator=g).to(dtype).to(dev) for _ in range(2))
    k, v = (torch.randn(T, Hk, 128, generator=g).to(dtype).to(dev) for _ in range(2))
    diag = torch.cat([torch.arange(n) // 64 for n in lens])
    blocks = torch.arange(nblk)
    mask = (torch.rand(Hk, T, nblk, generator=g) < density) & (blocks[None, None] < diag[None, :, None])
    mask |= (blocks[None] == diag[:, None])[None]              # every token has its own block
    idx = torch.where(mask, blocks[None, None], nblk).sort(2).values
    idx = torch.where(idx == nblk, -1, idx).to(torch.int32).to(dev)
    grads = []
    for deterministic in (False, True):
        qg, kg, vg = (t.clone().requires_grad_(True) for t in (q, k, v))
        out = ops.infllmv2_attn_varlen_func(qg, kg, vg, cu, cu, max(lens), max(lens), causal=True, topk_idx=idx, deterministic=deterministic)
        grads.append(torch.autograd.grad(out, (kg, vg), dout))
    for got, det, ref in zip(*grads, causal_reference(q, k, v, dout, mask, lens, Hk)):
        scale = max(1.0, float(ref.abs().max()))
        err = (got.float() - ref).abs()
        assert err.max() <= 2e-2 * scale and err.mean() <= 1e-3 * scale
        # another order of the same fp32 sums: at most one rounding of the 16-bit result apart (bf16: 2^-8 of the value)
        assert ((got.float() - det.float()).abs() <= 2 ** -7 * det.float().abs() + 1e-4 * scale).all()
