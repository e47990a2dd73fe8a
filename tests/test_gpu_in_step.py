"""Stage-2 forward on long sequences, where workgroups wait for the generation of their XCD before them: the same bits as the launches
that do not wait (images packed beforehand, or a workspace of the images' size alone), with several generations, short sequences and
sequences without queries in between, rows with blocks of their own and window rows, and a second launch into the same workspace."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # query lengths, key lengths, KV heads, blocks chosen per row
    ([9000], [33000], 1, 24),
    ([2100, 300, 0, 2500], [40000, 300, 50, 32769], 2, 24),
    ([5000, 9], [36000, 34000], 1, 0),                         # window rows
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sq, sk, Hk, scattered", CASES)
def test_in_step(sq, sk, Hk, scattered, dtype):
    from infllmv2_cuda_impl_amd import _lib
    dev = torch.device("cuda:0")
    g = torch.Generator(device="cpu").manual_seed(11)
    cu = lambda ns: torch.from_numpy(np.cumsum([0] + ns).astype(np.int32)).to(dev)
    T, S, n64 = sum(sq), sum(sk), ((max(sk) + 63) // 64 + 63) // 64
    q = torch.randn(T, Hk * 16, 128, generator=g).to(dtype).to(dev)
    k, v = (torch.randn(S, Hk, 128, generator=g).to(dtype).to(dev) for _ in range(2))
    pos = torch.cat([torch.arange(n) + m - n for n, m in zip(sq, sk)])
    diag = (pos // 64)[None, :, None].expand(Hk, -1, -1)
    picks = torch.cat([diag - j for j in range(4)] + [(torch.rand(Hk, T, 24, generator=g) * (diag + 1)).long()][:1 if scattered else 0], 2).clamp(min=0)
    words = torch.zeros(Hk, T, n64 * 64, dtype=torch.bool).scatter_(2, picks, True).view(Hk, T, n64, 64)
    mask = torch.from_numpy(np.packbits(words.numpy(), axis=-1, bitorder="little").view(np.int64).reshape(Hk, T, n64)).to(dev)
    cu_q, cu_k = cu(sq), cu(sk)
    size = _lib.lib.infllmv2_kv_image_bytes(S, len(sq), Hk)
    qs, ks, ls = _lib.i64_array([q.stride(0), 128, 16 * 128]), _lib.i64_array([Hk * 128, 128]), _lib.i64_array([16, 1, T * 16])

    def launch(ws, size, prepacked):
        out, lse = torch.full_like(q, float("nan")), torch.full((Hk, T * 16), float("nan"), device=dev)
        _lib.call_for(dtype, "infllmv2_varlen_fwd", torch.cuda.current_stream(dev).cuda_stream, q.data_ptr(), k.data_ptr(), v.data_ptr(),
                      out.data_ptr(), lse.data_ptr(), cu_q.data_ptr(), cu_k.data_ptr(), mask.data_ptr(), ws.data_ptr(), size, prepacked,
                      len(sq), T, S, Hk * 16, Hk, 128, max(sq), max(sk), qs, ks, ks, qs, ls, n64, 128 ** -0.5, 1)
        torch.cuda.synchronize()
        return out, lse

    ws = torch.full((size,), 255, dtype=torch.uint8, device=dev)
    runs = [launch(ws, size, 0), launch(ws, size, 0), launch(ws, size, 1), launch(ws, size - 1024, 0)]
    assert not torch.isnan(runs[0][0]).any()
    for out, lse in runs[1:]:
        assert torch.equal(out, runs[0][0]) and torch.equal(lse, runs[0][1])
    # a few rows against fp32 attention over their blocks
    for t in range(0, T, max(1, T // 7)):
        b = int(np.searchsorted(np.cumsum(sq), t, side="right"))
        k0 = sum(sk[:b])
        for h in range(Hk):
            keys = torch.nonzero(words[h, t].reshape(-1))[:, 0][:, None] * 64 + torch.arange(64)[None]
            keys = (keys[keys <= int(pos[t])] + k0).to(dev)
            s = q[t, 16 * h:16 * h + 16].float() @ k[keys, h].float().t() * 128 ** -0.5
            ref = torch.softmax(s, 1) @ v[keys, h].float()
            err = (runs[0][0][t, 16 * h:16 * h + 16].float() - ref).abs()
            assert err.max() <= 2e-2 and err.mean() <= 1e-3
