"""A one-token append into a cache whose unwritten rows hold NaN (memory from ``torch.empty``, or a recycled page): none of it may
reach the output.  Lengths at the ends of 64-key blocks and of pages, the first token of a sequence included; dense, mask and index
list; plain and paged; workgroups of one wavefront and of four; the C ABI entry that allocates nothing and the native module.
Against fp32 attention over the written rows; tolerances of the decode tests (2e-2 on an output of order one, 1e-3 on average)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
LENS = [0, 1, 62, 63, 64, 126, 127, 128, 190]
CAP, HK, PAGE = 192, 2, 64


def make(dtype, repeat, seed=1):
    """(q, k, v with NaN behind each sequence's end, new k, new v, lengths, reference output, k and v after the step)"""
    g = torch.Generator(device="cpu").manual_seed(seed)
    lens = LENS * repeat
    B = len(lens)
    mk = lambda *s: torch.randn(*s, generator=g).to(dtype)
    q, kc, vc, kn, vn = mk(B, 1, 16 * HK, 128), mk(B, CAP, HK, 128), mk(B, CAP, HK, 128), mk(B, 1, HK, 128), mk(B, 1, HK, 128)
    ref = torch.zeros(B, 1, 16 * HK, 128)
    for b, n in enumerate(lens):
        kc[b, n:], vc[b, n:] = float("nan"), float("nan")
    after_k, after_v = kc.clone(), vc.clone()
    for b, n in enumerate(lens):
        after_k[b, n], after_v[b, n] = kn[b, 0], vn[b, 0]
        for h in range(HK):
            s = (q[b, 0, 16 * h:16 * h + 16].float() @ after_k[b, :n + 1, h].float().t()) * 128 ** -0.5
            ref[b, 0, 16 * h:16 * h + 16] = torch.softmax(s, -1) @ after_v[b, :n + 1, h].float()
    d = lambda t: t.cuda()
    return d(q), d(kc), d(vc), d(kn), d(vn), torch.tensor(lens, dtype=torch.int32).cuda(), ref.cuda(), after_k.cuda(), after_v.cuda()


def check(out, ref, *pairs):
    err = (out.float() - ref).abs()
    assert err.max() <= 2e-2 and err.mean() <= 1e-3, (err.max().item(), err.mean().item())
    for got, want in pairs:
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def selection(form, B):
    if form == "dense":
        return {}
    if form == "mask":
        return {"block_mask": torch.full((B, HK, 1, 1), -1, dtype=torch.int64, device="cuda")}
    return {"topk_idx": torch.arange(3, dtype=torch.int32, device="cuda").flip(0).expand(B, HK, 1, 3).contiguous()}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", ["dense", "mask", "index"])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("repeat, splits", [(1, 1), (1, 3), (15, 1)])      # 18, 54 and 270 workgroups: 256 at most are of four wavefronts
def test_append_into_unwritten_rows(dtype, form, paged, repeat, splits):
    import infllmv2_cuda_impl_amd as ops
    q, kc, vc, kn, vn, L, ref, ak, av = make(dtype, repeat)
    B = q.shape[0]
    table = None
    if paged:
        per_seq = CAP // PAGE
        table = torch.randperm(B * per_seq, generator=torch.Generator().manual_seed(2)).to(torch.int32).view(B, per_seq).cuda()
        pages = lambda t: torch.empty_like(t).view(B * per_seq, PAGE, HK, 128).index_copy_(0, table.view(-1).long(), t.view(B * per_seq, PAGE, HK, 128))
        kc, vc, ak, av = pages(kc), pages(vc), pages(ak), pages(av)
    out = ops.infllmv2_attn_with_kvcache(q, kc, vc, k=kn, v=vn, cache_seqlens=L, block_table=table, num_splits=splits, **selection(form, B))
    check(out, ref, (kc, ak), (vc, av))


@pytest.mark.parametrize("form", ["dense", "mask"])
def test_append_into_unwritten_rows_through_the_other_entries(form):
    import infllmv2_cuda_impl_amd.C as pure
    from infllm_v2 import C as compiled
    from infllmv2_cuda_impl_amd import _lib
    for entry in (compiled, pure):
        q, kc, vc, kn, vn, L, ref, ak, av = make(torch.bfloat16, 1)
        words = selection(form, q.shape[0]).get("block_mask")
        out, _ = entry.fwd_kvcache(q, kc, vc, kn, vn, L, None, None, None, None, None, None, None, 128 ** -0.5, False, -1, -1, 0.0, True, 2, words)
        check(out, ref, (kc, ak), (vc, av))
    q, kc, vc, kn, vn, L, ref, ak, av = make(torch.bfloat16, 1)
    words = selection(form, q.shape[0]).get("block_mask")
    out, lse = torch.empty_like(q), torch.empty((q.shape[0], q.shape[2], 1), dtype=torch.float32, device="cuda")
    s3 = lambda t: _lib.i64_array(t.stride()[:3])
    two = lambda t: _lib.i64_array([t.stride(0), t.stride(2)])
    _lib.call("infllmv2_fwd_kvcache_static", torch.cuda.current_stream().cuda_stream, q.data_ptr(), kc.data_ptr(), vc.data_ptr(), kn.data_ptr(),
              vn.data_ptr(), L.data_ptr(), out.data_ptr(), lse.data_ptr(), None if words is None else words.data_ptr(), q.shape[0], 1, q.shape[2],
              HK, 128, CAP, 1, two(q), s3(kc), s3(vc), s3(kn), s3(vn), two(out), 0 if words is None else 1, 3, 128 ** -0.5, None, None, None,
              0, 0, None, None, 0, 0)
    check(out, ref, (kc, ak), (vc, av))
