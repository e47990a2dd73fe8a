"""The mask words of a top-k selection without its list: the same words as with the list, for rows of one register to the longest, few rows
(a workgroup each) and many (a wavefront each, several in turn), whole registers and not, ties, columns of -inf kept or dropped, more
wanted than there are, and mask rows wider than the scores."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [1, 63, 64, 257, 512, 513, 1024, 2048, 5000, 8192])
@pytest.mark.parametrize("rows", [3, 513, 2100])
def test_mask_alone_equals_mask_with_list(n, rows, dtype):
    import infllmv2_cuda_impl_amd as ops
    from infllmv2_cuda_impl_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(n * 7 + rows)
    x = torch.randn(rows, n, generator=gen, device="cuda")
    x = torch.where(torch.rand(rows, n, generator=gen, device="cuda") < 0.3, (x * 2).round(), x)              # ties
    x = x.masked_fill(torch.rand(rows, n, generator=gen, device="cuda") < 0.2, float("-inf"))
    x[::5, n // 2:] = float("-inf")
    x[1::7] = 0.0
    x = x.to(dtype)
    for k in (0, 1, 16, 64, 300):
        for drop in (0, 1):
            n64 = (n + 63) // 64 + drop
            want = torch.empty(rows, n64, dtype=torch.int64, device="cuda")
            idx = torch.empty(rows, max(k, 1), dtype=torch.int32, device="cuda")
            got = torch.full_like(want, -1)
            stream = torch.cuda.current_stream().cuda_stream
            _lib.call("infllmv2_topk_select", stream, x.data_ptr(), n, int(dtype == torch.bfloat16), idx.data_ptr(), want.data_ptr(), rows, n, k, n64, 0, drop)
            _lib.call("infllmv2_topk_mask", stream, x.data_ptr(), n, int(dtype == torch.bfloat16), got.data_ptr(), rows, n, k, n64, drop)
            assert torch.equal(got, want), (k, drop)
