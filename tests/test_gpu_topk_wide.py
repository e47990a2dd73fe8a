"""Top-k with a workgroup per row against a sort of unique keys (larger score first, equal scores by ascending column), on both sides of every number of
columns and rows at which the kernel or its registers change: rows of arbitrary bits, so that the search goes through both histograms, infinities more and
fewer than are wanted, rows of one value, and scores as Stage 1 makes them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def rows_of(kind, rows, n, gen, dtype=torch.bfloat16):
    if kind == "bits":                                           # NaN included: its bits order it
        return torch.randint(-32768, 32768, (rows, n), generator=gen, device="cuda", dtype=torch.int32).to(torch.int16).view(dtype)
    x = torch.rand(rows, n, generator=gen, device="cuda") ** 6
    if kind == "spread":                                         # over many powers of two, zeros and forced blocks among them
        x = 16 * torch.softmax(6 * torch.randn(rows, n, generator=gen, device="cuda"), 1)
        x[:, 3::11] = 0.0
        x[:, :2] = float("inf")
    if kind == "inf":
        x[torch.rand(rows, n, generator=gen, device="cuda") < 0.3] = float("-inf")
        x[:, ::5] = float("inf")
    if kind == "flat":
        x[:] = 0.25
        x[::2, 1::3] = -0.0
        x[::4, 2::7] = 0.0
    return x.to(dtype)


def check(x, k, drop=0):
    from infllmv2_cuda_impl_amd import _lib
    rows, n = x.shape
    bf16, neg_inf = int(x.dtype == torch.bfloat16), 0x80 if x.dtype == torch.bfloat16 else 0x400
    bits = x.view(torch.int16).to(torch.int64) & 0xffff
    key = torch.where(bits < 0x8000, bits + 0x8000, 0x10000 - bits)                                        # -0 and +0 alike
    order = torch.topk(key * 16384 + (16383 - torch.arange(n, device="cuda")), min(k, n), dim=1).values
    want = torch.full((rows, max(k, 1)), -1, dtype=torch.int64, device="cuda")
    want[:, :min(k, n)] = 16383 - (order & 16383)
    if drop:                                                     # what is not above -inf leaves the end of the list
        want[:, :min(k, n)][order >> 14 <= neg_inf] = -1
    n64, stream = (n + 63) // 64 + 1, torch.cuda.current_stream().cuda_stream
    idx = torch.empty(rows, max(k, 1), dtype=torch.int32, device="cuda")
    words = torch.empty(rows, n64, dtype=torch.int64, device="cuda")
    for by_index in (0, 1):
        _lib.call("infllmv2_topk_select", stream, x.data_ptr(), n, bf16, idx.data_ptr(), words.data_ptr(), rows, n, k, n64, by_index, drop)
        got = idx[:, :k].to(torch.int64)
        ref = want[:, :k]
        if by_index:
            ref = torch.where(ref < 0, 1 << 20, ref).sort(1).values
            ref = torch.where(ref == 1 << 20, -1, ref)
        assert torch.equal(got, ref), (rows, n, k, by_index)
        taken = torch.zeros(rows, n64 * 64 + 1, dtype=torch.bool, device="cuda").scatter_(1, torch.where(want[:, :k] < 0, n64 * 64, want[:, :k]), True)
        shown = (words[:, :, None] >> torch.arange(64, device="cuda") & 1).bool().view(rows, -1)
        assert torch.equal(shown, taken[:, :-1]), (rows, n, k)
    if k > 0 and not drop:
        stride = 1 << (k - 1).bit_length()                       # of this entry point's rows
        val, idx = torch.empty(rows, stride, dtype=x.dtype, device="cuda"), torch.empty(rows, stride, dtype=torch.int32, device="cuda")
        _lib.call("infllmv2_topk", stream, rows, n, k, bf16, x.data_ptr(), val.data_ptr(), idx.data_ptr())
        assert torch.equal(idx[:, :k].to(torch.int64), want[:, :k])
        got = x.gather(1, want[:, :min(k, n)])
        assert torch.equal(val[:, :min(k, n)].view(torch.int16), got.view(torch.int16))


@pytest.mark.parametrize("kind", ["bits", "inf", "flat", "scores"])
@pytest.mark.parametrize("n", [256, 257, 511, 512, 513, 1024, 1025, 2048, 2049, 4096, 4097, 8192])
def test_few_rows(n, kind):
    gen = torch.Generator(device="cuda").manual_seed(n)
    for k in (0, 1, 16, 64, 65, 300):
        check(rows_of(kind, 5, n, gen), k)


@pytest.mark.parametrize("rows, n", [(768, 400), (769, 400), (1024, 700), (1025, 700), (2048, 1100), (2049, 1100), (16384, 2100), (16385, 2100),
                                     (512, 400), (513, 400), (768, 1024), (769, 1024), (1536, 2048), (1537, 2048), (16384, 4096), (16385, 4096)])
def test_both_sides_of_the_rule(rows, n):
    gen = torch.Generator(device="cuda").manual_seed(rows)
    for kind in ("scores", "inf"):
        check(rows_of(kind, rows, n, gen), 32)


@pytest.mark.parametrize("rows, n", [(16384, 2100), (16385, 2100), (4096, 4096), (4097, 4096)])
def test_both_sides_of_the_rule_for_words_alone(rows, n):
    """The words without a list against those with it, which another kernel makes on one side."""
    from infllmv2_cuda_impl_amd import _lib
    x = rows_of("spread", rows, n, torch.Generator(device="cuda").manual_seed(rows), torch.float16)
    n64, stream = (n + 63) // 64, torch.cuda.current_stream().cuda_stream
    idx = torch.empty(rows, 48, dtype=torch.int32, device="cuda")
    want, got = torch.empty(2, rows, n64, dtype=torch.int64, device="cuda").unbind(0)
    _lib.call("infllmv2_topk_select", stream, x.data_ptr(), n, 0, idx.data_ptr(), want.data_ptr(), rows, n, 48, n64, 1, 0)
    _lib.call("infllmv2_topk_mask", stream, x.data_ptr(), n, 0, got.data_ptr(), rows, n, 48, n64, 0)
    assert torch.equal(got, want)


@pytest.mark.parametrize("drop", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["bits", "inf", "flat", "scores", "spread"])
def test_both_types_and_dropped_columns(kind, dtype, drop):
    """The histogram's bins hold another number of keys in IEEE half: every kind of row in both types, columns of -inf kept and dropped, more wanted than
    the first histogram holds, and the smallest key of a row."""
    gen = torch.Generator(device="cuda").manual_seed(5 + drop)
    for n in (513, 700, 2048, 4097):
        x = rows_of(kind, 6, n, gen, dtype)
        x[::3, 1::2] = float("-inf")
        for k in (1, 17, 64, 400, 1500, n):
            check(x, min(k, 2048), drop)


def test_more_long_rows_than_a_dispatch_holds():
    """Rows of more than 4096 columns take a workgroup of 512 threads each, and a dispatch fewer than 2^32 threads: 8 388 608 rows and some more, all of them
    the same one (row stride 0), so that the scores take little memory."""
    from infllmv2_cuda_impl_amd import _lib
    n, rows = 4097, (1 << 23) + 5
    x = torch.rand(1, n, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda").to(torch.bfloat16)
    idx = torch.full((rows, 1), -7, dtype=torch.int32, device="cuda")
    _lib.call("infllmv2_topk_select", torch.cuda.current_stream().cuda_stream, x.data_ptr(), 0, 1, idx.data_ptr(), None, rows, n, 1, 0, 0, 0)
    best = int((x[0] == x[0].max()).nonzero()[0])
    assert (idx == best).all()
