"""Compressed keys at the sizes where the kernel's tiling can go wrong: sequences around one window and around the rows
one workgroup takes (8 at 32/16, 2 at 128/64), windows longer than the staging buffer, head sizes other than 128, and
several heads and sequences.  Bit for bit against an fp32 sum in window order, rounded once."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def reference(k, cu, kernel, stride, dtype):
    rows = []
    for b in range(len(cu) - 1):
        seq = k[cu[b]:cu[b + 1]].astype(np.float32)
        for j in range((len(seq) - kernel) // stride + 1 if len(seq) >= kernel else 0):
            acc = np.zeros(seq.shape[1:], dtype=np.float32)
            for i in range(kernel):
                acc += seq[j * stride + i]
            rows.append(acc / np.float32(kernel))
    out = np.stack(rows) if rows else np.zeros((0,) + k.shape[1:], dtype=np.float32)
    return torch.from_numpy(out).to(dtype)


@pytest.mark.parametrize("lens,hk,d,sets", [
    ([31, 32, 33, 127, 128, 159, 160, 161], 2, 128, [(32, 16), (128, 64)]),
    ([64 * 3 + 127, 64 * 2 + 128, 1], 1, 128, [(32, 16), (128, 64)]),
    ([500, 700], 3, 64, [(32, 16), (256, 7)]),
    ([420], 2, 136, [(1, 1), (256, 16)]),
])
def test_compressed_keys_at_tile_edges(lens, hk, d, sets):
    from infllmv2_cuda_impl_amd import compress_keys
    from infllmv2_cuda_impl_amd.selection import compress_keys_pair
    cu = np.cumsum([0] + lens)
    g = torch.Generator(device="cpu").manual_seed(3)
    for dtype in (torch.bfloat16, torch.float16):
        k = torch.randn(int(cu[-1]), hk, d, generator=g).to(dtype)
        kd, cud = k.cuda(), torch.tensor(cu, dtype=torch.int32, device="cuda")
        pair = compress_keys_pair(kd, cud, max(lens), *sets)
        for n, (kernel, stride) in enumerate(sets):
            want = reference(k.float().numpy(), cu, kernel, stride, dtype)
            counts = np.cumsum([0] + [(s - kernel) // stride + 1 if s >= kernel else 0 for s in lens])
            for got, cu_got in (compress_keys(kd, cud, max(lens), kernel, stride), pair[2 * n:2 * n + 2]):
                assert np.array_equal(cu_got.cpu().numpy(), counts)
                assert torch.equal(got[:counts[-1]].cpu(), want)
