"""Host-side argument logic that needs no GPU."""
import pytest


def test_causal_flag_is_derived_from_the_window_as_in_the_reference():
    """flash_api.cpp:621-622 (a window side >= max_seqlen_k is unbounded), :600 (causal closes the right side),
    :137 (causal launch iff left unbounded and right == 0), :144-147 (anything else is local attention: rejected)."""
    from infllmv2_cuda_impl_amd.attention import normalise_causal as f
    assert f(True, (-1, -1)) is True
    assert f(False, (-1, -1)) is False
    assert f(False, (-1, 0)) is True                       # the case an int(bool(causal)) launch gets wrong
    assert f(True, (-1, 5)) is True                        # causal overrides the right side
    assert f(False, (-1, 5)) is None
    assert f(False, (7, 0)) is None and f(True, (7, -1)) is None
    assert f(False, (128, 0), max_seqlen_k=128) is True    # left side reaches the keys: unbounded
    assert f(False, (127, 0), max_seqlen_k=128) is None
    assert f(False, (500, 500), max_seqlen_k=128) is False
    assert f(False, (-1, 128), max_seqlen_k=128) is False
    assert f(False, (128, 0)) is None                      # without max_seqlen_k nothing is widened


def test_reject_unsupported_returns_the_launch_flag_and_keeps_the_reference_messages():
    from infllmv2_cuda_impl_amd.attention import _reject_unsupported as r
    assert r(0.0, (-1, 0), 0.0, None, False, 64) is True
    assert r(0.0, (-1, -1), 0.0, None, False, 64) is False
    with pytest.raises(RuntimeError, match="does not support local attention"):
        r(0.0, (3, 0), 0.0, None, False, 64)
    with pytest.raises(RuntimeError, match="does not support softcap"):
        r(0.0, (-1, -1), 1.0, None, True, 64)
    with pytest.raises(RuntimeError, match="does not support dropout"):
        r(0.5, (-1, -1), 0.0, None, True, 64)
    with pytest.raises(RuntimeError, match="does not support alibi"):
        r(0.0, (-1, -1), 0.0, object(), True, 64)


def test_native_module_binds_the_reference_names():
    """`infllm_v2.C` is the compiled extension and exports what csrc/entry.cu:197-215 binds; argument errors that need
    no GPU are reported on the host."""
    import pytest
    import torch
    from infllm_v2 import C
    import infllmv2_cuda_impl_amd._C as ext
    names = ["topk", "get_probs", "blockmask_to_uint64", "topk_to_uint64", "uint64_to_bool", "max_pooling_1d",
             "max_pooling_1d_varlen", "fwd", "varlen_fwd", "varlen_fwd_stage1", "bwd", "varlen_bwd", "fwd_kvcache"]
    for n in names:
        assert getattr(C, n) is getattr(ext, n), n
    with pytest.raises(NotImplementedError):
        C.get_probs()
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16)
    cu = torch.tensor([0, 4], dtype=torch.int32)
    with pytest.raises(RuntimeError, match="no CPU path"):
        C.varlen_fwd(z(4, 32, 128), z(4, 2, 128), z(4, 2, 128), None, cu, cu, None, None, None, None, 4, 4, 0.0, 0.088,
                     False, True, -1, -1, 0.0, False, None, None)
    with pytest.raises(RuntimeError, match="same dtype"):
        C.varlen_fwd(z(4, 32, 128), z(4, 2, 128).float(), z(4, 2, 128), None, cu, cu, None, None, None, None, 4, 4, 0.0,
                     0.088, False, True, -1, -1, 0.0, False, None, None)
    with pytest.raises(RuntimeError, match="does not support softcap"):
        C.fwd_kvcache(z(1, 1, 32, 128), z(1, 64, 2, 128), z(1, 64, 2, 128), None, None, None, None, None, None, None, None,
                      None, None, 0.088, False, -1, -1, 1.0, True, 0, None)


def _stub_forward(monkeypatch):
    """The operator's host call replaced by one that runs without a GPU: what is tested is the route to it."""
    from types import SimpleNamespace
    import torch
    from infllmv2_cuda_impl_amd import _lib
    monkeypatch.setattr(_lib, "host", SimpleNamespace(varlen_fwd=lambda q, k, *rest: (q * 1.0, torch.zeros(q.shape[1], q.shape[0]), None)))


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("grad", [False, True])
def test_tangents_are_not_dropped(monkeypatch, which, grad):
    """A forward-mode tangent on q, k or v does not set requires_grad; the operator has no forward-mode derivative and says so."""
    import torch
    import torch.autograd.forward_ad as fwd
    from infllmv2_cuda_impl_amd import infllmv2_attn_varlen_func
    _stub_forward(monkeypatch)
    qkv = [torch.randn(4, 32, 128), torch.randn(4, 2, 128), torch.randn(4, 2, 128)]
    cu = torch.tensor([0, 4], dtype=torch.int32)
    f = lambda *t: infllmv2_attn_varlen_func(*t, cu, cu, 4, 4, causal=True)
    with torch.set_grad_enabled(grad):
        assert torch.equal(f(*qkv), qkv[0])
        with fwd.dual_level():
            assert torch.equal(f(*qkv), qkv[0])                # no tangent: as outside
            qkv[which] = fwd.make_dual(qkv[which], torch.ones_like(qkv[which]))
            with pytest.raises(RuntimeError, match="jvp"):
                f(*qkv)
        with pytest.raises(RuntimeError):                      # neither are torch.func's transforms served
            torch.func.jvp(f, tuple(torch.zeros_like(t) for t in (qkv[0], qkv[1], qkv[2])), tuple(torch.ones_like(t) for t in (qkv[0], qkv[1], qkv[2])))


@pytest.mark.parametrize("selection", ["sparse", "dense", "window"])
def test_decode_on_cpu_tensors_says_that_there_is_no_cpu_path(selection):
    import torch
    from infllmv2_cuda_impl_amd import BatchCache, InfLLMv2Attention, SequenceCache
    layer = InfLLMv2Attention(selection=selection)
    q, kv = torch.zeros(1, 1, 32, 128, dtype=torch.bfloat16), torch.zeros(1, 1, 2, 128, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU path"):
        layer.decode(q, kv, kv, SequenceCache.empty(128, 2, 128, "cpu"))
    with pytest.raises(RuntimeError, match="no CPU path"):
        layer.decode_batch(q, kv, kv, BatchCache.empty(1, 128, 2, 128, "cpu"))


def test_the_autograd_function_defaults_the_softmax_scale(monkeypatch):
    """Infllmv2AttnVarlenFunc.apply with no scale: the head size to the power -1/2, as the operator defaults it."""
    from types import SimpleNamespace
    import torch
    from infllmv2_cuda_impl_amd import _lib
    from infllmv2_cuda_impl_amd.attention import Infllmv2AttnVarlenFunc
    scales = []
    monkeypatch.setattr(_lib, "host", SimpleNamespace(varlen_fwd=lambda q, k, v, cq, ck, mq, mk, scale, *rest: (scales.append(scale), (q * 1.0, q, None))[1]))
    q, kv, cu = torch.zeros(4, 32, 128), torch.zeros(4, 2, 128), torch.tensor([0, 4], dtype=torch.int32)
    Infllmv2AttnVarlenFunc.apply(q, kv, kv, cu, cu, 4, 4, 0.0, None, True, (-1, -1), 0.0, None, False, False, None, None)
    assert scales == [128 ** -0.5]


def test_which_walk_a_dense_forward_takes():
    """Sizes at which both walks were timed and differ by more than the timings scatter (query lengths, keys before the first query, KV
    heads, group, by tiles); a number of tiles taken from the longest sequence, or a number of tiles alone, gets several of them wrong."""
    from infllmv2_cuda_impl_amd import _lib
    from test_gpu_tile_walk import CASES, GROUP_CASES
    f = lambda sq, sk, hk, g, causal=True: bool(_lib.lib.infllmv2_varlen_fwd_dense_tiles(len(sq), sum(sq), sum(sk), hk * g, hk, max(sq), max(sk), int(causal)))
    for sq, before, hk, g, tiles in (([3800], 0, 1, 16, False), ([5000], 0, 1, 16, True), ([16000], 0, 1, 16, True), ([1000], 0, 2, 16, False),
                                     ([2200], 0, 2, 16, True), ([1000], 0, 4, 16, True), ([3800], 0, 2, 8, True), ([800], 0, 8, 8, True),
                                     ([1000] + [16] * 3, 0, 2, 16, False), ([1000] + [16] * 30, 0, 4, 16, True), ([4000] + [16] * 100, 0, 2, 16, True),
                                     ([24] * 80, 0, 2, 16, False), ([17] * 130, 0, 2, 16, False), ([130] * 15, 2000, 2, 16, False), ([300] * 2, 6000, 4, 16, True),
                                     ([300] * 2, 6000, 2, 16, False)):
        assert f(sq, [n + before for n in sq], hk, g) == tiles, (sq[:3], len(sq), before, hk, g)
    for sizes in ((0, 0, 0), (1, 1, 0), (1, 1, 1), (2 ** 31 - 1, 2 ** 31 - 1, 2 ** 31 - 1)):
        assert _lib.lib.infllmv2_varlen_fwd_dense_tiles(1, sizes[0], sizes[1], 32, 2, sizes[0], sizes[2], 1) in (0, 1)
    # the cases of the GPU test take the walk they are there for
    for cases, tiles in ((CASES, True), (GROUP_CASES, False)):
        for sq, sk, hk, g, kind in cases:
            assert kind == "all" or f(sq, sk, hk, g, kind != "acausal") == tiles, (sq[:3], len(sq), hk, g)
