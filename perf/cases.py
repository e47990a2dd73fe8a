"""Performance cases of the two-stage sparse attention path: what a user of the package has it do.

A case is a plain dict.  Its ``path`` says which public entry points a pass goes through:

* ``prefill``  - ``InfLLMv2Attention`` over packed prompts (selection and attention, no gradients);
* ``chunk``    - the operators called one by one, as a port of code written against the reference package calls them:
                 compressed keys, ``infllmv2_attn_stage1``, ``max_pooling_1d_varlen``, top-k, ``infllmv2_attn_varlen_func`` with
                 ``topk_idx``; the queries are the last ``queries`` tokens of every sequence (a chunk of a long prompt) or all of them;
* ``train``    - the layer forward and backward: output and gradients of q, k and v;
* ``decode``   - one step of ``decode_batch`` for a batch of sequences against its caches;
* ``decode_one`` - one step of ``decode`` for a single sequence;
* ``decode_paged`` - one step of a serving loop that calls the operators itself: Stage 1 against compressed-key caches, top-k,
                 attention over a paged cache with rotary embedding on append.

``lens`` lists the sequence lengths; where a batch is large they are drawn instead, from ``lens_seed`` over
``[lens_min, lens_max]``.  Values are i.i.d. N(0, 1), as in the repository's benchmark configurations: neighbouring tokens then
share few of the blocks that are chosen by score.
"""
from __future__ import annotations

import math
import random

import torch

import infllmv2_cuda_impl_amd as ops

D = 128            # head size
BLOCK = 64         # tokens per key block
FINE = (32, 16)    # window and stride of the compressed keys
COARSE = (128, 64)  # ... of the set the log-sum-exp is taken over


def _case(path, lens="", **more):
    case = {"path": path, "lens": lens, "lens_seed": 0, "lens_min": 0, "lens_max": 0, "batch": 0, "queries": 0, "heads_k": 2,
            "group": 16, "topk": 64, "local": 31, "init": 1, "dtype": "bf16", "selection": "sparse", "page": 0}
    case.update(more)
    return case


def listed():
    cases = {
        # a short prompt on its own: launches, host work and the kernels' fixed costs count (2048 tokens, top 16 blocks)
        "prefill_2k": _case("prefill", "2048", topk=16, local=1),
        # prompts of a serving batch prefilled together, lengths as they come
        "prefill_ragged": _case("prefill", "777,5003,1291,9173", dtype="fp16"),
        # the headline configuration: one 32K prompt
        "prefill_32k": _case("prefill", "32768"),
        # the longest context
        "prefill_128k": _case("prefill", "131072"),
        # prompts short enough that a model attends densely
        "prefill_dense": _case("prefill", "2500,6001,4096", selection="dense"),
        # chunked prefill of a long prompt through the reference's own sequence of calls
        "chunk_2k_of_20k": _case("chunk", "20011", queries=2049),
        # training on packed sequences: the benchmark's 4 sequences, multiples of 64 in [4096, 24576]
        "train_packed": _case("train", "14848,20480,24320,11904"),
        # fine-tuning on short samples, lengths as they come
        "train_short": _case("train", "1023,3001,517,2200", topk=16, local=4),
        # the benchmark's decode step: 64 sequences with 16K to 128K tokens held
        "decode_64": _case("decode", batch=64, lens_seed=1, lens_min=16383, lens_max=131071),
        # a few conversations at a time
        "decode_6": _case("decode", batch=6, lens_seed=2, lens_min=1500, lens_max=20000),
        # one user, interactive
        "decode_one_32k": _case("decode_one", "32767"),
        # a serving loop on a paged cache
        "decode_paged_24": _case("decode_paged", batch=24, lens_seed=3, lens_min=3000, lens_max=40000, page=128),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _split(rng, total, parts):
    """``parts`` ragged lengths that add up to about ``total``."""
    w = [rng.uniform(0.3, 1.7) for _ in range(parts)]
    return ",".join(str(max(130, int(total * x / sum(w)))) for x in w)


def draw(rng):
    path = rng.choice(["prefill", "prefill", "chunk", "train", "decode", "decode", "decode_one", "decode_paged"])
    topk = rng.choice([16, 32, 64])
    more = {"topk": topk, "local": rng.randint(1, topk // 2 - 1), "dtype": rng.choice(["bf16", "bf16", "bf16", "fp16"]),
            "heads_k": rng.choice([1, 2, 2, 4]), "group": rng.choice([16, 16, 16, 8])}
    if path == "prefill":
        more["selection"] = rng.choice(["sparse", "sparse", "sparse", "sparse", "dense", "window"])
        total = _log_int(rng, 1000, 16000 if more["selection"] == "dense" else 120000 // more["heads_k"])
        return _case(path, _split(rng, total, rng.choice([1, 1, 2, 5]) if total >= 4000 else 1), **more)
    if path == "chunk":
        total = _log_int(rng, 2000, 60000 // more["heads_k"])
        return _case(path, _split(rng, total, rng.choice([1, 1, 3])), queries=rng.choice([0, _log_int(rng, 256, 4096)]), **more)
    if path == "train":
        total = _log_int(rng, 1500, 64000 // more["heads_k"])
        return _case(path, _split(rng, total, rng.choice([1, 2, 4])), **more)
    if path == "decode_one":
        return _case(path, str(_log_int(rng, 1000, 131071)), **more)
    batch = _log_int(rng, 1, 64)
    lens_max = _log_int(rng, 2000, 120000 // max(1, more["heads_k"] // 2) if path == "decode" else 40000)
    return _case(path, batch=batch, lens_seed=rng.randrange(1 << 20), lens_min=max(500, lens_max // rng.randint(2, 12)),
                 lens_max=lens_max, page=rng.choice([64, 128, 256]) if path == "decode_paged" else 0, **more)


def _lens(case):
    if case["lens"]:
        return [int(x) for x in case["lens"].split(",")]
    r = random.Random(case["lens_seed"])
    return [r.randint(case["lens_min"], case["lens_max"]) for _ in range(case["batch"])]


def _queries(case, n):
    return min(case["queries"], n) if case["queries"] else n


def _rows(n, window, stride):
    """Compressed keys of n tokens."""
    return (n - window) // stride + 1 if n >= window else 0


def _layer(case):
    return ops.InfLLMv2Attention(topk=case["topk"], local_blocks=case["local"], init_blocks=case["init"], selection=case["selection"])


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
    hk, hq = case["heads_k"], case["heads_k"] * case["group"]
    lens, path = _lens(case), case["path"]
    rand = lambda *shape: torch.randn(shape, generator=gen, device=dev, dtype=dtype)
    cum = lambda ns: torch.tensor([sum(ns[:i]) for i in range(len(ns) + 1)], dtype=torch.int32, device=dev)
    s = {"path": path, "layer": _layer(case), "case": case}
    if path in ("prefill", "train"):
        total = sum(lens)
        s.update(q=rand(total, hq, D), k=rand(total, hk, D), v=rand(total, hk, D), cu=cum(lens), longest=max(lens))
        if path == "train":
            s["dout"] = rand(total, hq, D)
            for name in ("q", "k", "v"):
                s[name].requires_grad_(True)
    elif path == "chunk":
        n_q = [_queries(case, n) for n in lens]
        s.update(q=rand(sum(n_q), hq, D), k=rand(sum(lens), hk, D), v=rand(sum(lens), hk, D), cu_q=cum(n_q), cu_k=cum(lens),
                 longest_q=max(n_q), longest=max(lens), held=torch.tensor([n - c for n, c in zip(lens, n_q)], dtype=torch.int32, device=dev),
                 most_held=max(n - c for n, c in zip(lens, n_q)))
    elif path == "decode_one":
        n = lens[0]
        cache = ops.SequenceCache.empty(n + BLOCK, hk, D, dev, dtype=dtype)
        s["layer"](rand(n, hq, D), rand(n, hk, D), rand(n, hk, D), cum([n]), n, cache=cache)     # the prompt
        s.update(cache=cache, held=n, q=rand(1, 1, hq, D), k=rand(1, 1, hk, D), v=rand(1, 1, hk, D))
    elif path == "decode":
        b = len(lens)
        cache = ops.BatchCache.empty(b, max(lens) + BLOCK, hk, D, dev, dtype=dtype)
        s["layer"].fill_cache(cache, rand(sum(lens), hk, D), rand(sum(lens), hk, D), lens)
        s.update(cache=cache, lengths=cache.lengths, longest=cache.max_length, q=rand(b, 1, hq, D), k=rand(b, 1, hk, D), v=rand(b, 1, hk, D))
    else:
        b, page = len(lens), case["page"]
        per_seq = max(lens) // page + 1
        table = torch.randperm(b * per_seq, generator=gen, device=dev).to(torch.int32).view(b, per_seq)
        keys, values = rand(b * per_seq, page, hk, D), rand(b * per_seq, page, hk, D)
        held = torch.tensor(lens, dtype=torch.int32, device=dev)
        flat = keys[table.view(-1).long()].view(b, per_seq * page, hk, D)
        fine = torch.zeros(b, per_seq * page // FINE[1] + 1, hk, D, dtype=dtype, device=dev)
        coarse = torch.zeros(b, per_seq * page // COARSE[1] + 1, hk, D, dtype=dtype, device=dev)
        fine_lens, coarse_lens = ops.compress_keys_cache_pair(flat, held, FINE + (fine,), COARSE + (coarse,))
        angle = torch.arange(per_seq * page, device=dev)[:, None] * (10000.0 ** (-torch.arange(D // 2, device=dev) / (D // 2)))
        s.update(keys=keys, values=values, table=table, held=held, longest=max(lens), fine=fine, coarse=coarse, fine_lens=fine_lens,
                 coarse_lens=coarse_lens, cos=angle.cos().to(dtype), sin=angle.sin().to(dtype), q=rand(b, 1, hq, D), k=rand(b, 1, hk, D),
                 v=rand(b, 1, hk, D))
    return s


def run(s):
    path, layer, case = s["path"], s["layer"], s["case"]
    if path == "prefill":
        with torch.no_grad():
            return layer(s["q"], s["k"], s["v"], s["cu"], s["longest"])
    if path == "train":
        out = layer(s["q"], s["k"], s["v"], s["cu"], s["longest"])
        return (out.detach(),) + torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"])
    if path == "chunk":
        fine, cu_fine = ops.compress_keys(s["k"], s["cu_k"], s["longest"], *FINE)
        coarse, cu_coarse = ops.compress_keys(s["k"], s["cu_k"], s["longest"], *COARSE)
        most = _rows(s["longest"], *FINE)
        score = ops.infllmv2_attn_stage1(s["q"], fine, coarse, s["cu_q"], cu_fine, cu_coarse, s["longest_q"], most, causal=True)
        pooled = ops.max_pooling_1d_varlen(score, s["cu_q"], cu_fine, s["held"], s["longest_q"], most, case["local"], case["init"],
                                           max_cache_len=s["most_held"])
        idx = ops.topk_blocks(pooled, case["topk"])
        out = ops.infllmv2_attn_varlen_func(s["q"], s["k"], s["v"], s["cu_q"], s["cu_k"], s["longest_q"], s["longest"], causal=True,
                                            topk_idx=idx)
        return {"score": score, "idx": idx, "out": out}
    if path == "decode_one":
        cache = s["cache"]
        cache.length = s["held"]                                        # every pass is the step at this length
        out = layer.decode(s["q"], s["k"], s["v"], cache)
        return {"out": out, "k": cache.k, "v": cache.v, "k_fine": cache.k_fine, "k_coarse": cache.k_coarse}
    if path == "decode":
        cache = s["cache"]
        cache.lengths, cache.max_length = s["lengths"], s["longest"]
        out = layer.decode_batch(s["q"], s["k"], s["v"], cache)
        return {"out": out, "k": cache.k, "v": cache.v, "k_fine": cache.k_fine, "k_coarse": cache.k_coarse, "lengths": cache.lengths,
                "fine_lens": cache.fine_lens, "coarse_lens": cache.coarse_lens}
    pooled = ops.infllmv2_attn_stage1_kvcache(s["q"], s["fine"], s["coarse"], s["fine_lens"], s["coarse_lens"], s["held"], case["local"],
                                              case["init"], max_cache_len=s["longest"])
    idx = ops.topk_blocks(pooled, case["topk"])
    out = ops.infllmv2_attn_with_kvcache(s["q"], s["keys"], s["values"], k=s["k"], v=s["v"], rotary_cos=s["cos"], rotary_sin=s["sin"],
                                         cache_seqlens=s["held"], block_table=s["table"], rotary_interleaved=False,
                                         topk_idx=idx.unsqueeze(2))
    return {"idx": idx, "out": out, "keys": s["keys"], "values": s["values"]}


def work(case):
    """Bytes: inputs read and outputs written once (decode: the selected blocks, the compressed keys and the appended rows).  FLOPs: the
    Stage-1 products with the visible compressed keys and the attention products over the selected causal blocks (a
    backward 2.5 times the forward)."""
    hk, grp, path = case["heads_k"], case["group"], case["path"]
    row, hq = 2 * D, case["heads_k"] * case["group"]
    sparse = case["selection"] == "sparse"
    byts = flops = 0
    for n in _lens(case):
        if path.startswith("decode"):
            held = n + 1
            blocks = min(case["topk"], (held + BLOCK - 1) // BLOCK)
            comp = _rows(held, *FINE) + _rows(held, *COARSE)
            byts += hk * row * (2 * blocks * BLOCK + comp + 4) + 2 * hq * row
            flops += hk * grp * D * (4 * blocks * BLOCK + 2 * comp)
            continue
        n_q = _queries(case, n)
        picked = comp = 0
        most = {"sparse": case["topk"], "window": case["init"] + case["local"] + 1, "dense": n}[case["selection"]]
        for start in range((n - n_q) // BLOCK * BLOCK, n, BLOCK):          # the queries, a block at a time
            rows = min(start + BLOCK, n) - max(start, n - n_q)
            picked += rows * min(most, start // BLOCK + 1)
            comp += rows * (_rows(start, *FINE) + _rows(start, *COARSE))
        byts += 2 * hq * n_q * row + 2 * hk * n * row
        flops += hk * grp * D * (4 * BLOCK * picked + (2 * comp if sparse else 0))
        if path == "train":
            byts += 2 * hq * n_q * row + 2 * hk * n * row
            flops += hk * grp * D * 10 * BLOCK * picked
        elif path == "chunk":                                             # the operators hand scores and indices to their caller
            byts += hk * n_q * (2 * _rows(n, *FINE) + 4 * case["topk"])
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    """16-bit inputs, outputs and probabilities, 32-bit sums.  Where the selection runs inside a pass, two block scores that round to
    the same or neighbouring 16-bit values may be taken in the other order, and single rows then attend another block."""
    return {"rel": 1e-2, "max": 0.5, "differ": 2e-3}
