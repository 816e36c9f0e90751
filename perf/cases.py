"""What the framework is timed on: the operator stack of one attention layer, called as a serving or training
program calls it.

Sizes are the repository's own: head shapes 4/4, 16/2, 16/16, 32/4 and 32/8 (query / KV heads) of 64 or 128, chunks of
64 tokens, 8 to 32 selected chunks, a local window of 64 or 512 tokens, the batch and sequence lengths of its benchmark
and tests, and lengths that are no multiple of anything.  Paths:

* ``decode``   one token per sequence on the dense cache layer: local branch over the tail of the cache, chunk selection,
               sparse attention, merge.  With mean-pooled chunk keys or in the layer's default mode (attention-pooled
               keys, one per query head, and their entropy as prior bias).
* ``paged``    the remote branch of the same step on K and V in pages handed out in random order.
* ``extend``   a block of new tokens at the end of a longer cache (chunked prefill, a follow-up prompt).
* ``prefill``  the layer's forward on a whole prompt: norm + rotary embedding of q and k, chunk keys, local branch,
               selection, sparse attention with the merge.
* ``train``    the same with gradients, forward and backward.
* ``logz``     the exact per-chunk log-sum-exp (the selection scores of the exact variant), forward and backward.
"""
import math
import os

import torch

import __graft_entry__ as _entry

pkg = _entry.load_package()

S = 64  # chunk length, everywhere


def _case(name, path, batch, length, context, heads, topk, window, keys):
    hq, hkv, d = heads
    case = {"path": path, "batch": batch, "length": length, "context": context, "q_heads": hq, "kv_heads": hkv,
            "head_dim": d, "topk": topk, "window": window, "keys": keys}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one user's chat with a small model: a step is a handful of launches on a short cache
        _case("decode_b1_4k", "decode", 1, 1, 4097, (16, 2, 64), 16, 512, "mean"),
        # a few users, documents of different kinds, the layer's default chunk keys
        _case("decode_b4_30k_prior", "decode", 4, 1, 30001, (32, 4, 64), 32, 512, "attention"),
        # a busy server on the dense cache
        _case("decode_b8_100k", "decode", 8, 1, 100033, (32, 8, 128), 32, 512, "mean"),
        # the benchmark's decode step: 32 sequences of 128K tokens in pages
        _case("paged_b32_128k", "paged", 32, 1, 131072, (32, 8, 128), 32, 64, "mean"),
        # a short prompt of a small model, ragged, default chunk keys
        _case("prefill_2k_prior", "prefill", 1, 1999, 1999, (16, 2, 64), 8, 512, "attention"),
        # the benchmark's batch of 8K prompts
        _case("prefill_b4_8k", "prefill", 4, 8192, 8192, (16, 16, 64), 32, 64, "mean"),
        # the benchmark's 32K prompt
        _case("prefill_32k", "prefill", 1, 32768, 32768, (32, 8, 128), 32, 64, "mean"),
        # a slice of a chunked prefill deep in a long prompt
        _case("extend_2k_at_64k", "extend", 1, 2048, 65500, (32, 8, 128), 32, 512, "mean"),
        # fine-tuning on short sequences, default chunk keys
        _case("train_1k_prior", "train", 2, 1024, 1024, (16, 2, 64), 8, 512, "attention"),
        # the benchmark's training layer
        _case("train_b8_8k", "train", 8, 8192, 8192, (16, 16, 64), 32, 64, "mean"),
        # pretraining of a middle-sized model in the default mode
        _case("train_b2_8k_prior", "train", 2, 8192, 8192, (32, 4, 64), 32, 512, "attention"),
        # the exact variant's selection scores, trained through
        _case("logz_8k", "logz", 1, 8192, 8192, (32, 8, 128), 0, 64, "none"),
    ]


_HEADS = [(4, 4, 64), (16, 2, 64), (16, 16, 64), (32, 4, 64), (32, 4, 128), (32, 8, 128)]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["decode", "decode", "decode", "paged", "prefill", "prefill", "extend", "train", "train", "logz"])
    heads = rng.choice(_HEADS)
    hq, hkv, d = heads
    topk = rng.choice([8, 16, 32])
    window = rng.choice([64, 512])
    keys = rng.choice(["mean", "attention"])
    if path in ("decode", "paged"):
        context = _log_int(rng, 2048, 131072)
        # no more cache than the listed cases keep
        most = {"decode": 8 * 100033 * 8 * 128, "paged": 32 * 131072 * 8 * 128}[path]
        if path == "paged":
            keys = "mean"
        batch = _log_int(rng, 1, max(1, min(32, most // (context * hkv * d))))
        return _case(None, path, batch, 1, context, heads, topk, window, keys)
    if path == "extend":
        length = _log_int(rng, 128, 2048)
        context = _log_int(rng, 4096, 65500)
        return _case(None, path, 1, length, max(context, 2 * length), heads, topk, window, keys)
    if path == "logz":
        length = _log_int(rng, 512, 8192)
        batch = 1 if length > 2048 else rng.choice([1, 2])
        return _case(None, path, batch, length, length, heads, 0, window, "none")
    # whole sequences: up to the tokens (times heads) of the largest listed ones
    length = _log_int(rng, 1024, 16384 if path == "prefill" else 8192)
    most = {"prefill": 16384 * 32 * 128, "train": 8192 * 32 * 64}[path]
    batch = _log_int(rng, 1, max(1, min(8, most // (length * hq * d))))
    return _case(None, path, batch, length, length, heads, topk, window, keys)


# ---- inputs ------------------------------------------------------------------------------------

def _randn(shape, gen, scale=None, chunk=1 << 28):
    """bf16 N(0,1) made on the GPU in slices, times a scale per head (second to last dimension)."""
    out = torch.empty(shape, dtype=torch.bfloat16, device="cuda")
    flat = out.view(-1)
    for a in range(0, flat.numel(), chunk):
        flat[a:a + chunk].normal_(generator=gen)
    return out if scale is None else out.mul_(scale.to(torch.bfloat16).view(-1, 1))


def _tables(length, d, first=0):
    """Rotary tables (length, d), rotate-half convention, base 10000."""
    inv = 10000.0 ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float32) / d)
    ang = torch.arange(first, first + length, device="cuda", dtype=torch.float32)[:, None] * inv
    ang = torch.cat([ang, ang], -1)
    return ang.cos().bfloat16(), ang.sin().bfloat16()


def prepare(case, seed):
    b, length, context = case["batch"], case["length"], case["context"]
    hq, hkv, d, window = case["q_heads"], case["kv_heads"], case["head_dim"], case["window"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n = context // S
    # chunk scores are peaked in some heads and flat in others, as the benchmark's are
    head_scale = torch.rand(hq, device="cuda", generator=gen) * 1.5 + 0.5
    kv_scale = head_scale[:: hq // hkv].contiguous()
    st = {"case": dict(case), "path": case["path"]}

    if case["path"] in ("decode", "extend"):
        cache = pkg.HiLSDynamicLayer(chunk_size=S, offload=False, chunk_pooling=case["keys"] == "mean")
        k = _randn((b, context, hkv, d), gen, kv_scale)
        v = _randn((b, context, hkv, d), gen)
        mu = _randn((b, n, hq, d), gen) if case["keys"] == "attention" else None
        st["keys"], st["values"] = cache.update(k, v, mu_q=mu)  # the views that the last update handed out
        st["cache"] = cache
        st["q"] = _randn((b, length, hq, d), gen, head_scale)
    elif case["path"] == "paged":
        pages = b * n
        st["k_pages"] = _randn((pages, hkv, S, d), gen)
        st["k_pages"].mul_(kv_scale.to(torch.bfloat16).view(-1, 1, 1))
        st["v_pages"] = _randn((pages, hkv, S, d), gen)
        table = torch.randperm(pages, device="cuda", generator=gen).view(b, n)
        st["table"] = table.to(torch.int32).contiguous()
        pooled = pkg.chunk_mean_pool(st["k_pages"].view(-1, S, 1, d), S).view(pages, hkv, d)
        st["chunk_keys"] = pooled[table].permute(0, 2, 1, 3).contiguous()  # (b, hkv, n, d)
        st["q"] = _randn((b, 1, hq, d), gen, head_scale)
        st["lse"] = torch.randn(b, 1, hq, device="cuda", generator=gen) + 4.0  # of the local branch, fp32
    elif case["path"] in ("prefill", "train"):
        st["x_q"] = _randn((b, length, hq, d), gen)   # the projections' outputs
        st["x_k"] = _randn((b, length, hkv, d), gen)
        st["v"] = _randn((b, length, hkv, d), gen)
        # norm weights of the range of the head scales: scores of a standard deviation above one
        st["w_q"] = (torch.rand(d, device="cuda", generator=gen) * 1.5 + 0.5).bfloat16()
        st["w_k"] = (torch.rand(d, device="cuda", generator=gen) * 1.5 + 0.5).bfloat16()
        st["cos"], st["sin"] = _tables(length, d)
        if case["keys"] == "attention":
            st["mu"] = _randn((b, n, hq, d), gen)  # the chunks' prior queries
        if case["path"] == "train":
            st["d_o"] = _randn((b, length, hq, d), gen)
            st["wrt"] = [x for x in ("x_q", "x_k", "v", "w_q", "w_k", "mu") if x in st]
            for x in st["wrt"]:
                st[x].requires_grad_()
    else:
        st["q"] = _randn((b, length, hq, d), gen).requires_grad_()
        st["k"] = _randn((b, length, hkv, d), gen).requires_grad_()
        n_z = -(-length // S)
        t = torch.arange(length, device="cuda").view(-1, 1)
        c = torch.arange(n_z, device="cuda").view(1, -1)
        seen = (c + 1) * S <= t - window + 1  # chunks that lie wholly before the local window
        d_z = torch.randn((b, length, hq, n_z), device="cuda", generator=gen)
        st["d_z"] = d_z.mul_(seen.view(1, length, 1, n_z))
    return st


# ---- one pass ----------------------------------------------------------------------------------

def _on_cache(st, c):
    """The layer on a cache: the last `length` positions of `context`."""
    q, window = st["q"], c["window"]
    first = max(0, (c["context"] - c["length"] - window + 1) // S * S)  # where the first query's window begins
    swa_o, lse = pkg.flex_attn_tl(q, st["keys"][:, first:], st["values"][:, first:], window, S, training=False,
                                  kv_start=first)
    o, w, idx = st["cache"].hils_attend(q, lse, c["topk"], window)
    return {"o": torch.addcmul(o, swa_o, w[..., -1:]), "indices": idx}


def _chunk_keys(st, c, k):
    """(k chunks, mu) -> chunk keys and prior bias of the default mode."""
    b, length, hkv, d = k.shape
    n = length // S
    return pkg.chunk_attn_pool(st["mu"], k[:, : n * S].reshape(b, n, S, hkv, d))


def _keys_and_queries(st, c):
    q, _ = pkg.norm_rope_pool(st["x_q"], st["w_q"], st["cos"], st["sin"], S, pool=False)
    mean = c["keys"] == "mean"
    k, lmk = pkg.norm_rope_pool(st["x_k"], st["w_k"], st["cos"], st["sin"], S, pool=mean)
    prior = None
    if not mean:
        lmk, prior = _chunk_keys(st, c, k)
    return q, k, lmk, prior


def _prefill(st, c):
    with torch.no_grad():
        q, k, lmk, prior = _keys_and_queries(st, c)
        swa_o, lse = pkg.flex_attn_tl(q, k, st["v"], c["window"], S)
        idx, _, w = pkg.topk_chunk_weights(q, lmk, lse, c["topk"], S, c["window"], prior_b=prior,
                                           num_kv_heads=c["kv_heads"])
        o = pkg.HiLS_block_M_head(q, k, st["v"], w, idx, block_size=S, is_training=False, swa_o=swa_o)
    return {"o": o, "k": k, "chunk_keys": lmk, "indices": idx}  # k and the chunk keys go into the cache


def _train(st, c):
    q, k, lmk, prior = _keys_and_queries(st, c)
    swa_o, lse = pkg.flex_attn_tl(q, k, st["v"], c["window"], S)
    b, length, hq, d = q.shape
    grouped = q.view(b, length, c["kv_heads"], hq // c["kv_heads"], d)
    idx, scores = pkg.online_softmax_topk_head(grouped, lmk, lse.detach(), c["topk"], S, c["window"],
                                               bias=None if prior is None else prior.detach())
    w = pkg.chunk_weights(scores, lse, prior, idx)
    o = pkg.HiLS_block_M_head(q, k, st["v"], w, idx, block_size=S, swa_o=swa_o)
    grads = torch.autograd.grad(o, [st[x] for x in st["wrt"]], st["d_o"])
    return {"o": o, **{"d_" + x: g for x, g in zip(st["wrt"], grads)}}


def run(state):
    c = state["case"]
    path = state["path"]
    if path in ("decode", "extend"):
        return _on_cache(state, c)
    if path == "paged":
        o, w, idx = pkg.paged_hils_attend(state["q"], state["k_pages"], state["v_pages"], None, state["table"],
                                          state["lse"], c["context"], c["topk"], c["window"],
                                          lmk_dense=state["chunk_keys"])
        return {"o": o, "weights": w, "indices": idx}
    if path == "prefill":
        return _prefill(state, c)
    if path == "train":
        return _train(state, c)
    z = pkg.exact_chunk_log_z_tl(state["q"], state["k"], chunk_size=S, window_size=c["window"])
    d_q, d_k = torch.autograd.grad(z, [state["q"], state["k"]], state["d_z"])
    return {"log_z": z, "d_q": d_q, "d_k": d_k}


# ---- work --------------------------------------------------------------------------------------

def _positions(c):
    """(selected chunks, visible chunks, tokens in the local window), each summed over the queries of a sequence."""
    sel = vis = win = 0
    for t in range(c["context"] - c["length"], c["context"]):
        seen = min(max(0, (t - c["window"] + 1) // S), c["context"] // S)
        vis += seen
        sel += min(c["topk"], seen)
        win += t + 1 - max(0, (t - c["window"] + 1) // S * S)
    return sel, vis, win


def work(case):
    c = case
    b, length, context = c["batch"], c["length"], c["context"]
    hq, hkv, d = c["q_heads"], c["kv_heads"], c["head_dim"]
    n = context // S
    sel, vis, win = _positions(c)
    h_keys = hq if c["keys"] == "attention" else hkv
    q_bytes, kv_bytes = 2 * b * length * hq * d, 2 * b * length * hkv * d
    idx_bytes = 4 * b * length * hkv * c["topk"]
    score = 2 * d * hq * b * vis                   # query times chunk keys
    attend = 4 * d * S * hq * b * sel              # two products over the selected chunks
    local = 4 * d * hq * b * win                   # two products over the window
    if c["path"] in ("decode", "paged", "extend"):
        keys = 2 * b * h_keys * (vis // length if length == 1 else n) * d
        prior = 4 * b * n * hq if c["keys"] == "attention" else 0
        # K and V of the chunks that are selected (by many queries: of no more than there are), and of the window
        tokens = min(sel * S, context) + (0 if c["path"] == "paged" else win // length + length)
        rows = 4 * b * hkv * min(tokens, context) * d
        out = (2 * b * length * hq * (c["topk"] + 1) + 4 * b * length * hq) if c["path"] == "paged" else 0
        flops = score + attend + (0 if c["path"] == "paged" else local)
        return {"bytes": 2 * q_bytes + keys + prior + rows + idx_bytes + out, "flops": flops}
    if c["path"] == "prefill":
        # in: the projections, tables; out: o, k, chunk keys, indices
        extra = 2 * b * n * hq * d if c["keys"] == "attention" else 0
        return {"bytes": 2 * q_bytes + 3 * kv_bytes + 4 * length * d + 2 * b * n * h_keys * d + extra + idx_bytes,
                "flops": score + attend + local}
    if c["path"] == "train":
        # in: x_q, x_k, v, d_o; out: o and the gradients.  Backward: five products per pair of the attention (S again,
        # dP, dQ, dK, dV) for the forward's two, two for the selection scores' one
        extra = 4 * b * n * hq * d if c["keys"] == "attention" else 0
        return {"bytes": 4 * q_bytes + 4 * kv_bytes + 4 * length * d + extra,
                "flops": score + 3.5 * (attend + local) + 4 * d * hq * b * sel}
    # log-Z: the scores, once more in the backward, and the two gradient products; z is written and read, d_z read
    pairs = vis * S
    z = 4 * b * length * hq * (-(-length // S))
    return {"bytes": 2 * z + 2 * q_bytes + 2 * kv_bytes, "flops": 4 * 2 * d * hq * b * pairs}


def tolerance(case):
    """bf16 inputs and outputs, fp32 accumulation.  A few of the selected chunks may be others where scores tie to the
    last bits of a sum taken in another order."""
    return {"rel": 1e-2, "max": 0.5, "differ": 5e-3}
