"""The work whose speed is measured: one sparse attention layer as a serving process calls it.

Every case goes through the package's public entry points.  A case's ``kind`` is the call:

  decode    decode steps of one request over its arena (fused_decode_step), eight tokens in one
            HIP graph as vLLM's full-graph mode replays them, or eagerly
  dense     one query chunk of the dense prefix (dense_causal_attention)
  sparse    one query chunk past the dense prefix, its clusters already selected
            (kv_outer_attention)
  select    the cluster selection of one query chunk (theta_select_bitmask_flat)
  prefill   a whole prompt through the layer (SembloAttention.prefill): the block build, the
            packed K/V, every dense and sparse chunk, and the decode arena
  token     the same prompt in token order, slice by slice (SembloAttention.prefill_token_order)

Shapes are those of the benchmark's configurations (8 or 16 query heads, 2 or 4 KV heads, head
dimension 128 or 256, prompts of 8K to 512K, 2048 positions per cluster, at least 128 clusters, a
budget of a sixteenth of the prompt) and their neighbourhood: short and odd lengths, chunks
that are no multiple of a tile, 1 to 8 query heads per KV head.  Keys and queries are the benchmark's
Gaussian mixture (segments of consecutive positions share a centre, four large-norm sink keys,
values N(0, 1)), in bf16, the type the kernels take.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path.cwd() / "semantic-block-sparse-attention_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from semblo_amd.config import SembloRuntimeConfig  # noqa: E402
from semblo_amd.fused_decode import fused_decode_step  # noqa: E402
from semblo_amd.fused_select import theta_select_bitmask_flat  # noqa: E402
from semblo_amd.kv_outer import dense_causal_attention, kv_outer_attention  # noqa: E402
from semblo_amd.model import SembloAttention  # noqa: E402
from semblo_amd.state import ProductPostingIndex  # noqa: E402

TEMPERATURE, BETA, ITERS = 0.1, 0.25, 16     # the package's selection settings
PAGE = 16
DECODE_STEPS = 8


def listed():
    return [
        # decode of a short prompt at the CPU-sized configuration's heads: launch and latency
        dict(name="decode_8k_d128", kind="decode", length=8192, hq=8, hkv=2, d=128, suffix=37, graph=True),
        # decode without a graph (a step that is not captured): the host's share counts too
        dict(name="decode_5k_eager", kind="decode", length=5003, hq=16, hkv=4, d=256, suffix=5, graph=False),
        # the headline decode: 128K positions, some hundred tokens generated
        dict(name="decode_128k", kind="decode", length=131072, hq=16, hkv=4, d=256, suffix=200, graph=True),
        # decode at the longest prompt, well into the answer
        dict(name="decode_512k", kind="decode", length=524288, hq=16, hkv=4, d=256, suffix=3001, graph=True),
        # a dense-prefix chunk of an odd length, as the last one of a short prompt or a ragged slice
        dict(name="dense_5000_at_20011", kind="dense", start=20011, queries=5000, hq=16, hkv=4, d=256),
        # a ragged sparse chunk with eight query heads per KV head at the smaller head dimension
        dict(name="sparse_3001_at_40009_d128", kind="sparse", start=40009, queries=3001, length=65536, hq=16,
             hkv=2, d=128),
        # one of the headline prompt's late sparse chunks
        dict(name="sparse_8192_at_114688", kind="sparse", start=114688, queries=8192, length=131072, hq=16,
             hkv=4, d=256),
        # the selection of a slice of a 512K prompt
        dict(name="select_8192_c256", kind="select", start=300000, queries=8192, length=524288, hq=16, hkv=4,
             d=256),
        # the CPU-sized configuration's prompt with chunks of 1024: a small model's layer
        dict(name="prefill_8k_d128", kind="prefill", length=8192, hq=8, hkv=2, d=128, chunk=1024),
        # the 32K configuration
        dict(name="prefill_32k", kind="prefill", length=32768, hq=16, hkv=4, d=256, chunk=8192),
        # the headline prefill
        dict(name="prefill_128k", kind="prefill", length=131072, hq=16, hkv=4, d=256, chunk=8192),
        # the 512K configuration, streamed in token order
        dict(name="token_512k", kind="token", length=524288, hq=16, hkv=4, d=256, chunk=8192),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "dense", "dense", "sparse", "sparse", "sparse", "select",
                       "prefill", "prefill", "token"])
    d = rng.choice([128, 256, 256])
    hkv = rng.choice([1, 2, 4, 4])
    g = rng.choice([1, 2, 4, 4, 4, 8])
    heads = dict(hq=hkv * g, hkv=hkv, d=d)
    if kind == "decode":
        return dict(kind=kind, length=_log_int(rng, 2000, 524288), suffix=_log_int(rng, 1, 6000),
                    graph=rng.random() < 0.75, **heads)
    if kind == "dense":
        return dict(kind=kind, start=rng.choice([0, _log_int(rng, 100, 32768)]), queries=_log_int(rng, 130, 8192),
                    **heads)
    if kind in ("sparse", "select"):
        length = _log_int(rng, 8192, 393216)
        queries = _log_int(rng, 200, 8192)
        start = rng.randint(min(length // 4 + 1, length - queries), length - queries)
        return dict(kind=kind, start=max(1, start), queries=min(queries, length - 1), length=length, **heads)
    if kind == "prefill":
        return dict(kind=kind, length=_log_int(rng, 2000, 150000), chunk=rng.choice([1024, 2048, 4096, 8192, 8192]),
                    **heads)
    return dict(kind=kind, length=_log_int(rng, 70000, 200000), chunk=rng.choice([4096, 8192]), **heads)


# -- inputs -----------------------------------------------------------------------------------


def _clusters(length):
    """The partition's cluster count for a prompt: 2048 positions each, a power of two, at least 128."""
    return 1 << max(7, (max(length // 2048, 64) - 1).bit_length())


def _budget(length):
    return max(1, length // 16)


class _Source:
    """Seeded draws on the GPU and the prompt's segments (consecutive positions on one subject)."""

    def __init__(self, seed, length):
        self.gen = torch.Generator(device="cuda").manual_seed(1000003 * seed + 17)
        host = torch.Generator().manual_seed(seed)
        short = length <= 32768
        lo, hi = (32, 256) if short else (16, 2048)
        count = length // lo + 1
        u = torch.rand(count, generator=host)
        lens = (lo + u * (hi - lo)) if short else torch.exp(math.log(lo) + u * (math.log(hi) - math.log(lo)))
        lens = lens.round().long()
        used = int((lens.cumsum(0) < length).sum()) + 1
        self.segment = torch.arange(used).repeat_interleave(lens[:used])[:length].cuda()
        self.segments = used
        self.host = host

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.gen, device="cuda")


def _mixture(src, length, hkv, d):
    """Centres [Hkv, M, D], each segment's centre, and the keys and values of the prompt."""
    m = 256 if length <= 32768 else 1024
    centres = src.normal(hkv, m, d)
    which = torch.randint(0, m, (src.segments,), generator=src.host).cuda()[src.segment]
    k = torch.empty(length, hkv, d, dtype=torch.bfloat16, device="cuda")
    for h in range(hkv):
        x = centres[h, which] + 0.3 * src.normal(length, d)
        x[:4] *= 8.0
        k[:, h] = x
    v = torch.empty_like(k)
    for h in range(hkv):
        v[:, h] = src.normal(length, d)
    return centres, which, k, v


def _queries(src, centres, which, hq):
    """A query per position: its segment's centre and noise of its own per head."""
    hkv, _, d = centres.shape
    q = torch.empty(which.numel(), hq, d, dtype=torch.bfloat16, device="cuda")
    for j in range(hq):
        q[:, j] = centres[j // (hq // hkv), which] + 0.5 * src.normal(which.numel(), d)
    return q


def _partition(src, length, hkv, c):
    """A cluster per (head, position): segments fall into clusters of very unequal shares, as a
    k-means partition of such keys has them."""
    cluster = torch.empty(hkv, length, dtype=torch.int64, device="cuda")
    for h in range(hkv):
        share = torch.exp(torch.randn(c, generator=src.host))
        pick = torch.multinomial(share, src.segments, replacement=True, generator=src.host).cuda()
        cluster[h] = pick[src.segment]
    return cluster


def _runs(cluster, c, width_align=PAGE):
    """Run starts (whole pages), sizes and the posting lists (position per packed row) of a partition."""
    hkv, length = cluster.shape
    sizes = torch.stack([torch.bincount(cluster[h], minlength=c) for h in range(hkv)])
    rows = (sizes + width_align - 1) // width_align * width_align
    indptr = torch.zeros(hkv, c + 1, dtype=torch.int64, device="cuda")
    indptr[:, 1:] = rows.cumsum(1)
    width = int(indptr[:, -1].max())
    posting = torch.zeros(hkv, width, dtype=torch.int64, device="cuda")
    inverse = torch.empty(hkv, length, dtype=torch.int64, device="cuda")
    for h in range(hkv):
        order = torch.sort(cluster[h], stable=True).indices
        first = sizes[h].cumsum(0) - sizes[h]
        own = cluster[h][order]
        row = indptr[h][own] + torch.arange(length, device="cuda") - first[own]
        posting[h, row] = order
        inverse[h, order] = row
    return sizes, indptr, posting, inverse


def _descriptors(centres, which, cluster, c):
    """The partition's descriptors: the normalised mean of the centres each cluster's keys have."""
    hkv, _, d = centres.shape
    out = torch.zeros(hkv, 2, c, d // 2, dtype=torch.bfloat16, device="cuda")
    for h in range(hkv):
        pairs = torch.zeros(c, centres.shape[1], dtype=torch.float64, device="cuda")
        pairs.view(-1).index_add_(0, cluster[h] * centres.shape[1] + which,
                                  torch.ones(which.numel(), dtype=torch.float64, device="cuda"))
        mean = pairs @ centres[h].double()
        mean = mean / mean.norm(dim=1, keepdim=True).clamp_min(1e-12)
        out[h] = mean.view(c, 2, d // 2).transpose(0, 1).to(torch.bfloat16)
    return out


def _selected(src, visible, queries, target):
    """Which clusters each query reads: liked ones first (segments of queries like the same, small
    clusters count less against the budget), until the visible rows reach the budget."""
    hkv, c = visible.shape
    segment = src.segment[-queries:] - src.segment[-queries]
    n_seg = int(segment[-1]) + 1
    size = visible.float()
    chosen = torch.empty(queries, hkv, c, dtype=torch.bool, device="cuda")
    for h in range(hkv):
        like = 1.2 * src.normal(n_seg, c)[segment] + 0.5 * src.normal(queries, c) - torch.log1p(size[h])
        like = like.masked_fill(visible[h] <= 0, float("-inf"))
        order = like.argsort(dim=1, descending=True)
        got = visible[h][order]
        take = (got.cumsum(1) - got < target) & (got > 0)
        chosen[:, h] = torch.zeros_like(take).scatter(1, order, take)
    return chosen


def _words(chosen):
    q, hkv, c = chosen.shape
    bits = chosen.view(q, hkv, c // 32, 32).long() << torch.arange(32, device="cuda")
    w = bits.sum(-1)
    return torch.where(w >= 2 ** 31, w - 2 ** 32, w).to(torch.int32)


def _routing(q):
    """Unit routing vectors in bf16 (normalised, rounded, normalised again, rounded)."""
    for _ in range(2):
        x = q.float()
        q = (x / x.norm(dim=-1, keepdim=True).clamp_min(1e-12)).to(torch.bfloat16)
    return q


def _inputs(case, seed):
    """The tensors of a case, from its seed alone (plain torch)."""
    kind = case["kind"]
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    t = {}
    if kind == "decode":
        length, c = case["length"], _clusters(case["length"])
        src = _Source(seed, length)
        centres, which, t["k"], t["v"] = _mixture(src, length, hkv, d)
        cluster = _partition(src, length, hkv, c)
        t["sizes"], t["indptr"], t["posting"], t["inverse"] = _runs(cluster, c)
        t["codebooks"] = _descriptors(centres, which, cluster, c)
        t["suffix_k"] = src.normal(case["suffix"], hkv, d).to(torch.bfloat16)
        t["suffix_v"] = src.normal(case["suffix"], hkv, d).to(torch.bfloat16)
        pick = torch.randint(0, centres.shape[1], (DECODE_STEPS,), generator=src.host).cuda()
        t["q"] = _queries(src, centres, pick, hq)
        k_new = centres[:, pick].transpose(0, 1) + 0.3 * src.normal(DECODE_STEPS, hkv, d)
        t["k_new"] = k_new.to(torch.bfloat16).contiguous()
        t["v_new"] = src.normal(DECODE_STEPS, hkv, d).to(torch.bfloat16)
    elif kind == "dense":
        length = case["start"] + case["queries"]
        src = _Source(seed, length)
        centres, which, t["k"], t["v"] = _mixture(src, length, hkv, d)
        t["q"] = _queries(src, centres, which[case["start"]:], hq)
    elif kind == "sparse":
        end, c = case["start"] + case["queries"], _clusters(case["length"])
        src = _Source(seed, end)
        centres, which, t["k"], t["v"] = _mixture(src, end, hkv, d)
        t["q"] = _queries(src, centres, which[case["start"]:], hq)
        t["cluster"] = _partition(src, end, hkv, c)
        t["sizes"], t["indptr"], t["posting"], t["inverse"] = _runs(t["cluster"], c)
        t["visible"] = torch.stack([torch.bincount(t["cluster"][h, :case["start"]], minlength=c)
                                    for h in range(hkv)])
        t["chosen"] = _selected(src, t["visible"], case["queries"], _budget(case["length"]))
    elif kind == "select":
        end, c = case["start"] + case["queries"], _clusters(case["length"])
        src = _Source(seed, end)
        m = 1024
        centres = src.normal(hkv, m, d)
        which = torch.randint(0, m, (src.segments,), generator=src.host).cuda()[src.segment]
        cluster = _partition(src, end, hkv, c)
        t["sizes"] = torch.stack([torch.bincount(cluster[h, :case["start"]], minlength=c) for h in range(hkv)])
        t["codebooks"] = _descriptors(centres, which, cluster, c)
        t["vectors"] = _routing(_queries(src, centres, which[case["start"]:], hq))
    else:
        src = _Source(seed, case["length"])
        centres, which, t["k"], t["v"] = _mixture(src, case["length"], hkv, d)
        t["q"] = _queries(src, centres, which, hq)
    return t


def _layer(case, **more):
    cfg = SembloRuntimeConfig(num_q_heads=case["hq"], num_kv_heads=case["hkv"], head_dim=case["d"], **more)
    return SembloAttention(cfg, layer_name="perf.layer")


def _packed(t):
    """The cluster-ordered K/V store of a partition (a row per packed position, whole pages)."""
    hkv, width = t["posting"].shape
    rows = width + (-width) % 256
    packed = torch.zeros(2, rows, hkv, t["k"].shape[2], dtype=torch.bfloat16, device="cuda")
    for h in range(hkv):
        packed[0, :width, h] = t["k"][t["posting"][h], h]
        packed[1, :width, h] = t["v"][t["posting"][h], h]
    return packed


def prepare(case, seed):
    kind = case["kind"]
    t = _inputs(case, seed)
    state = {"case": case}
    if kind == "decode":
        length = case["length"]
        index = ProductPostingIndex(
            codebooks=t["codebooks"], posting_positions=t["posting"].int(), bucket_indptr=t["indptr"].int(),
            bucket_sizes=t["sizes"].int(), prompt_length=length, max_position=length - 1,
            flat_clusters=t["sizes"].shape[1], page_align=PAGE, _inverse_positions=t["inverse"].int())
        index.pack_prompt_kv(t["k"], t["v"])
        layer = _layer(case, suffix_reserve=8192)
        layer.adopt_index(index)
        layer.target_tokens = _budget(length)
        arena = layer.arena
        # the tokens generated so far, in the suffix store's blocks
        pos = torch.arange(length, length + case["suffix"], device="cuda")
        block = arena.suffix_table[pos // arena.suffix_block].long()
        arena.suffix_kv[0, block, pos % arena.suffix_block] = t["suffix_k"]
        arena.suffix_kv[1, block, pos % arena.suffix_block] = t["suffix_v"]
        first = length + case["suffix"]
        state.update(layer=layer, q=t["q"], k=t["k_new"], v=t["v_new"],
                     out=torch.empty(DECODE_STEPS, case["hq"] * case["d"], dtype=torch.bfloat16, device="cuda"),
                     positions=torch.arange(first, first + DECODE_STEPS, dtype=torch.int32, device="cuda"))
        if case["graph"]:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _decode(state)
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"]):
                _decode(state)
    elif kind == "dense":
        state.update(q=t["q"], k=t["k"], v=t["v"])
    elif kind == "sparse":
        window = (t["k"][case["start"]:], t["v"][case["start"]:])
        state.update(q=t["q"], packed=_packed(t), qmask=_words(t["chosen"]), visible=t["visible"].int(),
                     indptr=t["indptr"].int(), window=window)
    elif kind == "select":
        c = t["sizes"].shape[1]
        ones = torch.ones(case["queries"], case["hq"], 1, device="cuda")
        state.update(vectors=t["vectors"][:, :, None], logmix=ones.log(), codebooks=t["codebooks"],
                     sizes=t["sizes"].int()[None],
                     bitmask=torch.zeros(-(-case["queries"] // 32), case["hkv"], c // 32, dtype=torch.int32,
                                         device="cuda"),
                     qmask=torch.empty(case["queries"], case["hkv"], c // 32, dtype=torch.int32, device="cuda"),
                     theta=torch.empty(case["queries"], case["hkv"], device="cuda"))
    else:
        state.update(q=t["q"], k=t["k"], v=t["v"], out=torch.empty_like(t["q"]),
                     layer=_layer(case, query_chunk_size=case["chunk"]))
    return state


def _decode(s):
    layer = s["layer"]
    cfg = layer.runtime_config
    for i in range(DECODE_STEPS):
        fused_decode_step(layer, layer.arena, q_post=s["q"][i:i + 1], q_pre=s["q"][i:i + 1],
                          positions=s["positions"][i:i + 1], k_post=s["k"][i:i + 1], v_states=s["v"][i:i + 1],
                          output=s["out"][i:i + 1], temperature=cfg.selection_temperature,
                          beta=cfg.bucket_size_penalty, target_tokens=layer.decode_budget(),
                          sm_scale=layer.scaling, num_splits=cfg.decode_num_splits, iters=cfg.iters,
                          suffix_splits=cfg.decode_suffix_splits)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        if "graph" in s:
            s["graph"].replay()
        else:
            _decode(s)
        return s["out"]
    if kind == "dense":
        return dense_causal_attention(s["q"], s["k"], s["v"], sm_scale=case["d"] ** -0.5, chunk_start=case["start"])
    if kind == "sparse":
        out, _ = kv_outer_attention(s["q"], s["packed"], s["qmask"], s["visible"], s["indptr"],
                                    sm_scale=case["d"] ** -0.5, local_kv=s["window"], chunk_start=case["start"],
                                    wstart=case["start"])
        return out
    if kind == "select":
        s["bitmask"].zero_()
        counts, tokens = theta_select_bitmask_flat(
            s["vectors"], s["logmix"], s["codebooks"], s["sizes"], s["bitmask"], temperature=TEMPERATURE, beta=BETA,
            target_tokens=_budget(case["length"]), g_union=32, iters=ITERS, qmask=s["qmask"], theta_out=s["theta"])
        return {"theta": s["theta"], "counts": counts, "tokens": tokens, "qmask": s["qmask"], "bitmask": s["bitmask"]}
    layer = s["layer"]
    if kind == "prefill":
        layer.prefill(s["q"], s["q"], s["k"], s["k"], s["v"], s["out"])
    else:
        layer.prefill_token_order(s["q"], s["q"], s["k"], s["k"], s["v"], s["out"], case["chunk"])
    index = layer.index
    return {"out": s["out"], "codebooks": index.codebooks, "sizes": index.bucket_sizes, "indptr": index.bucket_indptr,
            "inverse": index.inverse_positions()}


# -- what a pass cannot do without -------------------------------------------------------------


def work(case):
    kind = case["kind"]
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    row = 2 * d * 2                      # one position's K and V of one head, bf16
    if kind == "decode":
        c, budget = _clusters(case["length"]), _budget(case["length"])
        rows = budget + case["suffix"] + DECODE_STEPS / 2
        step = hkv * (rows * row + c * d * 2) + 2 * hq * d * 2
        return {"bytes": DECODE_STEPS * step, "flops": DECODE_STEPS * (4.0 * d * hq * rows + 2.0 * d * hq * c)}
    if kind == "dense":
        return _dense_work(case["start"], case["queries"], hq, hkv, d)
    if kind == "sparse":
        n = case["queries"]
        return {"bytes": 2 * n * hq * d * 2 + (case["start"] + n) * hkv * row + n * hkv * _clusters(case["length"]) / 8,
                "flops": _sparse_flops(case["start"], n, case["length"], hq, d)}
    if kind == "select":
        n, c = case["queries"], _clusters(case["length"])
        return {"bytes": n * hq * d * 2 + hkv * c * d * 2 + n * hkv * (c / 8 * (1 + 1 / 32) + 12),
                "flops": 2.0 * n * hq * c * d}
    length, chunk, cap = case["length"], case["chunk"], 4 * _budget(case["length"])
    flops, first = 0.0, 0
    if kind == "token":      # exact until the clusters are fitted, on the first 64K and a slice more
        first = min(length, (min(65536, cap) // chunk + 1) * chunk)
    for start in range(0, length, chunk):
        n = min(chunk, length - start)
        if start <= cap or start < first:
            flops += _dense_work(start, n, hq, hkv, d)["flops"]
        else:
            flops += _sparse_flops(start, n, length, hq, d)
    # q and out, K and V read, the cluster-ordered copy written
    return {"bytes": 2 * length * hq * d * 2 + 2 * length * hkv * row, "flops": flops}


def _dense_work(start, n, hq, hkv, d):
    return {"bytes": 2 * n * hq * d * 2 + (start + n) * hkv * 2 * d * 2,
            "flops": 4.0 * d * hq * (n * (start + 1) + n * (n - 1) / 2)}


def _sparse_flops(start, n, length, hq, d):
    return 4.0 * d * hq * (n * min(_budget(length), start) + n * (n + 1) / 2)


def tolerance(case):
    # Attention: probabilities and outputs are rounded to bf16 (2^-9 of a value), and each cluster's
    # partial result once more in a prefill.  Selections, counts and the partition are whole numbers that
    # follow from fixed 32-bit sums; the cut is such a sum.
    if case["kind"] == "select":
        return {"rel": 5e-6, "differ": 1e-4}
    if case["kind"] in ("prefill", "token"):
        return {"rel": 1e-2, "differ": 0.0}
    return {"rel": 1e-2}


# -- the same results in 64 bits ----------------------------------------------------------------


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "token"):
        return None          # the partition (k-means over seeded draws) has no value of its own
    t = _inputs(case, seed)
    if kind == "decode":
        return _exact_decode(case, t)
    if kind == "select":
        theta = torch.empty(case["queries"], case["hkv"], dtype=torch.float64, device="cuda")
        for lo in range(0, case["queries"], 1024):
            v = t["vectors"][lo:lo + 1024]
            theta[lo:lo + 1024] = _exact_cut(v, t["codebooks"], t["sizes"], _budget(case["length"]))[0]
        return {"theta": theta, "counts": None, "tokens": None, "qmask": None, "bitmask": None}
    return _exact_chunk(case, t)


def _exact_cut(vectors, codebooks, sizes, target):
    """The cut theta [Q, Hkv] and the selection: cluster probabilities of each head's routing vector
    summed over the KV head's query heads, less the size penalty, bisected on the budget."""
    n, hq, d = vectors.shape
    hkv, _, c, _ = codebooks.shape
    words = codebooks.double().transpose(1, 2).reshape(hkv, c, d)
    theta = torch.empty(n, hkv, dtype=torch.float64, device="cuda")
    chosen = torch.empty(n, hkv, c, dtype=torch.bool, device="cuda")
    for h in range(hkv):
        q = vectors.double().view(n, hkv, hq // hkv, d)[:, h].reshape(-1, d)
        p = torch.softmax((q @ words[h].T / TEMPERATURE).view(n, hq // hkv, c), dim=-1).sum(1)
        size = sizes[h].double()
        live = size > 0
        score = p.clamp_min(1e-38).log() - BETA * torch.log1p(size)
        hi = score.masked_fill(~live, -3.4e38).amax(1) + 1e-6
        lo = torch.minimum(score.masked_fill(~live, 3.4e38).amin(1) - 1e-6, hi - 1e-5)
        for _ in range(ITERS):
            mid = (lo + hi) / 2
            reach = ((score >= mid[:, None]) * size).sum(1) >= target
            lo, hi = torch.where(reach, mid, lo), torch.where(reach, hi, mid)
        if float(size.sum()) < target:
            lo = torch.full_like(lo, -3.4e38)
        theta[:, h] = lo
        chosen[:, h] = live & (score >= lo[:, None])
    return theta, chosen


def _exact_decode(case, t):
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    g = hq // hkv
    _, chosen = _exact_cut(_routing(t["q"]), t["codebooks"], t["sizes"], _budget(case["length"]))
    k, v = t["k"], t["v"]
    out = torch.empty(DECODE_STEPS, hq, d, dtype=torch.float64, device="cuda")
    owner = torch.empty(hkv, case["length"], dtype=torch.int64, device="cuda")
    for h in range(hkv):
        owner[h] = torch.searchsorted(t["indptr"][h].contiguous(), t["inverse"][h].contiguous(), right=True) - 1
        # runs of empty clusters share a start: the last of them holds the rows
    for i in range(DECODE_STEPS):
        for h in range(hkv):
            at = torch.nonzero(chosen[i, h][owner[h]]).flatten()
            kk = torch.cat([k[at, h], t["suffix_k"][:, h], t["k_new"][:i + 1, h]]).double()
            vv = torch.cat([v[at, h], t["suffix_v"][:, h], t["v_new"][:i + 1, h]]).double()
            s = t["q"][i, h * g:(h + 1) * g].double() @ kk.T * d ** -0.5
            out[i, h * g:(h + 1) * g] = torch.softmax(s, dim=1) @ vv
    return out.view(DECODE_STEPS, hq * d)


def _exact_chunk(case, t):
    """Causal attention of a chunk; a sparse one sees only its chosen clusters' keys before the chunk."""
    n, start, hq, hkv, d = case["queries"], case["start"], case["hq"], case["hkv"], case["d"]
    g = hq // hkv
    out = torch.empty(n, hq, d, dtype=torch.float64, device="cuda")
    at = torch.arange(start + n, device="cuda")
    for h in range(hkv):
        k, v = t["k"][:, h].double(), t["v"][:, h].double()
        for lo in range(0, n, 256):
            hi = min(n, lo + 256)
            seen = at[None] <= (start + torch.arange(lo, hi, device="cuda"))[:, None]
            if case["kind"] == "sparse":
                seen &= (at[None] >= start) | t["chosen"][lo:hi, h][:, t["cluster"][h]]
            q = t["q"][lo:hi, h * g:(h + 1) * g].double().reshape(-1, d)
            s = (q @ k.T * d ** -0.5).view(hi - lo, g, -1).masked_fill_(~seen[:, None], float("-inf"))
            out[lo:hi, h * g:(h + 1) * g] = (torch.softmax(s, dim=-1).view(-1, start + n) @ v).view(hi - lo, g, d)
    return out
