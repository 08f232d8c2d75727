"""The calls that users of this package make, as benchmark cases with inputs made from a seed.

``listed()`` holds the fixed cases, ``draw(rng)`` gives further ones of the same ranges. A case is
prepared once (``prepare``: the tensors a program has in hand before the call, or the plan it keeps),
passed any number of times through the public entry points (``run``), and can be compared with the
same call in 64 bits (``exact``).

Kinds of case:
  index         ``lightning_indexer`` on BSND prompts (a whole prompt, or a chunk of its queries
                over the keys so far)
  index_paged   ``IndexerPlan`` over a serving engine's paged key cache: one token per sequence
                (or a few, with speculative tokens), at its own length
  attend        ``sparse_flash_attention`` on BSND or packed (TND) prompts, indices as an indexer
                gives them (distinct visible positions in no order of position, -1 behind them)
  attend_paged  ``AttentionPlan`` over a serving engine's paged latent cache
  prefill       ``dsa_prefill``: indexer and attention on one packed batch
  attend_grad   ``sparse_flash_attention_grad`` after its forward
  index_loss    ``sparse_lightning_indexer_grad_kl_loss`` after the attention's forward
  dense_loss    the warm-up stage's ``dense_lightning_indexer_softmax_lse`` and
                ``dense_loss_backward``
"""
import math
import random

import torch

import dsa_triton_ascend_amd as dsa
from dsa_triton_ascend_amd.lightning_indexer import IndexerPlan
from dsa_triton_ascend_amd.sparse_flash_attention import AttentionPlan

ROPE = 64
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _numbers(text):
    return [int(v) for v in text.split(",")]


def _text(values):
    return ",".join(str(int(v)) for v in values)


def _spread(n, low, high, seed):
    """n sequence lengths between low and high, even over the range, in no order."""
    r = random.Random(seed)
    got = [round(low + (high - low) * (i + 0.5) / n) for i in range(n)]
    r.shuffle(got)
    return got


def listed():
    return [
        # the smallest indexer call: one short prompt, few heads (host work and launches count)
        dict(name="index_short", kind="index", dtype="bf16", weights="fp32", batch=1, queries=256, keys=256,
             heads=8, top=64, values=True),
        # a whole 8K prompt with the model's 64 indexer heads
        dict(name="index_prompt_8k", kind="index", dtype="bf16", weights="fp32", batch=1, queries=8192,
             keys=8192, heads=64, top=2048, values=True),
        # a chunk of two longer fp16 prompts, odd sizes, no score values wanted
        dict(name="index_chunk_odd", kind="index", dtype="fp16", weights="fp16", batch=2, queries=509, keys=6007,
             heads=64, top=2048, values=False),
        # one decode step of the indexer: 64 sequences of 4K to 32K tokens in a paged cache
        dict(name="index_decode", kind="index_paged", dtype="bf16", weights="fp32", queries=1, heads=64,
             top=2048, page=64, kv=_text(_spread(64, 4096, 32768, 1))),
        # attention of a 4K prompt, all 128 heads on this GPU, statistics kept for the backward
        dict(name="attend_prompt_4k", kind="attend", dtype="bf16", heads=128, dim=512, top=2048, lse=True,
             batch=1, queries=4096, keys=4096, lengths=""),
        # packed ragged fp16 prompts with half the heads (two-way tensor parallel)
        dict(name="attend_packed_h64", kind="attend", dtype="fp16", heads=64, dim=512, top=2048, lse=False,
             batch=3, queries=0, keys=0, lengths="217,1500,2309"),
        # one decode step of the attention: 64 sequences, all heads, pages of 128 tokens
        dict(name="attend_decode", kind="attend_paged", dtype="bf16", heads=128, dim=512, top=2048, lse=False,
             queries=1, page=128, kv=_text(_spread(64, 4096, 32768, 2))),
        # decode with eight-way tensor parallel (16 heads here), some sequences shorter than top
        dict(name="attend_decode_h16", kind="attend_paged", dtype="bf16", heads=16, dim=512, top=2048, lse=False,
             queries=1, page=64, kv=_text(_spread(24, 700, 50000, 3))),
        # a prefill step of four packed prompts, indexer into attention
        dict(name="prefill_packed", kind="prefill", dtype="bf16", index_heads=64, heads=128, top=2048,
             lengths="1024,3000,6000,8192"),
        # backward of the attention over a training step's query block
        dict(name="attend_grad", kind="attend_grad", dtype="bf16", heads=64, dim=512, top=2048, queries=512,
             keys=4096),
        # the indexer's sparse training signal at the same block
        dict(name="index_loss", kind="index_loss", dtype="bf16", weights="bf16", heads=64, dim=512,
             index_heads=64, top=2048, queries=512, keys=4096),
        # the indexer's dense warm-up: statistics, then loss and gradients
        dict(name="dense_loss", kind="dense_loss", dtype="fp16", weights="fp16", heads=64, dim=128,
             index_heads=64, queries=512, keys=4096),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["index", "index_paged", "attend", "attend_paged", "prefill", "attend_grad", "index_loss",
                       "dense_loss"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    weights = rng.choice(["fp32", dtype])
    c = dict(kind=kind, dtype=dtype)
    if kind == "index":
        queries = _log(rng, 64, 8192)
        keys = min(16384, queries + rng.choice([0, _log(rng, 1, 12000)]))
        c.update(weights=weights, batch=1 if queries > 2048 else rng.randint(1, 4), queries=queries, keys=keys,
                 heads=rng.choice([8, 16, 32, 64, 64]), top=rng.choice([64, 512, 1024, 2048, 2048]),
                 values=rng.random() < 0.5)
    elif kind == "index_paged":
        n, high = _log(rng, 1, 64), _log(rng, 2000, 120000)
        c.update(weights=weights, queries=rng.choice([1, 1, 2, 3]), heads=rng.choice([32, 64, 64]),
                 top=rng.choice([1024, 2048, 2048]), page=rng.choice([16, 64, 128]),
                 kv=_text(_spread(n, max(8, high // 20), min(high, 1200000 // n), rng.randrange(1 << 20))))
    elif kind == "attend":
        c.update(heads=rng.choice([16, 32, 64, 128, 128]), dim=rng.choice([512, 512, 512, 256, 128]),
                 top=rng.choice([512, 1024, 2048, 2048]), lse=rng.random() < 0.5)
        if rng.random() < 0.5:
            n = rng.randint(1, 5)
            c.update(batch=n, queries=0, keys=0, lengths=_text([_log(rng, 20, 4096 // n) for _ in range(n)]))
        else:
            queries = _log(rng, 16, 3000)
            c.update(batch=1, queries=queries, keys=queries + _log(rng, 1, 9000), lengths="")
    elif kind == "attend_paged":
        n, high = _log(rng, 1, 96), _log(rng, 500, 120000)
        c.update(heads=rng.choice([16, 32, 64, 128, 128]), dim=512, top=rng.choice([1024, 2048, 2048]),
                 lse=False, queries=rng.choice([1, 1, 2, 3]), page=rng.choice([16, 64, 128]),
                 kv=_text(_spread(n, max(8, high // 20), min(high, 1200000 // n), rng.randrange(1 << 20))))
    elif kind == "prefill":
        n = rng.randint(1, 6)
        c.update(index_heads=rng.choice([32, 64]), heads=rng.choice([64, 128]), top=rng.choice([1024, 2048, 2048]),
                 lengths=_text([_log(rng, 100, 12000 // n) for _ in range(n)]))
    else:
        queries = _log(rng, 16, 512)
        c.update(queries=queries, keys=queries + _log(rng, 200, 4096 - 512))
        if kind == "attend_grad":
            c.update(heads=rng.choice([16, 32, 64, 128]), dim=rng.choice([512, 512, 256, 128]),
                     top=rng.choice([512, 1024, 2048]))
        elif kind == "index_loss":
            c.update(weights=weights, heads=rng.choice([32, 64, 128]), dim=512, index_heads=rng.choice([32, 64]),
                     top=rng.choice([512, 1024, 2048]))
        else:
            c.update(weights=weights, heads=rng.choice([32, 64]), dim=128, index_heads=rng.choice([32, 64]))
    return c


# ---- sequences of a case: query and key counts, causal against the end of the keys

def _sequences(case):
    kind = case["kind"]
    if kind in ("index_paged", "attend_paged"):
        return [(case["queries"], n) for n in _numbers(case["kv"])]
    if case.get("lengths"):
        return [(n, n) for n in _numbers(case["lengths"])]
    return [(case["queries"], case["keys"])] * case.get("batch", 1)


def _visible(case):
    """Visible keys of every query row, all sequences in turn (int64 tensor on the host)."""
    return torch.cat([torch.clamp(torch.arange(q) + (k - q + 1), 0, k) for q, k in _sequences(case)])


# ---- inputs

class _Maker:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, shape, dtype, scale=1.0):
        x = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return (x * scale if scale != 1.0 else x).to(dtype)

    def selection(self, visible, top):
        """Per row min(visible, top) distinct positions below visible, in no order, -1 behind them."""
        visible = visible.to("cuda")
        most = max(int(visible.max()), top)
        out = torch.empty((visible.numel(), top), dtype=torch.int32, device="cuda")
        step = max(1, (1 << 26) // most)
        position = torch.arange(most, device="cuda")
        for r in range(0, visible.numel(), step):
            v = visible[r:r + step, None]
            key = torch.rand((v.shape[0], most), generator=self.g, device="cuda")
            key = torch.where(position[None] < v, key, 2.0)
            got = torch.topk(key, top, dim=1, largest=False).indices
            out[r:r + step] = torch.where(got < v, got, -1).to(torch.int32)
        return out

    def pages(self, lengths, page):
        """A block table over a pool that holds every sequence's pages, scattered."""
        need = [(n + page - 1) // page for n in lengths]
        order = torch.randperm(sum(need), generator=self.g, device="cuda").to(torch.int32)
        table = torch.full((len(need), max(need)), -1, dtype=torch.int32, device="cuda")
        at = 0
        for b, n in enumerate(need):
            table[b, :n] = order[at:at + n]
            at += n
        return table, sum(need)


def _inputs(case, seed):
    m, kind, dt = _Maker(seed), case["kind"], DTYPES[case["dtype"]]
    wdt = DTYPES[case.get("weights", "fp32")]
    seqs = _sequences(case)
    rows = sum(q for q, _ in seqs)
    i = {}
    if kind == "index":
        b, s1, s2, n = case["batch"], case["queries"], case["keys"], case["heads"]
        i.update(query=m.normal((b, s1, n, 128), dt), key=m.normal((b, s2, 1, 128), dt),
                 weights=m.normal((b, s1, n), wdt, n ** -0.5))
    elif kind == "index_paged":
        b, n = len(seqs), case["heads"]
        i["table"], pool = m.pages([k for _, k in seqs], case["page"])
        i.update(query=m.normal((b, case["queries"], n, 128), dt), key=m.normal((pool, case["page"], 1, 128), dt),
                 weights=m.normal((b, case["queries"], n), wdt, n ** -0.5))
    elif kind in ("attend", "attend_paged"):
        n, d = case["heads"], case["dim"]
        packed = bool(case.get("lengths"))
        lead = (rows,) if packed else (len(seqs), seqs[0][0])
        if kind == "attend_paged":
            i["table"], pool = m.pages([k for _, k in seqs], case["page"])
            keys = (pool, case["page"])
        else:
            keys = (rows,) if packed else (len(seqs), seqs[0][1])
        i.update(query=m.normal(lead + (n, d), dt), query_rope=m.normal(lead + (n, ROPE), dt),
                 key=m.normal(keys + (1, d), dt), key_rope=m.normal(keys + (1, ROPE), dt),
                 indices=m.selection(_visible(case), case["top"]).reshape(lead + (1, case["top"])))
    elif kind == "prefill":
        n, ni = case["heads"], case["index_heads"]
        i.update(index_query=m.normal((rows, ni, 128), dt), index_key=m.normal((rows, 1, 128), dt),
                 index_weights=m.normal((rows, ni), torch.float32, ni ** -0.5),
                 query=m.normal((rows, n, 512), dt), key=m.normal((rows, 1, 512), dt),
                 query_rope=m.normal((rows, n, ROPE), dt), key_rope=m.normal((rows, 1, ROPE), dt))
    else:
        n, d, s1, s2 = case["heads"], case["dim"], case["queries"], case["keys"]
        n2 = n if kind == "dense_loss" else 1
        i.update(query=m.normal((1, s1, n, d), dt), query_rope=m.normal((1, s1, n, ROPE), dt),
                 key=m.normal((1, s2, n2, d), dt), key_rope=m.normal((1, s2, n2, ROPE), dt))
        if kind != "dense_loss":
            i["indices"] = m.selection(_visible(case), case["top"]).reshape(1, s1, 1, case["top"])
        if kind == "attend_grad":
            i["d_out"] = m.normal((1, s1, n, d), dt)
        else:
            ni = case["index_heads"]
            i.update(query_index=m.normal((1, s1, ni, 128), dt), key_index=m.normal((1, s2, 1, 128), dt),
                     weights=m.normal((1, s1, ni), wdt, ni ** -0.5))
        # what the forward left: its output and its softmax statistics
        if kind == "dense_loss":
            i["maximum"], i["total"] = _dense_statistics(case, i)
        else:
            out, maximum, total = _attention(case, i, i["indices"].reshape(s1, -1), torch.float32)
            i.update(out=out.to(dt).reshape(1, s1, n, d), maximum=maximum.reshape(1, 1, s1, n),
                     total=total.reshape(1, 1, s1, n))
    return i


def _scale(case):
    return 1.0 / math.sqrt(case.get("dim", 512) + ROPE)


def prepare(case, seed):
    i = _inputs(case, seed)
    state = {"case": case, "inputs": i}
    seqs = _sequences(case)
    if case["kind"] == "index_paged":
        state["plan"] = IndexerPlan(i["query"], i["key"], i["weights"], None, [k for _, k in seqs], i["table"], "BSND",
                                    "PA_BSND", case["top"], 3, False)
    elif case["kind"] == "attend_paged":
        state["plan"] = AttentionPlan(i["query"], i["key"], i["key"], i["indices"], _scale(case), i["table"], None,
                                      [k for _, k in seqs], i["query_rope"], i["key_rope"], layout_query="BSND",
                                      layout_kv="PA_BSND", sparse_mode=3, return_softmax_lse=case["lse"],
                                      block_size=case["page"])
    elif case.get("lengths"):
        state["ends"] = torch.cumsum(torch.tensor([q for q, _ in seqs]), 0).tolist()
    return state


def run(state):
    case, i = state["case"], state["inputs"]
    kind = case["kind"]
    if kind == "index":
        return dsa.lightning_indexer(i["query"], i["key"], i["weights"], sparse_count=case["top"], sparse_mode=3,
                                     return_value=case["values"])
    if kind in ("index_paged", "attend_paged"):
        return state["plan"].run()
    if kind == "attend":
        layout = "TND" if case["lengths"] else "BSND"
        ends = state.get("ends")
        return dsa.sparse_flash_attention(i["query"], i["key"], i["key"], i["indices"], _scale(case),
                                          actual_seq_lengths_query=ends, actual_seq_lengths_kv=ends,
                                          query_rope=i["query_rope"], key_rope=i["key_rope"], layout_query=layout,
                                          layout_kv=layout, sparse_mode=3, return_softmax_lse=case["lse"])
    if kind == "prefill":
        return dsa.dsa_prefill(i["index_query"], i["index_key"], i["index_weights"], i["query"], i["key"],
                               i["query_rope"], i["key_rope"], state["ends"], sparse_count=case["top"],
                               scale_value=_scale(case), return_softmax_lse=True)
    if kind == "attend_grad":
        return dsa.sparse_flash_attention_grad(i["query"], i["key"], i["key"], i["indices"], i["d_out"], i["out"],
                                               i["maximum"], i["total"], _scale(case), i["query_rope"],
                                               i["key_rope"])
    if kind == "index_loss":
        return dsa.sparse_lightning_indexer_grad_kl_loss(
            i["query"], i["key"], i["query_index"], i["key_index"], i["weights"], i["indices"], i["maximum"],
            i["total"], i["query_rope"], i["key_rope"], scale_value=_scale(case))
    maximum, total = dsa.dense_lightning_indexer_softmax_lse(i["query_index"], i["key_index"], i["weights"])
    return (maximum, total) + tuple(dsa.dense_loss_backward(
        i["query"], i["key"], i["query_index"], i["key_index"], i["weights"], i["maximum"], i["total"], maximum,
        total, _scale(case), i["query_rope"], i["key_rope"]))


# ---- what a pass cannot do without

def _size(case, name="dtype"):
    return 4 if case.get(name) == "fp32" else 2


def work(case):
    kind, seqs = case["kind"], _sequences(case)
    visible = _visible(case)
    rows, pairs = visible.numel(), int(visible.sum())
    picked = int(torch.clamp(visible, max=case["top"]).sum()) if "top" in case else pairs
    keys = sum(k for _, k in seqs)
    if kind in ("index", "index_paged"):
        n = case["heads"]
        out = rows * case["top"] * (6 if case.get("values") else 4)
        return {"bytes": rows * n * (256 + _size(case, "weights")) + keys * 256 + out, "flops": 2.0 * pairs * n * 128}
    if kind in ("attend", "attend_paged"):
        n, d = case["heads"], case["dim"]
        read = min(picked, keys) if kind == "attend" else sum(min(k, case["top"] * q) for q, k in seqs)
        stats = rows * n * 8 if case["lse"] else 0
        return {"bytes": rows * n * (2 * d + ROPE) * 2 + read * (d + ROPE) * 2 + picked * 4 + stats,
                "flops": 2.0 * picked * n * (2 * d + ROPE)}
    if kind == "prefill":
        n, ni = case["heads"], case["index_heads"]
        return {"bytes": rows * (ni * 260 + n * ((2 * 512 + ROPE) * 2 + 8) + case["top"] * 4) + keys * (256 + 1152),
                "flops": 2.0 * pairs * ni * 128 + 2.0 * picked * n * (2 * 512 + ROPE)}
    n, d = case["heads"], case["dim"]
    head = d + ROPE
    if kind == "attend_grad":
        # query, d_out, out in and the query's gradient out; keys in and their gradients out
        return {"bytes": rows * n * (4 * d + 2 * ROPE) * 2 + rows * n * 8 + keys * (3 * d + 2 * ROPE) * 2 + picked * 4,
                "flops": 2.0 * picked * n * (3 * head + 2 * d)}
    ni = case["index_heads"]
    index = rows * ni * (512 + 2 * _size(case, "weights")) + keys * 512
    if kind == "index_loss":
        return {"bytes": rows * n * (head * 2 + 8) + keys * head * 2 + picked * 4 + index,
                "flops": 2.0 * picked * (n * head + 3 * ni * 128)}
    return {"bytes": (rows + keys) * n * head * 2 + rows * n * 8 + index,
            "flops": 2.0 * pairs * (n * head + 3 * ni * 128)}


def tolerance(case):
    # about four times the distance from exact(): the rounding of the 16-bit outputs and, within them, of the
    # 16-bit probabilities. Positions: a score that rounds the other way moves those of its ties.
    kind, bf16 = case["kind"], case["dtype"] == "bf16"
    if kind in ("index", "index_paged"):
        return {"rel": 2e-3, "max": 0.02, "differ": 1e-3}
    most = {"rel": 9e-3, "max": 0.15} if bf16 else {"rel": 1.2e-3, "max": 0.015}
    return dict(most, differ=1e-3) if kind == "prefill" else most


# ---- the same calls in 64 bits

def _key_rows(case, i, name):
    """[keys, width] of every sequence in turn, in 64 bits, paged caches laid out by sequence."""
    x = i[name]
    if "table" in i:
        page = case["page"]
        flat = x.reshape(-1, x.shape[-1])
        parts = []
        for b, (_, k) in enumerate(_sequences(case)):
            t = torch.arange(k, device="cuda")
            parts.append(flat[i["table"][b, t // page].long() * page + t % page])
        x = torch.cat(parts)
    return x.reshape(-1, x.shape[-1]).double()


def _starts(case):
    """The first key of each row's sequence among the keys of all sequences."""
    at, got = 0, []
    for q, k in _sequences(case):
        got.append(torch.full((q,), at))
        at += k
    return torch.cat(got).to("cuda")


def _scores(q, k, w):
    """Indexer scores [rows, keys] of one sequence in 64 bits."""
    out = torch.empty((q.shape[0], k.shape[0]), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 28) // (q.shape[1] * k.shape[0]))
    kt = k.t().contiguous()
    for r in range(0, q.shape[0], step):
        part = q[r:r + step].double()
        dots = (part.reshape(-1, part.shape[-1]) @ kt).reshape(part.shape[0], part.shape[1], -1)
        out[r:r + step] = (dots.relu_() * w[r:r + step, :, None].double()).sum(1)
    return out


def _top(case, query, key, weights, dtype):
    """(positions, scores) of every row's first `top`, by 16-bit score, equal ones by position."""
    visible = _visible(case).to("cuda")
    at = row = 0
    places, values = [], []
    for q, k in _sequences(case):
        s = _scores(query[row:row + q], key[at:at + k], weights[row:row + q])
        hidden = torch.arange(k, device="cuda")[None] >= visible[row:row + q, None]
        s.masked_fill_(hidden, -math.inf)
        top = min(case["top"], k)
        pick = torch.sort(s.to(dtype).float(), dim=1, descending=True, stable=True).indices[:, :top]
        got = torch.gather(s, 1, pick)
        none = torch.isinf(got)
        pad = (0, case["top"] - top)
        places.append(torch.nn.functional.pad(pick.masked_fill(none, -1), pad, value=-1))
        values.append(torch.nn.functional.pad(got.masked_fill(none, 0.0), pad))
        at, row = at + k, row + q
    return torch.cat(places), torch.cat(values)


def _gathered(case, i, indices, dtype):
    """Yields (rows, key rows, selected, gathered [rows, top, dim + rope]) a block of rows at a time."""
    n_rows, top = indices.shape
    starts = _starts(case)
    k = torch.cat([_key_rows(case, i, "key"), _key_rows(case, i, "key_rope")], 1).to(dtype)
    step = max(1, (1 << 30) // (top * k.shape[1] * k.element_size()))
    for r in range(0, n_rows, step):
        part = indices[r:r + step].long()
        there = part >= 0
        place = part.clamp(min=0) + starts[r:r + step, None]
        yield slice(r, min(r + step, n_rows)), place, there, k[place]


def _attention(case, i, indices, dtype):
    """(out, maximum, total) of the selected tokens, rows of all sequences in turn."""
    n, d = i["query"].shape[-2:]
    q = torch.cat([i["query"].reshape(-1, n, d), i["query_rope"].reshape(-1, n, ROPE)], 2)
    out = torch.empty((q.shape[0], n, d), dtype=dtype, device="cuda")
    maximum = torch.empty((q.shape[0], n), dtype=dtype, device="cuda")
    total = torch.empty_like(maximum)
    for rows, _, there, k in _gathered(case, i, indices, dtype):
        s = torch.bmm(q[rows].to(dtype), k.transpose(1, 2).contiguous()) * _scale(case)
        s.masked_fill_(~there[:, None, :], -math.inf)
        top = s.amax(2)
        s.sub_(top[:, :, None]).exp_()
        maximum[rows], total[rows] = top, s.sum(2)
        out[rows] = torch.bmm(s, k[:, :, :d].contiguous()) / total[rows][:, :, None]
    return out, maximum, total


def _dense_statistics(case, i):
    """(maximum, total) [1, heads, queries, 1] of the attention over every visible key."""
    q = torch.cat([i["query"], i["query_rope"]], 3)[0].transpose(0, 1).float().contiguous()
    k = torch.cat([i["key"], i["key_rope"]], 3)[0].permute(1, 2, 0).float().contiguous()
    s = torch.bmm(q, k) * _scale(case)
    hidden = torch.arange(s.shape[2], device="cuda")[None] >= _visible(case).to("cuda")[:, None]
    s.masked_fill_(hidden[None], -math.inf)
    top = s.amax(2)
    return top[None, :, :, None].contiguous(), s.sub_(top[:, :, None]).exp_().sum(2)[None, :, :, None].contiguous()


def _loss_row(teacher, scores, dots, key, query, weights, maximum, total):
    """One row's loss and gradients: (loss, d_weights, d_query, d_key rows)."""
    student = torch.exp(scores - maximum) / total
    change = student - teacher
    p, s = teacher.clamp(min=1e-8), student.clamp(min=1e-8)
    flow = change[None] * weights[:, None] * (dots > 0)
    return (p * (p.log() - s.log())).sum(), dots @ change, flow @ key, flow.t() @ query


def _exact_grad(case, i):
    n, d, dt = case["heads"], case["dim"], torch.float64
    rows = case["queries"]
    q = torch.cat([i["query"], i["query_rope"]], 3)[0].to(dt)
    do, out = i["d_out"][0].to(dt), i["out"][0].to(dt)
    maximum, total = i["maximum"].reshape(rows, n).to(dt), i["total"].reshape(rows, n).to(dt)
    dq = torch.zeros_like(q)
    dk = torch.zeros((case["keys"], d + ROPE), dtype=dt, device="cuda")
    dv = torch.zeros((case["keys"], d), dtype=dt, device="cuda")
    for r, place, there, k in _gathered(case, i, i["indices"].reshape(rows, -1), dt):
        value = k[:, :, :d].contiguous()
        p = torch.bmm(q[r], k.transpose(1, 2).contiguous()) * _scale(case)
        p = torch.exp(p - maximum[r][:, :, None]) / total[r][:, :, None] * there[:, None, :]
        ds = torch.bmm(do[r], value.transpose(1, 2).contiguous()) - (do[r] * out[r]).sum(2)[:, :, None]
        ds = ds * p * _scale(case)
        dq[r] = torch.bmm(ds, k)
        at = place.reshape(-1)
        dk.index_add_(0, at, torch.bmm(ds.transpose(1, 2).contiguous(), q[r]).reshape(-1, d + ROPE))
        dv.index_add_(0, at, torch.bmm(p.transpose(1, 2).contiguous(), do[r]).reshape(-1, d))
    shape = (1, case["keys"], 1)
    return (dq[None, :, :, :d], dk[:, :d].reshape(shape + (d,)), dv.reshape(shape + (d,)), dq[None, :, :, d:],
            dk[:, d:].reshape(shape + (ROPE,)))


def _exact_loss(case, i):
    """Both losses: the sparse one over the selected keys, the dense one over every visible key."""
    dt, dense = torch.float64, case["kind"] == "dense_loss"
    rows, n = case["queries"], case["heads"]
    visible = _visible(case)
    q = torch.cat([i["query"], i["query_rope"]], 3)[0].to(dt)
    k = torch.cat([i["key"], i["key_rope"]], 3)[0].to(dt).transpose(0, 1).contiguous()   # [key heads, keys, width]
    maximum, total = (i[x].reshape(n, rows).t() if dense else i[x].reshape(rows, n) for x in ("maximum", "total"))
    qi, ki, w = i["query_index"][0].to(dt), i["key_index"][0, :, 0].to(dt), i["weights"][0].to(dt)
    tops, sums = torch.empty(rows, dtype=dt, device="cuda"), torch.empty(rows, dtype=dt, device="cuda")
    dqi, dki, dw = torch.zeros_like(qi), torch.zeros_like(ki), torch.zeros_like(w)
    loss = torch.zeros(1, dtype=dt, device="cuda")
    for r in range(rows):
        if dense:
            pick = torch.arange(int(visible[r]), device="cuda")
            s = torch.bmm(k[:, :pick.numel()], q[r][:, :, None])[:, :, 0] * _scale(case)
        else:
            pick = i["indices"][0, r, 0, :min(int(visible[r]), case["top"])].long()
            s = q[r] @ k[0, pick].t() * _scale(case)
        teacher = (torch.exp(s - maximum[r].to(dt)[:, None]) / (total[r].to(dt)[:, None] + 1e-8)).sum(0) / n
        key = ki[pick]
        dots = (qi[r] @ key.t()).relu()
        scores = w[r] @ dots
        tops[r], sums[r] = scores.max(), torch.exp(scores - scores.max()).sum()
        one, dw[r], dqi[r], part = _loss_row(teacher, scores, dots, key, qi[r], w[r], tops[r],
                                             sums[r] + (0.0 if dense else 1e-8))
        loss += one
        dki.index_add_(0, pick, part)
    got = (dqi[None], dki[None, :, None], dw[None], loss)
    return (tops.reshape(1, 1, -1), sums.reshape(1, 1, -1)) + got if dense else got


def exact(case, seed):
    """What run(prepare(case, seed)) returns, in 64 bits; None where an output is whole numbers."""
    i, kind = _inputs(case, seed), case["kind"]
    dt = DTYPES[case["dtype"]]
    if kind in ("index", "index_paged"):
        n = case["heads"]
        _, values = _top(case, i["query"].reshape(-1, n, 128), _key_rows(case, i, "key"),
                         i["weights"].reshape(-1, n), dt)
        lead = i["query"].shape[:2]
        return None, (values if case.get("values") else torch.zeros_like(values)).reshape(lead + (1, case["top"]))
    if kind == "attend_grad":
        return _exact_grad(case, i)
    if kind in ("index_loss", "dense_loss"):
        return _exact_loss(case, i)
    if kind == "prefill":
        indices, _ = _top(case, i["index_query"], _key_rows(case, i, "index_key"), i["index_weights"], dt)
    else:
        indices = i["indices"].reshape(-1, case["top"])
    out, maximum, total = _attention(case, i, indices, torch.float64)
    packed = bool(case.get("lengths"))
    b = 1 if packed else len(_sequences(case))
    shape = (1, out.shape[0], out.shape[1]) if packed else (b, 1, out.shape[0] // b, out.shape[1])
    maximum, total = maximum.reshape(shape), total.reshape(shape)
    if kind != "prefill" and not case["lse"]:
        maximum, total = torch.zeros_like(maximum), torch.zeros_like(total)
    got = (out.reshape(i["query"].shape), maximum, total)
    return (None,) + got if kind == "prefill" else got
