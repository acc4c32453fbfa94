"""Timed cases of the DSA path, each one pass through a drop-in module's forward.

Four kinds, one per way the path is called:
  attn         Task1 sparse attention with a sink (``task1_sparse_attn.Model``), head dim 128:
               a small shared kv block (n_kv <= 32) or rows gathered from a long one
  mla          sparse MLA of the DSA layer (the same module with v_dim): keys 576, values 512
  indexer      Task2 lightning indexer, 16 heads x 64 (q_lora_rank 256, dim 1024)
  dsa_indexer  the DSA layer's indexer, 64 heads x 128 (q_lora_rank 1536, dim 7168)

Sizes are those of the modules' own ``get_inputs`` builders and of the tests, with decode
steps, prefill chunks and ragged lengths between them. Inputs are drawn on the GPU from the
seed; queries, keys and activations are N(0, 1) in bf16 and weights N(0, 0.02), as in the
benchmark; selected rows are distinct and, in a prefill from position 0, causal.
"""
from __future__ import annotations

import math

import torch

from ascendc_kernel_amd import task1_sparse_attn as t1
from ascendc_kernel_amd import task2_indexer as t2

HEAD_DIM = 128              # Task1
D_QK, D_V = 576, 512        # sparse MLA: key and value channels of a latent row
INDEXERS = {                # kind: q_lora_rank, dim, heads, head dim, RoPE channels
    "indexer": (256, 1024, 16, 64, 32),
    "dsa_indexer": (1536, 7168, 64, 128, 64),
}


def _attn(name, b, m, h, n_kv, topk, causal, idx64):
    return dict(name=name, kind="attn", b=b, m=m, h=h, n_kv=n_kv, topk=topk, causal=causal, idx64=idx64)


def _mla(name, b, m, h, n_kv, topk, causal, idx64):
    return dict(name=name, kind="mla", b=b, m=m, h=h, n_kv=n_kv, topk=topk, causal=causal, idx64=idx64)


def _indexer(name, kind, b, s, start_pos, ratio, topk, offset=0):
    return dict(name=name, kind=kind, b=b, s=s, start_pos=start_pos, ratio=ratio, topk=topk, offset=offset)


def listed():
    return [
        # One short sequence over the smallest kv block: a call of a few microseconds, bound by
        # its launch.
        _attn("attn small", 1, 160, 64, 32, 16, False, False),
        # The same attention over a full batch of sequences: a stream of q in and out.
        _attn("attn full", 8, 2600, 64, 32, 16, False, False),
        # Prefill over a long kv block: every token gathers 512 rows of its past.
        _attn("attn gather prefill", 4, 4096, 64, 8192, 512, True, False),
        # A decode step of eight sequences over the same kv length, fed by the indexer's int64
        # picks: one token each.
        _attn("attn gather decode", 8, 1, 64, 8192, 512, False, True),
        # A prefill chunk with no round size anywhere: 48 heads (a tensor-parallel share), odd
        # token, row and slot counts.
        _attn("attn gather ragged", 3, 421, 48, 1531, 333, False, True),
        # The indexer's prefill over a full batch of sequences (ratio 4, top-128).
        _indexer("indexer prefill", "indexer", 8, 2600, 0, 4, 128),
        # A smaller, ragged prefill: three sequences of odd length, picks shifted by an offset.
        _indexer("indexer ragged", "indexer", 3, 1003, 0, 4, 128, 7),
        # A decode step of eight sequences at the end of the cache.
        _indexer("indexer decode", "indexer", 8, 1, 2599, 4, 128),
        # The DSA layer's indexer over an 8192-token prefill (top-2048 of the causal past).
        _indexer("dsa indexer prefill", "dsa_indexer", 1, 8192, 0, 1, 2048),
        # Its decode step: one new token at position 8191.
        _indexer("dsa indexer decode", "dsa_indexer", 1, 1, 8191, 1, 2048),
        # The DSA layer's attention over the same prefill: the largest call of the framework.
        _mla("mla prefill", 1, 8192, 128, 8192, 2048, True, True),
        # Its decode step: one token over the indexer's int64 picks.
        _mla("mla decode", 1, 1, 128, 8192, 2048, False, True),
    ]


def _log_int(rng, lo, hi):
    """A whole number from lo to hi, spread evenly over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("attn", "attn", "indexer", "indexer", "dsa_indexer", "mla"))
    decode = rng.random() < 0.4
    if kind == "attn":
        h = 16 * rng.randint(1, 8)
        small = rng.random() < 0.35                       # the small kv block, slots drawn with replacement
        n_kv = rng.randint(8, 32) if small else _log_int(rng, 64, 8192)
        topk = _log_int(rng, 4, 96) if small else _log_int(rng, 16, min(1024, n_kv))
        if decode:
            b, m = _log_int(rng, 1, 64), rng.randint(1, 4)
        else:
            b = rng.randint(1, 8)
            # no more work than the listed prefills
            most = min(8 * 2600 * 64 // (b * h), 4 * 4096 * 64 * 512 // (b * h * topk))
            m = _log_int(rng, 16, max(17, min(4096, most)))
        causal = not decode and not small and m <= n_kv and rng.random() < 0.5
        return dict(kind=kind, b=b, m=m, h=h, n_kv=n_kv, topk=topk, causal=causal, idx64=rng.random() < 0.5)
    if kind == "mla":
        h = rng.choice((64, 80, 96, 112, 128))
        n_kv = _log_int(rng, 512, 8192)
        topk = _log_int(rng, 128, min(2048, n_kv))
        if decode:
            b, m = _log_int(rng, 1, 16), rng.randint(1, 4)
        else:
            b, m = 1, _log_int(rng, 64, min(4096, n_kv))
        causal = not decode and rng.random() < 0.5
        return dict(kind=kind, b=b, m=m, h=h, n_kv=n_kv, topk=topk, causal=causal, idx64=rng.random() < 0.5)
    ratio = rng.choice((1, 2, 4))
    if kind == "indexer":
        longest = min(2600, 2048 * ratio)
        topk = _log_int(rng, 16, 256)
    else:
        longest = 8192
        topk = _log_int(rng, 256, 2048)
    if decode:
        b = _log_int(rng, 1, 16 if kind == "indexer" else 8)
        s = rng.randint(1, 2)
        start_pos = _log_int(rng, 4 * ratio * topk if 4 * ratio * topk < longest else longest // 2, longest) - s
    else:
        b = rng.randint(1, 8) if kind == "indexer" else 1
        s = _log_int(rng, 32 * ratio, longest)
        start_pos = 0
    return dict(kind=kind, b=b, s=s, start_pos=start_pos, ratio=ratio, topk=topk, offset=rng.choice((0, 0, 128)))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.bfloat16)


def _slots(g, case):
    """topk_idxs [b, m, topk]: with replacement from a small kv block; else distinct rows in
    random order, of the causally visible [0, t] (further slots -1) or of the whole cache."""
    b, m, n_kv, topk = case["b"], case["m"], case["n_kv"], case["topk"]
    dtype = torch.int64 if case["idx64"] else torch.int32
    if n_kv <= 32:
        return torch.randint(0, n_kv, (b, m, topk), generator=g, device="cuda", dtype=dtype)
    idx = torch.empty(b, m, topk, device="cuda", dtype=dtype)
    cols = torch.arange(n_kv, device="cuda")
    step = max(1, (1 << 24) // (b * n_kv))
    for at in range(0, m, step):
        t = torch.arange(at, min(m, at + step), device="cuda")
        order = torch.rand(b, len(t), n_kv, generator=g, device="cuda")
        if case["causal"]:
            order.masked_fill_(cols > t[:, None], -1.0)
        value, row = order.topk(topk, dim=-1)
        idx[:, at:at + len(t)] = row.masked_fill_(value < 0, -1)
    return idx


def _attention_inputs(case, seed):
    """q, kv, topk_idxs and the sink of an attn or mla case."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    d = D_QK if case["kind"] == "mla" else HEAD_DIM
    q = _randn(g, case["b"], case["m"], case["h"], d)
    kv = _randn(g, case["b"], case["n_kv"], d)
    sink = torch.randn(case["h"], generator=g, device="cuda")
    return q, kv, _slots(g, case), sink


def prepare(case, seed):
    if case["kind"] in ("attn", "mla"):
        q, kv, idx, sink = _attention_inputs(case, seed)
        model = t1.Model(case["h"], q.shape[-1], D_V if case["kind"] == "mla" else None)
        model = model.to("cuda").requires_grad_(False)
        model.attn_sink.copy_(sink)
        return model, (q, kv, idx)
    g = torch.Generator(device="cuda").manual_seed(seed)
    q_lora, dim, heads, head_dim, rope = INDEXERS[case["kind"]]
    b, s, ratio = case["b"], case["s"], case["ratio"]
    end = case["start_pos"] + s
    args = t2.ModelArgs(max_batch_size=b, max_seq_len=end, dim=dim, index_n_heads=heads, index_head_dim=head_dim,
                        index_topk=case["topk"], q_lora_rank=q_lora, rope_head_dim=rope)
    freqs = t2.precompute_freqs_cis(rope, end, device="cuda")
    kv_cache = _randn(g, b, end // ratio, head_dim)
    with torch.device("cuda"):
        model = t2.Model(args, freqs, kv_cache, ratio)
    model = model.requires_grad_(False)
    for w in (model.wq_b.weight, model.weights_proj.weight):
        w.copy_(torch.randn(w.shape, generator=g, device="cuda") * 0.02)
    return model, (_randn(g, b, s, dim), _randn(g, b, s, q_lora), case["start_pos"], case["offset"])


def run(state):
    model, inputs = state
    return model(*inputs)


def _valid_slots(case):
    """Slots of one batch row that hold a kv row."""
    m, topk = case["m"], case["topk"]
    if not case["causal"]:
        return m * topk
    full = max(0, m - topk)                               # tokens with topk visible rows
    part = m - full
    return full * topk + part * (part + 1) // 2


def work(case):
    if case["kind"] in ("attn", "mla"):
        b, m, h = case["b"], case["m"], case["h"]
        dk, dv = (D_QK, D_V) if case["kind"] == "mla" else (HEAD_DIM, HEAD_DIM)
        size = 8 if case["idx64"] else 4
        # q read, out written, each kv row once, the slot list
        nbytes = 2 * b * m * h * (dk + dv) + 2 * b * case["n_kv"] * dk + b * m * case["topk"] * size + 4 * h
        if case["n_kv"] <= 32:
            rows = b * m * min(case["topk"], case["n_kv"])  # slots repeat rows: score each row once
        else:
            rows = b * _valid_slots(case)
            nbytes = min(nbytes, nbytes - 2 * b * case["n_kv"] * dk + 2 * rows * dk)  # few tokens: not every row
        return {"bytes": nbytes, "flops": 2 * rows * h * (dk + dv)}
    q_lora, dim, heads, head_dim, rope = INDEXERS[case["kind"]]
    b, s, ratio = case["b"], case["s"], case["ratio"]
    n_cand = (case["start_pos"] + s) // ratio
    k_out = min(case["topk"], n_cand)
    # x, qr, both weights, keys and the RoPE rows read, int64 picks written
    nbytes = (2 * b * s * (dim + q_lora) + 2 * heads * (head_dim * q_lora + dim) + 2 * b * n_cand * head_dim
              + 4 * s * rope + 8 * b * s * k_out)
    pairs = b * (s * n_cand if case["start_pos"] else sum(min((t + 1) // ratio, n_cand) for t in range(s)))
    flops = 2 * b * s * heads * (head_dim * q_lora + dim) + 2 * pairs * heads * head_dim
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # The indexer returns indices, defined by every rounding of the reference module.
    if case["kind"] in ("indexer", "dsa_indexer"):
        return "exact"
    # bf16 outputs: one rounding (2^-9 at most, 1.7e-3 in the 2-norm) against 64 bits, times four.
    return {"rel": 7e-3, "max": 2e-2}


def exact(case, seed):
    if case["kind"] in ("indexer", "dsa_indexer"):
        return None                                       # indices: no value beyond the 16-bit rounding
    q, kv, idx, sink = _attention_inputs(case, seed)
    b, m, h, d = q.shape
    dv = D_V if case["kind"] == "mla" else d
    topk = idx.shape[-1]
    sink = sink.double().view(1, h, 1)
    out = torch.empty(b, m, h, dv, device="cuda", dtype=torch.float64)
    step = max(1, (1 << 26) // (topk * max(d, h)))
    for i in range(b):
        kvd = kv[i].double()
        for at in range(0, m, step):
            ix = idx[i, at:at + step].long()
            rows = kvd[ix.clamp(min=0)]                   # [t, topk, d]
            scores = torch.bmm(q[i, at:at + step].double(), rows.transpose(1, 2).contiguous()) * d ** -0.5
            scores.masked_fill_((ix < 0).unsqueeze(1), -math.inf)
            top = torch.maximum(scores.amax(-1, keepdim=True), sink)
            p = torch.exp(scores - top)
            p = p / (p.sum(-1, keepdim=True) + torch.exp(sink - top))
            out[i, at:at + step] = torch.bmm(p, rows[..., :dv].contiguous())
    return out
