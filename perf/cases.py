"""Workloads that stand for this framework's use, for timing it.

Every case goes through a public entry point of ``vecattention_amd`` on
seeded inputs made on the GPU: N(0, 1) queries, keys and values with the
vertical (column) structure of ``vecattention_amd.synth`` (sink keys and 2%
random keys along a per-head direction, queries along it, frame locality in
the video cases).  Kinds:

- ``decode``: one generated token's attention over a KV cache,
  ``single_decode_with_kv_cache``.
- ``prefill``: one layer's ``VecAttention_prefill``: causal GQA of a
  vision-language model, or non-causal self-attention of a video DiT.
- ``span``: the dispatcher on a prompt of text, vision tokens and text
  (``customize_prefill_attention`` with a vision span).
- ``full``: dense attention, ``Full_prefill`` (the 'full' metric).
- ``tuner``: the threshold tuner's recall / sparsity evaluation,
  ``seg_pr_perHead``, on fp32 copies of 16-bit queries and keys.
"""
import math

import torch

from vecattention_amd import (FastPrefillConfig, Full_prefill, VecAttention_prefill,
                              customize_prefill_attention, seg_pr_perHead,
                              single_decode_with_kv_cache)

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# Tile settings in use: the models' configuration defaults, the wider groups
# of the long-context configurations, the function signature's own defaults,
# and the video models' one group per row.  `keep` is the share of the
# selectable keys that these inputs keep at the threshold (for work()).
TILES = {
    "model": {"qps": 64, "bk": 16, "group": 1, "chunk": 8192, "threshold": 0.9, "keep": 0.137},
    "vlm": {"qps": 64, "bk": 16, "group": 16, "chunk": 32768, "threshold": 0.7551, "keep": 0.10},
    "long": {"qps": 64, "bk": 16, "group": 16, "chunk": 32768, "threshold": 0.8385, "keep": 0.05},
    "signature": {"qps": 128, "bk": 128, "group": 1, "chunk": 16384, "threshold": 0.9,
                  "keep": 0.017},
    "wan": {"qps": 64, "bk": 16, "group": 8192, "chunk": 32768, "threshold": 0.4248,
            "keep": 0.15},
    "hunyuan": {"qps": 64, "bk": 16, "group": 8192, "chunk": 32768, "threshold": 0.4277,
                "keep": 0.10},
    "fp32": {"qps": 64, "bk": 16, "group": 16, "chunk": 32768, "threshold": 0.6897,
             "keep": 0.10},
}


def listed():
    return [
        # The next token of a chat of two thousand tokens: the smallest call.
        {"name": "decode-2081", "kind": "decode", "S": 2081, "Hq": 28, "Hk": 4, "D": 128,
         "dtype": "bf16", "layout": "NHD"},
        # The next token after a 128K prompt: the cache's bytes count.
        {"name": "decode-131072", "kind": "decode", "S": 131072, "Hq": 28, "Hk": 4, "D": 128,
         "dtype": "bf16", "layout": "NHD"},
        # A short image prompt at the models' default tiles, on the projections' (B, S, H, D)
        # memory as the patched forwards hand it over; a ragged length.
        {"name": "vlm-2333", "kind": "prefill", "tiles": "model", "S": 2333, "Hq": 28, "Hk": 4,
         "D": 128, "dtype": "bf16", "causal": True, "bshd": True, "heads": False},
        # A 32K video prompt.
        {"name": "vlm-32768", "kind": "prefill", "tiles": "vlm", "S": 32768, "Hq": 28, "Hk": 4,
         "D": 128, "dtype": "bf16", "causal": True, "bshd": False, "heads": False},
        # A 128K video prompt: the headline workload.
        {"name": "vlm-131072", "kind": "prefill", "tiles": "long", "S": 131072, "Hq": 28, "Hk": 4,
         "D": 128, "dtype": "bf16", "causal": True, "bshd": False, "heads": False},
        # A program that leaves every option of VecAttention_prefill at its default; fp16, odd
        # length.
        {"name": "signature-16411", "kind": "prefill", "tiles": "signature", "S": 16411, "Hq": 28,
         "Hk": 4, "D": 128, "dtype": "fp16", "causal": True, "bshd": False, "heads": False},
        # One layer of a video DiT, 21 frames of 1560 tokens, tuned per-head thresholds.
        {"name": "dit-32760", "kind": "prefill", "tiles": "wan", "S": 32760, "Hq": 12, "Hk": 12,
         "D": 128, "dtype": "bf16", "causal": False, "bshd": False, "heads": True, "frame": 1560,
         "text": 0},
        # One layer of a larger video DiT, 33 frames of 3600 tokens and 256 text tokens: the
        # largest call.
        {"name": "dit-119056", "kind": "prefill", "tiles": "hunyuan", "S": 119056, "Hq": 24,
         "Hk": 24, "D": 128, "dtype": "bf16", "causal": False, "bshd": False, "heads": False,
         "frame": 3600, "text": 256},
        # fp32 queries, keys and values, head_dim 64.
        {"name": "fp32-4096", "kind": "prefill", "tiles": "fp32", "S": 4096, "Hq": 4, "Hk": 4,
         "D": 64, "dtype": "fp32", "causal": False, "bshd": False, "heads": False},
        # A chat prompt with a system text, one video and a question, through the dispatcher.
        {"name": "span-9001", "kind": "span", "tiles": "model", "S": 9001, "Hq": 28, "Hk": 4,
         "D": 128, "dtype": "bf16", "vs": 41, "ve": 8233},
        # Dense causal prefill, the 'full' metric.
        {"name": "full-16384", "kind": "full", "S": 16384, "Hq": 28, "Hk": 4, "D": 128,
         "dtype": "bf16", "causal": True},
        # One evaluation of the threshold tuner on a video DiT's dumped queries and keys.
        {"name": "tuner-32760", "kind": "tuner", "tiles": "wan", "S": 32760, "Hq": 12, "D": 128,
         "causal": False, "frame": 1560},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "vlm", "vlm", "vlm", "signature", "dit", "dit", "fp32",
                       "span", "full", "tuner"])
    dt = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    Hq, Hk = rng.choice([(28, 4), (28, 4), (32, 8), (16, 16), (12, 2)])
    if kind == "decode":
        return {"kind": "decode", "S": _log(rng, 128, 131072), "Hq": Hq, "Hk": Hk,
                "D": rng.choice([64, 128, 128]), "dtype": dt,
                "layout": rng.choice(["NHD", "NHD", "HND"])}
    if kind == "vlm":
        return {"kind": "prefill", "tiles": rng.choice(["model", "vlm", "long"]),
                "S": _log(rng, 400, 100000), "Hq": Hq, "Hk": Hk, "D": rng.choice([64, 128, 128]),
                "dtype": dt, "causal": True, "bshd": rng.random() < 0.5,
                "heads": rng.random() < 0.25}
    if kind == "signature":
        return {"kind": "prefill", "tiles": "signature", "S": _log(rng, 500, 50000), "Hq": Hq,
                "Hk": Hk, "D": rng.choice([64, 128]), "dtype": dt, "causal": True,
                "bshd": rng.random() < 0.5, "heads": False}
    if kind == "dit":
        frame, text, H, tiles = rng.choice([(1560, 0, 12, "wan"), (1350, 0, 16, "wan"),
                                            (3600, 256, 24, "hunyuan")])
        return {"kind": "prefill", "tiles": tiles, "S": frame * rng.randint(3, 25) + text, "Hq": H,
                "Hk": H, "D": 128, "dtype": "bf16", "causal": False, "bshd": rng.random() < 0.5,
                "heads": rng.random() < 0.5, "frame": frame, "text": text}
    if kind == "fp32":
        return {"kind": "prefill", "tiles": "fp32", "S": _log(rng, 500, 12000),
                "Hq": rng.choice([4, 8, 12]), "Hk": 4, "D": rng.choice([64, 128]),
                "dtype": "fp32", "causal": rng.random() < 0.5, "bshd": False, "heads": False}
    if kind == "span":
        vision, after = _log(rng, 500, 30000), _log(rng, 20, 2000)
        vs = rng.randint(10, 200)
        return {"kind": "span", "tiles": "model", "S": vs + vision + after, "Hq": Hq, "Hk": Hk,
                "D": 128, "dtype": dt, "vs": vs, "ve": vs + vision}
    if kind == "full":
        return {"kind": "full", "S": _log(rng, 300, 30000), "Hq": Hq, "Hk": Hk,
                "D": rng.choice([64, 128, 128]), "dtype": dt, "causal": rng.random() < 0.7}
    if rng.random() < 0.5:
        return {"kind": "tuner", "tiles": "wan", "S": 1560 * rng.randint(3, 21), "Hq": 12,
                "D": 128, "causal": False, "frame": 1560}
    return {"kind": "tuner", "tiles": "vlm", "S": _log(rng, 2000, 30000), "Hq": 28, "D": 128,
            "causal": True, "frame": 0}


def _inputs(case, seed):
    """q, k, v as (B, H, S, D) with B = 1 (decode: one query row)."""
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    g = torch.Generator(dev).manual_seed(seed)
    Hq, Hk, S, D = case["Hq"], case.get("Hk", case["Hq"]), case["S"], case["D"]
    Sq = 1 if case["kind"] == "decode" else S
    dtype = DTYPES[case.get("dtype", "bf16")]

    def rand(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    def unit(x):
        return x / x.norm(dim=-1, keepdim=True)

    u = unit(rand(Hk, D))
    q, k = rand(1, Hq, Sq, D), rand(1, Hk, S, D)
    text = case.get("text", 0)
    sinks = torch.arange(S - text, S, device=dev) if text else torch.arange(min(64, S), device=dev)
    for h in range(Hk):
        rnd = torch.randperm(S, generator=g, device=dev)[:round(0.02 * S)]
        k[:, h, torch.unique(torch.cat([sinks, rnd]))] += 4.0 * u[h]
    q += 1.5 * u.repeat_interleave(Hq // Hk, 0)[None, :, None]
    frame = case.get("frame", 0)
    if frame:
        for lo in range(0, S, frame):
            w = unit(rand(Hk, D))
            k[:, :, lo:lo + frame] += w[None, :, None]
            q[:, :, lo:lo + frame] += w.repeat_interleave(Hq // Hk, 0)[None, :, None]
    q, k = q.to(dtype), k.to(dtype)
    v = rand(1, Hk, S, D).to(dtype)
    if case.get("bshd"):  # (B, H, S, D) views of the projections' (B, S, H, D) memory
        q, k, v = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v))
    return q, k, v


def _threshold(case, dev):
    """The tiles' threshold, or one per head around it, as a tuner leaves them."""
    th = TILES[case["tiles"]]["threshold"]
    if not (case.get("heads") or case["kind"] == "tuner"):
        return th
    H = case["Hq"]
    step = torch.linspace(-1, 1, H, dtype=torch.float64)
    return (th + 0.05 * (1 - th) * step).to(dtype=torch.float32, device=dev)


class _Layer:
    layer_idx = 0


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    st = {"case": dict(case), "q": q, "k": k, "v": v}
    kind = case["kind"]
    if kind == "decode":
        st["q"] = q[0, :, 0].contiguous()
        perm = (1, 0, 2) if case["layout"] == "NHD" else (0, 1, 2)
        st["k"], st["v"] = (x[0].permute(*perm).contiguous() for x in (k, v))
    elif kind == "prefill":
        st["threshold"] = _threshold(case, q.device)
    elif kind == "span":
        t = TILES[case["tiles"]]
        st["layer"] = _Layer()
        st["config"] = FastPrefillConfig(
            metric="vecattention", threshold=t["threshold"], block_size_q=t["qps"],
            block_size_k=t["bk"], group_k_block=t["group"], chunk_size=t["chunk"],
            vision_start_position=case["vs"], vision_end_position=case["ve"], output_time=False)
    elif kind == "tuner":
        st["threshold"] = _threshold(case, q.device)
        st["q"], st["k"], st["v"] = q.float(), k.float(), None
    return st


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    kind = case["kind"]
    if kind == "decode":
        return single_decode_with_kv_cache(q, k, v, kv_layout=case["layout"])
    if kind == "span":
        return customize_prefill_attention(state["layer"], q, k, v, causal=True,
                                           config=state["config"])
    if kind == "full":
        return Full_prefill(q, k, v, causal=case["causal"])
    t = TILES[case["tiles"]]
    if kind == "tuner":
        return seg_pr_perHead(q, k, block_size_q=t["qps"], block_size_k=t["bk"],
                              group_size_k=t["group"], threshold=state["threshold"],
                              causal=case["causal"])
    if case["tiles"] == "signature":
        return VecAttention_prefill(q, k, v, threshold=state["threshold"], causal=case["causal"])
    return VecAttention_prefill(q, k, v, threshold=state["threshold"], q_pooling_size=t["qps"],
                                k_local_size=t["bk"], group_k_block=t["group"],
                                causal=case["causal"], chunk_size=t["chunk"])


def _pairs(S, causal, qps, keep):
    """(attended (row, key) pairs, scored (pooled row, key) pairs) of one head."""
    nqb = math.ceil(S / qps)
    if not causal:
        return keep * S * S, nqb * S
    scored = qps * nqb * (nqb - 1) / 2
    return qps * keep * scored + 1.5 * qps * S, scored


def work(case):
    Hq, Hk, S, D = case["Hq"], case.get("Hk", case["Hq"]), case["S"], case["D"]
    es = 4 if case.get("dtype") == "fp32" else 2
    kind = case["kind"]
    if kind == "decode":
        return {"bytes": es * D * (2 * Hk * S + 2 * Hq), "flops": 4 * D * Hq * S}
    causal = case.get("causal", True)
    dense = S * (S + 1) / 2 if causal else S * S
    if kind == "full":
        return {"bytes": es * D * S * (2 * Hq + 2 * Hk), "flops": 4 * D * Hq * dense}
    t = TILES[case["tiles"]]
    attended, scored = _pairs(S if kind != "span" else case["ve"], causal, t["qps"], t["keep"])
    if kind == "tuner":  # scores only: dense and selected rows, and the selection's
        return {"bytes": 4 * D * S * (Hq + Hk) + 8 * Hq,
                "flops": 2 * D * Hq * (dense + attended + scored)}
    flops = D * Hq * (4 * attended + 2 * scored)
    if kind == "span":
        after = S - case["ve"]
        flops += 4 * D * Hq * (after * (S - after / 2) + case["vs"] ** 2 / 2)
    return {"bytes": es * D * S * (2 * Hq + 2 * Hk), "flops": flops}


def tolerance(case):
    # 16-bit results: the probabilities and the output are rounded to the
    # type.  fp32: sums of fp32 products.  tuner: fp32 sums per row.
    # About four times the measured error against 64 bits (bf16 2.2e-3, fp16
    # 2.8e-4, fp32 4e-7, tuner 1e-7).
    if case["kind"] == "tuner":
        return {"rel": 2e-6}
    return {"rel": {"bf16": 1e-2, "fp16": 1.2e-3, "fp32": 2e-6}[case["dtype"]]}


# ---- the results in 64 bits --------------------------------------------------


def _keep_mask(q, k, gap, t, causal, chunk):
    """(nqb, Sk) bool of one head: the keys each query block keeps.

    q (S, D), k (Sk, D).  Blocks of queries are averaged (the mean and its
    scaling rounded to the inputs' type), scored against the keys, and a key is
    kept when its score + gap reaches the running maximum over its group's
    tiles up to its own.
    """
    S, D = q.shape
    Sk, qps, bk = k.shape[0], t["qps"], t["bk"]
    nqb = math.ceil(S / qps)
    pad = nqb * qps - S
    sums = torch.nn.functional.pad(q.double(), (0, 0, 0, pad)).view(nqb, qps, D).sum(1).float()
    rows = torch.full((nqb, 1), float(qps), device=q.device)
    if pad:
        rows[-1] = qps - pad
    pooled = (sums / rows).to(q.dtype)
    pooled = (pooled.float() * torch.tensor(1 / math.sqrt(D), dtype=torch.float32,
                                            device=q.device)).to(q.dtype)
    s = (pooled.double() @ k.double().T).float()
    first = qps if causal else 0
    s[:, :first] = -math.inf
    ntile = math.ceil(Sk / bk)
    tiles = torch.nn.functional.pad(s, (0, ntile * bk - Sk), value=-math.inf).view(nqb, ntile, bk)
    group = min(t["group"], ntile)
    ngroup = math.ceil(ntile / group)
    m = torch.nn.functional.pad(tiles.amax(-1), (0, ngroup * group - ntile), value=-math.inf)
    m = m.view(nqb, ngroup, group).cummax(-1).values.view(nqb, -1)[:, :ntile]
    kept = (tiles + gap >= m[..., None]).view(nqb, -1)[:, :Sk]
    if causal:
        J = torch.arange(nqb, device=q.device)
        # the first query block of each run of 64 rejects the tiles that begin
        # past the previous block's start
        head = (J % (chunk // qps)) % 64 == 0
        begin = torch.arange(Sk, device=q.device) // bk * bk
        limit = torch.where(head, (J - 1) * qps + 1, J * qps)
        kept = kept & (begin[None] < limit[:, None]) & (begin[None] >= first)
    return kept


def _local_mask(nqb, Sk, qps, causal, dev):
    if not causal:
        return torch.zeros(nqb, Sk, dtype=torch.bool, device=dev)
    J, c = torch.arange(nqb, device=dev)[:, None], torch.arange(Sk, device=dev)[None]
    return ((J >= 1) & (c < qps)) | ((c >= J * qps) & (c < (J + 1) * qps))


def _attend(q, k, v, blocks, qps, causal, rows=2048, masses=False):
    """Attention of one head over the keys of `blocks` (nqb, Sk) (None: all);
    causal rows aligned with the last key.  masses: instead of the output, the
    share of each row's dense softmax that the kept keys hold."""
    S, D = q.shape
    Sk = k.shape[0]
    kd = k.double()
    vd = None if masses else v.double()
    out = []
    for lo in range(0, S, rows):
        hi = min(lo + rows, S)
        n = min(Sk, hi + Sk - S) if causal else Sk
        s = (q[lo:hi].double() @ kd[:n].T).mul_(1 / math.sqrt(D))
        pos = torch.arange(lo, hi, device=q.device)
        if causal:
            s.masked_fill_(torch.arange(n, device=q.device)[None] > (pos + Sk - S)[:, None],
                           -math.inf)
        if masses:
            p = torch.softmax(s, -1)
            out.append((p * blocks[pos // qps, :n]).sum(-1))
            continue
        if blocks is not None:
            s.masked_fill_(~blocks[pos // qps, :n], -math.inf)
        none = torch.isinf(s).all(-1)
        out.append((torch.softmax(s, -1) @ vd[:n]).masked_fill_(none[:, None], 0.0))
    return torch.cat(out)


def _sparse(q, k, v, threshold, t, causal):
    # a tensor threshold takes its 1e-9 in its own type
    th = (threshold + 1e-9).double() if isinstance(threshold, torch.Tensor) else threshold + 1e-9
    outs = []
    for h in range(q.shape[0]):
        hk = h // (q.shape[0] // k.shape[0])
        gap = -math.log(float(th[h]) if isinstance(th, torch.Tensor) else th)
        gap = torch.tensor(gap, dtype=torch.float32, device=q.device)
        kept = _keep_mask(q[h], k[hk], gap, t, causal, t["chunk"])
        kept |= _local_mask(*kept.shape, t["qps"], causal, q.device)
        outs.append(_attend(q[h], k[hk], v[hk], kept, t["qps"], causal))
    return torch.stack(outs)


def _dense(q, k, v, causal):
    rep = q.shape[0] // k.shape[0]
    return torch.stack([_attend(q[h], k[h // rep], v[h // rep], None, 64, causal)
                        for h in range(q.shape[0])])


def exact(case, seed):
    S, Hq, kind = case["S"], case["Hq"], case["kind"]
    if kind != "decode" and Hq * S * S > 8e10:
        return None  # over about 20 seconds in 64 bits
    q, k, v = (x[0] for x in _inputs(case, seed))
    if kind == "decode":
        return _dense(q, k, v, False)[:, 0]
    if kind == "full":
        return _dense(q, k, v, case["causal"])[None]
    t = TILES[case["tiles"]]
    if kind == "prefill":
        return _sparse(q, k, v, _threshold(case, q.device), t, case["causal"])[None]
    if kind == "span":
        vs, ve = case["vs"], case["ve"]
        head = _dense(q[:, :vs], k[:, :vs], v[:, :vs], True)
        body = _sparse(q[:, :ve], k[:, :ve], v[:, :ve], t["threshold"], t, True)[:, vs:]
        tail = _dense(q[:, ve:], k, v, True)
        return torch.cat([head, body, tail], 1)[None]
    th, causal, qps = _threshold(case, q.device).double(), case["causal"], t["qps"]
    recall, sparsity = [], []
    nqb = math.ceil(S / qps)
    seen = torch.arange(1, S + 1, device=q.device).double() if causal else torch.full(
        (S,), float(S), device=q.device, dtype=torch.float64)
    for h in range(Hq):
        gap = torch.tensor(-math.log(float(th[h])), dtype=torch.float32, device=q.device)
        kept = _keep_mask(q[h].float(), k[h].float(), gap, t, causal, 8192)
        local = _local_mask(nqb, S, qps, causal, q.device)
        size = (kept.sum(-1) + local.sum(-1)).double().repeat_interleave(qps)[:S]
        recall.append(_attend(q[h], k[h], None, kept | local, qps, causal, masses=True).mean())
        sparsity.append(1 - (size / seen).mean())
    return torch.stack(recall), torch.stack(sparsity)
