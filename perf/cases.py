"""Performance cases of the sparse shared-KV attention operator.

Each case is one layer's call as a serving or training program makes it, through
the package's public entry points: ``sparse_attn_sharedkv`` (with the plan that
``sparse_attn_sharedkv_metadata`` built for the step), a replay of a captured call
(``SasGraph``), the metadata op and the call together (the first layer of a step),
and a launch with its backward (``build_launch``, ``run``, ``backward``).  The cases span the calls' real range: a two-sequence
window decode that is all latency, decode batches of ragged lengths, MTP decode
at 128k context, chunked and whole prefills, packed training batches; 16 heads (a
tensor-parallel shard) to 128; d_qk 512 and 576; bf16, fp16 and fp8 e4m3 KV; the window
alone, every compressed row (ratio 128) and per-token top-k rows (ratio 4).

Fields of a case:

* ``kind``: ``layer`` (one call, the plan kept), ``graph`` (a replay of the captured
  call), ``step`` (the metadata op, then the call), ``train`` (the call and the
  gradients of the queries, the KV pools and the sinks).
* ``B`` sequences of ``kv_lo`` .. ``kv_hi`` KV tokens (log-uniform), each with
  ``q_lo`` .. ``q_hi`` query tokens at its end (0: the whole sequence), drawn from
  ``shape_seed``; ``layout`` TND or BSND (one query length).
* ``H`` heads, ``D`` = d_qk, ``scenario`` 1 window, 2 window and every compressed row, 3
  window and top-k ``K``; ``ratio``, ``page``, ``q_dtype``, ``kv_dtype``.
"""

from __future__ import annotations

import math
import random

import torch

from dsv4_planb_amd import sparse_attn_sharedkv, sparse_attn_sharedkv_metadata
from dsv4_planb_amd.api import build_launch
from dsv4_planb_amd.graph import SasGraph

D_V = 512
WINDOW = 128
CUS = 256
MOST_FLOPS, MOST_BYTES = 2.6e12, 2.3e9  # of a drawn case: prefill8k_h128's
_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp8": torch.float8_e4m3fn}


def _case(kind, B, kv_lo, kv_hi, q_lo, q_hi, H, D, scenario, K, ratio, page, q_dtype, kv_dtype,
          layout="TND", shape_seed=0, **extra):
    return dict(kind=kind, B=B, kv_lo=kv_lo, kv_hi=kv_hi, q_lo=q_lo, q_hi=q_hi, H=H, D=D,
                scenario=scenario, K=K, ratio=ratio, page=page, q_dtype=q_dtype, kv_dtype=kv_dtype,
                layout=layout, shape_seed=shape_seed, **extra)


def listed():
    return [
        # The smallest call: a window-only layer of two sequences on a shard of 16 heads.
        dict(name="decode_window_h16",
             **_case("layer", 2, 1024, 1024, 1, 1, 16, 576, 1, 0, 4, 64, "bf16", "bf16")),
        # A decode layer of an ordinary batch: 32 sequences of 4k to 32k tokens, 64 heads,
        # called eagerly from Python.
        dict(name="decode32_h64",
             **_case("layer", 32, 4096, 32768, 1, 1, 64, 576, 3, 512, 4, 64, "bf16", "bf16", shape_seed=2)),
        # The same layer replayed from a graph, as a decode loop with captured steps runs it.
        dict(name="decode32_h64_graph",
             **_case("graph", 32, 4096, 32768, 1, 1, 64, 576, 3, 512, 4, 64, "bf16", "bf16", shape_seed=2)),
        # The first layer of an eager decode step on a tensor-parallel shard (16 heads,
        # fp16): the step's plan is built, then the layer runs.
        dict(name="decode_step_h16_fp16",
             **_case("step", 48, 1000, 60000, 1, 3, 16, 576, 3, 1024, 4, 64, "fp16", "fp16", shape_seed=3)),
        # Long-context decode with one draft token per sequence (MTP), all 128 heads.
        dict(name="decode128k_h128_mtp",
             **_case("layer", 128, 131072, 131072, 2, 2, 128, 576, 3, 2048, 4, 64, "bf16", "bf16")),
        # A mixed serving batch over an fp8 cache: lengths from 256 to 128k, 1 to 4 query
        # tokens each.
        dict(name="decode_ragged_fp8_h128",
             **_case("layer", 64, 256, 131072, 1, 4, 128, 576, 3, 2048, 4, 64, "bf16", "fp8", shape_seed=5)),
        # Prefill of one 8k prompt, all 128 heads, top-k 2048 (the largest forward).
        dict(name="prefill8k_h128",
             **_case("layer", 1, 8192, 8192, 0, 0, 128, 576, 3, 2048, 4, 64, "bf16", "bf16")),
        # Prefill of packed prompts by a 64-head model's top-k 512 layer.
        dict(name="prefill_packed_h64",
             **_case("layer", 3, 900, 5000, 0, 0, 64, 576, 3, 512, 4, 64, "bf16", "bf16", shape_seed=6)),
        # Prefill of an 8k prompt by a window-only layer: 64 heads, d 512, pages of 128, fp16.
        dict(name="prefill_window8k_h64_fp16",
             **_case("layer", 1, 8192, 8192, 0, 0, 64, 512, 1, 0, 4, 128, "fp16", "fp16")),
        # A chunk of four long prompts in a fixed-shape batch (BSND), a ratio-128 layer that
        # attends every compressed row, over an fp8 cache.
        dict(name="prefill_chunk_cfa_h64_fp8",
             **_case("layer", 4, 9000, 30000, 509, 509, 64, 512, 2, 0, 128, 128, "bf16", "fp8",
                     layout="BSND", shape_seed=8)),
        # A training layer: packed documents, all 128 heads, top-k 512, every gradient.
        dict(name="train_packed_h128",
             **_case("train", 4, 500, 2048, 0, 0, 128, 576, 3, 512, 4, 64, "bf16", "bf16", shape_seed=9)),
        # A window-only training layer of a 64-head model in fp16 at d 512.
        dict(name="train_window_h64_fp16",
             **_case("train", 2, 700, 1500, 0, 0, 64, 512, 1, 0, 4, 64, "fp16", "fp16", shape_seed=10)),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above."""
    while True:
        kind = rng.choice(["layer", "layer", "layer", "layer", "graph", "step", "train", "train"])
        train = kind == "train"
        prefill = train or (kind == "layer" and rng.random() < 0.5)
        q_dtype = rng.choice(["bf16", "bf16", "fp16"])
        kv_dtype = "fp8" if not train and rng.random() < 0.3 else q_dtype
        scenario = rng.choice([1, 2, 3, 3, 3])
        c = _case(kind, 1, 1, 1, 1, 1, rng.choice([16, 32, 64, 64, 100, 128, 128]),
                  rng.choice([512, 576, 576]), scenario,
                  _log_int(rng, 64, 2048) if scenario == 3 else 0,
                  128 if scenario == 2 else 4, rng.choice([64, 128]), q_dtype, kv_dtype,
                  shape_seed=rng.randrange(1 << 30))
        if not prefill:
            c.update(B=_log_int(rng, 1, 128), kv_lo=_log_int(rng, 200, 8000), q_lo=1,
                     q_hi=rng.choice([1, 1, 2, 4]))
            c["kv_hi"] = _log_int(rng, c["kv_lo"], 131072)
        else:
            c.update(B=_log_int(rng, 1, 6), kv_lo=_log_int(rng, 200, 1200))
            c["kv_hi"] = _log_int(rng, c["kv_lo"], 2500 if train else 9000)
            chunk = not train and rng.random() < 0.4
            c["q_lo"] = c["q_hi"] = _log_int(rng, 100, c["kv_lo"]) if chunk else 0
            if chunk and rng.random() < 0.5:
                c["layout"] = "BSND"
        w = work(c)
        if w["flops"] <= MOST_FLOPS * (0.25 if train else 1.0) and w["bytes"] <= MOST_BYTES:
            return c


# ---------------------------------------------------------------------------
# shapes
# ---------------------------------------------------------------------------
def _lengths(case):
    """(KV lengths, query lengths) of the sequences."""
    rng = random.Random(case["shape_seed"])
    kv = [_log_int(rng, case["kv_lo"], case["kv_hi"]) for _ in range(case["B"])]
    q = [rng.randint(case["q_lo"], case["q_hi"]) if case["q_hi"] else n for n in kv]
    return kv, [min(a, b) for a, b in zip(q, kv)]


def _rows(case, kv, q):
    """Per sequence: (window rows, compressed rows) attended by all its query tokens,
    and the distinct ones (expected, for random top-k lists)."""
    win = cmp = 0
    missed = 1.0  # the share of compressed rows that no token lists
    for s in range(q):
        sg = kv - q + s
        win += min(sg + 1, WINDOW)
        thr = (sg + 1) // case["ratio"] if case["scenario"] >= 2 else 0
        n = min(thr, case["K"]) if case["scenario"] == 3 else thr
        cmp += n
        if thr:
            missed *= 1.0 - n / thr
    distinct = (kv // case["ratio"]) * (1.0 - missed) if case["scenario"] >= 2 else 0.0
    return win, cmp, min(kv, q + WINDOW - 1), distinct


def work(case):
    kv, q = _lengths(case)
    H, D = case["H"], case["D"]
    T = sum(q)
    pairs = uniq = 0
    for a, b in zip(kv, q):
        w, c, uw, uc = _rows(case, a, b)
        pairs += w + c
        uniq += uw + uc
    row = D + 4 if case["kv_dtype"] == "fp8" else 2 * D
    idx = 4 * case["K"] * T
    nbytes = T * H * (2 * D + 2 * D_V + 4) + uniq * row + idx
    flops = 2 * pairs * H * (D + D_V)
    if case["kind"] == "train":
        # again q, the rows and the indices, and out, its gradient and the LSE; the
        # gradients of q and of the rows (K and V in one row)
        nbytes += T * H * (2 * D + 4 * D_V + 4) + uniq * row + idx + T * H * 2 * D + uniq * row
        flops += 2 * pairs * H * (3 * D + 2 * D_V)
    return {"bytes": int(nbytes), "flops": int(flops)}


def tolerance(case):
    """About four times the errors against 64 bits of a call with P and dS rounded to the
    query dtype (measured: relative 2.2e-3 in bf16 and 2.9e-4 in fp16; largest 3.3e-2 and
    3.2e-3 for outputs, 8.5e-2 and 7.1e-3 for gradients)."""
    if case["q_dtype"] == "bf16":
        return {"rel": 9e-3, "max": 0.35 if case["kind"] == "train" else 0.13}
    return {"rel": 1.2e-3, "max": 0.03 if case["kind"] == "train" else 0.013}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _pool(rows, D, page, kv_dtype, gen):
    """A paged pool of N(0, 1) rows; fp8: e4m3 codes and a scale per row (its largest
    element at 448)."""
    n = max(1, rows)
    if kv_dtype != "fp8":
        return torch.randn((n, page, 1, D), dtype=_DTYPES[kv_dtype], device="cuda", generator=gen), None
    x = torch.randn((n, page, 1, D), dtype=torch.float32, device="cuda", generator=gen)
    scale = x.abs().amax(dim=-1).clamp(min=1e-12) / 448.0
    return (x / scale[..., None]).to(torch.float8_e4m3fn), scale.contiguous()


def _table(pages, gen):
    """Every sequence's pages, a random permutation of the pool; -1 where unused."""
    B, width = len(pages), max(1, max(pages))
    perm = torch.randperm(max(1, sum(pages)), device="cuda", generator=gen).to(torch.int32)
    table = torch.full((B, width), -1, dtype=torch.int32, device="cuda")
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = perm[at:at + n]
        at += n
    return table


def _top_k(thr, K, gen):
    """Per token: min(K, thr) distinct compressed rows below thr in random order, -1 padded."""
    out = torch.full((thr.numel(), K), -1, dtype=torch.int32, device="cuda")
    space = max(1, int(thr.max()))
    col = torch.arange(space, device="cuda")
    for t0 in range(0, thr.numel(), 1024):
        th = thr[t0:t0 + 1024, None]
        keys = torch.rand((th.shape[0], space), generator=gen, device="cuda")
        keys.masked_fill_(col >= th, 2.0)
        pick = keys.argsort(dim=1)[:, :K].to(torch.int32)
        n = pick.shape[1]
        out[t0:t0 + 1024, :n] = torch.where(col[:n] < th, pick, -1)
    return out


def _inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kv, q_lens = _lengths(case)
    B, H, D, page, K = case["B"], case["H"], case["D"], case["page"], case["K"]
    T = sum(q_lens)
    cu = torch.tensor([0] + q_lens).cumsum(0).to(torch.int32)
    seqused = torch.tensor(kv, dtype=torch.int32, device="cuda")
    batch = torch.repeat_interleave(torch.arange(B), torch.tensor(q_lens)).cuda()
    pos = torch.arange(T, device="cuda") - cu.cuda()[batch] + (
        seqused - torch.tensor(q_lens, device="cuda"))[batch]  # the token's place in its sequence
    thr = (pos + 1) // case["ratio"] if case["scenario"] >= 2 else torch.zeros_like(pos)
    pages = [-(-n // page) for n in kv]
    ori, ori_scale = _pool(sum(pages), D, page, case["kv_dtype"], gen)
    x = dict(T=T, cu_host=cu, cu=cu.cuda(), q_prefix=cu[:-1].cuda(), seqused=seqused,
             act_q=torch.tensor(q_lens, dtype=torch.int32, device="cuda"), batch=batch, pos=pos, thr=thr,
             q=torch.randn((T, H, D), dtype=_DTYPES[case["q_dtype"]], device="cuda", generator=gen),
             sinks=torch.rand(H, device="cuda", generator=gen) * 2 - 1,
             ori=ori, ori_scale=ori_scale, ori_table=_table(pages, gen),
             cmp=None, cmp_scale=None, cmp_table=None, idx=None, max_q=max(q_lens), max_kv=max(kv))
    if case["scenario"] >= 2:
        cpages = [-(-(n // case["ratio"]) // page) for n in kv]
        x["cmp"], x["cmp_scale"] = _pool(sum(cpages), D, page, case["kv_dtype"], gen)
        x["cmp_table"] = _table(cpages, gen)
    if case["scenario"] == 3:
        x["idx"] = _top_k(thr, K, gen)
    if case["kind"] == "train":
        x["dout"] = torch.randn((T, H, D_V), dtype=_DTYPES[case["q_dtype"]], device="cuda", generator=gen)
    return x


def _metadata(case, x):
    kw = dict(num_heads_q=case["H"], num_heads_kv=1, head_dim=case["D"], seqused_kv=x["seqused"],
              batch_size=case["B"], max_seqlen_q=x["max_q"], max_seqlen_kv=x["max_kv"],
              layout_q=case["layout"], has_cmp_kv=case["scenario"] >= 2, aic_core_num=CUS)
    if case["layout"] == "TND":
        kw["cu_seqlens_q"] = x["cu_host"]
    if case["scenario"] >= 2:
        kw["cmp_ratio"] = case["ratio"]
    if case["scenario"] == 3:
        kw["cmp_topk"] = case["K"]
    return sparse_attn_sharedkv_metadata(**kw)


def _launch(case, x, metadata):
    return build_launch(
        q_flat=x["q"], ori_kv=x["ori"], ori_block_table=x["ori_table"], cmp_kv=x["cmp"],
        cmp_block_table=x["cmp_table"], cmp_indices=x["idx"], q_prefix=x["q_prefix"],
        act_q_lens=x["act_q"], seqused_kv=x["seqused"], sinks=x["sinks"], metadata=metadata,
        scenario=case["scenario"], topk=case["K"], cmp_ratio=case["ratio"],
        ori_win_left=WINDOW - 1, softmax_scale=1.0 / math.sqrt(case["D"]), core_num=CUS,
        ori_kv_scale=x["ori_scale"], cmp_kv_scale=x["cmp_scale"])


def prepare(case, seed):
    x = _inputs(case, seed)
    T, H, D, B, kind = x["T"], case["H"], case["D"], case["B"], case["kind"]
    s = dict(kind=kind, case=case, x=x)
    if kind != "step":
        s["metadata"] = _metadata(case, x)
    if kind == "graph":
        launch, s["out"], s["lse"] = _launch(case, x, s["metadata"])
        launch.run()
        torch.cuda.synchronize()
        s["graph"] = SasGraph(launch)
    if kind in ("graph", "train"):
        return s
    kw = dict(ori_kv=x["ori"], ori_block_table=x["ori_table"], seqused_kv=x["seqused"],
              sinks=x["sinks"], softmax_scale=1.0 / math.sqrt(D), layout_q=case["layout"],
              return_softmax_lse=True, core_num=CUS)
    s["q"] = x["q"]
    if case["layout"] == "TND":
        kw["cu_seqlens_q"] = x["cu"]
    else:
        s["q"] = x["q"].reshape(B, T // B, H, D)
    if case["scenario"] >= 2:
        kw.update(cmp_kv=x["cmp"], cmp_block_table=x["cmp_table"], cmp_ratio=case["ratio"])
    if case["scenario"] == 3:
        kw["cmp_sparse_indices"] = x["idx"].reshape(
            (T, 1, -1) if case["layout"] == "TND" else (B, T // B, 1, case["K"]))
    if case["kv_dtype"] == "fp8":
        kw["ori_kv_scale"] = x["ori_scale"]
        if case["scenario"] >= 2:
            kw["cmp_kv_scale"] = x["cmp_scale"]
    s["kw"] = kw
    return s


def run(s):
    if s["kind"] == "graph":
        s["graph"].replay()
        return s["out"], s["lse"]
    if s["kind"] == "train":
        launch, out, lse = _launch(s["case"], s["x"], s["metadata"])
        launch.run()
        return (out, lse) + launch.backward(s["x"]["dout"], kv_grad=True)
    metadata = _metadata(s["case"], s["x"]) if s["kind"] == "step" else s["metadata"]
    return sparse_attn_sharedkv(s["q"], metadata=metadata, **s["kw"])


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    x = _inputs(case, seed)
    T, H, D, page = x["T"], case["H"], case["D"], case["page"]
    scale = 1.0 / math.sqrt(D)
    train = case["kind"] == "train"
    ori = x["ori"].reshape(-1, D)
    cmp = None if x["cmp"] is None else x["cmp"].reshape(-1, D)

    def pool_row(table, b, p, ok):  # pool rows of places p of sequences b
        blk = torch.where(ok, p // page, 0)
        return table[b[:, None], blk].long() * page + p % page

    def rows(pool, scales, at, ok):
        v = pool[at.reshape(-1)].double().reshape(*at.shape, D)
        if scales is not None:
            v *= scales.reshape(-1)[at].double()[..., None]
        return v * ok[..., None]

    out = torch.empty((T, H, D_V), dtype=torch.float64, device="cuda")
    lse = torch.empty((T, H), dtype=torch.float64, device="cuda")
    if train:
        dq = torch.empty((T, H, D), dtype=torch.float64, device="cuda")
        dsink = torch.zeros(H, dtype=torch.float64, device="cuda")
        dori = torch.zeros(ori.shape, dtype=torch.float64, device="cuda")
        dcmp = None if cmp is None else torch.zeros(cmp.shape, dtype=torch.float64, device="cuda")
    sink = x["sinks"].double()
    chunk = 64
    for t0 in range(0, T, chunk):
        sl = slice(t0, min(T, t0 + chunk))
        b, pos, thr = x["batch"][sl], x["pos"][sl], x["thr"][sl]
        p = pos[:, None] - (WINDOW - 1) + torch.arange(WINDOW, device="cuda")
        wok = p >= 0
        wat = torch.where(wok, pool_row(x["ori_table"], b, p.clamp(min=0), wok), 0)
        kv, ok = rows(ori, x["ori_scale"], wat, wok), wok
        if case["scenario"] >= 2:
            if case["scenario"] == 3:
                ids = x["idx"][sl].long()
            else:
                ids = torch.arange(max(1, int(thr.max())), device="cuda").expand(b.numel(), -1)
            cok = (ids >= 0) & (ids < thr[:, None])
            ids = ids.clamp(min=0)
            cat = torch.where(cok, pool_row(x["cmp_table"], b, ids, cok), 0)
            kv = torch.cat([kv, rows(cmp, x["cmp_scale"], cat, cok)], 1)
            ok = torch.cat([ok, cok], 1)
        q = x["q"][sl].double()
        s = torch.matmul(q, kv.transpose(1, 2).contiguous()) * scale
        s.masked_fill_(~ok[:, None, :], -math.inf)
        full = torch.cat([s, sink[None, :, None].expand(s.shape[0], H, 1)], 2)
        L = torch.logsumexp(full, 2)
        P = torch.exp(s - L[..., None])
        v = kv[..., :D_V].contiguous()
        o = torch.matmul(P, v)
        out[sl], lse[sl] = o, L
        if train:
            g = x["dout"][sl].double()
            delta = (g * o).sum(-1)
            dS = P * (torch.matmul(g, v.transpose(1, 2).contiguous()) - delta[..., None])
            dq[sl] = torch.matmul(dS, kv) * scale
            dsink -= (torch.exp(sink - L) * delta).sum(0)
            dkv = torch.matmul(dS.transpose(1, 2).contiguous(), q) * scale
            dkv[..., :D_V] += torch.matmul(P.transpose(1, 2).contiguous(), g)
            dori.index_add_(0, wat[wok], dkv[:, :WINDOW][wok])
            if dcmp is not None:
                dcmp.index_add_(0, cat[cok], dkv[:, WINDOW:][cok])
    if case["layout"] == "BSND":
        B = case["B"]
        out, lse = out.reshape(B, T // B, H, D_V), lse.reshape(B, T // B, H)
    if not train:
        return out, lse
    return (out, lse, dq, dsink, dori.reshape(x["ori"].shape),
            None if dcmp is None else dcmp.reshape(x["cmp"].shape))
