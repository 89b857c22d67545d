"""Benchmark of the sparse shared-KV attention path on one MI355X.

Workloads (synthetic, seeded; q / KV ~ N(0, 1) bf16, sinks ~ U(-1, 1), page 64,
window 128, compression ratio 4, d_qk 576, d_v 512, scale 1/sqrt(576)):

* ``decode128k`` (default, the figure ``value`` reports): B=128 sequences of
  131072 tokens, 2 query tokens each (MTP), 128 heads, top-k 2048 compressed rows
  per token drawn without replacement from the causally valid ones; block tables
  a random permutation of a shared page pool.  HBM-bound.
* ``prefill8k``: one sequence, 8192 query tokens over 8192 KV, 128 heads, top-k
  2048 over the causally valid compressed rows (-1 padded).  MFMA-bound.
* ``decode32``: B=32, 64 heads, KV lengths U[4096, 32768], top-k 512.
* ``decode128k_fp8``: decode128k with the fp8 e4m3 pools of ``ragged_fp8``.
* ``ragged_fp8``: B=64, KV lengths log-uniform in [256, 131072], 1, 2 or 4 query
  tokens per sequence, 128 heads, top-k 2048 (-1 padded where fewer compressed
  rows are valid); KV pools fp8 e4m3 with a per-row fp32 scale (580 B per row).

A step is one forward call (row resolution, attention, split combine) with the
split-KV plan built beforehand by the metadata op, replayed from a hipGraph.
``value`` is microseconds per call (lower is better), timed over exactly
``--steps`` replays after ``--warmup`` untimed ones.  Before those, each workload
runs ``--settle`` seconds (default 0.25) of back-to-back replays, reported as
``settle``: the GPU clock ramps up over the first milliseconds of load (the first
20 replays from a cold start are reported one by one as ``cold_call_us``), and a
short warmup would otherwise time the ramp.  ``call_dist_us`` / ``attend_dist_us``
give the per-call distribution.  ``roofline`` rates the attention kernel alone:
``--steps`` back-to-back launches on its stream, each dispatch recording its own
start and end into HIP events (``sas_attend_timed``), so ``kernel_us`` is the
kernel's execution time as a kernel trace reports it; ``attend_us`` is the same
launches timed by events around them, dispatch gaps included.  After everything
else, the headline workload runs ``--sustain`` seconds (default 5) of
back-to-back replays and times ``--steps`` replays again, reported as
``sustained``: under the socket's power limit the clock keeps falling over
seconds of load.
``cpu_baseline`` times the C oracle on a bounded sample of the same workload on
the host cores and scales it to the full call.
"""

from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

import numpy as np  # noqa: E402
import torch  # noqa: E402

HBM_PEAK_GBS = 8000.0
MFMA_BF16_PEAK_TFLOPS = 2500.0
D_QK, D_V, PAGE, WIN, RATIO = 576, 512, 64, 128, 4
ROW_BYTES = D_QK * 2
ROW_BYTES_FP8 = D_QK + 4  # e4m3 payload + fp32 scale
KERNEL_NAME = {"decode128k": "sas::attend_kernel<576, bf16>", "prefill8k": "sas::attend_kernel<576, bf16>",
               "decode32": "sas::attend_kernel<576, bf16>",
               "decode128k_fp8": "sas::attend_kernel<576, bf16, fp8 KV>",
               "ragged_fp8": "sas::attend_kernel<576, bf16, fp8 KV>"}
FLOP_PER_ROW_HEAD = 2 * D_QK + 2 * D_V


# ---------------------------------------------------------------------------
# synthetic inputs, built on the GPU
# ---------------------------------------------------------------------------
def _random_subsets(n_tok, thr, K, space, gen, dev):
    """Per token: min(K, thr) distinct ids from [0, thr) in random order, -1 padded."""
    keys = torch.rand((n_tok, space), generator=gen, device=dev)
    col = torch.arange(space, device=dev)[None, :]
    keys = torch.where(col < thr[:, None], keys, torch.full_like(keys, 2.0))
    order = torch.argsort(keys, dim=1)[:, :K].to(torch.int32)
    take = torch.clamp(thr, max=K)
    return torch.where(torch.arange(K, device=dev)[None, :] < take[:, None], order,
                       torch.full_like(order, -1))


def _fp8_pool(n_pages, gen, dev):
    """N(0, 1) rows stored as e4m3 with a per-row fp32 scale (row max -> 448)."""
    x = torch.randn((n_pages, PAGE, 1, D_QK), dtype=torch.float32, device=dev, generator=gen)
    sc = x.abs().amax(dim=-1).clamp(min=1e-12) / 448.0
    return (x / sc[..., None]).to(torch.float8_e4m3fn), sc.contiguous()


def make_workload(name: str, seed: int = 0, dev="cuda", compact: bool = False):
    """Synthetic inputs of one workload.  compact: every sequence's block tables
    point at the first sequence's pages (a KV footprint that fits the 256 MB MALL;
    for locality experiments only, never the benchmark figure)."""
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    fp8 = False
    if name in ("decode128k", "decode128k_fp8"):
        B, q_per, H, ctx, K = 128, 2, 128, 131072, 2048
        kv = [ctx] * B
        q_lens = [q_per] * B
        fp8 = name.endswith("fp8")
    elif name == "prefill8k":
        B, q_per, H, K = 1, 8192, 128, 2048
        kv = [8192]
        q_lens = [q_per]
    elif name == "decode32":
        B, q_per, H, K = 32, 1, 64, 512
        rng = np.random.default_rng(seed)
        kv = rng.integers(4096, 32769, size=B).tolist()
        q_lens = [q_per] * B
    elif name == "ragged_fp8":
        B, H, K = 64, 128, 2048
        rng = np.random.default_rng(seed)
        kv = np.exp(rng.uniform(np.log(256), np.log(131072), size=B)).astype(np.int64).tolist()
        q_lens = rng.choice([1, 2, 4], size=B).tolist()
        q_per = max(q_lens)
        fp8 = True
    else:
        raise ValueError(name)
    T = sum(q_lens)
    pages = [math.ceil(x / PAGE) for x in kv]
    cpages = [math.ceil((x // RATIO) / PAGE) for x in kv]
    ori_scale = cmp_scale = None
    if fp8:
        ori_pool, ori_scale = _fp8_pool(sum(pages), gen, dev)
        cmp_pool, cmp_scale = _fp8_pool(sum(cpages), gen, dev)
    else:
        ori_pool = torch.randn((sum(pages), PAGE, 1, D_QK), dtype=torch.bfloat16, device=dev,
                               generator=gen)
        cmp_pool = torch.randn((sum(cpages), PAGE, 1, D_QK), dtype=torch.bfloat16, device=dev,
                               generator=gen)
    perm = torch.randperm(sum(pages), device=dev, generator=gen).to(torch.int32)
    cperm = torch.randperm(sum(cpages), device=dev, generator=gen).to(torch.int32)
    obt = torch.full((B, max(pages)), -1, dtype=torch.int32, device=dev)
    cbt = torch.full((B, max(cpages)), -1, dtype=torch.int32, device=dev)
    o = c = 0
    for b in range(B):
        obt[b, :pages[b]] = perm[o:o + pages[b]]
        cbt[b, :cpages[b]] = cperm[c:c + cpages[b]]
        o += pages[b]
        c += cpages[b]
    if compact:
        obt[:, :] = obt[0:1, :].clone()
        cbt[:, :] = cbt[0:1, :].clone()
    q = torch.randn((T, H, D_QK), dtype=torch.bfloat16, device=dev, generator=gen)
    sinks = (torch.rand(H, device=dev, generator=gen) * 2 - 1).float()
    qlen = torch.tensor(q_lens, dtype=torch.int32, device=dev)
    cu = torch.zeros(B + 1, dtype=torch.int32, device=dev)
    cu[1:] = torch.cumsum(qlen, 0)
    seqused = torch.tensor(kv, dtype=torch.int32, device=dev)
    b_of = torch.repeat_interleave(torch.arange(B, device=dev), qlen.long())
    s_loc = torch.arange(T, device=dev) - cu[b_of]
    s_g = seqused[b_of] - qlen[b_of] + s_loc
    thr = torch.div(s_g + 1, RATIO, rounding_mode="floor")
    space = int((max(kv) // RATIO))
    idx = _random_subsets(T, thr, K, space, gen, dev).reshape(T, 1, K)
    n_win = (s_g + 1 - torch.clamp(s_g - (WIN - 1), min=0)).clamp(min=0)
    n_cmp = torch.clamp(thr, min=0, max=K)
    # algorithmic work: unique KV rows per sequence, FLOPs per (row, head)
    flat = idx.reshape(T, K).long()
    keyed = torch.where(flat >= 0, b_of[:, None].long() * (space + 1) + flat, torch.full_like(flat, -1))
    distinct = int(torch.unique(keyed[keyed >= 0]).numel())
    win_lo = torch.full((B,), 1 << 40, dtype=torch.long, device=dev).scatter_reduce(
        0, b_of, torch.clamp(s_g - (WIN - 1), min=0).long(), reduce="amin")
    win_hi = torch.full((B,), -1, dtype=torch.long, device=dev).scatter_reduce(
        0, b_of, s_g.long(), reduce="amax")
    uniq = distinct + int((win_hi - win_lo + 1).clamp(min=0).sum().item())
    rows_total = int((n_win + n_cmp).sum().item())
    alg_bytes = (T * H * D_QK * 2 + T * H * D_V * 2 + T * H * 4 + T * K * 4 +
                 uniq * (ROW_BYTES_FP8 if fp8 else ROW_BYTES))
    alg_flops = rows_total * H * FLOP_PER_ROW_HEAD
    return dict(name=name, B=B, T=T, H=H, K=K, q_per=q_per, kv=kv, q=q, ori_kv=ori_pool,
                cmp_kv=cmp_pool, ori_scale=ori_scale, cmp_scale=cmp_scale, ori_bt=obt, cmp_bt=cbt,
                idx=idx, sinks=sinks, cu=cu, seqused=seqused, alg_bytes=alg_bytes,
                alg_flops=alg_flops, uniq_rows=uniq, rows_total=rows_total, fp8=fp8)


def build_call(wl, core_num=256):
    """The metadata op's plan and a launch object for one workload: (plan, launch, out, lse)."""
    from dsv4_planb_amd import metadata as M
    from dsv4_planb_amd.api import build_launch

    cu = wl["cu"]
    plan = M.sparse_attn_sharedkv_metadata(
        num_heads_q=wl["H"], num_heads_kv=1, head_dim=D_QK, cu_seqlens_q=cu,
        seqused_kv=wl["seqused"], batch_size=wl["B"], max_seqlen_q=wl["q_per"],
        max_seqlen_kv=max(wl["kv"]), cmp_topk=wl["K"], cmp_ratio=RATIO, layout_q="TND",
        has_cmp_kv=True, aic_core_num=core_num)
    launch, out, lse = build_launch(
        q_flat=wl["q"], ori_kv=wl["ori_kv"], ori_block_table=wl["ori_bt"], cmp_kv=wl["cmp_kv"],
        cmp_block_table=wl["cmp_bt"], cmp_indices=wl["idx"], q_prefix=cu[:-1],
        act_q_lens=cu[1:] - cu[:-1], seqused_kv=wl["seqused"], sinks=wl["sinks"],
        metadata=plan, scenario=3, topk=wl["K"], cmp_ratio=RATIO, ori_win_left=WIN - 1,
        softmax_scale=1.0 / math.sqrt(D_QK), core_num=core_num, ori_kv_scale=wl["ori_scale"],
        cmp_kv_scale=wl["cmp_scale"])
    return plan, launch, out, lse


# ---------------------------------------------------------------------------
# GPU timing
# ---------------------------------------------------------------------------
def _log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def _events_time(fn, n, stream):
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record(stream)
    for _ in range(n):
        fn()
    end.record(stream)
    end.synchronize()
    return start.elapsed_time(end) * 1000.0 / n  # us per call


def _per_call(fn, n, stream):
    """Each of n calls bracketed by its own events: the per-call distribution (us)."""
    evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
           for _ in range(n)]
    for a, b in evs:
        a.record(stream)
        fn()
        b.record(stream)
    evs[-1][1].synchronize()
    return [a.elapsed_time(b) * 1000.0 for a, b in evs]


RTC_HZ = 100e6  # the GPU's real-time counter (s_memrealtime)


def _dispatch_times(launch, n, stream):
    """n back-to-back attention launches, each dispatch recording its own start and
    end into HIP events and its span on the GPU's real-time counter (earliest
    workgroup start to latest workgroup end, sas_attend_timed): two readings of
    the kernel's execution per launch, in us."""
    evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
           for _ in range(n)]
    stamps = torch.zeros((n, 2), dtype=torch.int64, device=launch.device)
    stamps[:, 0] = -1  # UINT64_MAX for the atomic minimum
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(evs):
        launch.run_attend_timed(a, b, stamps[i])
    torch.cuda.synchronize()
    st = stamps.cpu().numpy().view(np.uint64)
    dev_us = [(int(e) - int(b)) / RTC_HZ * 1e6 for b, e in st]
    return [a.elapsed_time(b) * 1000.0 for a, b in evs], dev_us


def _dist(xs):
    v = np.sort(np.asarray(xs, np.float64))
    return {"n": int(v.size), "min": round(float(v[0]), 2), "p10": round(float(np.percentile(v, 10)), 2),
            "median": round(float(np.median(v)), 2), "p90": round(float(np.percentile(v, 90)), 2),
            "max": round(float(v[-1]), 2)}


def _settle(fn, secs, stream):
    """Back-to-back calls for `secs` seconds (host-synchronised every 32 calls so
    the queue stays short): the GPU's clock and power reach their steady state
    under this load before anything is timed.  Returns the number of calls."""
    n, t0 = 0, time.perf_counter()
    while time.perf_counter() - t0 < secs:
        for _ in range(32):
            fn()
        n += 32
        stream.synchronize()
    return n


def measure(wl, steps, warmup, core_num=256, settle_s=0.25, sustain_s=0.0):
    """Per workload: build the plan and launch, capture the forward call in a
    hipGraph, then (1) the first 20 replays timed one by one from a cold start
    (`cold_call_us`: the clock transient), (2) a settle phase of `settle_s`
    seconds of back-to-back replays, (3) `warmup` untimed replays, (4) the timed
    region: exactly `steps` replays between two events (`call_us`, the
    headline), (5) the per-call distribution of `steps` more replays, (6) the
    attention stage alone after a settle phase of its own: `steps` launches timed
    by their own dispatch events (`attend_kernel_us`, the roofline's kernel time)
    and by events around them (`attend_us`), (7) the other stages, the forward
    call launched eagerly through the C ABI (`eager_call_us`), the full op with
    the device planner captured ahead of the forward (`full_call_us`) and the
    eager API call, (8) with `sustain_s` > 0, last (so that no figure above moves): that
    many seconds of back-to-back replays, then `steps` replays timed again
    (`sustained`).  The socket's power limit keeps lowering the clock over
    seconds of load, so this reads above `call_us`."""
    from dsv4_planb_amd import sparse_attn_sharedkv
    from dsv4_planb_amd.graph import SasGraph

    dev = wl["q"].device
    scale = 1.0 / math.sqrt(D_QK)
    stream = torch.cuda.Stream(device=dev)  # all timed work runs on this stream
    with torch.cuda.stream(stream):
        t0 = time.perf_counter()
        plan, launch, out, lse = build_call(wl, core_num)
        torch.cuda.synchronize()
        plan_host_us = (time.perf_counter() - t0) * 1e6  # metadata op + launch set-up
        cu = wl["cu"]
        launch.run()
        torch.cuda.synchronize()
        graph = SasGraph(launch)
        replay = lambda: graph.replay(stream)  # noqa: E731
        cold = _per_call(replay, 20, stream)
        settle_calls = _settle(replay, settle_s, stream)
        for _ in range(warmup):
            replay()
        torch.cuda.synchronize()
        # the timed region: `steps` full forward calls replayed from the graph
        call_us = _events_time(replay, steps, stream)
        torch.cuda.synchronize()
        call_dist = _dist(_per_call(replay, max(steps, 10), stream))
        # the stages alone (same stream, same inputs).  The attention stage gets a
        # settle phase of its own: back-to-back attention launches draw more power
        # than the graph's, and the clock goes through the same transient again.
        attend = lambda: launch.run("attend")  # noqa: E731
        attend_settle = _settle(attend, settle_s, stream)
        kernel, kernel_dev = _dispatch_times(launch, max(steps, 10), stream)
        attend_kernel_us = float(np.mean(kernel))
        attend_dist = _dist(kernel)
        attend_kernel_dev_us = float(np.mean(kernel_dev))
        attend_us = _events_time(attend, steps, stream)
        resolve_us = _events_time(lambda: launch.run("resolve"), steps, stream)
        combine_us = _events_time(lambda: launch.run("combine"), steps, stream)
        # the same forward call launched eagerly through the C ABI, back to back (the
        # host runs ahead, so this is the device time without hipGraphLaunch's own
        # cost per replay)
        forward = lambda: launch.run("forward")  # noqa: E731
        _settle(forward, settle_s, stream)
        eager_call_us = _events_time(forward, steps, stream)
        # the full op: the device planner captured in the graph too, ahead of the
        # forward (the plan is rebuilt into the workspace on every replay)
        plan_keep, launch.plan = launch.plan, None
        graph_full = SasGraph(launch)
        launch.plan = plan_keep
        full_call_us = _events_time(lambda: graph_full.replay(stream), steps, stream)
        graph_full.close()
        plan_p = launch.params
        from dsv4_planb_amd.metadata import device_plan
        plan_us = _events_time(lambda: device_plan(plan_p, cu[:-1], cu[1:] - cu[:-1], wl["seqused"]),
                               steps, stream)
        # eager API call, host work included
        api_kw = dict(ori_kv=wl["ori_kv"], cmp_kv=wl["cmp_kv"], cmp_sparse_indices=wl["idx"],
                      ori_block_table=wl["ori_bt"], cmp_block_table=wl["cmp_bt"], cu_seqlens_q=cu,
                      seqused_kv=wl["seqused"], sinks=wl["sinks"], metadata=plan,
                      softmax_scale=scale, cmp_ratio=RATIO, topk_cmp=wl["K"],
                      ori_kv_scale=wl["ori_scale"], cmp_kv_scale=wl["cmp_scale"])
        sparse_attn_sharedkv(wl["q"], **api_kw)
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        for _ in range(steps):
            sparse_attn_sharedkv(wl["q"], **api_kw)
        torch.cuda.synchronize()
        eager_us = (time.perf_counter() - t1) * 1e6 / steps
        sustained = None
        if sustain_s > 0:
            n_sus = _settle(replay, sustain_s, stream)
            sustained = {"seconds": sustain_s, "calls": n_sus,
                         "call_us": _events_time(replay, steps, stream)}
        graph.close()
    ok = bool(torch.isfinite(out.float()).all().item())
    return dict(call_us=call_us, eager_call_us=eager_call_us, full_call_us=full_call_us,
                attend_us=attend_us,
                attend_kernel_us=attend_kernel_us, attend_kernel_rtc_us=attend_kernel_dev_us,
                attend_rtc_dist_us=_dist(kernel_dev), resolve_us=resolve_us,
                combine_us=combine_us, plan_us=plan_us, plan_host_us=plan_host_us,
                eager_api_us=eager_us, finite=ok, call_dist_us=call_dist,
                attend_dist_us=attend_dist, cold_call_us=[round(x, 1) for x in cold],
                settle={"seconds": settle_s, "calls": settle_calls,
                        "attend_calls": attend_settle}, sustained=sustained)


# FLOPs per (row, head) of the backward.  Algorithmic (FlashAttention-2's
# backward with P recomputed from the LSE): S = q K^T (2 d_qk), dP = dO V^T
# (2 d_v), dq = dS K (2 d_qk), dK = dS^T q (2 d_qk), dV = P^T dO (2 d_v).  Without
# key tiles (decode-like calls) the kernels run S and dP twice, once for dq and once for
# the pools' gradient; with them the dq kernel hands P and dS on through the workspace.
BWD_FLOP_DQ = 2 * D_QK + 2 * D_V + 2 * D_QK           # dq and dsinks
BWD_FLOP_ALG = BWD_FLOP_DQ + 2 * D_QK + 2 * D_V       # dq, dsinks, dK, dV
BWD_FLOP_EXEC = BWD_FLOP_DQ + 2 * D_QK + 2 * D_V + 2 * D_QK + 2 * D_V


def measure_backward(wl, steps, core_num=256, settle_s=0.25):
    """The backward of one forward call (16-bit KV): `steps` back-to-back calls of
    sas_backward with the plan passed in (resolve, D terms, dq, dsinks), then the
    same with the pools' gradients (adding the dK / dV kernel), each timed by
    events around the calls after a settle phase.  Reports us per call, TFLOP/s of
    the algorithmic FLOPs and the fraction of bf16 MFMA peak."""
    dev = wl["q"].device
    stream = torch.cuda.Stream(device=dev)
    with torch.cuda.stream(stream):
        plan, launch, out, lse = build_call(wl, core_num)
        launch.run()
        gen = torch.Generator(device=dev)
        gen.manual_seed(1)
        dout = torch.randn(out.shape, dtype=out.dtype, device=dev, generator=gen)
        res = {}
        for kv in (False, True):
            bufs = launch.backward_buffers(kv_grad=kv)
            if not kv:
                plain_ws = bufs["ws"].numel()
            tiled = kv and bufs["ws"].numel() > plain_ws
            call = lambda: launch.backward_into(dout, None, bufs)  # noqa: E731
            _settle(call, settle_s, stream)
            us = _events_time(call, steps, stream)
            rows_heads = wl["rows_total"] * wl["H"]
            flop_alg = rows_heads * (BWD_FLOP_ALG if kv else BWD_FLOP_DQ)
            flop_exec = rows_heads * (BWD_FLOP_DQ if not kv else BWD_FLOP_ALG if tiled else BWD_FLOP_EXEC)
            res["dq_dkv" if kv else "dq"] = dict(
                call_us=round(us, 2), alg_flops=flop_alg, exec_flops=flop_exec,
                tflops=round(flop_alg / (us * 1e-6) / 1e12, 2),
                frac_mfma=round(flop_alg / (us * 1e-6) / 1e12 / MFMA_BF16_PEAK_TFLOPS, 4),
                pool_grad_bytes=(0 if not kv else int(sum(
                    b.untyped_storage().nbytes() for b in (bufs["d_ori"], bufs["d_cmp"])
                    if b is not None))))
            del bufs
            torch.cuda.empty_cache()
        res["dkv_us"] = round(res["dq_dkv"]["call_us"] - res["dq"]["call_us"], 2)
        # fp32 atomic adds of the pools' gradient per call: every (token, list row)
        # adds one d_qk-wide row, summed over the heads first (with key tiles: one per
        # tile and token group, whose number is the device's choice)
        res["dkv_atomic_bytes"] = None if tiled else int(wl["rows_total"] * D_QK * 4)
    return res


def _traffic_from_profile(workload):
    """HBM bytes per attention launch measured with rocprofv3 counters, if a
    summary for this workload is committed (profiles/<kernel>_<workload>_pmc.json)."""
    path = os.path.join(ROOT, "profiles", f"sas_attend_{workload}_pmc.json")
    if not os.path.exists(path):
        return None
    try:
        with open(path) as f:
            return float(json.load(f)["hbm_bytes_per_launch"])
    except Exception:  # noqa: BLE001
        return None


# ---------------------------------------------------------------------------
# On-box peaks: what this GPU sustains for the two bounds the roofline uses
# ---------------------------------------------------------------------------
def measure_peaks(dev, secs=2.0):
    """Sustained bf16 MFMA rate (register-only, random operands that change every
    MFMA, one wave per SIMD) and HBM read bandwidth (16-B streaming loads over
    4 GiB), each after `secs` of back-to-back launches so the clock has settled
    under the power limit.  Kernels: dsv4_planb_amd/csrc/sas_probe.hip."""
    import ctypes

    from dsv4_planb_amd.build import PROBE_LIB

    if not os.path.exists(PROBE_LIB):
        raise RuntimeError(f"{PROBE_LIB} missing: run __graft_entry__.build()")
    lib = ctypes.CDLL(PROBE_LIB)
    stream = torch.cuda.current_stream(dev)
    sp = ctypes.c_void_p(stream.cuda_stream)

    def sustained(fn, n_timed):
        t0 = time.perf_counter()
        while time.perf_counter() - t0 < secs:
            fn()
            torch.cuda.synchronize()
        return _events_time(fn, n_timed, stream)

    blocks, iters = 256, 16000  # 1024 waves: one per SIMD
    out = torch.empty(blocks * 256, dtype=torch.float32, device=dev)
    ticks = torch.zeros(blocks * 4, dtype=torch.int64, device=dev)

    def mfma(dep=0):
        rc = lib.sas_probe_mfma(ctypes.c_void_p(out.data_ptr()), ctypes.c_void_p(ticks.data_ptr()),
                                iters, blocks, dep, sp)
        if rc:
            raise RuntimeError(f"sas_probe_mfma: {rc}")

    us = sustained(mfma, 10)
    n_mfma = iters * 8  # per wave
    mfma_tflops = blocks * 4 * n_mfma * 32768 / (us * 1e-6) / 1e12
    clock_ghz = float(ticks.double().mean().item()) / (us * 1e-6) / 1e9
    indep_cycles = float(ticks.double().mean().item()) / n_mfma
    mfma(1)  # one dependent chain per wave: cycles per MFMA when each waits for the last
    torch.cuda.synchronize()
    dep_cycles = float(ticks.double().mean().item()) / n_mfma
    del out, ticks
    nbytes = 4 << 30
    src = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    rblocks = 2048
    rout = torch.empty(rblocks * 256, dtype=torch.int32, device=dev)

    def read():
        rc = lib.sas_probe_read(ctypes.c_void_p(src.data_ptr()), ctypes.c_size_t(nbytes),
                                ctypes.c_void_p(rout.data_ptr()), rblocks, sp)
        if rc:
            raise RuntimeError(f"sas_probe_read: {rc}")

    us_r = sustained(read, 10)
    del src, rout
    torch.cuda.empty_cache()
    return {"mfma_bf16_tflops": round(mfma_tflops, 1), "mfma_clock_ghz": round(clock_ghz, 3),
            "mfma_cycles_independent": round(indep_cycles, 2), "mfma_cycles_dependent": round(dep_cycles, 2),
            "hbm_read_gbs": round(nbytes / (us_r * 1e-6) / 1e9, 1),
            "method": "sas_probe.hip: 32x32x16 bf16 MFMA on random operands, 1 wave/SIMD, "
                      "register-only; 16-B streaming reads of 4 GiB; each sustained for "
                      f"{secs:.0f} s before 10 timed launches"}


# ---------------------------------------------------------------------------
# CPU baseline: the C oracle on a bounded sample of the same workload
# ---------------------------------------------------------------------------
def cpu_baseline(name, n_seq, seed=0):
    from oracle import golden_c

    wl_shape = dict(decode128k=(128, 2, 128, 131072, 2048), decode32=(32, 1, 64, 32768, 512),
                    prefill8k=(1, 8192, 128, 8192, 2048))[name]
    B_full, q_per, H, ctx, K = wl_shape
    rng = np.random.default_rng(seed)
    cores = len(os.sched_getaffinity(0))

    def bf16_bits(n):
        return (rng.standard_normal(n, dtype=np.float32).view(np.uint32) >> 16).astype(np.uint16)

    if name == "prefill8k":
        # a stratified sample of query tokens of the one sequence
        n_tok_full = q_per
        tokens = np.linspace(0, q_per - 1, 256).astype(np.int64)
        nb, T = 1, q_per
        kv = [ctx]
        q = np.zeros((T, H, D_QK), np.uint16)
        q[tokens] = bf16_bits(len(tokens) * H * D_QK).reshape(len(tokens), H, D_QK)
        ori = bf16_bits(ctx // PAGE * PAGE * D_QK).reshape(ctx // PAGE, PAGE, D_QK)
        obt = np.arange(ctx // PAGE, dtype=np.int32)[None]
        ncp = ctx // RATIO // PAGE
        cmp = bf16_bits(ncp * PAGE * D_QK).reshape(ncp, PAGE, D_QK)
        cbt = np.arange(ncp, dtype=np.int32)[None]
        idx = np.full((T, K), -1, np.int32)
        for t in tokens:
            thr = (t + 1) // RATIO
            idx[t, :min(thr, K)] = rng.permutation(thr)[:K]
        sample = f"{len(tokens)} of {q_per} query tokens (stratified), scaled by token count"
        cu = np.array([0, T], np.int32)
        scale_up = n_tok_full / len(tokens)
    else:
        # Sequences share one window pool (3 pages) and one compressed pool: the
        # oracle's cost depends on the shapes, not on which pages hold the rows.
        nb = n_seq
        kv = [ctx] * nb
        T = nb * q_per
        tokens = None
        q = bf16_bits(T * H * D_QK).reshape(T, H, D_QK)
        npg = math.ceil(ctx / PAGE)
        obt = np.full((nb, npg), -1, np.int32)
        obt[:, npg - 3:] = np.arange(3, dtype=np.int32)
        ori = bf16_bits(3 * PAGE * D_QK).reshape(3, PAGE, D_QK)
        ncp = math.ceil(ctx // RATIO / PAGE)
        cmp = bf16_bits(ncp * PAGE * D_QK).reshape(ncp, PAGE, D_QK)
        cbt = np.tile(np.arange(ncp, dtype=np.int32), (nb, 1))
        idx = np.full((T, K), -1, np.int32)
        for t in range(T):
            thr = (ctx - q_per + t % q_per + 1) // RATIO
            take = min(thr, K)
            idx[t, :take] = rng.choice(thr, size=take, replace=False)
        cu = np.arange(0, T + 1, q_per, dtype=np.int32)
        sample = f"{nb} of {B_full} sequences ({T} query tokens), scaled by sequence count"
        scale_up = B_full / nb
    sinks = rng.uniform(-1, 1, H).astype(np.float32)
    t0 = time.perf_counter()
    golden_c.attention(q=q, ori_kv=ori, ori_block_table=obt, q_prefix=cu[:-1],
                       act_q=np.diff(cu), seqused_kv=kv, sinks=sinks,
                       softmax_scale=1.0 / math.sqrt(D_QK), scenario=3, cmp_kv=cmp,
                       cmp_block_table=cbt, cmp_sparse_indices=idx, cmp_ratio=RATIO,
                       d_v=D_V, q_dtype="bf16", kv_dtype="bf16", tokens=tokens, nthreads=cores)
    secs = time.perf_counter() - t0
    return dict(value=secs * 1e6 * scale_up, unit="us/call", cores=cores, kind="port",
                sample=f"{sample}; sample took {secs:.2f} s")


def profile_attend(name, steps, dev, core_num=256, stage="attend", compact=False):
    """Plan and resolve once, then launch only the attention stage `steps` times
    (the kernel the roofline rates), or the whole forward call (resolve,
    attention, combine) with stage="forward", for rocprofv3 counter runs.
    compact: the MALL-sized KV footprint of make_workload."""
    wl = make_workload(name, seed=0, dev=dev, compact=compact)
    _, launch, _, _ = build_call(wl, core_num)
    launch.run("resolve")
    for _ in range(steps):
        launch.run(stage)
    torch.cuda.synchronize()
    print(json.dumps({"mode": stage, "workload": name, "compact": compact, "launches": steps,
                      "alg_bytes": wl["alg_bytes"], "alg_flops": wl["alg_flops"]}))


def _smi_sample():
    """Socket power (W) and GFX clocks (MHz) from one `amd-smi metric -p -c` call."""
    import subprocess

    try:
        txt = subprocess.run(["amd-smi", "metric", "-p", "-c"], capture_output=True, text=True,
                             timeout=30).stdout
    except Exception as e:  # noqa: BLE001
        return {"error": str(e)}
    power, clocks, in_gfx = None, [], False
    for line in txt.splitlines():
        s = line.strip()
        if s.startswith("SOCKET_POWER:"):
            power = s.split(":", 1)[1].strip()
        elif s.startswith("GFX_"):
            in_gfx = True
        elif s.endswith(":") and not s.startswith("GFX_"):
            in_gfx = False
        elif in_gfx and s.startswith("CLK:"):
            clocks.append(s.split(":", 1)[1].strip())
            in_gfx = False
    return {"socket_power": power, "gfx_clk": clocks}


def power_mode(name, secs, dev, compact=False):
    """Run one stage back to back for `secs` s and sample power / clocks halfway:
    the attention stage of a workload, or a peak probe ('mfma_probe', 'read_probe')."""
    import ctypes

    stream = torch.cuda.current_stream(dev)
    if name in ("mfma_probe", "read_probe"):
        from dsv4_planb_amd.build import PROBE_LIB

        lib = ctypes.CDLL(PROBE_LIB)
        sp = ctypes.c_void_p(stream.cuda_stream)
        if name == "mfma_probe":
            out = torch.empty(256 * 256, dtype=torch.float32, device=dev)
            ticks = torch.zeros(256 * 4, dtype=torch.int64, device=dev)
            fn = lambda: lib.sas_probe_mfma(ctypes.c_void_p(out.data_ptr()),  # noqa: E731
                                            ctypes.c_void_p(ticks.data_ptr()), 16000, 256, 0, sp)
        else:
            src = torch.empty(4 << 30, dtype=torch.uint8, device=dev)
            out = torch.empty(2048 * 256, dtype=torch.int32, device=dev)
            fn = lambda: lib.sas_probe_read(ctypes.c_void_p(src.data_ptr()),  # noqa: E731
                                            ctypes.c_size_t(4 << 30), ctypes.c_void_p(out.data_ptr()),
                                            2048, sp)
    else:
        wl = make_workload(name, seed=0, dev=dev, compact=compact)
        _, launch, _, _ = build_call(wl)
        launch.run("resolve")
        fn = lambda: launch.run("attend")  # noqa: E731
    idle = _smi_sample()
    fn()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    n, sample = 0, None
    while time.perf_counter() - t0 < secs:
        fn()
        n += 1
        if sample is None and time.perf_counter() - t0 > secs / 2:
            for _ in range(5):  # keep the queue full while sampling
                fn()
            n += 5
            sample = _smi_sample()
        if n % 20 == 0:
            torch.cuda.synchronize()
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    print(json.dumps({"mode": "power", "stage": name, "compact": compact, "launches": n,
                      "us_per_launch": round(dt / n * 1e6, 1),
                      "under_load": sample, "before": idle}))


def main_r_batch(name):
    return dict(decode128k=128, decode32=32, prefill8k=1, decode128k_fp8=128, ragged_fp8=64)[name]


# ---------------------------------------------------------------------------
def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=100)
    ap.add_argument("--workload", default="decode128k",
                    choices=["decode128k", "prefill8k", "decode32", "decode128k_fp8", "ragged_fp8"])
    ap.add_argument("--extra", default="prefill8k,decode32,decode128k_fp8,ragged_fp8",
                    help="comma-separated extra workloads reported under 'workloads' ('' = none)")
    ap.add_argument("--settle", type=float, default=0.25,
                    help="seconds of back-to-back calls per workload before its warmup and timed "
                         "region (the clock and power reach steady state); reported as 'settle'")
    ap.add_argument("--cpu-seqs", type=int, default=0,
                    help="cap on sampled sequences for the CPU baseline (0 = size for ~10 s)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-peaks", action="store_true",
                    help="skip the on-box MFMA / HBM peak probes")
    ap.add_argument("--mode", default="bench", choices=["bench", "attend", "forward", "copy", "power"],
                    help="bench: the JSON line; attend: only the attention stage of --workload, "
                         "--steps launches (for counter runs); forward: the whole call (resolve, "
                         "attention, combine), --steps times; copy: a 1 GiB device copy, "
                         "--steps times (calibrates the HBM byte counters); power: --stage back "
                         "to back for --secs with a power / clock sample")
    ap.add_argument("--stage", default="decode128k",
                    choices=["decode128k", "prefill8k", "decode32", "decode128k_fp8", "ragged_fp8",
                             "mfma_probe", "read_probe"],
                    help="what --mode power runs")
    ap.add_argument("--secs", type=float, default=10.0, help="--mode power duration")
    ap.add_argument("--sustain", type=float, default=5.0,
                    help="seconds of back-to-back replays after every other timing of the headline "
                         "workload, then `steps` replays timed again (reported as 'sustained'; "
                         "0 skips it)")
    ap.add_argument("--backward", default="decode128k,prefill8k",
                    help="comma-separated workloads whose backward is timed, reported under "
                         "'backward' ('' = none; 16-bit KV workloads only)")
    ap.add_argument("--compact", action="store_true",
                    help="--mode power / attend / forward: all sequences read the first "
                         "sequence's KV pages")
    args = ap.parse_args()

    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print(json.dumps({"error": "the benchmark measures one GPU only: the operator is a "
                          "per-GPU kernel and sharding is data-parallel over sequences "
                          "(no exchange); run with --gpus 1"}))
        sys.exit(2)

    torch.backends.cuda.matmul.allow_tf32 = False
    dev = torch.device("cuda:0")
    if args.mode == "copy":
        src = torch.empty(1 << 30, dtype=torch.uint8, device=dev)
        dst = torch.empty_like(src)
        for _ in range(args.steps):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"mode": "copy", "bytes_per_copy": src.numel(), "copies": args.steps}))
        return
    if args.mode in ("attend", "forward"):
        profile_attend(args.workload, args.steps, dev, stage=args.mode, compact=args.compact)
        return
    if args.mode == "power":
        power_mode(args.stage, args.secs, dev, compact=args.compact)
        return
    results = {}
    for name in [args.workload] + [w for w in args.extra.split(",") if w and w != args.workload]:
        _log(f"{name}: building inputs")
        wl = make_workload(name, seed=0, dev=dev)
        _log(f"{name}: timing")
        r = measure(wl, args.steps, args.warmup, settle_s=args.settle,
                    sustain_s=args.sustain if name == args.workload else 0.0)
        _log(f"{name}: call {r['call_us']:.1f} us, attend {r['attend_us']:.1f} us "
             f"(kernel {r['attend_kernel_us']:.1f} us)")
        attend_s = r["attend_kernel_us"] * 1e-6  # the kernel's own dispatch time
        r.update(alg_bytes=wl["alg_bytes"], alg_flops=wl["alg_flops"], uniq_rows=wl["uniq_rows"],
                 rows_total=wl["rows_total"],
                 attend_gbs=wl["alg_bytes"] / attend_s / 1e9,
                 attend_tflops=wl["alg_flops"] / attend_s / 1e12,
                 call_gbs=wl["alg_bytes"] / (r["call_us"] * 1e-6) / 1e9,
                 call_tflops=wl["alg_flops"] / (r["call_us"] * 1e-6) / 1e12)
        results[name] = r
        del wl
        torch.cuda.empty_cache()

    backward = {}
    for name in [w for w in args.backward.split(",") if w]:
        if name.endswith("fp8"):
            continue  # the backward supports 16-bit KV pools only
        _log(f"{name}: backward")
        wl = make_workload(name, seed=0, dev=dev)
        b = measure_backward(wl, max(3, min(args.steps, 10)), settle_s=args.settle)
        _log(f"{name}: backward dq {b['dq']['call_us']:.1f} us, with dK/dV "
             f"{b['dq_dkv']['call_us']:.1f} us")
        backward[name] = b
        del wl
        torch.cuda.empty_cache()

    main_r = results[args.workload]
    bound = "mfma" if args.workload == "prefill8k" else "hbm"
    peaks = None
    if not args.no_peaks:
        _log("on-box peaks")
        peaks = measure_peaks(dev)
    if bound == "hbm":
        ach, peak, unit = main_r["attend_gbs"], HBM_PEAK_GBS, "GB/s"
        measured = peaks["hbm_read_gbs"] if peaks else None
    else:
        ach, peak, unit = main_r["attend_tflops"], MFMA_BF16_PEAK_TFLOPS, "TFLOP/s"
        measured = peaks["mfma_bf16_tflops"] if peaks else None
    if peaks:
        for r in results.values():
            r["frac_hbm_measured"] = round(r["attend_gbs"] / peaks["hbm_read_gbs"], 4)
            r["frac_mfma_measured"] = round(r["attend_tflops"] / peaks["mfma_bf16_tflops"], 4)
    roofline = {"bound": bound, "achieved": round(ach, 2), "peak": peak, "unit": unit,
                "frac": round(ach / peak, 4), "traffic": _traffic_from_profile(args.workload),
                "measured_peak": measured,
                "frac_of_measured": round(ach / measured, 4) if measured else None,
                "kernel": KERNEL_NAME[args.workload], "kernel_us": round(main_r["attend_kernel_us"], 2),
                "kernel_us_rtc": round(main_r["attend_kernel_rtc_us"], 2),
                "kernel_timing": "mean execution time of the attention dispatches as the forward "
                                 "launches them (with the units' own row resolution where the "
                                 "forward fuses it), their own start/end HIP events "
                                 "(sas_attend_timed), steps back-to-back launches; kernel_us_rtc: "
                                 "the same dispatches' span on the GPU's 100 MHz real-time counter "
                                 "(earliest workgroup start to latest workgroup end)",
                "algorithmic_bytes": main_r["alg_bytes"], "algorithmic_flops": main_r["alg_flops"]}
    cpu = None
    if not args.no_cpu_baseline and not args.workload.endswith("fp8"):
        _log("cpu baseline")
        if args.workload == "prefill8k":
            cpu = cpu_baseline(args.workload, 1)
        else:  # size the sample for ~10 s of CPU work, from a one-sequence probe
            probe = cpu_baseline(args.workload, 1)
            per_seq_s = probe["value"] * 1e-6 / main_r_batch(args.workload)
            n = int(max(1, min(main_r_batch(args.workload), 10.0 / max(per_seq_s, 1e-3))))
            cpu = cpu_baseline(args.workload, n if args.cpu_seqs <= 0 else min(n, args.cpu_seqs))
    desc = {
        "decode128k": "decode: B=128 seqs x 131072 KV, 2 query tokens/seq, H=128, top-k 2048, "
                      "window 128, ratio 4, page 64, d_qk 576 / d_v 512",
        "prefill8k": "prefill: B=1, 8192 query tokens over 8192 KV, H=128, top-k 2048, "
                     "window 128, ratio 4, page 64, d_qk 576 / d_v 512",
        "decode32": "decode: B=32 seqs x U[4096,32768] KV, 1 query token, H=64, top-k 512, "
                    "window 128, ratio 4, page 64, d_qk 576 / d_v 512",
        "decode128k_fp8": "decode: B=128 seqs x 131072 KV, 2 query tokens/seq, H=128, top-k 2048, "
                          "window 128, ratio 4, page 64, fp8 e4m3 KV with per-row fp32 scale, bf16 q",
        "ragged_fp8": "ragged: B=64 seqs x log-U[256,131072] KV, 1/2/4 query tokens/seq, H=128, "
                      "top-k 2048 (-1 padded), window 128, ratio 4, page 64, fp8 e4m3 KV with "
                      "per-row fp32 scale, bf16 q",
    }
    line = {
        "metric": "us/call of the sparse shared-KV attention forward (1x MI355X), with achieved "
                  "HBM GB/s (decode) and MFMA TFLOP/s (prefill)",
        "value": round(main_r["call_us"], 2),
        "unit": "us/call",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(main_r["call_us"] / 1000.0, 5),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded N(0,1) bf16 q/KV, random page permutation, random top-k)",
        "config": {"workload": desc[args.workload], "name": args.workload},
        "roofline": roofline,
        "measured_peaks": peaks,
        "cpu_baseline": cpu,
        "backward": backward or None,
        "workloads": {k: {kk: (round(vv, 3) if isinstance(vv, float) else vv) for kk, vv in v.items()}
                      for k, v in results.items()},
    }
    print(json.dumps(line))


if __name__ == "__main__":
    main()
