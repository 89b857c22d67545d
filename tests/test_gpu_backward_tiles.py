"""The KV pools' gradient by key tiles (prefill-like calls) against the oracle's
float64 gradient, at the sizes where its pieces meet: key tiles of 128 positions,
groups of tokens, 32-head chunks, rows listed more than once, tokens left to the
per-unit kernel, and a spill that takes several runs.

The tolerance is the backward tests' own (0.5% of the gradient's norm, 1% of its
largest element): P and dS enter both kernels with the same rounding.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.cases import make_case
from tests.test_gpu_backward import _check_grad, _check_pools, _dout, _exact_grads, _launch

pytestmark = pytest.mark.gpu


def _repeated():
    """Lists with ids repeated twice and three times, a terminator and ids past the
    threshold, 100 heads (a partial 32-head chunk)."""
    c = make_case(B=2, H=100, seq_kv=[600, 300], q_per_seq=[40, 30], scenario=3, K=64, seed=201)
    for t in range(0, c.T, 3):
        c.idx[t, 5] = c.idx[t, 2]
        c.idx[t, 9] = c.idx[t, 2]
        c.idx[t, 30] = c.idx[t, 11]
    c.idx[1, 7] = 10_000
    c.idx[2, 20] = -1
    return c


@pytest.mark.parametrize("name,build", [
    # window tiles: sequences that end at, just past and well inside a tile
    ("window", lambda: make_case(B=3, H=16, seq_kv=[128, 257, 40], q_per_seq=[128, 130, 40],
                                 scenario=1, seed=202)),
    ("window_d512_fp16", lambda: make_case(B=2, H=64, D=512, seq_kv=[300, 129], q_per_seq=[70, 129],
                                           scenario=1, win_left=200, q_dtype="fp16", kv_dtype="fp16",
                                           seed=203)),
    ("repeated_ids_h100", _repeated),
    # every compressed row (no index list), d 512
    ("cfa_d512", lambda: make_case(B=2, H=32, D=512, seq_kv=[1100, 513], q_per_seq=[33, 64],
                                   scenario=2, K=0, cmp_ratio=4, seed=204)),
    # few of many rows listed: window tiles, the compressed rows by the per-unit kernel
    ("sparse_lists", lambda: make_case(B=1, H=64, seq_kv=[4000], q_per_seq=[50], scenario=3, K=64,
                                       seed=205)),
    # a long list capacity: the spill holds about 1,000 tokens, so two runs
    ("two_runs", lambda: make_case(B=1, H=16, seq_kv=[1090], q_per_seq=[1090], scenario=3, K=16384,
                                   seed=206)),
])
def test_tiles_match_f64_gradient(name, build):
    c = build()
    print(f"\n[case] tiles_{name}: B={c.B} T={c.T} H={c.H} D={c.D} scen={c.scenario} K={c.K}", flush=True)
    launch, _, _ = _launch(c)
    g, g_np = _dout(c, seed=sum(name.encode()))
    dq, _, d_ori, d_cmp = launch.backward(g.cuda(), kv_grad=True)
    torch.cuda.synchronize()
    dq_ex, _, dori_ex, dcmp_ex = _exact_grads(c, g_np, kv_grad=True)
    _check_grad(f"tiles_{name}:dq", dq.cpu().numpy(), dq_ex)
    _check_pools(f"tiles_{name}", c, d_ori, d_cmp, dori_ex, dcmp_ex)


def test_the_queries_gradient_alone_takes_every_run():
    """dq and dsinks without the pools' gradient, of a call whose spill would take two runs."""
    c = make_case(B=1, H=16, seq_kv=[1090], q_per_seq=[1090], scenario=3, K=16384, seed=206)
    launch, _, _ = _launch(c)
    g, _ = _dout(c, seed=9)
    with_pools = launch.backward(g.cuda(), kv_grad=True)
    alone = launch.backward(g.cuda())
    torch.cuda.synchronize()
    # (no token is split: no atomics in dq)
    assert torch.equal(alone[0], with_pools[0]) and torch.equal(alone[1], with_pools[1])


def test_an_infinite_gradient_stays_with_the_rows_its_token_reads():
    """One element of one token's dO is infinite: the rows that token attends may be
    anything, every other row is the gradient without that token."""
    c = make_case(B=1, H=32, seq_kv=[400], q_per_seq=[400], scenario=1, seed=207)
    launch, _, _ = _launch(c)
    g, g_np = _dout(c, seed=4)
    bad = 150
    g[bad, 3, 17] = float("inf")
    _, _, d_ori, _ = launch.backward(g.cuda(), kv_grad=True)
    torch.cuda.synchronize()
    g_np[bad] = 0.0
    _, _, want, _ = _exact_grads(c, g_np, kv_grad=True)
    got = d_ori.squeeze(2).cpu().numpy()
    page = got.shape[1]
    reads = {(int(c.ori_block_table[0, p // page]), p % page) for p in range(max(0, bad - 127), bad + 1)}
    keep = np.array([[(b, r) not in reads for r in range(page)] for b in range(got.shape[0])])
    assert not np.isfinite(got[~keep]).all()
    _check_grad("tiles_inf:d_ori_kv", got[keep], want[keep])
