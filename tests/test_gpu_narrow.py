"""The two-wave attention kernel (at most 64 heads, 16-bit KV, more tokens than target
units: ``core_num`` is set below the token count) against the oracle and the exact
value, by the parity suite's own rules: rows at the edges of its 16-key tiles, one to
64 heads, both dtypes and widths, split tokens and their partials, the redo, tokens no
sequence owns and a plan for other arguments.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.cases import make_case
from tests.gpu_helpers import assert_parity, run_op, to_device

pytestmark = pytest.mark.gpu


def _check(name, c, core_num, rule="baseline"):
    print(f"\n[case] narrow_{name}: B={c.B} T={c.T} H={c.H} D={c.D} scen={c.scenario} K={c.K} "
          f"q={c.q_dtype} cores={core_num}", flush=True)
    assert c.H <= 64 and c.T > core_num
    out, lse = run_op(c, core_num=core_num)
    ref, ref_lse = c.oracle_c()
    assert_parity(out, lse, ref, ref_lse, dtype=c.q_dtype, label=f"narrow_{name}",
                  exact=c.oracle_exact(), rule=rule)


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("D", [512, 576])
@pytest.mark.parametrize("H", [1, 33, 64])
def test_every_row_count_of_the_first_tiles(H, D, dt):
    """A prompt's first tokens attend 1, 2, 3, ... rows: units of one to five tiles,
    every remainder; top-k rows from the fourth token on."""
    c = make_case(B=2, H=H, D=D, seq_kv=[70, 21], q_per_seq=[70, 21], scenario=3, K=16, q_dtype=dt,
                  kv_dtype=dt, seed=301 + H)
    _check(f"first_rows_h{H}_d{D}_{dt}", c, core_num=4)


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
def test_split_tokens(dt):
    """Long rows beside short ones on few units: partials (fp16 for bf16 queries, fp32 for
    fp16 ones) of a token with tens of splits."""
    c = make_case(B=3, H=40, seq_kv=[9000, 40, 700], q_per_seq=[2, 30, 9], scenario=3, K=2048,
                  q_dtype=dt, kv_dtype=dt, seed=311)
    _check(f"splits_{dt}", c, core_num=32)


def test_window_only_other_window():
    c = make_case(B=2, H=16, seq_kv=[400, 90], q_per_seq=[60, 90], scenario=1, win_left=45, seed=312)
    c.sinks[:5] = -np.inf
    _check("window45", c, core_num=16)


@pytest.mark.parametrize("D", [512, 576])
def test_redo_on_large_logits(D):
    """The reference's large-magnitude draws: later logits rise past the frame of the first
    32 keys, and units are redone."""
    c = make_case(B=1, H=64, D=D, seq_kv=[3000], q_per_seq=[24], scenario=3, K=512, dist="reference",
                  seed=313)
    _check(f"redo_d{D}", c, core_num=8, rule="reference")


def test_a_redone_split_unit_stores_fp32_partials():
    """Values past fp16's range in a split unit: the redo stores its partials in fp32."""
    c = make_case(B=1, H=16, seq_kv=[5000], q_per_seq=[12], scenario=3, K=1024, value_scale=1.0, seed=314)
    rows = c.ori_kv  # raw rows: V elements of +-99840 in one dimension
    big = np.float32(99840.0).view(np.uint32) >> 16
    rows[..., 7] = np.where(rows[..., 7] & 0x8000, big | 0x8000, big).astype(rows.dtype)
    c.q_bits[..., 7] = 0  # (not in the logits)
    out, lse = run_op(c, core_num=8)
    ref, ref_lse = c.oracle_exact()
    scale = np.abs(ref).max(axis=(0, 1))
    err = np.abs(out - ref).max(axis=(0, 1))
    # each dimension against its own size: two bf16 roundings
    assert (err <= 2.0 ** -7 * scale).all(), (err / scale).max()


def test_plan_for_other_arguments_zeroes_every_output():
    from dsv4_planb_amd.api import build_launch
    from dsv4_planb_amd.metadata import device_plan, plan_params

    c = make_case(B=2, H=64, seq_kv=[300, 200], q_per_seq=[20, 20], scenario=3, K=64, seed=315)
    d = to_device(c)
    cu = d["cu_seqlens_q"]
    p = plan_params(total_tokens=c.T, batch=c.B, num_heads_q=64, scenario=3, topk=c.K, cmp_ratio=2,
                    ori_win_left=c.win_left, core_num=8)
    plan = device_plan(p, cu[:-1], cu[1:] - cu[:-1], d["seqused_kv"])
    launch, out, lse = build_launch(
        q_flat=d["q"], ori_kv=d["ori_kv"], ori_block_table=d["ori_block_table"], cmp_kv=d["cmp_kv"],
        cmp_block_table=d["cmp_block_table"], cmp_indices=d["cmp_sparse_indices"], q_prefix=cu[:-1],
        act_q_lens=cu[1:] - cu[:-1], seqused_kv=d["seqused_kv"], sinks=d["sinks"], metadata=plan,
        scenario=3, topk=c.K, cmp_ratio=4, ori_win_left=c.win_left, softmax_scale=c.softmax_scale,
        core_num=8)
    out.fill_(1.0)
    lse.fill_(1.0)
    launch.run()
    torch.cuda.synchronize()
    assert launch.device_status() == -8
    assert out.abs().max().item() == 0 and lse.abs().max().item() == 0
