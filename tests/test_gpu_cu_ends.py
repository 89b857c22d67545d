"""The forward on cumulative sequence ends (``sas_forward_cu``, the path of a call
without a gradient) gives the bits of the forward on lengths: with and without a plan,
the units resolving their own rows or behind the resolver, empty sequences, query rows
past the last sequence, and BSND."""

from __future__ import annotations

import pytest
import torch

from tests.cases import make_case
from tests.gpu_helpers import to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("with_plan", [False, True])
@pytest.mark.parametrize("cores", [256, 8])  # 8: more tokens than target units
@pytest.mark.parametrize("H,kv_dtype", [(64, "bf16"), (128, "bf16"), (128, "fp8e4m3")])
def test_cumulative_ends_give_the_bits_of_lengths(H, kv_dtype, cores, with_plan):
    from dsv4_planb_amd import sparse_attn_sharedkv, sparse_attn_sharedkv_metadata
    from dsv4_planb_amd.api import build_launch

    c = make_case(B=4, H=H, seq_kv=[700, 64, 3000, 40], q_per_seq=[3, 0, 12, 5], scenario=3, K=128,
                  kv_dtype=kv_dtype, seed=401)
    d = to_device(c)
    extra = torch.randn((2, H, c.D), dtype=d["q"].dtype, device="cuda")  # rows no sequence owns
    q = torch.cat([d.pop("q"), extra])
    T = q.shape[0]
    idx = torch.cat([d.pop("cmp_sparse_indices"), torch.zeros((2, 1, c.K), dtype=torch.int32, device="cuda")])
    cu = d.pop("cu_seqlens_q")
    meta = None
    if with_plan:
        full = cu.clone()
        full[-1] = T  # the plan counts every row; the call's last sequence ends earlier
        meta = sparse_attn_sharedkv_metadata(
            num_heads_q=H, num_heads_kv=1, head_dim=c.D, cu_seqlens_q=full, seqused_kv=d["seqused_kv"],
            layout_q="TND", has_cmp_kv=True, cmp_ratio=4, cmp_topk=c.K, aic_core_num=max(cores, 40))
    cores = max(cores, 40) if with_plan else cores
    launch, out, lse = build_launch(
        q_flat=q, cmp_indices=idx, q_prefix=cu[:-1], act_q_lens=cu[1:] - cu[:-1], metadata=meta, scenario=3,
        topk=c.K, cmp_ratio=4, ori_win_left=127, softmax_scale=c.softmax_scale, core_num=cores, **d)
    launch.run()
    got, got_lse = sparse_attn_sharedkv(
        q, cmp_sparse_indices=idx, cu_seqlens_q=cu, metadata=meta, softmax_scale=c.softmax_scale, cmp_ratio=4,
        core_num=cores, return_softmax_lse=True, **d)
    torch.cuda.synchronize()
    assert torch.equal(got, out) and torch.equal(got_lse, lse)
    assert got[:15].abs().max().item() > 0


def test_bsnd_ends():
    from dsv4_planb_amd import sparse_attn_sharedkv
    from dsv4_planb_amd.api import build_launch

    c = make_case(B=3, H=16, seq_kv=[300, 77, 900], q_per_seq=7, scenario=1, seed=402)
    d = to_device(c)
    q = d.pop("q")
    cu = d.pop("cu_seqlens_q")
    launch, out, _ = build_launch(
        q_flat=q, cmp_kv=None, cmp_block_table=None, cmp_indices=None, q_prefix=cu[:-1],
        act_q_lens=cu[1:] - cu[:-1], metadata=None, scenario=1, topk=0, cmp_ratio=4, ori_win_left=127,
        softmax_scale=c.softmax_scale, core_num=256, **d)
    launch.run()
    got = sparse_attn_sharedkv(q.reshape(3, 7, 16, c.D), layout_q="BSND", softmax_scale=c.softmax_scale, **d)
    torch.cuda.synchronize()
    assert torch.equal(got.reshape(out.shape), out)
