"""What stays allocated while a model's backward runs.

During ``loss.backward()`` the graph is alive from its root, so whatever a layer's
autograd node holds adds up over the layers.  A layer's backward workspace (the forward's
lists, the spilled P and dS: up to 2 GiB and more) is used by its own launches only: the
caching allocator hands the block on in stream order, so nothing may hold it once they
are enqueued.
"""

from __future__ import annotations

import gc

import pytest
import torch

from tests.cases import make_case
from tests.gpu_helpers import to_device

pytestmark = pytest.mark.gpu


def _call(c, d, q, ori, cmp_):
    from dsv4_planb_amd import sparse_attn_sharedkv

    return sparse_attn_sharedkv(
        q, ori_kv=ori, cmp_kv=cmp_, cmp_sparse_indices=d["cmp_sparse_indices"],
        ori_block_table=d["ori_block_table"], cmp_block_table=d["cmp_block_table"],
        cu_seqlens_q=d["cu_seqlens_q"], seqused_kv=d["seqused_kv"], sinks=d["sinks"],
        softmax_scale=c.softmax_scale, cmp_ratio=c.cmp_ratio, ori_win_left=c.win_left)


@pytest.mark.parametrize("layers", [1, 3])
def test_a_layers_backward_workspace_is_given_back(layers):
    c = make_case(B=1, H=64, seq_kv=[900], q_per_seq=[900], scenario=3, K=256, seed=301)
    d = to_device(c)
    print(f"\n[case] autograd_memory: layers={layers} T={c.T} H={c.H} K={c.K}", flush=True)
    ori = d["ori_kv"].detach().requires_grad_()
    cmp_ = d["cmp_kv"].detach().requires_grad_()
    qs = [d["q"].detach().clone().requires_grad_() for _ in range(layers)]
    outs = [_call(c, d, q, ori, cmp_) for q in qs]
    g = torch.randn(outs[0].shape, device="cuda", generator=torch.Generator("cuda").manual_seed(6)).to(outs[0].dtype)
    # one layer's workspace, from a launch of the same call
    need = _workspace(c, d)
    assert need > 64 << 20
    gc.collect()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.autograd.backward(outs, [g] * layers)
    torch.cuda.synchronize()
    grads = sum(x.grad.numel() * x.grad.element_size() for x in [*qs, ori, cmp_])
    held = torch.cuda.memory_allocated() - before - grads
    print(f"held beside the gradients: {held / 2**20:.1f} MiB; a workspace: {need / 2**20:.1f} MiB", flush=True)
    assert held < need // 16  # (the outputs, and with them every layer's node, are alive)
    # the released workspaces were not reused too early: every layer has the same gradient
    for q in qs[1:]:
        assert torch.equal(q.grad, qs[0].grad)
    del outs


def _workspace(c, d):
    import ctypes

    from dsv4_planb_amd import _lib
    from dsv4_planb_amd.api import build_launch

    cu = d["cu_seqlens_q"]
    launch, _, _ = build_launch(
        q_flat=d["q"], ori_kv=d["ori_kv"], ori_block_table=d["ori_block_table"], cmp_kv=d["cmp_kv"],
        cmp_block_table=d["cmp_block_table"], cmp_indices=d["cmp_sparse_indices"], q_prefix=cu[:-1],
        act_q_lens=cu[1:] - cu[:-1], seqused_kv=d["seqused_kv"], sinks=d["sinks"], metadata=None,
        scenario=c.scenario, topk=c.K, cmp_ratio=c.cmp_ratio, ori_win_left=c.win_left,
        softmax_scale=c.softmax_scale, core_num=256)
    n = ctypes.c_size_t()
    assert _lib.load().sas_backward_workspace_size_for(ctypes.byref(launch.params), 1, ctypes.byref(n)) == 0
    return n.value
