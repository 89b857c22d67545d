"""A plan buffer that is shorter than the call's plan.

The C entry points take no plan size.  A plan that ``sas_plan`` built for fewer tokens or
a smaller target is a shorter buffer, and the kernels refuse it by its header: zeros and
SAS_ERR_PLAN, with nothing past the header read.  (The Python entry points refuse the size
on the host, so the launch is given the buffer behind them.)  A plan of the right size that
the caller keeps gives the same results as the call's own.
"""

from __future__ import annotations

import pytest
import torch

from tests.cases import make_case
from tests.test_gpu_backward import _launch
from tests.test_gpu_plan_reuse import _plan

pytestmark = pytest.mark.gpu

CASES = {
    # two-wave kernel (more tokens than target units, at most 64 heads); four-wave kernel
    # behind the resolver; units that resolve their own rows
    "narrow": dict(B=1, H=16, seq_kv=[700], q_per_seq=[300], scenario=1),
    "wide": dict(B=1, H=100, seq_kv=[700], q_per_seq=[300], scenario=3, K=64),
    "fused": dict(B=3, H=16, seq_kv=[900, 40, 500], q_per_seq=[1, 2, 1], scenario=3, K=64),
}


@pytest.mark.parametrize("short", ["tokens", "target", "header"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_a_short_plan_is_refused(name, short):
    c = make_case(seed=311, **CASES[name])
    print(f"\n[case] short_plan {name} {short}: B={c.B} T={c.T} H={c.H}", flush=True)
    launch, out, lse = _launch(c)
    assert launch.device_status() == 0 and out.any()
    small = make_case(B=1, H=c.H, seq_kv=[40], q_per_seq=[1], scenario=c.scenario, K=c.K, seed=312)
    args = small if short == "tokens" else c
    plan = _plan(args, torch.from_numpy(args.cu_seqlens_q), torch.from_numpy(args.seqused_kv).cuda(),
                 40 if short == "target" else 256)
    if short == "header":  # the header of another call's plan and nothing else
        plan = plan[:24].clone()
        plan[2] += 1  # its token count
    launch.plan = plan.clone()  # (without the host's record)
    for x in (out, lse):
        x.fill_(7.0)
    launch.run()
    assert launch.device_status() == -8
    assert not out.any() and not lse.any()
    dq, dsinks, d_ori, d_cmp = launch.backward(torch.ones_like(out), kv_grad=True)
    torch.cuda.synchronize()
    assert not dq.any() and not dsinks.any() and not d_ori.any()
    assert d_cmp is None or not d_cmp.any()


@pytest.mark.parametrize("name", sorted(CASES))
def test_a_callers_plan_gives_the_calls_own_results(name):
    """The kernels behind the resolver read the copy it makes of a caller's plan: forward and
    backward with a kept plan are those without one, also after a refused call has used
    the same workspace."""
    c = make_case(seed=313, **CASES[name])
    print(f"\n[case] kept_plan {name}: B={c.B} T={c.T} H={c.H}", flush=True)
    launch, out, lse = _launch(c)
    want = out.clone(), lse.clone()
    g = torch.randn(out.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(5)).to(out.dtype)
    want_dq = launch.backward(g, kv_grad=True)
    plan = _plan(c, torch.from_numpy(c.cu_seqlens_q), torch.from_numpy(c.seqused_kv).cuda(), 256)
    refused = plan.clone()
    refused[4:6] = 1 << 20  # (chunk and target: the target is checked)
    for p, ok in ((refused, False), (plan, True)):
        launch.plan = p
        launch.run()
        assert launch.device_status() == (0 if ok else -8)
    assert torch.equal(out, want[0]) and torch.equal(lse, want[1])
    dq, dsinks, d_ori, d_cmp = launch.backward(g, kv_grad=True)
    torch.cuda.synchronize()
    assert torch.equal(dsinks, want_dq[1])
    # sums of fp32 atomics in any order (dq of split tokens, the pools' rows): n terms in two
    # orders differ by at most 2 n 2^-24 of the sum of their magnitudes; n <= 300 tokens here
    # and those magnitudes are within a few times the largest sum
    for got, ref in ((dq, want_dq[0]), (d_ori, want_dq[2]), (d_cmp, want_dq[3])):
        if ref is not None:
            assert (got - ref).abs().max() <= 2 * 300 * 2.0 ** -24 * 4 * ref.abs().max()
