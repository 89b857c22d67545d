"""Host entry point of the MI355X sparse shared-KV attention operator.

Drop-in for the reference's ``sparse_attn_sharedkv_tilelang/api.py``: same
function name, keyword arguments, defaults, scenario resolution, layouts,
return convention and exception types (``api.py:129-397``).  Underneath, the
call goes through the C ABI of ``libsas_hip.so`` (``include/sas.h``) to gfx950
HIP kernels; there is no CPU fallback.

Differences from the reference, all extensions:

* ``num_heads_q`` may be 1..128 (reference: 64), ``head_dim`` 512 or 576; with
  576 the query/key width is 576 and the output is the first 512 (V) columns.
* ``ori_win_left`` may be any value >= 0 (reference kernel: 127).
* ``ori_kv`` / ``cmp_kv`` may be ``torch.float8_e4m3fn`` with per-row fp32
  scales ``ori_kv_scale`` / ``cmp_kv_scale`` ``[block_num, block_size, 1]``.
* paged KV may carry padded block / row strides (the reference benchmark's
  stride-padded layout, ``sparse_attn_sharedkv_perf_compare.py:220-247``).
* ``metadata`` may be the reference's int32[1024] table or a plan from
  :func:`dsv4_planb_amd.metadata.sparse_attn_sharedkv_metadata` with
  ``aic_core_num > 36``.  The 1024-entry table partitions query rows over the
  reference's 24-36 cores; the partition does not change any result, so the
  table is accepted by its size and the GPU builds its own split-KV plan for all
  CUs in the same stream (the planner kernel).  As with the reference's table, a
  plan may be reused while ``seqused_kv`` changes (the kernels read the KV
  lengths on every call).  A plan built for other arguments (token count, batch,
  scenario, window, ratio, top-k, CU count, or -- where the call's query lengths
  are known on the host -- other ``cu_seqlens_q``) raises ``ValueError``; one the
  host cannot check is checked on the device, which zeroes the outputs it
  refuses and sets the workspace status word (:meth:`SasLaunch.device_status`).
* No host synchronisation happens when every tensor is already on the device,
  so the call can be captured into a graph.
"""

from __future__ import annotations

import ctypes
from typing import Optional, Tuple, Union

import torch

from . import _lib
from ._lib import SasParams, SasTensors, SAS_META_SIZE

DEFAULT_CORE_NUM = 256  # compute units of one MI355X (reference default: 24 Ascend cores)
DEFAULT_BLOCK_I = 128  # the reference's KV tile width; kept for importers (api.py:44)

_KERNEL_CACHE: dict = {}


def _torch_to_sas_dtype(t: torch.dtype) -> int:
    """Query / output dtype code (reference ``_torch_to_tilelang_dtype``, api.py:51-56)."""
    if t == torch.bfloat16:
        return _lib.DT_BF16
    if t == torch.float16:
        return _lib.DT_FP16
    raise ValueError(f"unsupported torch dtype {t}")


def _kv_dtype_code(kv: torch.Tensor, q_code: int) -> int:
    if kv.dtype == torch.float8_e4m3fn:
        return _lib.DT_FP8E4M3
    code = _torch_to_sas_dtype(kv.dtype)
    if code != q_code:
        raise ValueError(f"kv dtype {kv.dtype} must match q dtype or be float8_e4m3fn")
    return code


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _dev_i32(t: torch.Tensor, device) -> torch.Tensor:
    # (the usual case first: a tensor that needs nothing costs no dispatch)
    if t.dtype is torch.int32 and t.device == device and t.is_contiguous():
        return t
    return t.to(device=device, dtype=torch.int32).contiguous()


def _dev_f32(t: torch.Tensor, device) -> torch.Tensor:
    if t.dtype is torch.float32 and t.device == device and t.is_contiguous():
        return t
    return t.to(device=device, dtype=torch.float32).contiguous()


def _paged_strides(kv: torch.Tensor, D: int, name: str):
    if kv.dim() != 4:
        raise ValueError(f"{name} must be paged [block_num, block_size, N2, D], got {tuple(kv.shape)}")
    if kv.shape[3] != D:
        raise ValueError(f"{name} head dim {kv.shape[3]} != q head dim {D}")
    stride = kv.stride()
    if stride[3] != 1:
        raise ValueError(f"{name} rows must be contiguous in the head dim")
    return stride[0], stride[1]


def _stream_handle(device) -> ctypes.c_void_p:
    if device.index is not None:  # (without building a Stream object)
        return ctypes.c_void_p(torch._C._cuda_getCurrentRawStream(device.index))
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)


def _check_plan_record(metadata: torch.Tensor, p: SasParams, host_lens, target: int) -> None:
    """Raise ``ValueError`` when the plan's own record (written by the metadata op,
    valid while the tensor is unmodified) names other arguments than this call:
    the host-side counterpart of the kernels' check, with the reason spelled out.
    host_lens: the call's (q_prefix, act_q) on the host (or a function that returns
    them), or None when they are on the device only (then the device check covers
    them, without a host sync); target: the call's balance target."""
    rec = getattr(metadata, "_sas_plan", None)
    if rec is None or rec.get("version") != metadata._version:
        return
    diffs = []

    def cmp(name, planned, called):
        if planned != called:
            diffs.append(f"{name}: planned {planned}, called with {called}")

    cmp("total_tokens", rec["T"], int(p.total_tokens))
    cmp("batch", rec["B"], int(p.batch))
    cmp("scenario", rec["scenario"], int(p.scenario))
    cmp("ori_win_left", rec["win_left"], int(p.ori_win_left))
    if p.scenario >= 2:
        cmp("cmp_ratio", rec["cmp_ratio"], int(p.cmp_ratio))
    if p.scenario == 3:
        cmp("topk", rec["K"], int(p.topk))
    cmp("work units (core_num)", rec["target"], target)
    if not diffs and host_lens is not None and rec.get("q_prefix") is not None:
        lens = host_lens() if callable(host_lens) else host_lens
        qp, aq = (x.to("cpu", torch.int64).reshape(-1) for x in lens)
        if not (torch.equal(qp, rec["q_prefix"]) and torch.equal(aq, rec["act_q"])):
            diffs.append("query layout (cu_seqlens_q / seqused_q) differs from the plan's")
    if diffs:
        raise ValueError("metadata was built for other arguments than this call ("
                         + "; ".join(diffs) + "): rebuild it with sparse_attn_sharedkv_metadata")


class SasLaunch:
    """One fully described call: parameter block, tensor block, workspace."""

    def __init__(self, params: SasParams, tensors: SasTensors, keep: list, plan, ws, device):
        self.params = params
        self.tensors = tensors
        self._keep = keep  # tensors whose storage the raw pointers refer to
        self.plan = plan
        self.ws = ws
        self.device = device
        self.ori_kv = None  # the pools (their shapes and strides lay out the KV gradient)
        self.cmp_kv = None

    def device_status(self) -> int:
        """The workspace status word of the last forward call: 0, or -8
        (``SAS_ERR_PLAN``) when the plan passed in was built for other arguments
        (the outputs it refused were zeroed).  Synchronises the device."""
        return int(self.ws[:4].view(torch.int32).item())

    def debug_lists(self):
        """The row lists the attention kernel read in the last forward (or
        resolve) on this launch's workspace: ``(addr [T, cap] int64, scale [T, cap]
        float32 or None, counts [T, 2] int32)`` on the device, counts being each
        token's (window rows, compressed rows)."""
        p = self.params
        K = p.topk if p.scenario >= 2 else 0
        cap = p.ori_win_left + 1 + K
        T = p.total_tokens
        addr = torch.empty((T, cap), dtype=torch.int64, device=self.device)
        kv8 = p.kv_dtype == _lib.DT_FP8E4M3
        scale = torch.empty((T, cap), dtype=torch.float32, device=self.device) if kv8 else None
        counts = torch.empty((T, 2), dtype=torch.int32, device=self.device)
        rc = _lib.load().sas_debug_lists(ctypes.byref(p), _ptr(self.ws), _ptr(addr), _ptr(scale),
                                         _ptr(counts), _stream_handle(self.device))
        _lib.check(rc, "sas_debug_lists")
        return addr, scale, counts

    def run_attend_timed(self, start: torch.cuda.Event, stop: torch.cuda.Event,
                         stamps: Optional[torch.Tensor] = None):
        """The attention stage alone (the dispatch as the forward launches it), its
        dispatch recording its own start and end into the two events (created with
        ``enable_timing=True``) and, with ``stamps`` (int64 [2] on the device,
        filled with {-1, 0}: read as unsigned), its span on the GPU's 100 MHz
        real-time counter."""
        stream = torch.cuda.current_stream(self.device)
        for e in (start, stop):  # torch creates the underlying event on first record
            if not e.cuda_event:
                e.record(stream)
        rc = _lib.load().sas_attend_timed(
            ctypes.byref(self.params), ctypes.byref(self.tensors), _ptr(self.plan), _ptr(self.ws),
            self.ws.numel(), _stream_handle(self.device), ctypes.c_void_p(start.cuda_event),
            ctypes.c_void_p(stop.cuda_event), _ptr(stamps))
        _lib.check(rc, "sas_attend_timed")

    def backward_buffers(self, kv_grad: bool = False) -> dict:
        """Device buffers of one backward call: ``dq [T, H, d_qk]`` and ``dsinks
        [H]`` (fp32), the backward workspace, and with ``kv_grad`` the pools'
        gradients (fp32, laid out like the pools over zeroed storage: the kernel
        adds into them and never touches a padded stride's padding)."""
        lib = _lib.load()
        p = self.params
        T, H = p.total_tokens, p.num_heads_q
        dev = self.device
        need = ctypes.c_size_t()
        _lib.check(lib.sas_backward_workspace_size_for(ctypes.byref(p), int(kv_grad), ctypes.byref(need)),
                   "sas_backward_workspace_size_for")

        def pool_grad(pool):
            n = 1 + sum((d - 1) * st for d, st in zip(pool.shape, pool.stride()))
            return torch.zeros(n, dtype=torch.float32, device=dev).as_strided(pool.shape,
                                                                               pool.stride())

        bufs = dict(dq=torch.empty((T, H, p.head_dim_qk), dtype=torch.float32, device=dev),
                    dsinks=torch.empty(H, dtype=torch.float32, device=dev),
                    ws=torch.empty(int(need.value), dtype=torch.uint8, device=dev),
                    d_ori=None, d_cmp=None)
        if kv_grad:
            bufs["d_ori"] = pool_grad(self.ori_kv)
            if p.scenario >= 2 and self.cmp_kv is not None:
                bufs["d_cmp"] = pool_grad(self.cmp_kv)
        return bufs

    def backward_into(self, dout: torch.Tensor, dlse: Optional[torch.Tensor], bufs: dict) -> None:
        """One backward call into ``bufs`` (from :meth:`backward_buffers`); ``dout``
        ``[T, H, d_v]`` in the query dtype and ``dlse`` ``[T, H]`` fp32 (or None),
        contiguous on the device.  The pools' gradients are added to what the
        buffers hold."""
        rc = _lib.load().sas_backward(
            ctypes.byref(self.params), ctypes.byref(self.tensors), _ptr(self.plan), _ptr(dout),
            _ptr(dlse), _ptr(bufs["dq"]), _ptr(bufs["dsinks"]), _ptr(bufs["d_ori"]),
            _ptr(bufs["d_cmp"]), _ptr(bufs["ws"]), bufs["ws"].numel(), _stream_handle(self.device))
        _lib.check(rc, "sas_backward")

    def backward(self, dout: torch.Tensor, dlse: Optional[torch.Tensor] = None,
                 kv_grad: bool = False):
        """Gradients of the last forward run through this launch (its out / lse hold
        that call's results) for ``dout = dL/dout`` ``[T, H, d_v]`` (and optionally
        ``dlse = dL/dlse`` ``[T, H]``): ``(dq [T, H, d_qk] fp32, dsinks [H] fp32)``,
        and with ``kv_grad`` also ``(d_ori_kv, d_cmp_kv)``: fp32 tensors with the
        pools' shapes and strides (``d_cmp_kv`` None in scenario 1)."""
        p = self.params
        T, H = p.total_tokens, p.num_heads_q
        dev = self.device
        q_dt = torch.bfloat16 if p.q_dtype == _lib.DT_BF16 else torch.float16
        g = dout.to(device=dev, dtype=q_dt).reshape(T, H, p.head_dim_v).contiguous()
        gl = None if dlse is None else dlse.to(device=dev, dtype=torch.float32).reshape(T, H).contiguous()
        bufs = self.backward_buffers(kv_grad)
        # The workspace (the spill: up to 2 GiB and more) and the converted gradients go back to
        # the allocator here, which hands them on in stream order; kept on the launch, every
        # layer of a model would hold its own until its graph is released.
        self.backward_into(g, gl, bufs)
        if kv_grad:
            return bufs["dq"], bufs["dsinks"], bufs["d_ori"], bufs["d_cmp"]
        return bufs["dq"], bufs["dsinks"]

    def drop_workspace(self):
        """Release the forward workspace (a later run or debug read needs a new
        launch); the tensors the pointers refer to stay alive."""
        self._keep = [x for x in self._keep if x is not self.ws]
        self.ws = None

    def run(self, stage: str = "forward"):
        lib = _lib.load()
        fn = getattr(lib, f"sas_{stage}")
        rc = fn(ctypes.byref(self.params), ctypes.byref(self.tensors), _ptr(self.plan),
                _ptr(self.ws), self.ws.numel(), _stream_handle(self.device))
        if rc:
            _lib.check(rc, f"sas_{stage}")


def build_launch(
    *,
    q_flat: torch.Tensor,
    ori_kv: torch.Tensor,
    ori_block_table: torch.Tensor,
    cmp_kv: Optional[torch.Tensor],
    cmp_block_table: Optional[torch.Tensor],
    cmp_indices: Optional[torch.Tensor],
    q_prefix: torch.Tensor,
    act_q_lens: torch.Tensor,
    seqused_kv: torch.Tensor,
    sinks: torch.Tensor,
    metadata: Optional[torch.Tensor],
    scenario: int,
    topk: int,
    cmp_ratio: int,
    ori_win_left: int,
    softmax_scale: float,
    core_num: int,
    ori_kv_scale: Optional[torch.Tensor] = None,
    cmp_kv_scale: Optional[torch.Tensor] = None,
    out: Optional[torch.Tensor] = None,
    lse: Optional[torch.Tensor] = None,
    units_per_cu: int = 0,
    host_lens=None,
) -> Tuple[SasLaunch, torch.Tensor, torch.Tensor]:
    """Validate, convert and lay out one call; returns (launch, out, lse).
    host_lens: the call's (q_prefix, act_q) on the host where the caller has them (or
    a function that returns them), for the check of a recorded plan (q_prefix /
    act_q_lens given as CPU tensors serve as well)."""
    lib = _lib.load()
    dev = q_flat.device
    if dev.type != "cuda":
        raise ValueError("sparse_attn_sharedkv runs on the GPU: q must be a device tensor")
    T, N1, D = q_flat.shape
    q_code = _torch_to_sas_dtype(q_flat.dtype)
    kv_code = _kv_dtype_code(ori_kv, q_code)
    q_flat = q_flat.contiguous()
    if ori_kv.device != dev:
        ori_kv = ori_kv.to(dev)
    obs, ors = _paged_strides(ori_kv, D, "ori_kv")
    ori_bt = _dev_i32(ori_block_table, dev)
    keep = [q_flat, ori_kv, ori_bt]
    cmp_bt = idx = None
    cmp_block_num = cmp_block_size = cmp_table_len = 1
    cbs = crs = D
    if scenario >= 2:
        if cmp_kv.device != dev:
            cmp_kv = cmp_kv.to(dev)
        if _kv_dtype_code(cmp_kv, q_code) != kv_code:
            raise ValueError("ori_kv and cmp_kv must share a dtype")
        cbs, crs = _paged_strides(cmp_kv, D, "cmp_kv")
        cmp_bt = _dev_i32(cmp_block_table, dev)
        cmp_block_num, cmp_block_size = cmp_kv.shape[0], cmp_kv.shape[1]
        cmp_table_len = cmp_bt.shape[1]
        keep += [cmp_kv, cmp_bt]
    else:
        cmp_kv = None
    if scenario == 3:
        idx = _dev_i32(cmp_indices, dev).reshape(T, -1)
        keep.append(idx)
    # scenario 3: index slots per token; scenario 2: capacity of the per-token list
    # of causally valid compressed rows -- the rows the block table covers
    slots = topk if scenario == 3 else (cmp_table_len * cmp_block_size if scenario == 2 else 0)
    # (the fields in the structure's order: one call instead of one per field)
    p = SasParams(q_prefix.numel(), T, N1, ori_kv.shape[2], D, 512,
                  ori_kv.shape[0], ori_kv.shape[1], ori_bt.shape[1],
                  cmp_block_num, cmp_block_size, cmp_table_len, obs, ors, cbs, crs,
                  slots, cmp_ratio, scenario, ori_win_left, 0, 4, 3, q_code, kv_code,
                  float(softmax_scale), int(core_num), int(units_per_cu))
    sizes = (ctypes.c_int64 * 3)()  # balance target, plan entries, workspace bytes
    rc = lib.sas_call_sizes(ctypes.byref(p), sizes)
    if rc:
        if rc == -6:  # heads: the reference raises ValueError for unsupported N1/N2 (api.py:279-282)
            raise ValueError(f"num_heads_kv must be 1 and num_heads_q in [1, 128] "
                             f"(got N1={N1}, N2={p.num_heads_kv}, D={D})")
        if rc == -2 and D not in (512, 576):
            raise ValueError(f"head_dim must be 512 or 576 (got {D})")
        _lib.check(rc, "sparse_attn_sharedkv")

    if host_lens is None and q_prefix.device.type == "cpu" and act_q_lens.device.type == "cpu":
        host_lens = (q_prefix, act_q_lens)
    qp = _dev_i32(q_prefix, dev)
    aq = _dev_i32(act_q_lens, dev)
    skv = _dev_i32(seqused_kv, dev)
    snk = _dev_f32(sinks, dev)
    if snk.numel() != N1:
        raise ValueError(f"sinks must have {N1} entries (got {snk.numel()})")
    keep += [qp, aq, skv, snk]
    osc = csc = None
    if kv_code == _lib.DT_FP8E4M3:
        if ori_kv_scale is None or (scenario >= 2 and cmp_kv_scale is None):
            raise ValueError("float8 KV needs ori_kv_scale (and cmp_kv_scale)")
        osc = _dev_f32(ori_kv_scale, dev)
        keep.append(osc)
        if scenario >= 2:
            csc = _dev_f32(cmp_kv_scale, dev)
            keep.append(csc)
    if out is None:
        out = torch.empty((T, N1, 512), dtype=q_flat.dtype, device=dev)
    if lse is None:
        lse = torch.empty((T, N1), dtype=torch.float32, device=dev)
    keep += [out, lse]

    plan = None
    if metadata is not None:
        n = metadata.numel()
        if n != SAS_META_SIZE:  # anything but the reference table must be our plan
            assert n == sizes[1], (
                f"metadata must have {SAS_META_SIZE} int32 entries (reference table) or "
                f"{sizes[1]} (split-KV plan for these shapes); got {n}")
            _check_plan_record(metadata, p, host_lens, sizes[0])
            plan = _dev_i32(metadata, dev)
            keep.append(plan)
    ws = torch.empty(sizes[2], dtype=torch.uint8, device=dev)
    keep.append(ws)

    t = SasTensors(
        q_flat.data_ptr(), ori_kv.data_ptr(), ori_bt.data_ptr(),
        None if cmp_kv is None else cmp_kv.data_ptr(), None if cmp_bt is None else cmp_bt.data_ptr(),
        None if idx is None else idx.data_ptr(), qp.data_ptr(), aq.data_ptr(), skv.data_ptr(),
        snk.data_ptr(), None if osc is None else osc.data_ptr(),
        None if csc is None else csc.data_ptr(), out.data_ptr(), lse.data_ptr())
    launch = SasLaunch(p, t, keep, plan, ws, dev)
    launch.ori_kv, launch.cmp_kv = ori_kv, cmp_kv
    return launch, out, lse


def _get_kernel(
    *,
    batch: int,
    max_seq: int,
    total_tokens: int,
    ori_block_num: int,
    ori_block_size: int,
    ori_table_len: int,
    cmp_block_num: int,
    cmp_block_size: int,
    cmp_table_len: int,
    n_heads: int,
    n_kv_heads: int,
    head_dim: int,
    topk_cmp: int,
    cmp_ratio: int,
    scenario: int,
    ori_win_left: int,
    softmax_scale: float,
    dtype: str,
    core_num: int,
):
    """The reference's compile-cache lookup (api.py:59-126).  HIP kernels are
    compiled ahead of time, so this only validates and caches the static
    parameters and returns ``func(11 tensors) -> (out, lse)`` with the
    reference kernel's argument order (api.py:372-384)."""
    key = (batch, max_seq, total_tokens, ori_block_num, ori_block_size, ori_table_len,
           cmp_block_num, cmp_block_size, cmp_table_len, n_heads, n_kv_heads, head_dim,
           topk_cmp, cmp_ratio, scenario, ori_win_left, round(softmax_scale, 8), dtype, core_num)
    fn = _KERNEL_CACHE.get(key)
    if fn is None:
        if dtype not in ("bfloat16", "float16"):
            raise ValueError(f"dtype must be bfloat16 or float16, got {dtype!r}")
        assert scenario in (1, 2, 3), "scenario must be 1 (SWA), 2 (CFA) or 3 (SCFA)"
        assert n_kv_heads == 1, "API constraint: n_kv_heads must be 1"
        assert head_dim in (512, 576), "API constraint: head_dim must be 512 or 576"
        assert topk_cmp >= 0
        assert batch > 0 and total_tokens > 0
        fn = _SasKernelFunc(scenario=scenario, topk=topk_cmp, cmp_ratio=cmp_ratio,
                            ori_win_left=ori_win_left, softmax_scale=softmax_scale,
                            core_num=core_num)
        _KERNEL_CACHE[key] = fn
    return fn


class _SasKernelFunc:
    """``func(Q, ori_KV, ori_block_table, cmp_KV, cmp_block_table, cmp_indices,
    q_prefix, actual_q_len, actual_kv_len, Sinks, Metadata) -> (Output, LSE)``."""

    def __init__(self, **static):
        self.static = static

    def __call__(self, Q, ori_KV, ori_block_table, cmp_KV, cmp_block_table, cmp_indices,
                 q_prefix, actual_q_len, actual_kv_len, Sinks, Metadata):
        s = self.static
        launch, out, lse = build_launch(
            q_flat=Q, ori_kv=ori_KV, ori_block_table=ori_block_table,
            cmp_kv=cmp_KV if s["scenario"] >= 2 else None,
            cmp_block_table=cmp_block_table if s["scenario"] >= 2 else None,
            cmp_indices=cmp_indices if s["scenario"] == 3 else None,
            q_prefix=q_prefix, act_q_lens=actual_q_len, seqused_kv=actual_kv_len, sinks=Sinks,
            metadata=Metadata, scenario=s["scenario"], topk=s["topk"],
            cmp_ratio=s["cmp_ratio"], ori_win_left=s["ori_win_left"],
            softmax_scale=s["softmax_scale"], core_num=s["core_num"])
        launch.run()
        return out, lse


class _SharedKVAttention(torch.autograd.Function):
    """Autograd of the operator for the queries, the sinks and the two KV pools:
    the forward is one launch; the backward runs ``sas_backward`` on the same launch
    (same plan and row lists) with the saved out / lse."""

    @staticmethod
    def forward(ctx, q_flat, sinks, ori_kv, cmp_kv, spec):
        launch, out, lse = build_launch(
            q_flat=q_flat.detach(), sinks=sinks.detach(), ori_kv=ori_kv.detach(),
            cmp_kv=None if cmp_kv is None else cmp_kv.detach(), **spec)
        launch.run()
        # The backward plans and resolves in a workspace of its own: the forward's is
        # released now (stream-ordered, so the kernels above still own it).
        launch.drop_workspace()
        # The backward reads these through the launch's raw pointers: saving them
        # lets autograd refuse a backward after any of them changed in place.
        ctx.save_for_backward(q_flat, sinks, ori_kv, cmp_kv, out, lse)
        ctx.launch = launch
        ctx.q_dtype, ctx.sinks_dtype = q_flat.dtype, sinks.dtype
        ctx.kv_dtype = ori_kv.dtype
        return out, lse

    @staticmethod
    def backward(ctx, dout, dlse):
        ctx.saved_tensors  # noqa: B018 -- raises if a saved tensor was modified in place
        T, H = ctx.launch.params.total_tokens, ctx.launch.params.num_heads_q
        if dout is None:
            dout = torch.zeros((T, H, 512), dtype=ctx.q_dtype, device=ctx.launch.device)
        kv = ctx.needs_input_grad[2] or ctx.needs_input_grad[3]
        res = ctx.launch.backward(dout, dlse, kv_grad=kv)
        dq, dsinks = res[0], res[1]
        d_ori = res[2] if kv and ctx.needs_input_grad[2] else None
        d_cmp = res[3] if kv and ctx.needs_input_grad[3] and res[3] is not None else None
        return (dq.to(ctx.q_dtype) if ctx.needs_input_grad[0] else None,
                dsinks.to(ctx.sinks_dtype) if ctx.needs_input_grad[1] else None,
                None if d_ori is None else d_ori.to(ctx.kv_dtype),
                None if d_cmp is None else d_cmp.to(ctx.kv_dtype), None)


def sparse_attn_sharedkv(
    q: torch.Tensor,
    *,
    ori_kv: torch.Tensor,
    cmp_kv: Optional[torch.Tensor] = None,
    cmp_sparse_indices: Optional[torch.Tensor] = None,
    ori_block_table: torch.Tensor,
    cmp_block_table: Optional[torch.Tensor] = None,
    cu_seqlens_q: Optional[torch.Tensor] = None,
    seqused_q: Optional[torch.Tensor] = None,
    seqused_kv: torch.Tensor,
    sinks: torch.Tensor,
    metadata: Optional[torch.Tensor] = None,
    softmax_scale: float,
    cmp_ratio: Optional[int] = None,
    ori_mask_mode: int = 4,
    cmp_mask_mode: int = 3,
    ori_win_left: int = 127,
    ori_win_right: int = 0,
    layout_q: str = "TND",
    layout_kv: str = "PA_ND",
    return_softmax_lse: bool = False,
    core_num: int = DEFAULT_CORE_NUM,
    topk_cmp: Optional[int] = None,
    ori_kv_scale: Optional[torch.Tensor] = None,
    cmp_kv_scale: Optional[torch.Tensor] = None,
) -> Union[torch.Tensor, Tuple[torch.Tensor, torch.Tensor]]:
    """Forward pass; returns ``attention_out`` in the layout of ``q`` (and the
    fp32 LSE with the sink folded in when ``return_softmax_lse``).  When ``q`` or
    ``sinks`` requires grad, the call is differentiable for them (the backward is
    an extension: the reference has none).

    Scenario by optional inputs (api.py:156-160, 196-202): no ``cmp_kv`` -> SWA
    (1); ``cmp_kv`` without ``cmp_sparse_indices`` -> CFA (2); both -> SCFA (3).
    ``seqused_q`` is accepted for API parity and unused, as in the reference.
    """
    del seqused_q
    assert ori_mask_mode == 4, "only ori_mask_mode=4 supported"
    assert cmp_mask_mode == 3 or cmp_kv is None, "only cmp_mask_mode=3 supported"
    assert ori_win_right == 0, "only ori_win_right=0 supported"
    assert layout_kv == "PA_ND", "only layout_kv=PA_ND supported"
    assert layout_q in ("TND", "BSND"), f"unsupported layout_q={layout_q!r}"
    _torch_to_sas_dtype(q.dtype)
    dev = q.device

    if cmp_kv is None:
        scenario = 1
    elif cmp_sparse_indices is None:
        scenario = 2
    else:
        scenario = 3

    # the query layout on the host where it is known there without a device sync
    # (for the check of a recorded plan)
    cu_host = None
    if cu_seqlens_q is not None and cu_seqlens_q.device.type == "cpu":
        cu_host = cu_seqlens_q.to(torch.int64).reshape(-1)
    host_lens = None
    grad = torch.is_grad_enabled() and any(
        x is not None and x.requires_grad for x in (q, sinks, ori_kv, cmp_kv))
    # without a gradient the forward takes the sequences' cumulative ends as they are
    # (sas_forward_cu): no kernel to form their lengths
    ends = False
    if layout_q == "TND":
        assert cu_seqlens_q is not None, "cu_seqlens_q is required for TND"
        cu = _dev_i32(cu_seqlens_q, dev)
        B = cu.numel() - 1
        T = q.shape[0]
        q_flat = q
        q_prefix = cu[:-1]
        ends = not grad
        act_q = cu[1:] if ends else cu[1:] - cu[:-1]
        idx = cmp_sparse_indices if scenario == 3 else None
        if cu_host is not None:
            host_lens = (cu_host[:-1], cu_host[1:] - cu_host[:-1])
    else:
        B, S, N1, D = q.shape
        T = B * S
        q_flat = q.reshape(T, N1, D)
        if cu_seqlens_q is not None:
            q_prefix = torch.arange(B, dtype=torch.int32, device=dev) * S
            cu = _dev_i32(cu_seqlens_q, dev)
            act_q = cu[1:] - cu[:-1]
            if cu_host is not None:
                host_lens = (torch.arange(B, dtype=torch.int64) * S, cu_host[1:] - cu_host[:-1])
        else:
            if grad:
                q_prefix = torch.arange(B, dtype=torch.int32, device=dev) * S
                act_q = torch.full((B,), S, dtype=torch.int32, device=dev)
            else:
                cu = torch.arange(B + 1, dtype=torch.int32, device=dev) * S
                q_prefix, act_q, ends = cu[:-1], cu[1:], True
            host_lens = lambda: (torch.arange(B, dtype=torch.int64) * S,  # noqa: E731
                                 torch.full((B,), S, dtype=torch.int64))
        idx = None
        if scenario == 3:
            ci = cmp_sparse_indices
            idx = ci.reshape(T, ci.shape[2], ci.shape[3])

    K = 0
    if scenario == 3:
        N2 = idx.shape[1]
        K = topk_cmp if topk_cmp is not None else idx.shape[2]
        assert K == idx.shape[2], "topk_cmp does not match cmp_sparse_indices last dim"
        if N2 != 1:
            raise ValueError(f"only N2=1 supported (got N2={N2})")
    cmp_ratio_eff = cmp_ratio if cmp_ratio is not None else 4

    spec = dict(
        ori_block_table=ori_block_table, cmp_block_table=cmp_block_table, cmp_indices=idx,
        q_prefix=q_prefix, act_q_lens=act_q, seqused_kv=seqused_kv,
        metadata=metadata, scenario=scenario, topk=K, cmp_ratio=cmp_ratio_eff,
        ori_win_left=ori_win_left, softmax_scale=softmax_scale, core_num=core_num,
        ori_kv_scale=ori_kv_scale, cmp_kv_scale=cmp_kv_scale, host_lens=host_lens)
    if grad:
        if ori_kv.dtype == torch.float8_e4m3fn:
            raise NotImplementedError("the backward supports 16-bit KV pools only")
        out, lse = _SharedKVAttention.apply(q_flat, sinks, ori_kv, cmp_kv, spec)
    else:
        launch, out, lse = build_launch(q_flat=q_flat, sinks=sinks, ori_kv=ori_kv, cmp_kv=cmp_kv,
                                        **spec)
        launch.run("forward_cu" if ends else "forward")

    if layout_q == "BSND":
        out = out.reshape(B, S, out.shape[1], out.shape[2])
        lse = lse.reshape(B, S, lse.shape[1])
    if return_softmax_lse:
        return out, lse
    return out
