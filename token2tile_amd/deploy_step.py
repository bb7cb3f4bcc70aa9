"""Token2Tile attention operator on MI355X: one sparse attention call.

Drop-in counterpart of ``token2tile/operator/deploy_step.py``: same module
surface (``MaskedStepDeploy``, ``online_u``, ``fast_assign``, ``fast_gather``),
same constructor, ``init_state`` / ``set_cfg_call`` / ``reset_cfg_reuse`` /
``step`` semantics, same snapshot reuse rules.  Every stage runs in the HIP
library (``libt2t_hip.so``); there is no CPU path.

``step(q, k, v, state)`` for q, k, v of shape [H, N, 128] (fp16, or bf16 -
the model dtype, accepted without a conversion pass):

  1. projection   QU = q Uq, KU = k Uk                       t2t_project
  2. clustering   one warm-started k-means update            t2t_kmm_run
  3. scoring      gl = QU cks^T                              t2t_score
  4. selection    per-query budget prefix + cluster union    t2t_select_run_packed
  5. attention    task plan, then one fused kernel: exact
                  attention over the unions, residual over
                  the other clusters, merge                  t2t_tile_plan,
                                                             t2t_tile_attn_run_planned

The output is in the original row order.  With ``mask_refresh=R`` the
structure (labels, permutations, sizes, centroids, union, task plan) is
rebuilt every R annotated steps and reused in between (deploy_step.py:296-316).
"""
from __future__ import annotations

import ctypes
import math
import threading
from contextlib import nullcontext

import torch

from . import _lib, ops
from .ops import fast_gather  # noqa: F401  (module surface of the reference)

__all__ = ["MaskedStepDeploy", "online_u", "fast_assign", "fast_gather", "fused_update_vstats"]


# ---------------------------------------------------------------------------
# low-rank space (deploy_step.py:104-149)
# ---------------------------------------------------------------------------

def _eigh_robust(M):
    """Batched symmetric eigendecomposition on M's device.  The device solver
    can fail to converge on nearly singular Grams, where the host LAPACK
    succeeds, so a failure is retried once on the host (the reference falls
    back the same way, deploy_step.py:104-111)."""
    if M.device.type == "cpu":
        return torch.linalg.eigh(M)
    try:
        return torch.linalg.eigh(M)
    except RuntimeError:                    # torch.linalg.LinAlgError derives from it
        return tuple(t.to(M.device) for t in torch.linalg.eigh(M.cpu()))


def _require_finite(**tensors):
    """Raise RuntimeError naming the heads of any input holding inf / NaN."""
    for name, t in tensors.items():
        per_head = torch.isfinite(t).logical_not_().flatten(1).sum(1)
        if bool(per_head.any()):
            heads = per_head.nonzero().flatten().tolist()
            raise RuntimeError(f"online_u: {name} {tuple(t.shape)} holds "
                               f"{int(per_head.sum())} non-finite values, in heads {heads}")


_EIG_FLOOR = 1e-8   # least Gram eigenvalue of the fit (smaller ones are raised to it)


def _fit_eigh(Mq, Mk, r):
    """The fit from the symmetric square roots of the Grams, eigenvalues below
    the floor raised to it: M = Rq Rk, whose top-r singular pairs come from the
    eigendecomposition of M^T M (U_r = M V_r / s_r)."""
    eq, Vq = _eigh_robust(Mq)
    ek, Vk = _eigh_robust(Mk)
    eq, ek = eq.clamp_min(_EIG_FLOOR), ek.clamp_min(_EIG_FLOOR)
    Rq = Vq @ (eq.sqrt().unsqueeze(-1) * Vq.transpose(1, 2))
    Rk = Vk @ (ek.sqrt().unsqueeze(-1) * Vk.transpose(1, 2))
    Rqi = Vq @ (eq.rsqrt().unsqueeze(-1) * Vq.transpose(1, 2))
    Rki = Vk @ (ek.rsqrt().unsqueeze(-1) * Vk.transpose(1, 2))
    M = Rq.transpose(1, 2) @ Rk
    w, V = _eigh_robust(M.transpose(1, 2) @ M)          # ascending eigenvalues
    Vr = V[:, :, -r:].flip(-1)
    sr = w[:, -r:].flip(-1).clamp_min(1e-30).sqrt()
    Ur = (M @ Vr) / sr.unsqueeze(1)
    root = sr.sqrt().unsqueeze(1)
    return (Rqi.transpose(1, 2) @ Ur) * root, (Rki @ Vr) * root


def _fit_chol(Mq, Mk, L, r):
    """The same fit where every Gram eigenvalue is above the floor.  Any factor
    of a Gram serves as its root: with Mk = L L^T and Mq = F F^T, M = F^T L has
    the singular values of Rq Rk and M^T M = L^T Mq L, so one eigensolution is
    left: Uq = F^-T U S^1/2 = L V S^-1/2 and Uk = L^-T V S^1/2.  (Uk also equals
    Mq L V S^-3/2, but the eigensolver's absolute noise in V, about the machine
    epsilon of the largest S, grows without bound there where S is small: inputs
    of few effective dimensions beside one large channel left fp16's range.)"""
    w, V = _eigh_robust(torch.bmm(L.transpose(1, 2).contiguous(), torch.bmm(Mq, L)))
    Vr = V[:, :, -r:].flip(-1).contiguous()
    sr = w[:, -r:].flip(-1).clamp_min(1e-30).sqrt().unsqueeze(1)
    Uk = torch.linalg.solve_triangular(L.transpose(1, 2), Vr, upper=True) * sr.sqrt()
    return torch.bmm(L, Vr) * sr.rsqrt(), Uk


def _fit_heads(Mq, Mk, L, low, r):
    """_fit_chol, and _fit_eigh for the heads ``low`` whose Grams have eigenvalues
    at the floor.  Those heads' places in the batch hold unit matrices, so what
    the others get does not depend on them."""
    if len(low) == Mq.shape[0]:
        return _fit_eigh(Mq, Mk, r)
    if not low:
        return _fit_chol(Mq, Mk, L, r)
    idx = torch.tensor(low, device=Mq.device)
    unit = torch.eye(Mq.shape[1], dtype=Mq.dtype, device=Mq.device).expand(len(low), -1, -1)
    fits = _fit_chol(*(M.index_copy(0, idx, unit) for M in (Mq, Mk, L)), r)
    return tuple(U.index_copy(0, idx, E) for U, E in zip(fits, _fit_eigh(Mq[idx], Mk[idx], r)))


def online_u(qf, kf, r=32):
    """Matched rank-r projections Uq, Uk [H, D, r] (fp32) minimising
    ||Q K^T - (Q Uq)(K Uk)^T||_F (deploy_step.py:122-149).

    The Gram matrices come from the HIP fp64 Gram kernel (16-bit inputs, read
    in place) or from fp64 matmul for fp32 inputs; the 128 x 128 problems run
    batched in fp64 on the GPU: a Cholesky factor and one symmetric
    eigensolution (_fit_chol), or three eigensolutions for the heads where a
    Gram has eigenvalues at the floor (_fit_eigh).  The reference backend's fast
    initialisation eigensolves in the same way (t2t_attn.py:211-239): a
    batched symmetric eigensolver is two orders of magnitude faster here than
    a batched SVD.  Raises RuntimeError on non-finite input."""
    half = (torch.float16, torch.bfloat16)
    if not (qf.is_cuda and kf.is_cuda and qf.dtype in half and kf.dtype in half
            and qf.shape[0] == kf.shape[0]):
        _require_finite(q=qf, k=kf)

        def gram(x):
            if x.dtype in half:
                return ops.gram(x.contiguous())
            xd = x.double()
            return xd.transpose(1, 2) @ xd / x.shape[1]

        Uq, Uk = _fit_eigh(gram(qf), gram(kf), r)
        return Uq.float().contiguous(), Uk.float().contiguous()

    H = qf.shape[0]
    rows = lambda x: x if x.stride(2) == 1 and x.stride(1) >= x.shape[2] else x.contiguous()  # noqa: E731
    # heads with non-finite q / k, heads with a small eigenvalue of Mq / Mk:
    # read back together
    flags = torch.empty(4, H, dtype=torch.int32, device=qf.device)
    Mq = ops.gram_strided(rows(qf), flags[0])
    Mk = ops.gram_strided(rows(kf), flags[1])
    L = ops.fit_chol(Mq, Mk, _EIG_FLOOR, flags[2:])
    bad_q, bad_k, small_q, small_k = flags.tolist()
    if any(bad_q) or any(bad_k):
        _require_finite(q=qf, k=kf)
    Uq, Uk = _fit_heads(Mq, Mk, L, [h for h in range(H) if small_q[h] or small_k[h]], r)
    return Uq.float().contiguous(), Uk.float().contiguous()


def fast_assign(x, centroids, out=None, **_tuning):
    """Nearest centroid (lowest index on ties), [H, N] int32
    (fast_assign.py:79-106).  Tuning keywords of the reference are accepted
    and ignored."""
    return ops.fast_assign_labels(x.contiguous(), centroids.contiguous(), out=out)


def fused_update_vstats(ku, labels, old_centroids, v=None, *, BLOCK_N=32, num_warps=2,
                        return_fp32=False):
    """One pass producing new centroids [H, C, DK], counts [H, C] int32 and,
    when ``v`` is given, the per-cluster mean values [H, C, DV]
    (fused_update_vstats.py:72-115).  Sums are fp32; an empty cluster keeps
    its old centroid and has a zero mean value.  Outputs are cast to the
    dtype of ku / v unless ``return_fp32``.  ``BLOCK_N`` and ``num_warps``
    are the reference's Triton tuning knobs: accepted and ignored."""
    del BLOCK_N, num_warps
    if ku.dim() != 3 or ku.shape[2] != 32:
        raise ValueError(f"fused_update_vstats: ku must be [H, N, 32] (the rank-32 space the "
                         f"HIP kernel is built for), got {tuple(ku.shape)}")
    if v is not None and (v.dim() != 3 or v.shape[2] != 128 or v.shape[:2] != ku.shape[:2]):
        raise ValueError(f"fused_update_vstats: v must be [H, N, 128] beside ku "
                         f"{tuple(ku.shape)}, got {tuple(v.shape)}")
    cent, counts, vmean = ops.fused_update_vstats(
        ku.contiguous(), labels.to(torch.int32).contiguous(), old_centroids.contiguous(),
        None if v is None else v.contiguous(), half=not return_fp32)
    return cent, counts, vmean


# ---------------------------------------------------------------------------
# the operator
# ---------------------------------------------------------------------------

class MaskedStepDeploy:
    """Persistent buffers and kernels for one (H, N, C_Q) attention shape.

    s_frac: per-query token budget as a fraction of N (``ns_t`` holds the token
        count on the device and may be overwritten between calls).
    mask_refresh: rebuild the structure every this many annotated steps.
    cfg_reuse: structure reuse across CFG branches even when mask_refresh is 1.
    pin_tail: the last pin_tail keys form one reserved key cluster that every
        query executes exactly.
    split_cap: accepted for interface compatibility; the HIP selection kernel
        balances rows per wave whatever the query-cluster sizes, so the split
        and unsplit variants are the same launch.
    (deploy_step.py:152-242)
    """

    def __init__(self, H, N, CQ, *, C=2048, D=128, r=32, s_frac=0.05, tailw=1.0, device="cuda",
                 mask_refresh=1, cfg_reuse=False, pin_tail=0, split_cap="auto"):
        if C != 2048 or D != 128:
            raise ValueError("the kernels require C=2048 and D=128")
        if r != 32:
            raise ValueError("the kernels require r=32")
        if not (1 <= CQ <= 4096):
            raise ValueError("CQ must be in [1, 4096]")
        if N >= 524288:
            raise ValueError("the selection packing requires N < 524288")
        if N < C or N < CQ:
            raise ValueError(f"N={N} tokens cannot seed {C} key clusters and {CQ} query clusters")
        self.H, self.N, self.CQ, self.C, self.D, self.r = H, N, CQ, C, D, r
        self.ns = max(1, int(s_frac * N))
        self.tailw = tailw
        self.dev = dev = torch.device(device)
        if dev.type != "cuda":
            raise ValueError("MaskedStepDeploy runs on a ROCm GPU device")
        self.scale = 1.0 / math.sqrt(D)
        self.pin_tail = int(pin_tail)
        if not (0 <= self.pin_tail <= N):
            raise ValueError("pin_tail must be in [0, N]")
        self.split_cap = 0 if split_cap in ("auto", None, 0) else int(split_cap)
        ops._lib.lib()  # fail loudly now if the HIP library is missing

        f16, f32, i32 = torch.float16, torch.float32, torch.int32
        self.QU = torch.empty(H, N, r, device=dev, dtype=f16)
        self.KU = torch.empty(H, N, r, device=dev, dtype=f16)
        self.klab = torch.empty(H, N, device=dev, dtype=i32)
        self.qlab = torch.empty(H, N, device=dev, dtype=i32)
        self.rowcnt = torch.empty(H, N, device=dev, dtype=i32)
        self._io = {}                 # dtype -> (kp, vp, out, attn workspace)
        self._tile_attn_plan_ints = ops.plan_ints(H, N, CQ)
        self.tailw_t = torch.tensor(float(tailw), device=dev, dtype=f32)
        # the exact-attention kernel reads K through kperm (kp = k[kperm] is
        # not materialised); False restores the reference's separate gather
        self.fuse_k_gather = True
        # ... and V through kperm too, so V_sorted is not materialised either;
        # the value statistics of a reuse call then run on s_side beside the
        # exact attention.  False restores the V_sorted buffer
        self.fuse_v_gather = True
        self._kmm_ck2 = torch.empty(H, C, r, device=dev, dtype=f32)
        self._kmm_kcounts = torch.empty(H, C, device=dev, dtype=i32)
        self._kmm_sumv = torch.empty(H, C, D, device=dev, dtype=f16)
        self._kmm_lam = torch.empty(H, device=dev, dtype=f32)
        self.ns_t = torch.tensor(self.ns, device=dev, dtype=i32)
        self._ws_kmm = torch.empty(ops.kmm_ws_bytes(H, N, CQ, C), dtype=torch.uint8, device=dev)
        self._ws_vst = torch.empty(ops.vstats_ws_bytes(H, N, C), dtype=torch.uint8, device=dev)
        self._ws_sel = torch.empty(ops.select_ws_bytes(H, N, CQ), dtype=torch.uint8, device=dev)
        # attention call scratch: lse of the exact part (sorted order) and the
        # centroid tile image the residual kernel stages from
        self._lse = torch.empty(H, N, dtype=torch.float32, device=dev)
        self._ctiles = torch.empty(ops.size_query("t2t_centroid_tiles_bytes", H), dtype=torch.uint8,
                                   device=dev)

        # fp32 parts of the exact attention of a small call (empty otherwise)
        self._ws_split = torch.empty(ops.attn_split_ws_bytes(H, N, CQ), dtype=torch.uint8, device=dev)

        self.cfg_reuse = bool(cfg_reuse)
        self.mask_refresh = max(1, int(mask_refresh))
        self._cfg_on = self.cfg_reuse or self.mask_refresh > 1
        self._cfg_hold = {}
        self._cfg_parity = None
        self._cfg_key = 0
        self._cfg_step = 0

        # default-priority streams (the two-stream schedule of the reference)
        self.s_main = torch.cuda.Stream(device=dev)
        self.s_side = torch.cuda.Stream(device=dev)
        self._lock = threading.Lock()
        # caller, fork, join, done.  Used once here: an event and a stream's queue
        # are made at their first use (200 us on the first reuse call otherwise)
        self._ev = [torch.cuda.Event() for _ in range(4)]
        for ev in self._ev:
            ev.record(self.s_main)
        self.s_side.wait_event(self._ev[1])
        self._ev[2].record(self.s_side)
        self.last_call_full = None
        # optional list: (stage name, start event, end event) per launch group
        # recorded on s_main, for the benchmark's per-kernel timing
        self.stage_events = None

    def _stage(self, name):
        deploy = self

        class _Ctx:
            def __enter__(self_):
                if deploy.stage_events is not None:
                    self_.a = torch.cuda.Event(enable_timing=True)
                    self_.a.record(deploy.s_main)

            def __exit__(self_, *exc):
                if deploy.stage_events is not None:
                    b = torch.cuda.Event(enable_timing=True)
                    b.record(deploy.s_main)
                    deploy.stage_events.append((name, self_.a, b))
        return _Ctx()

    def _buffers(self, dtype):
        io = self._io.get(dtype)
        if io is None:
            H, N, D = self.H, self.N, self.D
            # kp and vp are allocated on first use: the fused gathers need neither
            io = dict(kp=None, vp=None,
                      out=torch.empty(H, N, D, device=self.dev, dtype=dtype),
                      attn_out=None, lse=None)
            self._io[dtype] = io
        return io

    def _kp(self, dtype):
        io = self._buffers(dtype)
        if io["kp"] is None:
            io["kp"] = torch.empty(self.H, self.N, self.D, device=self.dev, dtype=dtype)
        return io["kp"]

    @property
    def kp(self):
        """The cluster-ordered K buffer; written by ``step`` only when
        ``fuse_k_gather`` is off (the fused kernel reads k through kperm)."""
        return self._kp(torch.float16)

    def _vp(self, dtype):
        io = self._buffers(dtype)
        if io["vp"] is None:
            io["vp"] = torch.empty(self.H, self.N, self.D, device=self.dev, dtype=dtype)
        return io["vp"]

    @property
    def vp(self):
        """The cluster-ordered V buffer (V_sorted); written by ``step`` only
        when a gather is unfused (the fused kernel reads v through kperm)."""
        return self._vp(torch.float16)

    @property
    def _fused_kv(self):
        return self.fuse_k_gather and self.fuse_v_gather

    # -- state init (deploy_step.py:245-266) ---------------------------------
    def init_state(self, q, k, *, warm_iters=4, seed=0):
        """Projections and initial centroids of one layer: the projections are
        kept for the whole request; the centroids warm-start every rebuild.
        Initial centroids are KU / QU rows picked by a seeded CPU randperm
        (the same indices as the reference), then ``warm_iters`` Lloyd
        iterations: nearest centroid (fast_assign) and the fp32 mean update
        of fused_update_vstats, as the reference operator's init_state does
        (deploy_step.py:245-266).  The backend's ``t2t_fast_init`` path keeps
        the deterministic fixed-point update instead (t2t_attn.py:242-281)."""
        N, r = self.N, self.r
        Uq, Uk = online_u(q, k, r)
        Uq = Uq.to(torch.float16).contiguous()
        Uk = Uk.to(torch.float16).contiguous()
        # strided views are read in place where the projection can (16-byte rows)
        rows = lambda x: x if ops.rows_in_place(x) else x.contiguous()  # noqa: E731
        KU = ops.project(rows(k), Uk)
        QU = ops.project(rows(q), Uq)
        g = torch.Generator(device="cpu").manual_seed(seed)
        kidx = torch.randperm(N, generator=g)[: self.C].sort().values.to(self.dev)
        qidx = torch.randperm(N, generator=g)[: self.CQ].sort().values.to(self.dev)
        ck = KU[:, kidx, :].contiguous()
        cq = QU[:, qidx, :].contiguous()
        iters = len(range(warm_iters))
        ops.lloyd(KU, ck, iters)
        ops.lloyd(QU, cq, iters)
        torch.cuda.synchronize(self.dev)
        return {"Uq": Uq, "Uk": Uk, "ck": ck.contiguous(), "cq": cq.contiguous()}

    def set_cfg_call(self, parity, key=0, step=0):
        """Annotate the next step() call (deploy_step.py:268-277)."""
        self._cfg_parity = int(parity)
        self._cfg_key = key
        self._cfg_step = int(step)

    def reset_cfg_reuse(self):
        """Drop all snapshots and any pending annotation (deploy_step.py:279-283)."""
        self._cfg_hold.clear()
        self._cfg_parity = None

    # -- the attention call (deploy_step.py:286-477) -------------------------
    def _launch(self, args, stages, stream):
        """Enqueue a call's stages on ``stream``: in one library call, or one
        per named stage between its two events while stage_events is set."""
        if self.stage_events is None or stream is not self.s_main:
            stages = (("", sum(bits for _, bits in stages)),)
        for name, bits in stages:
            with self._stage(name) if name else nullcontext():
                rc = _lib.lib().t2t_step(args, bits, stream.cuda_stream)
            if rc != 0:
                msg = _lib.lib().t2t_last_error().decode(errors="replace")
                raise RuntimeError(f"t2t_step failed (code {rc}): {msg}")

    def step(self, q, k, v, state, out=None):
        """q, k, v: [H, N, 128] fp16 (or bf16), original row order: contiguous,
        or strided views with contiguous rows, such as token-major [N, H, 128]
        tensors through ``.transpose(0, 1)`` (the kernels read them in place).
        state: dict(Uq, Uk, ck, cq) fp16; ck/cq are replaced by fresh tensors
        holding the centroids that warm-start the next call.  Returns out
        [H, N, 128] in q's dtype: the given ``out`` view (written in place), or
        a buffer reused by the next call.  Under graph capture a rebuilding call
        is recorded; a reuse call raises RuntimeError."""
        # the events and buffers serve one call at a time; the launches, events
        # and the capture query go to this object's GPU whichever is current
        with self._lock, torch.cuda.device(self.dev):
            return self._step(q, k, v, state, out)

    def _own_args(self):
        """A call's arguments that name this object's own settings and buffers, as
        they stand now."""
        H, N = self.H, self.N
        a = _lib.StepArgs()
        a.struct_bytes = ctypes.sizeof(a)
        a.H, a.N, a.CQ, a.CK = H, N, self.CQ, self.C
        a.pin_tail, a.scale = int(self.pin_tail), float(self.scale)
        for name, shape, dtype in (("QU", (H, N, self.r), torch.float16),
                                   ("KU", (H, N, self.r), torch.float16),
                                   ("rowcnt", (H, N), torch.int32), ("qlab", (H, N), torch.int32),
                                   ("klab", (H, N), torch.int32)):
            t = getattr(self, name)
            ops._check(t, shape, dtype, name, self.dev)
            setattr(a, name, t.data_ptr())
        for name, t in (("ck2", self._kmm_ck2), ("sumv", self._kmm_sumv), ("lam", self._kmm_lam),
                        ("tiles", self._ctiles), ("lse", self._lse)):
            setattr(a, name, t.data_ptr())
        for name in ("ws_kmm", "ws_vst", "ws_sel", "ws_split"):
            t = getattr(self, "_" + name)
            setattr(a, name, t.data_ptr())
            setattr(a, name + "_bytes", t.numel())
        return a

    def _step(self, q, k, v, state, out):
        H, N, C, CQ, D = self.H, self.N, self.C, self.CQ, self.D
        if not (q.dtype == k.dtype == v.dtype) or q.dtype not in (torch.float16, torch.bfloat16):
            raise TypeError("step: q, k, v must share dtype fp16 or bf16")
        a = self._own_args()
        a.dtype = _lib.dtype_code(q.dtype)
        io = self._buffers(q.dtype)
        dst = io["out"] if out is None else out
        for name, t in (("q", q), ("k", k), ("v", v), ("out", dst)):
            try:
                sh, sn = ops._rows(t, H, N, D, q.dtype, name, self.dev)
            except ValueError as e:
                raise ValueError(f"step: {e}") from None
            setattr(a, name, t.data_ptr())
            setattr(a, name + "_head_stride", sh)
            setattr(a, name + "_row_stride", sn)
        if not self.fuse_k_gather and not (q.is_contiguous() and k.is_contiguous()
                                           and (out is None or out.is_contiguous())):
            raise ValueError("step: strided q, k or out need fuse_k_gather (the separate gather "
                             "path reads and writes contiguous tensors)")
        # the kernels take raw pointers: a state of the wrong geometry would be
        # read out of bounds, so it is checked here
        for name, shape in (("Uq", (H, D, self.r)), ("Uk", (H, D, self.r)), ("ck", (H, C, self.r)),
                            ("cq", (H, CQ, self.r))):
            t = state.get(name)
            if (t is None or tuple(t.shape) != shape or t.dtype != torch.float16
                    or t.device != self.dev):
                raise ValueError(f"step: state[{name!r}] must be an fp16 {list(shape)} tensor on "
                                 f"{self.dev}")
        ops._check(self.tailw_t, (), torch.float32, "tailw_t", self.dev)
        a.tailw = self.tailw_t.data_ptr()
        # with the separate gathers K and V are copied to cluster order first
        if not self.fuse_k_gather:
            a.kp = self._kp(k.dtype).data_ptr()
        if not self._fused_kv:
            a.vp = self._vp(v.dtype).data_ptr()
        caller = torch.cuda.current_stream(self.dev)
        s0, s1 = self.s_main, self.s_side
        # this object's events order the streams; a call under graph capture
        # takes events of its own, which live and die with that capture
        capturing = torch.cuda.is_current_stream_capturing()

        def after(waits, which, signals):
            if capturing:
                waits.wait_stream(signals)
            else:
                self._ev[which].record(signals)
                waits.wait_event(self._ev[which])

        snap = None
        held = None
        cfg_parity = self._cfg_parity
        self._cfg_parity = None
        if self._cfg_on and cfg_parity is not None:
            held = self._cfg_hold.get(self._cfg_key)
            age = None if held is None else self._cfg_step - held["step"]
            refresh_due = age is None or age < 0 or age >= self.mask_refresh
            if held is not None and age >= 0 and not (cfg_parity == 0 and refresh_due):
                snap = held
        recycle = held is not None and snap is None
        if capturing and snap is not None:
            # s_main and s_side, both forked from the capturing stream, wait for
            # each other here: the end of such a capture crashed the process
            raise RuntimeError("step: a reuse call cannot be captured into a graph; capture "
                               "structure-rebuilding calls and run reuse calls outside")
        self.last_call_full = snap is None
        if caller != s0:
            after(s0, 0, caller)

        if snap is not None:
            st = snap
            self._point(a, st)
            a.Uq = st["Uq"].data_ptr()
            # reuse: project with the snapshot's Uq, group K and V through the
            # stored kperm, fresh value statistics from this call's V.  Only
            # the residual reads QU, lam and the tile image of cks and sumv: with
            # the fused gathers the projection and the value statistics run on
            # the side stream, under the exact attention.
            after(s1, 1, s0)
            side = (("", _lib.STEP_PROJECT_Q),)
            if self._fused_kv:
                side += (("", _lib.STEP_VSTATS | _lib.STEP_TILES),)
            self._launch(a, side, s1)
            self._ev[2].record(s1)
            main = ()
            if not self.fuse_k_gather:
                main += (("gather_k", _lib.STEP_GATHER_K),)
            if not self._fused_kv:
                main += (("vstats", _lib.STEP_VSTATS),)
            self._launch(a, main + (("attention_exact", _lib.STEP_EXACT),), s0)
            s0.wait_event(self._ev[2])
            tail = () if self._fused_kv else (("attention_prep", _lib.STEP_TILES),)
            self._launch(a, tail + (("attention_residual", _lib.STEP_RESIDUAL),), s0)
        else:
            for name in ("Uq", "Uk", "ck", "cq"):
                if not state[name].is_contiguous():
                    raise ValueError(f"step: state[{name!r}] must be contiguous")
            ops._check_ns(self.ns_t, self.dev)
            a.ns = self.ns_t.data_ptr()
            a.Uq, a.Uk = state["Uq"].data_ptr(), state["Uk"].data_ptr()
            a.cq0, a.ck0 = state["cq"].data_ptr(), state["ck"].data_ptr()
            with torch.cuda.stream(s0):
                e = lambda *shape, dtype=torch.int32: torch.empty(*shape, device=self.dev, dtype=dtype)  # noqa: E731
                f16 = torch.float16
                cq2, ck16, cks = (e(H, CQ, self.r, dtype=f16), e(H, C, self.r, dtype=f16),
                                  e(H, C, self.r, dtype=f16))
                if recycle:
                    st = dict(held, cks=cks)
                else:
                    st = {"qlab": self.qlab, "klab": self.klab, "counts": self._kmm_kcounts,
                          "tile_sizes": e(H, CQ), "qperm": e(H, N), "kperm": e(H, N),
                          "unip": e(H, CQ, C // 32), "tile_attn_plan": e(self._tile_attn_plan_ints),
                          "cks": cks}
                self._point(a, st)
                a.cq2, a.ck16 = cq2.data_ptr(), ck16.data_ptr()
                # scores fp16(QU . cks^T) and the selection in one kernel: the
                # [H, N, 2048] score tensor is never stored (the split variant
                # of the reference yields the same bitmap, so split_cap has no
                # effect here)
                gather = () if self.fuse_k_gather else (("gather_k", _lib.STEP_GATHER_K),)
                self._launch(a, (("project", _lib.STEP_PROJECT_Q | _lib.STEP_PROJECT_K),
                                 ("kmeans", _lib.STEP_KMEANS), ("score", _lib.STEP_FINALIZE),
                                 ("select", _lib.STEP_SELECT), *gather, ("plan", _lib.STEP_PLAN),
                                 ("attention_exact", _lib.STEP_EXACT),
                                 ("attention_prep", _lib.STEP_TILES),
                                 ("attention_residual", _lib.STEP_RESIDUAL)), s0)
                state["ck"], state["cq"] = ck16, cq2
                if self._cfg_on:
                    if recycle:
                        own = st
                    else:  # qlab, klab and counts are this object's own: copied
                        own = dict(st, **{n: st[n].clone() for n in ("qlab", "klab", "counts")})
                    self._cfg_hold[self._cfg_key] = dict(own, Uq=state["Uq"], step=self._cfg_step)
        if caller != s0:
            after(caller, 3, s0)
        self._last = dict(unip=st["unip"], qperm=st["qperm"], tile_sizes=st["tile_sizes"],
                          counts=st["counts"], qlab=st["qlab"], cks=st["cks"],
                          plan=st["tile_attn_plan"], kperm=st["kperm"])
        return dst

    @staticmethod
    def _point(a, st):
        """The structure's tensors as call arguments."""
        for name, key in (("qlab", "qlab"), ("klab", "klab"), ("qcounts", "tile_sizes"),
                          ("qperm", "qperm"), ("kcounts", "counts"), ("kperm", "kperm"),
                          ("unip", "unip"), ("plan", "tile_attn_plan"), ("cks", "cks")):
            setattr(a, name, st[key].data_ptr())
