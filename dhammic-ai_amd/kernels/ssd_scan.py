"""Fused chunked SSD scan on MI355X: the reference's Python API over the HIP C ABI.

Drop-in for r2/dhammic-ai/src/kernels/ssd_scan.py:
  * ``fused_ssd_scan(x, A, B, C, chunk_size, initial_states=None, cache=None)``
    -> ``(Y, final_state, cache)``                                  (:539-583)
  * ``FusedSSDScan.apply(x, A, B, C, chunk_size, initial_states, L, decay_chunk,
    A_cumsum)`` -> ``(Y, final_state, L, decay_chunk, A_cumsum)``; backward
    returns the nine slots of :533                                  (:427-533)
plus the extended entry ``ssd_scan_combined`` (dt, per-head A, grouped B/C,
D, gated RMSNorm, initial/final states, packed varlen via cu_seqlens) that
the caller composes around the op (r2/dhammic-ai/src/mamba_base_engine.py:
152-191).

All device work runs in libssd_mi355x.so (gfx950 HIP kernels) on the current
torch stream; torch only allocates the tensors and the workspaces. There is
no CPU or eager fallback: a CPU tensor or a missing library raises.

Reference behaviour kept: same signatures, shapes, dtypes and return
conventions; ``T % chunk_size == 0`` raises AssertionError; with a cache the
decay comes from ``cache["A_cumsum"]`` and A gets no gradient (:364-406,
:533). Differences (all below the parity tolerance): the acausal e^-20
entries of the reference's clamped -1e4 fill are exact zeros here, the
inter-chunk recurrence clamps each chunk's decay instead of multi-chunk
sums, and decays are computed in fp32 from an fp32 cumsum whatever the input
dtype. The returned cache's ``L`` and ``decay_chunk`` are materialised on
first access (they are never needed by the kernels).
"""
from __future__ import annotations

import contextlib
import ctypes
import functools
import weakref
from dataclasses import dataclass
from typing import NamedTuple

import torch

from . import _capi as C_

__all__ = ["fused_ssd_scan", "FusedSSDScan", "ssd_scan_combined"]

_DTYPES = {torch.float32: C_.SSD_DTYPE_F32, torch.bfloat16: C_.SSD_DTYPE_BF16}


def _code(dtype, what):
    if dtype not in _DTYPES:
        raise TypeError(f"{what}: dtype {dtype} is not supported (bfloat16 or float32)")
    return _DTYPES[dtype]


def _p(t):
    """The tensor's address as ctypes takes it (an int, or None)."""
    return None if t is None else t.data_ptr()


def _stream(dev):
    """The current stream's handle on dev (torch.cuda.current_stream builds a Stream object, 3 us a call)."""
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if dev.index is None else dev.index)


_HERE = contextlib.nullcontext()


def _on(dev):
    """A context with dev current: nothing to do where it already is (torch.cuda.device costs 5 us a call)."""
    return _HERE if dev.index is None or dev.index == torch.cuda.current_device() else torch.cuda.device(dev)


class _Cfg(NamedTuple):
    chunk: int
    a_mode: int
    nseq: int
    varlen: bool
    state_code: int
    want_acs: bool
    eps: float
    dA_skip: int = 0
    trapz: int = 0   # enum ssd_trapz (fused_trapezoidal_ssd_scan)


def _desc(cfg: _Cfg, x, B, dt, D, z, init, has_dfinal=False):
    return _desc_of(cfg, x.shape, B.shape[2], B.shape[3], x.dtype, dt is not None, D is not None, z is not None,
                    init is not None, has_dfinal)


def _desc_of(cfg: _Cfg, x_shape, G, N, dtype, has_dt, has_D, has_z, has_init, has_dfinal):
    d = C_.SsdDesc()
    d.batch, d.seqlen, d.nheads, d.headdim = x_shape
    d.ngroups, d.dstate, d.chunk, d.nseq = G, N, cfg.chunk, cfg.nseq
    d.dtype = _code(dtype, "x")
    d.state_dtype = cfg.state_code
    d.a_mode = cfg.a_mode
    d.has_dt = int(has_dt)
    d.has_D = int(has_D)
    d.has_z = int(has_z)
    d.has_init = int(has_init)
    d.has_dfinal = int(has_dfinal)
    d.varlen = int(cfg.varlen)
    d.want_final = int(not cfg.trapz)
    d.want_A_cumsum = int(cfg.want_acs)
    d.norm_eps = cfg.eps
    d.dA_skip = cfg.dA_skip
    d.trapz = cfg.trapz
    return d


def _check_device(*ts):
    for t in ts:
        if t is not None and not t.is_cuda:
            raise AssertionError("fused SSD scan: all tensors must be on the GPU (got a CPU tensor)")


def _head_split(lib, cfg: _Cfg, x, B, dt, D, z, init):
    """Smallest k dividing the head width P for which the C ABI takes heads of width P / k (1: as
    given). The kernels' tiles stop at a head width of 128 (64 in fp32 beside a state width above
    64), where the reference takes any; a head's P channels are independent given its dt, A, B and
    C, so a head of width P is exactly k heads of width P / k that share them: x, z, y, the states
    and their gradients keep their memory layout (heads are the slower dimension), B and C their
    groups (each of the k heads of a group's head reads the same group), and dt, A, D and the
    trapezoidal coefficients are repeated per head, their gradients summed back."""
    return _split_factor(lib, _desc(cfg, x, B, dt, D, z, init))


def _split_factor(lib, desc):
    H, P = desc.nheads, desc.headdim
    first = lib.ssd_validate(ctypes.byref(desc))
    if first != C_.SSD_ERR_UNSUPPORTED:
        return 1
    for k in range(2, P + 1):
        if P % k:
            continue
        desc.nheads, desc.headdim = H * k, P // k
        st = lib.ssd_validate(ctypes.byref(desc))
        if st == C_.SSD_OK:
            return k
        if st != C_.SSD_ERR_UNSUPPORTED:
            break
    return 1  # (the caller's own validation then reports the limit)


class _Plan(NamedTuple):
    """What one shape of call needs from the host: the heads' split (``_head_split``), the descriptor the library
    reads, the bytes of its workspaces, and whether the library halves the heads (bf16, 80 to 128 columns)."""
    k: int
    halves: bool
    desc: object   # ctypes.byref(SsdDesc), only read once made
    saved: int
    fwd: int
    bwd: int


@functools.lru_cache(maxsize=512)
def _plan(cfg: _Cfg, x_shape, G, N, dtype, has_dt, has_D, has_z, has_init, has_dfinal):
    """The plan by the sizes and options alone (no tensor, address or device enters it), so that a training loop's
    calls find it made; errors are raised anew each time. Building it took 15 of a call's 60 us on the host."""
    lib = C_.load()
    args = (G, N, dtype, has_dt, has_D, has_z, has_init, has_dfinal)
    k = _split_factor(lib, _desc_of(cfg, x_shape, *args))
    b, T, H, P = x_shape
    desc = _desc_of(cfg, (b, T, H * k, P // k), *args)
    ref = ctypes.byref(desc)
    C_.check(lib.ssd_validate(ref), "ssd_fwd")
    halves = dtype == torch.bfloat16 and 64 < P // k <= 128 and P // k % 16 == 0 and N % 8 == 0
    return _Plan(k, halves, ref, *(lib.ssd_workspace_bytes(ref, w)
                           for w in (C_.SSD_WS_SAVED, C_.SSD_WS_FWD_SCRATCH, C_.SSD_WS_BWD_SCRATCH)))


def _plan_for(cfg, x, B, dt, D, z, init, has_dfinal=False):
    return _plan(cfg, tuple(x.shape), B.shape[2], B.shape[3], x.dtype, dt is not None, D is not None, z is not None,
                 init is not None, has_dfinal)


def _on_grid(*tensors):
    """The tensors, copied where they start off the 16-byte grid, for heads that the library runs as two halves
    (``_Plan.halves``). Off the grid the halves take its general kernels, whose backward is slower on them than on whole
    heads (8 x 2048 tokens of 8 heads of 128, N = 128: 1463 us whole, 1876 in halves, 289 with the copies)."""
    return tuple(t if t is None or t.data_ptr() % 16 == 0 else t.clone() for t in tensors)


def _split_heads(k, cfg: _Cfg, x, dt, A, D, z, init, gamma, beta):
    """The inputs of one call as k-times as many heads of width P / k (``_head_split``)."""
    if k == 1:
        return x, dt, A, D, z, init, gamma, beta
    b, T, H, P = x.shape
    rep = lambda t, dim: None if t is None else t.repeat_interleave(k, dim=dim).contiguous()  # noqa: E731
    a_dim = {C_.SSD_A_PER_HEAD: 0, C_.SSD_A_PER_TOKEN: -1, C_.SSD_A_CUMSUM: 1}[cfg.a_mode]
    return (x.view(b, T, H * k, P // k), rep(dt, -1), rep(A, a_dim), rep(D, 0),
            None if z is None else z.view(b, T, H * k, P // k),
            None if init is None else init.view(init.shape[0], H * k, P // k, init.shape[-1]),
            rep(gamma, -1), rep(beta, -1))


def _merge_heads(k, t, dim):
    """Sum of a per-head gradient over the k heads each head was split into (fp32 sums)."""
    if k == 1 or t is None:
        return t
    shape = list(t.shape)
    dim = dim % len(shape)
    merged = t.float().view(*shape[:dim], shape[dim] // k, k, *shape[dim + 1:]).sum(dim + 1)
    return merged.to(t.dtype)


def _state_pieces(N):
    """Column ranges (start, width) of a state too wide for the C ABI (N > SSD_MAX_DSTATE), else one.
    Y is a sum over state columns, in the intra-chunk term (S = C B^T sums over them) and in the state
    term alike, and the decays do not depend on them: a wide state runs as one scan per range of
    B / C columns whose outputs add, whose final states sit side by side, and whose dA, dx and dt add."""
    m = -(-N // C_.SSD_MAX_DSTATE)
    w = -(-N // m)
    return [(s0, min(w, N - s0)) for s0 in range(0, N, w)]


def _gated_norm(y, z, w, eps):
    """rmsnorm over each token's H*P channels, times w and silu(z), in fp32 (the kernels' gated norm,
    for the wide-state path, where it follows the sum of the per-range scans)."""
    b, T, H, P = y.shape
    yf = y.float().reshape(b, T, H * P)
    rs = torch.rsqrt(yf.square().mean(-1, keepdim=True) + eps)
    zf = z.float().reshape(b, T, H * P)
    return (yf * rs * w.float() * torch.nn.functional.silu(zf)).reshape(b, T, H, P)


def _forward(cfg: _Cfg, x, dt, A, B, C, D, z, w, init, cu, events=None, gamma=None, beta=None):
    """Run ssd_fwd. Returns (y, final_state or None, A_cumsum_out or empty, saved workspace).
    ``events``: optional ctypes array of 2*SSD_NUM_PHASES hipEvent_t (profiling); ``gamma``,
    ``beta``: the trapezoidal mode's coefficients (cfg.trapz)."""
    lib = C_.load()
    _check_device(x, dt, A, B, C, D, z, w, init, cu, gamma, beta)
    b, T, H0, P0 = x.shape
    plan = _plan_for(cfg, x, B, dt, D, z, init)
    k = plan.k
    if k > 1:
        x, dt, A, D, z, init, gamma, beta = _split_heads(k, cfg, x, dt, A, D, z, init, gamma, beta)
    if plan.halves:
        x, B, C, z = _on_grid(x, B, C, z)
    b, T, H, P = x.shape
    N = B.shape[3]
    dev = x.device
    y = torch.empty_like(x)
    sdt = torch.float32 if cfg.state_code == C_.SSD_DTYPE_F32 else torch.bfloat16
    final = None if cfg.trapz else torch.empty((cfg.nseq, H, P, N), dtype=sdt, device=dev)
    acs = (torch.empty((b, H, T // cfg.chunk, cfg.chunk), dtype=x.dtype, device=dev)
           if cfg.want_acs else x.new_empty(0))
    saved = torch.empty(plan.saved, dtype=torch.uint8, device=dev)
    scratch = torch.empty(plan.fwd, dtype=torch.uint8, device=dev)
    args = C_.SsdFwdArgs(_p(x), _p(dt), _p(A), _p(B), _p(C), _p(D), _p(z), _p(w), _p(init), _p(cu),
                         _p(y), _p(final), _p(acs) if cfg.want_acs else None,
                         None if events is None else ctypes.cast(events, ctypes.c_void_p), _p(gamma), _p(beta))
    with _on(dev):
        st = lib.ssd_fwd(plan.desc, ctypes.byref(args), _p(saved), plan.saved, _p(scratch), plan.fwd, _stream(dev))
    C_.check(st, "ssd_fwd")
    if k > 1:  # back to the caller's heads (the k copies of a head's cumsum are equal)
        y = y.view(b, T, H0, P0)
        final = None if final is None else final.view(cfg.nseq, H0, P0, N)
        if cfg.want_acs:
            acs = acs.view(b, H0, k, T // cfg.chunk, cfg.chunk)[:, :, 0].contiguous()
    return y, final, acs, saved


def _dA_out(cfg: _Cfg, x, A):
    """The log-decay gradient buffer ssd_bwd writes, or None: A's own shape for a per-head or
    per-token A; with a cached A_cumsum, the per-token shape (b, T, H) when the intra-chunk term
    (the reference's L built from A) is not cached too."""
    if cfg.a_mode in (C_.SSD_A_PER_HEAD, C_.SSD_A_PER_TOKEN):
        return torch.empty_like(A)
    if not cfg.dA_skip & C_.SSD_DA_SKIP_INTRA:
        return torch.empty(x.shape[:3], dtype=x.dtype, device=x.device)
    return None


def _backward(cfg: _Cfg, saved_ws, x, dt, A, B, C, D, z, w, init, cu, dy, dfinal, events=None, gamma=None,
              beta=None):
    """Run ssd_bwd. Returns dict of gradients (None where the input is absent).
    ``A`` is the decay input the forward took (A_cumsum with a cache)."""
    lib = C_.load()
    b, T, H0, P0 = x.shape
    plan = _plan_for(cfg, x, B, dt, D, z, init, dfinal is not None)
    k = plan.k
    if k > 1:
        x, dt, A, D, z, init, gamma, beta = _split_heads(k, cfg, x, dt, A, D, z, init, gamma, beta)
    dev = x.device
    dy = torch.zeros_like(x) if dy is None else dy.contiguous().view(x.shape)
    if dy.dtype != x.dtype:
        dy = dy.to(x.dtype)
    if dfinal is not None:
        sdt = torch.float32 if cfg.state_code == C_.SSD_DTYPE_F32 else torch.bfloat16
        dfinal = dfinal.to(sdt).contiguous().view(dfinal.shape[0], *x.shape[2:], dfinal.shape[-1])
    if plan.halves:
        x, B, C, z, dy = _on_grid(x, B, C, z, dy)
    g = {
        "x": torch.empty_like(x), "B": torch.empty_like(B), "C": torch.empty_like(C),
        "dt": torch.empty_like(dt) if dt is not None else None,
        "A": _dA_out(cfg, x, A),
        "D": torch.empty_like(D) if D is not None else None,
        "z": torch.empty_like(z) if z is not None else None,
        "w": torch.empty_like(w) if (w is not None and z is not None) else None,
        "init": torch.empty_like(init) if init is not None else None,
        "gamma": torch.empty_like(gamma) if gamma is not None else None,
        "beta": torch.empty_like(beta) if beta is not None else None,
    }
    scratch = torch.empty(plan.bwd, dtype=torch.uint8, device=dev)
    args = C_.SsdBwdArgs(_p(x), _p(dt), _p(A), _p(B), _p(C), _p(D), _p(z), _p(w), _p(init), _p(cu),
                         _p(dy), _p(dfinal),
                         _p(g["x"]), _p(g["dt"]), _p(g["A"]), _p(g["B"]), _p(g["C"]), _p(g["D"]),
                         _p(g["z"]), _p(g["w"]), _p(g["init"]),
                         None if events is None else ctypes.cast(events, ctypes.c_void_p),
                         _p(gamma), _p(beta), _p(g["gamma"]), _p(g["beta"]))
    with _on(dev):
        st = lib.ssd_bwd(plan.desc, ctypes.byref(args), _p(saved_ws), saved_ws.numel(), _p(scratch), plan.bwd,
                         _stream(dev))
    C_.check(st, "ssd_bwd")
    if k > 1:  # back to the caller's heads: views of the split ones, or sums over each head's k copies
        a_dim = {C_.SSD_A_PER_HEAD: 0, C_.SSD_A_PER_TOKEN: -1}.get(cfg.a_mode, -1)
        g["x"] = g["x"].view(b, T, H0, P0)
        if g["z"] is not None:
            g["z"] = g["z"].view(b, T, H0, P0)
        if g["init"] is not None:
            g["init"] = g["init"].view(g["init"].shape[0], H0, P0, g["init"].shape[-1])
        g["dt"] = _merge_heads(k, g["dt"], -1)
        g["A"] = _merge_heads(k, g["A"], a_dim)
        g["D"] = _merge_heads(k, g["D"], 0)
        g["gamma"] = _merge_heads(k, g["gamma"], -1)
        g["beta"] = _merge_heads(k, g["beta"], -1)
    return g


class _SsdFunction(torch.autograd.Function):
    """Autograd node over ssd_fwd / ssd_bwd (inputs already contiguous). With ``acs`` (a cached
    A_cumsum, cfg.a_mode CUMSUM) the kernels take the decay from it and ``A`` (per token) only
    receives the gradient terms cfg.dA_skip leaves in."""

    @staticmethod
    def forward(ctx, cfg, x, dt, A, B, C, D, z, w, init, cu, acs=None):
        ctx.set_materialize_grads(False)
        a_arg = acs if cfg.a_mode == C_.SSD_A_CUMSUM else A
        y, final, acs_out, saved = _forward(cfg, x, dt, a_arg, B, C, D, z, w, init, cu)
        ctx.cfg = cfg
        ctx.ws = saved
        ctx.save_for_backward(x, dt, a_arg, B, C, D, z, w, init, cu)
        ctx.mark_non_differentiable(acs_out)
        return y, final, acs_out

    @staticmethod
    def backward(ctx, dy, dfinal, _dacs):
        x, dt, a_arg, B, C, D, z, w, init, cu = ctx.saved_tensors
        if dy is None and dfinal is None:
            return (None,) * 12
        g = _backward(ctx.cfg, ctx.ws, x, dt, a_arg, B, C, D, z, w, init, cu, dy, dfinal)
        ni = ctx.needs_input_grad
        pick = lambda k, i: g[k] if ni[i] else None  # noqa: E731
        return (None, pick("x", 1), pick("dt", 2), pick("A", 3), pick("B", 4), pick("C", 5),
                pick("D", 6), pick("z", 7), pick("w", 8), pick("init", 9), None, None)


# --------------------------------------------------------------------------- #
# Reference cache (L, decay_chunk, A_cumsum)
# --------------------------------------------------------------------------- #
def _cache_desc(a_like, chunk):
    b, T, H = a_like.shape[:3]
    d = C_.SsdDesc()
    d.batch, d.seqlen, d.nheads, d.headdim, d.ngroups, d.dstate, d.chunk = b, T, H, 1, 1, 1, chunk
    d.dtype = _code(a_like.dtype, "A")
    return d


class _LazyCache(dict):
    """The reference's cache dict {L, decay_chunk, A_cumsum}
    (ssd_scan.py:420, shapes pinned by tests/kernels/test_ssd_scan.py:104-110).
    ``A_cumsum`` is filled by the forward; ``L`` and ``decay_chunk`` are
    computed on first access from the per-token log-decay and A_cumsum."""

    def __init__(self, a, A_cumsum, chunk, tag=True):
        super().__init__(L=None, decay_chunk=None, A_cumsum=A_cumsum)
        self._a = a
        self._a_version = a._version
        self._chunk = chunk
        self._tag = tag
        if tag:
            _tag_origin(A_cumsum, a)

    def built_from(self, A):
        """Whether this cache is the one a call on this very A (same storage, unmodified since)
        returned: its A_cumsum is then the in-kernel fp32 cumsum of A, stored in A's dtype."""
        a = self._a
        return (A.data_ptr() == a.data_ptr() and A.shape == a.shape and A.stride() == a.stride()
                and A.dtype == a.dtype and A.device == a.device and A._version == self._a_version)

    def _fill(self, key):
        v = dict.__getitem__(self, key)
        if v is None and key in ("L", "decay_chunk"):
            lib = C_.load()
            acs = dict.__getitem__(self, "A_cumsum")
            b, H, nch, Q = acs.shape
            desc = _cache_desc(self._a, self._chunk)
            dev = acs.device
            with _on(dev):
                if key == "L":
                    v = torch.empty((b, H, nch, Q, Q), dtype=acs.dtype, device=dev)
                    C_.check(lib.ssd_materialize_L(ctypes.byref(desc), _p(self._a), _p(v), _stream(dev)),
                             "ssd_materialize_L")
                else:
                    v = torch.empty((b, H, nch + 1, nch + 1), dtype=acs.dtype, device=dev)
                    C_.check(lib.ssd_decay_chunk(ctypes.byref(desc), _p(acs), _p(v), _stream(dev)),
                             "ssd_decay_chunk")
            if self._tag:
                _tag_origin(v, self._a)
            dict.__setitem__(self, key, v)
        return v

    def __getitem__(self, key):
        return self._fill(key)

    def get(self, key, default=None):
        return self._fill(key) if key in self else default

    def __iter__(self):
        return iter(list(dict.keys(self)))

    def values(self):
        return [self._fill(k) for k in self]

    def items(self):
        return [(k, self._fill(k)) for k in self]

    def copy(self):
        c = _LazyCache(self._a, dict.__getitem__(self, "A_cumsum"), self._chunk, self._tag)
        for k in ("L", "decay_chunk"):
            dict.__setitem__(c, k, dict.__getitem__(self, k))
        return c

    def cumsum_tensor(self):
        return dict.__getitem__(self, "A_cumsum")


# A cache tensor this module computed remembers the per-token decays it came from (the tensor, its
# version then, and its own version then), so that a dict of such tensors passed back is known to
# hold the decays of that call without reading its values.
_ORIGIN = "_ssd_cache_origin"


def _same_tensor(a, b):
    return (a.data_ptr() == b.data_ptr() and a.shape == b.shape and a.stride() == b.stride()
            and a.dtype == b.dtype and a.device == b.device)


def _tag_origin(v, a):
    if v is not None:
        setattr(v, _ORIGIN, (weakref.ref(a), a._version, v._version))


def _origin(v):
    """The per-token decays tensor v was computed from by this module, if v is unmodified since."""
    tag = getattr(v, _ORIGIN, None)
    if tag is None:
        return None
    ref, a_version, v_version = tag
    a = ref()
    if a is None or a._version != a_version or v._version != v_version:
        return None
    return a


def _cache_is_ours(A, L_in, dc_in, acs_in):
    """Whether every cached tensor given came from one call of this module on unmodified decays,
    and (unless A_cumsum is given, which then supplies every decay) on this A."""
    given = [t for t in (L_in, dc_in, acs_in) if t is not None]
    srcs = [_origin(t) for t in given]
    if not given or any(a is None for a in srcs):
        return False
    if any(not _same_tensor(a, srcs[0]) for a in srcs[1:]):
        return False
    return acs_in is not None or _same_tensor(srcs[0], A)


def _log_close(given, ours, dtype, mag):
    """Decays compared in the log domain (both lie in [e^-20, e^20]). The reference builds them in
    the input dtype: bf16 segsum values are spaced up to 1/8 nat apart near |20|, and a decay taken
    as a difference of two bf16-rounded cumsums is off by about |cumsum| * 2^-9 even between
    adjacent tokens. So the bound grows with the exponent and with ``mag``, the largest |cumsum|
    the decay is a difference of (broadcast against the decay's shape)."""
    lo, hi = torch.exp(torch.tensor(-20.0)).item(), torch.exp(torch.tensor(20.0)).item()
    lg = given.float().clamp(lo, hi).log()
    lr = ours.float().clamp(lo, hi).log()
    tol = 2.0 ** -6 if dtype == torch.bfloat16 else 1e-4
    return bool(((lg - lr).abs() <= tol * (1.0 + lr.abs() + 2.0 * mag)).all())


def _verify_cached_decays(A, chunk, L_in, dc_in, acs_in):
    """The kernels compute every decay from A_cumsum (the cached one, else the cumsum of A); the
    reference uses a cached L or decay_chunk as given (ssd_scan.py:370-406). A cached L or
    decay_chunk that does not hold the decays the kernels will use (a cache from another call's A)
    raises ValueError rather than give a result the reference would not. Tensors this module
    computed for these very decays are known to match; others are checked against the decays'
    own L / decay_chunk (one materialisation each)."""
    if L_in is None and dc_in is None:
        return
    if _cache_is_ours(A, L_in, dc_in, acs_in):
        return
    b, T, H = A.shape
    nch = T // chunk
    if acs_in is not None:   # per-token decays of the cached cumsum
        a = torch.diff(acs_in.float(), dim=-1, prepend=torch.zeros_like(acs_in[..., :1], dtype=torch.float32))
        a = a.permute(0, 2, 3, 1).reshape(b, T, H).to(A.dtype).contiguous()
    else:
        a = A.detach().contiguous()
    acs = acs_in if acs_in is not None else \
        a.float().view(b, nch, chunk, H).cumsum(2).permute(0, 3, 1, 2).to(A.dtype).contiguous()
    ref = _LazyCache(a, acs, chunk, tag=False)
    acs32 = acs.float()
    mags = {"L": acs32.abs().amax(-1)[..., None, None],                                     # (b, H, nch, 1, 1)
            "decay_chunk": acs32[..., -1].cumsum(-1).abs().amax(-1)[..., None, None]}     # (b, H, 1, 1)
    for name, given in (("L", L_in), ("decay_chunk", dc_in)):
        if given is not None and not _log_close(given, ref[name], A.dtype, mags[name]):
            raise ValueError(f"fused_ssd_scan: cached {name} does not hold the decays of this call "
                             f"({'its A_cumsum' if acs_in is not None else 'A'}); the kernels compute every "
                             "decay from A_cumsum, so a cache must come from a call on the same decays")


def _check_reference_inputs(x, A, B, C, chunk_size):
    assert x.shape[1] % chunk_size == 0, (
        f"sequence length {x.shape[1]} not divisible by chunk_size {chunk_size}")
    _check_device(x, A, B, C)
    if not (x.dtype == A.dtype == B.dtype == C.dtype):
        raise RuntimeError(f"fused_ssd_scan: x, A, B, C must share one dtype "
                           f"(got {x.dtype}, {A.dtype}, {B.dtype}, {C.dtype})")


def _check_cached(name, t, shape, x):
    """A cached tensor must be what a prior call on inputs of x's shape returned: the reference
    combines it with this call's tensors in torch ops, which raise RuntimeError on a shape or
    dtype mismatch (ssd_scan.py:364-408); the kernels read A_cumsum by that shape."""
    if tuple(t.shape) != tuple(shape) or t.dtype != x.dtype:
        raise RuntimeError(f"fused_ssd_scan: cached {name} has shape {tuple(t.shape)} and dtype {t.dtype}; "
                           f"this call needs {tuple(shape)} and {x.dtype}")
    _check_device(t)
    if t.device != x.device:
        raise RuntimeError(f"fused_ssd_scan: cached {name} is on {t.device}, the inputs on {x.device}")


@dataclass(frozen=True)
class _CachePlan:
    cfg: _Cfg
    acs: torch.Tensor | None   # the cached A_cumsum the kernels read, or None (cumsum of A)
    A_used: bool               # A enters the computation (else its gradient is None, as in :533)


def _cache_plan(x, A, chunk, has_L, has_dc, acs, recompute=False):
    """Which decays come from a cache (ssd_scan.py:364-406): the intra-chunk L, the inter-chunk
    decay_chunk, A_cumsum (state build, Y_off, and decay_chunk when not cached itself). A cached
    tensor takes no gradient, so each one drops its terms from dA; A takes none at all when it feeds
    nothing (L and A_cumsum both cached). The kernels compute every decay from A_cumsum (the cached
    one, or the cumsum of A): a cached L or decay_chunk is taken to be the one a call on the same
    decays returned, which is how the reference's caller builds its cache
    (mamba_base_engine.py:170-181). ``recompute``: the cache came from this module's call on this
    same A, so the kernels rebuild that call's fp32 cumsum from A rather than read its stored copy.
    In bf16 the stored copy is rounded, and differences of rounded cumsums lose the intra-chunk
    decays of nearby tokens, which the reference takes from segsum(A) or its cached L (:104-116).
    The dropped gradient terms are the cache's all the same."""
    b, T, H = x.shape[:3]
    nch = T // chunk
    if acs is not None:
        _check_cached("A_cumsum", acs, (b, H, nch, chunk), x)
    skip = ((C_.SSD_DA_SKIP_INTRA if has_L else 0)
            | (C_.SSD_DA_SKIP_CUMSUM | C_.SSD_DA_SKIP_CHUNK if acs is not None else 0)
            | (C_.SSD_DA_SKIP_CHUNK if has_dc else 0))
    from_acs = acs is not None and not recompute
    a_mode = C_.SSD_A_CUMSUM if from_acs else C_.SSD_A_PER_TOKEN
    cfg = _Cfg(chunk=chunk, a_mode=a_mode, nseq=b, varlen=False, state_code=_code(x.dtype, "x"),
               want_acs=acs is None, eps=0.0, dA_skip=skip)
    return _CachePlan(cfg, acs.detach().contiguous() if from_acs else None, not (has_L and acs is not None))


def _kernel_chunk(chunk):
    """The chunk the kernels run: the caller's, or for one longer than SSD_MAX_CHUNK its largest
    divisor within the limit. Pairs of tokens in one caller chunk and two kernel chunks then meet
    through the state path, whose decays are the same cumsum differences, clamped per chunk: they
    differ from the reference's one clamp only where a decay is below e^-20."""
    if chunk <= C_.SSD_MAX_CHUNK:
        return chunk
    return max(q for q in range(1, C_.SSD_MAX_CHUNK + 1) if chunk % q == 0)


def _rechunk_plan(plan, chunk):
    """The cache plan at the kernels' chunk (``_kernel_chunk``): a cached A_cumsum restarted at every
    kernel chunk (fp32 differences), and no A_cumsum output (the caller's is built at its own chunk
    by ``_chunk_cumsum``)."""
    qk = _kernel_chunk(chunk)
    if qk == chunk:
        return plan
    acs = plan.acs
    if acs is not None:
        b, H, nch, Q = acs.shape
        a32 = acs.float().view(b, H, nch, Q // qk, qk)
        base = torch.cat([torch.zeros_like(a32[..., :1, -1:]), a32[..., :-1, -1:]], dim=-2)
        acs = (a32 - base).reshape(b, H, nch * (Q // qk), qk).to(acs.dtype).contiguous()
    return _CachePlan(plan.cfg._replace(chunk=qk, want_acs=False), acs, plan.A_used)


def _chunk_cumsum(a, chunk):
    """A_cumsum (b, H, T / chunk, chunk) of the per-token decays a (b, T, H): the fp32 cumsum within
    each chunk, stored in a's dtype (what the kernels write at chunks they run themselves)."""
    b, T, H = a.shape
    return a.float().view(b, T // chunk, chunk, H).cumsum(2).permute(0, 3, 1, 2).to(a.dtype).contiguous()


def fused_ssd_scan(x, A, B, C, chunk_size, initial_states=None, cache=None):
    """Fused SSD chunked-parallel scan (ssd_scan.py:539-583).

    Args:
        x: (b, seqlen, n_heads, d_head), bf16 or fp32, on the GPU.
        A: (b, seqlen, n_heads) per-token log-decay, same dtype.
        B, C: (b, seqlen, n_heads, d_state), same dtype.
        chunk_size: seqlen must be divisible by this (AssertionError otherwise).
        initial_states: optional (b, 1, n_heads, d_head, d_state); zeros if None.
        cache: optional dict from a prior call with any of the keys L, decay_chunk,
            A_cumsum (None values count as absent). Each cached decay replaces the one
            computed from A and carries no gradient, as in the reference: with the whole
            cache of a prior call (the β call of the Mamba-3 block), A gets no gradient.

    Returns:
        Y (b, seqlen, n_heads, d_head), final_state (b, n_heads, d_head, d_state),
        cache {L, decay_chunk, A_cumsum}; L and decay_chunk are computed on first access.
    """
    chunk = int(chunk_size)
    _check_reference_inputs(x, A, B, C, chunk)
    b, T, H, P = x.shape
    N = B.shape[-1]
    pieces = _state_pieces(N)
    if len(pieces) > 1:  # a state wider than the tiles: one scan per range of its columns
        ys, finals, out = [], [], None
        for s0, w in pieces:
            init_k = None if initial_states is None else initial_states[..., s0:s0 + w]
            y_k, f_k, c_k = fused_ssd_scan(x, A, B[..., s0:s0 + w], C[..., s0:s0 + w], chunk, init_k, cache)
            ys.append(y_k.float())
            finals.append(f_k)
            out = c_k if out is None else out
        return torch.stack(ys).sum(0).to(x.dtype), torch.cat(finals, -1), out
    init = None if initial_states is None else initial_states.reshape(b, H, P, N).contiguous()
    L_in = dc_in = acs_in = None
    recompute = False
    if isinstance(cache, _LazyCache):
        # every key is present (L and decay_chunk lazily, from the same decays)
        has_L = has_dc = True
        acs_in = cache.cumsum_tensor()
        recompute = cache.built_from(A)
    elif cache is not None:
        L_in, dc_in, acs_in = cache.get("L"), cache.get("decay_chunk"), cache.get("A_cumsum")
        has_L, has_dc = L_in is not None, dc_in is not None
        nch = T // chunk
        if has_L:
            _check_cached("L", L_in, (b, H, nch, chunk, chunk), x)
        if has_dc:
            _check_cached("decay_chunk", dc_in, (b, H, nch + 1, nch + 1), x)
        if acs_in is not None:
            _check_cached("A_cumsum", acs_in, (b, H, nch, chunk), x)
        _verify_cached_decays(A, chunk, L_in, dc_in, acs_in)
    else:
        has_L = has_dc = False
    plan = _cache_plan(x, A, chunk, has_L, has_dc, acs_in, recompute)
    kplan = _rechunk_plan(plan, chunk)
    a = A.contiguous()
    Y, final, acs = _SsdFunction.apply(kplan.cfg, x.contiguous(), None, a if plan.A_used else a.detach(),
                                       B.contiguous(), C.contiguous(), None, None, None, init, None, kplan.acs)
    if isinstance(cache, _LazyCache):
        return Y, final, cache.copy()
    if kplan is not plan and plan.acs is None:
        acs = _chunk_cumsum(a.detach(), chunk)
    out = _LazyCache(a.detach(), acs if plan.acs is None else acs_in, chunk)
    if L_in is not None:
        dict.__setitem__(out, "L", L_in)
    if dc_in is not None:
        dict.__setitem__(out, "decay_chunk", dc_in)
    return Y, final, out


class FusedSSDScan(torch.autograd.Function):
    """The reference's autograd op with its exact 9-in / 5-out contract
    (ssd_scan.py:427-533). Returns (Y, final_state, L, decay_chunk, A_cumsum): each
    cached tensor as given, the others computed (L from A, decay_chunk from A_cumsum,
    as the reference builds them). Backward returns the nine slots of :533; dA holds
    the terms of the decays not taken from a cache, and is None when A feeds nothing
    (L and A_cumsum both cached)."""

    @staticmethod
    def forward(ctx, x, A, B, C, chunk_size, initial_states, L_cache_in, decay_chunk_cache_in,
                A_cumsum_cache_in):
        chunk = int(chunk_size)
        _check_reference_inputs(x, A, B, C, chunk)
        b, T, H, P = x.shape
        N = B.shape[-1]
        nch = T // chunk
        if L_cache_in is not None:
            _check_cached("L", L_cache_in, (b, H, nch, chunk, chunk), x)
        if decay_chunk_cache_in is not None:
            _check_cached("decay_chunk", decay_chunk_cache_in, (b, H, nch + 1, nch + 1), x)
        if A_cumsum_cache_in is not None:
            _check_cached("A_cumsum", A_cumsum_cache_in, (b, H, nch, chunk), x)
        _verify_cached_decays(A, chunk, L_cache_in, decay_chunk_cache_in, A_cumsum_cache_in)
        init = None if initial_states is None else initial_states.reshape(b, H, P, N).contiguous()
        x, B, C = x.contiguous(), B.contiguous(), C.contiguous()
        plan = _cache_plan(x, A, chunk, L_cache_in is not None, decay_chunk_cache_in is not None,
                           A_cumsum_cache_in)
        kplan = _rechunk_plan(plan, chunk)
        a_tok = A.detach().contiguous()
        a_arg = kplan.acs if kplan.acs is not None else a_tok
        # one scan per range of state columns (one range unless N > SSD_MAX_DSTATE): outputs add,
        # final states sit side by side
        pieces = _state_pieces(N)
        outs = [_forward(kplan.cfg, x, None, a_arg, B[..., s0:s0 + w].contiguous(), C[..., s0:s0 + w].contiguous(),
                         None, None, None, None if init is None else init[..., s0:s0 + w].contiguous(), None)
                for s0, w in pieces]
        if len(outs) == 1:
            Y, final, acs, saved = outs[0]
        else:
            Y = torch.stack([o[0].float() for o in outs]).sum(0).to(x.dtype)
            final = torch.cat([o[1] for o in outs], -1)
            acs, saved = outs[0][2], [o[3] for o in outs]
        if A_cumsum_cache_in is not None:
            acs = A_cumsum_cache_in
        elif kplan is not plan:
            acs = _chunk_cumsum(a_tok, chunk)
        lazy = _LazyCache(a_tok, acs, chunk)
        L = L_cache_in if L_cache_in is not None else lazy["L"]
        dc = decay_chunk_cache_in if decay_chunk_cache_in is not None else lazy["decay_chunk"]
        ctx.cfg = kplan.cfg
        ctx.A_used = plan.A_used
        ctx.ws = saved
        ctx.init_shape = None if initial_states is None else initial_states.shape
        ctx.pieces = pieces
        ctx.save_for_backward(x, a_arg, B, C, init)
        ctx.set_materialize_grads(False)
        return Y, final, L, dc, acs

    @staticmethod
    def backward(ctx, dY, dfinal_state, dL_unused, ddecay_chunk_unused, dA_cumsum_unused):
        x, a_arg, B, C, init = ctx.saved_tensors
        if dY is None and dfinal_state is None:
            return (None,) * 9
        if len(ctx.pieces) == 1:
            g = _backward(ctx.cfg, ctx.ws, x, None, a_arg, B, C, None, None, None, init, None, dY, dfinal_state)
        else:  # per range of state columns: dx and dA add, dB, dC and dinit sit side by side
            parts = []
            for (s0, w), ws in zip(ctx.pieces, ctx.ws):
                cut = lambda t: None if t is None else t[..., s0:s0 + w].contiguous()  # noqa: E731
                parts.append(_backward(ctx.cfg, ws, x, None, a_arg, cut(B), cut(C), None, None, None, cut(init),
                                       None, dY, cut(dfinal_state)))
            add = lambda k: None if parts[0][k] is None else \
                torch.stack([q[k].float() for q in parts]).sum(0).to(parts[0][k].dtype)  # noqa: E731
            side = lambda k: None if parts[0][k] is None else torch.cat([q[k] for q in parts], -1)  # noqa: E731
            g = {"x": add("x"), "A": add("A"), "B": side("B"), "C": side("C"), "init": side("init")}
        ni = ctx.needs_input_grad
        dA = g["A"] if (ni[1] and ctx.A_used) else None
        dinit = g["init"].reshape(ctx.init_shape) if (ctx.init_shape is not None and ni[5]) else None
        return (g["x"] if ni[0] else None, dA, g["B"] if ni[2] else None, g["C"] if ni[3] else None,
                None, dinit, None, None, None)


def ssd_scan_combined(x, dt, A, B, C, chunk_size, D=None, z=None, norm_weight=None, norm_eps=1e-6,
                      initial_states=None, cu_seqlens=None, return_final_state=False):
    """Extended SSD: Y = SSD(x*dt, dt*A, B, C) + D*x, then optionally
    rmsnorm(Y over heads*headdim) * norm_weight * silu(z).

    x (b, L, H, P) bf16/fp32; dt (b, L, H) positive; A (H,); B, C (b, L, G, N)
    with head h reading group h // (H/G); D (H,); z like x; norm_weight (H*P,);
    initial_states (nseq, H, P, N) fp32; cu_seqlens (nseq+1,) int32 offsets of
    packed sequences (b must be 1; cu_seqlens[0] = 0, cu_seqlens[-1] = L).
    Sequences need not be chunk multiples: each ends in a partial chunk.
    Returns out (and final_states (nseq, H, P, N) fp32 when asked).
    """
    b, L, H, P = x.shape
    _check_device(x, dt, A, B, C, D, z, norm_weight, initial_states)
    if B.dtype != x.dtype or C.dtype != x.dtype or (z is not None and z.dtype != x.dtype):
        raise RuntimeError("ssd_scan_combined: B, C and z must have x's dtype")
    pieces = _state_pieces(B.shape[-1])
    if len(pieces) > 1:  # a state wider than the tiles: one scan per range of its columns, then D and the norm
        ys, finals = [], []
        for s0, w in pieces:
            init_k = None if initial_states is None else initial_states[..., s0:s0 + w]
            y_k, f_k = ssd_scan_combined(x, dt, A, B[..., s0:s0 + w], C[..., s0:s0 + w], chunk_size,
                                         initial_states=init_k, cu_seqlens=cu_seqlens, return_final_state=True)
            ys.append(y_k.float())
            finals.append(f_k)
        y = torch.stack(ys).sum(0)
        if D is not None:
            y = y + x.float() * D.float().view(1, 1, H, 1)
        if z is not None:
            w_ = norm_weight if norm_weight is not None else torch.ones(H * P, device=x.device)
            y = _gated_norm(y, z, w_, float(norm_eps))
        y = y.to(x.dtype)
        return (y, torch.cat(finals, -1)) if return_final_state else y
    f32 = lambda t: None if t is None else t.float().contiguous()  # noqa: E731
    cu = None
    nseq = b
    if cu_seqlens is not None:
        if b != 1:
            raise ValueError("ssd_scan_combined: cu_seqlens needs batch == 1")
        cu = cu_seqlens.to(device=x.device, dtype=torch.int32).contiguous()
        nseq = cu.numel() - 1
    if z is not None and norm_weight is None:
        norm_weight = torch.ones(H * P, dtype=torch.float32, device=x.device)
    cfg = _Cfg(chunk=_kernel_chunk(int(chunk_size)), a_mode=C_.SSD_A_PER_HEAD, nseq=nseq, varlen=cu is not None,
               state_code=C_.SSD_DTYPE_F32, want_acs=False, eps=float(norm_eps))
    init = f32(initial_states)
    out, final, _ = _SsdFunction.apply(cfg, x.contiguous(), f32(dt), f32(A), B.contiguous(), C.contiguous(),
                                       f32(D), None if z is None else z.contiguous(),
                                       f32(norm_weight) if z is not None else None, init, cu, None)
    return (out, final) if return_final_state else out
