"""CPU checks of the C ABI: the library loads, exports every symbol the header
declares, the ctypes layouts match the C structs, and host-side validation
returns the documented status for each bad descriptor (no GPU calls)."""
from __future__ import annotations

import ctypes
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "ssd_mi355x.h"
HEADERS = (HEADER, ROOT / "include" / "ssd_frontend.h", ROOT / "include" / "ssd_lmhead.h")


@pytest.fixture(scope="module")
def capi():
    from kernels import _capi
    _capi.load()
    return _capi


def _header_functions():
    text = "\n".join(h.read_text() for h in HEADERS)
    return sorted(set(re.findall(r"^\s*(?:int|size_t|const char\*)\s+(ssd_\w+)\s*\(", text, re.M)))


def test_library_exports_every_declared_symbol(capi):
    declared = _header_functions()
    assert set(declared) == set(capi.EXPORTS), declared
    lib = ctypes.CDLL(str(capi.LIB_PATH))
    for name in declared:
        assert hasattr(lib, name), name
    assert capi.load().ssd_abi_version() == capi.ABI_VERSION


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_ctypes_layout_matches_header(tmp_path, capi):
    src = tmp_path / "layout.c"
    fields = {
        "ssd_desc_t": [f[0] for f in capi.SsdDesc._fields_],
        "ssd_fwd_args_t": [f[0] for f in capi.SsdFwdArgs._fields_],
        "ssd_bwd_args_t": [f[0] for f in capi.SsdBwdArgs._fields_],
    }
    lines = ['#include <stdio.h>', '#include <stddef.h>', f'#include "{HEADER}"', "int main(void){"]
    for st, fs in fields.items():
        lines.append(f'printf("{st} %zu\\n", sizeof({st}));')
        for f in fs:
            lines.append(f'printf("{st}.{f} %zu\\n", offsetof({st}, {f}));')
    lines.append('printf("SSD_NOALLOC_SCRATCH_BYTES %zu\\n", (size_t)SSD_NOALLOC_SCRATCH_BYTES);')
    lines.append("return 0;}")
    src.write_text("\n".join(lines))
    exe = tmp_path / "layout"
    subprocess.run(["gcc", "-std=c99", str(src), "-o", str(exe)], check=True)
    out = dict(l.rsplit(" ", 1) for l in subprocess.run([str(exe)], capture_output=True, text=True,
                                                          check=True).stdout.splitlines())
    assert int(out["SSD_NOALLOC_SCRATCH_BYTES"]) == capi.SSD_NOALLOC_SCRATCH_BYTES
    for st, cls in (("ssd_desc_t", capi.SsdDesc), ("ssd_fwd_args_t", capi.SsdFwdArgs),
                    ("ssd_bwd_args_t", capi.SsdBwdArgs)):
        assert int(out[st]) == ctypes.sizeof(cls), st
        for f in fields[st]:
            assert int(out[f"{st}.{f}"]) == getattr(cls, f).offset, f"{st}.{f}"


def _desc(capi, **kw):
    d = capi.SsdDesc()
    base = dict(batch=4, seqlen=8192, nheads=64, headdim=64, ngroups=1, dstate=128, chunk=256,
                dtype=capi.SSD_DTYPE_BF16, state_dtype=capi.SSD_DTYPE_F32, a_mode=capi.SSD_A_PER_HEAD,
                has_dt=1, has_D=1, has_z=1, want_final=1, norm_eps=1e-6)
    base.update(kw)
    for k, v in base.items():
        setattr(d, k, v)
    return d


def _validate(capi, **kw):
    return capi.load().ssd_validate(ctypes.byref(_desc(capi, **kw)))


def test_validation_accepts_benchmark_configs(capi):
    assert _validate(capi) == capi.SSD_OK                                     # config 2
    assert _validate(capi, batch=8, seqlen=2048, nheads=24, has_z=0) == capi.SSD_OK  # config 1
    assert _validate(capi, batch=1, seqlen=65536, nheads=32, ngroups=8, dstate=64, varlen=1, nseq=15,
                     has_init=1) == capi.SSD_OK                               # config 3
    assert _validate(capi, batch=1, seqlen=512, nheads=4, headdim=32, dstate=32, chunk=64,
                     dtype=capi.SSD_DTYPE_F32, has_z=0) == capi.SSD_OK        # config 0
    # reference API: per-token A, no dt, state in the input dtype
    assert _validate(capi, a_mode=capi.SSD_A_PER_TOKEN, has_dt=0, has_D=0, has_z=0, ngroups=64,
                     state_dtype=capi.SSD_DTYPE_BF16, want_A_cumsum=1) == capi.SSD_OK
    # trapezoidal mode at config 4's layer shape (per-head B/C), both gradient settings
    for mode in (capi.SSD_TRAPZ_DROP_BETA_DA, capi.SSD_TRAPZ_EXACT_DA):
        assert _validate(capi, batch=4, seqlen=4096, nheads=32, ngroups=32, a_mode=capi.SSD_A_PER_TOKEN,
                         has_dt=0, want_final=0, trapz=mode) == capi.SSD_OK
    # reference cache path: cached A_cumsum, with and without a cached L
    for skip in (6, 7):
        assert _validate(capi, a_mode=capi.SSD_A_CUMSUM, has_dt=0, has_D=0, has_z=0, ngroups=64,
                         dA_skip=skip) == capi.SSD_OK


@pytest.mark.parametrize("kw,status", [
    (dict(batch=0), "SSD_ERR_INVALID"),
    (dict(nheads=6, ngroups=4), "SSD_ERR_INVALID"),
    (dict(dtype=7), "SSD_ERR_INVALID"),
    (dict(a_mode=1, has_dt=1), "SSD_ERR_INVALID"),
    (dict(varlen=1, nseq=3), "SSD_ERR_INVALID"),                 # varlen needs batch == 1
    (dict(a_mode=2, has_dt=0, seqlen=8000), "SSD_ERR_INVALID"),  # cumsum path needs T % Q == 0
    (dict(want_A_cumsum=1, varlen=1, batch=1, nseq=2), "SSD_ERR_INVALID"),
    (dict(norm_eps=float("nan")), "SSD_ERR_INVALID"),
    (dict(dA_skip=8), "SSD_ERR_INVALID"),                       # unknown dA_skip bit
    # a cached A_cumsum (cumsum mode) carries no gradient: CUMSUM and CHUNK must be skipped
    (dict(a_mode=2, has_dt=0, dA_skip=0), "SSD_ERR_INVALID"),
    (dict(a_mode=2, has_dt=0, dA_skip=2), "SSD_ERR_INVALID"),
    # trapezoidal mode: per-token decay, no dt, no initial / final state, no cache options
    (dict(trapz=3, a_mode=1, has_dt=0, want_final=0), "SSD_ERR_INVALID"),
    (dict(trapz=1, has_dt=0, want_final=0), "SSD_ERR_INVALID"),              # per-head A
    (dict(trapz=1, a_mode=1, has_dt=1, want_final=0), "SSD_ERR_INVALID"),    # dt given
    (dict(trapz=2, a_mode=1, has_dt=0, want_final=1), "SSD_ERR_INVALID"),    # final state asked
    (dict(trapz=2, a_mode=1, has_dt=0, want_final=0, has_init=1), "SSD_ERR_INVALID"),
    (dict(trapz=1, a_mode=1, has_dt=0, want_final=0, dA_skip=7), "SSD_ERR_INVALID"),
    (dict(chunk=512), "SSD_ERR_UNSUPPORTED"),
    (dict(headdim=256), "SSD_ERR_UNSUPPORTED"),
    (dict(dstate=160), "SSD_ERR_UNSUPPORTED"),
    (dict(dtype=0, headdim=128), "SSD_ERR_UNSUPPORTED"),         # fp32 tiles exceed LDS at N=128, P=128
])
def test_validation_rejects(capi, kw, status):
    assert _validate(capi, **kw) == getattr(capi, status)


@pytest.mark.parametrize("chunk", [1, 64, 65, 192, 256])
def test_fp32_shapes(capi, chunk):
    """The fp32 kernels take every pairing of 32, 64 and 128 padded columns but 128 x 128, whatever the chunk."""
    for P in (1, 32, 33, 64, 65, 128):
        for N in (1, 32, 33, 64, 65, 128):
            want = capi.SSD_ERR_UNSUPPORTED if P > 64 and N > 64 else capi.SSD_OK
            assert _validate(capi, dtype=capi.SSD_DTYPE_F32, headdim=P, dstate=N, chunk=chunk, has_z=0) == want, (P, N)


def test_fp32_workspaces_hold_no_tiles_that_nothing_reads(capi):
    """One head per group and N <= 32: S is multiplied in place, so the forward scratch is the chunk states and the
    decay factors alone, and the backward has dS tiles but none of S."""
    lib = capi.load()
    size = lambda kind, **kw: lib.ssd_workspace_bytes(ctypes.byref(_desc(  # noqa: E731
        capi, dtype=capi.SSD_DTYPE_F32, has_z=0, batch=8, seqlen=4096, nheads=32, headdim=32, **kw)), kind)
    chunks, unit = 8 * 16 * 32, 36 * 4096
    factors = chunks * 256 * 4
    assert size(capi.SSD_WS_FWD_SCRATCH, ngroups=32, dstate=16) == chunks * 32 * 32 * 4 + factors
    assert size(capi.SSD_WS_FWD_SCRATCH, ngroups=32, dstate=33) > 500 << 20  # (tiles, one batch)
    grown = size(capi.SSD_WS_BWD_SCRATCH, ngroups=32, dstate=16) - chunks * 10 * 256 * 4
    assert grown < chunks * unit + (64 << 20)


@pytest.mark.parametrize("kw,whole", [
    (dict(batch=32000, seqlen=64, nheads=65, ngroups=1, chunk=64), False),    # 2.08 M chunk-heads
    (dict(batch=32300, seqlen=64, nheads=65, ngroups=1, chunk=64), True),     # 2^32 threads of 1024 a kernel head
    (dict(batch=160, seqlen=8192, nheads=8, ngroups=8, chunk=256), False),    # 15.0 GiB of dS tiles
    (dict(batch=176, seqlen=8192, nheads=8, ngroups=8, chunk=256), True),     # 16.5 GiB
])
def test_wide_heads_run_whole_past_the_limits_of_pairs(capi, kw, whole):
    """Told apart by the decays' factors, one row per chunk and kernel head in the forward scratch."""
    d = _desc(capi, headdim=128, dstate=8, has_z=0, **kw)
    states = kw["batch"] * (kw["seqlen"] // kw["chunk"]) * kw["nheads"]
    fwd = capi.load().ssd_workspace_bytes(ctypes.byref(d), capi.SSD_WS_FWD_SCRATCH)
    assert fwd == states * (128 * 32 * 4 + (1 if whole else 2) * kw["chunk"] * 4)


def test_fused_backward_stays_below_32_bit_row_offsets(capi):
    """A chunk of B / C rows past 2 GiB takes the general kernels, told by the absence of dS tiles."""
    lib = capi.load()
    size = lambda G: lib.ssd_workspace_bytes(ctypes.byref(_desc(  # noqa: E731
        capi, batch=1, seqlen=256, nheads=G, ngroups=G, headdim=8, dstate=128, has_z=0)), capi.SSD_WS_BWD_SCRATCH) / G
    assert size(32767) > size(32769) + 16 * 4096 * 4


def test_workspace_sizes(capi):
    lib = capi.load()
    d = _desc(capi)
    saved = lib.ssd_workspace_bytes(ctypes.byref(d), capi.SSD_WS_SAVED)
    fwd = lib.ssd_workspace_bytes(ctypes.byref(d), capi.SSD_WS_FWD_SCRATCH)
    bwd = lib.ssd_workspace_bytes(ctypes.byref(d), capi.SSD_WS_BWD_SCRATCH)
    # saved: bf16 chunk-entering states (b*c*h*P*N*2) + y before the norm (b*L*H*P*2) + small
    assert saved >= 4 * 32 * 64 * 64 * 128 * 2 + 4 * 8192 * 64 * 64 * 2
    # fwd: fp32 chunk-local states (general path) + the fused state walk's per-token factors (c*h*Q*4)
    assert fwd == 4 * 32 * 64 * 64 * 128 * 4 + 4 * 32 * 64 * 256 * 4
    assert bwd > fwd
    assert lib.ssd_workspace_bytes(ctypes.byref(_desc(capi, batch=0)), 0) == 0


def test_entry_points_reject_null_pointers_without_touching_the_gpu(capi):
    lib = capi.load()
    d = _desc(capi)
    args = capi.SsdFwdArgs()
    assert lib.ssd_fwd(ctypes.byref(d), ctypes.byref(args), None, 0, None, 0, None) == capi.SSD_ERR_INVALID
    bargs = capi.SsdBwdArgs()
    assert lib.ssd_bwd(ctypes.byref(d), ctypes.byref(bargs), None, 0, None, 0, None) == capi.SSD_ERR_INVALID
    # pointers present but workspace missing -> workspace error
    fake = ctypes.c_void_p(16)
    args = capi.SsdFwdArgs(fake, fake, fake, fake, fake, fake, fake, fake, None, None, fake, fake, None)
    assert lib.ssd_fwd(ctypes.byref(d), ctypes.byref(args), None, 0, None, 0, None) == capi.SSD_ERR_WORKSPACE
    assert lib.ssd_status_string(capi.SSD_ERR_WORKSPACE) == b"workspace missing or too small"


def test_noalloc_rejects_inputs_beyond_its_scratch_without_touching_the_gpu(capi):
    """ssd_fwd_noalloc checks the workspace against its fixed scratch before any device call."""
    lib = capi.load()
    d = _desc(capi)                                   # config 2: far more than the scratch
    fake = ctypes.c_void_p(16)
    args = capi.SsdFwdArgs(fake, fake, fake, fake, fake, fake, fake, fake, None, None, fake, fake, None)
    need = (lib.ssd_workspace_bytes(ctypes.byref(d), capi.SSD_WS_SAVED) + 255) // 256 * 256 + \
        lib.ssd_workspace_bytes(ctypes.byref(d), capi.SSD_WS_FWD_SCRATCH)
    assert need > capi.SSD_NOALLOC_SCRATCH_BYTES
    assert lib.ssd_fwd_noalloc(ctypes.byref(d), ctypes.byref(args), None) == capi.SSD_ERR_TOO_LARGE
    assert b"no-allocation scratch" in lib.ssd_status_string(capi.SSD_ERR_TOO_LARGE)
    assert lib.ssd_fwd_noalloc(ctypes.byref(_desc(capi, batch=0)), ctypes.byref(args), None) == \
        capi.SSD_ERR_INVALID


def test_python_layer_maps_status_to_exceptions(capi):
    with pytest.raises(ValueError):
        capi.check(capi.SSD_ERR_INVALID, "x")
    with pytest.raises(NotImplementedError):
        capi.check(capi.SSD_ERR_UNSUPPORTED, "x")
    with pytest.raises(RuntimeError):
        capi.check(capi.SSD_ERR_HIP, "x")


def test_product_path_refuses_cpu_tensors():
    import torch
    import kernels
    x = torch.randn(1, 64, 2, 8)
    A = -torch.rand(1, 64, 2) * 0.1
    B = torch.randn(1, 64, 2, 4)
    with pytest.raises(AssertionError):
        kernels.fused_ssd_scan(x, A, B, B, 32)
    with pytest.raises(AssertionError):
        kernels.ssd_scan_combined(x, A.abs(), -torch.ones(2), B, B, 32)


def test_cached_tensor_rejections():
    """A cache from a call of another shape or dtype raises as the reference's torch ops would
    (RuntimeError); a CPU tensor fails the device assertion. No GPU calls."""
    import torch
    from kernels import ssd_scan as ks
    x = torch.zeros(2, 256, 4, 8)
    good = (2, 4, 4, 64)
    with pytest.raises(RuntimeError):
        ks._check_cached("A_cumsum", torch.zeros(2, 4, 2, 128), good, x)       # other chunking
    with pytest.raises(RuntimeError):
        ks._check_cached("A_cumsum", torch.zeros(1, 4, 4, 64), good, x)        # other batch
    with pytest.raises(RuntimeError):
        ks._check_cached("A_cumsum", torch.zeros(good, dtype=torch.bfloat16), good, x)
    with pytest.raises(AssertionError):
        ks._check_cached("A_cumsum", torch.zeros(good), good, x)               # CPU tensor


def test_cache_plan_gradient_terms(capi):
    """Which dA terms each cache combination leaves out (ssd_scan.py:364-406, :533)."""
    import torch
    from kernels import ssd_scan as ks
    x, A = torch.zeros(1, 128, 2, 8), torch.zeros(1, 128, 2)
    I, S, K = capi.SSD_DA_SKIP_INTRA, capi.SSD_DA_SKIP_CUMSUM, capi.SSD_DA_SKIP_CHUNK
    cases = {(False, False): (0, True), (True, False): (I, True), (False, True): (K, True),
             (True, True): (I | K, True)}
    for (has_L, has_dc), (skip, used) in cases.items():
        p = ks._cache_plan(x, A, 64, has_L, has_dc, None)
        assert p.cfg.dA_skip == skip and p.A_used == used and p.cfg.a_mode == capi.SSD_A_PER_TOKEN
    # with a cached A_cumsum the device check comes last, so build the plan from its parts
    for has_L in (False, True):
        skip = (I if has_L else 0) | S | K
        assert capi.load().ssd_validate(ctypes.byref(_desc(capi, a_mode=capi.SSD_A_CUMSUM, has_dt=0, has_D=0,
                                                              has_z=0, ngroups=64, dA_skip=skip))) == capi.SSD_OK


@pytest.mark.parametrize("P,N,dtype,k", [
    (64, 128, "bf16", 1), (128, 128, "bf16", 1), (256, 64, "bf16", 2), (192, 32, "bf16", 2),
    (384, 16, "bf16", 3), (130, 64, "bf16", 2), (128, 128, "f32", 2), (128, 64, "f32", 1), (96, 96, "f32", 2)])
def test_head_split_factor(capi, P, N, dtype, k):
    """Heads wider than the kernels' tiles run as k heads of width P / k: the smallest k the C ABI
    takes (host-side validation only)."""
    import torch
    from kernels import ssd_scan as S
    dt_ = torch.bfloat16 if dtype == "bf16" else torch.float32
    cfg = S._Cfg(chunk=128, a_mode=capi.SSD_A_PER_HEAD, nseq=1, varlen=False, state_code=capi.SSD_DTYPE_F32,
                 want_acs=False, eps=1e-6)
    x = torch.empty(1, 256, 2, P, dtype=dt_)
    B = torch.empty(1, 256, 1, N, dtype=dt_)
    dt = torch.empty(1, 256, 2)
    assert S._head_split(capi.load(), cfg, x, B, dt, None, None, None) == k


def test_state_pieces_and_limits_match_the_header(capi):
    from kernels import ssd_scan as S
    text = HEADER.read_text()
    for name in ("SSD_MAX_CHUNK", "SSD_MAX_HEADDIM", "SSD_MAX_DSTATE"):
        assert int(re.search(rf"#define {name} (\d+)", text).group(1)) == getattr(capi, name), name
    assert S._state_pieces(64) == [(0, 64)] and S._state_pieces(128) == [(0, 128)]
    assert S._state_pieces(256) == [(0, 128), (128, 128)]
    assert S._state_pieces(160) == [(0, 80), (80, 80)]
    assert S._state_pieces(300) == [(0, 100), (100, 100), (200, 100)]
    assert S._state_pieces(129) == [(0, 65), (65, 64)]


def test_head_merge_sums_each_heads_copies():
    import torch
    from kernels import ssd_scan as S
    t = torch.arange(24, dtype=torch.float32).view(2, 3, 4)   # 4 split heads = 2 heads x k = 2
    m = S._merge_heads(2, t, -1)
    assert m.shape == (2, 3, 2) and torch.equal(m, t[..., 0::2] + t[..., 1::2])
    h = torch.arange(6, dtype=torch.float32)                  # per-head vector, k = 3
    assert torch.equal(S._merge_heads(3, h, 0), torch.tensor([3.0, 12.0]))
    assert S._merge_heads(1, t, -1) is t


def test_product_path_never_imports_the_oracle():
    pkg = ROOT / "dhammic-ai_amd"
    for f in pkg.rglob("*.py"):
        assert "oracle" not in re.findall(r"^\s*(?:from|import)\s+(\w+)", f.read_text(), re.M), f


def test_lmhead_dtype_limit_raises_not_implemented():
    """The fused LM head takes hidden and weight of one dtype among bf16, fp16 and fp32 (the latter two on
    split bf16 operands); mixed dtypes and fp64 raise NotImplementedError before any device call."""
    import torch
    from kernels import lmhead
    for dt in (torch.bfloat16, torch.float16, torch.float32):
        lmhead.check_supported(dt, dt)
    for a, b in ((torch.float64, torch.float64), (torch.bfloat16, torch.float32), (torch.float16, torch.bfloat16)):
        with pytest.raises(NotImplementedError):
            lmhead.check_supported(a, b)


def test_lmhead_split_operands_carry_fp32_products():
    """[hi | hi | lo] . [hi | lo | hi] is an fp32 product to about 2^-16 (CPU, no kernels)."""
    import torch
    from kernels import lmhead
    g = torch.Generator().manual_seed(0)
    h, w = torch.randn(64, 40, generator=g), torch.randn(96, 40, generator=g)
    hs, ws = lmhead._split_operand(h, "hhl"), lmhead._split_operand(w, "hlh")
    assert hs.dtype == torch.bfloat16 and hs.shape == (64, 120) and ws.shape == (96, 120)
    exact = h.double() @ w.double().t()
    split = hs.double() @ ws.double().t()
    plain = h.bfloat16().double() @ w.bfloat16().double().t()
    err = lambda m: ((m - exact).abs().max() / exact.abs().max()).item()  # noqa: E731
    assert err(split) < 2e-5 < err(plain)


def test_lmhead_size_limits(capi):
    """ssd_lmhead_xent_* reject sizes whose launch grids would not fit 32 bits of threads, and widths
    that are not whole 16-byte rows, before touching the device (null pointers are never read)."""
    lib = capi.load()
    fake = ctypes.c_void_p(16)
    f = lib.ssd_lmhead_xent_fwd
    f.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int64] + [ctypes.c_void_p] * 3 + \
        [ctypes.c_int64] + [ctypes.c_void_p] * 4 + [ctypes.c_size_t, ctypes.c_void_p]
    f.restype = ctypes.c_int
    args = lambda M, V, d: (M, V, d, fake, fake, fake, -100, fake, fake, fake, None, 0, None)  # noqa: E731
    assert f(*args(1 << 27, 128, 64)) == capi.SSD_ERR_UNSUPPORTED
    assert f(*args(1 << 26, 1 << 30, 64)) == capi.SSD_ERR_UNSUPPORTED
    assert f(*args(64, 128, 12)) == capi.SSD_ERR_UNSUPPORTED
    assert f(*args(0, 128, 64)) == capi.SSD_ERR_INVALID
    assert f(*args(64, 128, 64)) == capi.SSD_ERR_WORKSPACE   # valid sizes: the missing workspace is next
