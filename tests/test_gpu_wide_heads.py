"""bf16 heads of 80 .. 128 columns, which the library runs as two kernel heads of half the width sharing the
head's dt, A, B, C and D: every entry point against the oracle, at the widths next to the rule's edges
(P % 16 == 0), odd head counts (the pair sums of the finish kernel then end on a half-filled block), packed
sequences, the cache, both trapezoidal gradient settings with steep tokens, rows that are not 16-byte aligned
(the general kernels on the same pairs), and the no-allocation forward on both sides of its scratch limit.
Tolerances: the flat 1e-2 of bf16 inputs (ssd_testlib.TOL)."""
from __future__ import annotations

import pytest
import torch

import test_gpu_parity as tp
import test_gpu_trapz as tz
from conftest import gpu_available
from oracle.inputs import SsdShape, make_inputs, make_reference_test_inputs
from ssd_testlib import TOL, assert_close, oracle_reference_api, rel_err

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X (HIP device)")]

DEV, BF = "cuda", torch.bfloat16


@pytest.mark.parametrize("P,H,G,N,Q,L,cu,with_z", [
    (80, 3, 1, 64, 64, 200, None, True),           # narrowest pair, odd head count, ragged length
    (96, 6, 3, 48, 128, 300, None, False),         # halves narrower than their tile, groups
    (112, 5, 5, 16, 256, 513, [0, 1, 258, 513], True),   # per-head B / C, packed sequences (one of a token)
    (128, 4, 1, 128, 256, 777, None, True),        # widest, full tiles, three chunk blocks and a remainder
    (104, 3, 3, 32, 64, 130, None, False),         # P / 2 not a multiple of 8: the head runs whole
])
def test_combined(P, H, G, N, Q, L, cu, with_z):
    tp._check_ext(SsdShape(1 if cu else 2, L, H, P, G, N, Q, cu_seqlens=cu), BF, with_z=with_z, seed=P + L, cu=cu,
                  randw=True)


@pytest.mark.parametrize("P,h", [(80, 3), (128, 2)])
def test_reference_api_and_cache(P, h):
    """fused_ssd_scan: values, gradients, the cache of the caller's heads, and that cache passed back both as
    the object and as a bare A_cumsum."""
    import kernels
    b, T, n, chunk = 2, 256, 32, 64
    x, A, B, C = [t.bfloat16().float() for t in make_reference_test_inputs(b, T, h, P, n, seed=P)]
    dY = torch.randn(b, T, h, P, generator=torch.Generator().manual_seed(3)).bfloat16().float()
    Yo, fo, go, co = oracle_reference_api(x, A, B, C, chunk, dY)
    leaves = [t.to(DEV, BF).requires_grad_(True) for t in (x, A, B, C)]
    Y, fs, cache = kernels.fused_ssd_scan(*leaves, chunk)
    Y.backward(dY.to(DEV, BF))
    for name, got, ref in [("Y", Y, Yo), ("final", fs, fo)] + [("d" + k, t.grad, go[k]) for k, t in zip("xABC", leaves)]:
        assert_close(name, got, ref, TOL[BF])
    for key in ("L", "A_cumsum"):
        assert cache[key].shape == co[key].shape
        assert_close(key, cache[key], co[key], TOL[BF])
    gx = [t.detach() for t in leaves]
    Y2, f2, _ = kernels.fused_ssd_scan(*gx, chunk, cache=cache)
    assert torch.equal(Y2, Y) and torch.equal(f2, fs)
    Y3 = kernels.fused_ssd_scan(*gx, chunk, cache={"A_cumsum": cache["A_cumsum"]})[0]
    assert_close("Y from A_cumsum", Y3, Yo, TOL[BF])


@pytest.mark.parametrize("exact", tz.MODES, ids=tz.MODE_IDS)
@pytest.mark.parametrize("P,H,G,steep", [(80, 3, 3, False), (128, 4, 2, False), (96, 4, 4, 2)])
def test_trapezoidal(P, H, G, steep, exact):
    t = tz.make(b=2, T=200, H=H, P=P, G=G, N=32, dtype=BF, seed=P, steep=steep)
    y, g = tz.native(t, 64, exact)
    yr, gr = tz.oracle(t, 64, exact)
    for name, got, ref in [("y", y, yr)] + [("d" + k, g[k], gr[k]) for k in tz.NAMES if k in g]:
        assert_close(name, got, ref, TOL[BF])


def test_rows_off_the_16_byte_grid():
    """x, B and C at storage offset 1: the general kernels run on the same pairs as the fused ones."""
    import kernels
    shape = SsdShape(1, 200, 3, 128, 1, 32, 64)
    inp = make_inputs(shape, seed=9)
    off = lambda t: torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)  # noqa: E731
    outs = []
    for place in (lambda t: t, off):
        leaves = {k: inp[k].to(DEV) for k in ("x", "dt", "A", "B", "C", "D")}
        for k in ("x", "B", "C"):
            leaves[k] = place(leaves[k].to(BF))
        leaves = {k: v.requires_grad_(True) for k, v in leaves.items()}
        out = kernels.ssd_scan_combined(*[leaves[k] for k in ("x", "dt", "A", "B", "C")], 64, D=leaves["D"])
        outs.append([out] + list(torch.autograd.grad(out, list(leaves.values()), inp["dy"].to(DEV, BF))))
    assert all(rel_err(a, b) <= TOL[BF] for a, b in zip(*outs)), [rel_err(a, b) for a, b in zip(*outs)]


@pytest.mark.parametrize("copies", [True, False], ids=["copied", "in place"])
@pytest.mark.parametrize("P,G,N,z", [(128, 3, 32, True), (96, 1, 64, False)])
def test_rows_off_the_grid_are_copied(P, G, N, z, copies, monkeypatch):
    """x, B, C, z and dy at storage offset 1: the Python layer copies them onto the grid, with the aligned call's bits;
    without the copies (as a caller of the C ABI has it) the general kernels run on the pairs."""
    import kernels
    from kernels import ssd_scan as ks
    if not copies:
        monkeypatch.setattr(ks, "_on_grid", lambda *t: t)
    inp = make_inputs(SsdShape(2, 200, 3, P, G, N, 64), seed=9, with_z=z)
    off = lambda t: torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)  # noqa: E731
    outs = []
    for place in (lambda t: t, off):
        t = {k: place(inp[k].to(DEV, BF)) if k in ("x", "B", "C", "z") else inp[k].to(DEV)
             for k in ("x", "dt", "A", "B", "C", "D") + (("z",) if z else ())}
        t = {k: v.requires_grad_(True) for k, v in t.items()}
        w = torch.ones(3 * P, device=DEV) if z else None
        y = kernels.ssd_scan_combined(*[t[k] for k in ("x", "dt", "A", "B", "C")], 64, D=t["D"], z=t.get("z"),
                                      norm_weight=w)
        outs.append([y] + list(torch.autograd.grad(y, list(t.values()), place(inp["dy"].to(DEV, BF)))))
    if copies:
        assert all(torch.equal(u, v) for u, v in zip(*outs))
    else:
        assert all(rel_err(u, v) <= TOL[BF] for u, v in zip(*outs)), [rel_err(u, v) for u, v in zip(*outs)]


def test_noalloc_forward_on_both_sides_of_the_pairs_limit():
    """A forward whose pairs fit the 64 MiB scratch, and one that fits only with whole heads, which
    ssd_fwd_noalloc then runs: the second agrees with ssd_fwd's pairs to bf16 rounding."""
    import test_zz_no_alloc as na
    from kernels import _capi as C_
    from kernels import ssd_scan as ks
    seen = set()
    for chunks in (8, 94, 95, 96, 97):
        shape = SsdShape(1, 64 * chunks, 12, 128, 1, 64, 64)
        inp = {k: v.to(DEV) for k, v in make_inputs(shape, seed=chunks).items()}
        cfg = ks._Cfg(chunk=64, a_mode=C_.SSD_A_PER_HEAD, nseq=1, varlen=False, state_code=C_.SSD_DTYPE_F32,
                      want_acs=False, eps=1e-6)
        args = (inp["x"].to(BF), inp["dt"], inp["A"], inp["B"].to(BF), inp["C"].to(BF), inp["D"], None, None, None, None)
        y0, f0, _, _ = ks._forward(cfg, *args)
        try:
            y1, f1, _ = na._noalloc(cfg, *args)
        except RuntimeError as e:
            assert "no-allocation scratch" in str(e)
            seen.add("too large")
            continue
        seen.add("pairs" if torch.equal(y1, y0) else "whole")
        assert_close("y", y1, y0, TOL[BF])
        assert_close("final", f1, f0, TOL[BF])
    print(seen)
    assert {"pairs", "whole", "too large"} <= seen


@pytest.mark.parametrize("P,N,chunk", [(80, 16, 64), (96, 128, 192), (128, 64, 256), (128, 32, 128)])
def test_forward_rounds_only_the_decayed_scores(P, N, chunk):
    """y without D: M's rounding and y's own, each uniform in half a bf16 ulp (1.66e-3 of the value in the root mean
    square), are 2.35e-3 together; one operand more would be 2.87e-3."""
    import kernels
    from oracle.ssd_chunked import fused_ssd_scan as ref_scan
    ins = [t.bfloat16() for t in make_reference_test_inputs(2, 768, 4, P, N, seed=N)]
    y = kernels.fused_ssd_scan(*[t.to(DEV) for t in ins], chunk)[0].double().cpu()
    ref = ref_scan(*[t.double() for t in ins], chunk)[0]
    err = ((y - ref).norm() / ref.norm()).item()
    print(P, N, chunk, err)
    assert err <= 2.6e-3, err


@pytest.mark.parametrize("P,H,b,L,Q,cu", [
    (104, 65, 2, 70, 64, None),                      # 130 (head, sequence) walks, two chunks
    (88, 33, 1, 300, 128, [0, 1, 90, 90, 200, 300]),  # 165 walks of packed sequences, one of them empty
    (120, 129, 1, 40, 256, None),
])
def test_whole_heads_with_128_state_columns(P, H, b, L, Q, cu):
    """Heads that do not halve (P % 16 != 0), states of 128 x 128 padded, more walks than half the CUs: a block per
    walk would need 1280 threads, so every walk is two blocks over half the columns."""
    tp._check_ext(SsdShape(b, L, H, P, 1, 128, Q, cu_seqlens=cu), BF, with_z=False, seed=P, cu=cu, randw=True)


def test_noalloc_whole_heads_with_128_state_columns():
    """The first head count whose pairs do not fit the no-allocation scratch: whole heads with 128 x 128 states."""
    import ctypes
    import test_zz_no_alloc as na
    from kernels import _capi as C_
    from kernels import ssd_scan as ks
    lib = C_.load()
    cfg = ks._Cfg(chunk=64, a_mode=C_.SSD_A_PER_HEAD, nseq=1, varlen=False, state_code=C_.SSD_DTYPE_F32, want_acs=False,
                  eps=1e-6)

    def need(H):
        d = ctypes.byref(ks._desc_of(cfg, (1, 64, H, 128), 1, 128, BF, True, True, False, False, False))
        saved, fwd = (lib.ssd_workspace_bytes(d, k) for k in (C_.SSD_WS_SAVED, C_.SSD_WS_FWD_SCRATCH))
        return (saved + 255) // 256 * 256 + fwd

    H = next(h for h in range(129, 2000) if need(h) > C_.SSD_NOALLOC_SCRATCH_BYTES)
    inp = {k: v.to(DEV) for k, v in make_inputs(SsdShape(1, 64, H, 128, 1, 128, 64), seed=1).items()}
    args = (inp["x"].to(BF), inp["dt"], inp["A"], inp["B"].to(BF), inp["C"].to(BF), inp["D"], None, None, None, None)
    y0, f0, _, _ = ks._forward(cfg, *args)
    y1, f1, _ = na._noalloc(cfg, *args)
    assert not torch.equal(y1, y0)  # (other kernels)
    assert_close("y", y1, y0, TOL[BF])
    assert_close("final", f1, f0, TOL[BF])


@pytest.mark.parametrize("exact", tz.MODES, ids=tz.MODE_IDS)
def test_trapezoidal_whole_heads_with_128_state_columns(exact):
    tz.check(tz.make(1, 100, 70, 104, 1, 128, BF, seed=4), 64, exact, BF, oracle_device=DEV, oracle_dtype=torch.float32,
             tag="whole P=104 N=128")
