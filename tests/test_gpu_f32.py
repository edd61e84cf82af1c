"""The fp32 kernels (ssd_f32.hip) at the edges of their tiles and of their dispatch, against the oracle to 1e-4
(ssd_testlib.TOL; they land near 1e-6): every chunk width in 64-token steps (a unit is one or two blocks from 192
tokens on), partial 32-token tiles, head widths of one, two and four 32-wide tiles, state widths on both sides of
32 (below it, with one head per group, S is multiplied in place), rows that are not whole 16-byte vectors or start
off the 16-byte grid, shared groups with several head slices, packed sequences; units past one batch of tiles, and
the no-allocation forward where its scratch holds only part of them."""
from __future__ import annotations

import pytest
import torch

import test_gpu_parity as tp
from conftest import gpu_available
from oracle.inputs import SsdShape, make_inputs
from ssd_testlib import TOL, rel_err

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X (HIP device)")]

DEV = "cuda"


@pytest.mark.parametrize("P,H,G,N,Q,L,cu", [
    (32, 4, 1, 16, 64, 65, None),               # one tile of the second chunk holds one token
    (33, 3, 3, 31, 64, 100, None),              # rows of odd width, S in place
    (64, 4, 4, 33, 128, 257, None),             # one head per group, N just past the in-place rule
    (8, 12, 1, 8, 192, 500, None),              # three blocks per chunk, many heads per group
    (64, 6, 2, 128, 192, 383, None),
    (128, 2, 1, 64, 256, 300, None),            # the widest head tile
    (100, 2, 2, 20, 256, 513, None),
    (64, 8, 1, 64, 256, 777, [0, 1, 33, 33, 300, 777]),   # packed, one sequence empty, one of a token
    (20, 2, 2, 12, 256, 700, [0, 256, 420, 700]),
])
def test_shapes(P, H, G, N, Q, L, cu):
    errs = tp._check_ext(SsdShape(1 if cu else 2, L, H, P, G, N, Q, cu_seqlens=cu), torch.float32, with_z=H % 4 == 0,
                         seed=P + N, cu=cu, randw=True)
    assert max(errs.values()) < 1e-5, errs


def _leaves(shape, seed):
    inp = make_inputs(shape, seed=seed)
    return {k: inp[k].to(DEV) for k in ("x", "dt", "A", "B", "C", "D")}, inp["dy"].to(DEV)


def _grads(t, dy, Q):
    import kernels
    t = {k: v.requires_grad_(True) for k, v in t.items()}
    y = kernels.ssd_scan_combined(t["x"], t["dt"], t["A"], t["B"], t["C"], Q, D=t["D"])
    return [y.detach()] + list(torch.autograd.grad(y, list(t.values()), dy))


def test_rows_off_the_16_byte_grid():
    shape = SsdShape(1, 300, 4, 64, 2, 64, 128)
    t, dy = _leaves(shape, 3)
    off = lambda v: torch.cat([v.new_zeros(1), v.flatten()])[1:].view(v.shape)  # noqa: E731
    a = _grads(t, dy, 128)
    b = _grads({k: off(v.detach()) if k in "xBC" else v.detach() for k, v in t.items()}, dy, 128)
    assert all(torch.equal(u, v) for u, v in zip(a, b))


def test_units_past_one_batch():
    """4096 (chunk, group) units, past the 3640 that one batch of 256-token tiles holds: every head's results are
    those of the call on half of the heads."""
    shape = SsdShape(1, 64 * 256, 64, 8, 64, 40, 256)
    t, dy = _leaves(shape, 5)
    whole = _grads(t, dy, 256)
    cut = {"x": (2, 1), "dt": (2, 2), "A": (0, 3), "B": (2, 4), "C": (2, 5), "D": (0, 6)}
    for lo in (0, 32):
        half = {k: t[k].detach().narrow(dim, lo, 32).contiguous() for k, (dim, _) in cut.items()}
        got = _grads(half, dy[:, :, lo:lo + 32].contiguous(), 256)
        assert torch.equal(got[0], whole[0][:, :, lo:lo + 32])
        for k, (dim, i) in cut.items():
            assert torch.equal(got[i], whole[i].narrow(dim, lo, 32)), k


def test_noalloc_forward_with_tiles_in_parts():
    """512 units whose S tiles (72 MiB) do not fit the 64 MiB scratch: they are multiplied in several batches in the
    chunk states' place, with the same results."""
    import test_zz_no_alloc as na
    from kernels import _capi as C_
    from kernels import ssd_scan as ks
    t, _ = _leaves(SsdShape(1, 64 * 256, 8, 32, 8, 40, 256), 7)
    cfg = ks._Cfg(chunk=256, a_mode=C_.SSD_A_PER_HEAD, nseq=1, varlen=False, state_code=C_.SSD_DTYPE_F32,
                  want_acs=False, eps=1e-6)
    args = (t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], None, None, None, None)
    y0, f0, _, _ = ks._forward(cfg, *args)
    y1, f1, _ = na._noalloc(cfg, *args)
    assert torch.equal(y1, y0) and torch.equal(f1, f0)
    assert rel_err(y1, y0) <= TOL[torch.float32]


def test_halves_of_wide_heads_at_the_largest_row_strides():
    """36 600 heads of 128 columns: rows 18.7 MB apart, so that one 64-column half's rows span more than 2 GiB from
    row 115 on. y of the last heads is that of the call on those heads alone."""
    import kernels
    H, L, k = 36600, 128, 8
    g = torch.Generator(device=DEV).manual_seed(11)
    x = torch.randn(1, L, H, 128, generator=g, device=DEV)
    dt = torch.rand(1, L, H, generator=g, device=DEV) * 0.1
    A = -torch.rand(H, generator=g, device=DEV) * 4 - 1
    B, C = (torch.randn(1, L, 1, 16, generator=g, device=DEV) for _ in range(2))
    with torch.no_grad():
        y = kernels.ssd_scan_combined(x, dt, A, B, C, 256)
        for lo in (0, H - k):
            got = kernels.ssd_scan_combined(x[:, :, lo:lo + k].contiguous(), dt[:, :, lo:lo + k].contiguous(),
                                            A[lo:lo + k].contiguous(), B, C, 256)
            assert torch.equal(y[:, :, lo:lo + k], got)
            assert y[:, 115:, lo:lo + k].abs().min() > 0


@pytest.mark.parametrize("off", [False, True], ids=["aligned", "unaligned"])
@pytest.mark.parametrize("P,H,G,N,Q,L", [
    (32, 4, 1, 16, 64, 65), (33, 3, 3, 31, 64, 100), (64, 4, 4, 33, 128, 257), (64, 6, 2, 128, 192, 383),
    (128, 2, 1, 64, 256, 300), (100, 2, 2, 20, 256, 513), (64, 3, 3, 32, 256, 256), (20, 2, 2, 12, 256, 31)])
def test_small_batches_are_the_same_bits(P, H, G, N, Q, L, off):
    """The scan's two splits (a wave per tile over 32 columns up to 2048 such waves, two tiles over 64 columns past
    them) and the states' two step lengths make the same sums: a batch past the rule against its first and last
    sequences alone."""
    import kernels
    per = -(-L // Q) * H * -(-P // 32) * (-(-Q // 64) * 2)
    b = 2048 // per + 1
    assert per <= 2048 < b * per
    inp = {k: v.to(DEV) for k, v in make_inputs(SsdShape(b, L, H, P, G, N, Q), seed=P, with_init=True).items()}
    place = (lambda t: torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)) if off else (lambda t: t.contiguous())

    def run(lo, hi):
        x, dt, B, C, init = (place(inp[k][lo:hi]) for k in ("x", "dt", "B", "C", "init"))
        with torch.no_grad():
            return kernels.ssd_scan_combined(x, dt, inp["A"], B, C, Q, D=inp["D"], initial_states=init,
                                             return_final_state=True)

    y, fin = run(0, b)
    for i in (0, b - 1):
        yi, fi = run(i, i + 1)
        assert torch.equal(y[i:i + 1], yi) and torch.equal(fin[i:i + 1], fi)
