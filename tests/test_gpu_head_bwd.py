"""The backward for B and C per head (one block per chunk and head, csrc/ssd_bwd_head.hip) at the edges of its tiles:
every chunk height it takes (2 to 8 tiles of 32 tokens), partial last tiles and chunks of one token, every width of
its column tiles full and partly filled, packed sequences, growing and steep heads, and both trapezoidal gradient
settings. Two checks each: against the oracle, and against the column / row kernels of larger groups on the same
inputs (SSD_ROW_KERNEL=block also turns this kernel off). Tolerances: 1e-2 of bf16 inputs against the oracle
(ssd_testlib.TOL). Between the two paths: both round M, dS and the outputs to bf16 (2^-9 each) along different
orders of sums, so normwise at most 4 * 2^-9 apart where nothing cancels."""
from __future__ import annotations

import pytest
import torch

import test_gpu_parity as tp
from conftest import gpu_available
from oracle.inputs import SsdShape, make_inputs
from oracle.ssd_extended import ssd_combined
from ssd_testlib import assert_close

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X (HIP device)")]

DEV, BF = "cuda", torch.bfloat16
SHAPES = [  # P, H, N, chunk, L, cu_seqlens
    (64, 3, 128, 64, 64, None),                     # one chunk of two tiles
    (64, 2, 128, 256, 513, None),                   # eight tiles, then a chunk of one token
    (64, 3, 64, 192, 31, None),                     # less than a tile
    (64, 3, 32, 128, 300, None),
    (64, 1, 16, 192, 400, None),                    # half a state tile; six waves
    (40, 3, 72, 128, 161, None),                    # partly filled column tiles
    (32, 4, 128, 256, 255, None),
    (16, 5, 32, 64, 129, None),
    (8, 2, 8, 256, 290, None),                      # narrowest
    (64, 3, 64, 256, 800, [0, 1, 1, 258, 514, 800]),  # packed: a token, none, 257, one chunk, a remainder
]


def _grads(shape, cu, monkeypatch, env, edit=lambda inp: inp):
    if env:
        monkeypatch.setenv("SSD_ROW_KERNEL", env)
    else:
        monkeypatch.delenv("SSD_ROW_KERNEL", raising=False)
    import kernels
    inp = edit(make_inputs(shape, seed=7, device=DEV, with_init=True, with_dfinal=True))
    leaves = {k: inp[k].to(BF).requires_grad_(True) for k in ("x", "B", "C")}
    leaves |= {k: inp[k].clone().requires_grad_(True) for k in ("dt", "A", "D", "init")}
    out, fin = kernels.ssd_scan_combined(
        leaves["x"], leaves["dt"], leaves["A"], leaves["B"], leaves["C"], shape.chunk, D=leaves["D"],
        initial_states=leaves["init"], return_final_state=True,
        cu_seqlens=None if cu is None else torch.tensor(cu, dtype=torch.int32, device=DEV))
    torch.autograd.backward([out, fin], [inp["dy"].to(BF), inp["dfinal"]])
    return {k: v.grad.float() for k, v in leaves.items()}


@pytest.mark.parametrize("P,H,N,Q,L,cu", SHAPES)
def test_shapes(P, H, N, Q, L, cu, monkeypatch):
    shape = SsdShape(1 if cu else 2, L, H, P, H, N, Q, cu_seqlens=cu)
    # (with z the norm's kernels round dY to bf16: dD of one or two heads, sums of 51200 and 4640 such terms that may
    # cancel to 1/24 and 1/70 of their root sum square, is then off by 2^-9 times that factor and more)
    tp._check_ext(shape, BF, with_z=bool(P % 3) and H > 2, seed=P + L, cu=cu, randw=True)
    head, general = (_grads(shape, cu, monkeypatch, e) for e in (None, "block"))
    for k in ("x", "B", "C"):
        assert_close("d" + k, head[k], general[k], 4 * 2.0 ** -9)
    for k in ("dt", "A", "D", "init"):  # (dA and ddt are differences of larger sums)
        assert_close("d" + k, head[k], general[k], 1e-2)


@pytest.mark.parametrize("Q", [64, 192, 256])
def test_growing_and_steep_heads(Q, monkeypatch):
    """A head with A > 0 and one past every decay's range, whose chunks the general path leaves to its exact fixup:
    every gradient, of either path, within the flat 1e-2 of the fp64 oracle (they land at 3.7e-3 and below)."""
    shape = SsdShape(2, 576, 8, 64, 8, 64, Q)

    def grow(inp):
        inp["A"][1], inp["A"][5] = 0.05, -400.0
        return inp

    head, general = (_grads(shape, None, monkeypatch, e, grow) for e in (None, "block"))
    inp = grow(make_inputs(shape, seed=7, device=DEV, with_init=True, with_dfinal=True))
    t = {k: (inp[k].to(BF) if k in ("x", "B", "C") else inp[k]).double().requires_grad_(True)
         for k in ("x", "dt", "A", "B", "C", "D", "init")}
    out, fin = ssd_combined(t["x"], t["dt"], t["A"], t["B"], t["C"], Q, D=t["D"], initial_states=t["init"])
    torch.autograd.backward([out, fin], [inp["dy"].to(BF).double(), inp["dfinal"].double()])
    for k, v in t.items():
        assert_close("d" + k, head[k], v.grad, 1e-2)
        assert_close("general d" + k, general[k], v.grad, 1e-2)


@pytest.mark.parametrize("exact", [False, True], ids=["drop_beta_dA", "exact_dA"])
@pytest.mark.parametrize("P,N,Q,L", [(64, 128, 256, 320), (32, 16, 64, 100), (16, 64, 192, 193), (48, 32, 128, 129)])
def test_trapezoidal(P, N, Q, L, exact):
    from test_gpu_trapz import check, make
    check(make(2, L, 4, P, 4, N, BF, seed=73), Q, exact, BF, oracle_device=DEV, oracle_dtype=torch.float32,
          tag=f"per-head P={P} N={N} Q={Q}")


def test_captured_backward_replays(monkeypatch):
    """A captured forward and backward, replayed with eager work between, equals the eager results each time."""
    import kernels
    monkeypatch.delenv("SSD_ROW_KERNEL", raising=False)
    inp = make_inputs(SsdShape(2, 384, 4, 64, 4, 64, 128), seed=9, device=DEV)
    leaves = {k: inp[k].to(BF).requires_grad_(True) for k in ("x", "B", "C")}
    leaves["dt"], leaves["A"] = (inp[k].clone().requires_grad_(True) for k in ("dt", "A"))
    dy = inp["dy"].to(BF)

    def run():
        out = kernels.ssd_scan_combined(leaves["x"], leaves["dt"], leaves["A"], leaves["B"], leaves["C"], 128)
        return torch.autograd.grad(out, list(leaves.values()), dy)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        got = run()
    for _ in range(3):
        want = run()
        g.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)


def test_more_groups_than_32_bit_offsets_reach(monkeypatch):
    """33 000 heads with B and C of their own, 128 columns each: a chunk's rows span 2.2 GB, so the general kernels run.
    The gradients of the first and last heads are those of the call on those heads alone, to the two paths' roundings."""
    import kernels
    monkeypatch.delenv("SSD_ROW_KERNEL", raising=False)
    H, L, k = 33000, 256, 4
    g = torch.Generator(device=DEV).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    full = {"x": rnd(1, L, H, 8).to(BF), "dt": torch.rand(1, L, H, generator=g, device=DEV) * 0.1,
            "A": -torch.rand(H, generator=g, device=DEV) * 4 - 1}
    for n in "BC":
        full[n] = torch.empty(1, L, H, 128, dtype=BF, device=DEV)
        for t in range(0, L, 32):
            full[n][:, t:t + 32] = rnd(1, 32, H, 128).div_(128 ** 0.5)
    dy = rnd(1, L, H, 8).to(BF)

    def grads(t, d):
        t = {n: v.requires_grad_(True) for n, v in t.items()}
        y = kernels.ssd_scan_combined(t["x"], t["dt"], t["A"], t["B"], t["C"], 256)
        return dict(zip(t, torch.autograd.grad(y, list(t.values()), d)))

    got = grads(full, dy)
    for lo in (0, H - k):
        cut = lambda n, v: (v[lo:lo + k] if n == "A" else v[:, :, lo:lo + k]).detach().contiguous()  # noqa: E731,B023
        want = grads({n: cut(n, v) for n, v in full.items()}, cut("dy", dy))
        for n in want:
            assert_close(f"d{n} from head {lo}", cut(n, got[n]), want[n], 1e-2)
