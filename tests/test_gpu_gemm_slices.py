"""dB / dC of the bf16 backward where few (chunk, group, 64-token) blocks split the heads and the tile terms of the
row kernel over more blocks (csrc/ssd_capi.hip, gemm_slices): both kinds of split and the sizes next to their
limits, head counts that leave a short last slice, partial and empty chunks, narrow states, heads that take the
exact fixup, the trapezoidal scan (each slice its share of the diagonal) in both gradient settings, all against the
oracle at 1e-2 of bf16 inputs (ssd_testlib.TOL); and two runs are the same bits."""
from __future__ import annotations

import pytest
import torch

import test_gpu_parity as tp
import test_gpu_rows as tr
from conftest import gpu_available
from oracle.inputs import SsdShape, make_inputs

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs an MI355X (HIP device)")]

DEV, BF = "cuda", torch.bfloat16


@pytest.mark.parametrize("b,L,H,P,G,N,Q,cu", [
    (1, 256, 24, 64, 1, 128, 256, None),               # one chunk: four slices, a slice per tile step
    (1, 200, 7, 64, 1, 64, 256, None),                 # 7 heads in slices of 3, 3 and 1; a partial chunk
    (1, 70, 6, 32, 1, 16, 64, None),                   # fewest heads that split; half a state tile
    (1, 1, 10, 64, 1, 128, 64, None),                  # one token
    (2, 256, 10, 48, 2, 40, 128, None),                # 5 heads per group: whole
    (1, 2048, 24, 64, 1, 32, 256, None),               # 32 blocks, the last of the first rule
    (1, 2304, 16, 64, 1, 32, 256, None),               # 36 blocks, two slices and one for the tile terms
    (2, 2048, 37, 32, 1, 64, 256, None),               # 64 blocks, 37 heads in slices of 13, 13 and 11
    (1, 256, 48, 64, 8, 128, 256, None),               # one chunk of eight groups: blocks on every XCD
    (1, 700, 18, 64, 3, 32, 256, None),                # three chunks of three groups, slices of 2
    (9, 128, 16, 32, 2, 32, 128, None),                # nine chunks: a second round of XCDs, padded to 16
    (1, 900, 16, 64, 2, 64, 256, [0, 1, 1, 258, 900]),  # packed: a token, none, two chunks, a remainder
])
def test_shapes(b, L, H, P, G, N, Q, cu):
    tp._check_ext(SsdShape(b, L, H, P, G, N, Q, cu_seqlens=cu), BF, with_z=False, seed=P + L, cu=cu, randw=True)


@pytest.mark.parametrize("H", [8, 18])
def test_growing_and_steep_heads(H):
    tr._ext_check(SsdShape(1, 512, H, 64, 1, 64, 256), seed=72, fix_heads=True, with_z=False)


@pytest.mark.parametrize("exact", [False, True], ids=["drop_beta_dA", "exact_dA"])
@pytest.mark.parametrize("L,H,P,N,Q", [(300, 8, 64, 128, 256), (2300, 16, 32, 32, 256), (65, 7, 64, 64, 64)])
def test_trapezoidal(L, H, P, N, Q, exact):
    from test_gpu_trapz import check, make
    check(make(1, L, H, P, 1, N, BF, seed=73), Q, exact, BF, oracle_device=DEV, oracle_dtype=torch.float32,
          tag=f"sliced H={H}")


def test_same_bits():
    import kernels
    inp = make_inputs(SsdShape(1, 300, 24, 64, 1, 64, 128), seed=5, device=DEV)
    x, B, C = (inp[k].to(BF).requires_grad_(True) for k in ("x", "B", "C"))
    runs = [torch.autograd.grad(kernels.ssd_scan_combined(x, inp["dt"], inp["A"], B, C, 128), [x, B, C],
                                inp["dy"].to(BF)) for _ in range(2)]
    assert all(torch.equal(a, b) for a, b in zip(*runs))
