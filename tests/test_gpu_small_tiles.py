"""The dense GEMM's small tiles (kern_mx_gemm_{bf16,e4m3}_t{rows}x{weights}) against the ring's 128 x 256 kernel, bit
for bit (every kernel of the family accumulates K in the same order), and the rule that picks one.

Each tile runs at its edges: one row, one row short of a whole tile, one past it; K from one k group of 512 to past two
rounds of its stages, every remainder among them; fewer and more tiles than the eight XCDs. The ring kernel is compared
with the CPU oracle in test_gpu_stack.py and test_gpu_sweep.py; here the entry as the C ABI picks it is as well, on both
sides of a switch and where it takes the ring for some rows and small tiles for the rest.
"""
import os

import pytest

from kern_amd import workload as wl
from tests._util import assert_gemm_close, bf16_to_f32, to_dev, to_np

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TILES = [(16, 32, 2, 8), (16, 64, 4, 8), (16, 128, 8, 4), (32, 128, 8, 4), (48, 128, 8, 4), (80, 128, 8, 3),
         (32, 256, 8, 3), (48, 256, 8, 3), (64, 256, 8, 3)]  # rows, weights, waves, stages


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from kern_amd import ops

    ops.lib()
    return ops


def _operands(ops, M, N, K, seed):
    w, s = (torch.empty((1, N, n), dtype=torch.uint8, device="cuda") for n in (K // 2, K // 32))
    ops.fill_random_u8(w, seed)
    ops.fill_random_u8(s, seed + 1, 119, 6)
    wp, sp = ops.repack_weights(w, s)
    q, qs = ops.quantize_mxfp8(to_dev(wl.activations_bf16(seed + 2, M, K, outlier_frac=0.01)))
    return wp[0], sp[0], q, qs


@pytest.mark.parametrize("rows,weights,waves,stages", TILES)
def test_tiles_have_the_rings_bits(ops, rows, weights, waves, stages):
    mod = ops.Module(ops.HSACO_PATH)
    N = 768
    for groups in list(range(1, stages + 2)) + [2 * stages, 2 * stages + 1]:
        K = 512 * groups
        M = {0: 1, 1: rows, 2: rows - 1}.get(groups % 4, 3 * rows + 1)
        print(f"[tile] {rows}x{weights} M={M} N={N} K={K}", flush=True)
        w, s, q, qs = _operands(ops, M, N, K, 40 + groups)
        ds = torch.tensor([1.0 / 16], dtype=torch.float32, device="cuda")
        lds = stages * rows * 512 + -(-rows * (K // 512 + 1) // 64) * 1024
        for out, extra in ((torch.bfloat16, ()), (torch.uint8, (ds,))):
            name = "kern_mx_gemm_" + ("bf16" if out == torch.bfloat16 else "e4m3")
            ring, tile = (torch.full((M + 2, N), 77, dtype=out, device="cuda") for _ in range(2))
            dbg = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
            mod.launch(name, (N // 256, -(-M // 128)), (512,), w, s, q, qs, ring, *extra, M, N, K, 0)
            for d in (0, dbg):
                tile.fill_(77)
                mod.launch(f"{name}_t{rows}x{weights}", (-(-N // weights), -(-M // rows)), (64 * waves,), w, s, q, qs,
                           tile, *extra, M, N, K, d, shared=lds)
                torch.cuda.synchronize()
                assert torch.equal(ring.view(torch.uint8), tile.view(torch.uint8)), (name, M, K)
            if out == torch.bfloat16:
                assert torch.equal(dbg.to(torch.bfloat16), tile[:M]), (M, K)
    mod.close()


@pytest.mark.parametrize("M,N,K", [(16, 256, 512), (100, 512, 1024), (130, 768, 1536), (40, 6144, 3584),
                                   (1100, 8192, 512), (1540, 5632, 512)])
def test_dense_gemm_as_picked(ops, oracle, M, N, K):
    """Against the oracle; (1540, 5632, 512) has 286 ring tiles, so rows past the ring's first round may go to small tiles."""
    print(f"[dense] M={M} N={N} K={K}", flush=True)
    w, s, q, qs = _operands(ops, M, N, K, 60)
    c = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.mxfp4_gemm_bf16(w, s, q, qs, c, M=M, m=N, k=K)
    torch.cuda.synchronize()
    _, acc = oracle.gemm_e4m3_pt(to_np(w), to_np(s), to_np(q), to_np(qs), N, K, 1.0)
    assert_gemm_close(bf16_to_f32(to_np(c)), acc, "dense")
