"""The dense GEMMs' small tiles: the MXFP4 ones (kern_mx_gemm_{bf16,e4m3}_t{rows}x{weights}) against the ring's
128 x 256 kernel, bit for bit (every kernel of the family accumulates K in the same order), the MXFP8 ones
(kern_mx_gemm_mxfp8_t{rows}x{weights}) against the oracle, and the rules that pick one.

Each tile runs at its edges: one row, one row short of a whole tile, one past it; K from one k group of 512 to past two
rounds of its stages, every remainder among them; fewer and more tiles than the eight XCDs. The ring kernel is compared
with the CPU oracle, by name, in test_gpu_large_tiles.py; here the entries as the C ABI picks them are as well, the walk
over wide weights is, and a launch that takes the ring for some rows and small tiles for the rest has the ring's bits
(test_pick.py holds which shapes those are).
"""
import numpy as np
import pytest

from kern_amd import workload as wl
from tests._util import assert_gemm_close, bf16_to_f32, r128c4_offsets, to_dev, to_np

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
    """Against the oracle, small tiles or (the last two, 288 and 286 ring tiles) the ring by the entry's choice."""
    print(f"[dense] M={M} N={N} K={K}", flush=True)
    w, s, q, qs = _operands(ops, M, N, K, 60)
    c = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.mxfp4_gemm_bf16(w, s, q, qs, c, M=M, m=N, k=K)
    torch.cuda.synchronize()
    _, acc = oracle.gemm_e4m3_pt(to_np(w), to_np(s), to_np(q), to_np(qs), N, K, 1.0)
    assert_gemm_close(bf16_to_f32(to_np(c)), acc, "dense")


def _mxfp8(ops, rows, K, seed):
    """MXFP8 rows as quantized on the device, scales tiled 128x4 with NaN codes in the padding."""
    q, sf = ops.quantize_mxfp8(to_dev(wl.activations_bf16(seed, rows, K, outlier_frac=0.01)))
    t = np.full(ops.r128c4_bytes(rows, K // 32), 255, np.uint8)
    t[r128c4_offsets(rows, K // 32)] = to_np(sf)
    return to_np(q), t


@pytest.mark.parametrize("rows,weights", [(16, 16), (16, 32), (16, 64), (32, 64), (32, 128), (48, 64), (64, 64)])
def test_mxfp8_tiles(ops, oracle, rows, weights):
    """K from one 32-wide block to past two k-tiles a wave (8 waves take every eighth 128-wide k-tile), partial last
    k-tiles; rows one short of and one past whole tiles and across a 128-row scale block; n and ldc odd."""
    mod = ops.Module(ops.HSACO_PATH)
    for M, N, K in [(1, 1, 32), (rows, weights, 128), (rows - 1, weights + 1, 1000 // 32 * 32), (3 * rows + 1, 263, 1120),
                    (130, 200, 2112), (rows + 1, 2 * weights - 3, 3200)]:
        print(f"[tile8] {rows}x{weights} M={M} N={N} K={K}", flush=True)
        (qa, ta), (qw, tw) = _mxfp8(ops, M, K, 80), _mxfp8(ops, N, K, 81)
        ldc = N + 3
        out = torch.full((M + 1, ldc), 7.0, dtype=torch.bfloat16, device="cuda")
        mt, ng = rows // 16, weights // 16
        mod.launch(f"kern_mx_gemm_mxfp8_t{rows}x{weights}", (-(-N // weights), -(-M // rows)), (512,), to_dev(qa), to_dev(qw),
                   out, to_dev(ta), to_dev(tw), M, N, K, ldc, shared=max(32768 * (mt + 1), 8192 * mt * ng))
        torch.cuda.synchronize()
        got = bf16_to_f32(to_np(out))
        assert (got[:, N:] == 7.0).all() and (got[M] == 7.0).all()
        assert_gemm_close(got[:M, :N], oracle.mxfp8_gemm(qa, qw, ta, tw, M, N, K), f"{rows}x{weights} {M}x{N}x{K}")
    mod.close()


@pytest.mark.parametrize("N,K,hb", [(256, 1024, 1), (4352, 2048, 3), (2304, 4096, 9), (9216, 7168, 5), (512, 8192, 2)])
def test_saved_walk_launch(ops, oracle, N, K, hb):
    """The walk (kern_mx_gemm_bf16_s{K / 1024}) as a manifest op saved before there were tiles launches it, with any share
    of half groups: against the oracle at ragged token counts."""
    from tests.test_pick import saved_walk_op

    op = ops.ManifestOp(saved_walk_op(N, K, hb))
    for M in (1, 17, 50, 64):
        print(f"[walk] M={M} N={N} K={K} hb={hb}", flush=True)
        w, s, q, qs = _operands(ops, M, N, K, 90)
        c = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
        op(w, s, q, qs, c, vars={"tokens": M})
        torch.cuda.synchronize()
        got = bf16_to_f32(to_np(c))
        assert (got[M] == 7.0).all()
        _, acc = oracle.gemm_e4m3_pt(to_np(w), to_np(s), to_np(q), to_np(qs), N, K, 1.0)
        assert_gemm_close(got[:M], acc, f"walk {M}x{N}x{K}")


@pytest.mark.parametrize("N,K", [(2048, 8192), (4352, 1024), (7168, 8192), (8448, 4096), (18688, 1024)])
def test_dense_op_has_the_c_abi_bits_up_to_64_rows(ops, N, K):
    """Each launch of the manifest op at the edges of its rows: the walk where the C ABI takes it, else the ring's bits."""
    from kern_amd import manifest as mf

    op = ops.ManifestOp(mf.mxfp4_gemm_bf16(N, K))
    w, s, q, qs = _operands(ops, 65, N, K, 95)
    for M in (1, 16, 17, 32, 33, 48, 49, 64, 65):
        print(f"[dense op] M={M} N={N} K={K}", flush=True)
        c, m = (torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        ops.mxfp4_gemm_bf16(w, s, q[:M], qs[:M], c, M=M, m=N, k=K)
        op(w, s, q[:M], qs[:M], m, vars={"tokens": M})
        torch.cuda.synchronize()
        assert torch.equal(c.view(torch.int16), m.view(torch.int16)), M


@pytest.mark.parametrize("M,N,K", [(2446, 3584, 1024), (1410, 6144, 1536)])  # "split" in test_pick.py's test_dense_routes
@pytest.mark.parametrize("dbg", [False, True])
def test_split_has_the_rings_bits(ops, oracle, M, N, K, dbg):
    """Whole rounds on the ring and the remaining rows on small tiles, in both outputs, against the ring alone: every
    operand's and output's offset of the second launch."""
    print(f"[split] M={M} N={N} K={K}", flush=True)
    mod = ops.Module(ops.HSACO_PATH)
    w, s, q, qs = _operands(ops, M, N, K, 70)
    ds = torch.tensor([1.0 / 16], dtype=torch.float32, device="cuda")
    for out, fn, extra in ((torch.bfloat16, ops.mxfp4_gemm_bf16, ()), (torch.uint8, ops.mxfp4_gemm_e4m3, (ds,))):
        ring, got = (torch.full((M + 1, N), 77, dtype=out, device="cuda") for _ in range(2))
        acc = [torch.full((M + 1, N), 7.0, dtype=torch.float32, device="cuda") for _ in range(2)] if dbg else [0, None]
        name = "kern_mx_gemm_" + ("bf16" if out == torch.bfloat16 else "e4m3")
        mod.launch(name, (N // 256, -(-M // 128)), (512,), w, s, q, qs, ring, *extra, M, N, K, acc[0])
        fn(w, s, q, qs, got, *extra, M=M, m=N, k=K, dbg=acc[1])
        torch.cuda.synchronize()
        assert torch.equal(ring.view(torch.uint8), got.view(torch.uint8)), name
        if dbg:
            assert torch.equal(acc[0], acc[1]), name
    mod.close()
