"""The large-tile GEMM kernels launched by name: the ring's 128 x 256 tiles (kern_mx_gemm_e4m3, kern_mx_gemm_bf16) and
kern_mx_gemm_mxfp8. The entry points send small shapes to small tiles, so the tests of those entry points reach these
kernels at whole tiles only; here the same tests run with the three GEMM entry points replaced by launches of the large
kernels: ragged last tiles (every case of the ring's activation loader), extreme scales, operands above address bit 31,
ragged m, n, k and row strides. Larger ragged batches of every caller run on them."""
import numpy as np
import pytest

from kern_amd import workload as wl
from tests import test_gpu_codecs as codecs
from tests import test_gpu_ops as gpu_ops
from tests import test_gpu_sweep as sweep
from tests._util import assert_gemm_close, bf16_to_f32, r128c4_offsets, to_dev, to_np

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


class LargeTiles:
    """kern_amd.ops with the GEMMs launched on the large kernels whatever their shape."""

    def __init__(self, ops):
        self._ops, self._mod = ops, ops.Module(ops.HSACO_PATH)

    def __getattr__(self, name):
        return getattr(self._ops, name)

    def mxfp4_gemm_e4m3(self, a, sf_a, b, sf_b, c, d_scale, *, M, m, k, dbg=None):
        assert m % 256 == 0 and k % 512 == 0 and b.numel() >= M * k and c.numel() >= M * m
        self._mod.launch("kern_mx_gemm_e4m3", (m // 256, -(-M // 128)), (512,), a, sf_a, b, sf_b, c, d_scale, M, m, k,
                         0 if dbg is None else dbg)

    def mxfp4_gemm_bf16(self, a, sf_a, b, sf_b, c, *, M, m, k, dbg=None):
        assert m % 256 == 0 and k % 512 == 0 and b.numel() >= M * k and c.numel() >= M * m
        self._mod.launch("kern_mx_gemm_bf16", (m // 256, -(-M // 128)), (512,), a, sf_a, b, sf_b, c, M, m, k,
                         0 if dbg is None else dbg)

    def cublaslt_mxfp8_tn(self, a, w, c, a_sf, w_sf, m, n, k, ldc=None):
        ldc = n if ldc is None else ldc
        assert k % 32 == 0 and a.numel() >= m * k and w.numel() >= n * k and c.numel() >= (m - 1) * ldc + n
        assert a_sf.numel() >= self._ops.r128c4_bytes(m, k // 32) and w_sf.numel() >= self._ops.r128c4_bytes(n, k // 32)
        self._mod.launch("kern_mx_gemm_mxfp8", (-(-n // 256), -(-m // 128)), (512,), a, w, c, a_sf, w_sf, m, n, k, ldc)


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from kern_amd import ops

    ops.lib()
    return LargeTiles(ops)


@pytest.mark.parametrize("M,m,k", [(1, 256, 512), (5, 512, 1024), (17, 512, 1536), (148, 512, 1024), (168, 512, 1024),
                                   (198, 512, 1024), (218, 512, 1024), (228, 512, 1024), (248, 512, 1024),
                                   (300, 512, 1024)])
def test_ring_e4m3(ops, oracle, M, m, k):
    gpu_ops.test_gemm_e4m3_per_tensor(ops, oracle, M, m, k)


@pytest.mark.parametrize("i,M,m,k", [(i,) + c for i, c in enumerate(sweep._gemm_cases())][::2])
def test_ring_bf16(ops, oracle, i, M, m, k):
    sweep.test_gemm_bf16_sweep(ops, oracle, i, M, m, k)


def test_ring_operands_above_bit31(ops, oracle):
    gpu_ops.test_ring_operands_above_bit31(ops, oracle)


def test_ring_extreme_scales(ops):
    codecs.test_gemm_extreme_scales(ops)


@pytest.mark.parametrize("m,n,k", [(300, 520, 1024), (64, 1000, 2080), (200, 256, 96)])
def test_mxfp8(ops, oracle, m, n, k):
    gpu_ops.test_mxfp8_gemm_random(ops, oracle, m, n, k)


def test_mxfp8_kat(ops):
    gpu_ops.test_mxfp8_gemm_kat(ops)


def test_mxfp8_extreme_scales(ops):
    codecs.test_mxfp8_gemm_extreme_scales(ops)


@pytest.mark.parametrize("M,N,K", [(1, 1, 32), (129, 257, 160), (255, 263, 1120), (383, 519, 2144), (127, 255, 384)])
def test_mxfp8_odd_edges(ops, oracle, M, N, K):
    """Odd n and ldc (stores not 8-byte aligned), rows one past and one short of whole tiles, a partial last k-tile, and
    NaN codes in the scales' padding."""
    print(f"[mxfp8] M={M} N={N} K={K}", flush=True)

    def operand(rows, seed):
        q, sf = ops.quantize_mxfp8(to_dev(wl.activations_bf16(seed, rows, K, outlier_frac=0.01)))
        t = np.full(ops.r128c4_bytes(rows, K // 32), 255, np.uint8)
        t[r128c4_offsets(rows, K // 32)] = to_np(sf)
        return to_np(q), t

    (qa, ta), (qw, tw) = operand(M, 84), operand(N, 85)
    ldc = N + 3
    out = torch.full((M + 1, ldc), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.cublaslt_mxfp8_tn(to_dev(qa), to_dev(qw), out, to_dev(ta), to_dev(tw), M, N, K, ldc=ldc)
    torch.cuda.synchronize()
    got = bf16_to_f32(to_np(out))
    assert (got[:, N:] == 7.0).all() and (got[M] == 7.0).all()
    assert_gemm_close(got[:M, :N], oracle.mxfp8_gemm(qa, qw, ta, tw, M, N, K), f"mxfp8 {M}x{N}x{K}")
