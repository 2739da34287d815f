"""The decode GEMV at every K of its range against the oracle: the row-group entries (kern_mx_gemv_bf16_r{K/512}) and
the persistent walk (kern_mx_gemv_bf16_p{ceil(K/1024)}, with an h where K is an odd multiple of 512), each launched
directly and through the C ABI's choice, which is also compared with the manifest op's. Past K = 8192 the looping and
slice-staging kernels. Row shares are ragged, x holds infinities next to the k-tiles that an `h` entry's waves skip."""
import numpy as np
import pytest

from kern_amd import manifest as mf
from kern_amd import workload as wl
from tests._util import bf16_to_f32, to_dev, to_np

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from kern_amd import ops

    ops.lib()
    return ops


def assert_gemm_close(got, ref, what):
    """The relative Frobenius error is at most that of one bf16 rounding, 2^-8 of each output, and 1e-4 for the f32
    sums in another order. (The 2e-3 that other tests hold averages over many outputs; 16 outputs need not meet it: one
    rounding of the largest gave 2.2e-3.) A k-tile left out or taken twice is at least 1/8 at K = 8192."""
    err = np.asarray(got, np.float64) - ref
    rel = np.sqrt((err**2).sum() / (np.asarray(ref, np.float64)**2).sum())
    assert rel <= 2.0**-8 + 1e-4, f"{what}: {rel:.3g}"


@pytest.mark.parametrize("kg", list(range(1, 17)) + [17, 19, 32])
def test_gemv_every_length(ops, oracle, kg):
    K, mod = 512 * kg, ops.Module(ops.HSACO_PATH)
    for M, N in [(1, 16), (2, 1040), (3, 528), (4, 4112), (5, 272), (16, 48)]:
        print(f"[gemv] M={M} N={N} K={K}", flush=True)
        x = wl.activations_bf16(400 + kg, M, K)
        w, sf = wl.mxfp4_weights(410 + kg, 1, N, K, 122, 132)
        wp, sfp = ops.repack_weights(to_dev(w[0]), to_dev(sf[0]))
        want = oracle.gemv_w4a16(x, w[0], sf[0])[1]
        xd, y = to_dev(x), torch.empty((M, N), dtype=torch.bfloat16, device="cuda")

        def check(name, launch):
            y.fill_(float("nan"))
            launch()
            torch.cuda.synchronize()
            assert_gemm_close(bf16_to_f32(to_np(y)), want, f"{name} M={M} N={N} K={K}")

        check("picked", lambda: ops.mxfp4_gemv_bf16(xd, wp, sfp, y, M, N=N, K=K))
        picked = y.clone()
        op = ops.ManifestOp(mf.mxfp4_gemv_bf16(N, K))
        check("manifest", lambda: op(xd, wp, sfp, y, vars={"tokens": M}))
        assert torch.equal(y.view(torch.int16), picked.view(torch.int16))
        if kg > 16:
            continue
        if 2 * M * K <= 144 * 1024:
            check("row groups", lambda: mod.launch(f"kern_mx_gemv_bf16_r{kg}", (N // 16,), (256,), xd, wp, sfp, y, M, N,
                                                   K, shared=2 * M * K))
        for hb in (1, 7, 9):
            check("walk", lambda: mod.launch(f"kern_mx_gemv_bf16_p{(kg + 1) // 2}{'h' if kg % 2 else ''}",
                                             (-(-(N // 8) // hb),), (512,), xd, wp, sfp, y, M, N, K, hb))
    mod.close()


@pytest.mark.parametrize("kg", [1, 5, 15])
def test_gemv_infinite_rows_stay_apart(ops, oracle, kg):
    """A token's infinities reach its own outputs only, the skipped k-tile's (the next token's first) among them."""
    M, N, K = 6, 128, 512 * kg
    mod = ops.Module(ops.HSACO_PATH)
    x = wl.activations_bf16(430, M, K)
    w, sf = wl.mxfp4_weights(431, 1, N, K, 122, 132)
    wp, sfp = ops.repack_weights(to_dev(w[0]), to_dev(sf[0]))
    want = oracle.gemv_w4a16(x, w[0], sf[0])[1]
    xi = x.copy()
    xi[1::2, :] = 0x7F80
    xd = to_dev(xi)
    for name, grid, block, extra, lds in [(f"r{kg}", N // 16, 256, (), 2 * M * K),
                                          (f"p{(kg + 1) // 2}h", N // 24 + 1, 512, (3,), 0)]:
        print(f"[gemv] infinities {name}", flush=True)
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        mod.launch("kern_mx_gemv_bf16_" + name, (grid,), (block,), xd, wp, sfp, y, M, N, K, *extra, shared=lds)
        torch.cuda.synchronize()
        got = bf16_to_f32(to_np(y))
        assert np.isfinite(got[0::2]).all()
        assert_gemm_close(got[0::2], want[0::2], name)
    mod.close()
