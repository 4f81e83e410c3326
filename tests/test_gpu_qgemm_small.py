"""q38a_qgemm at 9 to 64 rows (and fewer on narrow weights): every epilogue against the oracle's product
over the exact weights, at the edges of its row blocks, with fewer groups than waves, K shares of
unequal length, one and two column waves (weights wide enough for 64-column tiles over the whole K),
and stores that cannot be 16 bytes wide. Bounds as in test_gpu_qgemm.py."""
import numpy as np
import pytest
import torch

from q38a import gemm
from gpu_util import dev, host, stream
from test_gpu_qgemm import Weight, check_residual, close, row_scales, workspace
from util import assert_bits_equal, bf16_bits_to_f32, randn_bf16

pytestmark = pytest.mark.gpu

SHAPES = [(9, 256, 64), (31, 512, 320), (32, 12288, 128), (33, 12288, 192), (64, 2560, 1088), (63, 256, 2048),
          (5, 256, 576), (33, 256, 64), (64, 256, 192)]


@pytest.mark.parametrize("bits", [4, 5, 6])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_small_rows(orc, bits, m, n, k):
    w = Weight(orc, bits, n, k, seed=3 * bits + m)
    rng = np.random.default_rng(m + n)
    a = randn_bf16(rng, (m, k))
    hidden = 128 * max(1, k // 128)
    partials = rng.uniform(50.0, 200.0, (m, hidden // 128)).astype(np.float32)
    a_t, p_t = dev(a), dev(partials)
    ws, keep = workspace(m, n, k)
    want = orc.qgemm(a, w.w_exact, 3, partials_in=partials, hidden=hidden)
    rs = row_scales(partials, hidden)
    print(f"small: bits={bits} m={m} n={n} k={k}", flush=True)
    for ldo, n_store, shift in ((n, 0, 0), (n + 3, n - 5, 1)):
        runs = []
        for rep in range(2):
            out = torch.full((m * ldo + 8,), -21846, dtype=torch.int16, device="cuda")
            ep = gemm.GemmEpilogue(gemm.EPI_STORE_BF16, out.data_ptr() + 2 * shift, ldo, n_store, None, None, None,
                                   p_t.data_ptr(), hidden, 1e-6)
            gemm.qgemm(a_t.data_ptr(), m, w.desc, ep, ws, stream())
            runs.append(host(out, np.uint16))
        got, cols = runs[0][shift:shift + m * ldo].reshape(m, ldo), n_store or n
        close(bf16_bits_to_f32(got[:, :cols]), want[:, :cols], "bf16", a, w.w_offset_mag[:cols], rs)
        assert (got[:, cols:] == 0xAAAA).all(), "columns past n_store are not written"
        assert_bits_equal(runs[1], runs[0], "second launch")
    outf = torch.zeros(m * (n + 1), dtype=torch.float32, device="cuda")
    ep = gemm.GemmEpilogue(gemm.EPI_STORE_F32, outf.data_ptr(), n + 1, n - 1, None, None, None, None, 0, 1e-6)
    gemm.qgemm(a_t.data_ptr(), m, w.desc, ep, ws, stream())
    got = host(outf).reshape(m, n + 1)
    close(got[:, :n - 1], orc.qgemm(a, w.w_exact, 3)[:, :n - 1], "f32", a, w.w_offset_mag[:n - 1], out="f32")
    assert (got[:, n - 1:] == 0).all()
    if m > 8:  # (fewer rows: the wide-tile kernel or this one, by shape)
        res0 = rng.standard_normal((m, n)).astype(np.float32)
        res, xbf = dev(res0), torch.zeros(m * n, dtype=torch.int16, device="cuda")
        pout = torch.zeros(m * (n // 128), dtype=torch.float32, device="cuda")
        ep = gemm.GemmEpilogue(gemm.EPI_RESIDUAL, None, 0, 0, res.data_ptr(), xbf.data_ptr(), pout.data_ptr(), None, 0, 1e-6)
        gemm.qgemm(a_t.data_ptr(), m, w.desc, ep, ws, stream())
        check_residual(orc, w, a, res0, host(res).reshape(m, n), host(xbf, np.uint16).reshape(m, n),
                       host(pout).reshape(m, n // 128))


@pytest.mark.parametrize("m,n,k,kind", [(5, 256, 576, gemm.EPI_STORE_BF16), (9, 512, 320, gemm.EPI_STORE_F32),
                                        (33, 12288, 128, gemm.EPI_STORE_BF16), (64, 2560, 1088, gemm.EPI_RESIDUAL),
                                        (129, 512, 640, gemm.EPI_RESIDUAL), (200, 256, 448, gemm.EPI_STORE_BF16),
                                        (1800, 8192, 128, gemm.EPI_STORE_BF16)])
def test_unaligned_a(orc, m, n, k, kind):
    """A on a 2-byte boundary, which the copies into LDS are not made for: rows through registers, 64 a
    launch. The same bits as the oracle's bounds allow, with every row's scale, residual and sums in place."""
    w = Weight(orc, 6, n, k, seed=m + 1)
    rng = np.random.default_rng(m + k)
    a = randn_bf16(rng, (m, k))
    shifted = torch.zeros(m * k + 8, dtype=torch.int16, device="cuda")
    shifted[3:3 + m * k] = dev(a).view(-1)
    ap = shifted.data_ptr() + 6
    hidden = 128 * max(1, k // 128)
    partials = rng.uniform(50.0, 200.0, (m, hidden // 128)).astype(np.float32)
    p_t = dev(partials)
    ws, keep = workspace(m, n, k)
    print(f"unaligned A: m={m} n={n} k={k} kind={kind}", flush=True)
    if kind == gemm.EPI_RESIDUAL:
        res0 = rng.standard_normal((m, n)).astype(np.float32)
        res, xbf = dev(res0), torch.zeros(m * n, dtype=torch.int16, device="cuda")
        pout = torch.zeros(m * (n // 128), dtype=torch.float32, device="cuda")
        ep = gemm.GemmEpilogue(kind, None, 0, 0, res.data_ptr(), xbf.data_ptr(), pout.data_ptr(), None, 0, 1e-6)
        gemm.qgemm(ap, m, w.desc, ep, ws, stream())
        check_residual(orc, w, a, res0, host(res).reshape(m, n), host(xbf, np.uint16).reshape(m, n),
                       host(pout).reshape(m, n // 128))
        return
    f32 = kind == gemm.EPI_STORE_F32
    out = torch.zeros(m * n, dtype=torch.float32 if f32 else torch.int16, device="cuda")
    ep = gemm.GemmEpilogue(kind, out.data_ptr(), n, 0, None, None, None, p_t.data_ptr(), hidden, 1e-6)
    gemm.qgemm(ap, m, w.desc, ep, ws, stream())
    got = host(out).reshape(m, n) if f32 else bf16_bits_to_f32(host(out, np.uint16).reshape(m, n))
    want = orc.qgemm(a, w.w_exact, 3, partials_in=partials, hidden=hidden)
    close(got, want, "unaligned", a, w.w_offset_mag, row_scales(partials, hidden), out="f32" if f32 else "bf16")
