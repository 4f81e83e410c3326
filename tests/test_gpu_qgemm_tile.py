"""The 128- and 256-row tiles of q38a_qgemm (33 rows and more, below the large-M kernel): every epilogue
against the oracle's product over the exact weights, at the edges of the tiles (rows one past a tile,
one group of K, an odd number of groups for tiles that take two at a time, K slices of unequal length),
with stores that cannot be 16 bytes wide, and without the split workspace where it is optional. Bounds
as in test_gpu_qgemm.py: one rounding step of the output plus the fp32 accumulation."""
import numpy as np
import pytest
import torch

from q38a import gemm
from gpu_util import dev, host, stream
from test_gpu_qgemm import Weight, big_path, check_residual, close, row_scales, workspace
from util import assert_bits_equal, bf16_bits_to_f32, randn_bf16

pytestmark = pytest.mark.gpu

# (rows, columns, K): tile edges 64/128/256, one group, odd group counts, K slices that do not divide
SHAPES = [(33, 256, 64), (64, 256, 192), (65, 512, 576), (128, 256, 1088), (129, 512, 640), (255, 256, 448),
          (257, 768, 320), (300, 2560, 704)]


@pytest.mark.parametrize("bits", [4, 5, 6])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_tile_store(orc, bits, m, n, k):
    """StoreBF16 with the folded norm (aligned, and to rows of an odd stride with columns left out) and
    StoreF32, the same bits on a second launch."""
    assert not big_path(m, n)
    w = Weight(orc, bits, n, k, seed=7 * bits + m)
    rng = np.random.default_rng(m + n)
    a = randn_bf16(rng, (m, k))
    hidden = 128 * max(1, k // 128)
    partials = rng.uniform(50.0, 200.0, (m, hidden // 128)).astype(np.float32)
    a_t, p_t = dev(a), dev(partials)
    rs = row_scales(partials, hidden)
    want = orc.qgemm(a, w.w_exact, 3, partials_in=partials, hidden=hidden)
    ws, keep = workspace(m, n, k)
    for ldo, n_store, shift in ((n, 0, 0), (n + 3, n - 5, 1)):
        print(f"tile bf16: bits={bits} m={m} n={n} k={k} ldo={ldo}", flush=True)
        runs = []
        for rep in range(2):
            out = torch.full((m * ldo + 8,), -21846, dtype=torch.int16, device="cuda")
            ep = gemm.GemmEpilogue(gemm.EPI_STORE_BF16, out.data_ptr() + 2 * shift, ldo, n_store, None, None, None,
                                   p_t.data_ptr(), hidden, 1e-6)
            gemm.qgemm(a_t.data_ptr(), m, w.desc, ep, ws, stream())
            runs.append(host(out, np.uint16))
        got = runs[0][shift:shift + m * ldo].reshape(m, ldo)
        cols = n_store or n
        close(bf16_bits_to_f32(got[:, :cols]), want[:, :cols], "bf16", a, np.abs(w.w_exact[:cols]), rs)
        assert (got[:, cols:] == 0xAAAA).all(), "columns past n_store are not written"
        assert_bits_equal(runs[1], runs[0], "second launch")
    outf = torch.zeros(m * (n + 1), dtype=torch.float32, device="cuda")
    ep = gemm.GemmEpilogue(gemm.EPI_STORE_F32, outf.data_ptr(), n + 1, n - 1, None, None, None, None, 0, 1e-6)
    gemm.qgemm(a_t.data_ptr(), m, w.desc, ep, ws, stream())
    got = host(outf).reshape(m, n + 1)
    close(got[:, :n - 1], orc.qgemm(a, w.w_exact, 3)[:, :n - 1], "f32", a, np.abs(w.w_exact[:n - 1]), out="f32")
    assert (got[:, n - 1:] == 0).all()


@pytest.mark.parametrize("m,n,k,shift", [(33, 256, 64, 0), (129, 512, 640, 1), (300, 2560, 704, 0)])
def test_tile_residual(orc, m, n, k, shift):
    """The residual epilogue, also on buffers that take no 16-byte access."""
    w = Weight(orc, 5, n, k, seed=m)
    rng = np.random.default_rng(m)
    a = randn_bf16(rng, (m, k))
    res0 = rng.standard_normal((m, n)).astype(np.float32)
    a_t = dev(a)
    ws, keep = workspace(m, n, k)
    res = torch.zeros(m * n + 4, dtype=torch.float32, device="cuda")
    res[shift:shift + m * n] = dev(res0).view(-1)
    xbf = torch.zeros(m * n + 4, dtype=torch.int16, device="cuda")
    pout = torch.zeros(m * (n // 128), dtype=torch.float32, device="cuda")
    ep = gemm.GemmEpilogue(gemm.EPI_RESIDUAL, None, 0, 0, res.data_ptr() + 4 * shift, xbf.data_ptr() + 2 * shift,
                           pout.data_ptr(), None, 0, 1e-6)
    print(f"tile residual: m={m} n={n} k={k} shift={shift}", flush=True)
    gemm.qgemm(a_t.data_ptr(), m, w.desc, ep, ws, stream())
    check_residual(orc, w, a, res0, host(res)[shift:shift + m * n].reshape(m, n),
                   host(xbf, np.uint16)[shift:shift + m * n].reshape(m, n), host(pout).reshape(m, n // 128))


def test_tile_without_workspace(orc):
    """A launch that fills the GPU unsplit runs without the split workspace; a small one is refused."""
    from q38a import Q38AError
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    none = gemm.GemmWorkspace(None, 0, None, 0)
    n, k = 2560, 512
    m = 64 * (-(-2 * cus // (n // 256))) + 1  # two 64 x 256 tiles a CU
    assert not big_path(m, n)
    w = Weight(orc, 4, n, k, seed=3)
    a = randn_bf16(np.random.default_rng(5), (m, k))
    a_t = dev(a)
    out = torch.zeros(m * n, dtype=torch.int16, device="cuda")
    ep = gemm.GemmEpilogue(gemm.EPI_STORE_BF16, out.data_ptr(), n, 0, None, None, None, None, 0, 1e-6)
    print(f"no workspace: m={m}", flush=True)
    gemm.qgemm(a_t.data_ptr(), m, w.desc, ep, none, stream())
    rows = np.r_[0:3, m - 2:m]
    close(bf16_bits_to_f32(host(out, np.uint16).reshape(m, n)[rows]), orc.qgemm(a[rows], w.w_exact, 3), "bf16", a[rows],
          np.abs(w.w_exact))
    assert gemm.workspace_size(64, 512, 4096)[0] > 0
    small = gemm.BQWeight(w.desc.lo, None, w.desc.scales, 4, 512, 4096, 512)  # (refused before it is read)
    with pytest.raises(Q38AError):
        gemm.qgemm(a_t.data_ptr(), 64, small, ep, none, stream())


@pytest.mark.parametrize("n,k", [(14336, 5120), (5120, 6144), (512, 4096)])
def test_workspace_serves_fewer_rows(n, k):
    """The workspace of m rows is enough for every smaller m, also where m itself needs none."""
    last = (0, 0)
    for m in [*range(1, 140), *range(140, 2300, 37)]:
        size = gemm.workspace_size(m, n, k)
        assert size[0] >= last[0] and size[1] >= last[1], (m, size, last)
        last = size


def test_smaller_launch_in_a_larger_workspace(orc):
    """128 rows of the in-projection's shape split K; they run in the workspace of 512 rows, which do not."""
    n, k, m = 14336, 5120, 128
    w = Weight(orc, 4, n, k, seed=9)
    a = randn_bf16(np.random.default_rng(8), (m, k))
    a_t = dev(a)
    ws, keep = workspace(512, n, k)
    out = torch.zeros(m * n, dtype=torch.int16, device="cuda")
    ep = gemm.GemmEpilogue(gemm.EPI_STORE_BF16, out.data_ptr(), n, 0, None, None, None, None, 0, 1e-6)
    print(f"larger workspace: m={m} n={n} k={k}", flush=True)
    gemm.qgemm(a_t.data_ptr(), m, w.desc, ep, ws, stream())
    rows = np.r_[0:2, m - 1:m]
    close(bf16_bits_to_f32(host(out, np.uint16).reshape(m, n)[rows]), orc.qgemm(a[rows], w.w_exact, 3), "bf16", a[rows],
          np.abs(w.w_exact))
