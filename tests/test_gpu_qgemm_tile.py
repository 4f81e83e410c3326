"""The 128- and 256-row tiles of q38a_qgemm (65 rows and more, below the large-M kernel) and the large-M
kernel's loop: every epilogue against the oracle's product over the weights the kernel multiplies by, at the
edges of the tiles (rows one past a tile, one group of K, an odd number of groups for tiles that take two
at a time, K slices of unequal length, every remainder of the loops that are unrolled by four), with
stores that cannot be 16 bytes wide, and without the split workspace where it is optional. Bounds as in
test_gpu_qgemm.py: one rounding step of the output plus the fp32 accumulation. The tile height and the
number of slices that a shape is there for are asserted with tile_plan."""
import numpy as np
import pytest
import torch

from q38a import gemm
from gpu_util import dev, host, stream
from test_gpu_qgemm import Weight, big_path, check_residual, close, row_scales, workspace
from util import assert_bits_equal, bf16_bits_to_f32, randn_bf16

pytestmark = pytest.mark.gpu



def tile_plan(m, n, k):
    """(rows per tile, K slices, steps of the shortest and of the longest slice): csrc/qgemm.hip plan_tile."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    G = k // 64
    best = None
    for rows, us, kp in ((128, 1.12, 2), (256, 0.9, 1)):
        tiles = -(-m // rows) * (n // 128)
        for s in range(1, min(8, G) + 1):
            cost = -(-tiles * s // cus) * (-(-(-(-G // s)) // kp) * us + 12.0 + (5.0 + 3.0 * s if s > 1 else 0.0))
            if best is None or cost < best[0]:
                best = cost, rows, s, -(-(G // s) // kp), -(-(-(-G // s)) // kp)
    return best[1:]


# (rows, columns, K): tile edges 128/256, one group, odd group counts
SHAPES = [(65, 256, 64), (66, 256, 192), (65, 512, 576), (128, 256, 1088), (129, 512, 640), (255, 256, 448),
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


@pytest.mark.parametrize("m,n,k,shift", [(65, 256, 64, 0), (129, 512, 640, 1), (300, 2560, 704, 0)])
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


BF16, F32, RES = gemm.EPI_STORE_BF16, gemm.EPI_STORE_F32, gemm.EPI_RESIDUAL


def check_rows(orc, bits, m, n, k, kind, seed):
    """One launch with the epilogue `kind`, checked on rows at the edges of 32-, 64-, 128- and 256-row blocks
    and on the last ones."""
    w = Weight(orc, bits, n, k, seed=seed)
    rng = np.random.default_rng(seed)
    a = randn_bf16(rng, (m, k))
    rows = np.array(sorted({r for r in (0, 31, 32, 63, 64, 127, 128, 191, 192, 255, 256, 257, m - 2, m - 1) if r < m}))
    wo = w.w_ref if big_path(m, n) else w.w_exact
    hidden = 128 * max(1, k // 128)
    partials = rng.uniform(50.0, 200.0, (m, hidden // 128)).astype(np.float32)
    a_t, p_t = dev(a), dev(partials)
    ws, keep = workspace(m, n, k)
    print(f"tile rows: bits={bits} m={m} n={n} k={k} kind={kind}", flush=True)
    if kind == RES:
        res0 = rng.standard_normal((m, n)).astype(np.float32)
        res, xbf = dev(res0), torch.zeros(m * n, dtype=torch.int16, device="cuda")
        pout = torch.zeros(m * (n // 128), dtype=torch.float32, device="cuda")
        ep = gemm.GemmEpilogue(RES, None, 0, 0, res.data_ptr(), xbf.data_ptr(), pout.data_ptr(), None, 0, 1e-6)
        gemm.qgemm(a_t.data_ptr(), m, w.desc, ep, ws, stream())
        check_residual(orc, w, a[rows], res0[rows], host(res).reshape(m, n)[rows],
                       host(xbf, np.uint16).reshape(m, n)[rows], host(pout).reshape(m, n // 128)[rows], m=m)
        return
    out = torch.zeros(m * n, dtype=torch.float32 if kind == F32 else torch.int16, device="cuda")
    ep = gemm.GemmEpilogue(kind, out.data_ptr(), n, 0, None, None, None, p_t.data_ptr(), hidden, 1e-6)
    gemm.qgemm(a_t.data_ptr(), m, w.desc, ep, ws, stream())
    got = host(out).reshape(m, n)[rows] if kind == F32 else bf16_bits_to_f32(host(out, np.uint16).reshape(m, n)[rows])
    want = orc.qgemm(a[rows], wo, 3, partials_in=partials[rows], hidden=hidden)
    close(got, want, "rows", a[rows], np.abs(wo), row_scales(partials[rows], hidden), out="f32" if kind == F32 else "bf16")


@pytest.mark.parametrize("bits,m,n,k,kind,rows,split,steps", [
    # 256-row tiles over the whole K: 1 and 5 to 8 steps
    (6, 65, 256, 64, RES, 256, False, (1, 1)), (4, 257, 11008, 320, RES, 256, False, (5, 5)),
    (5, 257, 11008, 384, BF16, 256, False, (6, 6)), (6, 300, 11008, 448, F32, 256, False, (7, 7)),
    (6, 511, 11008, 512, RES, 256, False, (8, 8)),
    # 256-row tiles, three slices: 17 to 20 steps
    (4, 385, 4352, 3392, F32, 256, True, (17, 18)), (5, 385, 4352, 3520, RES, 256, True, (18, 19)),
    (6, 400, 4352, 3712, RES, 256, True, (19, 20)), (6, 500, 4352, 3392, BF16, 256, True, (17, 18)),
    # 128-row tiles (two groups a step) over the whole K: 1 to 4 steps
    (5, 65, 256, 128, RES, 128, False, (1, 1)), (6, 127, 256, 192, BF16, 128, False, (2, 2)),
    (4, 129, 512, 320, F32, 128, False, (3, 3)), (6, 100, 256, 448, RES, 128, False, (4, 4)),
    # 128-row tiles, three slices: 7 to 10 steps
    (4, 65, 256, 2496, RES, 128, True, (7, 7)), (5, 128, 256, 2752, BF16, 128, True, (7, 8)),
    (6, 65, 256, 3136, F32, 128, True, (8, 9)), (5, 120, 256, 3648, RES, 128, True, (10, 10)),
])
def test_tile_paths(orc, bits, m, n, k, kind, rows, split, steps):
    assert not big_path(m, n)
    plan = tile_plan(m, n, k)
    assert plan[0] == rows and (plan[1] > 1) == split and plan[2:] == steps, plan
    check_rows(orc, bits, m, n, k, kind, seed=bits + m + k)


@pytest.mark.parametrize("bits,k,kind", [(4, 64, BF16), (5, 128, RES), (6, 192, F32), (5, 256, BF16), (5, 320, BF16),
                                         (4, 384, RES), (6, 448, RES), (6, 512, BF16)])
def test_large_m_group_counts(orc, bits, k, kind):
    """The 256 x 256 tiles at one to eight groups of K."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n = 8192
    m = 256 * -(-cus // (n // 256)) - 200
    assert big_path(m, n)
    check_rows(orc, bits, m, n, k, kind, seed=bits + k)
