"""The append at 8,192 rows and more (four rows per wave): bit for bit against the oracle with means of
squares on rounding boundaries (the left-to-right replay), and against the one-row-per-wave kernel
(taken for a proj without 16-byte alignment) for head counts and token counts that leave the last wave
of each kind of row partly filled, with positions past the RoPE table and past the page table."""
import numpy as np
import pytest
import torch

import q38a
from q38a import gemm
from gpu_util import HD, LD, NQ, Batch, Pool, append_params, dev, host, paged_layout, rope_dev, stream
from test_append_mean import boundary_row
from test_gpu_append import run_append
from test_gpu_qgemm import InProj, workspace
from util import assert_bits_equal, f32_to_bf16_bits, randn_bf16

pytestmark = pytest.mark.gpu


def test_boundary_means(orc):
    rng = np.random.default_rng(3)
    for M in (5, 257):  # one row per wave; four rows per wave
        proj = randn_bf16(rng, (M, LD))
        kcol = 2 * NQ * HD
        for m in range(0, M, 2):
            for h in (0, 3, 23):
                proj[m, h * HD:(h + 1) * HD] = f32_to_bf16_bits(boundary_row(rng).astype(np.float32))
            proj[m, kcol + HD:kcol + 2 * HD] = f32_to_bf16_bits(boundary_row(rng).astype(np.float32))
        q, q_ref, pool, pool_ref = run_append(orc, [(0, 60, M)], q38a.KV_INT8, rng, proj=proj)[:4]
        assert_bits_equal(q, q_ref, "q fp16")
        assert_bits_equal(pool, pool_ref, "pool bytes")


@pytest.mark.parametrize("nq,nkv,kv_dtype", [(24, 4, q38a.KV_INT8), (7, 1, q38a.KV_INT8_VT), (9, 3, q38a.KV_BF16),
                                             (5, 5, q38a.KV_INT8)])
def test_rows_kernel_matches_one_row_per_wave(nq, nkv, kv_dtype):
    rng = np.random.default_rng(nq)
    M = -(-8192 // (nq + 2 * nkv)) + 3
    M += 1 - M % 2
    ld = 2 * (nq + nkv) * HD
    n0 = M // 2
    seqs = [(0, 33, n0), (1, 0, 1), (2, 900, M - n0 - 1)]
    b = Batch(seqs)
    bt, pages = paged_layout(rng, [p + n for _, p, n in seqs])
    bt = bt[:, :-1] if bt.shape[1] > 15 else bt  # the last pages' tokens have no page: not stored
    fill = rng.integers(0, 256, q38a.page_bytes(kv_dtype, nkv) * pages, dtype=np.uint8)
    proj = dev(randn_bf16(rng, (M, ld)))
    odd = torch.zeros(M * ld + 4, dtype=torch.int16, device="cuda")
    odd[4:] = proj.view(-1)  # 8 bytes past a 16-byte boundary
    qn, kn = dev(rng.normal(1.0, 0.2, HD).astype(np.float32)), dev(rng.normal(1.0, 0.2, HD).astype(np.float32))
    rope = rope_dev(900 + M - n0 - 40)  # the last positions lie past the table: NaN q, nothing stored
    got = []
    for p in (proj, odd[4:]):
        pool = Pool(kv_dtype, pages, bt, nkv=nkv, fill=fill)
        q = torch.zeros(M * nq * HD, dtype=torch.int16, device="cuda")
        print(f"append rows: nq={nq} nkv={nkv} M={M} dtype={kv_dtype}", flush=True)
        q38a.qk_norm_rope_append(append_params(p, qn, kn, q, rope, nq=nq, nkv=nkv, ld=ld), b.desc, pool.desc, stream())
        torch.cuda.synchronize()
        got.append((host(q, np.uint16), pool.download()))
    assert_bits_equal(got[0][0], got[1][0], "q")
    assert_bits_equal(got[0][1], got[1][1], "pool bytes")
    assert (got[0][0].reshape(M, -1)[-30:] == 0x7E00).all()


@pytest.mark.parametrize("kv_dtype", [q38a.KV_INT8, q38a.KV_INT8_VT, q38a.KV_BF16])
def test_non_finite_rows_match_one_row_per_wave(kv_dtype):
    """NaNs and infinities in q, k and v: the same bytes from both kernels. A K row with a NaN or a V
    group of NaNs alone keeps NaN as its scale, so that attention over it shows it; a NaN among other
    values of a V group is quantised to 0."""
    rng = np.random.default_rng(5)
    M, nkv = 8192 // 32 + 5, 4
    b = Batch([(0, 7, M)])
    bt, pages = paged_layout(rng, [7 + M])
    x = randn_bf16(rng, (M, LD)).reshape(M, LD // HD, HD)
    nan, inf = np.uint16(0x7FC1), np.uint16(0x7F80)
    k, v = 2 * NQ, 2 * NQ + nkv
    x[3, 5, 17] = nan
    x[4, 6, 40:44] = inf
    x[9, k + 1, 200] = nan  # the whole normalised row is NaN
    x[10, k + 2, 5] = inf
    x[11, v, 64:128] = nan
    x[12, v + 1, 70] = nan
    x[13, v + 2, 130] = inf | np.uint16(0x8000)
    proj = dev(x.reshape(M, LD))
    odd = torch.zeros(M * LD + 4, dtype=torch.int16, device="cuda")
    odd[4:] = proj.view(-1)
    ones = dev(np.ones(HD, np.float32))
    rope = rope_dev(7 + M)
    got = []
    for p in (proj, odd[4:]):
        pool = Pool(kv_dtype, pages, bt)
        q = torch.zeros(M * NQ * HD, dtype=torch.int16, device="cuda")
        print(f"append non-finite: dtype={kv_dtype}", flush=True)
        q38a.qk_norm_rope_append(append_params(p, ones, ones, q, rope), b.desc, pool.desc, stream())
        torch.cuda.synchronize()
        got.append((host(q, np.uint16), pool.download()))
    assert_bits_equal(got[0][0], got[1][0], "q")
    assert_bits_equal(got[0][1], got[1][1], "pool bytes")
    if kv_dtype == q38a.KV_INT8:
        page = got[0][1].reshape(pages, -1)
        at = lambda m: (page[bt[0, (7 + m) // 64]], (7 + m) % 64)
        scales = lambda m, plane, h: at(m)[0][2 * nkv * 64 * HD:].view(np.uint16).reshape(2, nkv, 64, 4)[plane, h, at(m)[1]]
        assert (scales(9, 0, 1) == 0x7E00).all()
        s = scales(11, 1, 0)
        assert s[1] == 0x7E00 and (s[[0, 2, 3]] < 0x7C00).all()
        assert (scales(12, 1, 1) < 0x7C00).all()


@pytest.mark.parametrize("M", [5, 40, 257])
def test_in_projection_any_row_stride(orc, M):
    """The in-projection with its append, proj's rows of an odd stride and on a 2-byte boundary (the append
    reads them back): the gate columns, q and the pool as with aligned rows, bit for bit."""
    ip = InProj(orc, [(60, M)], seed=M)

    def run(ld, shift):
        pool = Pool(ip.kv_dtype, ip.pages, ip.bt, fill=ip.pool_host)
        proj = torch.zeros(M * ld + shift, dtype=torch.int16, device="cuda")[shift:]
        q = torch.zeros(M * NQ * HD, dtype=torch.int16, device="cuda")
        ws, keep = workspace(M, ip.n, ip.k)
        ep = gemm.GemmEpilogue(gemm.EPI_STORE_BF16, proj.data_ptr(), ld, 0, None, None, None, ip.p_t.data_ptr(), ip.k,
                               1e-6)
        print(f"in-projection: M={M} ld={ld} shift={shift}", flush=True)
        gemm.qgemm_qkv_append(ip.a_t.data_ptr(), M, ip.w.desc, ep, ws,
                              append_params(proj, ip.qn_t, ip.kn_t, q, ip.rope_t, ld=ld), ip.b.desc, pool.desc, stream())
        torch.cuda.synchronize()
        return host(proj, np.uint16).reshape(M, ld)[:, NQ * HD:2 * NQ * HD], host(q, np.uint16), pool.download()

    want = run(LD, 0)
    for ld, shift in ((LD + 1, 0), (LD + 2, 0), (LD, 3)):
        for got, ref, what in zip(run(ld, shift), want, ("gate", "q fp16", "pool bytes")):
            assert_bits_equal(got, ref, what)
