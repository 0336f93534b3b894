"""GPU parity of rowstats, normadd and argmax/argmaxM (p0pc0rn_amd/csrc/misc.hip) through the C ABI: every result is
compared with the oracle (oracle/q4oracle.c, itself pinned in tests/test_misc_oracle.py) on the same inputs. The
kernels sum in the reference's order with no FMA contraction, so rowstats and normadd are bit-exact, and the argmax
(max, index) pairs are exact, ties included."""
import numpy as np
import pytest

from oracle import oracle as O
from p0pc0rn_amd import capi

pytestmark = pytest.mark.gpu
NAN = 0x7FC00000


@pytest.mark.parametrize("rows,cols,mode", [(1, 2048, 1), (7, 700, 0), (300000, 8, 0), (3, 3, 1), (2, 8192, 0)])
def test_rowstats_bit_exact(dev, rows, cols, mode):
    ld, c0 = cols + 5, 3
    x = (2.0 + O.randn(rows * ld, 70 + rows % 97)).astype(np.float32)
    want = np.full((rows + 1) * 2, np.nan, np.float32)
    O.rowstats(capi.rowstats_args(x=x.ctypes.data, x_ld=ld, x_c0=c0, rows=rows, cols=cols, mode=mode, eps=1e-5,
                                  st=want.ctypes.data, st_off=1))
    xb = capi.to_device(x)
    st = capi.Buffer(want.nbytes).fill_u32(NAN)
    capi.rowstats(capi.rowstats_args(x=xb, x_ld=ld, x_c0=c0, rows=rows, cols=cols, mode=mode, eps=1e-5, st=st,
                                     st_off=1))
    got = st.read(np.float32)
    print(f"rowstats rows {rows} cols {cols} mode {mode}: mismatches {int(np.sum(got.view(np.uint32) != want.view(np.uint32)))}",
          flush=True)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    xb.free(); st.free()


@pytest.mark.parametrize("D,M,nsrc,mode", [(2048, 1, 4, 0), (2048, 5, 1, 0), (3072, 2, 2, 1), (100, 3, 3, 0)])
def test_normadd_bit_exact(dev, D, M, nsrc, mode):
    ldp = M * D + 64
    t = O.randn(nsrc * ldp, D + M, 0.3).astype(np.float32)
    w = (0.5 + O.rng_uniform(D, D)).astype(np.float32)
    x0 = O.randn(M * D, D + 1).astype(np.float32)
    xw, sw = x0.copy(), np.full(M + 2, np.nan, np.float32)
    kw = dict(t_n=nsrc, t_ld=ldp, w_off=0, st_off=2, D=D, M=M, eps=1e-6, scale=0.9, mode=mode)
    O.normadd(capi.normadd_args(t=t.ctypes.data, w=w.ctypes.data, x=xw.ctypes.data, st=sw.ctypes.data, **kw))
    tb, wb, xb = capi.to_device(t), capi.to_device(w), capi.to_device(x0)
    sb = capi.Buffer(sw.nbytes).fill_u32(NAN)
    capi.normadd(capi.normadd_args(t=tb, w=wb, x=xb, st=sb, **kw))
    gx, gs = xb.read(np.float32), sb.read(np.float32)
    assert np.array_equal(gx.view(np.uint32), xw.view(np.uint32))
    assert np.array_equal(gs.view(np.uint32), sw.view(np.uint32))
    for b in (tb, wb, xb, sb):
        b.free()


@pytest.mark.parametrize("n,M", [(4096, 1), (4096, 5), (1, 1), (257, 3), (0, 1)])
def test_argmax_exact(dev, n, M):
    rng = np.random.default_rng(n + M)
    mx = np.zeros(2 * max(n, 1) * M, np.float32)
    vals = rng.integers(-50, 50, n * M).astype(np.float32)   # ties everywhere
    mx[0:2 * n * M:2] = vals
    mx[1:2 * n * M:2] = rng.integers(0, 1 << 24, n * M).astype(np.uint32).view(np.float32)
    want = O.argmaxM(mx, n, M)
    mb = capi.to_device(mx)
    out = capi.Buffer(8 * M).fill_u32(0)
    if M == 1:
        capi.argmax(mb, n, out)
    else:
        capi.argmaxM(mb, n, M, out)
    got = out.read(np.uint32)
    assert np.array_equal(got, want)
    mb.free(); out.free()


def test_argmax_of_a_softcap_gemv(dev):
    """the pipeline the reference runs at the end of a decode step: head GEMV (rms + softcap, per-tile max/argmax),
    then argmax over the tiles = the argmax of the softcapped logits (ties to the lower row)"""
    N, K = 8192, 512
    w, _ = O.pack_q4(O.randn(N * K, 81, 0.05), N, K)
    x = O.randn(K, 82)
    nw = np.ones(K, np.float32)
    NT = N // 64
    mx = np.zeros(2 * NT + 4, np.float32)
    mx[2 * NT + 1] = 1.0   # rstd slot
    wb, xb, nb, mb = (capi.to_device(a) for a in (w, x, nw, mx))
    y = capi.Buffer(N * 4)
    capi.q4_gemv(capi.gemv_args(w=wb, w_rows=N, w_cols=K, x=xb, N=N, K=K, pro=capi.PRO["rms"], epi=capi.EPI["softcap"],
                                y=y, stat=mb, stat_off=2 * NT + 1, norm=nb, mx=mb, cap=30.0))
    out = capi.Buffer(8).fill_u32(0)
    capi.argmax(mb, NT, out)
    logits = y.read(np.float32)
    got = out.read(np.uint32)
    assert got[0] == int(np.argmax(logits)) and got[1] == logits.max().view(np.uint32)
    for b in (wb, xb, nb, mb, y, out):
        b.free()


@pytest.mark.parametrize("n,M", [(1024, 1), (1025, 1), (1025, 171), (1026, 171), (1023, 700), (255, 1030), (9000, 2)])
def test_argmax_exact_wave_counts(dev, n, M):
    """both workgroup sizes: on both sides of 1024 pairs and of 6 pairs per row"""
    test_argmax_exact(dev, n, M)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("rows,cols", [(1, 4), (5, 252), (1027, 256), (3, 2048), (2, 2052), (5, 4096), (2, 4100), (1, 9000)])
def test_rowstats_aligned_rows_bit_exact(dev, rows, cols, mode):
    """16-byte aligned rows: a row held in registers (up to 2048 and 4096 columns), a longer one read twice, and the
    four-rows-a-workgroup launch with a ragged last workgroup. The same order of sums as the oracle: equal bits"""
    x = (2.0 + O.randn(rows * cols, 31 + cols)).astype(np.float32)
    want = np.full(rows * 2, np.nan, np.float32)
    O.rowstats(capi.rowstats_args(x=x.ctypes.data, rows=rows, cols=cols, mode=mode, eps=1e-5, st=want.ctypes.data))
    xb = capi.to_device(x)
    st = capi.Buffer(want.nbytes + 8).fill_u32(NAN)
    capi.rowstats(capi.rowstats_args(x=xb, rows=rows, cols=cols, mode=mode, eps=1e-5, st=st))
    got = st.read(np.float32).view(np.uint32)
    assert np.array_equal(got[:2 * rows], want.view(np.uint32))
    assert (got[2 * rows:2 * rows + 2] == NAN).all()
    xb.free(); st.free()


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("D,M,nsrc", [(4, 1, 1), (1000, 3, 5), (2048, 2, 8), (2052, 2, 4), (6148, 1, 3), (100, 256, 3),
                                      (100, 257, 3)])
def test_normadd_aligned_rows_bit_exact(dev, D, M, nsrc, mode):
    """16-byte aligned rows, few (up to 256: a workgroup a row) and many, in registers (up to 2048 values) and in two passes,
    partials in fours with a remainder"""
    t = O.randn(nsrc * M * D, D + nsrc, 0.3).astype(np.float32)
    w = (0.5 + O.rng_uniform(D, D)).astype(np.float32)
    x0 = O.randn(M * D, D + 1).astype(np.float32)
    xw, sw = x0.copy(), np.full(M, np.nan, np.float32)
    kw = dict(t_n=nsrc, D=D, M=M, eps=1e-6, scale=0.9, mode=mode)
    O.normadd(capi.normadd_args(t=t.ctypes.data, w=w.ctypes.data, x=xw.ctypes.data, st=sw.ctypes.data, **kw))
    tb, wb, xb = capi.to_device(t), capi.to_device(w), capi.Buffer(x0.nbytes + 16).fill_u32(NAN)
    xb.upload(x0)
    sb = capi.Buffer(sw.nbytes).fill_u32(NAN)
    capi.normadd(capi.normadd_args(t=tb, w=wb, x=xb, st=sb, **kw))
    gx, gs = xb.read(np.float32).view(np.uint32), sb.read(np.float32, M).view(np.uint32)
    assert np.array_equal(gx[:M * D], xw.view(np.uint32))
    assert (gx[M * D:M * D + 4] == NAN).all()
    assert np.array_equal(gs, sw.view(np.uint32))
    for b in (tb, wb, xb, sb):
        b.free()


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("D,M,nsrc,ldp_pad,w_off,shift", [
    (1, 3, 1, 1, 0, 0), (3, 2, 4, 5, 1, 1), (255, 300, 2, 1, 1, 0), (1027, 2, 3, 7, 0, 1), (2050, 1, 5, 0, 1, 0),
    (2048, 5, 4, 0, 0, 1), (2048, 2, 1, 0, 1, 0), (8193, 1, 2, 3, 3, 1), (38400, 1, 1, 1, 0, 0),
    (764, 257, 1, 0, 0, 0), (768, 257, 3, 0, 0, 0), (2048, 257, 2, 0, 0, 0), (3068, 2, 1, 0, 0, 0), (3072, 2, 5, 0, 0, 0),
])
def test_normadd_any_rows_bit_exact(dev, D, M, nsrc, ldp_pad, w_off, shift, mode):
    """rows, strides and buffers at any alignment, and both sides of the sizes where aligned rows take a wave or a workgroup
    each; nothing past x written"""
    ldp = M * D + ldp_pad
    t = O.randn(nsrc * ldp + 1, D + nsrc, 0.3).astype(np.float32)
    w = (0.5 + O.rng_uniform(D, D + w_off)).astype(np.float32)
    x0 = O.randn(M * D, D + 1).astype(np.float32)
    xw, sw = x0.copy(), np.full(M, np.nan, np.float32)
    kw = dict(t_n=nsrc, t_ld=ldp, w_off=w_off, D=D, M=M, eps=1e-6, scale=0.9, mode=mode)
    O.normadd(capi.normadd_args(t=t.ctypes.data, w=w.ctypes.data, x=xw.ctypes.data, st=sw.ctypes.data, **kw))
    tb, wb, xb = capi.to_device(t), capi.to_device(w), capi.Buffer(x0.nbytes + 32).fill_u32(NAN)
    xb.upload(x0, 4 * shift)
    sb = capi.Buffer(sw.nbytes).fill_u32(NAN)
    capi.normadd(capi.normadd_args(t=tb, w=wb, x=xb.ptr + 4 * shift, st=sb, **kw))
    gx, gs = xb.read(np.float32).view(np.uint32), sb.read(np.float32, M).view(np.uint32)
    assert np.array_equal(gx[shift:M * D + shift], xw.view(np.uint32))
    assert (gx[:shift] == NAN).all() and (gx[M * D + shift:M * D + 8] == NAN).all()
    assert np.array_equal(gs, sw.view(np.uint32))
    for b in (tb, wb, xb, sb):
        b.free()


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("rows,cols", [(1, 4095), (2, 4097), (256, 4096), (257, 511), (257, 513), (1030, 515)])
def test_rowstats_unaligned_rows_bit_exact(dev, rows, cols, mode):
    """rows that are not 16-byte aligned, on both sides of the sizes where a row takes a wave or a workgroup"""
    test_rowstats_bit_exact(dev, rows, cols, mode)
