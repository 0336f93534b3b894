"""GPU parity of the q4 dequant-GEMM (p0_q4_gemm) against the CPU oracle, through the C ABI.

Tolerance: relative L2 <= 1e-3 against the oracle's float64 sum over the same fp16 operands,
plus this build's bar of 1e-5 for fp32 outputs (MFMA accumulates in fp32; the operands are bit-identical fp16) and
2e-3 where the output itself is fp16 (half an fp16 ulp is 2^-11 relative).
"""
import numpy as np
import pytest

from oracle import oracle as O
from p0pc0rn_amd import capi
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-3
NAN32, NAN16x2 = 0x7FC00000, 0x7E007E00


def _weights(rows, K, seed):
    return O.pack_q4(O.randn(rows * K, seed, 0.05), rows, K)[0]


def run(fields, arrays, out_dtype, out_len, init=None):
    """run the same call on the oracle (host pointers) and on the GPU (device copies); returns (oracle, gpu)"""
    y_host = np.full(out_len, np.nan, out_dtype) if init is None else init.astype(out_dtype).copy()
    host = {k: v.ctypes.data for k, v in arrays.items()}
    O.q4_gemm(capi.gemm_args(**fields, **host, y=y_host.ctypes.data))
    dev = {k: capi.to_device(v) for k, v in arrays.items()}
    if init is None:
        yb = capi.Buffer(max(y_host.nbytes, 16)).fill_u32(NAN32 if out_dtype == np.float32 else NAN16x2)
    else:
        yb = capi.to_device(init.astype(out_dtype))
    flops = capi.q4_gemm(capi.gemm_args(**fields, **dev, y=yb))
    assert flops == 2.0 * fields["M"] * fields["N"] * fields["K"]
    got = yb.read(out_dtype, out_len)
    for b in list(dev.values()) + [yb]:
        b.free()
    return y_host, got


def check(got, want, what, tol_build):
    got = np.asarray(got, np.float64)
    want = np.asarray(want, np.float64)
    r = rel_l2(got, want)
    print(f"{what}: rel_l2 {r:.3e}", flush=True)
    assert np.all(np.isfinite(got)), what + ": unwritten outputs"
    assert r <= TOL and r <= tol_build, what


@pytest.mark.parametrize("M,N,K", [(40, 128, 256), (128, 256, 512), (300, 200, 96), (1, 64, 32), (257, 384, 1024)])
def test_gemm_f16_f32(dev, M, N, K):
    Nw = -(-N // 64) * 64                      # records hold 64 rows; a ragged N reads the first N of them
    w = _weights(Nw, K, 11)
    x = O.randn(M * K, 7).astype(np.float16)
    f = dict(w_rows=Nw, w_cols=K, M=M, N=N, K=K, x_mode=capi.XMODE["f16"], epi=capi.GEPI["f32"])
    want, got = run(f, dict(w=w, x=x), np.float32, M * N)
    check(got, want, f"gemm f16->f32 {M}x{N}x{K}", 1e-5)


def test_gemm_f16_out(dev):
    M, N, K = 96, 256, 256
    w = _weights(N, K, 12)
    x = O.randn(M * K, 8).astype(np.float16)
    f = dict(w_rows=N, w_cols=K, M=M, N=N, K=K, x_mode=capi.XMODE["f16"], epi=capi.GEPI["f16"])
    want, got = run(f, dict(w=w, x=x), np.float16, M * N)
    check(got, want, "gemm f16->f16", 2e-3)


@pytest.mark.parametrize("M,N,y_ld,y_n0", [(96, 251, 260, 4), (70, 131, 131, 0), (33, 128, 139, 3), (33, 128, 128, 1)])
def test_gemm_f16_out_layouts(dev, M, N, y_ld, y_n0):
    """fp16 outputs are stored two columns per 4-byte store when Y's rows allow it (even row stride, even first
    column) and one by one otherwise; ragged N (an odd last column) and offset rows, with every element outside the
    written block left untouched"""
    K = 256
    Nw = -(-N // 64) * 64
    w = _weights(Nw, K, 31)
    x = O.randn(M * K, 32).astype(np.float16)
    f = dict(w_rows=Nw, w_cols=K, M=M, N=N, K=K, x_mode=capi.XMODE["f16"], epi=capi.GEPI["f16"], y_ld=y_ld, y_n0=y_n0)
    n_out = (M * y_ld + y_n0 + 9) // 2 * 2   # whole 4-byte words: the device buffer is NaN-filled by words
    want, got = run(f, dict(w=w, x=x), np.float16, n_out)
    idx = np.concatenate([y_n0 + m * y_ld + np.arange(N) for m in range(M)])
    check(got[idx], want[idx], f"gemm f16 out M={M} N={N} ld={y_ld} n0={y_n0}", 2e-3)
    untouched = np.setdiff1d(np.arange(n_out), idx)
    assert np.all(np.isnan(got[untouched].astype(np.float32)))


def test_gemm_bf16_activations(dev):
    M, N, K = 64, 128, 512
    w = _weights(N, K, 14)
    xf = O.randn(M * K, 9)
    xb = (xf.view(np.uint32) >> 16).astype(np.uint16)          # bf16 by truncation: exact bf16 values
    f = dict(w_rows=N, w_cols=K, M=M, N=N, K=K, x_mode=capi.XMODE["bf16"], epi=capi.GEPI["f32"])
    want, got = run(f, dict(w=w, x=xb), np.float32, M * N)
    check(got, want, "gemm bf16->f32", 1e-5)


@pytest.mark.parametrize("mode", ["lnmod", "rms"])
def test_gemm_fused_norm_prologues(dev, mode):
    """engine/ops/gemm.js:59-63: X f32, (mean, rstd) per row, scale / shift vectors (shift base = off + stride, u32)"""
    M, N, K = 72, 192, 256
    w = _weights(N, K, 15)
    x = O.randn(M * K, 10, 2.0)
    st = np.zeros(2 * (M + 3), np.float32)
    xr = x.reshape(M, K).astype(np.float64)
    st[6::2] = xr.mean(1)
    st[7::2] = 1 / np.sqrt(xr.var(1) + 1e-6)
    pv = O.randn(4 * K, 16, 0.1)
    f = dict(w_rows=N, w_cols=K, M=M, N=N, K=K, x_mode=capi.XMODE[mode], epi=capi.GEPI["f32"], stats_off=3,
             pv_off=2 * K, pv_stride=(1 << 32) - 2 * K)           # shift at off - 2K, the reference's neg(stride) wrap
    want, got = run(f, dict(w=w, x=x, stats=st, pv=pv), np.float32, M * N)
    check(got, want, f"gemm {mode}", 1e-5)


@pytest.mark.parametrize("act", ["silu", "gelu"])
def test_gemm_swiglu_with_bias(dev, act):
    M, MLP, K = 80, 192, 256
    w = _weights(2 * MLP, K, 17)                                 # rows [gate | up]
    x = O.randn(M * K, 18).astype(np.float16)
    bv = O.randn(2 * MLP + 8, 19, 0.1)
    f = dict(w_rows=2 * MLP, w_cols=K, M=M, N=2 * MLP, K=K, x_mode=0, epi=capi.GEPI["swiglu"], wr0=0, wr1=MLP,
             y_ld=MLP, bv_off=4, bv_up=MLP, act=capi.ACT[act])
    want, got = run(f, dict(w=w, x=x, bv=bv), np.float16, M * MLP)
    check(got, want, f"gemm swiglu {act}", 2e-3)


@pytest.mark.parametrize("store", [0, 1])
def test_gemm_resadd_gate_bias(dev, store):
    M, N, K = 64, 256, 512
    w = _weights(N, K, 20)
    x = O.randn(M * K, 21).astype(np.float16)
    gate = O.randn(N, 22)
    bv = O.randn(N, 23, 0.1)
    resid = O.randn(M * N, 24)
    f = dict(w_rows=N, w_cols=K, M=M, N=N, K=K, x_mode=0, epi=capi.GEPI["resadd"], store=store)
    want, got = run(f, dict(w=w, x=x, ev=gate, bv=bv), np.float32, M * N, init=resid)
    check(got, want, f"gemm resadd store={store}", 1e-5)


@pytest.mark.parametrize("epi,N,y_ld,y_n0", [("f32", 131, 140, 2), ("f32", 128, 133, 1), ("resadd", 131, 140, 2),
                                            ("resadd", 128, 133, 3), ("bias", 131, 140, 2), ("bias", 128, 129, 1)])
def test_gemm_output_layouts(dev, epi, N, y_ld, y_n0):
    """the f32, resadd (accumulating) and bias (with residual) epilogues read and write two adjacent columns per
    access when Y's rows allow it and element by element otherwise; ragged N, offset rows, elements outside the block
    keep their values"""
    M, K = 45, 256
    Nw = -(-N // 64) * 64
    w = _weights(Nw, K, 41)
    x = O.randn(M * K, 42).astype(np.float16)
    ev = O.randn(N, 43)
    bv = O.randn(N, 44, 0.1)
    n_out = (M * y_ld + y_n0 + 9) // 2 * 2
    f = dict(w_rows=Nw, w_cols=K, M=M, N=N, K=K, x_mode=0, epi=capi.GEPI[epi], y_ld=y_ld, y_n0=y_n0)
    arrays = dict(w=w, x=x, ev=ev)
    if epi == "resadd":
        f.update(store=0)
        arrays.update(bv=bv)
    if epi == "bias":
        f.update(res=1)
    dt = np.float16 if epi == "bias" else np.float32
    init = O.randn(n_out, 45)
    want, got = run(f, arrays, dt, n_out, init=init)
    idx = np.concatenate([y_n0 + m * y_ld + np.arange(N) for m in range(M)])
    check(got[idx], want[idx], f"gemm {epi} out N={N} ld={y_ld} n0={y_n0}", 2e-3 if dt == np.float16 else 1e-5)
    untouched = np.setdiff1d(np.arange(n_out), idx)
    assert np.array_equal(got[untouched], init.astype(dt)[untouched])


def test_gemm_bias_residual_in_place(dev):
    M, N, K = 48, 128, 128
    w = _weights(N, K, 25)
    x = O.randn(M * K, 26).astype(np.float16)
    b = O.randn(N, 27, 0.1)
    prev = O.randn(M * N, 28).astype(np.float16)
    f = dict(w_rows=N, w_cols=K, M=M, N=N, K=K, x_mode=0, epi=capi.GEPI["bias"], res=1)
    want, got = run(f, dict(w=w, x=x, ev=b), np.float16, M * N, init=prev)
    check(got, want, "gemm bias res", 2e-3)


def test_gemm_offsets(dev):
    """a sub-block of a larger weight (wr0 rows, wk0 columns), x with a k offset and row stride, y with n0 and ld"""
    M, N, K, Nw, Kw = 50, 128, 128, 320, 256
    w = _weights(Nw, Kw, 29)
    ldx = 400
    x = O.randn(M * ldx + 64, 30).astype(np.float16)
    f = dict(w_rows=Nw, w_cols=Kw, M=M, N=N, K=K, wr0=64, wk0=128, x_mode=0, x_off=16, x_ld=ldx, x_k0=40,
             epi=capi.GEPI["f32"], y_off=32, y_ld=N + 40, y_n0=8)
    n_out = 8 + M * (N + 40) + 32
    want, got = run(f, dict(w=w, x=x), np.float32, n_out)
    idx = np.concatenate([8 + 8 + m * (N + 40) + np.arange(N) for m in range(M)])
    check(got[idx], want[idx], "gemm offsets", 1e-5)
    untouched = np.setdiff1d(np.arange(n_out), idx)
    assert np.all(np.isnan(got[untouched]))


def test_gemm_flux_shape_sampled_rows(dev):
    """FLUX.2-klein QKV at full size (M=4608, N=9216, K=3072): every row computed on the GPU, a sample checked"""
    M, N, K = 4608, 9216, 3072
    w = O.fill_q4_sym(N, K, 7, 0.02)
    x32, x16 = O.fill_randn(M * K, 8)
    wb, xb = capi.to_device(w), capi.to_device(x16)
    yb = capi.Buffer(M * N * 4).fill_u32(NAN32)
    capi.q4_gemm(capi.gemm_args(w=wb, w_rows=N, w_cols=K, x=xb, M=M, N=N, K=K, x_mode=0, epi=capi.GEPI["f32"], y=yb))
    rows = np.array([0, 1, 127, 128, 2047, 4095, 4096, 4607])
    y = yb.read(np.float32).reshape(M, N)
    assert np.all(np.isfinite(y))
    sub = np.ascontiguousarray(x16.reshape(M, K)[rows])
    ys = np.zeros(len(rows) * N, np.float32)
    O.q4_gemm(capi.gemm_args(w=w.ctypes.data, w_rows=N, w_cols=K, x=sub.ctypes.data, M=len(rows), N=N, K=K, x_mode=0,
                             epi=capi.GEPI["f32"], y=ys.ctypes.data))
    check(y[rows].ravel(), ys, "FLUX QKV sampled rows", 1e-5)
    for b in (wb, xb, yb):
        b.free()


@pytest.mark.parametrize("mode", ["f16", "bf16", "lnmod", "rms"])
@pytest.mark.parametrize("M,K,pad", [(3, 544, 0), (9001, 32, 0), (33005, 32, 0), (2051, 2592, 1), (131077, 32, 0),
                                     (700, 96, 1), (8200, 544, 0), (2100, 512, 1)])
def test_gemm_staging_rows_per_wave(dev, mode, M, K, pad):
    """the activation staging where a wave walks 1, 4 and 8 steps, a step 1 to 16 rows side by side (as many lanes a row as K
    fills), with a ragged last step and row group, 16-byte aligned rows and rows that are not (a leading element). One fp32
    rounding may differ from the oracle's before the value is rounded to fp16, which flips about 2^-12 of the fp16
    roundings by 2^-11: 1.3e-5 relative; the bar is four times that"""
    N, ld, c0 = 64, K + 8 * pad, pad if mode != "f16" else 1
    ld += 1 if mode == "f16" else 0
    w = _weights(N, K, 21)
    xf = O.randn(M * ld, 10, 1.5)
    x = (xf if mode in ("lnmod", "rms") else xf.astype(np.float16) if mode == "f16"
         else (xf.view(np.uint32) >> 16).astype(np.uint16))
    st = np.empty(2 * M, np.float32)
    xr = xf.reshape(M, ld).astype(np.float64)
    st[0::2] = xr.mean(1)
    st[1::2] = 1 / np.sqrt(xr.var(1) + 1e-6)
    pv = O.randn(2 * (K + 8), 16, 0.1)
    f = dict(w_rows=N, w_cols=K, M=M, N=N, K=K, x_ld=ld, x_k0=c0, x_mode=capi.XMODE[mode], epi=capi.GEPI["f32"],
             pv_off=K + 8, pv_stride=(1 << 32) - (K + 8))
    f["x_ld"] = ld + (0 if c0 + K <= ld else 8)
    if f["x_ld"] != ld:
        x = np.concatenate([x.reshape(M, ld), np.zeros((M, 8), x.dtype)], 1).ravel()
    arrays = dict(w=w, x=x)
    if mode in ("lnmod", "rms"):
        arrays.update(stats=st, pv=pv)
    want, got = run(f, arrays, np.float32, M * N)
    check(got, want, f"gemm staging {mode} {M}x{K}", 5e-5)


_SMALL = [  # (M, N, K, first weight row, its columns before K, epilogue): edges of 128 x 128 tiles, 64-k steps, K slices
    (1, 64, 32, 0, 0, "f32"), (127, 128, 96, 64, 32, "f16"), (129, 200, 1056, 0, 64, "f32"), (130, 131, 4128, 128, 0, "bias"),
    (257, 448, 2048, 0, 0, "resadd"), (64, 384, 544, 0, 32, "swiglu"), (200, 130, 2080, 64, 0, "swiglu"),
    (77, 384, 1088, 0, 0, "heads-inter"), (140, 640, 96, 0, 0, "heads-half"), (300, 128, 8192, 0, 0, "resadd"),
]


@pytest.mark.parametrize("M,N,K,wr0,wk0,epi", _SMALL)
def test_gemm_small_tiles_against_large(dev, M, N, K, wr0, wk0, epi):
    """calls of one or a few tiles run in 128 x 128 tiles with K cut into slices (gemm_n128.hip); the same call on a weight
    at a 4-byte offset runs in 256 x 256 tiles (gemm.hip). Both sum the same fp16 operands in fp32: each is within the
    oracle's bar, and they differ by the order of the sums only (2e-6 relative in fp32 over K <= 8192: sqrt(K) roundings
    of 2^-24; one fp16 ulp where the output is fp16)"""
    sw, heads = epi == "swiglu", epi.startswith("heads")
    rows = -(-(wr0 + (N if not sw else N // 2)) // 64) * 64
    wr1 = rows if sw else 0
    rows *= 2 if sw else 1
    Kw = wk0 + K + 32
    w = O.pack_q4(np.clip(O.randn(rows * Kw, M + N, 0.05), -0.3, 0.3), rows, Kw)[0]
    x = O.randn(M * (K + 8), 7).astype(np.float16)
    f32 = epi in ("f32", "resadd")
    dt, ncol = (np.float32 if f32 else np.float16), (N // 2 if sw else N)
    f = dict(w_rows=rows, w_cols=Kw, M=M, N=N, K=K, x_ld=K + 8, wr0=wr0, wr1=wr1, wk0=wk0, x_mode=0,
             epi=capi.GEPI["heads" if heads else epi], y_ld=ncol + 3, y_n0=1)
    arrays, n_out = dict(x=x), M * (ncol + 3) + 16
    if epi in ("bias", "resadd"):
        arrays.update(ev=O.randn(N, 43), bv=O.randn(N, 44, 0.1)) if epi == "resadd" else arrays.update(ev=O.randn(N, 43))
        f.update(res=1) if epi == "bias" else None
    if sw:
        arrays.update(bv=O.randn(2 * N, 45, 0.1))
        f.update(bv_up=N, act=capi.ACT["silu"])
    if heads:
        H, Ltot = N // 128, M + 5
        rope = np.stack([np.cos(np.arange(Ltot * 64) * 0.01), np.sin(np.arange(Ltot * 64) * 0.01)], -1).astype(np.float32)
        arrays.update(ev=(1 + O.randn(256, 46, 0.1)).astype(np.float32), rope=rope)
        f.update(heads_ltot=Ltot, heads_row_off=3, heads_hq=H // 2, heads_hkv=1, heads_rope=capi.ROPE[epi[6:]])
        n_out = H * Ltot * 128 + 16
    init = O.randn(n_out, 47)
    shifted = np.concatenate([np.zeros(4, np.uint8), np.asarray(w).view(np.uint8).ravel()])
    want, small = run(f, dict(arrays, w=w), dt, n_out, init=init)
    _, large = run(dict(f, w_off=4), dict(arrays, w=shifted), dt, n_out, init=init)
    check(small, want, f"gemm small tiles {epi} {M}x{N}x{K}", 1e-5 if f32 else 2e-3)
    check(small, large, f"gemm small against large tiles {epi}", 2e-6 if f32 else 1e-3)
    untouched = want == init.astype(dt)
    assert np.array_equal(small[untouched], want[untouched])


@pytest.mark.parametrize("M,mode", [(40, "f16"), (300, "f16"), (40, "bf16")])
def test_gemm_rows_going_down_in_memory(dev, M, mode):
    """a negative x_ld walks the rows of X from the last in memory to the first: 64-bit offsets, so gemm.hip's (the 32-bit
    buffer offsets of gemm_n128.hip reach upwards only), or the staging's, whose X' rows go up again"""
    N, K, ld = 128, 288, 296
    w = _weights(N, K, 31)
    xf = O.randn(M * ld, 32)
    x = xf.astype(np.float16) if mode == "f16" else (xf.view(np.uint32) >> 16).astype(np.uint16)
    f = dict(w_rows=N, w_cols=K, M=M, N=N, K=K, x_mode=capi.XMODE[mode], epi=capi.GEPI["f32"])
    want, got = run(dict(f, x_ld=-ld, x_off=(M - 1) * ld * 2), dict(w=w, x=x), np.float32, M * N)
    check(got, want, f"gemm {mode} rows down {M}x{N}x{K}", 1e-5)
    up, _ = run(dict(f, x_ld=ld), dict(w=w, x=np.ascontiguousarray(x.reshape(M, ld)[::-1])), np.float32, M * N)
    assert np.array_equal(up.view(np.uint32), want.view(np.uint32))


def _hard_records(N, K, seed):
    """q4 records a third of whose (row, group) pairs have q s + m inexact in fp32: a scale far above its minimum (odd
    mantissas, so that 3 s, 6 s and 12 s lie half way between fp16 values and the minimum decides), a minimum far above its
    scale, subnormals of either"""
    rng = np.random.default_rng(seed)
    w = O.pack_q4(O.randn(N * K, seed, 0.05), N, K)[0].copy().view(np.uint32).reshape(N // 64, K // 32, 320)
    w[..., :256] = rng.integers(0, 1 << 32, w[..., :256].shape, dtype=np.uint32)
    sm = w[..., 256:].copy().view(np.float16).reshape(N // 64, K // 32, 64, 2)
    kind = rng.integers(0, 9, sm.shape[:3])
    odd = (rng.integers(512, 682, sm.shape[:3]) * 2 + 1) / 1024.0
    e = rng.integers(2, 9, sm.shape[:3]).astype(np.float64)
    sign = rng.choice([-1.0, 1.0], sm.shape[:3])
    s = np.select([kind == 0, kind == 1, kind == 2], [odd * 2.0 ** e, odd * 2.0 ** (e - 14), odd * 2.0 ** -16], sm[..., 0])
    m = np.select([kind == 0, kind == 1, kind == 2], [sign * odd * 2.0 ** (e - 25), sign * odd * 2.0 ** e, sign * odd], sm[..., 1])
    sm[..., 0], sm[..., 1] = s.astype(np.float16), m.astype(np.float16)
    w[..., 256:] = sm.reshape(N // 64, K // 32, 128).view(np.uint32)
    return w.reshape(-1).view(np.uint8), sm


def test_gemm_weights_that_round_twice(dev):
    """each weight is fl16(fl32(q s + m)), bit for bit, also where the one rounding of the packed fp16 path would differ: rows
    of X that pick one k each give the weights themselves, in 128 x 128 tiles with K slices and a last step of one group, and
    in 256 x 256 tiles (the weight at a 4-byte offset)"""
    M, N, K = 200, 192, 2080
    w, sm = _hard_records(N, K, 5)
    w16 = np.asarray(O.dequant_q4(w, N, K)[1]).view(np.float16)
    q = w.view(np.uint32).reshape(N // 64, K // 32, 320)[..., :256].reshape(N // 64, K // 32, 64, 4)
    q = ((q[..., None] >> (4 * np.arange(8, dtype=np.uint32))) & 15).reshape(N // 64, K // 32, 64, 32)
    one = (q * sm[..., :1].astype(np.float64) + sm[..., 1:].astype(np.float64)).astype(np.float16)   # exact, rounded once
    one = one.transpose(0, 2, 1, 3).reshape(N, K)
    differ = (one.view(np.uint16) != w16.view(np.uint16)).sum(0)
    ks = np.concatenate([np.argsort(-differ)[:M - 40], np.arange(K - 40, K)])   # the columns with most of them, and the tail
    print("weights that round twice among those compared:", int(differ[ks].sum()), flush=True)
    assert differ[ks].sum() > 500
    x = np.zeros((M, K), np.float16)
    x[np.arange(M), ks] = 1
    f = dict(w_rows=N, w_cols=K, M=M, N=N, K=K, x_mode=capi.XMODE["f16"], epi=capi.GEPI["f32"])
    want = np.ascontiguousarray(w16[:, ks].T.astype(np.float32))
    for off in (0, 4):
        wb = capi.to_device(np.concatenate([np.zeros(off, np.uint8), w]))
        xb, yb, hb = capi.to_device(x), capi.Buffer(want.nbytes).fill_u32(NAN32), capi.Buffer(2 * N * K)
        capi.q4_dequant(wb, N, K, out16=hb, w_off=off)
        assert np.array_equal(hb.read(np.uint16), w16.view(np.uint16).ravel())
        capi.q4_gemm(capi.gemm_args(**f, w=wb, w_off=off, x=xb, y=yb))
        got = yb.read(np.float32).reshape(M, N)
        assert np.array_equal(got, want), f"weight offset {off}: {int((got != want).sum())} differ"
        for b in (wb, xb, yb, hb):
            b.free()
