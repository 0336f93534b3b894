"""The workloads whose speed this repository stands for, through its C ABI as p0pc0rn_amd.capi binds it.

A decode token is one GEMV per projection, recorded or chained; a verify pass the same with 2-16 rows; prefill chunks
and the DiT blocks are dequant-GEMMs with their fused prologues and epilogues; a weight is now and then dequantised as a
whole. Shapes are the Gemma-4-E2B, FLUX.2-klein and SANA-Video shaped ones that bench.py and the tests use.

listed() names the cases, draw() gives more of the same ranges, prepare() makes what a program holds before the call
(its inputs, weights, recordings and chains), run() is one pass, exact() the same outputs in float64 with plain torch.
"""
import math

import torch

from p0pc0rn_amd import capi

D, QKV, MLP, VOCAB = 2048, 3072, 8192, 262144   # the E2B-shaped decoder layer and head
Q4_REC, Q8_REC = 1280, 4224                     # bytes of one weight record: 64 rows x 32 k, 64 rows x 64 k
EPS = 1e-6


def listed():
    return [
        # the smallest call of a decode token, run eagerly: the 8-bit per-layer gate of the E2B balanced pack
        dict(name="gemv_q8_gate", kind="gemv", enc="q8", M=1, N=256, K=1536, kPer=0, pro="raw", epi="store", calls=1,
             mode="eager"),
        # one int4 projection at M = 1 over 32 layers' weights, recorded once and replayed: cold weights each call
        dict(name="gemv_q4_layers", kind="gemv", enc="q4", M=1, N=8192, K=2048, kPer=0, pro="raw", epi="store", calls=32,
             mode="record"),
        # speculative verification, 1 + 4 draft rows: the gated FFN's first half, its int4 weights read once for 5 rows
        dict(name="gemvM_geglu_m5", kind="gemv", enc="q4", M=5, N=MLP, K=D, kPer=0, pro="rms", epi="geglu", calls=8,
             mode="record"),
        # the same pass over the 8-bit layers of the balanced pack
        dict(name="gemvM_q8_m5", kind="gemv", enc="q8", M=5, N=5120, K=1536, kPer=0, pro="rms", epi="store", calls=24,
             mode="record"),
        # the decode token as one persistent launch: 30 layers with the residual norm updates between the projections,
        # the head, the argmax over its tile maxima
        dict(name="token_chain", kind="step", M=1, layers=30, vocab=VOCAB, mode="chain"),
        # the same token as DecodeRunner records it by default
        dict(name="token_record", kind="step", M=1, layers=30, vocab=VOCAB, mode="record"),
        # the verify pass of 5 rows as one persistent launch
        dict(name="verify_chain_m5", kind="step", M=5, layers=30, vocab=VOCAB, mode="chain"),
        # prefill: one decoder layer's linears over a chunk of 256 prompt tokens
        dict(name="prefill_256", kind="prefill", M=256, D=D, Nqkv=QKV, MLP=MLP),
        # the text stream of a FLUX.2-klein double block: 512 text tokens
        dict(name="dit_text_512", kind="dit", M=512, D=3072, MLP=9216, heads=24),
        # a FLUX.2-klein block at 1024 x 1024: 4096 image and 512 text tokens
        dict(name="dit_flux_4608", kind="dit", M=4608, D=3072, MLP=9216, heads=24),
        # SANA-Video's gated FFN input over 21 x 30 x 52 video tokens, bf16 activations
        dict(name="glu_sana_32760", kind="gemm", M=32760, N=16384, K=3072, x="bf16", epi="swiglu"),
        # a whole weight to fp16, as a loader that hands a layer to another library does
        dict(name="dequant_9216x3072", kind="dequant", N=9216, K=3072, out="f16"),
    ]


def _log(rng, lo, hi, step):
    """a multiple of step in [lo, hi], its logarithm uniform"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemvM", "gemvM", "step", "prefill", "dit", "gemm", "gemm", "dequant"])
    if kind in ("gemv", "gemvM"):
        enc = rng.choice(["q4", "q4", "q8"])
        epi = rng.choice(["store", "store", "geglu", "softcap"])
        K = _log(rng, 256, 2048, 64)
        kPer = 0
        if epi == "store" and rng.random() < 0.3:   # a long K in partial sums of 2048, as the down projections have it
            K, kPer = _log(rng, 2112, 8192, 64), 2048
        return dict(kind="gemv", enc=enc, M=1 if kind == "gemv" else rng.randint(2, 16), N=_log(rng, 256, 16384, 64), K=K,
                    kPer=kPer, pro=rng.choice(["raw", "rms"]), epi=epi, calls=rng.randint(1, 12),
                    mode=rng.choice(["eager", "record"]))
    if kind == "step":
        return dict(kind="step", M=rng.choice([1, 1, 1, 2, 3, 4, 5, 6, 8, 12, 16]), layers=rng.randint(1, 10),
                    vocab=_log(rng, 2048, 65536, 64), mode=rng.choice(["chain", "record"]))
    if kind == "prefill":
        return dict(kind="prefill", M=_log(rng, 17, 700, 1), D=64 * rng.randint(16, 40), Nqkv=64 * rng.randint(40, 64),
                    MLP=64 * rng.randint(64, 160))
    if kind == "dit":
        heads = rng.randint(12, 28)
        return dict(kind="dit", M=_log(rng, 64, 4608, 1), D=128 * heads, MLP=128 * rng.randint(36, 72), heads=heads)
    if kind == "gemm":
        return dict(kind="gemm", M=_log(rng, 17, 16384, 1), N=_log(rng, 256, 12288, 64), K=_log(rng, 256, 8192, 32),
                    x=rng.choice(["f16", "bf16"]), epi=rng.choice(["f16", "f32", "swiglu"]))
    return dict(kind="dequant", N=_log(rng, 256, 9216, 64), K=_log(rng, 256, 8192, 32), out=rng.choice(["f16", "f32"]))


# ------------------------------------------------------------------------------------------------ inputs
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def randn(self, *shape, dtype=torch.float32):
        return torch.randn(*shape, generator=self.g, device="cuda").to(dtype)

    def q4(self, N, K, sigma):
        """q4g32a.t64 records: uniform codes, scales |N(0, sigma)|, minima that centre each group"""
        w = torch.empty(N // 64, K // 32, Q4_REC // 4, dtype=torch.int32, device="cuda")
        w.random_(-(1 << 31), 1 << 31, generator=self.g)
        s = (self.randn(N // 64, K // 32, 64).abs_() * sigma).half()
        m = (-7.5 * s.float()).half()
        w[..., 256:] = torch.stack((s, m), -1).view(torch.int32).view(N // 64, K // 32, 64)
        return w

    def q8(self, N, K, sigma):
        """q8g64s.t64 records: byte codes, scales |N(0, sigma)| / 127"""
        w = torch.empty(N // 64, K // 64, Q8_REC, dtype=torch.int8, device="cuda")
        w.random_(-127, 128, generator=self.g)
        s = (self.randn(N // 64, K // 64, 64).abs_() * (sigma / 127)).half()
        w[..., 4096:] = s.view(torch.int8).view(N // 64, K // 64, 128)
        return w


def _unit(K):
    """sigma of q4 scales whose weights keep the magnitude of a K-long input (codes about their centre: rms 4.61)"""
    return 1.0 / (4.61 * math.sqrt(K))


def _f32(*shape):
    return torch.full(shape, float("nan"), device="cuda")


def _f16(*shape):
    return torch.full(shape, float("nan"), dtype=torch.float16, device="cuda")


class _Held:
    """a recording or chain, given back with the state that holds it"""

    def __init__(self, h):
        self.h = h
        self.go = h.replay if isinstance(h, capi.Recording) else h.run

    def __del__(self):
        self.h.free()


def _enqueue(ops, mode):
    """how a program runs its op list: call by call, or recorded or chained once and launched as a whole"""
    if mode == "eager":
        return None
    return _Held(capi.record(lambda: _calls(ops)) if mode == "record" else capi.chain(lambda: _calls(ops)))


def _calls(ops):
    for fn, args in ops:
        fn(*args)


def _data(case, seed):
    """the case's tensors, from the seed alone"""
    g, k = _Gen(seed), case["kind"]
    t = {}
    if k == "gemv":
        M, N, K = case["M"], case["N"], case["K"]
        rows = 2 * N if case["epi"] == "geglu" else N
        make = (lambda: g.q4(rows, K, _unit(K))) if case["enc"] == "q4" else (lambda: g.q8(rows, K, 1.7 / math.sqrt(K)))
        t["w"] = [make() for _ in range(case["calls"])]
        t["x"] = g.randn(M, K)
        t["st"] = 0.8 + 0.4 * torch.rand(M, 2, generator=g.g, device="cuda")
        t["nw"] = 1.0 + 0.2 * g.randn(K)
    elif k == "step":
        M = case["M"]
        t["layers"] = [dict(qkv=g.q4(QKV, D, _unit(D)), o=g.q4(D, D, _unit(D)), gu=g.q4(2 * MLP, D, _unit(D)),
                            down=g.q4(D, MLP, 2.0 * _unit(MLP)), nw=1.0 + 0.2 * g.randn(4, D))
                       for _ in range(case["layers"])]
        t["head"] = g.q4(case["vocab"], D, 4.0 * _unit(D))
        t["hnw"] = 1.0 + 0.2 * g.randn(D)
        t["x"] = g.randn(M, D)
    elif k == "prefill":
        M, d, n, h = case["M"], case["D"], case["Nqkv"], case["MLP"]
        t.update(x=g.randn(M, d), qkv=g.q4(n, d, _unit(d)), o=g.q4(d, d, _unit(d)), gu=g.q4(2 * h, d, _unit(d)),
                 down=g.q4(d, h, 2.0 * _unit(h)), nw=1.0 + 0.2 * g.randn(4, d))
    elif k == "dit":
        M, d, h = case["M"], case["D"], case["MLP"]
        t.update(x=g.randn(M, d), att=g.randn(M, d, dtype=torch.float16), qkv=g.q4(3 * d, d, _unit(d)),
                 proj=g.q4(d, d, _unit(d)), up=g.q4(2 * h, d, _unit(d)), down=g.q4(d, h, 2.0 * _unit(h)),
                 mod=0.2 * g.randn(6, d), qknorm=1.0 + 0.2 * g.randn(2, 128))
        ang = torch.rand(M, 64, generator=g.g, device="cuda") * 6.28
        t["rope"] = torch.stack((ang.cos(), ang.sin()), -1).contiguous()
    elif k == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        t["x"] = g.randn(M, K, dtype=torch.float16 if case["x"] == "f16" else torch.bfloat16)
        t["w"] = g.q4(N, K, _unit(K))
    else:
        t["w"] = g.q4(case["N"], case["K"], 0.02)
    return t


def prepare(case, seed):
    capi.open_device(0)
    t = _data(case, seed)
    k = case["kind"]
    keep, mode = [t], "eager"
    ops = []
    if k == "gemv":
        out, mode = _gemv_ops(case, t, ops), case["mode"]
    elif k == "step":
        out, mode = _step_ops(case, t, ops, keep), case["mode"]
    elif k == "prefill":
        out = _prefill_ops(case, t, ops, keep)
    elif k == "dit":
        out = _dit_ops(case, t, ops, keep)
    elif k == "gemm":
        out = _gemm_ops(case, t, ops)
    else:
        N, K = case["N"], case["K"]
        out = (_f16 if case["out"] == "f16" else _f32)(N, K)
        ops.append((capi.q4_dequant, (t["w"].data_ptr(), N, K, None if case["out"] == "f16" else out.data_ptr(),
                                      out.data_ptr() if case["out"] == "f16" else None)))
    if k in ("prefill", "dit", "gemm"):   # a program sizes the library's staging workspace with its first layer
        _calls(ops)
    torch.cuda.synchronize()
    return dict(ops=ops, held=_enqueue(ops, mode), out=out, keep=keep)


def run(state):
    if state["held"] is None:
        _calls(state["ops"])
    else:
        state["held"].go()
    return state["out"]


def _gemv_ops(case, t, ops):
    M, N, K, kPer = case["M"], case["N"], case["K"], case["kPer"]
    geglu, softcap = case["epi"] == "geglu", case["epi"] == "softcap"
    ns = -(-K // kPer) if kPer else 1
    out = dict(y=_f32(case["calls"], ns, M, N))
    mx = None
    if softcap:   # the tile maxima; behind them the rstd slot, which a softcap gemv takes from there
        mx = _f32(case["calls"], M * (N // 64) * 2 + 2)
        mx[:, -2] = t["st"][0, 1]
    kw = dict(w_enc=1 if case["enc"] == "q4" else 2, w_rows=2 * N if geglu else N, w_cols=K, x=t["x"].data_ptr(), N=N, K=K,
              kPer=kPer, pro=capi.PRO[case["pro"]], epi=capi.EPI[case["epi"]], stat=t["st"].data_ptr(), stat_off=1,
              norm=t["nw"].data_ptr())
    for i, w in enumerate(t["w"]):
        a = dict(kw, w=w.data_ptr(), y=out["y"][i].data_ptr(), mx=mx[i].data_ptr() if softcap else None)
        if softcap and M == 1:
            a["stat_off"] = N // 64 * 2
        ops.append((capi.q4_gemv, (capi.gemv_args(**a),)) if M == 1 else
                   (capi.q4_gemvM, (capi.gemvm_args(M=M, stat_ld=2, **a),)))
    if softcap:
        # (max, bits of the row index) pairs: the index words are whole numbers
        mx = mx[:, :-2].unflatten(1, (M, N // 64, 2))
        out["mx"] = dict(value=mx[..., 0], row=mx.view(torch.int32)[..., 1])
    return out


def _step_ops(case, t, ops, keep):
    """one decode token (M = 1) or verify pass: the residual stream x and its rstd, updated by a normadd after each half
    layer. o reads the q rows of qkv's output in place of the attention's"""
    M, V = case["M"], case["vocab"]
    b = dict(x=_f32(M, D), st=_f32(M), qkv=_f32(M, QKV), o=_f32(M, D), m=_f32(M, MLP), dp=_f32(4, M, D),
             logits=_f32(M, V), mx=_f32(M * (V // 64) * 2 + 2), arg=torch.zeros(M, 2, dtype=torch.int32, device="cuda"))
    keep.append(b)

    def gemv(w, n, k, x, ldx, y, pro="raw", epi="store", kPer=0, st=None, st_off=0, nw=None, mx=None):
        N = n // 2 if epi == "geglu" else n
        kw = dict(w=w.data_ptr(), w_rows=n, w_cols=k, x=x.data_ptr(), N=N, K=k, kPer=kPer, pro=capi.PRO[pro],
                  epi=capi.EPI[epi], y=y.data_ptr(), stat=st, stat_off=st_off,
                  norm=None if nw is None else nw.data_ptr(), mx=mx)
        ops.append((capi.q4_gemv, (capi.gemv_args(**kw),)) if M == 1 else
                   (capi.q4_gemvM, (capi.gemvm_args(M=M, x_ldx=ldx, stat_ld=1, **kw),)))

    def normadd(src, n, w, mode):
        ops.append((capi.normadd, (capi.normadd_args(t=src.data_ptr(), t_n=n, w=None if w is None else w.data_ptr(),
                                                     x=b["x"].data_ptr(), st=b["st"].data_ptr(), D=D, M=M, eps=EPS,
                                                     mode=mode),)))

    normadd(t["x"], 1, None, 1)   # the embedding becomes the residual stream
    x, st = b["x"], b["st"].data_ptr()
    for ly in t["layers"]:
        gemv(ly["qkv"], QKV, D, x, D, b["qkv"], "rms", st=st, nw=ly["nw"][0])
        gemv(ly["o"], D, D, b["qkv"], QKV, b["o"], kPer=2048)
        normadd(b["o"], 1, ly["nw"][1], 0)
        gemv(ly["gu"], 2 * MLP, D, x, D, b["m"], "rms", "geglu", st=st, nw=ly["nw"][2])
        gemv(ly["down"], D, MLP, b["m"], MLP, b["dp"], kPer=2048)
        normadd(b["dp"], 4, ly["nw"][3], 0)
    if M == 1:   # a softcap gemv takes its rstd slot from behind the tile maxima
        ops.append((capi.copy, (st, 0, b["mx"].data_ptr(), V // 64 * 8, 4)))
    gemv(t["head"], V, D, x, D, b["logits"], "rms", "softcap", st=st, st_off=V // 64 * 2 if M == 1 else 0, nw=t["hnw"],
         mx=b["mx"].data_ptr())
    ops.append((capi.argmax, (b["mx"].data_ptr(), V // 64, b["arg"].data_ptr())) if M == 1 else
               (capi.argmaxM, (b["mx"].data_ptr(), V // 64, M, b["arg"].data_ptr())))
    return dict(logits=b["logits"], top=b["arg"].view(torch.float32)[:, 1])


def _prefill_ops(case, t, ops, keep):
    """one decoder layer's linears over M prompt tokens: the residual stream x in fp32, RMS prologues, the gated FFN with
    tanh-GELU, a normadd after each half. The q rows of qkv stand in for the attention's output"""
    M, d, n, h = case["M"], case["D"], case["Nqkv"], case["MLP"]
    b = dict(x=_f32(M, d), st=_f32(M, 2), rs=_f32(M), qkv=_f16(M, n), t=_f32(M, d), m=_f16(M, h))
    keep.append(b)
    p = {k: v.data_ptr() for k, v in b.items()}

    def gemm(w, N, K, x, epi, y, **kw):
        ops.append((capi.q4_gemm, (capi.gemm_args(w=w.data_ptr(), w_rows=N, w_cols=K, x=x, M=M, N=N, K=K,
                                                  epi=capi.GEPI[epi], y=y, **kw),)))

    def rms(nw):
        ops.append((capi.rowstats, (capi.rowstats_args(x=p["x"], rows=M, cols=d, mode=1, eps=EPS, st=p["st"]),)))
        return dict(x_mode=capi.XMODE["rms"], stats=p["st"], pv=nw.data_ptr())

    def normadd(w):
        ops.append((capi.normadd, (capi.normadd_args(t=p["t"], w=w.data_ptr(), x=p["x"], st=p["rs"], D=d, M=M, eps=EPS),)))

    ops.append((capi.copy, (t["x"].data_ptr(), 0, p["x"], 0, 4 * M * d)))
    gemm(t["qkv"], n, d, p["x"], "f16", p["qkv"], **rms(t["nw"][0]))
    gemm(t["o"], d, d, p["qkv"], "f32", p["t"], x_ld=n)
    normadd(t["nw"][1])
    gemm(t["gu"], 2 * h, d, p["x"], "swiglu", p["m"], wr1=h, act=capi.ACT["gelu"], y_ld=h, **rms(t["nw"][2]))
    gemm(t["down"], d, h, p["m"], "f32", p["t"])
    normadd(t["nw"][3])
    return dict(qkv=b["qkv"], m=b["m"], x=b["x"], rstd=b["rs"])


def _dit_ops(case, t, ops, keep):
    """a DiT block's linears over M tokens: LayerNorm statistics and modulation in the qkv and FFN prologues, QK-norm and
    RoPE in the heads epilogue, gated residual adds. att stands for the attention's output"""
    M, d, h, H = case["M"], case["D"], case["MLP"], case["heads"]
    b = dict(x=_f32(M, d), st=_f32(M, 2), y=_f16(3 * H, M, 128), m=_f16(M, h))
    keep.append(b)
    p = {k: v.data_ptr() for k, v in b.items()}

    def gemm(w, N, K, x, epi, y, **kw):
        ops.append((capi.q4_gemm, (capi.gemm_args(w=w.data_ptr(), w_rows=N, w_cols=K, x=x, M=M, N=N, K=K,
                                                  epi=capi.GEPI[epi], y=y, **kw),)))

    def lnmod(i):   # rows of mod: shift, scale, gate of the attention half, then of the FFN half
        ops.append((capi.rowstats, (capi.rowstats_args(x=p["x"], rows=M, cols=d, mode=0, eps=EPS, st=p["st"]),)))
        return dict(x_mode=capi.XMODE["lnmod"], stats=p["st"], pv=t["mod"].data_ptr(), pv_off=(3 * i + 1) * d,
                    pv_stride=(1 << 32) - d)

    ops.append((capi.copy, (t["x"].data_ptr(), 0, p["x"], 0, 4 * M * d)))
    gemm(t["qkv"], 3 * d, d, p["x"], "heads", p["y"], ev=t["qknorm"].data_ptr(), heads_ltot=M, heads_hq=H, heads_hkv=H,
         heads_eps=EPS, heads_rope=capi.ROPE["inter"], rope=t["rope"].data_ptr(), **lnmod(0))
    gemm(t["proj"], d, d, t["att"].data_ptr(), "resadd", p["x"], ev=t["mod"].data_ptr(), ev_off=2 * d)
    gemm(t["up"], 2 * h, d, p["x"], "swiglu", p["m"], wr1=h, act=capi.ACT["silu"], y_ld=h, **lnmod(1))
    gemm(t["down"], d, h, p["m"], "resadd", p["x"], ev=t["mod"].data_ptr(), ev_off=5 * d)
    return dict(heads=b["y"], m=b["m"], x=b["x"])


def _gemm_ops(case, t, ops):
    M, N, K, sw = case["M"], case["N"], case["K"], case["epi"] == "swiglu"
    y = (_f32 if case["epi"] == "f32" else _f16)(M, N // 2 if sw else N)
    ops.append((capi.q4_gemm, (capi.gemm_args(w=t["w"].data_ptr(), w_rows=N, w_cols=K, x=t["x"].data_ptr(), M=M, N=N, K=K,
                                              x_mode=capi.XMODE[case["x"]], epi=capi.GEPI[case["epi"]], y=y.data_ptr(),
                                              y_ld=y.shape[1], wr1=N // 2 if sw else 0, act=capi.ACT["silu"]),)))
    return y


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _q4_bytes(n, k):
    return n // 64 * (k // 32) * Q4_REC


def work(case):
    k = case["kind"]
    M, byt, fl = case.get("M", 1), 0, 0
    if k == "gemv":
        N, K, c = case["N"], case["K"], case["calls"]
        rows = 2 * N if case["epi"] == "geglu" else N
        ns = -(-K // case["kPer"]) if case["kPer"] else 1
        byt = c * (_q4_bytes(rows, K) if case["enc"] == "q4" else rows // 64 * (K // 64) * Q8_REC) + M * K * 4
        byt += c * (M * N * ns * 4 + (M * (N // 64) * 8 if case["epi"] == "softcap" else 0))
        fl = c * 2 * M * rows * K
    elif k == "step":
        n = [(QKV, D), (D, D), (2 * MLP, D), (D, MLP)] * case["layers"] + [(case["vocab"], D)]
        byt = sum(_q4_bytes(a, b) for a, b in n) + M * case["vocab"] * 4 + M * D * 4
        fl = sum(2 * M * a * b for a, b in n)
    elif k == "prefill":
        d, h = case["D"], case["MLP"]
        n = [(case["Nqkv"], d), (d, d), (2 * h, d), (d, h)]
        byt = sum(_q4_bytes(a, b) for a, b in n) + M * (case["Nqkv"] * 2 + h * 2 + d * 8)
        fl = sum(2 * M * a * b for a, b in n)
    elif k == "dit":
        d, h = case["D"], case["MLP"]
        n = [(3 * d, d), (d, d), (2 * h, d), (d, h)]
        byt = sum(_q4_bytes(a, b) for a, b in n) + M * (d * 2 + 3 * d * 2 + h * 2 + d * 8 + 512)
        fl = sum(2 * M * a * b for a, b in n)
    elif k == "gemm":
        N, K = case["N"], case["K"]
        byt = _q4_bytes(N, K) + M * K * 2 + M * N * {"f16": 2, "f32": 4, "swiglu": 1}[case["epi"]]
        fl = 2 * M * N * K
    else:
        N, K = case["N"], case["K"]
        byt = _q4_bytes(N, K) + N * K * (2 if case["out"] == "f16" else 4)
        fl = 2 * N * K
    return dict(bytes=byt, flops=fl)


def tolerance(case):
    """about four times what this path is off exact() (in brackets: the largest relative errors seen over drawn cases)"""
    k = case["kind"]
    if k == "dequant":
        return "exact"                  # fl32(q s + m), and fl16 of that: one value
    if k == "gemv":                     # fp32 sums of fp32 activations (7e-7); a tile's row index where two rows tie
        return dict(rel=5e-6, max=5e-5, differ=0.01 if case["epi"] == "softcap" else 0)
    if k == "step":                     # the same through every layer, at most 30 of them (1.2e-6)
        return dict(rel=1e-5, max=1e-4)
    if k == "gemm" and case["epi"] == "f32":   # fp32 sums over fp16 tiles (2e-7; bf16 inputs below 2^-14 round: 1e-6)
        return dict(rel=5e-6, max=5e-5)
    if k == "gemm":                     # the same, rounded to fp16 (2.1e-4)
        return dict(rel=1e-3, max=5e-3)
    return dict(rel=2e-3, max=2e-2)     # prologue values rounded to fp16 tiles, fp16 outputs between GEMMs (4.7e-4)


# ------------------------------------------------------------------------------------------------ the same in float64
def _deq64(w, N, K, half=False, r0=0, r1=None):
    """rows r0 .. r1 - 1 (whole 64-row tiles) of a q4 weight; half: rounded to fp16, as the GEMM's tile holds it"""
    w = w[r0 // 64:(N if r1 is None else r1) // 64]
    n = w.shape[0]
    c = w[..., :256].reshape(n, K // 32, 64, 4, 1)
    q = ((c >> torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)) & 15).double()
    sm = w[..., 256:].contiguous().view(torch.float16).view(n, K // 32, 64, 2).double()
    v = q * sm[..., 0, None, None] + sm[..., 1, None, None]
    if half:
        v = v.float().half().double()
    return v.permute(0, 2, 1, 3, 4).reshape(n * 64, K)


def _deq64_q8(w, N, K):
    q = w[..., :4096].reshape(N // 64, K // 64, 64, 64).double()
    s = w[..., 4096:].contiguous().view(torch.float16).view(N // 64, K // 64, 64, 1).double()
    return (q * s).permute(0, 2, 1, 3).reshape(N, K)


def _gelu64(v):
    t = 0.7978845608028654 * (v + 0.044715 * v ** 3)
    return v * 0.5 * (1.0 + torch.tanh(t.clamp(-15, 15)))


def _softcap64(v):
    return 30.0 * torch.tanh((v / 30.0).clamp(-15, 15))


def _mm(x, w, N, K, half=False, rows=16384):
    """x W^T over a q4 weight, some rows of W at a time"""
    return torch.cat([x @ _deq64(w, N, K, half, r, min(N, r + rows)).T for r in range(0, N, rows)], 1)


def _rstd64(x):
    return 1.0 / torch.sqrt((x * x).mean(1, keepdim=True) + EPS)


def exact(case, seed):
    t, k = _data(case, seed), case["kind"]
    if k == "gemv":
        M, N, K, kPer = case["M"], case["N"], case["K"], case["kPer"] or case["K"]
        x = t["x"].double()
        if case["pro"] == "rms":
            x = x * t["st"][:, 1:].double() * t["nw"].double()
        ys = []
        for w in t["w"]:
            rows = 2 * N if case["epi"] == "geglu" else N
            w = _deq64(w, rows, K) if case["enc"] == "q4" else _deq64_q8(w, rows, K)
            y = torch.stack([x[:, a:a + kPer] @ w[:, a:a + kPer].T for a in range(0, K, kPer)])
            if case["epi"] == "geglu":
                y = _gelu64(y[..., :N]) * y[..., N:]
            ys.append(_softcap64(y) if case["epi"] == "softcap" else y)
        y = torch.stack(ys)
        if case["epi"] == "softcap":
            return dict(y=y, mx=dict(value=y[:, 0].reshape(case["calls"], M, N // 64, 64).amax(-1), row=None))
        return dict(y=y)
    if k == "step":
        x = t["x"].double()
        for ly in t["layers"]:
            nw = ly["nw"].double()
            a = _mm(x * _rstd64(x) * nw[0], ly["qkv"], QKV, D)
            v = _mm(a[:, :D], ly["o"], D, D)
            x = x + v * _rstd64(v) * nw[1]
            g = _mm(x * _rstd64(x) * nw[2], ly["gu"], 2 * MLP, D)
            v = _mm(_gelu64(g[:, :MLP]) * g[:, MLP:], ly["down"], D, MLP)
            x = x + v * _rstd64(v) * nw[3]
        h = x * _rstd64(x) * t["hnw"].double()
        logits = _softcap64(_mm(h, t["head"], case["vocab"], D))
        return dict(logits=logits, top=logits.amax(1))
    if k == "prefill":
        d, n, h = case["D"], case["Nqkv"], case["MLP"]
        x, nw = t["x"].double(), t["nw"].double()
        a = _mm(x * _rstd64(x) * nw[0], t["qkv"], n, d, True)
        v = _mm(a[:, :d], t["o"], d, d, True)
        x = x + v * _rstd64(v) * nw[1]
        g = _mm(x * _rstd64(x) * nw[2], t["gu"], 2 * h, d, True)
        m = _gelu64(g[:, :h]) * g[:, h:]
        v = _mm(m, t["down"], d, h, True)
        x = x + v * _rstd64(v) * nw[3]
        return dict(qkv=a, m=m, x=x, rstd=_rstd64(x).view(-1))
    if k == "dit":
        M, d, h, H = case["M"], case["D"], case["MLP"], case["heads"]
        x, mod = t["x"].double(), t["mod"].double()

        def ln(v, i):
            c = v - v.mean(1, keepdim=True)
            return c / torch.sqrt((c * c).mean(1, keepdim=True) + EPS) * (1 + mod[3 * i + 1]) + mod[3 * i]

        a = _mm(ln(x, 0), t["qkv"], 3 * d, d, True).view(M, 3 * H, 128).transpose(0, 1)
        nw = t["qknorm"].double().repeat_interleave(H, 0).view(2 * H, 1, 128)
        qk = a[:2 * H] / torch.sqrt((a[:2 * H] ** 2).mean(-1, keepdim=True) + EPS) * nw
        c, s = t["rope"].double().unbind(-1)
        e, o = qk[..., 0::2], qk[..., 1::2]
        qk = torch.stack((e * c - o * s, e * s + o * c), -1).flatten(-2)
        x = x + mod[2] * _mm(t["att"].double(), t["proj"], d, d, True)
        g = _mm(ln(x, 1), t["up"], 2 * h, d, True)
        m = torch.nn.functional.silu(g[:, :h]) * g[:, h:]
        return dict(heads=torch.cat((qk, a[2 * H:])), m=m, x=x + mod[5] * _mm(m, t["down"], d, h, True))
    if k == "gemm":
        N, K = case["N"], case["K"]
        y = _mm(t["x"].double(), t["w"], N, K, True)
        return torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:] if case["epi"] == "swiglu" else y
    v = _deq64(t["w"], case["N"], case["K"]).float()
    return v.half() if case["out"] == "f16" else v
