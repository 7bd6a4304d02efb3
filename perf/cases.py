"""The work a user of this library has it do, as cases to be timed: dense projections of a decode step, the dense half of a
decode layer, the decode MoE step of each weight format, and prefill chunks, each through the public entry points of
dsgx10_amd.lib.

Shapes: the FP8 layer (hidden 4096, intermediate 2048, 256 experts, top-8, FP8 shared expert), the INT4 layer (hidden 6144,
intermediate 2048, 168 experts, top-8, BF16 shared expert) and DeepSeek's MXFP4 layer (hidden 5120, intermediate 2304, 256
experts, top-6, FP8 shared expert), with their attention projections; draw() spreads over the sizes around them. Weights are
N(0, 0.02) values quantised as the formats' checkpoints are, rows N(0, 1), the prefill chunks' picks follow a Zipf popularity."""
import math

import numpy as np
import torch

from dsgx10_amd import abi, lib
from dsgx10_amd.layer import DESC_DTYPE, mat_bytes

FMT = {"fp8": abi.FMT_FP8, "int4": abi.FMT_INT4, "bf16": abi.FMT_BF16}
OUT = {"bf16": abi.OUT_BF16, "f32": abi.OUT_F32, "swiglu": abi.OUT_SWIGLU}
STEP_LAYERS = 4  # MoE layers of one decode pass: a step goes through layer after layer, each with its own routing
ZIPF = 1.1


def listed():
    fp8 = dict(fmt="fp8", H=4096, I=2048, E=256, topk=8, shared=True)
    int4 = dict(fmt="int4", H=6144, I=2048, E=168, topk=8, shared=True)
    dsk = dict(H=5120, I=2304, E=256, topk=6, shared=True)
    return [
        # the smallest call: one token through one small projection, where the launch and the call itself are the time
        dict(name="gemv fp8 1 row", kind="gemv", fmt="fp8", N=2048, K=4096, rows=1, out="bf16", splitk=2),
        # speculative decoding: a few drafted tokens of the widest INT4 projection (64 heads x 256 back to the hidden size)
        dict(name="gemv int4 4 rows", kind="gemv", fmt="int4", N=6144, K=16384, rows=4, out="f32", splitk=1),
        # one token through the projections of a layer: norm, x-projection, q_b, o_proj, norm + router
        dict(name="dense half fp8 1 row", kind="dense", fmt="fp8", H=4096, XR=2112, QL=1536, NQ=16384, E=256, rows=1),
        # the same in the INT4 checkpoint for a few concurrent streams
        dict(name="dense half int4 3 rows", kind="dense", fmt="int4", H=6144, XR=2752, QL=2048, NQ=16384, E=168, rows=3),
        # one stream's decode step through MoE layers with the routing inside
        dict(name="moe fp8 1 row", kind="moe", M=1, **fp8),
        # many streams at once: more rows than one pass of the kernels takes, an odd number of them
        dict(name="moe fp8 13 rows", kind="moe", M=13, **fp8),
        # the INT4 checkpoint beside its BF16 shared expert, a handful of streams
        dict(name="moe int4 6 rows", kind="moe", M=6, **int4),
        # DeepSeek's layer, two streams
        dict(name="dsk 2 rows", kind="dsk", M=2, **dsk),
        # a short prompt
        dict(name="prefill fp8 200 rows", kind="prefill", T=200, act_fp8=True, **fp8),
        # the largest chunk a call takes
        dict(name="prefill fp8 8192 rows", kind="prefill", T=8192, act_fp8=True, **fp8),
        # an ordinary prompt of an odd length in the INT4 checkpoint
        dict(name="prefill int4 1111 rows", kind="prefill", T=1111, act_fp8=False, **int4),
        # an ordinary prompt through DeepSeek's layer
        dict(name="dsk prefill 3000 rows", kind="dsk_prefill", T=3000, **dsk),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, m):
    return m * rng.randint(-(-lo // m), hi // m)


def _max_k(rows):
    """The longest K whose activation rows (eight at a time) fit the LDS: 128 KiB of bf16, in whole segments of 2048 k"""
    return 65536 // min(rows, 8) // 2048 * 2048


def draw(rng):
    """One more case of the same ranges. Sizes keep to what the formats take: an FP8 matrix's K is whole 128-blocks, the
    expert kernels' sizes are multiples of 256 (BF16 experts: 512)."""
    kind = rng.choice(["gemv"] * 3 + ["dense"] * 2 + ["moe"] * 4 + ["dsk"] * 2 + ["prefill"] * 3 + ["dsk_prefill"])
    if kind == "gemv":
        fmt = rng.choice(["fp8", "int4", "bf16"])
        N, K = 8 * max(8, _log(rng, 64, 16384) // 8), 128 * max(2, _log(rng, 1024, 16384) // 128)
        if fmt == "int4":
            K = 256 * max(1, K // 256)
        if fmt == "bf16":  # (the checkpoints' BF16 matrices are the small ones: routers and x-projections)
            N, K = min(N, 4096), min(K, 8192)
        out = rng.choice(["bf16", "f32"]) if fmt == "fp8" else rng.choice(["bf16", "f32", "swiglu"])
        rows = rng.choice([1, 1, 2, 3, 4, 5, 6, 7, 8, 11, 16])
        return dict(kind=kind, fmt=fmt, N=N, K=min(K, _max_k(rows)), rows=rows, out=out, splitk=rng.choice([1, 1, 2, 4]))
    if kind == "dense":
        XR, rows = _mult(rng, 1024, 2816, 64), rng.choice([1, 1, 2, 3, 4, 6, 8])
        return dict(kind=kind, fmt=rng.choice(["fp8", "int4"]), H=rng.choice([2048, 4096, 6144]), XR=XR, QL=min(_mult(rng, 1024, 2048, 256), XR // 256 * 256),
                    NQ=min(_mult(rng, 4096, 16384, 1024), _max_k(rows)), E=_mult(rng, 64, 256, 8), rows=rows)
    H, I, E = _mult(rng, 1024, 6144, 256), _mult(rng, 512, 2304, 256), _log(rng, 16, 256)
    topk = rng.choice([4, 6, 8, 8])
    shared = rng.random() < 0.75
    if kind in ("moe", "dsk"):
        c = dict(kind=kind, H=H, I=I, E=E, topk=topk, shared=shared, M=rng.choice([1, 1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 16]))
        if kind == "moe":
            c["fmt"] = rng.choice(["fp8", "fp8", "fp8", "int4", "int4", "int4", "bf16"])
            if c["fmt"] == "bf16":  # (BF16 experts have no fused shared expert; a layer of them is small)
                c.update(shared=False, H=max(1, H // 512) * 512, I=max(1, I // 512) * 512, E=min(E, 64))
        return c
    if kind == "dsk_prefill":
        return dict(kind=kind, H=H, I=I, E=E, topk=min(topk, 6), shared=shared, T=_log(rng, 17, 6000))
    fmt = rng.choice(["fp8", "fp8", "int4"])
    return dict(kind=kind, fmt=fmt, H=min(H, 4096) if fmt == "fp8" else H, I=min(I, 2048), E=E, topk=topk, shared=shared,
                T=_log(rng, 17, 8192 if fmt == "fp8" else 2500), act_fp8=fmt == "fp8" and (rng.random() < 0.8 or H * I > 4096 * 1024))


# ---- weights, quantised as the formats define them ---------------------------------------------------------------------------
def _al256(n):
    return (n + 255) // 256 * 256


class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, shape, sigma=1.0, dtype=torch.float32):
        return (torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32) * sigma).to(dtype)


def _chunks(n, each):
    per = max(1, 200_000_000 // each)
    return [(a, min(n, a + per)) for a in range(0, n, per)]


def _fp8(w):
    """w f32 [c][N][K] (N whole 128-blocks) -> e4m3 codes [c][N][K], f32 scales [c][N/128][K/128]: scale = amax / 448"""
    c, N, K = w.shape
    blk = w.view(c, N // 128, 128, K // 128, 128)
    s = (blk.abs().amax(dim=(2, 4)) * (1.0 / 448.0)).clamp_min(1e-12)
    return (blk / s[:, :, None, :, None]).to(torch.float8_e4m3fn).view(torch.uint8).view(c, N, K), s


def _int4(w):
    """w f32 [c][N][K] -> packed i32 [c][N][K/8], bf16 scales [c][N][K/32], zero points i32 [c][N/8][K/32]: asymmetric, a
    scale and a zero point a group of 32 along K"""
    c, N, K = w.shape
    g = w.view(c, N, K // 32, 32)
    lo, hi = g.amin(-1).clamp_max(0.0), g.amax(-1).clamp_min(0.0)
    s = ((hi - lo) / 15.0).clamp_min(1e-8).to(torch.bfloat16)
    z = (-lo / s.float()).round().clamp(0, 15)
    u = ((g / s.float()[..., None]).round() + z[..., None]).clamp(0, 15).to(torch.int32)
    sh = torch.arange(8, device=w.device, dtype=torch.int32) * 4
    pack = lambda v, shift: (v << shift).sum(-1, dtype=torch.int32)  # (disjoint nibbles: the sum is their or)
    words = pack(u.view(c, N, K // 8, 8), sh)
    zp = pack(z.to(torch.int32).view(c, N // 8, 8, K // 32).transpose(2, 3), sh)
    return words, s, zp


def _mxfp4(w):
    """w f32 [c][N][K] -> e2m1 pairs u8 [c][N][K/2] (the low nibble the even k), ue8m0 scales u8 [c][N][K/32]"""
    c, N, K = w.shape
    g = w.view(c, N, K // 32, 32)
    e = torch.ceil(torch.log2((g.abs().amax(-1) / 6.0).clamp_min(2.0 ** -100)))
    v = g * torch.exp2(-e)[..., None]
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=w.device)
    code = torch.bucketize(v.abs(), edges, out_int32=True).to(torch.uint8) | ((v < 0).to(torch.uint8) << 3)
    code = code.view(c, N, K // 2, 2)
    return (code[..., 0] | (code[..., 1] << 4)), (e + 127.0).to(torch.uint8)


def _fp8e(w):
    """w f32 [N][K] -> e4m3 codes [N][K], ue8m0 scales u8 [N/32][K/32], one a 32 x 32 block"""
    N, K = w.shape
    blk = w.view(N // 32, 32, K // 32, 32)
    e = torch.ceil(torch.log2((blk.abs().amax(dim=(1, 3)) / 448.0).clamp_min(2.0 ** -100)))
    q = (blk * torch.exp2(-e)[:, None, :, None]).to(torch.float8_e4m3fn).view(torch.uint8).view(N, K)
    return q.contiguous(), (e + 127.0).to(torch.uint8).contiguous()


def _dense(g, fmt, N, K):
    """One dense matrix as lib.gemv takes it (without n, y, ldy)."""
    if fmt == "fp8":
        q, s = _fp8(g.normal((1, (N + 127) // 128 * 128, K), 0.02))
        return dict(fmt=FMT[fmt], w=q[0, :N].contiguous(), s=s[0].contiguous())
    if fmt == "int4":
        p, s, z = _int4(g.normal((1, N, K), 0.02))
        return dict(fmt=FMT[fmt], w=p[0], s=s[0], zp=z[0])
    return dict(fmt=FMT[fmt], w=g.normal((N, K), 0.02, torch.bfloat16))


def _pool(g, c):
    """The layer's experts in one pool and their descriptors (include/dsgx.h's layouts)."""
    fmt, H, I, E = FMT[c["fmt"]], c["H"], c["I"], c["E"]
    shapes = [(I, H), (I, H), (H, I)]
    per = [mat_bytes(fmt, N, K) for N, K in shapes]
    pool = torch.empty((E, sum(per)), dtype=torch.uint8, device="cuda")
    at = 0
    for (N, K), nbytes in zip(shapes, per):
        for a, b in _chunks(E, N * K):
            w = g.normal((b - a, N, K), 0.02)
            if c["fmt"] == "fp8":
                parts = _fp8(w)
            elif c["fmt"] == "int4":
                parts = _int4(w)
            else:
                parts = (w.to(torch.bfloat16),)
            o = at
            for p in parts:
                p = p.contiguous().view(torch.uint8).view(b - a, -1)
                pool[a:b, o:o + p.shape[1]] = p
                o += _al256(p.shape[1])
        at += nbytes
    desc = np.zeros((E, 3), DESC_DTYPE)
    desc["off"] = np.arange(E)[:, None] * sum(per) + np.cumsum([0] + per[:2])[None, :]
    desc["s2"], desc["fmt"] = 1.0, fmt
    return pool, torch.from_numpy(desc.view(np.uint8).reshape(-1).copy()).cuda()


def _layer_w(c, pool, desc, shared):
    L = abi.LayerW()
    L.pool, L.desc = pool.data_ptr(), desc.data_ptr()
    L.fmt, L.H, L.I, L.E, L.topk = FMT[c["fmt"]], c["H"], c["I"], c["E"], c["topk"]
    if shared and c["fmt"] == "fp8":
        (L.sh.g, L.sh.gs), (L.sh.u, L.sh.us), (L.sh.d, L.sh.ds) = [(q.data_ptr(), s.data_ptr()) for q, s in shared]
    elif shared:
        L.sh.bgu, L.sh.bd = [t.data_ptr() for t in shared]
    return L


def _shared(g, c):
    """A shared expert beside the layer's experts: FP8 beside FP8, BF16 (gate and up interleaved) beside INT4."""
    H, I = c["H"], c["I"]
    if not c["shared"]:
        return None
    if c["fmt"] == "fp8":
        return [tuple(t[0].contiguous() for t in _fp8(g.normal((1, N, K), 0.02))) for N, K in ((I, H), (I, H), (H, I))]
    return [g.normal((2 * I, H), 0.02, torch.bfloat16), g.normal((H, I), 0.02, torch.bfloat16)]


def _dsk_weights(g, c):
    """DeepSeek's layer: experts stacked by id as MXFP4, the shared expert as FP8 with ue8m0 scales per 32 x 32."""
    H, I, E = c["H"], c["I"], c["E"]
    t = {}
    for n, (N, K) in (("1", (I, H)), ("3", (I, H)), ("2", (H, I))):
        t["w" + n] = torch.empty((E, N, K // 2), dtype=torch.uint8, device="cuda")
        t["s" + n] = torch.empty((E, N, K // 32), dtype=torch.uint8, device="cuda")
        for a, b in _chunks(E, N * K):
            t["w" + n][a:b], t["s" + n][a:b] = _mxfp4(g.normal((b - a, N, K), 0.02))
        if c["shared"]:
            t["sh_w" + n], t["sh_s" + n] = _fp8e(g.normal((N, K), 0.02))
    names = ("w1", "s1", "w3", "s3", "w2", "s2", "sh_w1", "sh_s1", "sh_w3", "sh_s3", "sh_w2", "sh_s2")
    return t, abi.DskWeights(*[t[k].data_ptr() if k in t else None for k in names], H, I, E, c["topk"])


def _act_quant32(x):
    """Rows f32 [T][H] -> e4m3 codes and a ue8m0 scale per 32 values (the smallest power of two that covers amax / 448)"""
    T, H = x.shape
    blk = x.view(T, H // 32, 32)
    e = torch.ceil(torch.log2(blk.abs().amax(-1).clamp_min(1e-4) / 448.0))
    q = (blk * torch.exp2(-e)[..., None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8).view(T, H)
    return q.contiguous(), (e + 127.0).to(torch.uint8).contiguous()


def _zipf_logits(g, T, E):
    """Router logits whose top-k are drawn without replacement from a Zipf popularity over a seeded permutation of the experts"""
    logp = -ZIPF * torch.log(torch.randperm(E, generator=g.g, device="cuda").float() + 1.0)
    u = torch.rand((T, E), generator=g.g, device="cuda").clamp(1e-7, 1 - 1e-7)
    return (logp[None, :] - torch.log(-torch.log(u))).contiguous()


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda")


# ---- prepare and run ---------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    c, g = case, _Gen(seed)
    k = c["kind"]
    s = dict(case=c)
    if k == "gemv":
        ncol = c["N"] // 2 if c["out"] == "swiglu" else c["N"]
        s["x"] = g.normal((c["rows"], c["K"]), 1.0, torch.bfloat16)
        s["y"] = _empty(c["rows"], ncol, dtype=torch.float32 if c["out"] == "f32" else torch.bfloat16)
        s["segs"] = [dict(_dense(g, c["fmt"], c["N"], c["K"]), n=c["N"], y=s["y"], ldy=ncol)]
    elif k == "dense":
        M, H, XR, QL, NQ, E = c["rows"], c["H"], c["XR"], c["QL"], c["NQ"], c["E"]
        b16 = torch.bfloat16
        s["yr"], s["res"] = g.normal((M, H), 0.5), g.normal((M, H), 1.0, b16)
        s["n1"], s["n2"] = (1.0 + g.normal((H,), 0.1)).to(b16), (1.0 + g.normal((H,), 0.1)).to(b16)
        o = s["out"] = dict(res1=_empty(M, H, dtype=b16), xn1=_empty(M, H, dtype=b16), xg=_empty(M, XR, dtype=b16), q=_empty(M, NQ, dtype=b16),
                            part=_empty(M, H), res2=_empty(M, H, dtype=b16), xn2=_empty(M, H, dtype=b16), logits=_empty(M, E))
        s["xproj"] = [dict(_dense(g, "bf16", XR, H), n=XR, y=o["xg"], ldy=XR)]
        s["qb"] = [dict(_dense(g, c["fmt"], NQ, QL), n=NQ, y=o["q"], ldy=NQ)]
        s["oproj"] = [dict(_dense(g, c["fmt"], H, NQ), n=H, y=o["part"], ldy=H)]
        s["router"] = [dict(_dense(g, "bf16", E, H), n=E, y=o["logits"], ldy=E)]
    elif k == "moe":
        M, H = c["M"], c["H"]
        pool, desc = _pool(g, c)
        s["keep"] = [pool, desc, [_shared(g, c) for _ in range(STEP_LAYERS)]]
        s["layers"] = [_layer_w(c, pool, desc, sh) for sh in s["keep"][2]]
        s["x"] = g.normal((STEP_LAYERS, M, H), 1.0, torch.bfloat16)
        s["logits"] = g.normal((STEP_LAYERS, M, c["E"]), 1.0)
        s["yr"] = _empty(STEP_LAYERS, M, H)
        s["ys"] = _empty(STEP_LAYERS, M, H) if c["shared"] else None
        s["ws"] = torch.zeros(lib.decode_ws_bytes(s["layers"][0]), dtype=torch.uint8, device="cuda")
    elif k == "dsk":
        M, H = c["M"], c["H"]
        s["keep"], s["weights"] = _dsk_weights(g, c)
        rows = [_act_quant32(g.normal((M, H), 1.5)) for _ in range(STEP_LAYERS)]
        s["xq"], s["xs"] = [r[0] for r in rows], [r[1] for r in rows]
        s["logits"] = g.normal((STEP_LAYERS, M, c["E"]), 1.0)
        s["y"] = _empty(STEP_LAYERS, M, H)
        s["idx"], s["w"] = _empty(STEP_LAYERS, M, c["topk"], dtype=torch.int32), _empty(STEP_LAYERS, M, c["topk"])
        s["ws"] = torch.zeros(lib.dsk_ws_bytes(H, c["I"]), dtype=torch.uint8, device="cuda")
    elif k in ("prefill", "dsk_prefill"):
        T, H = c["T"], c["H"]
        s["logits"] = _zipf_logits(g, T, c["E"])
        s["idx"], s["w"] = _empty(T, c["topk"], dtype=torch.int32), _empty(T, c["topk"])
        if k == "prefill":
            pool, desc = _pool(g, c)
            sh = _shared(g, c)
            s["keep"], s["layer"] = [pool, desc, sh], _layer_w(c, pool, desc, sh)
            s["x"] = g.normal((T, H), 1.0, torch.bfloat16)
            s["yr"] = _empty(T, H)
            if c["shared"]:
                s["ys"], s["y"] = _empty(T, H), _empty(T, H, dtype=torch.bfloat16)
            s["ws"] = _empty(lib.prefill_ws_bytes(s["layer"], T), dtype=torch.uint8)
        else:
            s["keep"], s["weights"] = _dsk_weights(g, c)
            s["xq"], s["xs"] = _act_quant32(g.normal((T, H), 1.5))
            s["y"] = _empty(T, H)
            s["ws"] = _empty(lib.dsk_prefill_ws_bytes(H, c["I"], c["E"], c["topk"], T), dtype=torch.uint8)
    else:
        raise ValueError(k)
    return s


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "gemv":
        lib.gemv(s["x"], c["K"], c["rows"], c["K"], s["segs"], OUT[c["out"]], splitk=c["splitk"])
        return s["y"]
    if k == "dense":
        # the order of a decode layer's calls (dsgx10_amd/chain.py), without the MoE step at its end
        M, H, o = c["rows"], c["H"], s["out"]
        lib.add_norm(s["yr"], None, M, H, s["res"], o["res1"], s["n1"], 1e-5, o["xn1"])
        lib.gemv(o["xn1"], H, M, H, s["xproj"], abi.OUT_BF16, splitk=2)
        lib.gemv(o["xg"], c["XR"], M, c["QL"], s["qb"], abi.OUT_BF16)
        lib.gemv(o["q"], c["NQ"], M, c["NQ"], s["oproj"], abi.OUT_F32)
        lib.add_norm_gemv(o["part"], None, o["res1"], o["res2"], s["n2"], 1e-5, o["xn2"], M, H, s["router"], abi.OUT_F32, splitk=4)
        return o
    if k == "moe":
        for l, L in enumerate(s["layers"]):
            lib.moe_decode(L, s["x"][l], None, None, c["M"], s["ws"], s["yr"][l], s["ys"][l] if c["shared"] else None, logits=s["logits"][l],
                           route_scale=1.0 if c["fmt"] == "fp8" else 2.5, ysum=c["shared"])
        return [s["yr"], s["ys"]] if c["shared"] else [s["yr"]]
    if k == "dsk":
        for l in range(STEP_LAYERS):
            lib.dsk_moe_stacked(s["weights"], s["xq"][l], s["xs"][l], None, None, c["M"], s["ws"], s["y"][l], logits=s["logits"][l],
                                route_scale=1.5, idx_out=s["idx"][l], wts_out=s["w"][l])
        return [s["y"], s["idx"], s["w"]]
    if k == "prefill":
        lib.route(s["logits"], None, s["idx"], s["w"], route_scale=1.0 if c["fmt"] == "fp8" else 2.5)
        lib.moe_prefill(s["layer"], s["x"], s["idx"], s["w"], c["T"], s["ws"], s["yr"], s.get("ys"), shared=c["shared"], act_fp8=c["act_fp8"])
        if not c["shared"]:
            return [s["idx"], s["w"], s["yr"]]
        lib.finalize(s["yr"], s["ys"], c["T"] * c["H"], s["y"])
        return [s["idx"], s["w"], s["yr"], s["ys"], s["y"]]
    lib.route(s["logits"], None, s["idx"], s["w"], route_scale=1.5, score_fn=1)
    lib.dsk_moe_prefill(s["weights"], s["xq"], s["xs"], s["idx"], s["w"], c["T"], s["ws"], s["y"])
    return [s["idx"], s["w"], s["y"]]


# ---- what a pass cannot do without, and how far apart two correct ones may be ------------------------------------------------
def _dense_bytes(fmt, N, K):
    return {"fp8": N * K + (N + 127) // 128 * (K // 128) * 4, "int4": N * K // 2 + N * K // 16 + N * K // 64, "bf16": 2 * N * K}[fmt]


def work(case):
    c = case
    k = c["kind"]
    if k == "gemv":
        ncol = c["N"] // 2 if c["out"] == "swiglu" else c["N"]
        return {"bytes": _dense_bytes(c["fmt"], c["N"], c["K"]) + c["rows"] * (2 * c["K"] + (4 if c["out"] == "f32" else 2) * ncol),
                "flops": 2 * c["rows"] * c["N"] * c["K"]}
    if k == "dense":
        M, H, XR, QL, NQ, E = c["rows"], c["H"], c["XR"], c["QL"], c["NQ"], c["E"]
        values = XR * H + NQ * QL + H * NQ + E * H
        return {"bytes": _dense_bytes("bf16", XR, H) + _dense_bytes(c["fmt"], NQ, QL) + _dense_bytes(c["fmt"], H, NQ) + _dense_bytes("bf16", E, H) +
                M * (4 * H + 2 * H + 4 * 2 * H + 2 * XR + 2 * NQ + 4 * H + 4 * E), "flops": 2 * M * values}
    H, I, E, topk = c["H"], c["I"], c["E"], c["topk"]
    T, steps = (c["M"], STEP_LAYERS) if k in ("moe", "dsk") else (c["T"], 1)
    if steps > 1:  # the expected number of distinct experts of T rows: uniform picks, or Zipf's
        union = E * (1.0 - (1.0 - topk / E) ** T)
    else:
        p = [(r + 1.0) ** -ZIPF for r in range(E)]
        union = sum(1.0 - (1.0 - min(1.0, topk * v / sum(p))) ** T for v in p)
    if k in ("dsk", "dsk_prefill"):
        expert, shared, row = 3 * H * I * 17 // 32, 3 * H * I + 3 * H * I // 1024, H + H // 32 + 4 * H
    else:
        expert = sum(_dense_bytes(c["fmt"], N, K) for N, K in ((I, H), (I, H), (H, I)))
        shared = expert if c["fmt"] == "fp8" else 6 * H * I
        row = 2 * H + 4 * H + (4 * H if c["shared"] else 0) + (2 * H if c["shared"] and k == "prefill" else 0)
    sh = 1 if c["shared"] else 0
    return {"bytes": steps * (union * expert + sh * shared + T * (row + 4 * E)), "flops": steps * 6 * H * I * T * (topk + sh)}


def tolerance(case):
    """About four times what two orders of the sums give (K split over 1 and over 4 waves; the vector-unit and the MFMA decode
    kernels; prefill against decode; f64 sums): f32 sums 1e-7; where bf16 values are rounded on the way 3e-5 .. 2e-4 (a flipped
    rounding is one bf16 step of one value); where h is quantised to e4m3 on the way 1.2e-3 .. 1.9e-3."""
    c = case
    k = c["kind"]
    if k == "gemv":
        return {"rel": 1e-5, "max": 1e-4} if c["out"] == "f32" else {"rel": 5e-4, "max": 2e-2}
    if k == "dense":
        return {"rel": 5e-4, "max": 2e-2}
    if k == "moe":
        return {"rel": 2e-4, "max": 5e-3}
    if k == "prefill":
        return {"rel": 8e-3, "max": 0.15} if c["act_fp8"] else {"rel": 1e-3, "max": 2e-2}
    return {"rel": 5e-3, "max": 5e-2}


# ---- the same outputs in 64 bits ---------------------------------------------------------------------------------------------
def _up(s, b0, b1):
    return s.double().repeat_interleave(b0, 0).repeat_interleave(b1, 1)


def _deq(fmt, w, s=None, zp=None):
    """A stored matrix as the f64 values its format defines (INT4: W = bf16((u - u_z) s), the checkpoints' own rounding)"""
    if fmt == "fp8":
        return w.view(torch.float8_e4m3fn).double() * _up(s, 128, 128)[:w.shape[0]]
    if fmt == "fp8e":
        return w.view(torch.float8_e4m3fn).double() * _up(torch.exp2(s.double() - 127.0), 32, 32)
    if fmt == "int4":
        sh = torch.arange(8, device=w.device, dtype=torch.int32) * 4
        u = ((w[..., None] >> sh) & 15).flatten(-2).double()
        z = ((zp[:, None, :] >> sh[None, :, None]) & 15).flatten(0, 1)
        return ((u - _up(z, 1, 32)) * _up(s, 1, 32)).to(torch.bfloat16).double()
    if fmt == "mxfp4":
        val = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], device=w.device, dtype=torch.float64)
        code = torch.stack([w & 15, w >> 4], -1).flatten(-2).long()
        v = val[code & 7] * (1.0 - 2.0 * (code >> 3))
        return v * _up(torch.exp2(s.double() - 127.0), 1, 32)
    return w.double()


def _experts(c, s):
    """e -> (gate, up, down) in f64"""
    H, I = c["H"], c["I"]
    if c["kind"] in ("dsk", "dsk_prefill"):
        t = s["keep"]
        return lambda e: tuple(_deq("mxfp4", t["w" + n][e], t["s" + n][e]) for n in "132")
    pool, fmt = s["keep"][0], c["fmt"]

    def get(e):
        at, out = 0, []
        for N, K in ((I, H), (I, H), (H, I)):
            o, parts = at, []
            for shape, dt in {"fp8": [((N, K), torch.uint8), ((N // 128, K // 128), torch.float32)], "bf16": [((N, K), torch.bfloat16)],
                              "int4": [((N, K // 8), torch.int32), ((N, K // 32), torch.bfloat16), ((N // 8, K // 32), torch.int32)]}[fmt]:
                n = math.prod(shape) * dt.itemsize
                parts.append(pool[e, o:o + n].view(dt).view(shape))
                o += _al256(n)
            out.append(_deq(fmt, *parts))
            at += mat_bytes(FMT[fmt], N, K)
        return out
    return get


def _shared64(c, sh):
    if c["kind"] in ("dsk", "dsk_prefill"):
        return tuple(_deq("fp8e", sh["sh_w" + n], sh["sh_s" + n]) for n in "132")
    if c["fmt"] == "fp8":
        return tuple(_deq("fp8", q, sc) for q, sc in sh)
    return sh[0][0::2].double(), sh[0][1::2].double(), sh[1].double()


def _route64(logits, topk, scale, softplus):
    l = logits.double()
    key = torch.nn.functional.softplus(l).sqrt() if softplus else torch.sigmoid(l)
    v, idx = key.topk(topk, dim=-1)
    return idx, v / v.sum(-1, keepdim=True) * scale


def _mlp(x, w, limit):
    g, u = x @ w[0].T, x @ w[1].T
    if limit:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return (torch.nn.functional.silu(g) * u) @ w[2].T


def _moe64(c, x, idx, w, experts, shared, limit=None):
    """x f64 [T][H] -> the picks' weighted sum, the shared expert's rows"""
    y = torch.zeros_like(x)
    for e in idx.unique().tolist():
        r, k = (idx == e).nonzero(as_tuple=True)
        y[r] += _mlp(x[r], experts(e), limit) * w[r, k, None]
    return y, _mlp(x, shared, limit) if shared is not None else None


def exact(case, seed):
    c, s = case, prepare(case, seed)
    k = c["kind"]
    mat = lambda segs: _deq(c["fmt"] if segs[0]["fmt"] == FMT[c["fmt"]] else "bf16", segs[0]["w"], segs[0].get("s"), segs[0].get("zp"))
    if k == "gemv":
        y = s["x"].double() @ mat(s["segs"]).T
        return torch.nn.functional.silu(y[:, 0::2]) * y[:, 1::2] if c["out"] == "swiglu" else y
    if k == "dense":
        norm = lambda h, w: h * torch.rsqrt((h * h).mean(-1, keepdim=True) + 1e-5) * w.double()
        o = {"res1": s["res"].double() + s["yr"].double()}
        o["xn1"] = norm(o["res1"], s["n1"])
        o["xg"] = o["xn1"] @ mat(s["xproj"]).T
        o["q"] = o["xg"][:, :c["QL"]] @ mat(s["qb"]).T
        o["part"] = o["q"] @ mat(s["oproj"]).T
        o["res2"] = o["res1"] + o["part"]
        o["xn2"] = norm(o["res2"], s["n2"])
        o["logits"] = o["xn2"] @ mat(s["router"]).T
        return {n: o[n] for n in s["out"]}
    dsk = k in ("dsk", "dsk_prefill")
    scale = 1.5 if dsk else 1.0 if c["fmt"] == "fp8" else 2.5
    layers = range(STEP_LAYERS) if k in ("moe", "dsk") else [None]
    at = lambda v, l: v if l is None else v[l]
    res = []
    for l in layers:
        idx, w = _route64(at(s["logits"], l), c["topk"], scale, dsk)
        if dsk:
            x = at(s["xq"], l).view(torch.float8_e4m3fn).double() * _up(torch.exp2(at(s["xs"], l).double() - 127.0), 1, 32)
        else:
            x = at(s["x"], l).double()
        sh = None if not c["shared"] else s["keep"] if dsk else at(s["keep"][2], l)
        y, ys = _moe64(c, x, idx, w, _experts(c, s), _shared64(c, sh) if c["shared"] else None, 10.0 if dsk else None)
        res.append((w, y, ys))
    w, y, ys = [torch.stack(v) if v[0] is not None else None for v in zip(*res)]
    both = y + ys if ys is not None else y
    if k == "moe":
        return [both, ys] if c["shared"] else [both]
    if k == "dsk":
        return [both, None, w]
    if dsk:
        return [None, w[0], both[0]]
    return [None, w[0], y[0], ys[0], both[0]] if c["shared"] else [None, w[0], y[0]]
