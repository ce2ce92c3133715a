"""The work that a program built on this framework has it do, as cases that a timing program can run.

A case is one call (or one chain of calls) of h3metal_amd.ops on buffers of one device context, the way a diffusion
transformer, its text encoder, its vision tower and its autoencoder make them. `listed()` holds the fixed cases,
`draw()` makes more of the same ranges, `prepare()` makes a case's inputs and buffers on the GPU, `run()` is one
pass, `exact()` the same outputs in 64 bits by plain torch.
"""

import math

import torch

from h3metal_amd import ops
from h3metal_amd.gpu import Gpu

DEV = "cuda"
HD_OUTLIERS, OUTLIER = 4, 20.0  # channels of a head that are larger, and by how much (the int8 benchmark recipe)
EPS = 1e-6


# -- the cases ------------------------------------------------------------------------------------------------------

def listed():
    return [
        # The smallest call: 4 heads over 256 rows. What counts is the latency of the call.
        dict(name="attn_256", op="attention", path="bf16", H=4, KVH=4, D=128, Lq=256, L=256, causal=False, seqs=1),
        # Joint text + image attention of a 1024 x 1024 image with padded text: 4096 image rows, 259 valid of 512
        # text rows (a ragged key count), 16-bit scores.
        dict(name="attn_1024_keys", op="attention", path="bf16", H=30, KVH=30, D=128, Lq=4608, L=4355, causal=False,
             seqs=1),
        # Joint attention of a 2048 x 2048 image with int8 scores: the headline call and the largest one here.
        dict(name="attn_2048_int8", op="attention", path="int8", H=32, KVH=32, D=128, Lq=16896, L=16896,
             causal=False, seqs=1),
        # The text encoder: causal, grouped heads, a prompt of 512 rows.
        dict(name="attn_text_causal", op="attention", path="f16", H=32, KVH=8, D=128, Lq=512, L=512, causal=True,
             seqs=1),
        # The vision tower: head dim 72 padded to 96, a ragged number of patches.
        dict(name="attn_vision_96", op="attention", path="f16", H=16, KVH=16, D=96, Lq=1037, L=1037, causal=False,
             seqs=1),
        # The autoencoder's batched tiles: 32 sequences of 4 heads with 64 channels, 256 rows each.
        dict(name="attn_tiles_64", op="attention", path="f16", H=128, KVH=128, D=64, Lq=256, L=256, causal=False,
             seqs=32),
        # The pre-pass in front of int8 attention at 2048 x 2048: RMS norm, rotary embedding, rotation, int8.
        dict(name="prepass_2048", op="prepass", M=16896, Hq=32, Hk=32, Hv=32, hd=128, rot=96, q8=True, norm=True),
        # The int8 producer in front of the MLP's second projection, gated, at 2048 x 2048.
        dict(name="rot_q8_gated", op="rot_q8", M=16896, D=4096, dtype="bf16", swiglu=True, half=False),
        # The int8 qkv projection at 2048 x 2048.
        dict(name="gemm_qkv_2048", op="gemm", fmt="q8", M=16896, N=12288, K=4096, epi=0, out="bf16", bias=False),
        # An unquantised qkv projection at 1024 x 1024 (24 heads).
        dict(name="gemm_bf16_1024", op="gemm", fmt="bf16", M=4608, N=9216, K=3072, epi=0, out="bf16", bias=False),
        # A projection of the text encoder: few rows, int8 weights, half activations.
        dict(name="gemm_text_h8", op="gemm", fmt="h8", M=300, N=4096, K=4096, epi=0, out="f16", bias=False),
        # The attention half of a transformer block at 1024 x 1024: qkv projection, pre-pass, int8 attention, row
        # quantisation, output projection into the gated residual.
        dict(name="block_1024", op="block", S=4608, H=32, hd=128, rot=96),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


LARGEST = 4.0 * 32 * 16896 * 16896 * 128  # operations of the largest listed case


def draw(rng):
    kind = rng.choice(["dit", "dit", "text", "vision", "tiles", "prepass", "rot_q8", "gemm", "gemm", "block"])
    if kind == "dit":
        H, path = rng.choice([4, 24, 30, 32]), rng.choice(["int8", "int8", "bf16", "f16"])
        Lq = _log(rng, 64, 16896)
        L = max(1, Lq - rng.randrange(0, min(481, Lq))) if rng.random() < 0.5 else Lq
        return dict(op="attention", path=path, H=H, KVH=H, D=128, Lq=Lq, L=L, causal=False, seqs=1)
    if kind == "text":
        H = rng.choice([8, 16, 32])
        S = _log(rng, 16, 2048)
        return dict(op="attention", path=rng.choice(["f16", "f16", "bf16"]), H=H, KVH=H // rng.choice([2, 4]), D=128,
                    Lq=S, L=S, causal=True, seqs=1)
    if kind == "vision":
        N = _log(rng, 64, 4096)
        return dict(op="attention", path=rng.choice(["f16", "bf16"]), H=16, KVH=16, D=96, Lq=N, L=N, causal=False,
                    seqs=1)
    if kind == "tiles":
        seqs, sh, N = _log(rng, 1, 64), rng.choice([2, 4, 8]), _log(rng, 40, 1024)
        return dict(op="attention", path=rng.choice(["f16", "bf16"]), H=seqs * sh, KVH=seqs * sh, D=64, Lq=N, L=N,
                    causal=False, seqs=seqs)
    if kind == "prepass":
        M, H, q8 = _log(rng, 32, 16896), rng.choice([8, 24, 30, 32]), rng.random() < 0.6
        kv = H if q8 or rng.random() < 0.5 else max(1, H // 4)
        return dict(op="prepass", M=M, Hq=H, Hk=kv, Hv=kv, hd=128, rot=rng.choice([96, 128]), q8=q8, norm=True)
    if kind == "rot_q8":
        return dict(op="rot_q8", M=_log(rng, 32, 16896), D=256 * _log(rng, 4, 56), dtype=rng.choice(["bf16", "f16"]),
                    swiglu=rng.random() < 0.5, half=rng.random() < 0.25)
    if kind == "gemm":
        fmt = rng.choice(["q8", "q8", "h8", "f16", "bf16"])
        while True:
            M, N, K = _log(rng, 16, 16896), 256 * _log(rng, 4, 48), 256 * _log(rng, 4, 40)
            if 2.0 * M * N * K <= 2.0 * 16896 * 12288 * 4096:
                break
        epi = rng.choice([0, 0, 1])
        return dict(op="gemm", fmt=fmt, M=M, N=N, K=K, epi=epi,
                    out="f32" if epi else "bf16" if fmt in ("q8", "bf16") else "f16", bias=rng.random() < 0.3)
    return dict(op="block", S=_log(rng, 256, 8192), H=rng.choice([24, 32]), hd=128, rot=96)


# -- buffers --------------------------------------------------------------------------------------------------------

_gpu = None


def gpu():
    """The program's device context."""
    global _gpu
    if _gpu is None:
        _gpu = Gpu()
    return _gpu


_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i8": torch.int8, "u8": torch.uint8}
_TYPESTR = {"f32": "<f4", "f16": "<f2", "bf16": "<i2", "i8": "|i1", "u8": "|u1"}


class _Device:
    """What torch makes a tensor from; it lives as long as that tensor's storage, and the buffer as long as it."""

    def __init__(self, ptr, t):
        self.buf = t.buf
        self.__cuda_array_interface__ = dict(shape=tuple(t.shape), typestr=_TYPESTR[t.dtype], data=(ptr, False),
                                             version=2)


def view(t):
    """A torch tensor over the device memory of a framework tensor."""
    from h3metal_amd.gpu import lib
    x = torch.as_tensor(_Device(lib().h3_buffer_device(t.buf.handle) + t.offset, t), device=DEV)
    return x.view(torch.bfloat16) if t.dtype == "bf16" else x


def empty(shape, dtype):
    return gpu().empty(shape, dtype)


def upload(x, dtype, rows=None):
    """`x` on the device; with `rows`, in the first of that many rows."""
    t = empty((rows or x.shape[0],) + tuple(x.shape[1:]), dtype)
    view(t)[:x.shape[0]].copy_(x.to(_TORCH[dtype]))
    return t


# -- inputs ---------------------------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _hadamard(n):
    h = torch.ones(1, 1, device=DEV)
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(n)


def _codes(x):
    """Per-row int8 codes and scales."""
    s = x.abs().amax(-1) / 127
    s = torch.where(s > 0, s, torch.ones_like(s))
    return torch.round(x / s[..., None]).to(torch.int8), s


def _attention_inputs(c, seed):
    g = _gen(seed)
    D = c["D"]
    q, k, v = _normal(g, c["H"], c["Lq"], D), _normal(g, c["KVH"], c["L"], D), _normal(g, c["KVH"], c["L"], D)
    if D == 96:  # 72 real channels
        for t in (q, k, v):
            t[..., 72:] = 0
    if c["path"] != "int8":
        return q.to(_TORCH[c["path"]]), k.to(_TORCH[c["path"]]), v.to(_TORCH[c["path"]]), None, None
    # outlier channels of each head, rotated, then rounded to int8 row by row
    rot = _hadamard(D) * torch.where(torch.rand(D, generator=g, device=DEV) < 0.5, -1.0, 1.0)[:, None]
    for t in (q, k):
        for h in range(t.shape[0]):
            t[h, :, torch.randperm(D, generator=g, device=DEV)[:HD_OUTLIERS]] *= OUTLIER
    (qi, qs), (ki, ks) = _codes(q @ rot), _codes(k @ rot)
    return qi, ki, v.to(torch.bfloat16), qs, ks


def _attention_scale(c):
    return (72 if c["D"] == 96 else c["D"]) ** -0.5


def _rope(S, rot, base=10000.0):
    f = base ** (-torch.arange(rot // 2, device=DEV, dtype=torch.float32) * 2 / rot)
    a = torch.arange(S, device=DEV, dtype=torch.float32)[:, None] * f
    return torch.cos(a), torch.sin(a)


def _prepass_inputs(c, seed):
    g = _gen(seed)
    n = c["Hq"] + c["Hk"] + c["Hv"]
    x = _normal(g, c["M"], n, c["hd"])
    boost = torch.ones(n, c["hd"], device=DEV)
    for h in range(c["Hq"] + c["Hk"]):
        boost[h, torch.randperm(c["hd"], generator=g, device=DEV)[:HD_OUTLIERS]] = OUTLIER
    x = (x * boost).to(torch.bfloat16).reshape(c["M"], n * c["hd"])
    wq, wk = (1 + 0.1 * _normal(g, c["hd"]) for _ in range(2))
    return x, wq, wk, *_rope(c["M"], c["rot"])


def _rot_inputs(c, seed):
    g = _gen(seed)
    return (2 * _normal(g, c["M"], (2 if c["swiglu"] else 1) * c["D"])).to(_TORCH[c["dtype"]])


def _weights(g, N, K):
    q = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    return q, torch.rand(N, generator=g, device=DEV) * 1e-4 + 1e-4


def _residual(g, M, N):
    """The residual stream, the rows' modality and the gate table (text rows, image rows)."""
    return (_normal(g, M, N), (torch.arange(M, device=DEV) >= max(1, M // 8)).to(torch.uint8),
            1 + 0.1 * _normal(g, 2, N))


def _gemm_inputs(c, seed):
    g = _gen(seed)
    M, N, K, fmt = c["M"], c["N"], c["K"], c["fmt"]
    d = {}
    if fmt == "q8":
        d["a"], d["sa"] = _codes(_normal(g, M, K))
    else:
        d["a"] = _normal(g, M, K).to(torch.bfloat16 if fmt == "bf16" else torch.float16)
    if fmt in ("q8", "h8"):
        d["w"], d["sw"] = _weights(g, N, K)
    else:
        d["w"] = (_normal(g, N, K) / math.sqrt(K)).to(_TORCH[fmt])
    if c["bias"]:
        d["bias"] = _normal(g, N)
    if c["epi"]:
        d["x"], d["rtype"], d["gate"] = _residual(g, M, N)
    return d


def _block_inputs(c, seed):
    g = _gen(seed)
    S, E = c["S"], c["H"] * c["hd"]
    a, sa = _codes(_normal(g, S, E))
    wqkv, swqkv = _weights(g, 3 * E, E)
    wo, swo = _weights(g, E, E)
    wq, wk = (1 + 0.1 * _normal(g, c["hd"]) for _ in range(2))
    x, rtype, gate = _residual(g, S, E)
    cos, sin = _rope(S, c["rot"])
    return dict(a=a, sa=sa, wqkv=wqkv, swqkv=swqkv, wo=wo, swo=swo, wq=wq, wk=wk, x=x, rtype=rtype, gate=gate, cos=cos,
                sin=sin)


def prepare(case, seed):
    c, op = case, case["op"]
    s = dict(case=c)
    if op == "attention":
        q, k, v, qs, ks = _attention_inputs(c, seed)
        t, vt = ("i8", "bf16") if c["path"] == "int8" else (c["path"], c["path"])
        s.update(q=upload(q, t), k=upload(k, t), v=upload(v, vt))
        if qs is not None:
            s.update(qs=upload(qs, "f32"), ks=upload(ks, "f32"))
        sh = c["H"] // c["seqs"]
        s["o"] = empty((c["seqs"] * c["Lq"], sh * c["D"]), vt)
        s["out"] = view(s["o"])
    elif op == "prepass":
        x, wq, wk, cos, sin = _prepass_inputs(c, seed)
        s.update(x=upload(x, "bf16"), wq=upload(wq, "f32"), wk=upload(wk, "f32"), cos=upload(cos, "f32"),
                 sin=upload(sin, "f32"))
        t = "i8" if c["q8"] else "bf16"
        for n, heads in (("Q", "Hq"), ("K", "Hk"), ("V", "Hv")):
            s[n] = empty((c[heads], c["M"], c["hd"]), "bf16" if n == "V" else t)
        s["out"] = [view(s[n]) for n in "QKV"]
        if c["q8"]:
            s.update(qs=empty((c["Hq"], c["M"]), "f32"), ks=empty((c["Hk"], c["M"]), "f32"))
            s["out"] += [view(s["qs"]), view(s["ks"])]
    elif op == "rot_q8":
        s["x"] = upload(_rot_inputs(c, seed), c["dtype"])
        s["o"] = empty((c["M"], c["D"]), "f16" if c["half"] else "i8")
        s["sa"] = None if c["half"] else empty((c["M"],), "f32")
        s["out"] = [view(s["o"])] + ([] if c["half"] else [view(s["sa"])])
    elif op == "gemm":
        d = _gemm_inputs(c, seed)
        at, wt = ops.GEMM_ACT[c["fmt"]], "i8" if c["fmt"] in ("q8", "h8") else c["fmt"]
        M, rows = c["M"], ops.pad_rows(c["M"], 64)  # row counts are padded to the default tile's height
        s["a"], s["sa"] = upload(d["a"], at, rows), upload(d["sa"], "f32", rows) if "sa" in d else None
        s["w"] = ops.QWeight(c["fmt"], upload(d["w"], wt), upload(d["sw"], "f32") if "sw" in d else None, c["N"],
                             c["K"], bias=upload(d["bias"], "f32") if "bias" in d else None)
        if c["epi"]:
            s.update(o=upload(d["x"], "f32", rows), rtype=upload(d["rtype"], "u8", rows), gate=upload(d["gate"], "f32"))
        else:
            s.update(o=empty((rows, c["N"]), c["out"]), rtype=None, gate=None)
        s["out"] = view(s["o"])[:M]
    else:
        d = _block_inputs(c, seed)
        S, H, hd, E = c["S"], c["H"], c["hd"], c["H"] * c["hd"]
        rows = ops.pad_rows(S, 64)
        s.update(a=upload(d["a"], "i8", rows), sa=upload(d["sa"], "f32", rows), rtype=upload(d["rtype"], "u8", rows),
                 x=upload(d["x"], "f32", rows))
        for n in ("wq", "wk", "cos", "sin", "gate"):
            s[n] = upload(d[n], "f32")
        s["wqkv"] = ops.QWeight("q8", upload(d["wqkv"], "i8"), upload(d["swqkv"], "f32"), 3 * E, E)
        s["wo"] = ops.QWeight("q8", upload(d["wo"], "i8"), upload(d["swo"], "f32"), E, E)
        s.update(qkv=empty((rows, 3 * E), "bf16"), Q=empty((H, S, hd), "i8"), K=empty((H, S, hd), "i8"),
                 V=empty((H, S, hd), "bf16"), qs=empty((H, S), "f32"), ks=empty((H, S), "f32"), o=empty((S, E), "bf16"),
                 o8=empty((rows, E), "i8"), so=empty((rows,), "f32"))
        s["out"] = [view(s["x"])[:S], view(s["o"])]
    torch.cuda.synchronize()
    return s


# -- one pass -------------------------------------------------------------------------------------------------------

def run(s):
    c, g = s["case"], gpu()
    op = c["op"]
    if op == "attention":
        more = dict(q_scale=s["qs"], k_scale=s["ks"]) if c["path"] == "int8" else {}
        if c["seqs"] > 1:
            more.update(seq_heads=c["H"] // c["seqs"], seq_rows=c["Lq"])
        ops.attention(g, s["q"], s["k"], s["v"], s["o"], Lq=c["Lq"], L=c["L"], H=c["H"], KVH=c["KVH"], D=c["D"],
                      q_rows=c["Lq"], k_rows=c["L"], scale=_attention_scale(c), causal=c["causal"], **more)
    elif op == "prepass":
        more = dict(q_scale=s["qs"], k_scale=s["ks"], qk_rot=True) if c["q8"] else {}
        ops.qk_norm_rope(g, s["x"], s["wq"], s["wk"], s["cos"], s["sin"], s["Q"], s["K"], s["V"], M=c["M"], Hq=c["Hq"],
                         Hk=c["Hk"], Hv=c["Hv"], hd=c["hd"], out_rows=c["M"], rot=c["rot"], eps=EPS, norm=c["norm"],
                         **more)
    elif op == "rot_q8":
        ops.rot_q8(g, s["x"], s["o"], s["sa"], c["M"], c["D"], swiglu=c["swiglu"], out_hr=c["half"])
    elif op == "gemm":
        ops.gemm(g, s["a"], s["w"], s["o"], c["M"], sa=s["sa"], epi=c["epi"], rtype=s["rtype"], gate=s["gate"])
    else:
        S, H, hd = c["S"], c["H"], c["hd"]
        ops.gemm(g, s["a"], s["wqkv"], s["qkv"], S, sa=s["sa"])
        ops.qk_norm_rope(g, s["qkv"], s["wq"], s["wk"], s["cos"], s["sin"], s["Q"], s["K"], s["V"], M=S, Hq=H, Hk=H,
                         Hv=H, hd=hd, out_rows=S, rot=c["rot"], eps=EPS, q_scale=s["qs"], k_scale=s["ks"], qk_rot=True)
        ops.attention(g, s["Q"], s["K"], s["V"], s["o"], Lq=S, L=S, H=H, KVH=H, D=hd, q_rows=S, k_rows=S,
                      scale=hd ** -0.5, q_scale=s["qs"], k_scale=s["ks"])
        ops.rot_q8(g, s["o"], s["o8"], s["so"], S, H * hd)
        ops.gemm(g, s["o8"], s["wo"], s["x"], S, sa=s["so"], epi=1, rtype=s["rtype"], gate=s["gate"])
    return s["out"]


# -- what a pass cannot do without ------------------------------------------------------------------------------------

def _attention_work(H, KVH, D, Lq, L, causal, qk_bytes):
    pairs = sum(min(L, i + 1) for i in range(Lq)) if causal else Lq * L
    rows = H * Lq + KVH * L
    return rows * D * (qk_bytes + 2) + (rows * 4 if qk_bytes == 1 else 0), 4.0 * H * pairs * D


def _prepass_bytes(M, Hq, Hk, Hv, hd, rot, q8):
    out = (Hq + Hk) * (hd + 4) if q8 else (Hq + Hk) * hd * 2
    return M * ((Hq + Hk + Hv) * hd * 2 + out + Hv * hd * 2) + M * rot * 4


def _gemm_work(M, N, K, a, w, out, epi):
    return M * K * a + N * K * w + M * N * out * (2 if epi else 1), 2.0 * M * N * K


def work(case):
    c, op = case, case["op"]
    if op == "attention":
        b, f = _attention_work(c["H"], c["KVH"], c["D"], c["Lq"], c["L"], c["causal"], 1 if c["path"] == "int8" else 2)
    elif op == "prepass":
        b, f = _prepass_bytes(c["M"], c["Hq"], c["Hk"], c["Hv"], c["hd"], c["rot"], c["q8"]), 0.0
    elif op == "rot_q8":
        b = c["M"] * c["D"] * ((4 if c["swiglu"] else 2) + (2 if c["half"] else 1)) + (0 if c["half"] else 4 * c["M"])
        f = 0.0
    elif op == "gemm":
        b, f = _gemm_work(c["M"], c["N"], c["K"], 1 if c["fmt"] == "q8" else 2, 1 if c["fmt"] in ("q8", "h8") else 2,
                          4 if c["out"] == "f32" else 2, c["epi"])
    else:
        S, H, hd, E = c["S"], c["H"], c["hd"], c["H"] * c["hd"]
        parts = [_gemm_work(S, 3 * E, E, 1, 1, 2, 0), (_prepass_bytes(S, H, H, H, hd, c["rot"], True), 0.0),
                 _attention_work(H, H, hd, S, S, False, 1), (S * E * 3 + 4 * S, 0.0), _gemm_work(S, E, E, 1, 1, 4, 1)]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    return dict(bytes=float(b), flops=float(f))


def tolerance(case):
    """About four times the distance from the 64-bit result that the rounding of the stored types alone leaves (a
    16-bit result is 1.7e-3 away in bf16 and 2.1e-4 in f16; attention also rounds its weights). Codes are the same
    but for the gated rows, whose exponential may round differently."""
    op = case["op"]
    if op == "attention":
        return {"rel": 1.2e-3 if case["path"] == "f16" else 1e-2}
    if op == "prepass":
        return {"rel": 1e-6} if case["q8"] else {"rel": 7e-3}
    if op == "rot_q8":
        return {"rel": 1e-3 if case["half"] else 1e-6, "differ": 2e-4 if case["swiglu"] else 0.0}
    if op == "gemm":
        return {"rel": {"bf16": 7e-3, "f16": 1e-3, "f32": 1e-6 if case["fmt"] == "q8" else 1e-5}[case["out"]]}
    return {"rel": 1e-2}


# -- the same in 64 bits ----------------------------------------------------------------------------------------------

def _exact_attention(q, k, v, scale, causal=False, seqs=1):
    """q [H][Lq][D], k and v [KVH][L][D] in float64 -> [seqs * Lq][H / seqs * D]."""
    H, Lq, D = q.shape
    per, sh = H // k.shape[0], H // seqs
    out = torch.empty(seqs * Lq, sh * D, device=DEV, dtype=torch.float64)
    chunk = max(1, (1 << 26) // k.shape[1])
    for h in range(H):
        kt, vh = k[h // per].t().contiguous(), v[h // per]
        for r in range(0, Lq, chunk):
            x = (q[h, r:r + chunk] @ kt) * scale
            if causal:
                rows = torch.arange(r, r + x.shape[0], device=DEV)[:, None]
                x.masked_fill_(torch.arange(x.shape[1], device=DEV)[None] > rows, float("-inf"))
            x = torch.softmax(x, -1)
            r0 = (h // sh) * Lq + r
            out[r0:r0 + x.shape[0], (h % sh) * D:(h % sh + 1) * D] = x @ vh
    return out


def _exact_prepass(x, wq, wk, cos, sin, Hq, Hk, Hv, hd, rot, rotate):
    """Rotated queries and keys [heads][M][hd] in float64 before any rounding, and the values."""
    M = x.shape[0]
    x = x.double().reshape(M, Hq + Hk + Hv, hd).transpose(0, 1)
    out = []
    for part, w in ((x[:Hq], wq), (x[Hq:Hq + Hk], wk)):
        t = part / torch.sqrt((part * part).mean(-1, keepdim=True) + EPS) * w.double()
        a, b, c, s = t[..., :rot // 2], t[..., rot // 2:rot], cos.double(), sin.double()
        t = torch.cat([a * c - b * s, b * c + a * s, t[..., rot:]], -1)
        if rotate:
            sign = [-1.0 if bin((i * 0x2545F491) & 0xFFFFFFFF).count("1") & 1 else 1.0 for i in range(hd)]
            t = (t * torch.tensor(sign, device=DEV, dtype=torch.float64)) @ (_hadamard(hd).double() * math.sqrt(hd))
            t = t / math.sqrt(hd)
        out.append(t)
    return out[0], out[1], x[Hq + Hk:]


def _exact_rows(x):
    """Rows in float64 times the 256-point Walsh-Hadamard matrix, block by block."""
    return (x.reshape(x.shape[0], -1, 256) @ _hadamard(256).double()).reshape(x.shape)


def _exact_codes(x):
    s = x.abs().amax(-1) / 127
    s = torch.where(s > 0, s, torch.ones_like(s))
    return torch.round(x / s[..., None]), s


def _rows_product(a, w, chunk=2048):
    wt = w.double().t().contiguous()
    return torch.cat([a[r:r + chunk].double() @ wt for r in range(0, a.shape[0], chunk)])


def exact(case, seed):
    c, op = case, case["op"]
    if op == "attention":
        q, k, v, qs, ks = _attention_inputs(c, seed)
        q, k = q.double(), k.double()
        if qs is not None:
            q, k = q * qs.double()[..., None], k * ks.double()[..., None]
        return _exact_attention(q, k, v.double(), _attention_scale(c), c["causal"], c["seqs"])
    if op == "prepass":
        x, wq, wk, cos, sin = _prepass_inputs(c, seed)
        q, k, v = _exact_prepass(x, wq, wk, cos, sin, c["Hq"], c["Hk"], c["Hv"], c["hd"], c["rot"], c["q8"])
        if not c["q8"]:
            return [q, k, v.contiguous()]
        return [None, None, v.contiguous(), q.abs().amax(-1) / 127, k.abs().amax(-1) / 127]
    if op == "rot_q8":
        x = _rot_inputs(c, seed).double()
        if c["swiglu"]:
            x = x[:, :c["D"]] * torch.nn.functional.silu(x[:, c["D"]:])
        x = _exact_rows(x)
        return [x] if c["half"] else [None, _exact_codes(x)[1]]
    if op == "gemm":
        d = _gemm_inputs(c, seed)
        v = _rows_product(d["a"], d["w"])
        if "sa" in d:
            v *= d["sa"].double()[:, None]
        if "sw" in d:
            v *= d["sw"].double()
        if "bias" in d:
            v += d["bias"].double()
        return d["x"].double() + d["gate"].double()[d["rtype"].long()] * v if c["epi"] else v
    d = _block_inputs(c, seed)
    S, H, hd = c["S"], c["H"], c["hd"]
    qkv = _rows_product(d["a"], d["wqkv"]) * d["sa"].double()[:, None] * d["swqkv"].double()
    q, k, v = _exact_prepass(qkv.to(torch.bfloat16), d["wq"], d["wk"], d["cos"], d["sin"], H, H, H, hd, c["rot"], True)
    (qi, qs), (ki, ks) = _exact_codes(q), _exact_codes(k)
    o = _exact_attention(qi * qs[..., None], ki * ks[..., None], v, hd ** -0.5)
    oi, so = _exact_codes(_exact_rows(o.to(torch.bfloat16).double()))
    v = _rows_product(oi, d["wo"]) * so[:, None] * d["swo"].double()
    return [d["x"].double() + d["gate"].double()[d["rtype"].long()] * v, o]
