"""Short attention calls: the 32-row tiles whose waves split the keys (csrc/attention_small.hip; SMALL names them) and
what the size chooses, against float64 attention and against the 256-row tiles, whole (SPLIT=0) and with a split last
round (GROUPS=1), on the same inputs: every head dim, score type and
output type, causal masks with offsets, grouped heads, batched sequences, ragged query and key counts around the
32-key blocks and the four waves, rows reserved past the valid ones holding NaN, and rows that see no key. The
max-abs tolerances are the attention tests' own, 5e-3 with half values and 2e-2 with bf16 (the rounding of P and of the
output); the mean-abs one is 2^-9, half a bf16 ulp of a unit value, since over few keys the outputs are as large as
the values. Both kernels round P with a maximum of their own, so they agree to that."""

import numpy as np
import pytest

from h3metal_amd import ops
from h3metal_amd.gpu import GpuError
from oracle import attention as oa
from oracle.bf16 import from_bf16, to_bf16

pytestmark = pytest.mark.gpu

CASES = [  # path, D, H, KVH, Lq, L, causal, offset, sequences, output
    ("f16", 128, 2, 2, 1, 1, False, 0, 1, "f16"), ("bf16", 128, 4, 2, 31, 33, False, 0, 1, "f32"),
    ("int8", 128, 3, 3, 33, 127, False, 0, 1, "bf16"), ("f16", 128, 2, 1, 129, 129, True, 0, 1, "f16"),
    ("int8", 128, 4, 2, 70, 95, True, 25, 1, "f32"), ("bf16", 128, 8, 2, 200, 160, True, -40, 1, "bf16"),
    ("f16", 96, 2, 2, 65, 97, False, 0, 1, "bf16"), ("bf16", 96, 3, 1, 64, 64, True, 0, 1, "f16"),
    ("int8", 96, 2, 2, 40, 300, False, 0, 1, "f32"), ("f16", 64, 6, 6, 40, 40, False, 0, 3, "f16"),
    ("bf16", 64, 4, 4, 257, 31, False, 0, 2, "bf16"), ("int8", 64, 4, 2, 128, 128, True, 0, 1, "f16"),
    ("f16", 64, 128, 128, 256, 256, False, 0, 32, "f16"), ("bf16", 64, 8, 4, 100, 200, False, 0, 2, "f32"),
    ("int8", 64, 6, 6, 33, 129, False, 0, 3, "bf16"), ("f16", 64, 3, 3, 97, 130, True, 30, 1, "f32"),
    ("f16", 96, 16, 16, 1500, 1500, False, 0, 1, "f16"), ("int8", 96, 3, 3, 129, 200, True, 71, 1, "bf16"),
    ("bf16", 96, 4, 2, 65, 300, False, 0, 2, "bf16"),
]


def rows(gpu, x, n, dtype, fill=None):
    """x [heads][rows][..] in tensors of n rows per head; the rows past x's hold `fill`."""
    full = np.zeros((x.shape[0], n) + x.shape[2:], x.dtype)
    if fill is not None:
        full[:] = fill
    full[:, :x.shape[1]] = x
    t = gpu.empty(full.shape, dtype)
    t.write(full)
    return t


@pytest.mark.parametrize("path,D,H,KVH,Lq,L,causal,off,seqs,out", CASES)
def test_short_calls(gpu, path, D, H, KVH, Lq, L, causal, off, seqs, out):
    rng = np.random.default_rng(Lq * 1000 + L + D)
    print(f"[short] {path} D={D} H={H}/{KVH} Lq={Lq} L={L} causal={causal} off={off} seqs={seqs}", flush=True)
    q, k, v = (rng.standard_normal((n, r, D)).astype(np.float32) for n, r in ((H, Lq), (KVH, L), (KVH, L)))
    vt = "f16" if path == "f16" else "bf16"
    bits = (lambda x: x.astype(np.float16)) if vt == "f16" else to_bf16
    val = (lambda x: x.astype(np.float64)) if vt == "f16" else (lambda x: from_bf16(x).astype(np.float64))
    nan = np.float16(np.nan) if vt == "f16" else np.uint16(0x7FC0)
    qr, kr = Lq + 5, L + 9
    extra = {}
    if path == "int8":
        q[..., :2] *= 8
        (qs, ks) = (np.abs(x).max(-1) / 127 for x in (q, k))
        qi, ki = (np.rint(x / s[..., None]).astype(np.int8) for x, s in ((q, qs), (k, ks)))
        qs, ks = qs.astype(np.float32), ks.astype(np.float32)
        Q, K = rows(gpu, qi, qr, "i8", 127), rows(gpu, ki, kr, "i8", 127)
        extra = dict(q_scale=rows(gpu, qs, qr, "f32", np.nan), k_scale=rows(gpu, ks, kr, "f32", np.nan))
        qv, kv = qi * qs[..., None].astype(np.float64), ki * ks[..., None].astype(np.float64)
    else:
        qb, kb = bits(q), bits(k)
        Q, K, qv, kv = rows(gpu, qb, qr, vt, nan), rows(gpu, kb, kr, vt, nan), val(qb), val(kb)
    vb = bits(v)
    V = rows(gpu, vb, kr, vt, nan)
    sh, seq_rows = H // seqs, Lq + 3
    with np.errstate(invalid="ignore"):
        want = oa.ref_attention(qv, kv, val(vb), D ** -0.5, causal=causal, off=off)
    want = np.nan_to_num(want.reshape(Lq, H, D))  # a row that sees no key is zero
    outs = []
    for variant in ({}, {"SPLIT": 0}, {"GROUPS": 1}, {"SMALL": 1}, *([{"SMALL": 2}] if D == 96 else [])):
        O = gpu.empty((seqs * seq_rows, sh * D), out)
        ops.attention(gpu, Q, K, V, O, Lq=Lq, L=L, H=H, KVH=KVH, D=D, q_rows=qr, k_rows=kr, scale=D ** -0.5,
                      causal=causal, causal_off=off, seq_heads=sh, seq_rows=seq_rows, **extra, **variant)
        gpu.wait()
        o = O.numpy()
        o = (from_bf16(o) if out == "bf16" else o).astype(np.float64).reshape(seqs, seq_rows, sh, D)
        assert (o[:, Lq:] == 0).all()
        got = o[:, :Lq].transpose(1, 0, 2, 3).reshape(Lq, H, D)
        err = np.abs(got - want)
        assert np.isfinite(got).all(), variant
        outs.append(got)
        assert err.max() < (5e-3 if path == "f16" and out != "bf16" else 2e-2) and err.mean() < 2 ** -9, (variant, err.max())
    if D == 96:  # two query tiles per workgroup: each row's keys, waves and merge are those of one
        assert np.array_equal(outs[4], outs[3])


def test_small_macro_refusals(gpu):
    """SMALL is 1, or 2 at head dim 96, and names a kernel: not beside SPLIT=0 or GROUPS=1, nor for the scores hook where
    that runs another one."""
    for fn, m in (("attention", dict(HD=128, SMALL=2)), ("attention", dict(HD=96, SMALL=3)),
                  ("attention", dict(HD=64, SMALL=-1)), ("attention", dict(HD=128, SMALL=1, SPLIT=0)),
                  ("attention", dict(HD=128, SMALL=1, GROUPS=1)), ("attention_scores", dict(HD=64, SMALL=1)),
                  ("attention_scores", dict(HD=128, SMALL=1, CAUSAL=1))):
        with pytest.raises(GpuError, match="SMALL"):
            gpu.kernel("attention", fn, **m)


@pytest.mark.parametrize("path,D,H,Lq,L", [("int8", 128, 4, 32, 20000), ("bf16", 128, 1, 200, 20000),
                                           ("f16", 64, 16, 1, 8000), ("int8", 96, 4, 32, 8000)])
def test_long_keys_for_few_queries(gpu, path, D, H, Lq, L):
    """Few query rows against many keys leave a workgroup of the small tiles a long chain of key blocks (43 -> 163 us
    at int8, 4 heads, 32 x 32 768): these calls split the keys of 256-row tiles over workgroups, so that they are
    GROUPS=1's, bit for bit."""
    rng = np.random.default_rng(L)
    print(f"[long keys] {path} D={D} H={H} Lq={Lq} L={L}", flush=True)
    vt = "f16" if path == "f16" else "bf16"
    q, k, v = (rng.standard_normal((H, r, D), dtype=np.float32) for r in (Lq, L, L))
    bits = (lambda x: x.astype(np.float16)) if vt == "f16" else to_bf16
    V, extra = gpu.upload(bits(v), vt), {}
    if path == "int8":
        Q, K = (gpu.upload(np.rint(x * 30).clip(-127, 127).astype(np.int8)) for x in (q, k))
        extra = dict(q_scale=gpu.upload(np.full((H, Lq), 1 / 30, np.float32)),
                     k_scale=gpu.upload(np.full((H, L), 1 / 30, np.float32)))
    else:
        Q, K = (gpu.upload(bits(x), vt) for x in (q, k))
    outs = []
    for variant in ({}, {"GROUPS": 1}):
        O = gpu.empty((Lq, H * D), "f32")
        ops.attention(gpu, Q, K, V, O, Lq=Lq, L=L, H=H, KVH=H, D=D, q_rows=Lq, k_rows=L, scale=D ** -0.5, **extra,
                      **variant)
        gpu.wait()
        outs.append(O.numpy())
    assert np.abs(outs[0]).max() > 0 and np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
