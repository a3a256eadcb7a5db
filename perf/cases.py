"""Performance cases of the framework: what its users have it do, over the sizes they do it at.

Five kinds of call make up a model served with int8 attention and GGUF k-quant weights:

  prefill   `attn_int8_fwd` on fp16/bf16 Q/K/V (int8 QK^T, or full W8A8 with `int8_pv`)
  build     `quantize_kv_cache`: a prompt's K/V into the contiguous int8 cache
  append    `quantize_kv_write_paged`: one new token per sequence into the paged int8 cache
  decode    one query token per sequence against a cache: contiguous with fp16 or int8 V,
            paged int8, paged int8-K / 3-bit-V
  linear    `linear_q4k` / `linear_q5k` / `linear_q6k` on native GGUF bytes, M tokens

`listed()` holds the workloads of this repository's benchmark and typical ones around them;
`draw` samples the ranges that they stand for. A case is a dict of plain values.
"""
from __future__ import annotations

import math
import random

import torch

import superl8_amd as sl8
from superl8_amd import _C
from superl8_amd.quant.lloydmax import gaussian_codebook

DEV = "cuda" if torch.cuda.is_available() else "cpu"
LOG2E = math.log2(math.e)
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
BLOCK_BYTES = {"q4k": 144, "q5k": 176, "q6k": 210}
LINEAR = {"q4k": sl8.linear_q4k, "q5k": sl8.linear_q5k, "q6k": sl8.linear_q6k}


def _prefill(B, Hq, Hkv, M, N, D, causal=True, dtype="fp16", window=-1, int8_pv=False):
    return dict(kind="prefill", B=B, Hq=Hq, Hkv=Hkv, M=M, N=N, D=D, causal=causal, dtype=dtype,
                window=window, int8_pv=int8_pv)


def _decode(cache, B, Hq, Hkv, N, D=128, block=0, splits=0, rotate=False):
    return dict(kind="decode", cache=cache, B=B, Hq=Hq, Hkv=Hkv, N=N, D=D, block=block,
                splits=splits, rotate=rotate)


def _linear(fmt, M, N, K, dtype="fp16", bias=False):
    return dict(kind="linear", fmt=fmt, M=M, N=N, K=K, dtype=dtype, bias=bias)


def listed() -> list[dict]:
    return [
        # a short prompt on a small model: launches and latency count
        dict(name="prefill_512", **_prefill(1, 8, 8, 512, 512, 64)),
        # the flagship: a 4k prompt of a GQA model, prologue and outlier gate included
        dict(name="prefill_4k", **_prefill(1, 32, 8, 4096, 4096, 128)),
        # chunked prefill of a bf16 model: an odd-sized chunk behind a cached prefix
        dict(name="prefill_chunk_bf16", **_prefill(1, 32, 8, 1000, 6121, 128, dtype="bf16")),
        # full W8A8 with outlier channels, head dim 256: the largest call
        dict(name="w8a8_8k", **_prefill(2, 16, 2, 8192, 8192, 256, int8_pv=True)),
        # a 16k prompt's K/V quantised once for decoding
        dict(name="build_16k", kind="build", B=1, Hkv=8, N=16384, D=128, dtype="fp16", rotate=False),
        # the new tokens of a batch of 32 written into the paged cache: the smallest call
        dict(name="append_32", kind="append", B=32, Hkv=8, D=128, block=16, rotate=True),
        # long-context decode of a batch, int8 K and fp16 V
        dict(name="decode_32k", **_decode("k8", 16, 32, 8, 32768, splits=16)),
        # serving: sequences of mixed lengths in 16-token blocks, int8 K and V
        dict(name="decode_paged_mixed", **_decode("paged", 32, 32, 8, 8192, block=16, rotate=True)),
        # the same with 3-bit Lloyd-Max V
        dict(name="decode_k8v3_mixed", **_decode("k8v3", 16, 32, 8, 16384, block=16, rotate=True)),
        # one token through the up projection of an MLP
        dict(name="linear_q4k_m1", **_linear("q4k", 1, 17408, 5120)),
        # a decode batch through the down projection, bf16 activations
        dict(name="linear_q6k_m8", **_linear("q6k", 8, 5120, 17408, dtype="bf16")),
        # a prompt chunk through the up projection
        dict(name="linear_q4k_m512", **_linear("q4k", 512, 17408, 5120)),
    ]


def _log(rng: random.Random, lo: float, hi: float) -> int:
    return max(int(lo), min(int(hi), round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _heads(rng: random.Random) -> tuple[int, int]:
    hkv = rng.choice([2, 4, 8])
    return hkv * rng.choice([1, 2, 4, 8] if hkv < 8 else [1, 2, 4]), hkv


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["prefill", "prefill", "w8a8", "build", "append", "decode", "decode",
                       "decode", "linear", "linear", "linear", "linear"])
    if kind == "prefill":
        if rng.random() < 0.2:  # a vision tower: head dims 72 / 80, no mask
            h = rng.choice([8, 16])
            S = _log(rng, 196, 4096)
            return _prefill(rng.choice([1, 2, 4]), h, h, S, S, rng.choice([72, 80]), causal=False,
                            dtype=rng.choice(["fp16", "bf16"]))
        hq, hkv = _heads(rng)
        M = _log(rng, 64, 6000)
        N = M + (_log(rng, 64, 12000) if rng.random() < 0.5 else 0)
        causal = rng.random() < 0.85
        window = _log(rng, 512, 4096) if causal and rng.random() < 0.2 else -1
        return _prefill(1 if M * N > 4 << 20 else rng.choice([1, 2]), hq, hkv, M, N,
                        rng.choice([64, 128, 128]), causal=causal,
                        dtype=rng.choice(["fp16", "bf16"]), window=window)
    if kind == "w8a8":
        hq, hkv = _heads(rng)
        S = _log(rng, 256, 5000)
        return _prefill(1, hq, hkv, S, S, rng.choice([64, 128, 256]), causal=rng.random() < 0.8,
                        dtype=rng.choice(["fp16", "bf16"]), int8_pv=True)
    if kind == "build":
        return dict(kind="build", B=rng.choice([1, 1, 2]), Hkv=rng.choice([2, 4, 8]),
                    N=_log(rng, 256, 32768), D=rng.choice([64, 128, 256]),
                    dtype=rng.choice(["fp16", "bf16"]), rotate=rng.random() < 0.3)
    if kind == "append":
        return dict(kind="append", B=_log(rng, 1, 256), Hkv=rng.choice([2, 4, 8]),
                    D=rng.choice([64, 128, 256]), block=rng.choice([16, 32]),
                    rotate=rng.random() < 0.8)
    if kind == "decode":
        cache = rng.choice(["k8", "kv8", "kv8", "paged", "paged", "k8v3"])
        hq, hkv = _heads(rng)
        B = _log(rng, 1, 64)
        D = rng.choice([128, 128, 256]) if cache == "k8v3" else rng.choice([64, 128, 128, 256])
        most = (1 << 29) // (B * hkv * D)  # keys: K and V codes stay below the listed caches'
        N = _log(rng, 300, min(65536, most))
        paged = cache in ("paged", "k8v3")
        return _decode(cache, B, hq, hkv, N, D, block=rng.choice([16, 32, 64]) if paged else 0,
                       rotate=rng.random() < (0.8 if paged else 0.3) and cache != "k8")
    N, K = rng.choice([(4096, 3072), (4096, 4096), (1024, 5120), (5120, 5120), (17408, 5120),
                       (5120, 17408), (14336, 4096), (4096, 14336), (rng.randrange(1000, 8000), 2048)])
    M = _log(rng, 1, 2048) if rng.random() < 0.6 else _log(rng, 1, 16)
    return _linear(rng.choice(["q4k", "q5k", "q6k"]), M, N, K, dtype=rng.choice(["fp16", "bf16"]),
                   bias=rng.random() < 0.25)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.float16):
    return torch.randn(*shape, device=DEV, dtype=dtype, generator=g)


def _qkv(c, seed):
    """Q and V are N(0, 1); K has a per-channel offset, as the keys of trained models do
    (what K smoothing is for). W8A8: three channels of Q and K are 20 times larger."""
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    q = _randn(g, c["B"], c["Hq"], c["M"], c["D"], dtype=dt)
    k = _randn(g, c["B"], c["Hkv"], c["N"], c["D"], dtype=dt)
    v = _randn(g, c["B"], c["Hkv"], c["N"], c["D"], dtype=dt)
    k += _randn(g, 1, c["Hkv"], 1, c["D"], dtype=dt)
    if c["int8_pv"]:
        ch = [c["D"] // 15, 2 * c["D"] // 5, 4 * c["D"] // 5]
        q[..., ch] *= 20
        k[..., ch] *= 20
    return q, k, v


def _cache_inputs(c, seed):
    """The query and the cache of a decode step: int8 K rows of N(0, 1) keys with their scales;
    V as the cache stores it; for paged caches a shuffled block table and mixed lengths."""
    g = _gen(seed)
    B, Hq, Hkv, N, D = (c[x] for x in ("B", "Hq", "Hkv", "N", "D"))
    s = {"q": _randn(g, B, Hq, 1, D)}
    if c["block"]:
        nb = -(-N // c["block"])
        lead = (B * nb, Hkv, c["block"])
        s["table"] = torch.randperm(B * nb, device=DEV, generator=g).to(torch.int32).reshape(B, nb)
        # lengths spread evenly (in the logarithm) from N / 16 to N, in a seeded order
        lens = [max(1, round(N * 16 ** -(i / max(1, B - 1)))) for i in range(B)]
        random.Random(seed).shuffle(lens)
        s["lens"] = torch.tensor(lens, device=DEV, dtype=torch.int32)
    else:
        lead = (B, Hkv, N)

    def rows():
        x = torch.empty(*lead, D, device=DEV, dtype=torch.int8)
        sc = torch.empty(lead, device=DEV, dtype=torch.float32)
        for i in range(0, lead[0], max(1, (1 << 27) // (math.prod(lead[1:]) * D))):
            part = slice(i, i + max(1, (1 << 27) // (math.prod(lead[1:]) * D)))
            x[part], sc[part] = _rows_int8(_randn(g, *x[part].shape))
        return x, sc

    s["k"], s["k_scale"] = rows()
    if c["cache"] == "k8":
        s["v"] = _randn(g, *lead, D)
    elif c["cache"] == "kv8":
        s["v"] = torch.randint(-127, 128, (*lead, D), device=DEV, dtype=torch.int8, generator=g)
        s["v_scale"] = torch.rand(B, Hkv, D, device=DEV, generator=g) * 0.01 + 0.02
    elif c["cache"] == "paged":
        s["v"], s["v_scale"] = rows()
    else:
        s["v"] = torch.randint(-2 ** 31, 2 ** 31 - 1, (*lead, 3 * D // 32), device=DEV,
                               dtype=torch.int32, generator=g)
        s["v_norm"] = torch.rand(*lead, D // 128, device=DEV, generator=g) * 4 + 9
        s["codebook"] = gaussian_codebook(3, 128).to(DEV)
    return s


def _kquant_fields(fmt, N, K, g):
    """Random super-blocks: (scale per sub-block, offset per sub-block or None, codes) and bytes."""
    nb = K // 256
    d = (torch.randn(N, nb, device=DEV, generator=g).abs() * 1e-2).half()
    if fmt == "q6k":
        d = (d * 0.1).half()
        sc = torch.randint(-128, 128, (N, nb, 16), device=DEV, dtype=torch.int8, generator=g)
        q = torch.randint(0, 64, (N, nb, 2, 4, 32), device=DEV, dtype=torch.uint8, generator=g)
        lo, hi = q & 15, q >> 4
        ql = lo[..., :2, :] | (lo[..., 2:, :] << 4)
        qh = hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)
        w = torch.cat([ql.reshape(N, nb, 128), qh.reshape(N, nb, 64), sc.view(torch.uint8),
                       d.view(torch.uint8).reshape(N, nb, 2)], -1)
        return d, None, sc, None, q.reshape(N, nb, 16, 16), w.reshape(N, -1)
    dmin = (torch.randn(N, nb, device=DEV, generator=g).abs() * 1e-2).half()
    sc = torch.randint(0, 64, (N, nb, 8), device=DEV, dtype=torch.uint8, generator=g)
    mn = torch.randint(0, 64, (N, nb, 8), device=DEV, dtype=torch.uint8, generator=g)
    q = torch.randint(0, 16 if fmt == "q4k" else 32, (N, nb, 8, 32), device=DEV, dtype=torch.uint8,
                      generator=g)
    packed = torch.cat([(sc[..., :4] & 63) | ((sc[..., 4:] >> 4) << 6),
                        (mn[..., :4] & 63) | ((mn[..., 4:] >> 4) << 6),
                        (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)
    parts = [d.view(torch.uint8).reshape(N, nb, 2), dmin.view(torch.uint8).reshape(N, nb, 2), packed]
    if fmt == "q5k":
        qh = torch.zeros(N, nb, 32, device=DEV, dtype=torch.uint8)
        for j in range(8):
            qh |= (q[..., j, :] >> 4) << j
        parts.append(qh)
    parts.append(((q[..., 0::2, :] & 15) | ((q[..., 1::2, :] & 15) << 4)).reshape(N, nb, 128))
    return d, dmin, sc, mn, q, torch.cat(parts, -1).reshape(N, -1)


def _linear_inputs(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    fields = _kquant_fields(c["fmt"], c["N"], c["K"], g)
    x = _randn(g, c["M"], c["K"], dtype=dt)
    bias = _randn(g, c["N"], dtype=dt) if c["bias"] else None
    return fields, x, bias


def _append_inputs(c, seed):
    g = _gen(seed)
    blocks = c["B"] * 4
    pool = (blocks, c["Hkv"], c["block"])
    s = {"k_new": _randn(g, c["B"], c["Hkv"], c["D"]), "v_new": _randn(g, c["B"], c["Hkv"], c["D"])}
    s["k"], s["v"] = (torch.randint(-127, 128, (*pool, c["D"]), device=DEV, dtype=torch.int8,
                                    generator=g) for _ in range(2))
    s["k_scale"], s["v_scale"] = (torch.rand(pool, device=DEV, generator=g) for _ in range(2))
    s["slots"] = torch.randperm(blocks * c["block"], device=DEV, generator=g)[:c["B"]].to(torch.int32)
    return s


def prepare(case: dict, seed: int) -> dict:
    c, kind = case, case["kind"]
    if kind == "prefill":
        q, k, v = _qkv(c, seed)
        return {"case": c, "q": q, "k": k, "v": v}
    if kind == "build":
        g, dt = _gen(seed), DTYPES[c["dtype"]]
        k, v = (_randn(g, c["B"], c["Hkv"], c["N"], c["D"], dtype=dt) for _ in range(2))
        return {"case": c, "k": k + _randn(g, 1, c["Hkv"], 1, c["D"], dtype=dt), "v": v}
    if kind == "append":
        return {"case": c, **_append_inputs(c, seed)}
    if kind == "decode":
        s = _cache_inputs(c, seed)
        if c["cache"] == "k8":  # the entry point takes the query already quantised
            s["q"], qs = _C.quantize_i8_rowwise(s["q"].reshape(-1, c["D"]))
            s["q"] = s["q"].reshape(c["B"], c["Hq"], 1, c["D"])
            s["q_scale"] = (qs * (LOG2E / math.sqrt(c["D"]))).reshape(c["B"], c["Hq"], 1)
        return {"case": c, **s}
    fields, x, bias = _linear_inputs(c, seed)
    return {"case": c, "x": x, "w": fields[-1], "bias": bias}


def run(state: dict):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "prefill":
        # W8A8 of outlier inputs: the caller opts out of the gate, which would send them to fp16
        return sl8.attn_int8_fwd(s["q"], s["k"], s["v"], causal=c["causal"], int8_pv=c["int8_pv"],
                                 window_left=c["window"], internal_accuracy_gate=not c["int8_pv"])
    if kind == "build":
        return sl8.quantize_kv_cache(s["k"], s["v"], rotate=c["rotate"])
    if kind == "append":
        sl8.quantize_kv_write_paged(s["k_new"], s["v_new"], s["k"], s["k_scale"], s["v"],
                                    s["v_scale"], s["slots"], rotate=c["rotate"])
        return s["k"], s["k_scale"], s["v"], s["v_scale"]
    if kind == "decode":
        if c["cache"] == "k8":
            return _C.attn_int8_decode(s["q"], s["q_scale"], s["k"], s["k_scale"], s["v"],
                                       c["splits"] or -1)
        if c["cache"] == "kv8":
            return sl8.attn_decode_cached(s["q"], s["k"], s["k_scale"], s["v"], s["v_scale"],
                                          rotate=c["rotate"])
        if c["cache"] == "paged":
            return sl8.attn_paged_decode_cached(s["q"], s["k"], s["k_scale"], s["v"], s["v_scale"],
                                                s["table"], s["lens"], c["block"],
                                                max_context_len=c["N"], rotate=c["rotate"])
        return sl8.attn_paged_decode_k8v3(s["q"], s["k"], s["k_scale"], s["v"], s["v_norm"],
                                          s["codebook"], s["table"], s["lens"], c["block"],
                                          max_context_len=c["N"], rotate=c["rotate"])
    return LINEAR[c["fmt"]](s["x"], s["w"], bias=s["bias"], out_dtype=s["x"].dtype)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case: dict) -> dict:
    c, kind = case, case["kind"]
    if kind == "prefill":
        B, Hq, Hkv, M, N, D = (c[x] for x in ("B", "Hq", "Hkv", "M", "N", "D"))
        # causal: query i sees the last `window` (all, if -1) of the keys up to i + N - M
        past = [i + N - M + 1 for i in range(M)] if c["causal"] else [N] * M
        pairs = sum(min(n, c["window"]) if c["window"] >= 0 else n for n in past)
        return {"bytes": 2 * D * (2 * B * Hq * M + 2 * B * Hkv * N), "flops": 4 * B * Hq * D * pairs}
    if kind == "build":
        n = c["B"] * c["Hkv"] * c["N"]
        return {"bytes": 2 * n * c["D"] * 3 + 4 * n + 4 * c["B"] * c["Hkv"] * c["D"],
                "flops": 6 * n * c["D"]}
    if kind == "append":
        n = c["B"] * c["Hkv"]
        rot = 2 * n * c["D"] ** 2 if c["rotate"] else 0
        return {"bytes": n * (6 * c["D"] + 8) + 4 * c["B"], "flops": 6 * n * c["D"] + rot}
    if kind == "decode":
        B, Hq, Hkv, N, D = (c[x] for x in ("B", "Hq", "Hkv", "N", "D"))
        keys = B * N
        if c["block"]:
            keys = sum(max(1, round(N * 16 ** -(i / max(1, B - 1)))) for i in range(B))
        per_key = {"k8": 3 * D + 4, "kv8": 2 * D + 4, "paged": 2 * D + 8,
                   "k8v3": D + 4 + 3 * D // 8 + 4 * (D // 128)}[c["cache"]]
        return {"bytes": keys * Hkv * per_key + 4 * B * Hq * D, "flops": 4 * keys * Hq * D}
    M, N, K = c["M"], c["N"], c["K"]
    return {"bytes": N * (K // 256) * BLOCK_BYTES[c["fmt"]] + 2 * M * K + 2 * M * N,
            "flops": 2 * M * N * K}


def tolerance(case: dict):
    c, kind = case, case["kind"]
    bf16 = c.get("dtype") == "bf16"
    if kind == "prefill":
        if c["int8_pv"]:
            # P is requantised to int8 against an implementation's own reference points
            return {"rel": 6e-3, "max": 0.1}
        # fp16 (bf16) probabilities and outputs
        return {"rel": 8e-3, "max": 0.1} if bf16 else {"rel": 1e-3, "max": 0.02}
    if kind in ("build", "append"):
        # codes and scales follow from the inputs; the rotation's 32-bit sums move a rounding to
        # 16 bits now and then, and with it a code and a row's scale
        if c["rotate"]:
            return {"rel": 1e-4, "max": 1e-2, "differ": 2e-3}
        return {"rel": 1e-6, "max": 1e-5, "differ": 1e-6}
    if kind == "decode":
        # fp16 output and probabilities; with the rotation the query's codes move as above
        return {"rel": 4e-3, "max": 0.05} if c["rotate"] else {"rel": 1.2e-3, "max": 0.02}
    # exact integer sums per super-block, 32-bit sums over them, one rounding to the output
    return {"rel": 4e-3, "max": 0.02} if bf16 else {"rel": 5e-4, "max": 3e-3}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------
def _codes(x, s):
    return torch.clamp(torch.round(x.float() / s), -127, 127)


def _rows_int8(x):
    """The row-wise int8 contract: scale = max|x| * fp32(1/127) (1 for a zero row)."""
    s = x.float().abs().amax(-1, keepdim=True) * torch.tensor(1.0 / 127.0, device=x.device)
    s = torch.where(s == 0, torch.ones_like(s), s)
    return _codes(x, s).to(torch.int8), s.squeeze(-1)


def _rows_value(x):
    q, s = _rows_int8(x)
    return q.double() * s.double()[..., None]


def _smooth(k):
    return (k.float() - k.double().mean(-2, keepdim=True).float()).to(k.dtype)


def _rotated(x):
    """x times the normalised Sylvester-Hadamard matrix of its last dim, in x's dtype."""
    h = torch.ones(1, 1, device=x.device, dtype=torch.float64)
    while h.shape[0] < x.shape[-1]:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x.double() @ h / math.sqrt(x.shape[-1])).to(x.dtype)


def _exact_prefill(c, seed):
    q, k, v = _qkv(c, seed)
    B, Hq, Hkv, M, N, D = (c[x] for x in ("B", "Hq", "Hkv", "M", "N", "D"))
    q, k = _rows_value(q), _rows_value(_smooth(k))
    if c["int8_pv"]:
        s = v.float().abs().amax(-2, keepdim=True) * torch.tensor(1.0 / 127.0, device=v.device)
        v = _codes(v, s).double() * s.double()
    else:
        v = v.double()
    out = torch.empty(B, Hq, M, D, device=q.device, dtype=torch.float64)
    j = torch.arange(N, device=q.device)
    for b in range(B):
        for h in range(Hq):
            kk, vv = k[b, h // (Hq // Hkv)], v[b, h // (Hq // Hkv)]
            for m0 in range(0, M, 4096):
                m1 = min(M, m0 + 4096)
                s = q[b, h, m0:m1] @ kk.T / math.sqrt(D)
                i = torch.arange(m0, m1, device=q.device)[:, None] + (N - M)
                if c["causal"]:
                    s.masked_fill_(j > i, -math.inf)
                if c["window"] >= 0:
                    s.masked_fill_(j <= i - c["window"], -math.inf)
                out[b, h, m0:m1] = torch.softmax(s, -1) @ vv
    return out


def _exact_decode(c, seed):
    s = _cache_inputs(c, seed)
    B, Hq, Hkv, N, D = (c[x] for x in ("B", "Hq", "Hkv", "N", "D"))
    q = _rows_value(_rotated(s["q"]) if c["rotate"] else s["q"])[:, :, 0]
    out = torch.empty(B, Hq, 1, D, device=q.device, dtype=torch.float64)

    def rows(x, b):  # [Hkv, keys of sequence b, ...]
        if not c["block"]:
            return x[b]
        x = x[s["table"][b].long()].transpose(0, 1).flatten(1, 2)
        return x[:, :int(s["lens"][b])]

    for b in range(B):
        k = rows(s["k"], b).double() * rows(s["k_scale"], b).double()[..., None]
        v = rows(s["v"], b)
        if c["cache"] == "k8v3":
            bits = (v.long()[..., None] >> torch.arange(32, device=v.device)) & 1
            codes = bits.flatten(-2).unflatten(-1, (D, 3))
            codes = codes[..., 0] + 2 * codes[..., 1] + 4 * codes[..., 2]
            norm = rows(s["v_norm"], b).repeat_interleave(128, -1)
            v = (s["codebook"][codes] * norm).half()
        v = v.double()
        if c["cache"] == "kv8":
            v = v * s["v_scale"][b].double()[:, None]
        elif c["cache"] == "paged":
            v = v * rows(s["v_scale"], b).double()[..., None]
        for h in range(Hkv):
            heads = slice(h * (Hq // Hkv), (h + 1) * (Hq // Hkv))
            p = torch.softmax(q[b, heads] @ k[h].T / math.sqrt(D), -1)
            out[b, heads, 0] = p @ v[h]
    return out


def _exact_linear(c, seed):
    (d, dmin, sc, mn, q, _), x, bias = _linear_inputs(c, seed)
    x = _rows_value(x)
    out = torch.empty(c["M"], c["N"], device=x.device, dtype=torch.float64)
    for n in range(0, c["N"], 2048):
        r = slice(n, n + 2048)
        code = q[r].double() - (32 if c["fmt"] == "q6k" else 0)
        w = (d[r].double()[..., None] * sc[r].double())[..., None] * code
        if dmin is not None:
            w -= (dmin[r].double()[..., None] * mn[r].double())[..., None]
        out[:, r] = x @ w.reshape(-1, c["K"]).T
    return out if bias is None else out + bias.double()


def exact(case: dict, seed: int):
    c, kind = case, case["kind"]
    if kind == "prefill":
        return _exact_prefill(c, seed)
    if kind == "decode":
        return _exact_decode(c, seed)
    if kind == "linear":
        return _exact_linear(c, seed)
    if kind == "append":
        s = _append_inputs(c, seed)
        k = _rotated(s["k_new"]) if c["rotate"] else s["k_new"]
        i = s["slots"].long()
        for x, sc in ((k, s["k_scale"]), (s["v_new"], s["v_scale"])):
            sc[i // c["block"], :, i % c["block"]] = x.float().abs().amax(-1) / 127
        return None, s["k_scale"].double(), None, s["v_scale"].double()
    s = prepare(c, seed)
    k = _smooth(s["k"])
    if c["rotate"]:
        k = _rotated(k)
    return (None, k.double().abs().amax(-1) / 127, None, s["v"].double().abs().amax(-2) / 127)
