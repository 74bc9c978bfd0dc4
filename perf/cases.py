"""The work whose time this repository is judged by: listed cases, drawn ones of
the same ranges, their inputs, one pass of each, and what a pass should give.

Sizes are the repository's own: the five benchmark configurations
(``amd_optimization_challenge_amd.inputs.CONFIGS``), the task's shapes (16 heads,
batch 4 to 256, 1024 or 8192 cached tokens, contiguous) and the options the
entry points take (cache formats, Q precisions, pages, causal multi-token rows,
log-sum-exp).  Inputs are N(0, 1) bf16 as in the benchmark; the caches are
quantized here in plain torch, so that ``exact`` needs none of the
repository's code.
"""
from __future__ import annotations

import math
import random

import torch

from amd_optimization_challenge_amd import custom_kernel, kv_cache, neighbours, ops

QK, V = 576, 512          # latent + rope, latent
NOPE, ROPE, VH = 128, 64, 128
ROW_BYTES = {"fp8": 576, "mxfp4": 306, "auto": 306, "mxfp4k_fp8v": 818, "bf16": 1152}
DEV = "cuda"


def _decode(name, batch, heads, lens, lo, hi, mode, q_dtype="fp8", qlen=1, page=1, permute=True, lse=False,
            lens_seed=0):
    c = dict(kind="decode", batch=batch, heads=heads, lens=lens, lo=lo, hi=hi, mode=mode, q_dtype=q_dtype,
             qlen=qlen, page=page, permute=permute, lse=lse, lens_seed=lens_seed)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest benchmark configuration: four short sequences, where
        # launches and host time are the call
        _decode("a8w8_b4_l256", 4, 16, "uniform", 256, 256, "fp8"),
        # one of eight head shards of a 128-head model, a small serving batch
        _decode("a8w8_b32_l1024", 32, 16, "uniform", 1024, 1024, "fp8"),
        # the task's largest shape on the fastest route (contiguous cache)
        _decode("auto_b256_l8192", 256, 16, "uniform", 8192, 8192, "auto", q_dtype="auto", permute=False),
        # the task's shape of few, long sequences on the same route: every
        # sequence is cut into pieces to fill the card
        _decode("auto_b4_l8192", 4, 16, "uniform", 8192, 8192, "auto", q_dtype="auto", permute=False),
        # all 128 heads on one card, ragged lengths, fp8 cache
        _decode("h128_a8w8_b64", 64, 128, "uniform", 512, 8192, "fp8", lens_seed=3),
        # the mxfp4 cache over scattered slots
        _decode("mxfp4_b128_l4096", 128, 16, "uniform", 4096, 4096, "mxfp4"),
        # a serving batch with a long tail, 128 heads, mxfp4 K and fp8 V
        _decode("h128_mixed_b256", 256, 128, "lognormal", 1, 32768, "mxfp4k_fp8v", lens_seed=5),
        # speculative decoding: four new tokens a sequence, causal, with the
        # log-sum-exp a caller merges other context with
        _decode("causal4_b32", 32, 16, "uniform", 512, 8192, "fp8", qlen=4, lse=True, lens_seed=7),
        # bf16 queries over pages of two tokens
        _decode("a16w8_page2_b64_l8192", 64, 16, "uniform", 8192, 8192, "fp8", q_dtype="bf16", page=2),
        # a prefill's tokens written into both caches at scattered slots
        dict(name="append_8192", kind="append", tokens=8192, capacity=32768),
        # both caches built whole from a bf16 latent buffer
        dict(name="build_131072", kind="build", tokens=131072),
        # the per-head products before and after the decode (128 heads), the
        # second one quantized for the product that follows
        dict(name="proj_b64_h128", kind="proj", batch=64, heads=128),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 8 + ["append", "build", "proj"])
    if kind == "append":
        n = _log_uniform(rng, 1, 65536)
        return dict(kind="append", tokens=n, capacity=n + _log_uniform(rng, 64, 65536))
    if kind == "build":
        return dict(kind="build", tokens=_log_uniform(rng, 17, 262144))
    if kind == "proj":
        return dict(kind="proj", batch=_log_uniform(rng, 1, 512), heads=rng.choice([16, 128]))
    heads = rng.choice([16, 16, 16, 128])
    if heads == 128:
        mode = rng.choice(["fp8", "mxfp4k_fp8v"])
        q_dtype, qlen = "fp8", rng.choice([1, 1, 1, 2])
        most = 500_000 // qlen
    else:
        mode = rng.choice(["fp8", "fp8", "mxfp4", "auto", "auto", "mxfp4k_fp8v", "bf16"])
        q_dtype = "auto" if mode == "auto" else rng.choice(["fp8", "bf16"]) if mode == "fp8" else "fp8"
        qlen = rng.choice([1, 1, 2, 4])
        most = {"fp8": 1_000_000, "bf16": 500_000, "mxfp4k_fp8v": 600_000}.get(mode, 2_000_000) // qlen
    batch = _log_uniform(rng, 1, 300)
    mean = _log_uniform(rng, 32, min(32768, max(64, most // batch)))
    page = rng.choice([1, 1, 1, 2, 16])
    lens = rng.choice(["fixed", "ragged"])
    lo, hi = (mean, mean) if lens == "fixed" else (max(1, mean // 4), mean + (mean - max(1, mean // 4)))
    return _decode(None, batch, heads, "uniform", lo, hi, mode, q_dtype, qlen, page,
                   page > 1 or rng.random() < 0.5, rng.random() < 0.3, rng.randrange(1 << 20))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _lengths(c):
    rng = random.Random(c["lens_seed"])
    if c["lens"] == "lognormal":  # median 1000, sigma 1, as the benchmark's long-tail batch
        return [min(max(round(math.exp(math.log(1000.0) + rng.gauss(0.0, 1.0))), c["lo"]), c["hi"])
                for _ in range(c["batch"])]
    return [rng.randint(c["lo"], c["hi"]) for _ in range(c["batch"])]


def _fp8_rows(x, scale):
    return (x / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)


def _fp8_scale(x, dim=None):
    a = x.abs()
    a = a.amax() if dim is None else a.amax(dim=dim, keepdim=True)
    return a.clamp(min=1e-12) / 448.0


def _pack_fp4(x):
    """bf16 [n, 576] -> (packed e2m1 [n, 288], e8m0 [n, 18]) uint8."""
    n = x.shape[0]
    packed = torch.empty((n, QK // 2), dtype=torch.uint8, device=x.device)
    scales = torch.empty((n, QK // 32), dtype=torch.uint8, device=x.device)
    for i in range(0, n, 1 << 17):
        y = x[i:i + (1 << 17)].float().reshape(-1, QK // 32, 32)
        bits = (y.abs().amax(dim=2).view(torch.int32) + 0x200000) >> 23
        e = (bits - 129).clamp(-127, 127)
        scales[i:i + y.shape[0]] = (e + 127).to(torch.uint8)
        y = y * torch.exp2(-e.float()).unsqueeze(2)
        a = y.abs()
        code = torch.where(a < 2, torch.round(2 * a), torch.where(a < 4, torch.round(a) + 2,
                                                                  torch.round(a.clamp(max=6) / 2) + 4))
        code = code.to(torch.uint8) | ((y < 0).to(torch.uint8) << 3)
        code = code.reshape(-1, QK // 2, 2)
        packed[i:i + code.shape[0]] = code[..., 0] | (code[..., 1] << 4)
    return packed, scales


def _decode_inputs(c, seed):
    """Plain tensors: q, caches by token slot, and for each sequence its length
    and the slots of its tokens (a permutation of all slots, by page)."""
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    lens, P = _lengths(c), c["page"]
    pages = [-(-n // P) for n in lens]
    n_pages = sum(pages)
    q = torch.randn((c["batch"] * c["qlen"], c["heads"], QK), dtype=torch.bfloat16, device=DEV, generator=gen)
    kv = torch.randn((n_pages * P, QK), dtype=torch.bfloat16, device=DEV, generator=gen)
    if c["permute"]:
        ids = torch.randperm(n_pages, device=DEV, generator=gen).to(torch.int32)
    else:
        ids = torch.arange(n_pages, dtype=torch.int32, device=DEV)
    x = dict(q=q, lens=lens, pages=pages, ids=ids)
    if c["mode"] == "bf16":
        x["bf16"] = kv
    if c["mode"] in ("fp8", "mxfp4k_fp8v"):
        s = _fp8_scale(kv)
        x["fp8"], x["fp8_scale"] = _fp8_rows(kv, s), s.float().reshape(1)
    if c["mode"] in ("mxfp4", "auto", "mxfp4k_fp8v"):
        x["fp4"], x["fp4_scales"] = _pack_fp4(kv)
    return x


def _indptr(counts):
    return torch.tensor([0] + list(counts), dtype=torch.int32).cumsum(0).to(torch.int32).to(DEV)


def _prepare_decode(c, seed):
    x = _decode_inputs(c, seed)
    P, n = c["page"], len(x["ids"]) * c["page"]

    def rows(t):
        return t.reshape(n, 1, -1) if P == 1 else t.reshape(n // P, P, 1, -1)

    kv = {}
    if "bf16" in x:
        kv["bf16"] = rows(x["bf16"])
    if "fp8" in x:
        kv["fp8"] = (rows(x["fp8"]), x["fp8_scale"])
    if "fp4" in x:
        kv["mxfp4"] = (rows(x["fp4"]).view(torch.float4_e2m1fn_x2), x["fp4_scales"].view(torch.float8_e8m0fnu))
    cfg = dict(batch_size=c["batch"], num_heads=c["heads"], num_kv_heads=1, qk_head_dim=QK, kv_lora_rank=V,
               qk_rope_head_dim=ROPE, v_head_dim=V, q_seq_len=c["qlen"], kv_seq_len=max(x["lens"]),
               sm_scale=_sm_scale(c), kv_mode=c["mode"], return_lse=c["lse"])
    if c["q_dtype"] != "auto":
        cfg["q_dtype"] = c["q_dtype"]
    if c["permute"] or P > 1:
        cfg["kv_indices"] = x["ids"]
    if P > 1:
        cfg["page_size"] = P
        cfg["kv_last_page_lens"] = torch.tensor([L - (p - 1) * P for L, p in zip(x["lens"], x["pages"])],
                                                dtype=torch.int32).to(DEV)
    kv_indptr = _indptr(x["pages"])
    qo_indptr = torch.arange(c["batch"] + 1, dtype=torch.int32, device=DEV) * c["qlen"]
    return (x["q"], kv, qo_indptr, kv_indptr, cfg)


def _sm_scale(c):
    return 1.0 / math.sqrt(192.0 if c["permute"] else 576.0)


def _append_inputs(c, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    x = torch.randn((c["tokens"], QK), dtype=torch.bfloat16, device=DEV, generator=gen)
    slots = torch.randperm(c["capacity"], device=DEV, generator=gen)[:c["tokens"]].to(torch.int32)
    return x, slots


def _proj_inputs(c, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed))

    def randn(*shape, std=1.0):
        return (torch.randn(shape, dtype=torch.float32, device=DEV, generator=gen) * std).to(torch.bfloat16)

    B, H = c["batch"], c["heads"]
    return dict(q_nope=randn(B, H, NOPE), q_rope=randn(B, H, ROPE), w_uk=randn(H, NOPE, V, std=NOPE ** -0.5),
                o=randn(B, H, V), w_uv=randn(H, V, VH, std=V ** -0.5))


FP8_SCALE = 4.8 / 448.0  # of a cache calibrated on N(0, 1) latents


def prepare(case, seed):
    if case["kind"] == "decode":
        return dict(case=case, data=_prepare_decode(case, seed))
    if case["kind"] == "append":
        x, slots = _append_inputs(case, seed)
        return dict(case=case, x=x, slots=slots, cache=kv_cache.KVCache(case["capacity"], fp8_scale=FP8_SCALE))
    if case["kind"] == "build":
        gen = torch.Generator(device=DEV).manual_seed(int(seed))
        return dict(case=case, x=torch.randn((case["tokens"], 1, QK), dtype=torch.bfloat16, device=DEV, generator=gen))
    return dict(case=case, **_proj_inputs(case, seed))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(state):
    kind = state["case"]["kind"]
    if kind == "decode":
        return custom_kernel(state["data"])
    if kind == "append":
        cache = state["cache"]
        cache.write(state["x"], state["slots"])
        return dict(fp8=cache.fp8, fp4=cache.fp4, fp4_scales=cache.fp4_scales, amax=cache.amax_bits)
    if kind == "build":
        fp8, scale = ops.quant_fp8_per_tensor(state["x"])
        fp4, fp4_scales = ops.pack_mxfp4(state["x"])
        return dict(fp8=fp8, fp8_scale=scale, fp4=fp4, fp4_scales=fp4_scales)
    q = neighbours.absorb_q(state["q_nope"], state["q_rope"], state["w_uk"])
    y, scale = neighbours.v_up_proj(state["o"], state["w_uv"], quant_fp8=True)
    return dict(q=q, y=y, y_scale=scale)


# ---------------------------------------------------------------------------
# what a pass cannot do without, and what it should give
# ---------------------------------------------------------------------------


def work(case):
    if case["kind"] == "append":  # the token, its slot; its row of both caches
        return dict(bytes=case["tokens"] * (2 * QK + 4 + 576 + 306), flops=0)
    if case["kind"] == "build":
        return dict(bytes=case["tokens"] * (2 * QK + 576 + 306), flops=0)
    if case["kind"] == "proj":
        B, H = case["batch"], case["heads"]
        weights = H * (NOPE * V + V * VH)
        rows = B * H * (NOPE + ROPE + QK + V)
        return dict(bytes=2 * (weights + rows) + B * H * VH, flops=2 * B * weights)
    lens, rows = _lengths(case), case["batch"] * case["qlen"]
    per_token = ROW_BYTES[case["mode"]] + (4 / case["page"] if case["permute"] or case["page"] > 1 else 0)
    io = rows * case["heads"] * (2 * QK + 2 * V + (4 if case["lse"] else 0))
    return dict(bytes=sum(lens) * per_token + io, flops=2 * case["heads"] * (QK + V) * sum(lens) * case["qlen"])


def tolerance(case):
    if case["kind"] in ("append", "build"):
        return "exact"  # bytes of the cache formats
    if case["kind"] == "proj":
        # bf16 results of f32 sums; the fp8 codes of two results that round to
        # neighbouring bf16 values may differ by a step
        return {"rel": 4e-3, "max": 0.25}
    # bf16 results (one rounding 1.7e-3 in the 2-norm), the split pieces in bf16
    # too, the probabilities at seven to eight significant bits
    return {"rel": 1e-2, "max": 0.1}


E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _fp4_rows(packed, scales):
    lut = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device=packed.device)
    codes = torch.stack((packed & 15, packed >> 4), dim=-1).reshape(packed.shape[0], QK).long()
    s = torch.exp2(scales.double() - 127.0).repeat_interleave(32, dim=1)
    return lut[codes] * s


def _exact_decode(c, seed):
    x = _decode_inputs(c, seed)
    q = x["q"]
    if c["mode"] == "bf16" or c["q_dtype"] == "bf16":
        q = q.double()
    else:  # per tensor, or per head row on the fastest route
        s = _fp8_scale(q, dim=2 if c["q_dtype"] == "auto" else None)
        q = _fp8_rows(q, s).float().double() * s.float().double()
    out = torch.zeros((q.shape[0], c["heads"], V), dtype=torch.float64, device=DEV)
    lse = torch.full((q.shape[0], c["heads"]), -math.inf, dtype=torch.float64, device=DEV)
    P, at = c["page"], 0
    within = torch.arange(P, device=DEV)
    for b, (L, n) in enumerate(zip(x["lens"], x["pages"])):
        slots = (x["ids"][at:at + n].long()[:, None] * P + within).reshape(-1)[:L]
        at += n
        if c["mode"] == "bf16":
            k = v = x["bf16"][slots].double()
        else:
            f8 = x["fp8"][slots].float().double() * x["fp8_scale"].double() if "fp8" in x else None
            k = _fp4_rows(x["fp4"][slots], x["fp4_scales"][slots]) if "fp4" in x else f8
            v = k if f8 is None else f8
        for i in range(c["qlen"]):
            r, m = b * c["qlen"] + i, L - (c["qlen"] - 1 - i)
            if m > 0:
                s = (q[r] @ k[:m].T) * _sm_scale(c)
                lse[r] = torch.logsumexp(s, dim=1)
                out[r] = torch.softmax(s, dim=1) @ v[:m, :V]
    return (out, lse) if c["lse"] else out


def exact(case, seed):
    if case["kind"] == "decode":
        return _exact_decode(case, seed)
    if case["kind"] == "append":
        x, slots = _append_inputs(case, seed)
        fp8 = torch.zeros((case["capacity"], 1, QK), dtype=torch.float64, device=DEV)
        y = (x.float() / torch.tensor(FP8_SCALE, dtype=torch.float32, device=DEV)).to(torch.bfloat16)
        fp8[slots.long(), 0] = y.clamp(-448.0, 448.0).to(torch.float8_e4m3fn).float().double()
        return dict(fp8=fp8, fp4=None, fp4_scales=None, amax=None)
    if case["kind"] == "build":
        gen = torch.Generator(device=DEV).manual_seed(int(seed))
        x = torch.randn((case["tokens"], 1, QK), dtype=torch.bfloat16, device=DEV, generator=gen)
        s = _fp8_scale(x)
        return dict(fp8=_fp8_rows(x, s).float().double(), fp8_scale=s.double().reshape(1), fp4=None, fp4_scales=None)
    x = {k: v.double() for k, v in _proj_inputs(case, seed).items()}
    q = torch.cat(((x["q_nope"].transpose(0, 1) @ x["w_uk"]).transpose(0, 1), x["q_rope"]), dim=2)
    y = (x["o"].transpose(0, 1) @ x["w_uv"]).transpose(0, 1)
    return dict(q=q, y=None, y_scale=_fp8_scale(y).reshape(1))
