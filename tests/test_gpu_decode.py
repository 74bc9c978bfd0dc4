"""HIP decode vs the CPU oracle on the same seeded inputs (atol = rtol = 2e-2
on the bf16 output, plus a relative-L2 bound), and exact invariances."""
import math

import numpy as np
import pytest
import torch

from amd_optimization_challenge_amd import custom_kernel
from mla_cases import assert_close, case_from_tensors, device_data, host_case, run_and_reference, run_case

pytestmark = pytest.mark.gpu

LENS = [
    [1],
    [63, 64, 65],
    [0, 200, 7],
    [3000, 10, 129],
    [1024] * 5,
]
MODES = [(16, "fp8"), (16, "mxfp4"), (16, "mxfp4k_fp8v"), (128, "fp8"), (128, "mxfp4k_fp8v")]


@pytest.mark.parametrize("heads,mode", MODES)
@pytest.mark.parametrize("lens", LENS)
def test_decode_matches_oracle(cuda, heads, mode, lens):
    print(f"decode H={heads} mode={mode} lens={lens[:4]}", flush=True)
    got, ref, _ = run_and_reference(lens, heads, mode, seed=len(lens) * 31 + heads)
    assert np.all(np.isfinite(got))
    assert_close(got, ref)
    for b, L in enumerate(lens):
        if L == 0:
            assert np.all(got[b] == 0)


@pytest.mark.parametrize("mode", ["fp8", "mxfp4k_fp8v"])
@pytest.mark.parametrize("lens", LENS[:4])
def test_h128_contiguous_cache_matches_oracle(cuda, mode, lens):
    """128 heads on a contiguous cache (no kv_indices: each sequence's rows in
    order from kv_indptr[b]): within tolerance of the oracle, and bit-equal to
    the same cache addressed through identity kv_indices (the 128-head plan does
    not depend on whether indices are given)."""
    from oracle import mla_oracle as O

    print(f"contiguous H=128 mode={mode} lens={lens}", flush=True)
    q, kv, indptr, idx, qb, caches = host_case(lens, 128, mode, seed=len(lens) * 7 + 3, permute=False)
    sm = 1 / math.sqrt(192)
    contig = custom_kernel(device_data(q, kv, indptr, idx, caches, mode, sm, pass_indices=False)).clone()
    indexed = custom_kernel(device_data(q, kv, indptr, idx, caches, mode, sm, pass_indices=True))
    torch.cuda.synchronize()
    _, ref = O.reference_path(qb, mode, caches, indptr.numpy(), idx.numpy(), sm)
    got = contig.float().cpu().numpy()
    assert np.all(np.isfinite(got))
    assert_close(got, ref)
    assert torch.equal(contig, indexed)


@pytest.mark.parametrize("heads,mode", MODES)
def test_sm_scale_is_honoured(cuda, heads, mode):
    print(f"sm_scale H={heads} mode={mode}", flush=True)
    for sm in (1 / math.sqrt(576), 0.3):
        got, ref, _ = run_and_reference([300, 77], heads, mode, seed=5, sm_scale=sm)
        assert_close(got, ref)


@pytest.mark.parametrize("heads,mode", MODES)
def test_wide_score_range(cuda, heads, mode):
    """Scores that climb by 25 log2 units per 64-token tile: beyond the fp8 range
    of P, so every tile needs its own offset (items that run again from higher
    references: test_gpu_second_pass.py)."""
    print(f"wide score range H={heads} mode={mode}", flush=True)
    g = torch.Generator().manual_seed(17)
    lens = [700, 130, 5]
    T = sum(lens)
    q = torch.randn(len(lens), heads, 576, generator=g)
    q[..., 7] = 40.0
    kv = 0.25 * torch.randn(T, 1, 576, generator=g)
    pos = torch.cat([torch.arange(L) for L in lens]).float()
    kv[:, 0, 7] = 6.0 * torch.floor(pos / 64) - 20.0 + 0.1 * torch.randn(T, generator=g)
    indptr = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    idx = torch.randperm(T, generator=g).to(torch.int32)
    # kv rows are addressed through idx: place token j of the flattened sequences at row idx[j]
    rows = torch.empty_like(kv)
    rows[idx.long()] = kv
    case = case_from_tensors(q.to(torch.bfloat16), rows.to(torch.bfloat16), indptr, idx, mode)
    got, ref, _ = run_case(case, mode, 1 / math.sqrt(192))
    assert np.all(np.isfinite(got))
    assert_close(got, ref)


@pytest.mark.parametrize("growth", [20, 45, 90])
def test_mxfp4_value_scale_growth(cuda, growth):
    """fp4 V (H = 16): the per-token MX block scales are folded into P relative
    to a per-item reference exponent.  Latent values that grow by 2^growth
    over the sequence give its 128-token items different references, each with
    later block exponents up to 17 above it (past 31 an item runs again:
    test_gpu_second_pass.py); Q is zero on dims 0..511, so the scores stay
    ordinary while V (and K's first 512 dims) change scale."""
    print(f"mxfp4 V scale growth 2^{growth}", flush=True)
    g = torch.Generator().manual_seed(23)
    lens = [700, 129, 64]
    T = sum(lens)
    q = torch.randn(len(lens), 16, 576, generator=g)
    q[..., :512] = 0.0
    kv = torch.randn(T, 1, 576, generator=g)
    pos = torch.cat([torch.arange(L) for L in lens]).float()
    grow = torch.exp2(growth * pos / 700.0)
    kv[:, 0, :512] *= grow[:, None]
    indptr = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    idx = torch.randperm(T, generator=g).to(torch.int32)
    rows = torch.empty_like(kv)
    rows[idx.long()] = kv
    case = case_from_tensors(q.to(torch.bfloat16), rows.to(torch.bfloat16), indptr, idx, "mxfp4")
    got, ref, _ = run_case(case, "mxfp4", 1 / math.sqrt(192))
    assert np.all(np.isfinite(got))
    # compare relative to each row's own magnitude (the outputs span 2^growth)
    for b in range(len(lens)):
        s = float(np.abs(ref[b]).max()) or 1.0
        assert_close(got[b] / s, ref[b] / s)


@pytest.mark.parametrize("contiguous", [False, True])
@pytest.mark.parametrize("log2k", [10, 22, 30])
def test_mxfp4_huge_scores(cuda, log2k, contiguous):
    """Scores up to 2^42, whose references round by more than a pass may leave above
    them: the call ends, at the row of the one largest score."""
    from oracle import mla_oracle as O

    print(f"mxfp4 huge scores 2^{log2k}", flush=True)
    lens = [200, 70, 700]
    q, kv, indptr, idx, _, _ = host_case(lens, 16, "mxfp4", seed=31, permute=not contiguous)
    q, kv = torch.zeros_like(q), kv.clone()
    q[..., 575] = 2.0 ** 14
    kv[:, 0, 544:575] = 0.0
    kv[:, 0, 575] = 2.0 ** log2k
    for b in range(len(lens)):  # past the first tile; the factor 4 is exact in any format
        kv[idx[int(indptr[b]) + 66].long(), 0, 575] = 2.0 ** (log2k + 2)
    case = case_from_tensors(q, kv, indptr, idx, "mxfp4")
    data = device_data(q, kv, indptr, idx, case[5], "mxfp4", 0.0712, pass_indices=not contiguous)
    got = custom_kernel(data)
    torch.cuda.synchronize()
    _, ref = O.reference_path(case[4], "mxfp4", case[5], indptr.numpy(), idx.numpy(), 0.0712)
    assert_close(got.float().cpu().numpy(), ref)


@pytest.mark.parametrize("heads,mode", [(16, "mxfp4"), (16, "mxfp4k_fp8v"), (128, "mxfp4k_fp8v")])
def test_mxfp4_scale_row_stride(cuda, heads, mode):
    """The e8m0 scale rows may be padded (stride > 18, odd or even); every
    stride gives the stride-18 result bit for bit."""
    print(f"scale stride H={heads} mode={mode}", flush=True)
    case = host_case([700, 129, 64, 1], heads, mode, seed=29, permute=True)
    q, kv, indptr, idx, qb, caches = case
    data = device_data(q, kv, indptr, idx, caches, mode, 1 / math.sqrt(192))
    from oracle import mla_oracle as O

    base = custom_kernel(data).clone()
    torch.cuda.synchronize()
    _, ref = O.reference_path(qb, mode, caches, indptr.numpy(), idx.numpy(), 1 / math.sqrt(192))
    assert_close(base.float().cpu().numpy(), ref)
    packed, sc = data[1]["mxfp4"]
    for cols in (19, 24, 25):
        wide = torch.full((sc.shape[0], cols), 127, dtype=torch.uint8, device=sc.device)
        wide[:, :18] = sc.view(torch.uint8)
        data[1]["mxfp4"] = (packed, wide.view(torch.float8_e8m0fnu))
        got = custom_kernel(data)
        torch.cuda.synchronize()
        assert torch.equal(got, base), cols


@pytest.mark.parametrize("heads,mode", [(16, "mxfp4"), (16, "mxfp4k_fp8v"), (128, "mxfp4k_fp8v")])
def test_mxfp4_scales_in_row(cuda, heads, mode):
    """Scales stored inside each 320-byte packed row (inputs.mxfp4_in_row:
    both caches strided views of one buffer) give the separate-array result
    bit for bit, and so does the whole operator on that layout."""
    from amd_optimization_challenge_amd import inputs

    print(f"in-row scales H={heads} mode={mode}", flush=True)
    q, kv, indptr, idx, qb, caches = host_case([700, 129, 64, 1], heads, mode, seed=31, permute=True)
    data = device_data(q, kv, indptr, idx, caches, mode, 1 / math.sqrt(192))
    base = custom_kernel(data).clone()
    qd, kv_data, qo, kv_indptr, cfg = data
    inrow = inputs.mxfp4_in_row(kv_data)
    k, s = inrow["mxfp4"]
    assert k.stride(0) == s.stride(0) == 320 and s.data_ptr() == k.data_ptr() + 288
    got = custom_kernel((qd, inrow, qo, kv_indptr, cfg))
    torch.cuda.synchronize()
    assert torch.equal(got, base)


@pytest.mark.parametrize("heads,mode", [(16, "fp8"), (128, "fp8"), (16, "mxfp4"), (128, "mxfp4k_fp8v")])
def test_cache_permutation_is_exact(cuda, heads, mode):
    # moving cache rows together with kv_indices leaves the output bit-identical
    print(f"permutation H={heads} mode={mode}", flush=True)
    q, kv, indptr, idx, qb, caches = host_case([500, 90], heads, mode, seed=9)
    out1 = custom_kernel(device_data(q, kv, indptr, idx, caches, mode, 0.07)).clone()
    perm = torch.randperm(kv.shape[0], generator=torch.Generator().manual_seed(1))
    inv = torch.argsort(perm)
    c2 = {}
    for k, v in caches.items():
        c2[k] = v[perm.numpy()] if isinstance(v, np.ndarray) and v.ndim == 2 else v
    out2 = custom_kernel(device_data(q, kv[perm], indptr, inv[idx.long()].to(torch.int32), c2, mode, 0.07))
    torch.cuda.synchronize()
    assert torch.equal(out1, out2)


@pytest.mark.parametrize("heads,mode,return_lse", [(16, "fp8", False), (128, "fp8", True),
                                                    (128, "mxfp4k_fp8v", False)])
def test_output_buffer_is_reused(cuda, heads, mode, return_lse):
    """In steady state a call allocates nothing: the result (and lse) come back
    in the operator's buffer for that shape (as the reference caches its
    output), overwritten by the next call, and the allocator's count of live
    allocations does not move from one call to the next."""
    q, kv, indptr, idx, qb, caches = host_case([300, 77], heads, mode, seed=13)
    data = device_data(q, kv, indptr, idx, caches, mode, 0.07)
    if return_lse:
        data = data[:4] + (dict(data[4], return_lse=True),)
    first = custom_kernel(data)
    torch.cuda.synchronize()
    before = torch.cuda.memory_stats()["allocation.all.current"]
    second = custom_kernel(data)
    torch.cuda.synchronize()
    assert torch.cuda.memory_stats()["allocation.all.current"] == before
    if return_lse:
        assert first[0].data_ptr() == second[0].data_ptr() and first[1].data_ptr() == second[1].data_ptr()
    else:
        assert first.data_ptr() == second.data_ptr()


def test_identity_indices_equal_explicit_arange(cuda):
    q, kv, indptr, idx, qb, caches = host_case([100, 30], 16, "fp8", seed=2, permute=False)
    d1 = device_data(q, kv, indptr, idx, caches, "fp8", 0.05, pass_indices=True)
    d2 = device_data(q, kv, indptr, idx, caches, "fp8", 0.05, pass_indices=False)
    assert torch.equal(custom_kernel(d1).clone(), custom_kernel(d2))


def test_golden_decode_fixture(cuda):
    import os

    from oracle import mla_oracle as O

    d = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "decode_fp8.npz"))
    T = d["kv"].shape[0]
    dev = torch.device("cuda")
    q = torch.from_numpy(d["q"].view(np.int16)).view(torch.bfloat16).to(dev)
    kv_data = {"fp8": (torch.from_numpy(d["kv_codes"].reshape(T, 1, 576)).to(dev).view(torch.float8_e4m3fn),
                       torch.tensor([float(d["kv_scale"])], dtype=torch.float32, device=dev))}
    cfg = {"num_heads": 16, "q_seq_len": 1, "sm_scale": float(d["sm_scale"]),
           "kv_indices": torch.from_numpy(d["kv_indices"]).to(dev)}
    out = custom_kernel((q, kv_data, None, torch.from_numpy(d["kv_indptr"]).to(dev), cfg))
    assert_close(out.float().cpu().numpy(), d["out_f32"])
    assert O.f32_to_bf16(d["out_f32"]).shape == tuple(out.shape)


@pytest.mark.parametrize("heads,mode", MODES)
def test_fused_pipeline_matches_staged(cuda, heads, mode):
    """custom_kernel (for H = 16 the decode kernel quantizes Q itself from
    the amax partials) equals the staged entry points (quant kernel, plan,
    decode, combine) bit for bit, and a second decode + combine on the same
    plan reproduces it."""
    from amd_optimization_challenge_amd import ops

    print(f"fused vs staged H={heads} mode={mode}", flush=True)
    q, kv, indptr, idx, qb, caches = host_case([3000, 10, 129, 700, 1], heads, mode, seed=41)
    data = device_data(q, kv, indptr, idx, caches, mode, 0.07)
    fused = custom_kernel(data)
    qd, kv_data, _, kv_indptr, cfg = data
    B = qd.shape[0]
    ws = ops.workspace(B, heads, mode, qd.device)
    qf8 = torch.empty(qd.shape, dtype=torch.float8_e4m3fn, device=qd.device)
    qsc = torch.empty(1, dtype=torch.float32, device=qd.device)
    ops.quant_fp8_per_tensor(qd, qf8, qsc)
    ops.plan(kv_indptr, B, heads, mode, ws)
    outs = []
    for _ in range(2):
        out = torch.full((B, heads, 512), float("nan"), dtype=torch.bfloat16, device=qd.device)
        ops.decode(qf8, qsc, kv_data, kv_indptr, cfg["kv_indices"], heads, cfg["sm_scale"], mode, ws, out)
        ops.combine(B, heads, ws, out)
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], fused)
    assert torch.equal(outs[1], fused)
    # the whole operator on a workspace of garbage bytes, twice in a row: the
    # call owns every workspace word it reads
    ws2 = torch.full_like(ws, 0x5A)
    for _ in range(2):
        out = ops.decode_fwd(qd, kv_data, kv_indptr, cfg["kv_indices"], cfg["sm_scale"], mode, ws=ws2)
        torch.cuda.synchronize()
        assert torch.equal(out, fused)


def _lse_close(got, ref, tol=1e-2):
    # an lse error d scales the row's softmax weights by e^d ~ 1 + d, so 1e-2
    # stays inside the 2e-2 output tolerance; the bf16 P of the fp4-V path
    # (relative rounding 2^-9 per weight) moves a one-dominant-token lse by ~4e-3
    inf_ref = np.isneginf(ref)
    assert np.array_equal(np.isneginf(got), inf_ref)
    err = np.abs(got[~inf_ref] - ref[~inf_ref])
    assert np.all(err <= tol + tol * np.abs(ref[~inf_ref])), err.max()


@pytest.mark.parametrize("heads,mode", MODES)
@pytest.mark.parametrize("qlen", [1, 2, 4])
def test_causal_multi_token_rows_and_lse(cuda, heads, mode, qlen):
    """q_seq_len = qlen rows per sequence (causal prefixes, reference.py:188-193)
    and return_lse, against the oracle; rows left with no key give 0 / -inf."""
    from oracle import mla_oracle as O

    print(f"mtp H={heads} mode={mode} qlen={qlen}", flush=True)
    lens = [300, 7, 1, 64, 2000, 2]
    S = len(lens)
    g = torch.Generator().manual_seed(100 + qlen + heads)
    q = torch.randn(S * qlen, heads, 576, generator=g).to(torch.bfloat16)
    _, kv, indptr, idx, _, caches = host_case(lens, heads, mode, seed=7 + qlen)
    qb = O.bf16_tensor_bits(q)
    dev = torch.device("cuda")
    data = device_data(q[:S], kv, indptr, idx, caches, mode, 0.08)
    _, kv_data, _, kv_indptr, cfg = data
    cfg = dict(cfg, q_seq_len=qlen, return_lse=True)
    qo = torch.arange(S + 1, dtype=torch.int32, device=dev) * qlen
    out, lse = custom_kernel((q.to(dev), kv_data, qo, kv_indptr, cfg))
    torch.cuda.synchronize()
    _, ref, ref_lse = O.reference_path(qb, mode, caches, indptr.numpy(), idx.numpy(), 0.08, q_seq_len=qlen,
                                       return_lse=True)
    got = out.float().cpu().numpy()
    assert_close(got, ref)
    _lse_close(lse.cpu().numpy(), ref_lse)
    for b, L in enumerate(lens):
        for i in range(qlen):
            if L - (qlen - 1 - i) <= 0:
                assert np.all(got[b * qlen + i] == 0)
