"""Items that run a second time from higher references: scores, and at 16 heads the
block exponents of an fp4 V, that rise within one work item by more than its first
tile's reference may carry.  Each case checks from the plan the call left behind
that some item holds such a rise, so that the second pass is what is compared with
the oracle."""
import numpy as np
import pytest
import torch

from amd_optimization_challenge_amd import ops
from mla_cases import assert_close, case_from_tensors, device_data
from oracle import mla_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
SM = 1 / np.sqrt(192)
MODES = [(16, "fp8"), (16, "mxfp4"), (16, "mxfp4k_fp8v"), (128, "fp8"), (128, "mxfp4k_fp8v")]
LEVELS = torch.tensor([0.0, 1.0, 2.0, 4.0])  # by 64-token stretch of a sequence; a level is 130 log2 units


def _case(q, kv, lens, mode, contiguous, seed):
    """(q, kv) with kv in sequence order -> the case with the rows at their slots."""
    T = sum(lens)
    idx = torch.arange(T) if contiguous else torch.randperm(T, generator=torch.Generator().manual_seed(seed))
    rows = torch.empty_like(kv)
    rows[idx] = kv
    indptr = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    return case_from_tensors(q.to(torch.bfloat16), rows.to(torch.bfloat16), indptr, idx.to(torch.int32), mode)


def _run(case, mode, qlen, contiguous, rows_route=False, monkeypatch=None, **kw):
    """(out, items of the call's plan [n, 4]: row or sequence, first token, end, slot)"""
    q, kv, indptr, idx, _, caches = case
    S = indptr.numel() - 1
    _, kv_data, _, kv_indptr, cfg = device_data(q[:S], kv, indptr, idx, caches, mode, SM, pass_indices=not contiguous)
    if monkeypatch is not None:
        monkeypatch.setattr(ops, "_rows_together", lambda *a: rows_route)
    heads = q.shape[1]
    ws = torch.empty(ops.workspace_bytes(S * qlen, heads, mode, qlen), dtype=torch.uint8, device=DEV)
    out = ops.decode_fwd(q.to(DEV), kv_data, kv_indptr, cfg["kv_indices"], SM, mode, ws=ws, q_seq_len=qlen, **kw)
    return out.float().cpu().numpy(), ops.read_plan(ws, S * qlen, heads, mode)["items"].numpy()


def _reference(case, mode, qlen):
    """The oracle's decode in float64 on the device (float32 on the host takes 40 s
    at 90000 tokens x 4 rows)."""
    _, _, indptr, idx, qb, caches = case
    codes, scale = O.quantize_fp8_per_tensor(qb)
    q = torch.from_numpy(O.dequant_fp8(codes, scale)).to(DEV).double()
    k, v = (torch.from_numpy(t[idx.numpy()]).to(DEV).double() for t in O.dequant_kv(mode, **caches))
    out = torch.zeros(q.shape[0], q.shape[1], 512, dtype=torch.float64, device=DEV)
    for r in range(q.shape[0]):
        a, z = int(indptr[r // qlen]), int(indptr[r // qlen + 1]) - (qlen - 1 - r % qlen)
        if z > a:
            out[r] = torch.softmax((q[r] @ k[a:z].T) * SM, dim=1) @ v[a:z, :512]
    return out.float().cpu().numpy()


def _score_rise(case, mode, items, tile):
    """(largest rise of an item's scores above its first tile's, tiles of that item)"""
    q, _, _, idx, qb, caches = case
    k = O.dequant_kv(mode, **caches)[0][idx.numpy()]
    codes, scale = O.quantize_fp8_per_tensor(qb)
    s = k @ O.dequant_fp8(codes, scale)[0, 0] * np.float32(SM * 1.4426950408889634)
    return max((s[a:e].max() - s[a:a + tile].max(), -(-(e - a) // tile)) for _, a, e, _ in items if e > a)


def _levels(lens, heads, qlen, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(len(lens) * qlen, heads, 576, generator=g)
    q[..., 7] = 40.0
    kv = 0.25 * torch.randn(sum(lens), 1, 576, generator=g)
    pos = torch.cat([torch.arange(L) for L in lens])
    kv[:, 0, 7] = 31.25 * LEVELS[(pos // 64) % 4]
    return q, kv


@pytest.mark.parametrize("heads,mode", MODES)
@pytest.mark.parametrize("lens,contiguous", [([700, 130, 5], False), ([700, 130, 5], True), ([10277], True)])
def test_scores_that_rise_within_an_item(heads, mode, lens, contiguous):
    q, kv = _levels(lens, heads, 1, 17)
    case = _case(q, kv, lens, mode, contiguous, 3)
    got, items = _run(case, mode, 1, contiguous)
    rise, tiles = _score_rise(case, mode, items, 64 if heads == 16 else 32)
    assert rise > 97 and tiles >= (5 if heads == 16 and lens[0] > 10000 else 2), (rise, tiles)
    _, ref = O.reference_path(case[4], mode, case[5], case[2].numpy(), case[3].numpy(), SM)
    assert_close(got, ref)


@pytest.mark.parametrize("qlen", [2, 4])
@pytest.mark.parametrize("lens,contiguous", [([700, 130, 5], False), ([700, 130, 5], True), ([10277], True),
                                             ([45011, 44990], False)])
def test_scores_that_rise_within_an_item_of_several_rows(monkeypatch, qlen, lens, contiguous):
    q, kv = _levels(lens, 16, qlen, 19)
    case = _case(q, kv, lens, "fp8", contiguous, 5)
    got, items = _run(case, "fp8", qlen, contiguous, True, monkeypatch)
    rise, tiles = _score_rise(case, "fp8", items, 64)
    assert rise > 97 and tiles >= (5 if sum(lens) > 10000 else 2), (rise, tiles)
    assert_close(got, _reference(case, "fp8", qlen))


@pytest.mark.parametrize("q_dtype", ["fp8", "fp8_row"])
@pytest.mark.parametrize("blocks", [slice(0, 512), slice(96, 128)])
@pytest.mark.parametrize("jump", [40, 70, -40])
@pytest.mark.parametrize("lens,contiguous", [([700, 130, 5], False), ([700, 130, 5], True), ([10277], True)])
def test_fp4_value_exponents_that_jump_within_an_item(q_dtype, blocks, jump, lens, contiguous):
    """Ordinary scores (Q is zero on the latent dims); every second stretch of 64
    tokens has V 2^jump as large in all, or one, of its blocks.  Past 31 the item runs
    again from the higher exponent."""
    g = torch.Generator().manual_seed(23)
    q = torch.randn(len(lens), 16, 576, generator=g)
    q[..., :512] = 0.0
    kv = torch.randn(sum(lens), 1, 576, generator=g)
    pos = torch.cat([torch.arange(L) for L in lens])
    kv[(pos // 64) % 2 == 1, :, blocks] *= 2.0 ** jump
    case = _case(q, kv, lens, "mxfp4", contiguous, 7)
    got, items = _run(case, "mxfp4", 1, contiguous, q_dtype=q_dtype)
    e = case[5]["fp4_scales"][case[3].numpy()][:, :16].max(axis=1).astype(int)  # of the V blocks, by token
    rise = max(e[a:z].max() - e[a:a + 64].max() for _, a, z, _ in items if z > a)
    assert jump < 0 or rise > 31, rise
    _, ref = O.reference_path(case[4], "mxfp4", case[5], case[2].numpy(), case[3].numpy(), SM, q_dtype=q_dtype)
    for b in range(len(lens)):
        for d in (blocks, slice(0, 96), slice(128, 512)):  # relative to the dims' own magnitude
            s = float(np.abs(ref[b, :, d]).max())
            assert_close(got[b, :, d] / s, ref[b, :, d] / s)
