"""The causal rows of a sequence as one work item (16 heads, fp8 cache, q_seq_len 2
to 4) at the edges of its tiles: one-token to many-tile sequences, rows that see
nothing, pieces whose end lies inside the last rows' masked tail, scores and codes at
the ends of their ranges, a captured graph, more sequences than the planner sorts,
and workspaces of both sizes; against the oracle."""
import ctypes

import numpy as np
import pytest
import torch

from amd_optimization_challenge_amd import _lib, ops
from mla_cases import assert_close, case_from_tensors, device_data, host_case
from oracle import mla_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.fixture(autouse=True)
def _rows_route(monkeypatch):
    """Every test here takes the route, whatever its size."""
    monkeypatch.setattr(ops, "_rows_together", lambda *a: True)


def _run(case, q, qlen, sm, contiguous=False, ws=None):
    _, kv, indptr, idx, _, caches = case
    S = indptr.numel() - 1
    _, kv_data, _, kv_indptr, cfg = device_data(q[:S], kv, indptr, idx, caches, "fp8", sm, pass_indices=not contiguous)
    return ops.decode_fwd(q.to(DEV), kv_data, kv_indptr, cfg["kv_indices"], sm, "fp8", ws=ws, q_seq_len=qlen,
                          return_lse=True)


def _check(case, q, qlen, sm, out, lse):
    _, _, indptr, idx, _, caches = case
    _, ref, ref_lse = O.reference_path(O.bf16_tensor_bits(q), "fp8", caches, indptr.numpy(), idx.numpy(), sm,
                                       q_seq_len=qlen, return_lse=True)
    assert_close(out.float().cpu().numpy(), ref)
    got = lse.cpu().numpy()
    assert np.array_equal(np.isneginf(got), np.isneginf(ref_lse))
    fin = ~np.isneginf(ref_lse)
    # an lse error d scales the row's weights by e^d: 1e-2 stays inside the 2e-2 of the output
    assert np.all(np.abs(got[fin] - ref_lse[fin]) <= 1e-2 + 1e-2 * np.abs(ref_lse[fin]))


@pytest.mark.parametrize("qlen", [2, 3, 4])
@pytest.mark.parametrize("contiguous", [False, True])
@pytest.mark.parametrize("lens", [[1], [3, 2, 64], [63, 65, 66], [130, 0, 127, 129], [2049], [191] * 40])
def test_rows_match_oracle(qlen, contiguous, lens):
    g = torch.Generator().manual_seed(sum(lens) + qlen)
    q = torch.randn(len(lens) * qlen, 16, 576, generator=g).to(torch.bfloat16)
    case = host_case(lens, 16, "fp8", seed=3 + qlen, permute=not contiguous)
    out, lse = _run(case, q, qlen, 0.08, contiguous)
    _check(case, q, qlen, 0.08, out, lse)


def test_more_sequences_than_the_planner_sorts():
    lens = [(7 * i) % 90 for i in range(300)]
    q = torch.randn(600, 16, 576, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
    case = host_case(lens, 16, "fp8", seed=9)
    out, lse = _run(case, q, 2, 0.08)
    _check(case, q, 2, 0.08, out, lse)


def test_scores_that_climb():
    """Scores that climb by 25 log2 units per tile, past the fp8 range of P: every half
    tile needs its own exponent (the second pass: test_gpu_second_pass.py)."""
    g = torch.Generator().manual_seed(17)
    lens, qlen = [700, 130, 5], 4
    T = sum(lens)
    q = torch.randn(len(lens) * qlen, 16, 576, generator=g)
    q[..., 7] = 40.0
    kv = 0.25 * torch.randn(T, 1, 576, generator=g)
    pos = torch.cat([torch.arange(L) for L in lens]).float()
    kv[:, 0, 7] = 6.0 * torch.floor(pos / 64) - 20.0 + 0.1 * torch.randn(T, generator=g)
    indptr = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    idx = torch.randperm(T, generator=g).to(torch.int32)
    rows = torch.empty_like(kv)
    rows[idx.long()] = kv
    case = case_from_tensors(q[:3].to(torch.bfloat16), rows.to(torch.bfloat16), indptr, idx, "fp8")
    qb = q.to(torch.bfloat16)
    out, lse = _run(case, qb, qlen, 1 / np.sqrt(192))
    assert torch.isfinite(out).all()
    _check(case, qb, qlen, 1 / np.sqrt(192), out, lse)


# sm_scale where the largest score is an odd multiple of 16 in [2^27, 2^28) log2 units:
# half an ulp from its neighbours after adding the 8 that scales P to its fp8 range
TIES = [0.048, 0.0635, 0.0765]


def _log2_score(q_code, kv_code, qs, kvs, sm):
    c = np.float32(qs) * np.float32(kvs) * np.float32(sm) * np.float32(1.4426950408889634)
    return np.float32(q_code * kv_code) * c


@pytest.mark.parametrize("contiguous", [False, True])
@pytest.mark.parametrize("log2k,sm", [(15, s) for s in TIES] + [(10, 0.0712), (16, 0.0712), (18, 0.0712), (30, 0.0712)])
def test_huge_scores(log2k, sm, contiguous):
    """One largest score a sequence, up to 2^43: each row is that key's value."""
    lens, qlen = [200, 70, 700], 3
    _, kv, indptr, idx, _, _ = host_case(lens, 16, "fp8", seed=31, permute=not contiguous)
    q, kv = torch.zeros(len(lens) * qlen, 16, 576, dtype=torch.bfloat16), kv.clone()
    q[..., 575] = 2.0 ** 14
    kv[:, 0, 544:575] = 0.0
    kv[:, 0, 575] = 2.0 ** log2k
    for b in range(len(lens)):  # past the first tile; the factor 4 is exact in e4m3
        kv[idx[int(indptr[b]) + 66].long(), 0, 575] = 2.0 ** (log2k + 2)
    kv[:, 0, :512] *= 2.0 ** (log2k - 1)
    case = case_from_tensors(q[:3], kv, indptr, idx, "fp8")
    _, qs = O.quantize_fp8_per_tensor(O.bf16_tensor_bits(q))
    top = _log2_score(448, 448, qs, case[5]["fp8_scale"], sm)
    if sm in TIES:
        assert 2 ** 27 <= np.ceil(top) < 2 ** 28 and np.ceil(top) // 16 % 2 == 1, top
    out, lse = _run(case, q, qlen, sm, contiguous)
    _, ref, ref_lse = O.reference_path(O.bf16_tensor_bits(q), "fp8", case[5], indptr.numpy(), idx.numpy(), sm,
                                       q_seq_len=qlen, return_lse=True)
    got, unit = out.float().cpu().numpy(), 2.0 ** (log2k - 1)
    assert_close(got / unit, ref / unit)
    assert np.allclose(lse.cpu().numpy(), ref_lse, rtol=1e-2)


@pytest.mark.parametrize("qlen", [2, 4])
@pytest.mark.parametrize("outlier", [1.0, 2.0 ** 12])
def test_pieces_cost_no_precision(qlen, outlier):
    """Rows in up to eight pieces: 1.66e-3 for the bf16 result and 0.55e-3 for the two
    fp8 terms of P, 1.75e-3 together in the 2-norm (a bf16 rounding of the pieces would
    make it 2.2 to 2.35e-3), also where one large value leaves the others small codes."""
    lens = [260, 300, 400, 513, 600, 777, 900, 1024, 64]
    q = torch.randn(len(lens) * qlen, 16, 576, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16)
    _, kv, indptr, idx, _, _ = host_case(lens, 16, "fp8", seed=6)
    kv = kv.clone()
    kv[idx[int(indptr[-2])].long(), 0, 3] = 4.0 * outlier  # in the last sequence, left out below
    case = case_from_tensors(q[:len(lens)], kv, indptr, idx, "fp8")
    out, _ = _run(case, q, qlen, 0.08)
    _, ref = O.reference_path(O.bf16_tensor_bits(q), "fp8", case[5], indptr.numpy(), idx.numpy(), 0.08, q_seq_len=qlen)
    got, ref = out.float().cpu().numpy()[:-qlen], ref[:-qlen]
    assert np.linalg.norm(got - ref) <= 1.95e-3 * np.linalg.norm(ref)


@pytest.mark.parametrize("contiguous", [False, True])
def test_first_tile_of_minus_infinity(contiguous):
    """Scores of a piece's first tile that overflow to -inf, finite ones after it: the
    row is the mean of the finite keys' values."""
    lens, qlen = [120, 100, 77], 3
    _, kv, indptr, idx, _, _ = host_case(lens, 16, "fp8", seed=33, permute=not contiguous)
    q, kv = torch.zeros(len(lens) * qlen, 16, 576, dtype=torch.bfloat16), kv.clone()
    q[..., 575] = 2.0 ** 104
    kv[:, 0, 512:575] = 0.0
    kv[:, 0, :512] *= 2.0 ** 26
    for b in range(len(lens)):  # a sequence is one piece of two tiles
        slots = idx[int(indptr[b]):int(indptr[b + 1])].long()
        kv[slots[:64], 0, 575] = -(2.0 ** 30)
        kv[slots[64:], 0, 575] = -(2.0 ** 20)
    case = case_from_tensors(q[:3], kv, indptr, idx, "fp8")
    out, lse = _run(case, q, qlen, 0.0712, contiguous)
    _, ref = O.reference_path(O.bf16_tensor_bits(q), "fp8", case[5], indptr.numpy(), idx.numpy(), 0.0712,
                              q_seq_len=qlen)
    assert np.isfinite(ref).all() and lse.isfinite().all()
    assert_close(out.float().cpu().numpy() / 2.0 ** 26, ref / 2.0 ** 26)


@pytest.mark.parametrize("qlen", [2, 3, 4])
@pytest.mark.parametrize("contiguous", [False, True])
@pytest.mark.parametrize("back", [1, 2, 3])
@pytest.mark.parametrize("dim", [100, 550])
def test_nan_codes_stay_with_the_rows_that_see_them(qlen, contiguous, back, dim):
    """A NaN code in one of a sequence's last keys (latent and rope dims; the masked
    tail inside one tile, over two, and repeated past the item's end): the rows that
    see the key are NaN throughout, the others as without it."""
    lens = [70, 130, 5, 64, 65, 66, 192]
    q = torch.randn(len(lens) * qlen, 16, 576, generator=torch.Generator().manual_seed(back)).to(torch.bfloat16)
    case = host_case(lens, 16, "fp8", seed=5, permute=not contiguous)
    _, kv, indptr, idx, _, caches = case
    codes = caches["fp8_codes"].copy()
    for b in range(len(lens)):
        codes[int(idx[int(indptr[b + 1]) - back]), dim] = 0x7F if b % 2 else 0xFF
    out, lse = _run((*case[:5], dict(caches, fp8_codes=codes)), q, qlen, 0.08, contiguous)
    _, ref, ref_lse = O.reference_path(O.bf16_tensor_bits(q), "fp8", caches, indptr.numpy(), idx.numpy(), 0.08,
                                       q_seq_len=qlen, return_lse=True)
    sees = np.array([i >= qlen - back for _ in lens for i in range(qlen)])  # row i ends qlen - 1 - i keys early
    assert out[torch.from_numpy(sees).to(DEV)].isnan().all()
    assert_close(out.float().cpu().numpy()[~sees], ref[~sees])
    got, want = lse.cpu().numpy()[~sees], ref_lse[~sees]
    assert np.all(np.abs(got - want) <= 1e-2 + 1e-2 * np.abs(want))


@pytest.mark.parametrize("qlen", [2, 4])
def test_workspace_sizes(qlen):
    """The size of mla_workspace_bytes is accepted (fewer pieces), a byte less refused."""
    lens = [3000, 900, 40]
    q = torch.randn(3 * qlen, 16, 576, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16)
    case = host_case(lens, 16, "fp8", seed=4)
    n = ctypes.c_int64(0)
    _lib.check(_lib.load().mla_workspace_bytes(3 * qlen, 16, 0, ctypes.byref(n)), "mla_workspace_bytes")
    assert ops.workspace_bytes(3 * qlen, 16, "fp8", qlen) >= n.value == ops.workspace_bytes(3 * qlen, 16, "fp8")
    ws = torch.empty(n.value, dtype=torch.uint8, device=DEV)
    out, lse = _run(case, q, qlen, 0.08, ws=ws)
    _check(case, q, qlen, 0.08, out, lse)
    with pytest.raises(_lib.MlaLibraryError):
        _run(case, q, qlen, 0.08, ws=ws[:-256])


def test_captured_calls_follow_their_inputs():
    """The route in a graph, replayed with eager calls between: new queries and other
    lengths in the same buffers give the eager call's bits each time."""
    lens, qlen = [1500, 700, 64, 3], 4
    case = host_case(lens, 16, "fp8", seed=8)
    q, kv, indptr, idx, _, caches = case
    _, kv_data, _, kv_indptr, cfg = device_data(q, kv, indptr, idx, caches, "fp8", 0.08)
    g = torch.Generator(device=DEV).manual_seed(1)
    q = torch.randn(16, 16, 576, device=DEV, generator=g).to(torch.bfloat16)
    ws = torch.empty(ops.workspace_bytes(16, 16, "fp8", qlen), dtype=torch.uint8, device=DEV)
    out = torch.empty(16, 16, 512, dtype=torch.bfloat16, device=DEV)
    lse = torch.empty(16, 16, dtype=torch.float32, device=DEV)

    def call(ws, out, lse):
        ops.decode_fwd(q, kv_data, kv_indptr, cfg["kv_indices"], 0.08, "fp8", out=out, ws=ws, q_seq_len=qlen,
                       return_lse=True, lse=lse)

    call(ws, out, lse)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(ws, out, lse)
    for i, cut in enumerate([0, 100, 700, 1436]):  # the first sequence loses its last keys to the second
        q.normal_(generator=g)
        kv_indptr[1] = lens[0] - cut
        out.fill_(0)
        graph.replay()
        torch.cuda.synchronize()
        want, want_lse = torch.empty_like(out), torch.empty_like(lse)
        call(torch.full_like(ws, 0x5A), want, want_lse)
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)) and torch.equal(lse, want_lse), i
