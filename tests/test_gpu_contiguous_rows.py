"""Contiguous 16-head caches: whole tiles are gathered from one scalar base per
tile, partial tiles and rows too far apart for 32-bit lane offsets (a stride
above 2^24 bytes) by an address per row.  Same plan, same rows, so the far cache
gives the near one's bits, and the near one is checked against the oracle."""
import math

import pytest
import torch

import mla_cases as M
from amd_optimization_challenge_amd import custom_kernel
from oracle import mla_oracle as O

pytestmark = pytest.mark.gpu
FAR = (1 << 24) + 16  # bytes between rows, past the near-row rule


def _far(t, rows):
    """The same rows FAR bytes apart (uint8 view)."""
    row = t.reshape(rows, -1).view(torch.uint8)
    buf = torch.empty(rows * FAR, dtype=torch.uint8, device=t.device)
    out = buf.as_strided((rows, row.shape[1]), (FAR, 1))
    out.copy_(row)
    return out


@pytest.mark.parametrize("mode", ["fp8", "mxfp4", "mxfp4k_fp8v", "bf16"])
@pytest.mark.parametrize("lens", [[1], [64], [63, 2], [65, 1], [128], [1, 64, 127]])
def test_near_and_far_rows(mode, lens):
    case = M.host_case(lens, 16, mode, seed=sum(lens), permute=False)
    q, kv, indptr, idx, qb, caches = case
    sm = 1 / math.sqrt(192)
    data = M.device_data(q, kv, indptr, idx, caches, mode, sm, pass_indices=False)
    near = custom_kernel(data).clone()
    kvd, T = data[1], kv.shape[0]
    if "fp8" in kvd:
        kvd["fp8"] = (_far(kvd["fp8"][0], T), kvd["fp8"][1])
    if "mxfp4" in kvd:
        kvd["mxfp4"] = (_far(kvd["mxfp4"][0], T), kvd["mxfp4"][1])
    if mode == "bf16":
        kvd["bf16"] = _far(kvd["bf16"], T).view(torch.bfloat16)
    far = custom_kernel(data)
    assert torch.equal(near.view(torch.int16), far.view(torch.int16))
    if mode != "bf16":
        _, ref = O.reference_path(qb, mode, caches, indptr.numpy(), idx.numpy(), sm)
        M.assert_close(near.float().cpu().numpy(), ref)
