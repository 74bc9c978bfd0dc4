"""Which calls run a sequence's causal rows together (ops._rows_together): both sides
of every line of the rule, and calls measured to be faster one way or the other."""
import pytest
import torch

from amd_optimization_challenge_amd import ops, submission


@pytest.mark.parametrize("qlen,seqs,tokens,indexed", [
    # (a pass per row was faster)
    (4, 1, 32768, True), (4, 1, 32768, False), (2, 1, 1 << 20, False), (4, 2, 1 << 20, False), (3, 2, 32768, True),
    (2, 4, 1 << 20, False), (3, 8, 32768, True), (4, 8, 32768, False), (2, 16, 32768, True), (2, 32, 32768, False),
    (4, 60, 9600, True), (2, 300, 65400, False), (3, 257, 49087, False), (2, 1000, 131072, False),
    # one token, sequence or row below each line
    (2, 192, 32767, True), (2, 191, 32768, True), (4, 96, 10922, True), (3, 383, 32768, True), (2, 384, 32768, True),
    (4, 2, (1 << 18) - 1, True), (3, 3, 1 << 20, False), (3, 257, (1 << 17) - 1, True),
    (3, 257, (3 << 16) - 1, False), (2, 24, (3 << 15) - 1, True), (4, 23, 32768, True), (2, 256, 98304, False),
    (4, 3, 43690, True)])
def test_a_pass_per_row(qlen, seqs, tokens, indexed):
    assert not ops._rows_together(qlen, 16, 0, tokens, seqs, indexed)


@pytest.mark.parametrize("qlen,seqs,tokens,indexed", [
    (4, 32, 139000, True), (2, 128, 384000, True), (4, 280, 280000, True), (4, 300, 262144, False), (4, 16, 65536, False),
    (3, 2, 1 << 18, True), (2, 192, 32768, True), (4, 96, 10923, True), (3, 384, 32768, True), (4, 2, 1 << 18, True),
    (4, 3, 43691, False), (3, 257, 1 << 17, True), (3, 257, 3 << 16, False), (2, 24, 3 << 15, True),
    (4, 24, 32768, False), (2, 256, 1 << 17, False), (4, 3, 43691, True)])
def test_rows_together(qlen, seqs, tokens, indexed):
    assert ops._rows_together(qlen, 16, 0, tokens, seqs, indexed)


@pytest.mark.parametrize("qlen,heads,mode", [(1, 16, 0), (5, 16, 0), (4, 128, 0), (4, 16, 1), (4, 16, 2), (4, 16, 3)])
def test_what_the_kernel_does_not_take(qlen, heads, mode):
    assert not ops._rows_together(qlen, heads, mode, 1 << 30, 32, True)


@pytest.mark.parametrize("kv_seq_len,tokens,indexed,together", [
    (160, 9600, True, False), (160, 1 << 17, True, False), (160, 1 << 17, False, False),  # room to spare
    (None, 9600, True, False), (None, 1 << 17, True, True), (0, 1 << 17, True, True), (4000, 1 << 17, True, True),
    (4000, 1 << 17, False, True)])
def test_tokens_are_bounded_by_the_longest_sequence(monkeypatch, kv_seq_len, tokens, indexed, together):
    """Sixty sequences x 4 rows through custom_kernel: a cache or an index list larger
    than the sequences fill does not take a short call to the route of a long one."""
    called = []
    monkeypatch.setattr(ops, "_require_cuda", lambda *a: None)
    monkeypatch.setattr(ops, "workspace", lambda *a: torch.empty(0, dtype=torch.uint8))
    monkeypatch.setattr(ops, "_call", lambda name, *a: called.append(name))
    monkeypatch.setattr(submission, "_out_cache", {})
    monkeypatch.setattr(ops, "_ws_cache", {})
    kv = {"fp8": (torch.empty((1, 1, 576), dtype=torch.uint8).expand(tokens, 1, 576), torch.ones(1))}
    cfg = dict(q_seq_len=4, kv_indices=torch.zeros(1, dtype=torch.int32).expand(tokens) if indexed else None)
    if kv_seq_len is not None:
        cfg["kv_seq_len"] = kv_seq_len
    submission.custom_kernel((torch.zeros((240, 16, 576), dtype=torch.bfloat16), kv, None,
                              torch.zeros(61, dtype=torch.int32), cfg))
    assert called == ["mla_decode_fwd_rows" if together else "mla_decode_fwd"]
