"""Which calls run a sequence's causal rows together (ops._rows_together): both sides
of every line of the rule, and calls measured to be faster one way or the other."""
import pytest

from amd_optimization_challenge_amd import ops


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
