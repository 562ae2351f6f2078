"""Which calls of the MLP and the head the few-row kernels take: those that were measured to gain by
them, at the lines of the rule."""
import pytest
import torch

from kernels import few_rows


@pytest.mark.parametrize("rows,vocab,hidden,pays", [
    (1, 32000, 896, True), (16, 32000, 768, True), (16, 32000, 512, False), (17, 32000, 1536, False),
    (33, 64000, 1536, False), (17, 151936, 1536, True), (40, 151936, 1536, True),
    (48, 151936, 1536, False), (64, 32000, 2048, False), (16, 151936, 2048, True)])
def test_head(rows, vocab, hidden, pays):
    w = torch.empty(vocab, hidden, dtype=torch.bfloat16, device="meta")
    assert few_rows.linear_pays(rows, w) == pays


@pytest.mark.parametrize("rows,hidden,pays", [(1, 256, True), (64, 1536, True), (65, 1536, False),
                                              (32, 2048, True), (33, 2048, False), (33, 1792, False)])
def test_mlp(rows, hidden, pays):
    assert few_rows.mlp_pays(rows, hidden) == pays
