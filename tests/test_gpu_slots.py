"""Selections whose valid slots are scattered: the per-row merges read only the slots a row has."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import msa_triton_amd as msa
from oracle import msa_oracle as O
from tests.helpers import check_bf16_stated, cu_tensor, np64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,groups,dimension,topk", [(3, 1, 64, 40), (6, 2, 136, 33), (8, 2, 128, 7)])
def test_scattered_slots_against_fp64(heads, groups, dimension, topk, device):
    """Valid ids at random slots among -1 and future ids (more than 32 slots, and heads of two
    tokens sharing a wave where their number is odd; some rows with no valid slot at all)."""
    lengths, block = [230, 1, 74], 4
    rng = np.random.default_rng(heads * topk)
    total = sum(lengths)
    ids = np.full((total, groups, topk), -1, dtype=np.int32)
    at = 0
    for length in lengths:
        for pos in range(length):
            own = pos // block
            for g in range(groups):
                n = int(rng.integers(0, min(topk, own + 1) + 1))
                row = np.concatenate([rng.permutation(own + 1)[:n],
                                      rng.choice([-1, own + 1, own + 7], size=topk - n)])
                ids[at + pos, g] = rng.permutation(row)
        at += length
    gen = torch.Generator().manual_seed(11)
    q, k, v, dout = (torch.randn(total, n, dimension, generator=gen).bfloat16()
                     for n in (heads, groups, groups, heads))
    cu = cu_tensor(lengths)
    out, lse, dq, dk, dv = O.sparse_attention(np64(q), np64(k), np64(v), ids, cu.numpy(), block_size=block, scale=None,
                                              dout=np64(dout))
    leaves = [x.to(device).requires_grad_() for x in (q, k, v)]
    ids_d = torch.from_numpy(ids).to(device)
    got, got_lse = msa.m3_sparse_attention(*leaves, ids_d, cu.to(device), max(lengths), block_size=block,
                                           return_lse=True)
    got.backward(dout.to(device))
    with torch.no_grad():  # forward only: no row state is kept
        again = msa.m3_sparse_attention(*leaves, ids_d, cu.to(device), max(lengths), block_size=block)
    assert torch.equal(again, got)
    np.testing.assert_allclose(got_lse.detach().cpu().numpy(), lse, atol=1e-5, rtol=1e-5)
    for actual, ref, what in zip((got, *(x.grad for x in leaves)), (out, dq, dk, dv), ("out", "dq", "dk", "dv")):
        check_bf16_stated(actual.detach(), ref, what)
