"""fp32 attention on the FP64 matrix products against the FP64 oracle, and where it ends."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import msa_triton_amd as msa
from oracle import msa_oracle as O
from tests.helpers import cu_tensor, np64, random_selection

pytestmark = pytest.mark.gpu


def _close_f32(actual, expected, what):
    """FP64 arithmetic rounded once to fp32: within 2^-23 of each value, plus the FP64 sums'
    own rounding (1e-11: 2^-53 of sums of up to ~1e4 in magnitude)."""
    act = actual.detach().cpu().numpy().astype(np.float64)
    worst = np.max(np.abs(act - expected) - 2.0 ** -23 * np.abs(expected))
    assert worst <= 1e-11, f"{what}: {worst}"


_FEW = [1] * 9 + [2, 0, 3, 5, 130, 1, 33]


@pytest.mark.parametrize("dimension", [32, 64, 96, 128])
@pytest.mark.parametrize("lengths,groups,ratio,block,topk", [
    # tiles with fewer than 100 (row, key) pairs (the KV pass's vector kernel) beside others
    (_FEW, 2, 4, 16, 3), (_FEW, 1, 1, 128, 2), ([60, 41], 2, 1, 5, 4), ([100], 1, 6, 1, 8),
    ([1], 1, 8, 128, 1), ([17, 0, 15, 130], 2, 4, 16, 3), ([300, 33], 1, 8, 128, 2), ([95, 64], 2, 3, 5, 6),
    ([210], 1, 5, 100, 2), ([257], 2, 8, 200, 1), ([40, 90], 2, 2, 24, 3), ([70], 1, 12, 16, 4),
])
def test_f32_forward_backward_against_fp64(lengths, groups, ratio, block, topk, dimension, device):
    """3 to 8 heads per group (matrix products in every pass), and 2 and 12 (the query passes on
    the vector unit); tiles of fewer than 16 keys and rows, blocks above 128 keys, slots with
    -1 and future ids."""
    gen = torch.Generator().manual_seed(dimension + block)
    total = sum(lengths)
    q, k, v, dout = (torch.randn(total, n, dimension, generator=gen)
                     for n in (groups * ratio, groups, groups, groups * ratio))
    ids = random_selection(total, groups, topk, lengths, block, 1, gen)
    ids[2::5, :, -1] = 1000  # after every query
    cu = cu_tensor(lengths)
    out, lse, dq, dk, dv = O.sparse_attention(np64(q), np64(k), np64(v), ids.numpy(), cu.numpy(), block_size=block,
                                              scale=None, dout=np64(dout))
    leaves = [x.to(device).requires_grad_() for x in (q, k, v)]
    got, got_lse = msa.m3_sparse_attention(*leaves, ids.to(device), cu.to(device), max(lengths), block_size=block,
                                           return_lse=True)
    got.backward(dout.to(device))
    finite = np.isfinite(lse)
    assert np.array_equal(finite, np.isfinite(got_lse.cpu().numpy()))
    _close_f32(got_lse[torch.from_numpy(finite).to(device)], lse[finite], "lse")
    for actual, ref, what in zip((got, *(x.grad for x in leaves)), (out, dq, dk, dv), ("out", "dq", "dk", "dv")):
        _close_f32(actual, ref, what)


def test_f32_rows_off_16_byte_boundaries_equal_aligned_ones(device):
    """The same values one element past a 16-byte boundary take the vector kernels, forward and
    backward: both within one fp32 rounding of the same FP64 result."""
    gen = torch.Generator().manual_seed(3)
    lengths, groups, ratio, dimension, block, topk = [150, 37], 2, 4, 64, 32, 3
    total = sum(lengths)
    values = [torch.randn(total, n, dimension, generator=gen) for n in (groups * ratio, groups, groups)]
    ids = random_selection(total, groups, topk, lengths, block, 1, gen).to(device)
    cu = cu_tensor(lengths, device)

    def shifted(x):
        flat = torch.empty(x.numel() + 1, device=device)
        flat[1:] = x.to(device).flatten()
        return flat[1:].view(x.shape)

    dout = torch.randn(values[0].shape, generator=gen)
    results = []
    for place in (lambda x: x.to(device), shifted):
        leaves = [place(x).requires_grad_() for x in values]
        out = msa.m3_sparse_attention(*leaves, ids, cu, max(lengths), block_size=block)
        results.append([out.detach(), *torch.autograd.grad(out, leaves, place(dout))])
    for a, b in zip(*results):  # (1e-11: the FP64 sums' own rounding, as above)
        assert bool(((a - b).abs() <= 2.0 ** -22 * b.abs() + 1e-11).all())


@pytest.mark.parametrize("dimension", [32, 64, 96, 128])
@pytest.mark.parametrize("tensor", ["q", "dout"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_f32_non_finite_query_row_stays_with_the_keys_it_sees(value, tensor, dimension, device):
    """A token whose q or dO row (one head) holds a NaN or an infinity: dK and dV of the keys it does
    not see, later ones of its own block among them, are those of the call in which its dO is zero."""
    gen = torch.Generator().manual_seed(dimension)
    lengths, groups, ratio, block, topk = [70, 41], 2, 4, 32, 2
    total, bad = sum(lengths), 37  # token 37: position 5 of its block of 32 keys, tile of 16 keys 32..47
    q, k, v, dout = (torch.randn(total, n, dimension, generator=gen)
                     for n in (groups * ratio, groups, groups, groups * ratio))
    ids = random_selection(total, groups, topk, lengths, block, 1, gen)
    cu = cu_tensor(lengths)
    without = dout.clone()
    without[bad] = 0.0
    _, _, _, dk, dv = O.sparse_attention(np64(q), np64(k), np64(v), ids.numpy(), cu.numpy(), block_size=block,
                                         scale=None, dout=np64(without))
    dout[bad] = 0.0
    (q if tensor == "q" else dout)[bad, 1, dimension // 2] = value
    leaves = [x.to(device).requires_grad_() for x in (q, k, v)]
    got = msa.m3_sparse_attention(*leaves, ids.to(device), cu.to(device), max(lengths), block_size=block)
    got.backward(dout.to(device))
    seen = torch.zeros(total, dtype=torch.bool)
    seen[:bad + 1] = True  # (a superset: both selected blocks are earlier keys)
    for leaf, ref, what in ((leaves[1], dk, "dk"), (leaves[2], dv, "dv")):
        _close_f32(leaf.grad[~seen.to(device)], ref[~seen.numpy()], what)
        _close_f32(leaf.grad[:, 1], ref[:, 1], what + " of the other group")


@pytest.mark.parametrize("dimension", [32, 64, 96, 128])
def test_f32_infinite_value_at_the_end_of_a_partial_tile(dimension, device):
    """V = inf at the last key of a partial tile of 16 keys: inf in the output of the rows that see it
    (not the NaN that 0 times a repetition of that key would give), the rest as without it."""
    gen = torch.Generator().manual_seed(dimension)
    lengths, groups, ratio, block = [21], 1, 4, 21
    total = sum(lengths)
    q, k, v = (torch.randn(total, n, dimension, generator=gen) for n in (ratio, groups, groups))
    ids = torch.zeros(total, groups, 1, dtype=torch.int32)
    cu = cu_tensor(lengths)
    v[20, 0, 3] = 0.0
    out, _, _, _, _ = O.sparse_attention(np64(q), np64(k), np64(v), ids.numpy(), cu.numpy(), block_size=block,
                                         scale=None, dout=np64(q))
    v[20, 0, 3] = float("inf")  # tile of keys 16..20, seen by token 20 only
    got = msa.m3_sparse_attention(*(x.to(device) for x in (q, k, v)), ids.to(device), cu.to(device), total,
                                  block_size=block)
    assert bool((got[20, :, 3] == float("inf")).all())
    rest = torch.ones(total, ratio, dimension, dtype=torch.bool)
    rest[20, :, 3] = False
    _close_f32(got[rest.to(device)], out[rest.numpy()], "out")


@pytest.mark.parametrize("dimension", [32, 64, 96, 128])
def test_f32_infinite_value_counts_once_in_the_row_statistics(dimension, device):
    """A row whose only infinite dP is that of the last key of a partial tile of 16 keys: its delta
    (row_state[3]) is inf, not the NaN that a repetition of that key with weight 0 would give."""
    total, ratio = 17, 4
    q = torch.zeros(total, ratio, dimension)
    k = torch.zeros(total, 1, dimension)
    v = torch.zeros(total, 1, dimension)
    v[16, 0, 0] = float("inf")  # second tile: one key of 16, seen by token 16 only
    out = torch.zeros(total, ratio, dimension)
    dout = torch.zeros(total, ratio, dimension)
    dout[16, :, 0] = 1.0
    from msa_triton_amd.layout import prepare_sequences
    from msa_triton_amd.sparse_attention import _attn_backward

    seqs = prepare_sequences(torch.tensor([0, total], dtype=torch.int32, device=device), block_size=32)
    state = torch.zeros(total, ratio, 4, dtype=torch.float64, device=device)
    state[..., 0] = torch.arange(1, total + 1, dtype=torch.float64, device=device).log()[:, None]  # lse of equal logits
    state[..., 1] = 1.0
    ids = torch.zeros(total, 1, 1, dtype=torch.int32, device=device)
    _attn_backward(*(x.to(device) for x in (q, k, v)), ids, seqs.cu_seqlens, out.to(device), state, dout.to(device),
                   seqs.meta, 32, 1.0, seqs, True, False, False)
    assert bool((state[16, :, 3] == float("inf")).all())


@pytest.mark.parametrize("dimension", [32, 128])
def test_f32_tile_of_minus_infinite_logits(dimension, device):
    """Keys whose logits are -inf have weight 0, also when they fill the first tile of 16 keys: the
    output and lse are those of the remaining keys, and 0 and -inf where no other key is visible."""
    gen = torch.Generator().manual_seed(dimension)
    total, ratio, block = 90, 4, 128
    q, k, v = (torch.randn(total, n, dimension, generator=gen) for n in (ratio, 1, 1))
    q = q.abs()
    ids = torch.zeros(total, 1, 1, dtype=torch.int32)
    cu = cu_tensor([total])
    k[:16, 0, 0] = -1e30  # (for the oracle: exp of its logits is 0 as well)
    out, lse, _, _, _ = O.sparse_attention(np64(q), np64(k), np64(v), ids.numpy(), cu.numpy(), block_size=block,
                                           scale=None, dout=np64(q))
    k[:16, 0, 0] = -float("inf")
    got, got_lse = msa.m3_sparse_attention(*(x.to(device) for x in (q, k, v)), ids.to(device), cu.to(device), total,
                                           block_size=block, return_lse=True)
    assert bool((got[:16] == 0).all()) and bool((got_lse[:16] == -float("inf")).all())
    _close_f32(got[16:], out[16:], "out")
    _close_f32(got_lse[16:], lse[16:], "lse")


def _grads(q, k, v, dout, ids, cu, longest, block):
    leaves = [x.clone().requires_grad_() for x in (q, k, v)]
    msa.m3_sparse_attention(*leaves, ids, cu, longest, block_size=block).backward(dout)
    return [x.grad for x in leaves]


@pytest.mark.parametrize("block", [1 << 20, 2 ** 31 - 17, 2 ** 31 - 1])
def test_f32_backward_with_a_block_far_above_the_sequences(block, device):
    """The KV pass's workgroups follow the tokens, not the block size: the same bits as with blocks
    of the longest sequence, up to the largest block size."""
    gen = torch.Generator(device=device).manual_seed(1)
    lengths, ratio, dimension = [70, 3, 0, 41], 4, 64
    total = sum(lengths)
    q, k, v, dout = (torch.randn(total, n, dimension, generator=gen, device=device) for n in (ratio, 1, 1, ratio))
    ids = torch.zeros(total, 1, 1, dtype=torch.int32, device=device)
    cu = cu_tensor(lengths, device)
    for a, b in zip(_grads(q, k, v, dout, ids, cu, 70, block), _grads(q, k, v, dout, ids, cu, 70, 70)):
        assert torch.equal(a, b)


def test_f32_backward_does_not_take_the_number_of_blocks_from_the_caller(device):
    """total_blocks of msa_attn_bwd describes the edge rows of the KV-major kernels; the fp32 pass
    writes every key whatever it says."""
    from msa_triton_amd import _lib
    from msa_triton_amd.k2q import build_k2q_csr

    gen = torch.Generator(device=device).manual_seed(2)
    lengths, ratio, dimension, block = [70, 41], 4, 64, 16
    total = sum(lengths)
    q, k, v, dout = (torch.randn(total, n, dimension, generator=gen, device=device) for n in (ratio, 1, 1, ratio))
    ids = random_selection(total, 1, 2, lengths, block, 1, torch.Generator().manual_seed(2)).to(device)
    cu = cu_tensor(lengths, device)
    want = _grads(q, k, v, dout, ids, cu, 70, block)
    csr = build_k2q_csr(ids, cu, block_size=block)
    out, lse = torch.empty_like(q), torch.empty(total, ratio, device=device)
    state = torch.empty(total, ratio, 4, dtype=torch.float64, device=device)
    scale, lib, stream = dimension ** -0.5, _lib.lib(), _lib.stream_of(q.device)
    sizes = (2, total, ratio, 1, dimension, 2, block, scale)
    assert lib.msa_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), 0, ids.data_ptr(), cu.data_ptr(), *sizes, None, 0,
                            None, None, None, None, 0, out.data_ptr(), lse.data_ptr(), state.data_ptr(), None,
                            stream) == 0
    for total_blocks in (0, 1):
        got = [torch.full_like(x, float("nan")) for x in (q, k, v)]
        assert lib.msa_attn_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), 0, out.data_ptr(), dout.data_ptr(),
                                state.data_ptr(), None, ids.data_ptr(), cu.data_ptr(), *sizes,
                                csr.cu_block_lens.data_ptr(), total_blocks, csr.row_ptr.data_ptr(),
                                csr.query_indices.data_ptr(), csr.slot_indices.data_ptr(),
                                *(x.data_ptr() for x in got), None, 0, stream) == 0
        for a, b, what in zip(got, want, ("dq", "dk", "dv")):
            assert bool(((a - b).abs() <= 2.0 ** -22 * b.abs() + 1e-11).all()), (total_blocks, what)
