"""Key-split prefill launches around the table width up to which K tiles are loaded in place (two key tiles)
against the oracle's gather path and float64 brute force: tables of one to three 16-key tiles, every key split,
block sizes 16 and 32."""

from __future__ import annotations

import pytest
import torch

from tests.paged_cases import ATOL, RTOL, Scenario

# (heads, sequences): heads x row tiles x sequences choose the waves per tile (8, 4, 2).
SPLITS = [(2, 3), (64, 4), (64, 9)]


@pytest.mark.gpu
@pytest.mark.parametrize("heads,seqs", SPLITS)
@pytest.mark.parametrize("bs", [16, 32])
@pytest.mark.parametrize("longest", [2, 16, 17, 31, 32, 33, 48])
def test_matches_the_oracle(heads, seqs, bs, longest):
    lens = [max(2, longest - 5 * i) for i in range(seqs)]
    starts = [0 if i % 2 else min(i, longest - n) for i, n in enumerate(lens)]
    sc = Scenario(starts, lens, block_size=bs, n_head=heads, seed=longest + seqs)
    pool_ref, out_ref = sc.reference()
    pool, out, batch = sc.run_product()
    assert torch.equal(pool, pool_ref)
    torch.testing.assert_close(out, sc.packed_reference(out_ref, batch.token_index), rtol=RTOL, atol=ATOL)
    at = 0
    for want in sc.brute_force(pool_ref):
        got = out[at : at + want.shape[0]].view(-1, heads, 64).double()
        want = torch.from_numpy(want)
        assert (got - want).norm() <= 1e-6 * want.norm()
        at += want.shape[0]
