"""Prefill and mixed launches with block size 8 (a key tile is two blocks) against the oracle's gather path and
float64 brute force: key counts around the 8-row blocks, the 16-key tiles and a refresh of 64 block ids, starts
inside blocks, every number of waves per query tile and two tiles per wave, decode rows beside."""

from __future__ import annotations

import pytest
import torch

from tests.paged_cases import ATOL, RTOL, Scenario
from tokquay_amd import ops

# (heads, starts, lens): heads x ceil(longest / 16) x sequences row tiles choose the waves per tile.
SHAPES = [
    (2, [0, 0, 0, 0, 0, 3], [1, 2, 7, 8, 9, 5]),  # one or two blocks
    (2, [0, 7, 8, 15, 500, 505], [15, 16, 17, 33, 12, 23]),  # 8 waves a tile; past 64 ids
    (12, [16, 509, 9, 1000], [100, 64, 31, 128]),  # 4 waves
    (12, [0, 100, 33, 250, 7], [129, 200, 140, 100, 199]),  # 2 waves
    (64, [0, 24, 510], [300, 257, 131]),  # one wave
    (64, [1, 300], [1030, 1020]),  # one wave, two tiles of a sequence each
    (12, [40, 600, 0, 12], [1, 1, 1, 90]),  # decode rows beside
    (12, [514, 7, 31, 500, 3], [1, 1, 200, 190, 180]),
]


@pytest.mark.gpu
@pytest.mark.parametrize("heads,starts,lens", SHAPES)
def test_matches_the_oracle(heads, starts, lens):
    sc = Scenario(starts, lens, block_size=8, n_head=heads, seed=sum(lens))
    pool_ref, out_ref = sc.reference()
    pool, out, batch = sc.run_product()
    assert torch.equal(pool, pool_ref)
    torch.testing.assert_close(out, sc.packed_reference(out_ref, batch.token_index), rtol=RTOL, atol=ATOL)
    at = 0
    for want in sc.brute_force(pool_ref):
        got = out[at : at + want.shape[0]].view(-1, heads, 64)
        torch.testing.assert_close(got.double(), torch.from_numpy(want), rtol=RTOL, atol=ATOL)
        at += want.shape[0]


@pytest.mark.gpu
@pytest.mark.parametrize("entry", [4, 5])
def test_a_bad_block_counts_as_zeros(entry):
    """Either block of a pair past the pool: reported, the rows before it unchanged, nothing non-finite."""
    sc = Scenario([0], [100], block_size=8, n_head=2)
    pool, out, batch = sc.run_product()
    qkv, gpu_pool = sc.packed_qkv(batch.token_index).cuda(), pool.cuda()
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    tables = batch.prefill_block_tables.clone()
    tables[0, entry] = gpu_pool.size(0)
    got = torch.empty(100, sc.C, device="cuda")
    ops.paged_prefill(got, qkv[:, : sc.C], gpu_pool, 0, tables, batch.prefill_cu_seqlens, batch.prefill_start,
                      batch.prefill_max_q, d_error=err)  # fmt: skip
    got = got.cpu()
    assert int(err) == 1 and got.isfinite().all()
    assert torch.equal(got[: 8 * entry], out[: 8 * entry]) and not torch.equal(got[8 * entry :], out[8 * entry :])
