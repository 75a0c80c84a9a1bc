"""Prefill launches with many query rows (128-query workgroups on the bf16 matrix cores) against the
oracle's gather path and float64 brute force, at the edges of their tiles: query counts around 32 and
128, key counts around 32 and past one refresh of 64 block ids, starts inside blocks, block sizes 16
and 32. 64 heads give a launch the rows it needs from short sequences."""

from __future__ import annotations

import math

import pytest
import torch

from tests.paged_cases import ATOL, RTOL, Scenario
from tokquay_amd import ops

H = 64
SHAPES = [
    ([0, 0, 0, 0, 0], [256, 200, 129, 128, 97]),
    ([1000, 37, 300, 5], [300, 257, 31, 255]),
    ([0, 64, 511, 15, 16, 100], [385, 161, 160, 159, 2, 384]),
    ([3, 200, 31, 2000], [128, 127, 140, 250]),
]


# Relative 2-norm against float64: the six limb products measure 1e-7 to 4e-7 here; with the three largest only,
# which RTOL and ATOL would let pass, it is 6e-6.
NORM = 1e-6


def _sixteen_row(sc, batch, pool):
    """The same rows from the 16-row kernels: sequences without rows beside them leave 128-query workgroups
    too empty to be taken, and change nothing else."""
    qkv, B = sc.packed_qkv(batch.token_index).cuda(), len(sc.starts)
    tables = torch.cat([batch.prefill_block_tables] + [batch.prefill_block_tables] * 2)
    cu = torch.cat([batch.prefill_cu_seqlens, batch.prefill_cu_seqlens[-1:].expand(2 * B)]).contiguous()
    start = torch.cat([batch.prefill_start, torch.zeros_like(batch.prefill_start).repeat(2)])
    out = torch.empty(qkv.size(0), sc.C, device="cuda")
    ops.paged_prefill(out, qkv[:, : sc.C], pool.cuda(), 0, tables, cu, start, batch.prefill_max_q)
    return out.cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("starts,lens", SHAPES)
@pytest.mark.parametrize("bs", [16, 32])
def test_matches_the_oracle(starts, lens, bs):
    sc = Scenario(starts, lens, block_size=bs, n_head=H, seed=sum(lens))
    pool_ref, out_ref = sc.reference()
    pool, out, batch = sc.run_product()
    assert torch.equal(pool, pool_ref)
    torch.testing.assert_close(out, sc.packed_reference(out_ref, batch.token_index), rtol=RTOL, atol=ATOL)
    at = 0
    for want in sc.brute_force(pool_ref):
        got, want = out[at : at + want.shape[0]].view(-1, H, 64).double(), torch.from_numpy(want)
        torch.testing.assert_close(got, want, rtol=RTOL, atol=ATOL)
        assert (got - want).norm() <= NORM * want.norm()
        at += want.shape[0]
    # The launch is the 128-query one: its bits are not those of the 16-row kernels.
    other = _sixteen_row(sc, batch, pool)
    torch.testing.assert_close(out, other, rtol=RTOL, atol=ATOL)
    assert not torch.equal(out, other)


@pytest.mark.gpu
def test_too_few_rows_stay_on_the_16_row_kernels():
    """What the check above rests on: a launch that is not well filled has the 16-row kernels' bits already."""
    sc = Scenario([0, 64, 511, 15, 16], [385, 161, 160, 159, 2], n_head=H, seed=5)
    pool, out, batch = sc.run_product()
    assert torch.equal(out, _sixteen_row(sc, batch, pool))


@pytest.mark.gpu
def test_dispatch_order_keeps_the_bits_and_bad_metadata_is_reported():
    sc = Scenario(*SHAPES[0], n_head=H)
    pool, out, batch = sc.run_product()
    qkv, gpu_pool = sc.packed_qkv(batch.token_index).cuda(), pool.cuda()
    err = torch.zeros(1, dtype=torch.int32, device="cuda")

    def run(tables, order):
        got = torch.empty(qkv.size(0), sc.C, device="cuda")
        ops.paged_prefill(got, qkv[:, : sc.C], gpu_pool, 0, tables, batch.prefill_cu_seqlens, batch.prefill_start,
                          batch.prefill_max_q, d_error=err, seq_order=order)  # fmt: skip
        return got.cpu()

    for perm in ([4, 3, 2, 1, 0], [2, 0, 4, 1, 3]):
        assert torch.equal(run(batch.prefill_block_tables, torch.tensor(perm, dtype=torch.int32, device="cuda")), out)
    assert torch.equal(run(batch.prefill_block_tables, None), out) and int(err) == 0
    tables = batch.prefill_block_tables.clone()
    tables[1, 3] = gpu_pool.size(0)  # a block past the pool: its keys count as zeros, the others run on
    got = run(tables, None)
    assert int(err) == 1 and got.isfinite().all()
    keep = torch.ones(out.size(0), dtype=torch.bool)
    keep[256 + 48 : 456] = False  # sequence 1's rows from the bad block's first position on
    assert torch.equal(got[keep], out[keep])


@pytest.mark.gpu
def test_non_finite_keys_follow_fp32_softmax():
    """An infinite key gives a query that sees it what fp32 softmax gives (NaN, or no weight), and the queries
    and heads that do not see it keep their bits, those of the same wave too."""
    starts, lens = SHAPES[0]
    sc = Scenario(starts, lens, n_head=H)
    sc.k[0, 3, 100, 7] = float("inf")
    sc.k[2, 5, 40, 0] = float("-inf")
    pool, out, batch = sc.run_product()
    clean, want, _ = Scenario(starts, lens, n_head=H).run_product()
    unseen = torch.ones(want.size(0), H, dtype=torch.bool)
    same = want.view(-1, H, 64)
    want = want.double().view(-1, H, 64).clone()
    at = [0, 256, 456, 585, 713]
    for b, h, pos in ((0, 3, 100), (2, 5, 40)):
        q, k, v = (t[b, h].double() for t in (sc.q, sc.k, sc.v))
        unseen[at[b] + pos : at[b] + lens[b], h] = False
        for t in range(pos, lens[b]):
            p = torch.softmax(k[: t + 1] @ q[t] / math.sqrt(64), 0)
            want[at[b] + t, h] = p @ v[: t + 1]
    got = out.double().view(-1, H, 64)
    assert torch.equal(out.view(-1, H, 64)[unseen], same[unseen])
    assert want.isnan().any() and want[at[0] + 100 : at[0] + 256, 3].isfinite().any()
    torch.testing.assert_close(got, want, rtol=RTOL, atol=ATOL, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("bs", [16, 32])
def test_tiny_operands_keep_fp32(bs):
    """Values below 2^-110, whose limbs do not add up to them, and tiny queries against huge keys (and the
    reverse) give what fp32 gives, dims of zeros give zeros; heads without any keep their bits."""
    starts, lens = SHAPES[1]
    sc = Scenario(starts, lens, block_size=bs, n_head=H)
    _, clean, _ = Scenario(starts, lens, block_size=bs, n_head=H).run_product()
    for h, scale in ((3, 1e-34), (17, 1e-36), (40, 1e-39)):
        sc.v[:, h] *= scale
        for b, s in enumerate(starts):
            for p in range(s):
                sc.pool[sc.tables[b][p // bs], 0, 1, h, p % bs] *= scale
    sc.v[:, 5, ::2, :7] = 0.0
    for h, scale in ((20, 1e34), (50, 1e-34)):
        sc.q[:, h] *= scale
        sc.k[:, h] /= scale
        for b, s in enumerate(starts):
            for p in range(s):
                sc.pool[sc.tables[b][p // bs], 0, 0, h, p % bs] /= scale
    pool, out, batch = sc.run_product()
    same = [h for h in range(H) if h not in (3, 5, 17, 20, 40, 50)]
    got = out.view(-1, H, 64)
    assert torch.equal(got[:, same], clean.view(-1, H, 64)[:, same])
    at = 0
    for want in sc.brute_force(pool):
        have = got[at : at + want.shape[0]].double()
        want = torch.from_numpy(want)
        for h, scale in ((3, 1e-34), (5, 1.0), (17, 1e-36), (20, 1.0), (40, 1e-39), (50, 1.0)):
            err = (have[:, h] - want[:, h]).abs().max()
            assert err <= 1e-5 * scale + 2.0**-140, (h, float(err))  # 2^-140: subnormal products of fp32
        at += want.shape[0]
