"""The prefill's split work list (LongPlan.work, split_rows): every key tile of every row tile in exactly one
piece, slots and merge entries that agree, on the host."""
import numpy as np
import pytest
import torch

from kvq import cuda_kernels as ck

ROWS = 128


def _lists(q_lens, seq_lens, group, hkv, d, fill=256, max_parts=64):
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    plan = ck.plan_long(cu, seq_lens, 16)
    req, row, keys = plan._row_tiles(group, ROWS)
    tiles = np.maximum(-(-keys // ck.PREFILL_TILE), 1)
    return plan, req, row, keys, tiles, ck.split_rows(req, row, tiles, hkv, d, fill, max_parts)


def test_row_tiles_match_the_loop():
    """The vectorised row tiles: rows of `rows` (token, q head) pairs, the keys the last of them reads."""
    q_lens, seq_lens = [100, 3, 37, 700, 9], [100, 9, 517, 2000, 5000]
    plan, req, row, keys, _, _ = _lists(q_lens, seq_lens, 7, 4, 128)
    want = []
    for r, (Q, L) in enumerate(zip(q_lens, seq_lens)):
        if Q > ck.SHORT_Q:
            for r0 in range(0, Q * 7, ROWS):
                want.append((r, r0, L - Q + 1 + min(Q - 1, (r0 + ROWS - 1) // 7)))
    assert list(zip(req.tolist(), row.tolist(), keys.tolist())) == want
    tr, tw = plan.tiles(7, "cpu", rows=ROWS)
    order = np.argsort(-keys, kind="stable")
    assert tr.tolist() == req[order].tolist() and tw.tolist() == row[order].tolist()
    assert tr.dtype == torch.int32


@pytest.mark.parametrize("batch", [([512], [8192]), ([16], [16384]), ([64, 1, 200], [8192, 50, 300]),
                                   ([9, 700, 333], [4000, 700, 2500]), ([40], [70000])])
@pytest.mark.parametrize("group,hkv,d", [(7, 4, 128), (4, 8, 128), (1, 16, 64), (6, 1, 64)])
def test_split_rows_covers_every_tile_once(batch, group, hkv, d):
    _, req, row, keys, tiles, got = _lists(*batch, group, hkv, d)
    if got is None:
        assert req.shape[0] * hkv >= 1
        return
    preq, prow, piece, slot, merge, longest, slots = got
    part, parts = piece & 0xffff, piece >> 16
    count = {}
    for i in range(preq.shape[0]):
        count.setdefault((int(preq[i]), int(prow[i]), int(parts[i])), []).append((int(part[i]), int(slot[i])))
    assert len(count) == req.shape[0]
    used, longest_seen, shortest = [], 0, max(tiles)
    cut = {(int(a), int(b)): (int(c), int(n)) for a, b, c, n in merge}
    for (r, w, n), got_parts in count.items():
        t = int(tiles[(req == r) & (row == w)][0])
        assert sorted(p for p, _ in got_parts) == list(range(n)) and n <= min(64, t)
        longest_seen = max(longest_seen, -(-t // n))
        if n > 1:
            shortest = min(shortest, t // n)
            first, merged = cut.pop((r, w))
            assert merged == n and all(s == first + p for p, s in got_parts)
            used += [s for _, s in got_parts]
    assert not cut and sorted(used) == list(range(slots)) and longest_seen == longest
    # equal shares of rows longer than the length aimed at: at least half of it (rounded up)
    assert shortest >= (ck.PREFILL_MIN_PIECE + 1) // 2
    assert preq.shape[0] * hkv <= ck.PREFILL_PER_CU * 256 and longest >= ck.PREFILL_MIN_PIECE


def test_full_devices_and_short_rows_are_not_cut():
    assert _lists([16384] * 4, [16384] * 4, 4, 8, 128)[-1] is None       # 4,096 workgroups
    assert _lists([256], [256], 7, 4, 128)[-1] is None                    # 8 tiles at most
    assert _lists([512], [8192], 7, 4, 128)[-1] is not None
