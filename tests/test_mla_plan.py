"""Checks of the balanced MLA launch plan as the Python surface reports it
(mla.get_mla_metadata's num_splits): on the CPU against a direct simulation of
the launch's share walk, share by share and request by request; on the GPU
against the prefix sums that the split kernel writes for the merge.

The walk: a request's units are a weight and then one per 32-token tile; n
shares take [w U / n, (w + 1) U / n) of the U units, and a request gets one
partial result per share that holds some of its tiles. The row groups, and with
them the shares, follow the work of the longest possible batch; a batch of as
many tiles in every request (16 or more per share) whose shares its requests
divide is cut without the weight."""

import random

import numpy as np
import pytest
import torch

import capi
from mla import get_mla_metadata

WEIGHT = 8


def row_groups(B, rows, block_size, width, nwg):
    """(row groups, weight) of a launch on a table `width` tokens wide."""
    if block_size % 8:
        return -(-rows // 128), 0
    sizes = [r for r in (16, 32, 64, 128) if r == 16 or r < 2 * rows]
    tiles = -(-width // 32)
    groups = lambda r: -(-rows // r)  # noqa: E731
    work = B * tiles * groups(16) / nwg
    r = min(16 if work <= 12 else 32 if work <= 28 else 64 if work <= 160 else 128, sizes[-1])
    if tiles <= 2:
        r = next((x for x in sizes if x >= r and B * groups(x) <= nwg), sizes[-1])
    if tiles >= 8 and B * groups(sizes[-1]) % nwg == 0:
        r = sizes[-1]
    return groups(r), WEIGHT


def simulate(S_list, rows, block_size, longest, nwg):
    B, width = len(S_list), max(1, -(-longest // block_size)) * block_size
    tiles = [-(-min(max(s, 0), width) // 32) for s in S_list]
    T, live = sum(tiles), sum(t > 0 for t in tiles)
    groups, weight = row_groups(B, rows, block_size, width, nwg)
    U = T + live * weight
    n = min(max(1, nwg // groups), U)
    if weight:
        n = min(n, max(B, 1 + int(np.float32(5) * np.sqrt(np.float32(U)))))
        if min(tiles) == max(tiles) and T > 0 and T >= 16 * n and n % B == 0:
            weight, U = 0, T
    ranges, at = [], 0  # each request's tiles in the line of units
    for t in tiles:
        at += weight if t else 0
        ranges.append((at, at + t))
        at += t
    out = [0]
    for t0, t1 in ranges:
        out.append(out[-1] + sum(max(t0, w * U // n) < min(t1, (w + 1) * U // n)
                                 for w in range(n)))
    return out


BATCHES = [([4096] * 8, 128), ([0, 1, 33, 0, 5000], 128), ([100000], 128), ([31, 32, 33] * 50, 256),
           ([0, 0], 64), ([7000, 1, 1, 1, 9000], 300), ([4096], 128), ([4096], 16),
           ([4096, 4096], 128), ([33] * 256, 64), ([500] * 256, 128), ([2048] * 128, 128),
           ([4096] * 128, 256), ([64], 512), ([1], 1), ([16] * 200, 64), ([50] * 300, 40)]


@pytest.mark.parametrize("S_list,rows", BATCHES)
@pytest.mark.parametrize("block_size", [64, 16, 20])  # (20: the 8-wave kernels)
def test_plan_pieces(S_list, rows, block_size):
    sl = torch.tensor(S_list, dtype=torch.int32)
    meta, splits = get_mla_metadata(sl, rows, 1, block_size=block_size)
    assert int(meta[0, 0]) == 0
    nwg = int(meta[0, 1])
    assert splits.tolist() == simulate(S_list, rows, block_size, max(S_list), nwg)
    # A table of another width than the longest request's, told as max_seqlen.
    for longest in (max(S_list) // 2, max(S_list) + 1000, 131072):
        _, splits = get_mla_metadata(sl, rows, 1, longest, block_size)
        assert splits.tolist() == simulate(S_list, rows, block_size, longest, nwg)


def test_plan_of_one_request():
    # 128 heads of one request of 4096 tokens on 256 CUs: 32 shares of 4.25 units
    # in 16-row groups, of which the weight of 8 takes the first two.
    _, splits = get_mla_metadata(torch.tensor([4096], dtype=torch.int32), 128, 1)
    assert splits.tolist() == [0, 30]


@pytest.mark.parametrize("seed", range(8))
def test_plan_across_the_rules(seed):
    # Few and many workgroups, lengths on both sides of every row rule.
    rng = random.Random(seed)
    for _ in range(40):
        B, top = rng.choice([1, 2, 3, 8, 40, 128]), rng.choice([20, 64, 65, 250, 256, 300, 2000])
        S_list = [rng.randint(0, top) if seed % 2 else top for _ in range(B)]
        rows, nwg = rng.choice([1, 16, 17, 64, 65, 128, 321, 512]), rng.choice([1, 2, 4, 30, 256])
        sl = torch.tensor(S_list, dtype=torch.int32)
        splits = torch.empty(B + 1, dtype=torch.int32)
        for blocks in (0, 1, 7, 100):
            assert capi.mla_balanced_num_splits(sl.data_ptr(), splits.data_ptr(), B, 1, rows, 64,
                                                blocks, nwg, 1, None) == 0
            longest = 64 * blocks if blocks else max(S_list)
            assert splits.tolist() == simulate(S_list, rows, 64, longest, nwg)


def test_num_splits_refuses():
    sl, out = torch.ones(1, dtype=torch.int32), torch.empty(2, dtype=torch.int32)
    good = [sl.data_ptr(), out.data_ptr(), 1, 1, 128, 64, 1, 256, 1, None]
    assert capi.mla_balanced_num_splits(*good) == 0
    for i, bad in ((0, None), (1, None), (2, -1), (3, 0), (4, 0), (4, 1 << 21), (5, 0), (6, -1),
                   (6, 1 << 26)):
        args = list(good)
        args[i] = bad
        assert capi.mla_balanced_num_splits(*args) == capi.HIP_ERROR_INVALID_VALUE


@pytest.mark.gpu
@pytest.mark.parametrize("block_size", [64, 16, 20])
def test_plan_is_the_launch(gpu, block_size):
    # The pieces that the merge finds in the prefix sums of the launch.
    from test_mla import SCALE
    rng = random.Random(block_size)
    batches = BATCHES + [([rng.randint(0, 6000) for _ in range(rng.randint(1, 60))],
                          rng.choice([1, 16, 40, 128, 256])) for _ in range(12)]
    for S_list, rows in batches:
        if sum(S_list) > 300000:
            continue
        B, width = len(S_list), max(1, -(-max(S_list) // block_size))
        sl = torch.tensor(S_list, dtype=torch.int32, device="cuda")
        meta, splits = get_mla_metadata(sl, rows, 1, block_size=block_size)
        nwg = int(meta[0, 1])
        kv = torch.zeros(1, block_size, 1, 576, dtype=torch.bfloat16, device="cuda")
        bt = torch.zeros(B, width, dtype=torch.int32, device="cuda")
        q = torch.zeros(B, 1, rows, 576, dtype=torch.bfloat16, device="cuda")
        out = torch.empty(B, 1, rows, 512, dtype=torch.bfloat16, device="cuda")
        wsb = capi.mla_balanced_workspace_bytes(B, 1, rows, nwg)
        ws = torch.zeros(wsb, dtype=torch.uint8, device="cuda")
        assert capi.mla_balanced_launch(
            q.data_ptr(), kv.data_ptr(), bt.data_ptr(), sl.data_ptr(), out.data_ptr(), None, B, 1,
            rows, block_size, width, SCALE, 0, nwg, ws.data_ptr(), wsb,
            torch.cuda.current_stream().cuda_stream) == 0
        *pre, last = ws[wsb - 8 * (B + 2):].view(torch.int64).tolist()
        n, weight, U = last & 0xFFFFFFFF, last >> 32, pre[-1]
        want = [0]
        for p0, p1 in zip(pre, pre[1:]):
            held = 0 if p0 == p1 else ((p1 * n - 1) // U) - (((p0 + weight + 1) * n - 1) // U) + 1
            want.append(want[-1] + held)
        assert splits.tolist() == want, f"{S_list[:8]} rows {rows}"


def test_fixed_plan():
    sl = torch.tensor([100, 2000, 0], dtype=torch.int32)
    meta, splits = get_mla_metadata(sl, 128, 1, num_splits=4)
    assert int(meta[0, 0]) == 4 and splits.tolist() == [0, 4, 8, 12]
    with pytest.raises(ValueError):
        get_mla_metadata(sl, 128, 2)


@pytest.mark.parametrize("B,s_q,h_q,cus,want", [(32, 1, 128, 256, 8), (64, 1, 128, 256, 4),
                                                (128, 1, 128, 256, 2), (1, 1, 128, 256, 128),
                                                (8, 2, 128, 256, 16), (3, 1, 200, 256, 43),
                                                (256, 1, 64, 256, 1), (300, 1, 128, 256, 1)])
def test_pick_num_splits_covers_cus(B, s_q, h_q, cus, want):
    # The (row group, request, split) grid covers num_cus workgroups with the
    # fewest splits: B * ceil(s_q h_q / 128) row groups per split. Long
    # sequences (1 << 20 tokens), so the 256-token minimum does not bind.
    ns = capi.mla_pick_num_splits(B, s_q, h_q, 64, (1 << 20) // 64, cus)
    groups = B * -(-(s_q * h_q) // 128)
    assert ns == want
    assert ns == 128 or groups * ns >= cus  # 128: MLA_DECODE_MAX_SPLITS
    assert ns == 1 or groups * (ns - 1) < cus


def test_pick_num_splits_min_chunk():
    # 1000 tokens (125 blocks of 8): at most 1000 // 256 = 3 splits, however
    # few the requests; 128 tokens: one.
    assert capi.mla_pick_num_splits(1, 1, 128, 8, 125, 256) == 3
    assert capi.mla_pick_num_splits(1, 1, 128, 64, 2, 256) == 1
