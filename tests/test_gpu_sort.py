"""The library's device radix sort and scan against NumPy: stable order by a key bit
range (unsigned), values carried along, for 32- and 64-bit keys, sizes around the
4096-element tile and heavy duplicates; prefix sums against ``np.cumsum``."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [1, 63, 4095, 4096, 4097, 100_003, 1_000_000]


def _ref(keys_u: np.ndarray, begin: int, end: int):
    """Stable order of the unsigned keys by bits [begin, end)."""
    width = end - begin
    field = keys_u >> np.uint64(begin)
    if width < 64:
        field = field & np.uint64((1 << width) - 1)
    return np.argsort(field, kind="stable")


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("dtype,bits", [(torch.int32, (0, 32)), (torch.int32, (5, 29)), (torch.int32, (0, 7)),
                                        (torch.int64, (0, 64)), (torch.int64, (3, 47))])
def test_sort_pairs_matches_numpy_stable(cuda, n, dtype, bits):
    from hi3d_amd import sort

    rng = np.random.default_rng(n + bits[0] * 7 + bits[1])
    if dtype == torch.int32:
        raw = rng.integers(0, 2**32, size=n, dtype=np.uint64)
        keys = torch.as_tensor(raw.astype(np.uint32).view(np.int32))
    else:
        raw = rng.integers(0, 2**64, size=n, dtype=np.uint64)
        keys = torch.as_tensor(raw.view(np.int64))
    vals = torch.arange(n, dtype=torch.int32)
    sk, sv = sort.sort_pairs(keys.to(cuda), vals.to(cuda), *bits)
    order = _ref(raw, *bits)
    assert np.array_equal(sv.cpu().numpy(), order)
    assert torch.equal(sk.cpu(), keys[torch.as_tensor(order)])


@pytest.mark.parametrize("n", [4097, 300_001])
def test_sort_pairs_stable_on_duplicates(cuda, n):
    """Seven distinct keys: equal keys keep their input order (values ascend inside each
    run), over one digit pass and over four."""
    from hi3d_amd import sort

    rng = np.random.default_rng(5)
    raw = rng.integers(0, 7, size=n).astype(np.uint64) * np.uint64(0x01010101)
    keys = torch.as_tensor(raw.astype(np.uint32).view(np.int32))
    vals = torch.as_tensor(rng.permutation(n).astype(np.int32))
    for bits in ((0, 8), (0, 32)):
        sk, sv = sort.sort_pairs(keys.to(cuda), vals.to(cuda), *bits)
        order = _ref(raw, *bits)
        assert np.array_equal(sv.cpu().numpy(), vals.numpy()[order])
        assert torch.equal(sk.cpu(), keys[torch.as_tensor(order)])


def test_sort_pairs_empty_and_empty_range(cuda):
    from hi3d_amd import sort

    k = torch.tensor([5, 3, 9], dtype=torch.int32, device=cuda)
    v = torch.tensor([0, 1, 2], dtype=torch.int32, device=cuda)
    sk, sv = sort.sort_pairs(k, v, 4, 4)
    assert sk.cpu().tolist() == [5, 3, 9] and sv.cpu().tolist() == [0, 1, 2]
    sk, sv = sort.sort_pairs(k[:0], v[:0])
    assert sk.numel() == 0 and sv.numel() == 0


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("inclusive", [False, True])
def test_scan_matches_cumsum(cuda, n, inclusive):
    from hi3d_amd import sort

    rng = np.random.default_rng(n)
    x = rng.integers(-50, 100, size=n).astype(np.int32)
    got = sort.scan(torch.as_tensor(x).to(cuda), inclusive).cpu().numpy()
    c = np.cumsum(x, dtype=np.int64).astype(np.int32)
    ref = c if inclusive else np.concatenate([[0], c[:-1]]).astype(np.int32)
    assert np.array_equal(got, ref)


def _al(x: int) -> int:
    return (x + 255) // 256 * 256


def _least(n: int) -> int:
    """Sort and scan scratch with tiles of 4096 elements."""
    return 1024 * max((n + 4095) // 4096, 1) + 1024


LEAST = {
    "hi3d_sort_pairs_workspace": _least,
    "hi3d_unique_keys_workspace": lambda n: 2 * _al(8 * n) + 5 * _al(4 * n) + _least(n) + 256,
    "hi3d_conv_plan_workspace": lambda n: 2 * _al(8 * n) + 3 * _al(4 * n) + _least(n) + 256,
    "hi3d_halo_plan_workspace": lambda n: 2 * _al(8 * n) + 3 * _al(4 * n) + _least(n) + 256,
    "hi3d_downsample_workspace": lambda n: 2 * _al(8 * n) + 3 * _al(4 * n) + _least(n) + 256,
    "hi3d_stride2_up_plan_workspace": lambda n: 4 * _al(4 * n) + _least(n),
    "hi3d_child_table_workspace": lambda n: 2 * _al(32 * n) + _al(32 * n + 32) + _least(8 * n),
    "hi3d_kmap_dense_order_workspace": lambda n: 4 * _al(4 * n) + _least(n),
    "hi3d_kmap_workspace": lambda n, cap, key64: _al(8 * cap) + _al(32 * cap) + 4 * _al(4 * n) + _least(n) + _al(16 * n),
}


@pytest.mark.parametrize("n", [1, 5000, 150_001, 1_100_000])
def test_least_workspaces_are_enough(cuda, monkeypatch, n):
    """Every call that sorts or scans, with the least workspace it takes (tiles of 4096
    keys, whatever faster tiles the size query leaves room for): the results of the
    reported size, and nothing written behind the workspace."""
    from hi3d_amd import _lib, fast_unique, kmap, sort

    rng = np.random.default_rng(n)
    side = 128
    cells = torch.as_tensor(rng.permutation(side ** 3)[:n])
    idx = torch.stack([0 * cells, cells // side ** 2, cells // side % side, cells % side], 1).int().to(cuda)
    keys = torch.as_tensor(rng.integers(0, 2**31, n).astype(np.int32)).to(cuda)
    vals = torch.arange(n, dtype=torch.int32, device=cuda)
    mask = torch.as_tensor(rng.random((n, 8)) < 0.4).to(cuda)

    def run():
        monkeypatch.setattr(kmap, "KMAP_DENSE_ORDER_MIN_BYTES", 0)
        m = kmap.build_kernel_map(idx, [side] * 3, 1)
        far = idx * torch.tensor([1, 16, 16, 16], dtype=torch.int32, device=cuda)
        hashed = [kmap.build_kernel_map(c, [s] * 3, 1, capacity=1 << 21).table for c, s in ((idx, 512), (far, 2048))]
        plan = kmap.build_plan(m.table, n, idx)
        s2 = kmap.stride2_structure(idx, [side] * 3, 1)
        return [*sort.sort_pairs(keys, vals), sort.scan(vals % 7), m.table, *hashed, plan.rows, plan.gidx, plan.tile_mask,
                s2.low, s2.inverse, s2.counts, *s2.up_order(), *kmap.child_neighbour_table(m.table, mask),
                *fast_unique.unique_rows(idx[:, 1:] // 3, True, True)]

    want = run()
    guards, query = [], _lib.query

    def least(name, *args):
        if name not in LEAST:
            return query(name, *args)
        b = LEAST[name](*args)
        assert b <= query(name, *args)
        return b

    def workspace(nbytes, device):
        t = torch.full((int(nbytes) + 4096,), 0xA5, dtype=torch.uint8, device=device)
        guards.append(t[int(nbytes):])
        return t[:int(nbytes)]

    monkeypatch.setattr(_lib, "query", least)
    monkeypatch.setattr(_lib, "workspace", workspace)
    for g, w in zip(run(), want, strict=True):
        assert torch.equal(g, w)
    assert len(guards) >= 10 and all((g == 0xA5).all() for g in guards)
