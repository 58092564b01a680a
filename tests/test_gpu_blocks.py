"""Whole-block movement parity (bit-exact): gather, scatter, compaction copy and
the DMA offload moves, on the engine's [2, L, blocks, page, KVH, D] pool."""
import numpy as np
import pytest
import torch

from nanovllm_amd import _native as nat
from nanovllm_amd.engine.kv_runner import BlockMover
from oracle import kv_oracle as ko

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _pool(L=3, blocks=20, kvh=4, seed=0, page=256):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(2, L, blocks, page, kvh, 128, generator=g).to(torch.bfloat16).to(DEV)


def _np(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy()


def test_gather_into_device_staging_and_pinned_host():
    pool = _pool()
    mover = BlockMover(pool)
    ids = [7, 0, 19, 3, 3]
    print("[blocks] gather", flush=True)
    dev = mover.gather(ids)                      # [n, 2, L, page, KVH, D] device
    host = torch.empty((len(ids),) + tuple(pool[:, :, 0].shape), dtype=pool.dtype, pin_memory=True)
    mover.gather(ids, out=host)                  # kernel writes pinned host memory
    torch.cuda.synchronize()
    ref = ko.block_gather(_np(pool).reshape(2 * pool.size(1), pool.size(2), -1), ids)
    assert np.array_equal(_np(dev).reshape(ref.shape), ref)
    assert np.array_equal(_np(host).reshape(ref.shape), ref)


def test_scatter_from_pinned_host():
    pool = _pool(seed=1)
    mover = BlockMover(pool)
    ids = [2, 11, 5]
    g = torch.Generator().manual_seed(2)
    items = torch.randn((3,) + tuple(pool[:, :, 0].shape), generator=g).to(torch.bfloat16).pin_memory()
    expect = _np(pool).reshape(2 * pool.size(1), pool.size(2), -1).copy()
    ko.block_scatter(expect, ids, _np(items).reshape(3, 2 * pool.size(1), -1))
    print("[blocks] scatter", flush=True)
    mover.scatter(items, ids)
    torch.cuda.synchronize()
    assert np.array_equal(_np(pool).reshape(expect.shape), expect)


def test_compaction_copy_disjoint_and_overlapping():
    pool = _pool(seed=3, blocks=32)
    mover = BlockMover(pool)
    expect = _np(pool).reshape(2 * pool.size(1), pool.size(2), -1).copy()
    src, dst = [1, 5, 9, 30], [2, 6, 10, 31]
    ko.block_copy(expect, src, dst)
    print("[blocks] copy disjoint", flush=True)
    mover.copy(src, dst)
    torch.cuda.synchronize()
    assert np.array_equal(_np(pool).reshape(expect.shape), expect)
    # A chain (dst of one pair is the src of another) must behave as a
    # simultaneous copy, like pool[:, :, dst] = pool[:, :, src].
    src, dst = [3, 4, 8], [4, 8, 12]
    ko.block_copy(expect, src, dst)
    print("[blocks] copy overlapping", flush=True)
    mover.copy(src, dst)
    torch.cuda.synchronize()
    assert np.array_equal(_np(pool).reshape(expect.shape), expect)


def test_dma_offload_roundtrip():
    pool = _pool(seed=4)
    mover = BlockMover(pool)
    ids = [4, 17, 0]
    host = torch.empty((3,) + tuple(pool[:, :, 0].shape), dtype=pool.dtype, pin_memory=True)
    print("[blocks] d2h dma", flush=True)
    mover.d2h(ids, host)
    torch.cuda.synchronize()
    ref = ko.block_gather(_np(pool).reshape(2 * pool.size(1), pool.size(2), -1), ids)
    assert np.array_equal(_np(host).reshape(ref.shape), ref)
    new_ids = [9, 1, 13]
    expect = _np(pool).reshape(2 * pool.size(1), pool.size(2), -1).copy()
    ko.block_scatter(expect, new_ids, _np(host).reshape(ref.shape))
    print("[blocks] h2d dma", flush=True)
    mover.h2d(host, new_ids)
    torch.cuda.synchronize()
    assert np.array_equal(_np(pool).reshape(expect.shape), expect)


def test_overlapped_swap_step_matches_sequential_moves():
    # One offload step with its moves on two copy-engine streams plus the
    # compaction on the current stream: the result equals the closed forms
    # (victims land in the host buffer, revived blocks come from the other host
    # buffer, compaction copies src -> dst); overlapping id sets are rejected.
    pool = _pool(L=2, blocks=24, seed=5)
    before = _np(pool).reshape(2 * pool.size(1), pool.size(2), -1).copy()
    mover = BlockMover(pool)
    out_ids, in_ids, src, dst = [3, 17, 8], [0, 21, 12], [5, 6, 22, 1], [9, 10, 2, 23]
    shape = (3,) + tuple(pool[:, :, 0].shape)
    host_out = torch.empty(shape, dtype=pool.dtype, pin_memory=True)
    g = torch.Generator().manual_seed(6)
    host_in = torch.randn(shape, generator=g).to(torch.bfloat16).pin_memory()
    print("[blocks] overlapped swap", flush=True)
    mover.swap(out_ids, host_out, in_ids, host_in, src, dst)
    torch.cuda.synchronize()
    assert np.array_equal(_np(host_out).reshape(3, *before.shape[:1], -1),
                          ko.block_gather(before, out_ids))
    expect = before.copy()
    ko.block_scatter(expect, in_ids, _np(host_in).reshape(3, before.shape[0], -1))
    ko.block_copy(expect, src, dst)
    assert np.array_equal(_np(pool).reshape(expect.shape), expect)
    with pytest.raises(ValueError):
        mover.swap([1], host_out[:1], [1], host_in[:1])


@pytest.mark.parametrize("planes,row_bytes,n", [
    (1, 16, 1),                    # one vector, one workgroup of the eight launched
    (1, 16 * 1024, 7),             # one full piece per row, 7 pieces over 8 XCDs
    (3, 16 * 1024 + 16, 3),        # a second piece of one vector; 18 pieces
    (5, 3 * 16 * 1024 - 16, 13),   # a last piece one vector short; 195 pieces
    (2, 48, 256), (2, 48, 257), (1, 16, 600),  # 256 host ids go with one launch
])
def test_device_moves_at_piece_and_xcd_edges(planes, row_bytes, n):
    g = torch.Generator().manual_seed(7)
    pool = torch.randint(0, 256, (1, planes, 2 * n + 1, row_bytes), generator=g,
                         dtype=torch.uint8).to(DEV)
    ids = torch.randperm(2 * n + 1, generator=g).tolist()
    src, dst = ids[:n], ids[n:2 * n]
    mover = BlockMover(pool)
    before = pool.clone()
    print(f"[blocks] edges planes={planes} row={row_bytes} n={n}", flush=True)
    items = mover.gather(src)
    assert torch.equal(items, before[:, :, src].movedim(2, 0))
    # ids on the device (read there) and in a pinned-host destination's move
    assert torch.equal(mover.gather(torch.tensor(src, device=DEV)), items)
    host = torch.empty_like(items, device="cpu", pin_memory=True)
    mover.gather(torch.tensor(src), out=host)
    torch.cuda.synchronize()
    assert torch.equal(host, items.cpu())
    expect = before.clone()
    expect[:, :, dst] = before[:, :, src]
    mover.copy(src, dst)
    assert torch.equal(pool, expect)
    expect[:, :, src] = items.movedim(0, 2).flip(2)
    mover.scatter(items.flip(0), src)
    assert torch.equal(pool, expect)
    expect[:, :, src] = items.movedim(0, 2)
    mover.scatter(host, src)
    assert torch.equal(pool, expect)


@pytest.mark.parametrize("planes,row_bytes,n", [
    (2, 1 << 20, 7),       # 14 MiB: plain stores
    (2, 1 << 20, 8),       # 16 MiB: non-temporal stores
    (1, 1 << 16, 255), (1, 1 << 16, 256),
    (1, 16 << 20, 17),     # past the memory-side cache
])
def test_device_moves_around_the_streaming_store_size(planes, row_bytes, n):
    g = torch.Generator(device=DEV).manual_seed(3)
    pool = torch.randint(0, 1 << 62, (1, planes, 2 * n + 1, row_bytes // 8), generator=g,
                         dtype=torch.int64, device=DEV)
    ids = torch.randperm(2 * n + 1, generator=torch.Generator().manual_seed(3)).tolist()
    src, dst = ids[:n], ids[n:2 * n]
    mover = BlockMover(pool)
    expect = pool.clone()
    print(f"[blocks] streaming stores planes={planes} row={row_bytes} n={n}", flush=True)
    items = mover.gather(src)
    assert torch.equal(items, expect[:, :, src].movedim(2, 0))
    expect[:, :, dst] = expect[:, :, src]
    mover.copy(src, dst)
    assert torch.equal(pool, expect)
    expect[:, :, src] = items.movedim(0, 2).flip(2)
    mover.scatter(items.flip(0).contiguous(), torch.tensor(src, device=DEV))
    assert torch.equal(pool, expect)


@pytest.mark.parametrize("n,inline", [(256, (True, True)), (257, (False, True)),
                                      (512, (False, True)), (513, (False, False))])
def test_id_lists_go_with_the_launch_or_are_uploaded(monkeypatch, n, inline):
    # A gather / scatter list of up to 256 ids and a copy's lists of up to 512
    # go with the launches; a host tensor does at any length.
    pool = torch.arange(2 * n, dtype=torch.int64, device=DEV).view(1, 1, -1, 1).repeat(1, 2, 1, 2)
    mover, called = BlockMover(pool), []
    real = nat.call
    monkeypatch.setattr(nat, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
    ids = torch.randperm(2 * n, generator=torch.Generator().manual_seed(n)).tolist()
    src, dst = ids[:n], ids[n:]
    print(f"[blocks] id lists n={n}", flush=True)
    items = mover.gather(src)
    assert torch.equal(mover.gather(torch.tensor(src)), items)
    host = torch.empty(items.shape, dtype=items.dtype, pin_memory=True)
    mover.gather(src, out=host)
    expect = pool.clone()
    expect[:, :, dst] = expect[:, :, src]
    assert torch.equal(items, expect[:, :, dst].movedim(2, 0))
    mover.copy(src, dst)
    assert torch.equal(pool, expect) and torch.equal(host, items.cpu())
    mover.scatter(items.flip(0).contiguous(), src)
    expect[:, :, src] = items.flip(0).movedim(0, 2)
    assert torch.equal(pool, expect)
    form = ["_ids" if i else "" for i in inline]
    assert called == ["kvc_block_gather" + form[0], "kvc_block_gather_ids",
                      "kvc_block_gather" + form[0], "kvc_block_copy" + form[1],
                      "kvc_block_scatter" + form[0]]
