"""GPU parity of the group kernel (rows of 1, 3, 5, 7 or 9 power-of-two groups
of 16-byte vectors) with plain torch indexing: every width class, token counts
around a wave's and a block's rows, one to three planes, flat and block-strided
caches, int32 and int64 slots with -1 padding and out-of-range slots, a pointer
table entry that is only 8-byte aligned, and batches with ragged objects, more
objects than a launch holds and grids past the linear layout's line."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    import lmcache_amd

    return lmcache_amd.c_ops


def _slots(T, num, seed, dtype):
    g = torch.Generator().manual_seed(seed)
    s = torch.randperm(num, generator=g)[:T].clone()
    if T > 2:
        s[T // 2] = -1
        s[T - 1] = num + 3
    return s.to(dtype)


def _copy(obj_rows, paged, slots, num, store):
    """obj_rows [T, W] and paged [num, W] views of the expected buffers."""
    for t, s in enumerate(slots.tolist()):
        if 0 <= s < num:
            if store:
                obj_rows[t] = paged[s]
            else:
                paged[s] = obj_rows[t]


def _bits(t):
    return t.view(torch.int16)


@pytest.mark.parametrize("store", [True, False])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
@pytest.mark.parametrize("W,L,T", [
    (64, 3, 1), (64, 2, 129), (128, 1, 16), (128, 5, 17), (192, 3, 8), (192, 2, 33), (320, 2, 31), (384, 3, 17),
    (448, 2, 9), (512, 2, 5), (576, 3, 8), (576, 2, 37), (640, 1, 13), (768, 3, 9), (896, 2, 7), (1536, 2, 3),
])
def test_object_vs_indexing(ops, W, L, T, dtype, store):
    num = 2 * T + 64
    g = torch.Generator().manual_seed(W + L + T)
    pool = torch.randn((L, 2, num, W), generator=g).to(torch.bfloat16)
    obj = torch.randn((2, L, T, W), generator=g).to(torch.bfloat16)
    slots = _slots(T, num, T, dtype)
    dpool, dobj = pool.to(DEV), obj.to(DEV)
    ptrs = torch.tensor([dpool[l, p].data_ptr() for l in range(L) for p in range(2)], dtype=torch.int64, device=DEV)
    ops.multi_layer_kv_transfer(dobj, ptrs, slots.to(DEV), torch.device(DEV), num, store, False, 2)
    for p in range(2):
        for l in range(L):
            _copy(obj[p, l], pool[l, p], slots, num, store)
    assert torch.equal(_bits(dobj.cpu()), _bits(obj))
    assert torch.equal(_bits(dpool.cpu()), _bits(pool))


@pytest.mark.parametrize("store", [True, False])
@pytest.mark.parametrize("W", [64, 192, 576])
def test_misaligned_table_entry(ops, W, store):
    L, T, num = 2, 21, 80
    g = torch.Generator().manual_seed(W)
    flat = torch.randn((L * 2, num * W + 8), generator=g).to(torch.bfloat16)
    obj = torch.randn((2, L, T, W), generator=g).to(torch.bfloat16)
    slots = _slots(T, num, 1, torch.int64)
    dflat, dobj = flat.to(DEV), obj.to(DEV)
    shift = [0, 4, 0, 0]  # elements: the second table entry is 8 bytes past a 16-byte boundary
    ptrs = torch.tensor([dflat[i].data_ptr() + 2 * shift[i] for i in range(2 * L)], dtype=torch.int64, device=DEV)
    ops.multi_layer_kv_transfer(dobj, ptrs, slots.to(DEV), torch.device(DEV), num, store, False, 2)
    for p in range(2):
        for l in range(L):
            i = 2 * l + p
            _copy(obj[p, l], flat[i, shift[i]:shift[i] + num * W].view(num, W), slots, num, store)
    assert torch.equal(_bits(dobj.cpu()), _bits(obj))
    assert torch.equal(_bits(dflat.cpu()), _bits(flat))


@pytest.mark.parametrize("store", [True, False])
@pytest.mark.parametrize("W", [64, 384])
def test_three_equal_planes(ops, W, store):
    L, T, num = 2, 19, 70
    g = torch.Generator().manual_seed(W)
    pool = torch.randn((L, 3, num, W), generator=g).to(torch.bfloat16)
    obj = torch.randn((1, L, T, 3 * W), generator=g).to(torch.bfloat16)
    slots = _slots(T, num, 2, torch.int64)
    dpool, dobj = pool.to(DEV), obj.to(DEV)
    ptrs = torch.tensor([dpool[l, p].data_ptr() for l in range(L) for p in range(3)], dtype=torch.int64, device=DEV)
    ops.multi_layer_kv_transfer(dobj, ptrs, slots.to(DEV), torch.device(DEV), num, store, True, 4, W, W, W)
    for p in range(3):
        for l in range(L):
            _copy(obj[0, l, :, p * W:(p + 1) * W], pool[l, p], slots, num, store)
    assert torch.equal(_bits(dobj.cpu()), _bits(obj))
    assert torch.equal(_bits(dpool.cpu()), _bits(pool))


@pytest.mark.parametrize("store", [True, False])
@pytest.mark.parametrize("block", [16, 48])  # 48: no power of two, the tile kernel
@pytest.mark.parametrize("H,D,T", [(1, 64, 50), (3, 128, 77), (9, 64, 1)])
def test_single_layer_blocks(ops, H, D, T, block, store):
    nb, W = 9, H * D
    g = torch.Generator().manual_seed(T)
    # Block-strided caches: blocks 0, 2, 4, ... of a larger allocation.
    pool = torch.randn((2, 2 * nb, block, H, D), generator=g).to(torch.bfloat16)
    lmc = torch.randn((2, T, W), generator=g).to(torch.bfloat16)
    num = nb * block
    slots = _slots(T, num, 3, torch.int64)
    dpool, dl = pool.to(DEV), lmc.to(DEV)
    ops.single_layer_kv_transfer(dl, (dpool[0, ::2], dpool[1, ::2]), slots.to(DEV), store, 2)
    for p in range(2):
        rows = pool[p, ::2].reshape(num, W).clone()
        _copy(lmc[p], rows, slots, num, store)
        pool[p, ::2] = rows.view(nb, block, H, D)
    assert torch.equal(_bits(dl.cpu()), _bits(lmc))
    assert torch.equal(_bits(dpool.cpu()), _bits(pool))


@pytest.mark.parametrize("store", [True, False])
@pytest.mark.parametrize("W,L,sizes", [
    (128, 2, [17, 1, 64, 5]),          # one launch, ragged objects
    (64, 1, [3] * 70),                 # more objects than a launch holds
    (192, 40, [256, 256, 100]),        # past the linear layout's line, a ragged last object
    (576, 61, [256] * 5 + [7]),
])
def test_batch_vs_indexing(ops, W, L, sizes, store):
    T = sum(sizes)
    num = T + 30
    gen = torch.Generator(device=DEV).manual_seed(T)
    pool = torch.randn((L, 2, num, W), generator=gen, device=DEV).to(torch.bfloat16)
    objs = [torch.randn((2, L, n, W), generator=gen, device=DEV).to(torch.bfloat16) for n in sizes]
    slots = _slots(T, num, 4, torch.int64).to(DEV)
    starts = [sum(sizes[:i]) for i in range(len(sizes))]
    want_pool, want = pool.clone(), [o.clone() for o in objs]
    for o, st in zip(want, starts):
        s = slots[st:st + o.shape[2]]
        ok = (s >= 0) & (s < num)
        if store:
            o[:, :, ok] = want_pool[:, :, s[ok]].transpose(0, 1)
        else:
            want_pool[:, :, s[ok]] = o[:, :, ok].transpose(0, 1)
    ptrs = torch.tensor([pool[l, p].data_ptr() for l in range(L) for p in range(2)], dtype=torch.int64, device=DEV)
    ops.multi_layer_kv_transfer_batched(objs, ptrs, slots, starts, torch.device(DEV), num, store, False, 2)
    for o, w in zip(objs, want):
        assert torch.equal(_bits(o), _bits(w))
    assert torch.equal(_bits(pool), _bits(want_pool))
