"""GPU parity of copy_blocks against the CPU oracle (bit-exact, whole pool)."""
import numpy as np
import pytest
import torch

import lmserve_amd as kvc
from lmserve_amd import _lib
import workloads as wl
from oracle import kvc_oracle as orc
from tests.helpers import bits_of, random_pool, to_bf16

pytestmark = pytest.mark.gpu


def _run(gpu, shape, src_to_dst, seed=0, **kw):
    pool = random_pool(shape, seed)
    want = pool.copy()
    orc.c_copy_blocks(want, np.asarray(kvc.flatten_block_maps(src_to_dst), dtype=np.int64))
    dpool = to_bf16(pool, gpu)
    kvc.copy_blocks(dpool, src_to_dst, **kw)
    torch.cuda.synchronize()
    return bits_of(dpool), want, pool


@pytest.mark.parametrize("shape_name,L,nb,P", [
    ("llama-3-8b", 4, 256, 64),       # 64 KiB blocks
    ("llama-3.2-1b", 16, 128, 40),    # 32 KiB blocks, all 16 layers
    ("qwen2.5-7b", 3, 96, 17),
])
def test_copy_blocks_matches_oracle(gpu, shape_name, L, nb, P):
    s = {"llama-3-8b": wl.LLAMA_3_8B, "llama-3.2-1b": wl.LLAMA_3_2_1B,
         "qwen2.5-7b": wl.QWEN_2_5_7B}[shape_name]
    _, d = wl.copy_on_write_pairs(nb, P, seed=L)
    got, want, before = _run(gpu, (L, nb, 2, s.block_size, s.num_kv_heads, s.head_dim), d, seed=P)
    assert np.array_equal(got, want)
    assert not np.array_equal(got, before)


def test_copy_blocks_one_to_many_self_pair_and_empty(gpu):
    shape = (3, 32, 2, 16, 2, 64)
    got, want, before = _run(gpu, shape, {5: [0, 9, 31], 7: [7], 2: [3]}, seed=1)
    assert np.array_equal(got, want)
    for d in (0, 9, 31):
        assert np.array_equal(got[:, d], before[:, 5])
    got, want, before = _run(gpu, shape, {}, seed=2)
    assert np.array_equal(got, before)
    got, want, before = _run(gpu, shape, {4: []}, seed=3)
    assert np.array_equal(got, before)


@pytest.mark.parametrize("block_shape", [
    (2, 3, 1, 5),     # 60-byte blocks: 4-byte vectors
    (2, 1, 1, 3),     # 12-byte blocks
    (2, 1, 1, 1),     # 4-byte blocks
    (2, 16, 1, 72),   # 4608-byte blocks: a partial last chunk
    (2, 16, 8, 100),  # 51200-byte blocks, not a power of two
])
def test_copy_blocks_odd_block_sizes(gpu, block_shape):
    L, nb = 3, 24
    _, d = wl.copy_on_write_pairs(nb, 9, seed=5)
    got, want, _ = _run(gpu, (L, nb) + block_shape, d, seed=6)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("unroll", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("nt", [0, 1])
@pytest.mark.parametrize("max_wgs", [0, 7])
def test_copy_blocks_every_launch_shape(gpu, unroll, nt, max_wgs):
    """All unroll / load-store kind / grid-cap instantiations give the same bits."""
    s = wl.LLAMA_3_8B
    L, nb = 2, 64
    _, d = wl.copy_on_write_pairs(nb, 13, seed=unroll)
    _lib.set_tuning("copy_unroll", unroll)     # the autouse fixture puts the defaults back
    _lib.set_tuning("copy_nt", nt)
    _lib.set_tuning("copy_max_wgs", max_wgs)
    got, want, _ = _run(gpu, (L, nb, 2, s.block_size, s.num_kv_heads, s.head_dim), d, seed=8)
    ran = _lib.last_launch()
    assert ran["kernel"] == _lib.KVC_KERNEL_COPY_TILES and ran["per_lane"] == unroll
    assert ran["non_temporal"] == nt and ran["vec_bytes"] == 16
    assert ran["grid"] == (7 if max_wgs else 13 * L * (65536 // (256 * 16 * unroll)))
    assert np.array_equal(got, want)


def test_copy_blocks_accepts_a_device_pair_tensor_and_validates_on_request(gpu):
    s = wl.LLAMA_3_2_1B
    shape = (2, 40, 2, s.block_size, s.num_kv_heads, s.head_dim)
    flat, d = wl.copy_on_write_pairs(40, 10, seed=3)
    pool = random_pool(shape, 4)
    want = pool.copy()
    orc.copy_blocks_np(want, flat)
    dpool = to_bf16(pool, gpu)
    kvc.copy_blocks(dpool, torch.from_numpy(flat).to(gpu))
    torch.cuda.synchronize()
    assert np.array_equal(bits_of(dpool), want)
    with pytest.raises(ValueError):
        kvc.copy_blocks(dpool, {1: [2], 2: [3]}, validate=True)
    with pytest.raises(IndexError):
        kvc.copy_blocks(dpool, {1: [40]}, validate=True)
    with pytest.raises(ValueError):
        kvc.copy_blocks(dpool, torch.zeros(3, dtype=torch.int64, device=gpu))


def test_copy_blocks_skips_out_of_range_ids_on_the_device(gpu):
    """Ids the host never saw (device tensor input) cannot fault: pairs with an
    id outside the pool are skipped."""
    shape = (2, 16, 2, 16, 1, 64)
    pool = random_pool(shape, 9)
    want = pool.copy()
    orc.copy_blocks_np(want, np.asarray([1, 2], dtype=np.int64))
    dpool = to_bf16(pool, gpu)
    maps = torch.tensor([1, 2, 3, 16, -1, 5, 99, 7], dtype=torch.int64, device=gpu)
    kvc.copy_blocks(dpool, maps)
    torch.cuda.synchronize()
    assert np.array_equal(bits_of(dpool), want)


@pytest.mark.parametrize("n", [1, 2, 4, 8, 16, 32, 100])
def test_every_launch_shape_the_size_rule_picks_matches_the_oracle(gpu, n):
    """Bytes per workgroup follow the launch size (1, 2, 4, 8 or 16 vectors per lane
    for small launches, 2 or 1 for large ones): copy, gather and scatter at sizes
    that reach each choice, Llama-3-8B block shape over 32 layers."""
    s = wl.LLAMA_3_8B
    L, nb = 32, 256
    pool = random_pool((L, nb, 2, s.block_size, s.num_kv_heads, s.head_dim), seed=n)
    flat, pairs = wl.copy_on_write_pairs(nb, n, seed=n)
    want = pool.copy()
    orc.c_copy_blocks(want, flat)
    dpool = to_bf16(pool, gpu)
    assert _lib.lib().kvc_tuning_modified() == 0 and _lib.get_tuning("copy_unroll") == 0
    # vectors per lane the size rule must pick on a 256-CU part (2048 resident workgroups):
    # the smallest depth that fits n * 32 tiles of 64 KiB into 512 workgroups, a whole tile
    # per workgroup while that stays within 1024, else 2 (copy, scatter) or 1 (gather)
    small = {1: 1, 2: 2, 4: 4, 8: 8, 16: 16, 32: 16}
    kvc.copy_blocks(dpool, pairs)
    assert _lib.last_launch()["per_lane"] == small.get(n, 2)
    ids = torch.from_numpy(flat[1::2].copy()).to(gpu)               # the blocks just written
    dense = kvc.gather_blocks(dpool, ids)
    assert _lib.last_launch()["per_lane"] == small.get(n, 1)
    back = torch.from_numpy(flat[0::2].copy()).to(gpu)              # scatter them over their sources
    kvc.scatter_blocks(dpool, back, dense)
    assert _lib.last_launch()["per_lane"] == small.get(n, 2)
    torch.cuda.synchronize()
    view = want.reshape(L, nb, -1)
    want_dense = view[:, flat[1::2]].swapaxes(0, 1)
    assert np.array_equal(bits_of(dense), want_dense)
    view[:, flat[0::2]] = want_dense.swapaxes(0, 1)                 # a no-op by value: dst == src content
    assert np.array_equal(bits_of(dpool), want)


@pytest.mark.parametrize("tile_bytes,n,L,per_lane", [
    (65536, 6, 32, 4),       # 768 workgroups of 16 KiB: three eighths of the resident ones
    (65536, 7, 32, 8),       # more
    (36864, 20, 12, 4),      # the last workgroup of a tile a quarter full: three quarters of all lanes
    (34816, 20, 12, 16),     # less than that at 4 and at 8 vectors: a tile per workgroup
    (4112, 30, 8, 2),        # one vector past a chunk
    (4096, 96, 8, 1),
])
def test_depth_of_small_copies(gpu, tile_bytes, n, L, per_lane):
    """Vectors per lane by launch size and by how far a tile fills its workgroups; copy, gather and scatter against
    NumPy, at tiles that end inside a workgroup's chunk."""
    nb = 2 * n + 3
    pool = random_pool((L, nb, tile_bytes // 2), seed=n)
    ids = np.random.default_rng(n).permutation(nb)
    src, dst = ids[:n], ids[n:2 * n]
    dpool = to_bf16(pool, gpu)
    kvc.copy_blocks(dpool, {int(a): [int(b)] for a, b in zip(src, dst)})
    assert _lib.last_launch()["per_lane"] == per_lane
    pool[:, dst] = pool[:, src]
    assert np.array_equal(bits_of(dpool), pool)
    dense = kvc.gather_blocks(dpool, torch.from_numpy(dst.copy()).to(gpu))
    assert _lib.last_launch()["per_lane"] == per_lane
    assert np.array_equal(bits_of(dense), pool[:, dst].swapaxes(0, 1))
    kvc.scatter_blocks(dpool, torch.from_numpy(ids[3:3 + n].copy()).to(gpu), dense)
    pool[:, ids[3:3 + n]] = pool[:, dst].copy()
    assert np.array_equal(bits_of(dpool), pool)


@pytest.mark.parametrize("tile_bytes,n,L", [
    (8192, 400, 3),        # one chunk per tile
    (8208, 400, 3),        # a second chunk of one vector
    (20480, 350, 3),       # two and a half chunks
    (65552, 176, 3),       # one vector past 64 KiB; a last span of chunks that is not full
    (65536, 129, 8),       # whole spans and a remainder
])
def test_stream_kernel_edges(gpu, tile_bytes, n, L):
    """Launches beyond the small regime: tiles that end inside a chunk, spans of chunks that the launch does not
    fill, ids that are skipped; copy, gather and scatter against NumPy, dense buffers below 256 MiB."""
    nb = 2 * n + 5
    pool = random_pool((L, nb, tile_bytes // 2), seed=n)
    rng = np.random.default_rng(n)
    ids = rng.permutation(nb)
    src, dst = ids[:n].copy(), ids[n:2 * n].copy()
    src[3], dst[5] = nb, -1                                # outside the pool: skipped
    dst[7] = src[7]                                        # a pair onto itself
    want = pool.copy()
    ok = (src < nb) & (dst >= 0)
    want[:, dst[ok]] = pool[:, src[ok]]
    dpool = to_bf16(pool, gpu)
    maps = torch.from_numpy(np.stack([src, dst], 1).reshape(-1)).to(gpu)
    kvc.copy_blocks(dpool, maps)
    ran = _lib.last_launch()
    assert ran["kernel"] == _lib.KVC_KERNEL_COPY_TILES and ran["per_lane"] == 2
    assert ran["grid"] == n * L * ((tile_bytes + 8191) // 8192)
    assert np.array_equal(bits_of(dpool), want)
    picked = torch.from_numpy(ids[:n].copy()).to(gpu)
    dense = kvc.gather_blocks(dpool, picked)
    assert _lib.last_launch()["threads"] == 64 and _lib.last_launch()["per_lane"] == 1
    assert np.array_equal(bits_of(dense), want[:, ids[:n]].swapaxes(0, 1))
    back = torch.from_numpy(ids[5:5 + n].copy()).to(gpu)   # overlaps the blocks that were gathered
    kvc.scatter_blocks(dpool, back, dense)
    assert _lib.last_launch()["per_lane"] == 2
    want[:, ids[5:5 + n]] = want[:, ids[:n]].copy()
    assert np.array_equal(bits_of(dpool), want)


def test_stream_kernel_dense_buffer_beyond_the_last_level_cache(gpu):
    """Past 256 MiB the dense side is read and written non-temporally too."""
    L, nb, n = 16, 300, 257                                # 257 MiB of dense buffer
    pool = torch.randint(-2**15, 2**15, (L, nb, 32768), dtype=torch.int16, device=gpu)
    ids = torch.from_numpy(np.random.default_rng(1).permutation(nb)).to(gpu)
    dense = kvc.gather_blocks(pool, ids[:n].contiguous())
    assert _lib.last_launch()["non_temporal"] == 1
    assert torch.equal(dense, pool[:, ids[:n]].transpose(0, 1))
    want = pool.clone()
    want[:, ids[nb - n:]] = dense.transpose(0, 1)
    kvc.scatter_blocks(pool, ids[nb - n:].contiguous(), dense)
    assert _lib.last_launch()["non_temporal"] == 1 and torch.equal(pool, want)


@pytest.mark.parametrize("block_elems,n,L", [
    (4096, 1, 2),
    (4096, 447, 2),        # with the pair that is skipped a list of 448: the longest in a launch's own arguments
    (4096, 448, 2),        # one more: staged
    (4096, 300, 8),        # the stream kernel
    (2051, 20, 2),         # 2-byte vectors: staged
    (8, 65001, 1),         # staged in two pieces
])
def test_pairs_from_a_dict_reach_the_device_with_the_launch(gpu, block_elems, n, L):
    """Lists on either side of what a launch's arguments hold, ids outside the pool skipped, back to back with
    other lists and no synchronisation between, and from another stream; also with the call extension's place
    taken by the list in device memory."""
    nb = 2 * n + 6
    pool = random_pool((L, nb, block_elems), seed=n)
    dpool, dlist = to_bf16(pool, gpu), to_bf16(pool, gpu)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for rep in range(7):
        ids = np.random.default_rng(rep).permutation(nb).tolist()
        d = {}
        for i in range(n):
            d.setdefault(ids[i - i % 2], []).append(ids[n + 2 + i])
        d[ids[0]].append([nb, -1, 2**40, 1 - 2**63][rep % 4])
        for src, dsts in d.items():
            for dst in dsts:
                if 0 <= dst < nb:
                    pool[:, dst] = pool[:, src]
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side if rep == 5 else torch.cuda.current_stream()):
            kvc.copy_blocks(dpool, d)
        torch.cuda.current_stream().wait_stream(side)
        kvc.copy_blocks(dlist, torch.tensor(kvc.flatten_block_maps(d), device=gpu))
    assert np.array_equal(bits_of(dpool), pool) and np.array_equal(bits_of(dlist), pool)
    with pytest.raises((TypeError, ValueError)):
        kvc.copy_blocks(dpool, {0: ["x"]})


@pytest.mark.parametrize("tile_bytes,L,fans,per_lane", [
    (65536, 2, (2, 1, 3), 1),              # items of up to 3 destinations, one short of full
    (65536, 16, (3, 3, 2, 4, 1, 3), 4),    # a group of 4 is two items
    (65536, 16, (7, 7, 7, 16, 14), 4),     # up to 7 an item; groups beyond
    (65552, 30, (3,) * 12, 8),             # one vector past 64 KiB
    (65552, 60, (3,) * 12, 1),             # 2160 workgroups of 8 vectors: the large form
    (65536, 32, (2,) * 30, 8),             # 1920 workgroups: two per tile, paced
    (36864, 12, (3,) * 20, 4),
    (8192, 30, (3,) * 300, 1),             # longer than a launch's arguments: staged; the large form
    (8208, 3, (1,) * 400 + (2,) * 30, 4),  # staged, most items of one destination
])
def test_copies_of_blocks_with_several_destinations(gpu, tile_bytes, L, fans, per_lane):
    """One read for several destinations, with ids outside the pool and a pair onto itself among them; then the same
    as a list of pairs on the device, which reads once per copy."""
    n = sum(fans)
    nb = n + len(fans) + 3
    pool = random_pool((L, nb, tile_bytes // 2), seed=n)
    ids = np.random.default_rng(n).permutation(nb).tolist()
    d, at = {}, len(fans)
    for src, fan in zip(ids, fans):
        d[src] = ids[at:at + fan]
        at += fan
    dpool, dlist = to_bf16(pool, gpu), to_bf16(pool, gpu)
    for src, dsts in d.items():
        pool[:, dsts] = pool[:, src:src + 1]
    d[ids[0]][1:1] = [nb, -1, 2**40]       # outside the pool
    d[ids[1]] = [ids[1]] + d[ids[1]]       # onto itself
    kvc.copy_blocks(dpool, d)
    ran = _lib.last_launch()
    assert ran["kernel"] == _lib.KVC_KERNEL_COPY_TILES and ran["per_lane"] == per_lane
    assert np.array_equal(bits_of(dpool), pool)
    kvc.copy_blocks(dlist, torch.tensor(kvc.flatten_block_maps(d), device=gpu))
    assert np.array_equal(bits_of(dlist), pool)


@pytest.mark.parametrize("tile_bytes,L,fans,per_lane", [
    (8192, 30, (1,) * 540 + (2,) * 30, 2),       # beyond one resident set: one pair in ten is not worth the fan form,
    (8192, 30, (1,) * 250 + (2,) * 175, 2),      # nor more than half; at 7 items for 10 pairs
    (8192, 30, (1,) * 240 + (2,) * 180, 1),      # it is
    (65536, 50, (1,) * 14 + (2,), 8),            # within it 15 items for 16 pairs are enough,
    (65536, 50, (1,) * 15 + (2,), 16),           # 16 for 17 not
    (65536, 2, (1,) * 200 + (2,) * 60, 16),      # pairs that travel with the launch, and more items than would
])
def test_the_fan_form_is_taken_where_enough_pairs_share_a_source(gpu, tile_bytes, L, fans, per_lane):
    n = sum(fans)
    nb = n + len(fans) + 1
    pool = random_pool((L, nb, tile_bytes // 2), seed=n)
    dpool = to_bf16(pool, gpu)
    ids = np.random.default_rng(n).permutation(nb).tolist()
    d, at = {}, len(fans)
    for i, src in zip(np.random.default_rng(1).permutation(len(fans)), ids):
        d[src] = ids[at:at + fans[i]]
        at += fans[i]
    for src, dsts in d.items():
        pool[:, dsts] = pool[:, src:src + 1]
    kvc.copy_blocks(dpool, d)
    assert _lib.last_launch()["per_lane"] == per_lane
    assert np.array_equal(bits_of(dpool), pool)


@pytest.mark.parametrize("n", [6, 600])     # in the launch's arguments, and staged
def test_a_list_of_which_nothing_copies(gpu, n):
    pool = random_pool((2, 8, 4096), seed=n)
    dpool = to_bf16(pool, gpu)
    pairs = np.stack([np.full(n, 3), np.resize([3, 8, -1], n)], axis=1).astype(np.int64)
    scratch = torch.zeros(2 * n, dtype=torch.int64, device=gpu)
    _lib.check(_lib.lib().kvc_copy_blocks_host_pairs(dpool.data_ptr(), pairs.ctypes.data, n, scratch.data_ptr(), 2, 8 * 8192,
                                                     8192, 8, torch.cuda.current_stream().cuda_stream))
    assert np.array_equal(bits_of(dpool), pool)


def test_pairs_that_travel_with_the_launch_are_recorded_with_or_without_scratch(gpu):
    """300 pairs of which two share a source, and scratch at hand: nothing of the list may be left to a staging buffer
    that a replay would read again."""
    n, L, elems = 300, 2, 4096
    nb = 2 * n
    pool = random_pool((L, nb, elems), seed=5)
    dpool = to_bf16(pool, gpu)
    ids = np.random.default_rng(5).permutation(nb)
    pairs = np.stack([ids[:n], ids[n:]], axis=1).astype(np.int64)
    pairs[8, 0] = pairs[7, 0]
    scratch = torch.zeros(2 * n, dtype=torch.int64, device=gpu)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _lib.check(_lib.lib().kvc_copy_blocks_host_pairs(
            dpool.data_ptr(), pairs.ctypes.data, n, scratch.data_ptr(), L, nb * elems * 2, elems * 2, nb,
            torch.cuda.current_stream().cuda_stream))
    kept, at = pairs.copy(), dpool.clone()
    pairs[:] = 0
    for rep in range(3):
        scratch.fill_(rep)
        dpool.copy_(at)
        graph.replay()
        torch.cuda.synchronize()
        want = pool.copy()
        want[:, kept[:, 1]] = want[:, kept[:, 0]]
        assert np.array_equal(bits_of(dpool), want)
    with torch.cuda.graph(torch.cuda.CUDAGraph()):     # a longer list is refused there, also where its items are few
        long = np.stack([np.repeat(ids[:100], 5), np.resize(ids[100:], 500)], axis=1).astype(np.int64)
        rc = _lib.lib().kvc_copy_blocks_host_pairs(
            dpool.data_ptr(), long.ctypes.data, 500, torch.zeros(1000, dtype=torch.int64, device=gpu).data_ptr(), L,
            nb * elems * 2, elems * 2, nb, torch.cuda.current_stream().cuda_stream)
        assert rc == _lib.KVC_ERR_UNSUPPORTED
        torch.zeros(4, device=gpu).add_(1)


@pytest.mark.parametrize("block_bytes,n,per_lane,grid", [
    (1 << 20, 131071, 2, 131071 * 128),                # the largest that the stream kernel takes: 2^32 - 2^15 lanes
    (1 << 20, 131073, 2, (2**32 - 1) // 256),          # past it: chunks walked grid-stride
    ((1 << 20) + 8, 70000, 2, (2**32 - 1) // 256),     # 8-byte vectors, never taken by the stream kernel
])
def test_copies_of_more_lanes_than_a_launch_has(gpu, block_bytes, n, per_lane, grid):
    """A list of that many pairs over a small pool: all but the first and the last are outside the pool."""
    pool = random_pool((1, 8, block_bytes // 2), seed=n)
    dpool = to_bf16(pool, gpu)
    pairs = torch.full((n, 2), -1, dtype=torch.int64, device=gpu)
    pairs[0] = torch.tensor([0, 1])
    pairs[-1] = torch.tensor([2, 7])
    kvc.copy_blocks(dpool, pairs.flatten())
    ran = _lib.last_launch()
    assert (ran["per_lane"], ran["grid"]) == (per_lane, grid)
    pool[0, 1], pool[0, 7] = pool[0, 0], pool[0, 2]
    assert np.array_equal(bits_of(dpool), pool)


def test_a_gather_of_more_lanes_than_a_launch_has(gpu):
    """67 million chunks of 1 KiB, all but the first block's outside the pool: nothing is written for those."""
    block_bytes, n = 1 << 20, 65537
    pool = torch.randint(-2**15, 2**15, (1, 2, block_bytes // 2), dtype=torch.int16, device=gpu)
    dense = torch.zeros(block_bytes // 2, dtype=torch.int16, device=gpu)
    ids = torch.full((n,), -1, dtype=torch.int64, device=gpu)
    ids[0] = 1
    rc = _lib.lib().kvc_gather_blocks(pool.data_ptr(), dense.data_ptr(), ids.data_ptr(), n, 1, block_bytes * 2,
                                      block_bytes, 2, 0, 1, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and _lib.last_launch()["threads"] == 256 and _lib.last_launch()["grid"] == (2**32 - 1) // 256
    assert torch.equal(dense, pool[0, 1])


@pytest.mark.parametrize("tile_bytes,L,fans,threads", [
    (65552, 60, (2,) * 20, 64),            # one vector past 64 KiB: a wavefront with one lane of work
    (8208, 30, (2,) * 150, 64),
    (8208, 30, (2, 1) * 200, 64),          # staged
    (8208, 30, (3, 1) * 110, 64),          # two an item on average
    (8208, 30, (3, 2) * 80, 256),          # more
])
def test_large_copies_with_two_destinations_a_block(gpu, tile_bytes, L, fans, threads):
    """Up to two destinations an item go out in single wavefronts: against NumPy at tiles that end inside a chunk."""
    n = sum(fans)
    nb = n + len(fans) + 1
    pool = random_pool((L, nb, tile_bytes // 2), seed=n)
    dpool = to_bf16(pool, gpu)
    ids = np.random.default_rng(n).permutation(nb).tolist()
    d, at = {}, len(fans)
    for src, fan in zip(ids, fans):
        d[src] = ids[at:at + fan]
        at += fan
    for src, dsts in d.items():
        pool[:, dsts] = pool[:, src:src + 1]
    kvc.copy_blocks(dpool, d)
    ran = _lib.last_launch()
    assert (ran["per_lane"], ran["threads"]) == (1, threads)
    assert np.array_equal(bits_of(dpool), pool)


@pytest.mark.parametrize("tile_bytes,n,order", [(65536, 1023, 1), (65536, 1024, 0), (65552, 1024, 0), (65520, 1025, 1)])
def test_order_of_large_copies(gpu, tile_bytes, n, order):
    """Tiles of 64 KiB and more: below 64 MiB a layer the launch walks layers, from there on blocks."""
    L = 2
    g = torch.Generator(device=gpu).manual_seed(n)
    pool = torch.randint(-2**31, 2**31 - 1, (L, 2 * n + 3, tile_bytes // 4), dtype=torch.int32, device=gpu, generator=g)
    ids = torch.randperm(2 * n + 3, device=gpu, generator=g)
    want = pool.clone()
    want[:, ids[n:2 * n]] = pool[:, ids[:n]]
    kvc.copy_blocks(pool, torch.stack([ids[:n], ids[n:2 * n]], 1).flatten().contiguous())
    assert _lib.last_launch()["order"] == order
    assert torch.equal(pool, want)


@pytest.mark.parametrize("tile_bytes,L,fans,threads", [
    (65536, 28, (4,) * 19, 64),            # items of three and one by turns, a tile to a run
    (65536, 28, (4, 1, 1) * 10, 64), (131088, 12, (1, 7) * 11, 64), (49152, 28, (4, 2) * 18, 64),
    (65536, 28, (5, 6, 7) * 16, 256), (65552, 9, (3, 2, 3) * 30, 256),
    (65536, 28, (2,) * 37 + (1,), 64),     # a last span that is not full
])
def test_large_forks_of_uneven_items(gpu, tile_bytes, L, fans, threads):
    """Items of few and of many destinations by turns, which the XCDs share out between them: against NumPy."""
    n = sum(fans)
    nb = n + len(fans) + 1
    pool = random_pool((L, nb, tile_bytes // 2), seed=n)
    dpool = to_bf16(pool, gpu)
    ids = np.random.default_rng(n).permutation(nb).tolist()
    d, at = {}, len(fans)
    for src, fan in zip(ids, fans):
        d[src] = ids[at:at + fan]
        at += fan
    for src, dsts in d.items():
        pool[:, dsts] = pool[:, src:src + 1]
    kvc.copy_blocks(dpool, d)
    ran = _lib.last_launch()
    assert (ran["per_lane"], ran["threads"], ran["order"]) == (1, threads, 1)
    assert np.array_equal(bits_of(dpool), pool)


@pytest.mark.parametrize("tile_bytes,n,L,run", [
    (8192, 6143, 1, 64), (8192, 6144, 1, 256), (8208, 1023, 3, 64), (8208, 1024, 3, 256),   # either side of three spans
])
def test_runs_of_scatters(gpu, tile_bytes, n, L, run):
    g = torch.Generator(device=gpu).manual_seed(n)
    nb = n + 9
    pool = torch.randint(-2**31, 2**31 - 1, (L, nb, tile_bytes // 4), dtype=torch.int32, device=gpu, generator=g)
    dense = torch.randint(-2**31, 2**31 - 1, (n, L, tile_bytes // 4), dtype=torch.int32, device=gpu, generator=g)
    ids = torch.randperm(nb, device=gpu, generator=g)[:n].contiguous()
    want = pool.clone()
    want[:, ids] = dense.transpose(0, 1)
    kvc.scatter_blocks(pool, ids, dense)
    assert _lib.last_launch()["run"] == run
    assert torch.equal(pool, want)
