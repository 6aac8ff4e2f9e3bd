"""GPU parity of the page-table index preparation against the CPU oracle."""
import numpy as np
import pytest
import torch

import lmserve_amd as kvc
from lmserve_amd import _lib
from oracle import kvc_oracle as orc
from tests.helpers import MAPPED_FORMS, mapped_requests

pytestmark = pytest.mark.gpu


def _up(a, gpu):
    return torch.from_numpy(np.asarray(a, dtype=np.int32)).to(gpu)


@pytest.mark.parametrize("page_size", [16, 4, 3])
def test_get_seq_lens_matches_oracle(gpu, page_size):
    rng = np.random.default_rng(page_size)
    B = 300
    pages = rng.integers(0, 40, size=B)
    pages[::17] = 0                                    # requests without pages: clamp
    indptr = np.cumsum(np.concatenate([[0], pages])).astype(np.int32)
    last = rng.integers(1, page_size + 1, size=B).astype(np.int32)
    want = orc.c_get_seq_lens(indptr, last, page_size)
    assert np.array_equal(want, orc.get_seq_lens_np(indptr, last, page_size))
    got = kvc.get_seq_lens(_up(indptr, gpu), _up(last, gpu), page_size)
    assert got.dtype == torch.int32
    assert np.array_equal(got.cpu().numpy(), want)
    assert kvc.get_seq_lens(_up([0], gpu), _up([], gpu), page_size).numel() == 0


def test_get_batch_indices_positions_matches_oracle(gpu):
    rng = np.random.default_rng(1)
    B = 257
    n_new = rng.integers(0, 9, size=B)                 # includes requests with no new token
    n_new[5] = 2048                                    # one long prefill chunk
    filled = rng.integers(0, 5000, size=B)
    seq_lens = (filled + n_new).astype(np.int32)
    indptr = np.cumsum(np.concatenate([[0], n_new])).astype(np.int32)
    nnz = int(indptr[-1])
    want_b, want_p = orc.c_get_batch_indices_positions(indptr, seq_lens, nnz)
    np_b, np_p = orc.get_batch_indices_positions_np(indptr, seq_lens, nnz)
    assert np.array_equal(want_b, np_b) and np.array_equal(want_p, np_p)
    got_b, got_p = kvc.get_batch_indices_positions(_up(indptr, gpu), _up(seq_lens, gpu), nnz)
    assert np.array_equal(got_b.cpu().numpy(), want_b)
    assert np.array_equal(got_p.cpu().numpy(), want_p)
    # positions are exactly range(filled, filled + n_new) per request
    at = 0
    for b in range(B):
        assert got_p[at:at + n_new[b]].cpu().tolist() == list(range(filled[b], filled[b] + n_new[b]))
        at += n_new[b]


def test_index_prep_rejects_wrong_dtypes_and_lengths(gpu):
    with pytest.raises(TypeError):
        kvc.get_seq_lens(torch.zeros(3, dtype=torch.int64, device=gpu), _up([1, 1], gpu), 16)
    with pytest.raises(ValueError):
        kvc.get_seq_lens(_up([0, 1], gpu), _up([1, 1], gpu), 16)
    with pytest.raises(ValueError):
        kvc.get_batch_indices_positions(_up([0, 1], gpu), _up([1, 1], gpu), 1)


@pytest.mark.parametrize("kind", ["decode", "chunked_prefill", "mixed", "large_batch", "empty"])
def test_one_launch_index_build_matches_the_host_construction(gpu, kind):
    """Prefix sums, last-page lengths, request indices, positions and slots from
    one device launch equal what the host-side construction (the restatement of
    the reference's list building) produces."""
    import workloads as wl
    rng = np.random.default_rng(11)
    bs = 16
    if kind == "decode":
        reqs = wl.decode_step(wl.LLAMA_3_8B, num_blocks=4096, batch=256, max_context=200, seed=5).inputs
    elif kind == "chunked_prefill":
        reqs = wl.chunked_prefill(wl.QWEN_2_5_7B, num_blocks=16384, seed=6).inputs
    elif kind == "mixed":
        filled = [0, 37, 5, 64, 200, 16, 15, 0]
        new = [70, 1, 1, 33, 1, 16, 2, 1]
        reqs = wl._write_workload(wl.LLAMA_3_2_1B, 256, filled, new, rng).inputs
    elif kind == "large_batch":                       # more requests than one scan chunk
        filled = rng.integers(0, 40, size=2500).tolist()
        new = rng.integers(1, 4, size=2500).tolist()
        reqs = wl._write_workload(wl.LLAMA_3_2_1B, 16384, filled, new, rng).inputs
    else:
        reqs = []
    host = kvc.make_kv_index_inputs(reqs, bs)
    dev = kvc.to_device_one_launch(reqs, bs, gpu)
    torch.cuda.synchronize()
    # the oracle's statement of the same index, from the per-request scalars in batch order
    ordered = [reqs[i] for i in host.order]
    want = orc.build_write_index_np([r.input_len for r in ordered], [r.context_len for r in ordered],
                                    [len(r.block_ids) for r in ordered],
                                    [b for r in ordered for b in r.block_ids], bs)
    for got, exp in zip((dev.cu_seqlens_q, dev.kv_block_indptrs, dev.kv_last_block_lens,
                         dev.batch_indices, dev.positions, dev.slot_mapping), want):
        assert np.array_equal(got.cpu().numpy(), exp)
    assert np.array_equal(dev.cu_seqlens_q.cpu().numpy(), host.cu_seqlens_q)
    assert np.array_equal(dev.kv_block_indptrs.cpu().numpy(), host.kv_block_indptrs)
    assert np.array_equal(dev.kv_last_block_lens.cpu().numpy(), host.kv_last_block_lens)
    assert np.array_equal(dev.kv_block_indices.cpu().numpy(), host.kv_block_indices)
    assert np.array_equal(dev.batch_indices.cpu().numpy(), host.batch_indices)
    assert np.array_equal(dev.positions.cpu().numpy(), host.position_ids)
    assert np.array_equal(dev.slot_mapping.cpu().numpy(), host.slot_mapping)
    assert dev.prefill_input_len == host.prefill_input_len
    # and it agrees with the two-call device path
    two = kvc.to_device(host, bs, gpu)
    assert torch.equal(two.batch_indices, dev.batch_indices)
    assert torch.equal(two.positions, dev.positions)


def test_one_launch_index_build_marks_positions_outside_the_table(gpu):
    cu, indptr, last, bi, pos, slots = kvc.build_write_index(
        _up([2, 1], gpu), _up([40, 5], gpu), _up([1, 1], gpu), _up([7, 3], gpu), 16, 3)
    assert cu.tolist() == [0, 2, 3] and indptr.tolist() == [0, 1, 2] and last.tolist() == [8, 5]
    assert pos.tolist() == [38, 39, 4]
    # request 0 claims 40 tokens with a single block: positions 38, 39 index past its table
    assert slots.tolist()[2] == 3 * 16 + 4
    assert slots.tolist()[0] == -1 and slots.tolist()[1] == -1
    # a position past the request's OWN table must not borrow the next request's block
    _, _, _, _, pos, slots = kvc.build_write_index(
        _up([1, 1], gpu), _up([20, 5], gpu), _up([1, 1], gpu), _up([7, 3], gpu), 16, 2)
    assert pos.tolist() == [19, 4] and slots.tolist() == [-1, 3 * 16 + 4]


@pytest.mark.parametrize("sizes", [
    [1], [1] * 1024, [1] * 1025,                     # one scan chunk, and one request beyond it
    [1024], [1025], [700, 324, 1], [2048, 1, 1],     # a round of 1024 tokens per workgroup, and one token more
    [5000, 3, 2, 1],                                 # 20 000 block ids: several workgroups upload them
], ids=str)
def test_index_from_requests_at_the_edges_of_its_launch(gpu, sizes):
    """Requests packed into the staging ring, against the oracle's statement of the index: every remainder of
    the 16-byte upload, more calls in flight than the ring has buffers, on two streams."""
    rng = np.random.default_rng(len(sizes) + sizes[0])
    ps = 4
    calls = []
    for k in range(9):
        reqs = []
        for i, n in enumerate(sizes[:len(sizes) - (k % 2 if len(sizes) > 1 else 0)]):
            filled = int(rng.integers(0, 50))
            blocks = (filled + n + ps - 1) // ps + (k if i == 0 else 0)    # tables may be longer than needed
            blocks += 20000 if n == 5000 else 0
            reqs.append(kvc.InferInput(i, [], n, filled, filled + n, rng.integers(0, 1 << 20, blocks).tolist()))
        calls.append([reqs[i] for i in rng.permutation(len(reqs))])
    streams = [torch.cuda.current_stream(gpu), torch.cuda.Stream(gpu)]
    got = []
    for k, reqs in enumerate(calls):
        with torch.cuda.stream(streams[k % 2]):
            got.append(kvc.to_device_one_launch(reqs, ps, gpu))
    torch.cuda.synchronize()
    for reqs, dev in zip(calls, got):
        ordered = sorted(reqs, key=lambda r: -r.input_len)
        ids = [b for r in ordered for b in r.block_ids]
        want = orc.build_write_index_np([r.input_len for r in ordered], [r.context_len for r in ordered],
                                        [len(r.block_ids) for r in ordered], ids, ps)
        for g, w in zip((dev.cu_seqlens_q, dev.kv_block_indptrs, dev.kv_last_block_lens, dev.batch_indices,
                         dev.positions, dev.slot_mapping, dev.kv_block_indices), list(want) + [np.asarray(ids)]):
            assert np.array_equal(g.cpu().numpy(), w)


def test_a_step_beyond_what_is_staged(gpu):
    """Block tables of 16 MiB and one request more than that take the unstaged path: the same index."""
    small = kvc.InferInput(1, [], 3, 5, 8, [9])
    for ids in ((16 << 20) // 4 - 2000, (16 << 20) // 4):
        table = list(range(ids))
        reqs = [small, kvc.InferInput(0, [], 2, 16 * ids - 2, 16 * ids, table)]
        got = kvc.to_device_one_launch(reqs, 16, gpu)
        step = kvc.KVWriteStep(1, 64, 16, torch.bfloat16, gpu, max_requests=2, max_tokens=5, max_block_ids=ids + 1)
        assert step.set_requests(reqs) == [0, 1]
        step.build_index()
        want = [9 * 16 + 5, 9 * 16 + 6, 9 * 16 + 7, 16 * ids - 2, 16 * ids - 1]
        assert got.slot_mapping.tolist() == want and step.slot_mapping.tolist() == want
        assert torch.equal(got.kv_block_indices, torch.tensor([9] + table, dtype=torch.int32, device=gpu))
        assert torch.equal(step.kv_indices, got.kv_block_indices)


def _check_build(reqs, gpu):
    want = kvc.to_device(kvc.make_kv_index_inputs(reqs, 16), 16, gpu)
    got = kvc.to_device_one_launch(reqs, 16, gpu)
    for name in ("cu_seqlens_q", "kv_block_indptrs", "kv_last_block_lens", "kv_block_indices", "batch_indices",
                 "positions", "slot_mapping"):
        assert torch.equal(getattr(got, name), getattr(want, name)), name


@pytest.mark.parametrize("ids", [1, 3, 4095, 4096, 4097, 4099])
@pytest.mark.parametrize("tokens", [1, 1500])
def test_tables_that_one_workgroup_reads_whole_and_longer_ones(gpu, ids, tokens):
    """On either side of 4096 block ids, with one workgroup of tokens and with two."""
    table = np.random.default_rng(ids + tokens).integers(0, 1 << 20, ids).tolist()
    cut = ids - ids // 3
    _check_build([kvc.InferInput(i, [], n, 16 * len(t) - n, 16 * len(t), t)
                  for i, t in enumerate((table[:cut], table[cut:])) if t for n in (min(tokens, 16 * len(t)),)], gpu)


def test_one_launch_index_build_reports_an_allocation_that_fails(gpu):
    """As an exception of the interpreter; the next call works."""
    huge = [kvc.InferInput(seq_id=0, input_ids=[], input_len=1 << 29, filled_token_len=0, context_len=1 << 29,
                           block_ids=[0])]
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(0.01)       # below the 8 GiB of output tensors
    try:
        with pytest.raises(torch.cuda.OutOfMemoryError):
            kvc.to_device_one_launch(huge, 16, gpu)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    import workloads as wl
    _check_build(wl.decode_step(wl.LLAMA_3_8B, num_blocks=256, batch=8, max_context=100, seed=1).inputs, gpu)


def _long_work(gpu, x):
    """About 0.2 s on the current stream; the event behind it."""
    for _ in range(150):
        x @ x
    done = torch.cuda.Event()
    done.record()
    return done


def test_index_builds_far_ahead_of_the_device_and_from_threads_that_end(gpu):
    """More builds than staging buffers behind long work: the fifth waits for a buffer without the interpreter's lock.
    Of threads that end, the fifth comes round to a buffer whose reader, an ended thread's, is still queued. Every
    build reads its own requests."""
    import threading
    import time
    import workloads as wl
    steps = [wl.decode_step(wl.LLAMA_3_8B, num_blocks=512, batch=8 + i, max_context=300, seed=i).inputs
             for i in range(12)]
    want = [kvc.to_device(kvc.make_kv_index_inputs(r, 16), 16, gpu) for r in steps]
    x = torch.ones(4096, 4096, device=gpu)
    _long_work(gpu, x)
    torch.cuda.synchronize()
    ticks, stop, got, waits = [0], threading.Event(), [], []

    def tick():
        while not stop.is_set():
            time.sleep(0.001)
            ticks[0] += 1

    def build(requests):
        t0 = time.perf_counter()
        got.append(kvc.to_device_one_launch(requests, 16, gpu))
        waits.append(time.perf_counter() - t0)

    ticker = threading.Thread(target=tick)
    ticker.start()
    try:
        _long_work(gpu, x)
        for r in steps[:4]:
            build(r)
        before = ticks[0]
        build(steps[4])
        ticked = ticks[0] - before
        for r in steps[5:6]:
            build(r)
        torch.cuda.synchronize()
        _long_work(gpu, x)
        for r in steps[6:]:
            worker = threading.Thread(target=build, args=(r,))
            worker.start()
            worker.join()
    finally:
        stop.set()
        ticker.join()
    torch.cuda.synchronize()
    assert len(got) == len(steps)
    assert waits[4] >= 0.05 and ticked >= waits[4] / 0.005, (waits, ticked)
    assert waits[10] >= 0.05 and max(waits[6:10]) < waits[10], waits
    for g, w in zip(got, want):
        assert torch.equal(g.slot_mapping, w.slot_mapping) and torch.equal(g.kv_block_indices, w.kv_block_indices)


def test_staging_grows_while_its_readers_are_queued(gpu):
    """A step whose tables outgrow the buffers behind long work: the call waits for no buffer and for no device, and
    the builds queued before it still read what they were given."""
    def step(ids, start):
        return [kvc.InferInput(0, [], 2, 16 * ids - 2, 16 * ids, list(range(start, start + ids)))]

    small, large = [step(3000, k) for k in range(8)], [step(20000 << k, 7) for k in range(3)]
    _lib.check(_lib.lib().kvc_thread_release())
    for r in small[:4]:                                      # four buffers of 64 KiB
        kvc.to_device_one_launch(r, 16, gpu)
    x = torch.ones(4096, 4096, device=gpu)
    torch.empty(1 << 22, device=gpu)                         # room for the outputs below in the allocator's cache
    _long_work(gpu, x)
    torch.cuda.synchronize()
    done = _long_work(gpu, x)
    got = [kvc.to_device_one_launch(r, 16, gpu) for r in small[4:] + large]
    assert not done.query()
    for g, r in zip(got, small[4:] + large):
        ids = r[0].block_ids
        assert torch.equal(g.kv_block_indices, torch.tensor(ids, dtype=torch.int32, device=gpu))
        assert g.slot_mapping.tolist() == [16 * ids[-1] + 14, 16 * ids[-1] + 15]


@pytest.mark.parametrize("tokens,page", [(1, 16), (3, 1), (1023, 16), (4099, 7)])
def test_host_arrays_on_the_device_in_every_form(gpu, tokens, page):
    """Dense arrays through the staging ring, more calls than it has buffers, on two streams; strided
    arrays take the copies: the same tensors."""
    rng = np.random.default_rng(tokens)
    filled = int(rng.integers(0, 40))
    # tables of exactly the blocks a context needs: the device derives the context from the table's length
    reqs = [kvc.InferInput(i, [], n, filled, filled + n, rng.integers(0, 1 << 24, -(-(filled + n) // page)).tolist())
            for i, n in enumerate([1, tokens, 2])]
    host = kvc.make_kv_index_inputs(reqs, page)
    strided = kvc.KVIndexInputs(**{k: np.repeat(v, 2)[::2] if isinstance(v, np.ndarray) else v
                                   for k, v in vars(host).items()})
    side = torch.cuda.Stream(gpu)
    got = [kvc.to_device(h, page, gpu, slots) for h in (host, strided) for slots in (True, False)]
    with torch.cuda.stream(side):
        got += [kvc.to_device(host, page, gpu) for _ in range(7)]
    torch.cuda.synchronize()
    for dev in got:
        for name in ("position_ids", "cu_seqlens_q", "kv_block_indices", "kv_block_indptrs", "kv_last_block_lens",
                     "batch_indices", "positions", "slot_mapping"):
            t, want = getattr(dev, name), getattr(host, name)
            if t is not None:
                assert t.is_contiguous() and t.device == gpu and np.array_equal(t.cpu().numpy(), want), name
    assert got[1].slot_mapping is None and got[3].slot_mapping is None
    host.slot_mapping = None
    assert kvc.to_device(host, page, gpu, False).slot_mapping is None
    with pytest.raises(TypeError):                        # slots wanted, none there
        kvc.to_device(host, page, gpu)


# (a general path reads what an int subclass stores, by struct.pack: "ids converted" is the host arrays' own)
@pytest.mark.parametrize("form", MAPPED_FORMS[:-1])
def test_requests_are_read_as_they_read_themselves(gpu, form):
    """Subclasses that map or load their elements on read, by both ways to the device; an empty step only
    where the requests are empty."""
    reqs, _ = mapped_requests(form)
    got = kvc.to_device_one_launch(reqs, 16, gpu)
    assert got.slot_mapping.tolist() == [107 * 16 + 1, 107 * 16 + 2, 103 * 16]
    assert got.kv_block_indices.tolist() == [107, 103]
    step = kvc.KVWriteStep(1, 64, 16, torch.bfloat16, gpu, max_requests=3, max_tokens=4, max_block_ids=5)
    assert step.set_requests(reqs) == [0, 1]
    step.build_index()
    assert step.slot_mapping.tolist() == [107 * 16 + 1, 107 * 16 + 2, 103 * 16, -1]


@pytest.mark.parametrize("sizes", [
    [1], [0, 5, 0], [1] * 15 + [300], [1] * 17, [2] * 1030, [4099, 1, 64, 65, 0, 63],
    [1] * 16500,        # more than a lane of every workgroup has
])
def test_host_arrays_uploaded_in_one_launch(gpu, sizes):
    """batch_indices and positions that the upload derives, against the host's own, requests without new tokens among
    them."""
    rng = np.random.default_rng(len(sizes))
    reqs = []
    for i, n in enumerate(sizes):
        filled = int(rng.integers(0 if n else 1, 40))
        reqs.append(kvc.InferInput(seq_id=i, input_ids=[0] * n, input_len=n, filled_token_len=filled, context_len=filled + n,
                                   block_ids=rng.integers(0, 1000, (filled + n + 15) // 16).tolist()))
    host = kvc.make_kv_index_inputs(reqs, 16)
    got = kvc.to_device(host, 16, gpu)
    want = np.repeat(np.arange(len(sizes)), np.diff(host.cu_seqlens_q))
    assert np.array_equal(got.batch_indices.cpu().numpy(), want)
    assert np.array_equal(got.positions.cpu().numpy(), host.position_ids)
    for name in ("position_ids", "cu_seqlens_q", "kv_block_indices", "kv_block_indptrs", "kv_last_block_lens", "slot_mapping"):
        assert np.array_equal(getattr(got, name).cpu().numpy(), getattr(host, name)), name


def test_upload_of_index_arrays_refuses_what_lies_outside(gpu):
    lib = _lib.lib()
    dst = torch.zeros(64, dtype=torch.int32, device=gpu)
    out = torch.zeros(8, dtype=torch.int32, device=gpu)
    for bytes_, cu, ptr, last, batch in ((64, 0, 16, 52, 4), (64, -4, 16, 32, 2), (64, 2, 16, 32, 2), (60, 0, 16, 32, 2),
                                         (64, 0, 60, 32, 2), (64, 0, 16, 32, 0), (64, 0, 16, 32, 2**40)):
        rc = lib.kvc_staging_upload_index(dst.data_ptr(), bytes_, cu, ptr, last, batch, 16, 4, out.data_ptr(),
                                          out.data_ptr(), torch.cuda.current_stream().cuda_stream)
        assert rc == _lib.KVC_ERR_INVALID_ARG


@pytest.mark.parametrize("sizes", [
    [256], [257], [1, 256, 257, 0, 512, 255], [70001, 3],
    [1] * 33000 + [300, 2, 258],       # in the second round of a workgroup's lanes
])
def test_long_requests_uploaded_in_one_launch(gpu, sizes):
    """Requests of more tokens than a workgroup has lanes, among short ones, in the order given."""
    sizes = np.asarray(sizes)
    rng = np.random.default_rng(len(sizes))
    filled = rng.integers(1, 40, len(sizes))
    blocks = (filled + sizes + 15) // 16
    i32 = lambda a: np.asarray(a, dtype=np.int32)
    cu, indptr = i32(np.concatenate([[0], np.cumsum(sizes)])), i32(np.concatenate([[0], np.cumsum(blocks)]))
    requests = np.repeat(np.arange(len(sizes)), sizes)
    positions = np.arange(cu[-1]) - cu[requests] + filled[requests]
    host = kvc.KVIndexInputs(i32(positions), cu, 0, i32(rng.integers(0, 1000, indptr[-1])), indptr,
                             i32((filled + sizes - 1) % 16 + 1), i32(requests), i32(positions),
                             positions.astype(np.int64), list(range(len(sizes))))
    got = kvc.to_device(host, 16, gpu)
    for name in ("batch_indices", "positions", "position_ids", "cu_seqlens_q", "kv_block_indices", "kv_block_indptrs",
                 "kv_last_block_lens", "slot_mapping"):
        assert np.array_equal(getattr(got, name).cpu().numpy(), getattr(host, name)), name
