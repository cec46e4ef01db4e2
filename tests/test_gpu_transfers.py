"""Host <-> device transfers: the pinned upload ring, staged and direct downloads, host arrays of the library's own.  Values
travel as they are, so every comparison is of bits."""
import gc
import os
import resource

import numpy as np
import pytest

from deepj_amd import HipNative, Tensor
from deepj_amd._native import host_array, library
from deepj_amd.fused import DeviceBuffers
from gpu_util import backend, tensor

pytestmark = pytest.mark.gpu

PIECE = 1 << 16                  # floats of one piece of the upload ring
SEGMENT = 1 << 18                # of one of its four segments: the pieces of uploads of more than two
RING = 1 << 20                   # floats it holds; larger uploads are copied by two threads


@pytest.fixture
def dev():
    d = DeviceBuffers()
    yield d
    d.release_all()


def values(n, seed):
    return np.random.default_rng(seed).integers(-2 ** 31, 2 ** 31, n, dtype=np.int64).astype(np.int32)


def read(dev, buf, n):
    out = np.empty(n, np.int32)
    HipNative.nativeDownloadBuffer(buf, out)
    return out


@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 1021, PIECE - 1, PIECE, PIECE + 1, 2 * PIECE + 3, SEGMENT - 1, SEGMENT, SEGMENT + 1,
                               2 * SEGMENT, 2 * SEGMENT + 1, 3 * SEGMENT + 5, RING, RING + 1, RING + SEGMENT + 33, 4 * RING + 3])
def test_an_upload_of_any_size_arrives_whole_and_nothing_behind_it(dev, n):
    """Parts of a piece, several pieces, large ones, those that two threads copy; from a source that is not 16-byte aligned."""
    a, old = values(n + 1, n)[1:], values(n + 7, n + 1)
    buf = dev.upload(old)
    dev.write(buf, a)
    got = read(dev, buf, n + 7)
    assert np.array_equal(got[:n], a) and np.array_equal(got[n:], old[n:])


def test_uploads_of_several_rings_before_anything_waits(dev):
    """More than the ring holds, many times over, in sizes that leave every segment's end ragged: none may be overwritten in
    the ring before its launch has read it."""
    sizes, total, rng = [], 0, np.random.default_rng(5)
    while total < 8 * RING:
        sizes.append(int(rng.choice([1, 7, 300, 5000, PIECE - 5, PIECE, 2 * PIECE + 9, SEGMENT, RING + 77])))
        total += (sizes[-1] + 63) // 64 * 64
    sent = [values(n, i) for i, n in enumerate(sizes)]
    bufs = [dev.upload(a) for a in sent]
    for i in range(0, len(sent), 3):                       # a third of them again, while the first may still be on the link
        sent[i] = values(sizes[i], 1000 + i)
        dev.write(bufs[i], sent[i])
    for a, b in zip(sent, bufs):
        assert np.array_equal(read(dev, b, a.size), a)


@pytest.mark.parametrize("large", [100, SEGMENT + 64, RING + 64])
def test_uploads_into_the_same_buffer_land_in_their_order(dev, large):
    """The whole buffer, its beginning, the whole again and a shorter beginning, before anything waits: staged words are replaced,
    or launched before the later ones are sent."""
    whole, first, again, short = values(large, 1), values(large // 2, 2), values(large, 3), values(17, 4)
    buf = dev.alloc(large)
    for seq in ([whole, first], [first, whole], [whole, first, again, short], [short, short + 1, first, whole, short]):
        exp = read(dev, buf, large)
        for a in seq:
            dev.write(buf, a)
            exp[:a.size] = a
        assert np.array_equal(read(dev, buf, large), exp)


def test_a_released_buffer_takes_no_upload_of_its_predecessor(dev):
    """The block of a released buffer goes to the next one of its size: what was staged for the first is written first."""
    for n in (40, 5000):
        for seed in range(4):
            a = dev.upload(values(n, seed))
            dev.release(a)
            b = dev.upload(values(n, 100 + seed))
            assert np.array_equal(read(dev, b, n), values(n, 100 + seed))
            dev.release(b)


@pytest.mark.parametrize("n", [1, 3, 2047, 2048, 2049, (512 << 10) // 4, (512 << 10) // 4 + 1, (1 << 20) - 1, (1 << 20) + 1, 2 * (1 << 20) + 4099])
@pytest.mark.parametrize("offset", [0, 1])
def test_a_download_into_ordinary_memory(dev, n, offset):
    """Through the stage: parts of a chunk, chunk edges, both chunk sizes, more than the 4 MiB stage; into memory that is not
    16-byte aligned, of a buffer that holds more; what surrounds the destination stays."""
    a = values(n + 9, n)
    buf, out = dev.upload(a), np.full(n + offset + 3, 7, np.int32)
    HipNative.nativeDownloadBuffer(buf, out[offset:offset + n])
    assert np.array_equal(out[offset:offset + n], a[:n])
    assert np.all(out[:offset] == 7) and np.all(out[offset + n:] == 7)


def test_a_small_buffer_is_read_while_uploads_to_others_are_staged(dev):
    """A download launches staged uploads only where it reads them."""
    a, b = values(33, 1), values(70, 2)
    ba, bb = dev.upload(a), dev.upload(b)
    assert np.array_equal(read(dev, ba, 33), a)
    dev.write(bb, b + 1)
    assert np.array_equal(read(dev, ba, 33), a)
    assert np.array_equal(read(dev, bb, 70), b + 1)


@pytest.fixture
def blocks():
    """host_alloc on a pool without blocks and without history."""
    HipNative.init(0)
    gc.collect()
    HipNative.trim()
    lib, taken = library(), []

    def take(size):
        p = lib.deepj_hip_host_alloc(size)
        if p:
            taken.append(p)
        return p

    def give(p):
        taken.remove(p)
        lib.deepj_hip_host_free(p)
    yield take, give
    for p in taken:
        lib.deepj_hip_host_free(p)
    HipNative.trim()


def test_pinned_blocks_are_made_for_sizes_that_are_asked_for_again_and_again(blocks):
    take, give = blocks
    size = 10 << 20
    assert [take(size - 100 * i) for i in range(4)] == [None] * 4      # the first results of about a size: ordinary memory
    a, b = take(size), take(size)
    assert a and b and a != b
    assert take(size) is None                                          # kept, not given back: no more of them
    for _ in range(2):
        assert take(size) is None
        give(a)
        assert take(size - 4096) == a
    c = take(size)                                                     # used again twice: one more is worth making
    assert c and take(size) is None
    give(b)
    assert take(3 << 20) == b                                          # up to four times what is asked for
    give(c)
    assert take(2 << 20) is None and take(65535) is None
    give(b)
    HipNative.trim()
    assert take(size) is None                                          # nothing kept, nothing remembered
    small = [take(1 << 20) for _ in range(4 + 16 + 2)]
    assert small[:4] == [None] * 4 and all(small[4:20]) and small[20:] == [None] * 2      # 16 MiB of them ahead of their use


def test_a_pinned_block_leaves_no_page_to_its_reader(blocks, dev):
    """Its pages are in use before it is handed out: the first look at a result must not pay for them."""
    take, _ = blocks
    n = 1 << 20
    for _ in range(4):
        take(4 * n)
    out = host_array(n)
    assert library().deepj_hip_host_alloc(0) is None and type(out.base).__name__ == "_HostBlock"
    buf = dev.upload(np.arange(n, dtype=np.int32))
    HipNative.nativeDownloadBuffer(buf, out)
    before = resource.getrusage(resource.RUSAGE_SELF).ru_minflt
    last = int(out.view(np.int32)[::1024].max())
    assert resource.getrusage(resource.RUSAGE_SELF).ru_minflt - before < 64 and last == n - 1024


def test_the_bound_on_pinned_memory_ends_in_ordinary_memory(blocks):
    take, give = blocks
    size = 300 << 20
    for _ in range(4):
        assert take(size) is None
    a, b = take(size), take(size)
    for _ in range(2):
        give(a)
        a = take(size)
    c = take(size)                                                     # 900 MiB (and what the size class adds) are out
    assert a and b and c
    for _ in range(4):
        give(c)
        c = take(size)
    assert c and take(size) is None                                    # another block would pass 1 GiB


@pytest.mark.parametrize("n", [1 << 14, (1 << 18) + 3, (1 << 20) + 1, 5 * (1 << 20) + 7])
def test_a_view_keeps_its_pinned_block(blocks, dev, n):
    """Results land in the block itself; a view that outlives its array keeps the block from the next result."""
    take, _ = blocks
    for _ in range(4):
        take(4 * n)
    a, b = values(n, 1), values(n, 2)
    ba, bb = dev.upload(a), dev.upload(b)
    first = host_array(n)
    assert type(first.base).__name__ == "_HostBlock"
    HipNative.nativeDownloadBuffer(ba, first)
    view = first[5:n - 1].view(np.int32)
    address = first.ctypes.data
    del first
    second = host_array(n)
    assert second.ctypes.data != address
    HipNative.nativeDownloadBuffer(bb, second)
    assert np.array_equal(view, a[5:n - 1]) and np.array_equal(second.view(np.int32), b)
    HipNative.nativeDownloadBuffer(bb, second[3:])                     # inside the block, where 128-bit words do not fit
    assert np.array_equal(second.view(np.int32)[3:], b[:n - 3]) and np.array_equal(second.view(np.int32)[:3], b[:3])
    del view
    third = host_array(n)
    assert third.ctypes.data == address


def test_a_forked_child_reads_results_in_pinned_memory(blocks, dev):
    """As a worker process does that was handed results: their values in the child, which changes its copy, gives it back and
    forks again; the parent's are untouched, and so is what it goes on to do."""
    take, _ = blocks
    n = (1 << 20) + 5
    for _ in range(4):
        take(4 * n)
    a, b = values(n, 1), values(n, 2)
    ba, bb = dev.upload(a), dev.upload(b)
    kept, dropped = host_array(n).view(np.int32), host_array(n).view(np.int32)
    assert type(kept.base.base).__name__ == "_HostBlock"
    HipNative.nativeDownloadBuffer(ba, kept)
    HipNative.nativeDownloadBuffer(bb, dropped)
    del dropped                                                        # a free block: the child has none
    pid = os.fork()
    if pid == 0:
        code = 1
        try:
            ok = np.array_equal(kept, a)
            kept[:] = 7
            grandchild = os.fork()
            if grandchild == 0:
                os._exit(0 if ok and int(kept.sum()) == 7 * n else 1)
            ok = ok and os.waitpid(grandchild, 0)[1] == 0
            other = host_array(n)
            ok = ok and type(other.base).__name__ != "_HostBlock"
            del kept
            code = 0 if ok else 2
        finally:
            os._exit(code)
    assert os.waitpid(pid, 0)[1] == 0
    assert np.array_equal(kept, a)
    again = host_array(n).view(np.int32)
    HipNative.nativeDownloadBuffer(bb, again)
    assert np.array_equal(again, b) and np.array_equal(kept, a)


@pytest.mark.parametrize("rows,cols", [(1, 1), (33, 7), (64, 64), (300, 1003)])
def test_tensors_nothing_was_written_to_are_zeros_on_the_device(rows, cols):
    """They are cleared there instead of being sent, in blocks that held other values before, next to tensors that are sent."""
    rng = np.random.default_rng(rows)
    with backend() as be:
        for _ in range(3):                                             # blocks of these sizes with something in them
            be.add(tensor(rng.standard_normal((rows, cols))), tensor(rng.standard_normal((rows, cols)))).numpy()
        be.graph.releaseAll()
        a = rng.standard_normal((rows, cols)).astype(np.float32)
        z1, z2, row = Tensor.zeros(rows, cols), Tensor.zeros(rows, cols), Tensor.zeros(1, cols)
        t = tensor(a)
        assert np.array_equal(be.add(be.add(t, z1), z2).numpy(), a)
        assert np.array_equal(be.addRowVector(t, row).numpy(), a)
        assert np.array_equal(be.multiply(z1, t).numpy(), np.zeros_like(a))
        late = Tensor.zeros(rows, cols)
        late.data[:] = a                                               # written before it was ever used: sent
        assert np.array_equal(be.add(late, z2).numpy(), a)
