"""Launches at the limits of sizes, on the CPU: the library's host code through the
stand-in HIP runtime (tests/fakehip), which reports a launch that the runtime would
refuse (a dimension of 2^32 threads or more) or that leaves bytes uncovered.  Device
memory is reserved and never touched, so sizes beyond a card's are fine.  CPU only.
"""
import ctypes
import threading

import pytest

from tests.test_host_launches import (BASIC, OK, TREE, Header, checkpoint, create, dev_alloc, fake, launches,  # noqa: F401
                                      violations)

GIB = 1 << 30


@pytest.mark.parametrize("size", [1, 4097, GIB, 64 * GIB - 1, 64 * GIB, 72 * GIB + 5])
@pytest.mark.parametrize("offset", [0, 4])
def test_device_copy_of_any_size(fake, size, offset):
    L = fake
    L.fakehip_reset()
    src, dst = dev_alloc(L, size), dev_alloc(L, size + offset)
    getattr(L, "_ZN3mtc11copy_deviceEPKhPhmP12ihipStream_t")(src, ctypes.c_void_p(dst.value + offset), ctypes.c_uint64(size), None)
    assert any("k_copy" in n for n in launches(L))
    assert violations(L) == []
    for p in (src, dst):
        L.hipFree(p)


@pytest.mark.parametrize("C,datalen", [(1000, 63 * GIB), (1000, 72 * GIB + 5), (1 << 20, 72 * GIB), (1 << 20, 256 * GIB + 7)])
@pytest.mark.parametrize("offset", [0, 4])
def test_restart_of_any_size(fake, C, datalen, offset):
    """A header without regions is a chain as far as the host sees it."""
    L = fake
    L.fakehip_reset()
    diff = Header(0, 0, datalen, C, 0, 0, 0)
    out = dev_alloc(L, datalen + offset)
    ptrs = (ctypes.c_void_p * 1)(ctypes.addressof(diff))
    sizes = (ctypes.c_uint64 * 1)(32)
    assert L.mtc_restart(ptrs, sizes, 1, 0, 0, ctypes.c_void_p(out.value + offset), ctypes.c_uint64(datalen), 0, None) == OK
    assert any("k_r_copy" in n for n in launches(L))
    assert violations(L) == []
    L.hipFree(out)


def test_batch_of_large_baselines(fake):
    """Sixteen baselines of 2^20 one-chunk tiles each."""
    L = fake
    L.fakehip_reset()
    b = ctypes.c_void_p()
    assert L.mtc_batch_create(ctypes.byref(b), 0, 0) == OK
    B, C = 16, 8193
    size = C << 20
    hs = [create(L, C, BASIC) for _ in range(B)]
    H = (ctypes.c_void_p * B)(*[h.value for h in hs])
    datas = [dev_alloc(L, size) for _ in range(B)]
    D = (ctypes.c_void_p * B)(*[d.value for d in datas])
    N = (ctypes.c_uint64 * B)(*[size] * B)
    assert L.mtc_checkpoint_batch(b, H, D, N, (ctypes.c_int * B)(*[1] * B), B, 1, None, None, None) == OK
    assert violations(L) == []
    for h in hs:
        L.mtc_destroy(h)
    for d in datas:
        L.hipFree(d)
    L.mtc_batch_destroy(b)


@pytest.mark.parametrize("C", [16384, 16385, 0xFFFFC000, 0xFFFFC001, 0xFFFFF001, 0xFFFFFFFF])
@pytest.mark.parametrize("approach", [TREE, BASIC])
def test_gather_tiles_of_the_largest_chunks(fake, C, approach):
    """A chunk larger than a gather tile (16 KiB) is sliced, up to the largest chunk
    size: a baseline of one chunk has a block for every slice and one for the header."""
    L = fake
    L.fakehip_reset()
    L.fakehip_launch_blocks.restype = ctypes.c_uint64
    h = create(L, C, approach)
    data = dev_alloc(L, 1000)
    rc, _ = checkpoint(L, h, data, 1000, baseline=True)
    assert rc == OK, L.mtc_last_error(h)
    blocks = [L.fakehip_launch_blocks(i) for i, n in enumerate(launches(L)) if "assemble" in n or "basic_diff" in n]
    assert blocks == [1 + -(-C // 16384)]
    assert violations(L) == []
    L.mtc_destroy(h)


def test_copies_of_one_handle_by_two_threads(fake):
    """Each copy takes its time between events of its own."""
    L = fake
    L.fakehip_reset()
    h = create(L, 128)
    data = dev_alloc(L, 1 << 20)
    L.fakehip_set_diff_size(ctypes.c_uint64(5000))
    assert checkpoint(L, h, data, 1 << 20, baseline=True)[0] == OK
    dst = [dev_alloc(L, 5000) for _ in range(2)]
    for _ in range(2):  # the second time with what the first one left in the handle
        L.fakehip_hold(2)
        rcs = []
        ts = [threading.Thread(target=lambda p=p: rcs.append(L.mtc_copy_diff(h, p, ctypes.c_uint64(5000), None))) for p in dst]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        L.fakehip_hold(0)
        assert rcs == [OK, OK]
        assert violations(L) == []
    L.fakehip_reset()
    L.mtc_destroy(h)


@pytest.mark.parametrize("room", [5000, 4999, 64])
def test_device_copy_stays_in_the_destination(fake, room):
    """The runtime refuses a copy past the end of the destination's allocation.  A
    capacity larger than the allocation still ends in that refusal, not in a kernel."""
    L = fake
    L.fakehip_reset()
    h = create(L, 128)
    data = dev_alloc(L, 1 << 20)
    L.fakehip_set_diff_size(ctypes.c_uint64(5000))
    assert checkpoint(L, h, data, 1 << 20, baseline=True)[0] == OK
    p = dev_alloc(L, room + 16)
    L.fakehip_reset()
    rc = L.mtc_copy_diff(h, ctypes.c_void_p(p.value + 16), ctypes.c_uint64(1 << 20), None)
    copied = any("k_copy" in n for n in launches(L))
    assert (rc, copied) == ((OK, True) if room >= 5000 else (6, False))
    L.fakehip_reset()
    L.mtc_destroy(h)


# What covers a chain's diffs, launch by launch: chunks (C) or shifted entries (S) of one diff by
# plain stores, or all that is left of several by atomics (A).
@pytest.mark.parametrize("chunks,shifted,order", [
    ([5], [0], "C"),
    ([5, 5, 5], [0, 0, 0], "CA"),                       # the oldest diff's chunks, then all others together
    ([5, 5, 5], [3, 3, 3], "CA"),
    ([5], [3], "CA"),
    ([1 << 22, 5, 5], [0, 0, 3], "CA"),
    ([0, 1 << 22, 5, 1 << 22], [0, 0, 0, 0], "CCAC"),   # in the chain's order
    ([0, 1 << 22, 5, 1 << 22], [3, 3, 3, 3], "CACACA"),
    ([5, 5, 1 << 22, (1 << 22) - 1], [0, 0, 0, 0], "CACA"),
    ([5], [1 << 22], "CS"),
    ([0], [(1 << 22) - 1], "CA"),
    ([5, 5, 5], [1 << 22, 0, 5], "CSA"),
    ([5, 5, 5], [5, 1 << 22, 5], "CASA"),
    ([0, 1 << 22, 1], [0, 1 << 22, 1], "CCSA"),
    ([0, 0, 0], [0, (1 << 22) - 1, 1 << 22], "CAS"),
])
def test_large_diffs_of_a_chain_are_covered_by_plain_stores(fake, chunks, shifted, order):
    L = fake
    L.fakehip_reset()
    n = 1 << 23
    bufs = [ctypes.create_string_buffer(bytes(Header(0, k, n, 1, 0, 0, s)), 32 + 8 * s + f) for k, (f, s) in enumerate(zip(chunks, shifted))]
    ptrs = (ctypes.c_void_p * len(bufs))(*[ctypes.addressof(b) for b in bufs])
    sizes = (ctypes.c_uint64 * len(bufs))(*[len(b) for b in bufs])
    out = dev_alloc(L, n)
    assert L.mtc_restart(ptrs, sizes, len(bufs), len(bufs) - 1, 0, out, ctypes.c_uint64(n), 0, None) == OK
    assert "".join("C" if "base" in k else "S" if "Lb1" in k else "A" for k in launches(L) if "k_r_cover" in k) == order
    assert violations(L) == []
    L.hipFree(out)


@pytest.mark.parametrize("hk,C,n,offset,alone,leaf", [
    # what one of the kernels for a chunk size takes, whatever its number
    (0, 128, 5, 0, 128, 128), (1, 4096, 9, 16, 4096, 4096),
    # Murmur3: 0 is the staged kernel, -1 the one by bytes
    (0, 19, 90_000, 0, -1, -1), (0, 20, 90_000, 0, -1, -1), (0, 25, 700_000, 1, 0, -1), (0, 26, 90_000, 0, 0, 0),
    (0, 50, 90_000, 0, 0, 0), (0, 64, 1 << 22, 4, 0, -1), (0, 64, 1 << 22, 1, 0, -1),
    (0, 1000, 200_000, 0, 0, 0), (0, 100, 5_000, 0, 0, -1), (0, 100, 5_243, 0, 0, 0), (0, 99, 5_000, 0, 0, 0),
    (0, 320, 100_000, 0, 0, -1), (0, 320, 110_000, 0, 0, 0), (0, 320, 100_000, 1, 0, 0),
    (0, 4096, 100_000, 4, 0, -1), (0, 4096, 1 << 17, 4, 0, 0), (0, 8192, 16_383, 0, -1, -1), (0, 8192, 16_384, 0, 0, -1),
    (0, 8192, 1 << 17, 0, 0, 0), (0, 8192, 1_000, 3, 0, 0),
    # MD5
    (1, 1000, 65_535, 0, -1, -1), (1, 1000, 65_536, 0, 0, 0), (1, 24, 1 << 20, 0, 0, -1), (1, 25, 1 << 20, 0, 0, 0),
    (1, 64, 1 << 20, 1, -1, -1), (1, 128, 1 << 20, 4, -1, -1), (1, 128, 1 << 20, 1, 0, 0), (1, 960, 1 << 20, 0, -1, -1),
    (1, 1024, 131_071, 4, -1, -1), (1, 1024, 131_072, 4, 0, 0), (1, 8192, 1 << 18, 0, 0, -1),
    (1, 72, 1 << 20, 0, 0, -1), (1, 200, 262_143, 0, -1, -1), (1, 200, 262_144, 0, 0, 0), (1, 200, 100_000, 2, 0, 0),
    (1, 204, 100_000, 0, 0, 0), (1, 5000, 100_000, 0, 0, 0),
])
def test_kernel_of_a_chunk_size(fake, hk, C, n, offset, alone, leaf):
    """Which kernel hashes chunks: where staging them was measured to be the slower way, alone or
    in a checkpoint, they go by bytes."""
    L = fake
    L.fakehip_reset()
    size = n * C
    data, out = dev_alloc(L, size + 16), dev_alloc(L, 16 * n)
    p = ctypes.c_void_p(data.value + offset)
    assert L.mtc_hash_chunks(p, ctypes.c_uint64(size), C, hk, out, None) == OK
    tag = lambda cb: f"ILi{hk}ELi{'n' if cb < 0 else ''}{abs(cb)}E"  # noqa: E731
    assert [k for k in launches(L) if "k_hash_chunks" + tag(alone) in k], launches(L)
    h = create(L, C, TREE, hk)
    L.fakehip_reset()
    assert checkpoint(L, h, p, size, baseline=True)[0] == OK
    names = [k for k in launches(L) if "k_leaf" in k]
    assert len(names) == 1 and tag(leaf) in names[0], names
    assert violations(L) == []
    L.mtc_destroy(h)
    L.hipFree(data)
    L.hipFree(out)


@pytest.mark.parametrize("entries,one_piece", [(0, True), (21 / 32, True), (22 / 32, True), (23 / 32, False), (3 / 4, False), (7 / 8, False)])
def test_a_step_that_could_fill_the_table_waits_for_its_bound(fake, entries, one_piece):
    """n = 2^12 chunks have 2^15 slots; a step may add 2^13 - 1 entries.  It runs in one piece
    only while that leaves a sixteenth of the slots empty (probes grow with the square of
    the empty share's inverse); else it pauses for the exact bound."""
    L = fake
    L.fakehip_reset()
    n, C = 1 << 12, 128
    h = create(L, C)
    data = dev_alloc(L, n * C)
    L.fakehip_set_claims(ctypes.c_uint64(int(entries * 8 * n)))
    assert checkpoint(L, h, data, n * C, baseline=True)[0] == OK
    L.fakehip_reset()
    assert checkpoint(L, h, data, n * C)[0] == OK
    assert any("k_leaf1_direct" in k for k in launches(L)) == one_piece
    assert violations(L) == []
    L.mtc_destroy(h)
    L.hipFree(data)


def test_a_table_of_half_the_usual_load_takes_a_baseline(fake):
    """At load factor 0.5 a baseline's 2n - 1 entries could fill the 2n slots: it pauses, and
    the table grows first."""
    L = fake
    L.fakehip_reset()
    n, C = 1 << 12, 128
    h = create(L, C)
    assert L.mtc_set_tuning(h, 1, ctypes.c_float(0.5), 8) == OK
    data = dev_alloc(L, n * C)
    for k in range(3):
        assert checkpoint(L, h, data, n * C, baseline=(k != 1))[0] == OK, L.mtc_last_error(h)
    assert violations(L) == []
    L.mtc_destroy(h)
    L.hipFree(data)


@pytest.mark.parametrize("C,datalen", [(15, 1), (15, 29 * GIB + 3), (4, 8 * GIB - 4), (16, 30 * GIB + 3), (17, 16)])
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_restart_copies_whole_words(fake, C, datalen, offset):
    """Chunks under 16 bytes by threads of a word each, larger ones by threads of four, from the word
    on that the output starts in."""
    L = fake
    L.fakehip_reset()
    diff = Header(0, 0, datalen, C, 0, 0, 0)
    out = dev_alloc(L, datalen + offset)
    ptrs = (ctypes.c_void_p * 1)(ctypes.addressof(diff))
    sizes = (ctypes.c_uint64 * 1)(32)
    assert L.mtc_restart(ptrs, sizes, 1, 0, 0, ctypes.c_void_p(out.value + offset), ctypes.c_uint64(datalen), 0, None) == OK
    copies = [n for n in launches(L) if "k_r_copy" in n]
    assert len(copies) == 1 and (C == 16 and offset == 0 or f"k_r_copy_anyILj{4 if C < 16 else 16}E" in copies[0]), copies
    assert violations(L) == []
    L.hipFree(out)
