"""Series at the sizes where a kernel's work split changes, byte for byte against the
oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import first_mismatch

torch = pytest.importorskip("torch")
import mtcheck_amd as M  # noqa: E402

pytestmark = pytest.mark.gpu


def same_as_oracle(versions, C, hk=0):
    """Diffs of a series equal the oracle's; returns them."""
    d, orc, diffs = M.TreeDeduplicator(C, hash_kind=hk), O.OracleDedup(C, hk), []
    for k, host in enumerate(versions):
        print(f"checkpoint {k} of {len(host)} bytes, C={C}, hash {hk}", flush=True)
        g = d.checkpoint(torch.from_numpy(host.copy()).to("cuda:0"), make_baseline=(k == 0))
        e = orc.checkpoint(host, make_baseline=(k == 0))
        assert g == e, (k, first_mismatch(g, e))
        diffs.append(g)
    d.close()
    return diffs


@pytest.mark.parametrize("patterns", [1, 4, 7])
@pytest.mark.parametrize("n", [63, 1025, 40_000])
def test_digests_shared_by_many_chunks(patterns, n):
    """Chunks that share few digests, in an order that mixes them within a wavefront:
    the lowest chunk of each is the first occurrence, at a baseline and later (one to
    more shared entries than a wavefront folds before its atomics)."""
    C = 32
    rng = np.random.default_rng(100 * patterns + n)
    bank = rng.integers(0, 256, (2 * patterns, C), dtype=np.uint8)
    v0 = bank[rng.integers(0, patterns, n)].reshape(-1)
    v1 = v0.copy().reshape(n, C)
    at = rng.random(n) < 0.5
    v1[at] = bank[patterns + rng.integers(0, patterns, int(at.sum()))]
    v2 = v1.copy()
    v2[rng.random(n) < 0.3] = bank[0]
    same_as_oracle([v0, v1.reshape(-1), v2.reshape(-1)], C)


@pytest.mark.parametrize("approach", [M.TREE, M.BASIC])
@pytest.mark.parametrize("C,n,tail", [
    (1, 3000, 0), (3, 5000, 0), (16, 4097, 5), (17, 3000, 16), (48, 2500, 47), (100, 1300, 3), (1000, 333, 999),
    (1024, 130, 1), (4096, 70, 4000), (4100, 40, 17), (16384, 9, 0), (16400, 11, 5), (32768, 5, 32767),
    (65536, 4, 100), (65536, 3, 0), (100_003, 5, 77)])
def test_gathered_chunks(approach, C, n, tail):
    """The diff's data section around the sizes at which its tiles change: chunks of
    one byte to several tiles, powers of two or not, with and without a short last
    chunk, runs and single chunks, and a buffer that is not 16-byte aligned."""
    rng = np.random.default_rng(C + n)
    size = n * C + tail
    v = [rng.integers(0, 256, size, dtype=np.uint8)]
    for k in range(3):
        w = v[-1].copy()
        for first in rng.integers(0, n, 1 + n // 40):
            e = min(size, (int(first) + int(rng.integers(1, 6))) * C)
            w[first * C:e] = rng.integers(0, 256, max(0, e - first * C), dtype=np.uint8)
        if k == 1:
            w[-1:] ^= 1
        v.append(w)
    for off in (0, 5):
        d = M.TreeDeduplicator(C, approach)
        orc = O.OracleDedup(C, M.MURMUR3) if approach == M.TREE else O.OracleBasic(C, M.MURMUR3)
        for k, host in enumerate(v):
            print(f"gather C={C} n={n} tail={tail} approach={approach} off={off} k={k}", flush=True)
            buf = torch.zeros(size + 16, dtype=torch.uint8, device="cuda:0")
            buf[off:off + size] = torch.from_numpy(host)
            g = d.checkpoint(buf[off:off + size], make_baseline=(k == 0))
            e = orc.checkpoint(host, make_baseline=(k == 0))
            assert g == e, (k, len(g), len(e))
        d.close()


@pytest.mark.parametrize("n", [(1 << 20) - 3, 1 << 21, 1 << 22])
def test_root_segments_per_wavefront(n):
    """Root segments of one tile each: 37 thousand (two segments per wavefront of the
    root compaction), 74 thousand (four) and 147 thousand (eight)."""
    C = 16
    rng = np.random.default_rng(n)
    v0 = rng.integers(0, 256, n * C, dtype=np.uint8)
    v1 = v0.copy().reshape(n, C)
    at = rng.random(n) < 0.02
    v1[at] = rng.integers(0, 256, (int(at.sum()), C), dtype=np.uint8)
    at = np.nonzero(rng.random(n) < 0.01)[0]
    v1[at] = v1[rng.integers(0, n, at.size)]
    v1 = v1.reshape(-1)
    d, orc = M.TreeDeduplicator(C), O.OracleDedup(C)
    d.set_sweep_tiles(1, 1)
    for k, host in enumerate((v0, v1)):
        print(f"segments n={n} k={k}", flush=True)
        g = d.checkpoint(torch.from_numpy(host).to("cuda:0"), make_baseline=(k == 0))
        e = orc.checkpoint(host, make_baseline=(k == 0), threads=8)
        assert g == e, (k, first_mismatch(g, e))
    d.close()


def test_handle_alternates_between_alone_and_a_large_batch():
    """A handle whose root segments are planned for steps alone joins a step of many
    tiles (a new plan with four tiles a segment) and returns: the oracle's diffs."""
    C, n, members = 8, 1 << 21, 8
    rng = np.random.default_rng(8)
    host = [rng.integers(0, 256, n * C, dtype=np.uint8)]
    for _ in range(4):
        w = host[-1].copy().reshape(n, C)
        at = rng.random(n) < 0.01
        w[at] = rng.integers(0, 256, (int(at.sum()), C), dtype=np.uint8)
        at = np.nonzero(rng.random(n) < 0.005)[0]
        w[at] = w[rng.integers(0, n, at.size)]
        host.append(w.reshape(-1))
    bufs = [torch.from_numpy(v).to("cuda:0") for v in host]
    ds, batch, orc = [M.TreeDeduplicator(C) for _ in range(members)], M.Batch(), O.OracleDedup(C)
    for k, b in enumerate(bufs):
        print(f"alternating step {k}", flush=True)
        if k % 2 == 0:
            got = [d.checkpoint(b, make_baseline=(k == 0)) for d in ds]
        else:
            got = batch.checkpoint(ds, [b] * members, copy=True)
        e = orc.checkpoint(host[k], make_baseline=(k == 0), threads=8)
        for g in got:
            assert g == e, (k, first_mismatch(g, e))
    for d in ds:
        d.close()
    batch.close()


@pytest.mark.parametrize("C,n,tail", [(1, 700, 0), (7, 1000, 3), (16, 513, 0), (48, 300, 47), (100, 2000, 1),
                                      (128, 4096, 0), (128, 1000, 5), (1000, 129, 999), (4096, 33, 17)])
def test_restart_copies(C, n, tail):
    """Restarts of every checkpoint from device and host chains: chunk sizes that are
    powers of two and not, short last chunks, outputs at any alignment, diffs that lie
    at odd addresses, and shifted entries from one leaf to the whole buffer."""
    size = n * C + tail
    rng = np.random.default_rng(7 * C + n)
    v0 = rng.integers(0, 256, size, dtype=np.uint8)
    v1 = v0.copy()
    half = n // 2 * C
    v1[half:2 * half] = v0[:half]                      # large shifted entries
    v2 = v1.copy()
    for first in rng.integers(0, n, 6):
        v2[first * C:(first + 2) * C] = rng.integers(0, 256, v2[first * C:(first + 2) * C].size, dtype=np.uint8)
    versions = [v0, v1, v2, v0, v2[::-1].copy(), v1]   # v0 again: every leaf shifted
    diffs = same_as_oracle(versions, C)
    dev = [torch.frombuffer(bytearray(d), dtype=torch.uint8).to("cuda:0") for d in diffs]
    odd = []
    for i, d in enumerate(diffs):
        t = torch.zeros(len(d) + 8, dtype=torch.uint8, device="cuda:0")
        t[i % 5:i % 5 + len(d)] = dev[i]
        odd.append(t[i % 5:i % 5 + len(d)])
    for off in (0, 4, 1):
        for chain in (dev, odd, diffs):
            for k in range(len(versions)):
                print(f"restart C={C} n={n} tail={tail} off={off} k={k}", flush=True)
                buf = torch.full((size + 32,), 0xA5, dtype=torch.uint8, device="cuda:0")
                M.restart_into(buf[off:off + size], chain, k)
                got = buf.cpu().numpy()
                assert np.array_equal(got[off:off + size], versions[k])
                assert (got[:off] == 0xA5).all() and (got[off + size:] == 0xA5).all()


def test_restart_of_a_late_chain():
    """A device chain that starts after checkpoint 4096: its headers are read from the
    chain's first diff on; what lies below it is not needed."""
    d, size = M.TreeDeduplicator(16), 16 * 50 + 3
    rng = np.random.default_rng(5)
    host = rng.integers(0, 256, size, dtype=np.uint8)
    buf = torch.from_numpy(host).to("cuda:0")
    chain = []
    for k in range(4099):
        d.checkpoint_device(buf, make_baseline=(k == 4094))
        chain.append(d.copy_last_diff_device() if k >= 4094 else None)
        if k >= 4094:
            buf[(k % 50) * 16:(k % 50) * 16 + 5] = k % 251
    d.close()
    want = torch.from_numpy(host).to("cuda:0")
    for k in range(4094, 4099):
        out = torch.zeros(size, dtype=torch.uint8, device="cuda:0")
        M.restart_into(out, chain, k)
        assert torch.equal(out, want), k
        want[(k % 50) * 16:(k % 50) * 16 + 5] = k % 251


def test_restart_refuses_short_data_and_leaves_the_output():
    """A diff whose data section is cut to fewer chunks than its regions (to some, to
    none) is refused before anything is written."""
    C, n = 64, 40
    rng = np.random.default_rng(9)
    v0 = rng.integers(0, 256, n * C, dtype=np.uint8)
    v1 = v0.copy()
    v1[5 * C:9 * C] = rng.integers(0, 256, 4 * C, dtype=np.uint8)
    diffs = same_as_oracle([v0, v1], C)
    for cut0, cut1 in ((0, 1), (0, 4), (1, 0)):
        chain = [torch.frombuffer(bytearray(d[:len(d) - cut * C]), dtype=torch.uint8).to("cuda:0")
                 for d, cut in zip(diffs, (cut0, cut1))]
        out = torch.full((n * C,), 7, dtype=torch.uint8, device="cuda:0")
        with pytest.raises(M.MtcError) as e:
            M.restart_into(out, chain, 1)
        assert e.value.code == 5
        assert bool((out == 7).all())
    M.restart_into(out, [torch.frombuffer(bytearray(d), dtype=torch.uint8).to("cuda:0") for d in diffs], 1)
    assert np.array_equal(out.cpu().numpy(), v1)


@pytest.mark.parametrize("hk", [M.MURMUR3, M.MD5])
@pytest.mark.parametrize("C", [16, 32, 64, 128, 256, 2048, 4096])
def test_hash_chunks_blocks(C, hk):
    """mtc_hash_chunks at one wavefront of chunks, one more, less, and short tails."""
    rng = np.random.default_rng(C + hk)
    for n, tail in ((1, 0), (63, 5), (64, 0), (64, 15), (65, C - 1), (300, 1)):
        a = rng.integers(0, 256, n * C + tail, dtype=np.uint8)
        print(f"hash_chunks C={C} hk={hk} n={n} tail={tail}", flush=True)
        got = M.hash_chunks(torch.from_numpy(a).to("cuda:0"), C, hk).cpu().numpy().reshape(-1, 16)
        assert len(got) == n + (tail > 0)
        for c in range(len(got)):
            assert got[c].tobytes() == O.hash_bytes(hk, a[c * C:(c + 1) * C]), c


@pytest.mark.parametrize("hk", [M.MURMUR3, M.MD5])
@pytest.mark.parametrize("C", [1, 5, 15, 17, 20, 24, 40, 51, 63, 100, 111, 112, 113, 127, 129, 144, 200, 255, 257, 1000])
def test_hash_chunks_any_size(C, hk):
    """Digests of chunk sizes that are no power of two, at every data alignment modulo
    16: chunks staged as one piece and by rows, tails of every class, wavefronts at the
    buffer's edges (first unaligned, last partial), and MD5 of few and many chunks."""
    rng = np.random.default_rng(3 * C + hk)
    n = 66_000 if hk == M.MD5 and C in (17, 100, 113) else 333
    a = rng.integers(0, 256, n * C + 16, dtype=np.uint8)
    some = range(n) if n < 1000 else sorted({*range(130), *range(n - 130, n), *rng.integers(0, n, 200).tolist()})
    for off, cut in ((0, 0), (1, 1), (4, 0), (7, 0), (8, C // 2), (13, 0), (15, 0)):
        size = n * C - cut
        buf = torch.zeros(size + 32, dtype=torch.uint8, device="cuda:0")
        buf[off:off + size] = torch.from_numpy(a[:size])
        print(f"hash any C={C} hk={hk} n={n} off={off} cut={cut}", flush=True)
        got = M.hash_chunks(buf[off:off + size], C, hk).cpu().numpy().reshape(-1, 16)
        assert len(got) == (size + C - 1) // C
        for c in some:
            if c * C < size:
                assert got[c].tobytes() == O.hash_bytes(hk, a[c * C:min((c + 1) * C, size)]), c


@pytest.mark.parametrize("C,hk,n", [(100, 0, 3000), (100, 1, 66_000), (20, 0, 3000), (333, 0, 1000), (1000, 1, 700)])
def test_series_of_any_chunk_size(C, hk, n):
    rng = np.random.default_rng(C * n)
    v = [rng.integers(0, 256, n * C + 3, dtype=np.uint8)]
    for _ in range(2):
        w = v[-1].copy()
        for first in rng.integers(0, n, 12):
            w[first * C:(first + 3) * C] = rng.integers(0, 256, w[first * C:(first + 3) * C].size, dtype=np.uint8)
        src, dst = rng.integers(0, n, 2)
        w[dst * C:(dst + 1) * C] = w[src * C:(src + 1) * C]
        v.append(w)
    same_as_oracle(v, C, hk)


def test_diff_copies_to_device_memory():
    """mtc_copy_diff to device memory at every word offset modulo 16, and at byte
    offsets: the diff's bytes and nothing around them."""
    rng = np.random.default_rng(2)
    for C, n in ((4, 1), (4, 3), (16, 5), (64, 700), (100, 333)):
        host = rng.integers(0, 256, n * C, dtype=np.uint8)
        d = M.TreeDeduplicator(C)
        want = d.checkpoint(torch.from_numpy(host).to("cuda:0"), make_baseline=True)
        for off in (0, 4, 8, 12, 1, 6):
            out = torch.full((len(want) + 48,), 0x5A, dtype=torch.uint8, device="cuda:0")
            got = d.copy_last_diff_device(out[16 + off:16 + off + len(want)])
            o = out.cpu().numpy()
            assert got.cpu().numpy().tobytes() == want
            assert (o[:16 + off] == 0x5A).all() and (o[16 + off + len(want):] == 0x5A).all()
        d.close()


@pytest.mark.parametrize("n", [3000, 36_000])
def test_shifted_chunks_of_many_checkpoints(n):
    """Shifted entries of one, a few and more than 256 sources (none, one and two sort
    passes; their counts added up by the sort's blocks or scanned first), beside the
    scan of the region sizes."""
    C, rng = 16, np.random.default_rng(n)
    cur = rng.integers(0, 256, (n, C), dtype=np.uint8)
    fresh, versions = [cur[:50].copy()], [cur.reshape(-1).copy()]
    for k in range(1, 290):
        new = rng.integers(0, 256, (20, C), dtype=np.uint8)
        cur[rng.choice(n, 20, replace=False)] = new
        fresh.append(new)
        if k in (2, 5, 40, 270, 289):  # chunks of every earlier checkpoint, at new places
            bank = np.concatenate(fresh)
            to = rng.choice(n, n // 3, replace=False)
            cur[to] = bank[rng.integers(0, len(bank), len(to))]
        versions.append(cur.reshape(-1).copy())
    same_as_oracle(versions, C)


@pytest.mark.parametrize("hk", [M.MURMUR3, M.MD5])
@pytest.mark.parametrize("C,n", [(16, 1), (128, 255), (32, 256), (64, 257), (128, 70_001), (512, 3000), (4096, 300)])
def test_basic_lists_are_ascending(C, n, hk):
    """The basic approach's lists from leaf blocks of one tile: no, one, few and all
    chunks of a block changed, in one and in several of its wavefronts."""
    rng = np.random.default_rng(C * n)
    v = [rng.integers(0, 256, n * C - 3, dtype=np.uint8)]
    for frac in (0.0, 0.01, 0.5, 1.0):
        w = v[-1].copy()
        for c in np.nonzero(rng.random(n) < frac)[0]:
            w[c * C] ^= 1
        v.append(w)
    w = v[-1].copy()
    w[-1] ^= 1
    v.append(w)
    d, orc = M.TreeDeduplicator(C, M.BASIC, hash_kind=hk), O.OracleBasic(C, hk)
    for k, host in enumerate(v):
        g = d.checkpoint(torch.from_numpy(host).to("cuda:0"), make_baseline=(k == 0))
        e = orc.checkpoint(host, make_baseline=(k == 0))
        assert g == e, (k, first_mismatch(g, e))
    d.close()


@pytest.mark.parametrize("hk", [M.MURMUR3, M.MD5])
@pytest.mark.parametrize("n,tail", [(1, 0), (64, 0), (65, 4095), (255, 1), (256, 0), (257, 77), (5000, 100)])
def test_series_of_large_chunks(n, tail, hk):
    """Leaf tiles hashed by blocks of one wavefront: part of a tile's wavefronts, all,
    several tiles, with and without a short last chunk."""
    C, rng = 4096, np.random.default_rng(n)
    v = [rng.integers(0, 256, n * C + tail, dtype=np.uint8)]
    for frac in (0.0, 0.02, 0.7, 0.01):
        w = v[-1].copy()
        for c in np.nonzero(rng.random(n) < frac)[0]:
            w[c * C + 17] ^= 5
        w[-1] ^= 1 if frac else 0
        v.append(w)
    same_as_oracle(v, C, hk)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 257, 300, 777, 5000])
def test_pending_leaves_decided_by_the_sweep(n):
    """Leaves whose label is open until every insert has landed (chunks that share
    digests, zero chunks after a second baseline), on one and on two tree depths."""
    C, rng = 32, np.random.default_rng(n)
    bank = rng.integers(0, 256, (3, C), dtype=np.uint8)
    bank[0] = 0
    d, orc = M.TreeDeduplicator(C), O.OracleDedup(C, M.MURMUR3)
    host = bank[rng.integers(0, 3, n)].copy()
    for k in range(5):
        if k:
            at = rng.random(n) < (0.6 if k < 4 else 0.05)
            host[at] = np.concatenate([bank, rng.integers(0, 256, (2, C), dtype=np.uint8)])[rng.integers(0, 5, int(at.sum()))]
        flat = host.reshape(-1).copy()
        g = d.checkpoint(torch.from_numpy(flat).to("cuda:0"), make_baseline=k in (0, 2))
        e = orc.checkpoint(flat, make_baseline=k in (0, 2))
        assert g == e, (k, first_mismatch(g, e))
    d.close()
