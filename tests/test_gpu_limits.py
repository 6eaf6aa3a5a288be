"""Sizes, table loads, chunk sizes and addresses at the limits of the kernels and their rules."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import first_mismatch

torch = pytest.importorskip("torch")
import mtcheck_amd as M  # noqa: E402

pytestmark = pytest.mark.gpu


def test_copy_and_restart_beyond_one_row_of_blocks():
    """33 GiB at 16 bytes a thread take two rows: the diff's copy to device memory and
    the restart by k_r_copy_any (a chunk size that is no power of two)."""
    n, C = (33 << 30) + 5, 1_000_000
    data = torch.empty(n, dtype=torch.uint8, device="cuda:0")
    for i in range(0, n, 1 << 30):
        data[i:i + (1 << 30)].random_(0, 256)
    d = M.TreeDeduplicator(C)
    print("checkpoint", flush=True)
    d.checkpoint_device(data, make_baseline=True)
    print("copy", flush=True)
    kept = d.copy_last_diff_device()
    d.close()
    out = torch.zeros_like(data)
    print("restart", flush=True)
    M.restart_into(out, [kept], 0)
    for i in range(0, n, 1 << 30):
        assert torch.equal(out[i:i + (1 << 30)], data[i:i + (1 << 30)]), i


def series(versions, C, hk=0, offset=0, load_factor=0.125):
    n = len(versions[0])
    buf = torch.zeros(n + 16, dtype=torch.uint8, device="cuda:0")
    d, orc = M.TreeDeduplicator(C, hash_kind=hk), O.OracleDedup(C, hk)
    d.set_tuning(1, load_factor, 8)
    for k, host in enumerate(versions):
        print(f"C={C} hash {hk} n={n} offset {offset} load factor {load_factor} checkpoint {k}", flush=True)
        buf[offset:offset + n] = torch.from_numpy(host)
        g = d.checkpoint(buf[offset:offset + n], make_baseline=(k == 0))
        e = orc.checkpoint(host, make_baseline=(k == 0), threads=8)
        assert g == e, (k, first_mismatch(g, e))
    d.close()


@pytest.mark.parametrize("C,hk,n,offset", [
    (100, 0, 5_000, 0), (100, 0, 5_300, 0), (25, 0, 5_000, 1), (64, 0, 9_000, 4), (320, 0, 300, 0), (320, 0, 106_000, 0),
    (4096, 0, 300, 4), (8192, 0, 150, 0), (8192, 0, 150, 3), (24, 1, 70_000, 0), (64, 1, 66_000, 1), (72, 1, 70_000, 0),
    (200, 1, 66_000, 0), (200, 1, 66_000, 2), (128, 1, 66_000, 1), (128, 1, 66_000, 4)])
def test_series_by_bytes_and_staged(C, hk, n, offset):
    """Chunk sizes, numbers and addresses on both sides of the rules that choose the leaf kernel."""
    rng = np.random.default_rng(C + n + offset)
    v = [rng.integers(0, 256, n * C - C // 3, dtype=np.uint8)]
    for _ in range(2):
        w = v[-1].copy()
        for first in rng.integers(0, n, 9):
            w[first * C:(first + 2) * C] = rng.integers(0, 256, w[first * C:(first + 2) * C].size, dtype=np.uint8)
        w[-1] ^= 1
        v.append(w)
    series(v, C, hk, offset)


@pytest.mark.parametrize("load_factor", [0.125, 0.5, 0.7])
@pytest.mark.parametrize("n", [1 << 12, 1 << 16])
def test_whole_rewrites_grow_the_table(n, load_factor):
    """Every chunk new in every version: each adds 2n - 1 entries to the table, which grows
    before it is nearly full (a baseline's table too, at load factors of a half and more)."""
    rng = np.random.default_rng(n)
    series([rng.integers(0, 256, n * 16, dtype=np.uint8) for _ in range(6)], 16, load_factor=load_factor)


@pytest.mark.parametrize("C", [2, 5, 6, 15, 17, 33, 4097, 5001, 8191, 20_001])
def test_chunks_gathered_and_restored_by_words(C):
    """Diffs and outputs that start at any byte of a word: single chunks, runs, and words of up to
    four chunks."""
    n = max(9, 60_000 // C)
    rng = np.random.default_rng(C)
    v = [rng.integers(0, 256, n * C - C // 2, dtype=np.uint8)]
    for _ in range(2):
        w = v[-1].copy()
        for first in rng.integers(0, n, n // 6):
            w[first * C:(first + int(rng.integers(1, 4))) * C] ^= 255
        v.append(w)
    hk, size = (M.MD5 if C < 16 else M.MURMUR3), len(v[0])
    for offset in (0, 3):
        for approach in (M.TREE, M.BASIC):
            buf = torch.zeros(size + 16, dtype=torch.uint8, device="cuda:0")
            d = M.TreeDeduplicator(C, approach, hash_kind=hk)
            orc = O.OracleDedup(C, hk) if approach == M.TREE else O.OracleBasic(C, hk)
            chain = []
            for k, host in enumerate(v):
                print(f"C={C} offset {offset} approach {approach} checkpoint {k}", flush=True)
                buf[offset:offset + size] = torch.from_numpy(host)
                g, e = d.checkpoint(buf[offset:offset + size], make_baseline=(k == 0)), orc.checkpoint(host, make_baseline=(k == 0))
                assert g == e, (k, first_mismatch(g, e))
                chain.append(torch.frombuffer(bytearray(g), dtype=torch.uint8).to("cuda:0"))
            d.close()
            if approach == M.BASIC:
                continue
            for at in (0, 1, 2, 3, 4):
                out = torch.full((size + 32,), 0xA5, dtype=torch.uint8, device="cuda:0")
                M.restart_into(out[at:at + size], chain, 2)
                got = out.cpu().numpy()
                assert np.array_equal(got[at:at + size], v[2])
                assert (got[:at] == 0xA5).all() and (got[at + size:] == 0xA5).all()
