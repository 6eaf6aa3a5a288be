"""Sizes beyond one row of a launch's blocks (2^31 threads)."""
import pytest

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
