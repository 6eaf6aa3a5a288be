"""Restarts of chains whose diffs cover many chunks at once."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import mtcheck_amd as M  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,n", [(16, (1 << 22) - 1), (8, 1 << 22), (12, (1 << 22) + 777), (8, 1 << 23)])
def test_large_diffs_between_small_ones(C, n):
    """Diffs below and from 2^22 chunks or shifted entries on, the oldest among them: every later
    one replaces what the earlier ones covered, in any order of the two kinds."""
    g = torch.Generator(device="cuda")
    g.manual_seed(n + C)
    rand = lambda k: torch.randint(0, 256, (k, C), dtype=torch.uint8, device="cuda", generator=g)  # noqa: E731
    v = [rand(n)]
    v[0][: 3 * n // 5] = 7                                    # a shifted entry for nearly each of these leaves
    for k in range(1, 9):
        w = v[-1].clone()
        if k in (1, 4, 6):                                    # few chunks
            at = torch.randint(0, n, (50,), device="cuda", generator=g)
            w[at] = rand(50)
            w[:20] = w[n // 2:n // 2 + 20]
        elif k == 2:
            w = rand(n)                                       # every chunk new
        elif k == 3:
            w[:] = 0                                          # one chunk, all others shifted
        elif k == 5:
            w = v[2].clone()                                  # the whole buffer from an earlier checkpoint
        elif k == 7:
            w = torch.where((torch.rand(n, 1, device="cuda", generator=g) < 0.5), v[0], w)
        else:
            w = rand(n)
            w[::2] = v[7][::2]
        v.append(w)
    d, chain = M.TreeDeduplicator(C, hash_kind=M.MD5), []  # (Murmur3's digests of so many 8-byte chunks collide)
    for k, w in enumerate(v):
        d.checkpoint_device(w.view(-1), make_baseline=(k == 0))
        s = d.stats()
        print(f"C={C} n={n} k={k} chunks {s.data_chunks} shifted {s.num_shift_dupl}", flush=True)
        chain.append(d.copy_last_diff_device())
    d.close()
    out = torch.zeros(n * C, dtype=torch.uint8, device="cuda")
    for k in list(range(9)) + [8]:
        M.restart_into(out, chain, k)
        assert torch.equal(out, v[k].view(-1)), k
