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
