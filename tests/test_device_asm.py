"""What the compiler cannot know about instructions written as text (gfx950 assembly of
this repository's own code).  CPU only."""
import re
import subprocess

import pytest

from mtcheck_amd import build as B

SRC = """
#include "device.hpp"
using namespace mtc;
__global__ void k(Slot* tab, uint64_t mask, const Digest* d, uint32_t* err, uint32_t* out) {
  bool claimed;
  out[threadIdx.x] = table_insert(tab, mask, d[threadIdx.x], threadIdx.x, false, err, &claimed, true);
}
"""


WHOLE = """
#include "dedup.hip"
namespace mtc {
__global__ void k_decide(SweepArgs a, uint8_t* out) { out[threadIdx.x] = decide_leaf(a, threadIdx.x); }
}
"""


@pytest.fixture(scope="module")
def whole(tmp_path_factory):
    """The assembly of dedup.hip, and of decide_leaf in a kernel of its own."""
    d = tmp_path_factory.mktemp("asm")
    (d / "k.hip").write_text(WHOLE)
    subprocess.run([B.HIPCC, *B.CFLAGS, "-I", B.CSRC, "--offload-device-only", "-S", str(d / "k.hip"), "-o", str(d / "k.s")],
                   check=True, capture_output=True)
    return (d / "k.s").read_text()


def kernel(text, name):
    return re.search(rf"^{name}\w*:.*?s_endpgm", text, re.M | re.S).group(0)


def test_sweep_a_reads_table_values_at_agent_scope(whole):
    """Sweep A inserts, so it reads a slot's value past the caches of its own die (sc1)
    where it decides a pending leaf too."""
    loads = re.findall(r"global_load_dwordx2 .*", kernel(whole, "_ZN3mtc8k_decide"))
    assert len(loads) == 1 and "sc1" in loads[0], loads


def test_pair_store_waits_before_its_data_is_overwritten(tmp_path):
    """A vector store of more than 8 bytes needs two wait states before an instruction
    overwrites its data registers.  The compiler keeps them after its own stores only."""
    src = tmp_path / "k.hip"
    src.write_text(SRC)
    out = tmp_path / "k.s"
    subprocess.run([B.HIPCC, *B.CFLAGS, "-I", B.CSRC, "--offload-device-only", "-S", str(src), "-o", str(out)], check=True,
                   capture_output=True)
    code = [s.split(";")[0].strip() for s in out.read_text().splitlines()]
    code = [s for s in code if s and not s.startswith((".", "#")) and not s.endswith(":")]
    at = [i for i, s in enumerate(code) if re.match(r"global_store_dwordx[34] .*\bsc1\b", s)]
    assert at
    for i in at:
        m = re.match(r"s_nop (\d+)", code[i + 1])
        assert m and int(m.group(1)) >= 1, code[i:i + 2]


def test_md5_by_bytes_issues_a_blocks_loads_together(whole):
    """The four 16-byte loads of a 64-byte block, with nothing between them: the other wavefronts
    of a compute unit push a line out of its cache before a late one of them reads it."""
    lines = [s.strip() for s in kernel(whole, "_ZN3mtc13k_hash_chunksILi1ELin1EE").splitlines()]
    lines = [s for s in lines if s and not s.startswith(";")]
    at = [i for i, s in enumerate(lines) if s.startswith("global_load_dwordx4")]
    assert len(at) == 4 and at[3] - at[0] == 3, lines[at[0]:at[-1] + 1]
