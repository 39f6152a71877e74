"""The blocks of an ensemble member hand their results over through memory: the waits that this
needs are in the compiled kernel.  Compiles the source for gfx950 and reads the assembly."""
import os
import re
import subprocess

import pytest

from dftbaby_amd import build

STORE = re.compile(r"\b(flat|global|buffer)_(store|atomic)")
MEMORY = re.compile(r"\b(flat|global|buffer|scratch)_(load|store|atomic)")


def _waits(line):
    return "s_waitcnt" in line and "vmcnt(0)" in line


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("asm") / "ensemble.s")
    subprocess.run([build.HIPCC] + build.FLAGS + ["-S", "--offload-device-only",
                                                  os.path.join(build.CSRC, "ensemble.hip"), "-o", out], check=True,
                   capture_output=True)
    return [x.split(";")[0].strip() for x in open(out)]


def test_stores_arrive_before_the_write_back(assembly):
    """Before each L2 write-back: a barrier, and before that, after the last store of every wave, a
    wait for the wave's stores.  After it a wait before anything else goes to memory."""
    sites = [i for i, x in enumerate(assembly) if x.startswith("buffer_wbl2")]
    assert len(sites) >= 7          # each form of a section of products, of the exchange, of a helper
    for i in sites:
        j = i
        while assembly[j] != "s_barrier":
            assert not STORE.search(assembly[j]) or "scratch" in assembly[j], (j + 1, assembly[j])
            j -= 1
        k = j
        while not _waits(assembly[k]):
            assert not MEMORY.search(assembly[k]) and not assembly[k].endswith(":"), (k + 1, assembly[k])
            k -= 1
        k = i + 1
        while not _waits(assembly[k]):
            assert not MEMORY.search(assembly[k]) and not assembly[k].endswith(":"), (k + 1, assembly[k])
            k += 1


def test_stale_lines_are_gone_before_the_barrier(assembly):
    """After each invalidation a wait before the barrier that lets the other waves read."""
    sites = [i for i, x in enumerate(assembly) if x.startswith("buffer_inv")]
    assert len(sites) >= 7
    for i in sites:
        k = i + 1
        while not _waits(assembly[k]):
            assert assembly[k] != "s_barrier" and not MEMORY.search(assembly[k]), (k + 1, assembly[k])
            k += 1
