"""What the launches ask for and refuse, by a host program linked to the library: nothing here reaches a GPU."""
import os
import shutil
import subprocess

import pytest

from vllm_neuron_amd import _native

CSRC = os.path.join(os.path.dirname(os.path.abspath(_native.__file__)), "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include <cstdio>
#include "attn_kernels.h"
int main() {
  using namespace mi;
  for (int hd : {64, 128})
    for (int kh : {1, 2})
      for (int splits : {1, 2, 8}) printf("lds %d %d %d %d\n", hd, kh, splits, attn_mixed_lds(hd, kh, splits));
}
"""


@pytest.fixture(scope="module")
def said(tmp_path_factory):
    _native.load_library()
    at = tmp_path_factory.mktemp("launch")
    (at / "p.cpp").write_text(PROGRAM)
    r = subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-std=c++17", "-I", CSRC, str(at / "p.cpp"), "-x", "none", _native.LIB_PATH,
                        "-Wl,-rpath," + os.path.dirname(_native.LIB_PATH), "-o", str(at / "p")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(at / "p")], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr[-3000:]
    return [line.split(" ", 1) for line in r.stdout.splitlines()]


def test_splits_are_merged_by_work_groups_that_have_their_cu_alone(said):
    """The merge of a context's splits hands partial sums over without a fence: its work-groups must not share a CU (160 KiB of LDS)."""
    lds = {tuple(map(int, s.split()[:3])): int(s.split()[3]) for k, s in said if k == "lds"}
    assert len(lds) == 12 and all(n <= 160 << 10 for n in lds.values())
    assert all(2 * n > 160 << 10 for (_, _, splits), n in lds.items() if splits > 1)
