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
#include "linear_kernels.h"
using namespace mi;
static void refused(const char* what, int rc) { printf("%s %d %s\n", what, rc, mi_last_error()); }
int main() {
  for (int hd : {64, 128})
    for (int kh : {1, 2})
      for (int splits : {1, 2, 8}) printf("lds %d %d %d %d\n", hd, kh, splits, attn_mixed_lds(hd, kh, splits));
  // a residual projection that is to hand the norm behind it on, where the kernel cannot
  EpiArgs e{};
  uint16_t x[1];
  e.next_x = x; e.ld_out = 256;
  const LinearW w{nullptr, 256, 256, MI_W_BF16}, w8{nullptr, 256, 256, MI_W_F8E4M3};
  refused("hand", launch_splitk_reduce(SlabSum{nullptr, 2, 4, 256, nullptr, nullptr, nullptr}, EPI_RESID, e, nullptr));
  refused("hand", launch_gemm(w, 33, x, 256, EPI_RESID, e, nullptr));
  refused("hand", launch_gemm_wide(w, 33, x, 256, EPI_RESID, e, nullptr));
  refused("hand", launch_gemm_a8(w8, 33, nullptr, 33, EPI_RESID, e, nullptr));
  refused("hand", launch_gemv(w, 4, PRO_BF16, ProArgs{}, EPI_F32, e, nullptr));
  e.ld_out = 512;
  refused("hand", launch_gemv(w, 4, PRO_BF16, ProArgs{}, EPI_RESID, e, nullptr));
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


def test_launches_that_cannot_hand_a_norm_on_refuse_to(said):
    lines = [s for k, s in said if k == "hand"]
    assert len(lines) == 6 and all(s.startswith("-1 ") and "norm" in s for s in lines), lines
