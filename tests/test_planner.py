"""The rules that choose a launch's shape, on the CPU: csrc/qa_api.cpp (plan_linear)
and qa_internal.h compiled into a small library of the test's own."""
from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import pytest

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
SOURCE = r"""
#include "qa_api.cpp"
// out: tile, splits, tiles over m, over n
extern "C" void test_plan_linear(uint32_t flags, int64_t m, int64_t n, int64_t k, int64_t batch, int cus, int64_t* out) {
  qa_linear_desc d{};
  d.flags = flags;
  d.m = m;
  d.n = n;
  d.k = k;
  d.batch = batch;
  const qa::Plan p = plan_linear(d, cus);
  out[0] = p.tile;
  out[1] = p.splits;
  out[2] = p.tiles_m;
  out[3] = p.tiles_n;
}
extern "C" int test_attention_32(int64_t rows, int64_t q0, int nkvh, int cus) {
  qa::AttnParams p{};
  p.rows = rows;
  p.q0 = q0;
  p.nkvh = nkvh;
  p.num_cus = cus;
  return qa::attention_32_row_blocks(p);
}
"""


@pytest.fixture(scope="module")
def planner(pkg, tmp_path_factory):
    if not shutil.which(HIPCC):
        pytest.skip("hipcc not available")
    td = tmp_path_factory.mktemp("planner")
    src, lib = td / "planner.cpp", td / "planner.so"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-std=c++17", "-O1", "-fPIC", "-shared", "-I", pkg.CSRC, "-I", os.path.join(pkg.CSRC, "..", "..", "include"),
                    str(src), "-o", str(lib), "-x", "none", pkg.LIB_PATH, f"-Wl,-rpath,{pkg.CSRC}"], check=True, capture_output=True)
    return ctypes.CDLL(str(lib))


def _linear(planner, m, n, k, batch=1, flags=0, cus=256):
    out = (ctypes.c_int64 * 4)()
    i64 = ctypes.c_int64
    planner.test_plan_linear(ctypes.c_uint32(flags), i64(m), i64(n), i64(k), i64(batch), cus, out)
    return tuple(out)


@pytest.mark.parametrize("m", [256, 512, 1024])
@pytest.mark.parametrize("n,k", [(128, 128), (256, 512), (512, 512), (1024, 1024), (3072, 1024), (1024, 3072)])
@pytest.mark.parametrize("batch", [2, 3, 16, 64, 256])
def test_batch_is_priced_as_a_whole(planner, m, n, k, batch):
    """A batch of problems of whole tiles costs what one problem of as many
    rows does: the same tile, or the one of the unsplit plan where that problem
    would split K (a batch never does)."""
    one = _linear(planner, batch * m, n, k)
    got = _linear(planner, m, n, k, batch)
    assert got[1] == 1
    if one[1] == 1:
        assert got[0] == one[0]
    assert _linear(planner, m, n, k, 0) == _linear(planner, m, n, k, 1)


@pytest.mark.parametrize("cus", [32, 64, 256])
def test_attention_shape_counts_the_devices_cus(planner, cus):
    """32-row blocks up to one 64-row block per CU of the device in use (a
    partition of the chip has fewer than 256), or, behind a long past, up to
    one 32-row block per CU."""
    def blocks32(rows, q0):
        i64 = ctypes.c_int64
        return bool(planner.test_attention_32(i64(rows), i64(q0), 8, cus))

    full = cus // 8  # blocks of one kv head in a round
    assert blocks32(64 * full, 0) and not blocks32(64 * full + 1, 0)
    assert blocks32(32 * full, 10 * 32 * full) and not blocks32(32 * full + 1, 2 * 32 * full)
