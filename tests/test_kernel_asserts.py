"""Kernel forms that would be silently wrong do not compile (checked by the compiler's front end
alone, for the device, in about a second each)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

KERNEL = """#include "pkv_decode.hip"
namespace pkv { namespace {
__global__ void probe(DecodeArgs a) {
  WaveState<1> st;
  u32x4 qf[1][4];
  %s
} } }
"""


def _compile(tmp_path, body):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    src = tmp_path / "probe.hip"
    src.write_text(KERNEL % body)
    return subprocess.run(
        [HIPCC, "--offload-arch=gfx950", "-std=c++17", "-fsyntax-only", "--cuda-device-only",
         "-I" + os.path.join(ROOT, "include"),
         "-I" + os.path.join(ROOT, "persistentkv-attention_amd", "csrc"), str(src)],
        capture_output=True, text=True)


@pytest.mark.parametrize("depth,allowed", [(2, True), (1, False)])
def test_fp8_append_needs_the_two_tile_loop(tmp_path, depth, allowed):
    r = _compile(tmp_path, f"stream_tiles<Half, 1, kPgFp8Append, {depth}>(a, st, qf, 0, 0, 0, 1, 1, 0);")
    assert (r.returncode == 0) == allowed, r.stderr[-2000:]
    assert allowed or "two-tile loop" in r.stderr
