"""The cross-lane helpers of bq_device.hpp that are written in inline asm keep
the wait states that gfx950 asks for between a vector write and a DPP or lane-
swap read of the same register (two).  The compiler counts them for its own
instructions and does not see the writes inside an asm block, so the helpers
end on the wait themselves.  Compiled here, read from the assembly: no GPU."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mojo-gemma4-cpu_amd")

# each kernel reads the register its helper writes last in the next instruction
SOURCE = r"""
#include "bq_device.hpp"
using namespace bq;
template <int ST> __device__ void swap_after_bfly(float* x) {
  float v[8], lo, hi;
  for (int i = 0; i < 8; ++i) v[i] = x[64 * i + threadIdx.x];
  dpp_bfly8<ST>(v, x[600 + threadIdx.x]);
  row_exchange<16>(v[6], v[7], lo, hi);
  x[threadIdx.x] = lo;
  x[64 + threadIdx.x] = hi;
  for (int i = 0; i < 6; ++i) x[128 + 64 * i + threadIdx.x] = v[i];
}
extern "C" __global__ void k_swap1(float* x) { swap_after_bfly<1>(x); }
extern "C" __global__ void k_swap8(float* x) { swap_after_bfly<8>(x); }
extern "C" __global__ void k_dpp_after_max(float* x) {
  float v[4];
  for (int i = 0; i < 4; ++i) v[i] = x[64 * i + threadIdx.x];
  row_max16_x4(v);
  x[threadIdx.x] = row_add_shl<1>(v[3]);
  for (int i = 0; i < 3; ++i) x[64 + 64 * i + threadIdx.x] = v[i];
}
"""


def registers(op):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", op)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(r"v(\d+)", op)
    return {int(m[1])} if m else set()


def closest(body):
    """{kind: fewest wait states between a vector write and the cross-lane read
    of the register} over a kernel's straight-line code."""
    now, wrote, least = 0, {}, {}
    for line in body.splitlines():
        line = line.split(";")[0].strip()
        m = re.match(r"([sv]_\w+|\w+_(?:load|store)\w*)\s*(.*)", line)
        if not m:
            continue
        name, rest = m.groups()
        if name == "s_nop":
            now += int(rest, 0) + 1
            continue
        ops = [o.strip().split(" ")[0] for o in rest.split(",")]
        swap = name.startswith("v_permlane")
        if swap or re.search(r"quad_perm|row_", rest):
            kind = "swap" if swap else "dpp"
            for r in (registers(ops[0]) if swap else set()) | registers(ops[1]):
                if r in wrote:
                    least[kind] = min(least.get(kind, 99), now - wrote[r] - 1)
        if name.startswith("v_"):
            for r in registers(ops[0]) | (registers(ops[1]) if swap else set()):
                wrote[r] = now
        now += 1
    return least


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    spec = importlib.util.spec_from_file_location("bq_build", os.path.join(PKG, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not shutil.which(build.HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("waits")
    (d / "waits.hip").write_text(SOURCE)
    subprocess.run([build.HIPCC, *build.CFLAGS, "-I", build.CSRC, "--cuda-device-only", "-S",
                    str(d / "waits.hip"), "-o", str(d / "waits.s")], check=True, capture_output=True)
    text = (d / "waits.s").read_text()
    return {n: re.search(rf"^{n}:(.*?)s_endpgm", text, re.S | re.M)[1]
            for n in ("k_swap1", "k_swap8", "k_dpp_after_max")}


@pytest.mark.parametrize("name,kind", [("k_swap1", "swap"), ("k_swap8", "swap"), ("k_dpp_after_max", "dpp")])
def test_wait_states_after_asm(kernels, name, kind):
    assert closest(kernels[name])[kind] >= 2, kernels[name]
