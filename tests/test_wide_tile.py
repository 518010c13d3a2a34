"""What the compiler makes of `csrc/wide_tile.h`, looked at without a GPU."""

import re
import subprocess

import pytest

from atomserve_amd.kernels import build

KERNEL = """
#include "wide_tile.h"
extern "C" __global__ void copies(const char* p, int bytes, char* out) {
  __shared__ __attribute__((aligned(128))) char lds[2048];
  typedef __attribute__((address_space(3))) char lds_char;
  const __amdgpu_buffer_rsrc_t buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p), 0, bytes, 0x00020000);
  const unsigned at = threadIdx.x * 16;
  __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, (__attribute__((address_space(3))) void*)lds, 16, at, 0, 0, 0);
  wide::copy_to_lds(buf, at, 1024, (unsigned)(uintptr_t)(lds_char*)lds + 1024);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, (__attribute__((address_space(3))) void*)lds, 16, at, 2048, 0, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  out[at] = lds[at];
}
"""


def test_a_copy_beside_the_large_tiles_goes_where_it_is_told(tmp_path):
    """The instruction takes its place in LDS from a register that the large tile's copy sets in inline assembly: a copy by the builtin to the
    same place as the one before has to set it again."""
    try:
        hipcc = build._hipcc()
    except build.BuildError:
        pytest.skip("no hipcc")
    source, listing = tmp_path / "copies.hip", tmp_path / "copies.s"
    source.write_text(KERNEL)
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC")]
    done = subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", "-I", build.CSRC, str(source), "-o", str(listing)],
                          capture_output=True, text=True, timeout=100)  # fmt: skip
    assert done.returncode == 0, done.stderr
    order = re.findall(r"^\s+(s_mov_b32 m0|buffer_load_dwordx4 .* lds)", listing.read_text(), re.M)
    assert [o[:8] for o in order] == ["s_mov_b3", "buffer_l"] * 3
