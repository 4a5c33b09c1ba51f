"""Direct loads to LDS (csrc/dma.h) take their LDS address from m0, and so do loads of the compiler's own builtin: neither
may leave the other's address behind.  Read off the assembly of a kernel that mixes them."""

import re
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "nanovllm-voxcpm_amd" / "csrc"

KERNEL = """
#include "dma.h"
extern "C" __global__ void probe(const char* src, uint32_t* out) {
  __shared__ char lds[16384];
  const uint32_t voff = threadIdx.x * 16, to = __builtin_amdgcn_readfirstlane(mlora::lds_address(lds));
  auto builtin = [&](int at) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) uint32_t*)(src + voff + at),
                                     (__attribute__((address_space(3))) uint32_t*)(lds), 4, 0, 0);
  };
  builtin(0);
  mlora::dma16(src, voff, to + 8192);
  builtin(4096);
  mlora::wait_loads<0>();
  __syncthreads();
  out[threadIdx.x] = *(uint32_t*)(lds + threadIdx.x * 4);
}
"""


def test_every_direct_load_finds_its_own_address_in_m0(tmp_path):
    src, asm = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(KERNEL)
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", f"-I{CSRC}", f"-I{CSRC.parent.parent / 'include'}", "-S",
                    "--cuda-device-only", str(src), "-o", str(asm)], check=True)
    steps = re.findall(r"^\s+(s_\w+ m0,.*|global_load_lds_\w+)", asm.read_text(), flags=re.M)
    assert [bool(re.match(r"s_\w+ m0", s)) for s in steps] == [True, False] * 3, steps
    addresses = [s.split("m0,")[1].strip() for s in steps[::2]]
    assert addresses[0] == addresses[2] != addresses[1], addresses
